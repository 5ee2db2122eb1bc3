"""Prefill chunks (more than 64 rows): the number of splits is chosen on the device from the position, and a slice that uses
one writes its output without a combiner.  Against the oracle, and against the decode kernel forced on the same rows."""
import numpy as np
import pytest

from tests.tolerances import assert_attn_close

pytestmark = pytest.mark.gpu


# rows around a row block (21 1/3 tokens), a slice (2,048) and its tail; contexts on both sides of one split
@pytest.mark.parametrize("M,ctx,max_ctx,paged", [
    (65, 0, 4096, False), (65, 3000, 32768, True), (85, 31, 512, False), (129, 700, 8192, True), (683, 0, 8192, False),
    (300, 5000, 32768, False), (1100, 33, 1280, True),
])
def test_against_the_oracle(native, oracle, M, ctx, max_ctx, paged):
    q, k, v, kn, vn, _ = oracle.make_inputs(M, ctx, M)
    oc = oracle.Cache(max_ctx)
    with native.KvCache(max_ctx=max_ctx, max_rows=M, paged=paged) as kv:
        if paged:
            kv.set_page_table(np.random.default_rng(M).permutation(max_ctx // 256).astype(np.int32))
        if ctx:
            oc.append(k, v, 0)
            kv.import_rows(0, 0, oc.kc[:, :ctx], oc.ks[:, :ctx], oc.vc[:, :ctx], oc.vs[:, :ctx])
        kv.poison_workspace()
        out = kv.layer_call(0, q, kn, vn, ctx)
        got = kv.export_rows(0, ctx, M)
    oc.append(kn, vn, ctx)
    for a, b in zip(got, (oc.kc, oc.ks, oc.vc, oc.vs)):
        assert (a == b[:, ctx:ctx + M]).all(), "appended rows differ"
    # rows of a handful of keys: two fp16 spacings on values in [2, 4] (tolerances.py)
    assert_attn_close(out, oc.attend_f32(q, ctx, None, threads=8, want_f32=True)[1], f"M={M} ctx={ctx}", two_spacings=ctx < 64)


# 2,049 and 2,100 rows: a second slice of 1 and 52 rows.  Option 4 (inverse rotation) and forced split counts keep the combiner.
# 661 and 662 rows: one split gives 124 and 128 workgroups, both sides of the two forms of the kernel, with one split in use and with several.
# Both sides round V and P to fp16 and sum in fp32 in another order: 1e-3 between them, two bf16 roundings (2^-8 each) on top.
@pytest.mark.parametrize("M,ctx,opts", [(2049, 0, []), (2100, 4000, []), (1500, 0, [(4, 1)]), (1500, 2000, [(4, 1)]), (700, 9000, [(2, 5)]),
                                        (333, 0, [(11, 1)]), (1500, 7000, [(11, 1)]), (90, 12000, [(10, 128)]),
                                        (661, 0, []), (662, 0, []), (661, 6000, [(11, 1)]), (662, 6000, [(11, 1)]), (661, 6000, []), (662, 6000, [])])
def test_against_the_decode_kernel(native, M, ctx, opts):
    rng = np.random.default_rng(M + ctx)
    bf16 = (11, 1) in opts

    def rows(n, heads):
        x = rng.standard_normal((n, heads, 128)).astype(np.float32)
        return (x.view(np.uint32) >> 16).astype(np.uint16).view(np.float16) if bf16 else x.astype(np.float16)

    with native.KvCache(max_ctx=16384, max_rows=max(M, 2048)) as kv:
        for key, val in opts:
            kv.set_opt(key, val)
        for p in range(0, ctx, 2048):
            n = min(2048, ctx - p)
            kv.append_host(0, rows(n, 4), rows(n, 4), p)
        q, k, v = rows(M, 24), rows(M, 4), rows(M, 4)
        kv.poison_workspace()
        out = kv.layer_call(0, q, k, v, ctx)
        kv.set_opt(3, 1)
        ref = kv.layer_call(0, q, k, v, ctx)
    wide = (lambda x: (x.view(np.uint16).astype(np.uint32) << 16).view(np.float32)) if bf16 else (lambda x: x.astype(np.float32))
    out, ref = wide(out), wide(ref)
    assert np.isfinite(out).all()
    assert np.linalg.norm(out - ref) <= (1e-3 + (2 * 2.0 ** -8 if bf16 else 0)) * np.linalg.norm(ref)
    per_row = np.linalg.norm(out - ref, axis=2) / np.linalg.norm(ref, axis=2)
    assert per_row.max() <= (4e-3 if not bf16 else 1.2e-2)


# the 256-channel formats: slices of 1,024 tokens on the wide kernels, row blocks of equal height; the same comparison
@pytest.mark.parametrize("kk", [0, 4, 5])
# 107 and 140 rows: six row blocks and seven, the last of six and five waves of rows, on either of the int4 kernels
@pytest.mark.parametrize("M,ctx,opts", [(65, 0, []), (22, 500, []), (43, 100, []), (107, 300, []), (140, 300, []), (1025, 0, []), (1100, 700, [(4, 1)]), (200, 3000, [(2, 3)])])
def test_256_channel_rows(native, kk, M, ctx, opts):
    from yasakani_amd import kvqp
    rng = np.random.default_rng(M + ctx + kk)

    def rows(n, heads):
        return rng.standard_normal((n, heads, 256)).astype(np.float16)

    with native.KvCache(max_ctx=8192, head_dim=256, max_rows=max(M, 1024)) as kv:
        if kk:
            kv.set_profile(kvqp.synthetic(layers=1, kk=kk, seed=5))
        for key, val in opts:
            kv.set_opt(key, val)
        for p in range(0, ctx, 1024):
            n = min(1024, ctx - p)
            kv.append_host(0, rows(n, 4), rows(n, 4), p)
        q, k, v = rows(M, 24), rows(M, 4), rows(M, 4)
        kv.poison_workspace()
        out = kv.layer_call(0, q, k, v, ctx).astype(np.float32)
        kv.set_opt(3, 1)
        ref = kv.layer_call(0, q, k, v, ctx).astype(np.float32)
    assert np.isfinite(out).all()
    assert np.linalg.norm(out - ref) <= 1e-3 * np.linalg.norm(ref)
    assert (np.linalg.norm(out - ref, axis=2) / np.linalg.norm(ref, axis=2)).max() <= 4e-3


@pytest.mark.parametrize("bf16", [0, 1])
@pytest.mark.parametrize("ctx", [0, 400])
def test_query_rows_that_are_not_numbers(native, ctx, bf16):
    """A query row with a NaN has no softmax: zeros, from a slice that writes its own output rows (one split) as from one whose
    partials a combiner merges (a split count set by the caller)."""
    rng = np.random.default_rng(ctx)

    def rows(n, heads):
        x = rng.standard_normal((n, heads, 128)).astype(np.float32)
        return native.bf16_bits(x) if bf16 else x.astype(np.float16)

    M, bad = 150, [(0, 0), (77, 5), (78, 23), (149, 11)]
    with native.KvCache(max_ctx=1024, max_rows=512) as kv:
        kv.set_opt(11, bf16)
        if ctx:
            kv.append_host(0, rows(ctx, 4), rows(ctx, 4), 0)
        q, k, v = rows(M, 24), rows(M, 4), rows(M, 4)
        clean = kv.layer_call(0, q, k, v, ctx)
        for t, h in bad:
            q.view(np.uint16)[t, h, 40] = 0x7fc0 if bf16 else 0x7e00
        touched = np.zeros((M, 24), bool)
        touched[tuple(np.array(bad).T)] = True
        for splits in (0, 3):
            kv.set_opt(2, splits)
            kv.poison_workspace()
            out = kv.layer_call(0, q, k, v, ctx)
            assert not (out[touched].view(np.uint16) & 0x7fff).any(), splits
            if splits == 0:                                        # the other rows do not notice
                assert np.array_equal(out[~touched].view(np.uint16), clean[~touched].view(np.uint16))


@pytest.mark.parametrize("dim,max_rows,pairs", [(128, 64, 4096), (128, 128, 4096), (128, 2048, 10899), (256, 341, 4096), (256, 2048, 5376)])
def test_a_handle_reserves_what_its_slices_can_use(native, dim, max_rows, pairs):
    """24 * (2 dim + 8) bytes for each (token, split) pair; everything else this handle holds is below 2 MB."""
    import ctypes
    hip = ctypes.CDLL("libamdhip64.so")
    free, total = ctypes.c_size_t(), ctypes.c_size_t()

    def free_bytes():
        assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    with native.KvCache(max_ctx=256, max_rows=max_rows, head_dim=dim):
        pass                                                       # whatever the runtime itself keeps is there from now on
    before = free_bytes()
    with native.KvCache(max_ctx=32768 if max_rows > 64 else 256, max_rows=max_rows, head_dim=dim) as kv:
        used = before - free_bytes()
        cache = kv.max_ctx * 4 * (2 * (dim // 2) + (16 if dim == 128 else 8))
    assert used - cache <= pairs * 24 * (2 * dim + 8) + (10 << 20), used       # each of six allocations rounds up to 2 MB at most
