"""Decode over trellis-coded rows: the encoder's search rides in the attention launch, which attends to the rows in front of the
position; the combiner adds the new rows.  Against the general path (option 3: encoder launches first, every key in the
attention launch), from the empty cache to the last row of the container."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kk", [4, 5])
@pytest.mark.parametrize("M,ctx,opts", [(1, 0, []), (2, 0, []), (1, 1, []), (2, 31, []), (2, 32, []), (1, 500, [(4, 1)]), (2, 1023, [(1, 200)]),
                                        (2, 2046, []), (1, 2047, []), (1, 700, [(11, 1)]), (2, 65, [(11, 1)])])
def test_against_the_general_path(native, kk, M, ctx, opts):
    from yasakani_amd import kvqp
    rng = np.random.default_rng(100 * M + ctx + kk)
    bf16 = (11, 1) in opts

    def rows(n, heads):
        x = rng.standard_normal((n, heads, 256)).astype(np.float32)
        return native.bf16_bits(x) if bf16 else x.astype(np.float16)

    with native.KvCache(n_layers=2, max_ctx=2048, head_dim=256, max_rows=2048) as kv:
        kv.set_profile(kvqp.synthetic(layers=2, kk=kk, seed=11))
        for key, val in opts:
            kv.set_opt(key, val)
        if ctx:
            kv.append_host(1, rows(ctx, 4), rows(ctx, 4), 0)
        q, k, v = rows(M, 24), rows(M, 4), rows(M, 4)
        kv.poison_workspace()
        out = kv.layer_call(1, q, k, v, ctx)
        kv.set_opt(3, 1)
        kv.poison_workspace()
        ref = kv.layer_call(1, q, k, v, ctx)
    if bf16:
        out, ref = native.bf16_to_f32(out), native.bf16_to_f32(ref)
    out, ref = out.astype(np.float32), ref.astype(np.float32)
    assert np.isfinite(out).all()
    # the same codes; the general path rounds P (times the V scale) and its partials to fp16, both round the output (bf16: 2^-8 each)
    assert np.linalg.norm(out - ref) <= (1e-3 + (2 * 2.0 ** -8 if bf16 else 0)) * np.linalg.norm(ref)


@pytest.mark.parametrize("kk", [4, 5])
def test_splits_change_with_the_position(native, kk):
    """A container of more than 98,304 tokens: half of the launched splits are in use up to that position, all beyond it."""
    from yasakani_amd import kvqp
    rng = np.random.default_rng(kk)
    half = lambda n, heads: rng.standard_normal((n, heads, 256)).astype(np.float16)    # noqa: E731
    with native.KvCache(n_layers=1, max_ctx=98304 + 512, head_dim=256, max_rows=2048) as kv:
        kv.set_profile(kvqp.synthetic(layers=1, kk=kk, seed=11))
        k, v = half(2048, 4), half(2048, 4)
        for at in range(0, 98304 + 2048, 2048):
            n = min(2048, 98304 + 300 - at)
            kv.append_host(0, np.roll(k, at // 2048, axis=2)[:n], np.roll(v, at // 2048 + 1, axis=0)[:n], at)
        for ctx, M in ((0, 2), (1, 1), (300, 1), (4095, 2), (98302, 2), (98303, 2), (98304, 1), (98305, 2), (98304 + 511, 1), (98304 + 510, 2)):
            q, kn, vn = half(M, 24), half(M, 4), half(M, 4)
            got = []
            for splits in (0, 48):
                kv.set_opt(1, splits)
                kv.poison_workspace()
                got.append(kv.layer_call(0, q, kn, vn, ctx).astype(np.float32))
            assert np.isfinite(got[0]).all(), ctx
            # other splits: partials and outputs rounded to fp16 once each (2^-11), sums in fp32
            assert np.linalg.norm(got[0] - got[1]) <= 1e-3 * np.linalg.norm(got[1]), ctx


@pytest.mark.parametrize("kk", [4, 5])
@pytest.mark.parametrize("M,bad,which", [(1, 0, "k"), (2, 0, "k"), (2, 1, "k"), (1, 0, "v"), (1, 0, "q"), (2, 1, "q")])
def test_rows_that_are_not_numbers(native, kk, M, bad, which):
    """A new K row with a NaN has a NaN scale: a query that sees its key has no softmax, whichever launch attends to the key.
    500 tokens: the new keys share a workgroup's tiles with cached ones in the general path, too."""
    from yasakani_amd import kvqp
    rng = np.random.default_rng(kk + M)
    half = lambda n, heads: rng.standard_normal((n, heads, 256)).astype(np.float16)    # noqa: E731
    with native.KvCache(n_layers=1, max_ctx=1024, head_dim=256, max_rows=512) as kv:
        kv.set_profile(kvqp.synthetic(layers=1, kk=kk, seed=11))
        kv.append_host(0, half(500, 4), half(500, 4), 0)
        new = dict(q=half(M, 24), k=half(M, 4), v=half(M, 4))
        new[which][bad, 2, 17] = np.nan
        out = kv.layer_call(0, new["q"], new["k"], new["v"], 500).astype(np.float32)
        kv.set_opt(3, 1)
        ref = kv.layer_call(0, new["q"], new["k"], new["v"], 500).astype(np.float32)
    heads = slice(2, 3) if which == "q" else slice(12, 18)         # query head 2, or the query heads of KV head 2
    touched = np.zeros(out.shape[:2], bool)
    touched[bad if which == "q" else slice(bad, None), heads] = True
    assert np.isnan(out[touched]).all() if which == "v" else not out[touched].any()
    assert np.array_equal(np.isnan(out), np.isnan(ref)) and np.array_equal(out[touched] == 0, ref[touched] == 0)
    # as in test_against_the_general_path
    assert np.linalg.norm(out[~touched] - ref[~touched]) <= 1e-3 * np.linalg.norm(ref[~touched])


@pytest.mark.parametrize("kk", [4, 5])
@pytest.mark.parametrize("heads,n_mult", [(1, 1), (1, 16), (2, 9), (3, 2)])
@pytest.mark.parametrize("M,post", [(1, False), (2, False), (3, False), (5, False), (16, False), (17, False), (1, True)])
def test_rows_as_the_oracle_codes_them(native, oracle, kk, heads, n_mult, M, post):
    """Rows coded by the combiner of a decode pass (M <= 2), by the attention launch of a window (up to 16 rows) and by a launch of their own
    (wider; `post`: fp32 rows), in handles whose rows do not fill the waves of a workgroup (2 to 102 rows, four to a workgroup), with one
    multiplier and with as many as a profile may have."""
    from yasakani_amd import kvqp
    blob = kvqp.synthetic(layers=1, kv_heads=heads, kk=kk, seed=kk, n_mult=n_mult, mu=M == 2)
    rng = np.random.default_rng(10 * M + heads)
    k, v = (rng.standard_normal((M, heads, 256)).astype(np.float16) for _ in range(2))
    k[0, 0] = 0                                                    # a row of zeros: its residual has no length
    q = rng.standard_normal((M, 6 * heads, 256)).astype(np.float16)
    pos = 256 - M                                                  # up to the last row of the container
    with native.KvCache(n_heads=6 * heads, n_kv_heads=heads, max_ctx=256, head_dim=256, max_rows=24) as kv:
        kv.set_profile(blob)
        if post:
            kv.append256_f32_host(0, k.astype(np.float32), v.astype(np.float32), pos, rotate=False)
        else:
            kv.layer_call(0, q, k, v, pos)
        kw, ks, vw, vs = kv.export_rows(0, pos, M)
    for kind, x, words, scales in ((0, k, kw, ks), (1, v, vw, vs)):
        for h in range(heads):
            ref = oracle.tb_encode_rows(blob, np.full(M, 2 * h + kind, np.int32), np.arange(M, dtype=np.int32), x[:, h].astype(np.float32))
            assert np.array_equal(words[h], ref["words"][:, :8 * kk]), (kind, h)
            assert np.array_equal(np.asarray(scales[h]).view(np.uint32), np.asarray(ref["scale"]).view(np.uint32)), (kind, h)


@pytest.mark.parametrize("kk", [4, 5])
@pytest.mark.parametrize("M", [3, 16])                        # 17: both passes below would be the same launches; see the test above and the next
@pytest.mark.parametrize("pos,splits", [(0, 0), (30, 0), (250, 0), (250, 1), (250, 97), (1008 - 3, 0)])
@pytest.mark.parametrize("siblings", [False, True])
def test_windows_store_every_row(native, kk, M, pos, splits, siblings):
    """Rows stored by the attention launch of a window: over two tiles, in a share of one split and of many, in front of the end of the
    container, and siblings (a depth table of zeros) that no query row's tiles reach.  Against the rows of an append."""
    from yasakani_amd import kvqp
    rng = np.random.default_rng(M + pos)
    half = lambda n, heads: rng.standard_normal((n, heads, 256)).astype(np.float16)    # noqa: E731
    blob = kvqp.synthetic(layers=1, kk=kk, seed=11, mu=True)
    q, k, v = half(M, 24), half(M, 4), half(M, 4)
    old_k, old_v = half(max(pos, 1), 4), half(max(pos, 1), 4)
    n = min(M, 1024 - pos)
    stored, outs = [], []
    for fused in (True, False):
        with native.KvCache(max_ctx=1024, head_dim=256, max_rows=1024) as kv:
            kv.set_profile(blob)
            kv.set_opt(2, splits)
            if pos:
                kv.append_host(0, old_k[:pos], old_v[:pos], 0)
            depth = np.zeros(M, np.uint8) if siblings else None
            if fused:
                kv.poison_workspace()
                outs.append(kv.layer_call(0, q, k, v, pos, depth))
            else:
                kv.append_host(0, k, v, pos)
                outs.append(kv.layer_call(0, q, None, None, pos, depth))
            stored.append([np.ascontiguousarray(x).view(np.uint8) for x in kv.export_rows(0, 0, pos + n)])
    for a, b in zip(*stored):
        assert np.array_equal(a, b)
    a, b = (x.astype(np.float32) for x in outs)
    # the same rows, other split bounds: partials and outputs rounded to fp16 once each (2^-11), sums in fp32
    assert np.isfinite(a).all() and np.linalg.norm(a - b) <= 1e-3 * np.linalg.norm(b)


@pytest.mark.parametrize("form", ["kv4", "kv5", "256"])
@pytest.mark.parametrize("M", [1, 2, 3, 16, 17, 21, 22, 32, 33])    # edges of who stores the rows, and of a row block (21 rows are one, 22 are two)
@pytest.mark.parametrize("bf16", [False, True])
def test_passes_read_the_rows_they_store(native, form, M, bf16):
    """A pass over rows that others occupied, then the same pass over its own: the same launches, so the same bits, unless the first one read
    something it had yet to store.  One split and many, over two tiles, up to the end of the container; a depth table."""
    from yasakani_amd import kvqp
    rng = np.random.default_rng(M)

    def rows(n, heads):
        x = rng.standard_normal((n, heads, 256)).astype(np.float32)
        return native.bf16_bits(x) if bf16 else x.astype(np.float16)

    with native.KvCache(max_ctx=1024, head_dim=256, max_rows=1024) as kv:
        if form != "256":
            kv.set_profile(kvqp.synthetic(layers=1, kk=int(form[2]), seed=11, mu=True))
        kv.set_opt(11, int(bf16))
        kv.append_host(0, rows(1024, 4), rows(1024, 4), 0)
        q, k, v = rows(M, 24), rows(M, 4), rows(M, 4)
        for pos, splits, tree in ((0, 0, False), (30, 3, True), (250, 1, False), (250, 97, False), (700, 5, True), (700, 0, False), (1024 - M, 0, False)):
            kv.set_opt(2, splits)
            if M <= 2:
                kv.set_opt(1, splits)
            depth = (np.arange(M) // 2).astype(np.uint8) if tree else None
            kv.append_host(0, rows(M, 4), rows(M, 4), pos)
            outs = []
            for _ in range(2):
                kv.poison_workspace()
                outs.append(kv.layer_call(0, q, k, v, pos, depth).view(np.uint16))
            f = native.bf16_to_f32(outs[0]) if bf16 else outs[0].view(np.float16)
            assert np.isfinite(f.astype(np.float32)).all(), (pos, splits)
            assert np.array_equal(outs[0], outs[1]), (pos, splits)
