"""The combiner of decode, small windows and multi-stream passes where its sets of 64 splits begin and end: a split more or less than
a set holds, the most splits there are, rows of splits nobody wrote, the inverse rotation, and a stream whose share spans sets; and the combiner of prefill slices, which takes 1 to 8 rows at a time by the splits the device has chosen."""
import numpy as np
import pytest

from oracle import yko
from tests.tolerances import assert_attn_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S", [1, 4, 15, 16, 17, 63, 64, 65, 127, 128, 129, 255, 256])
@pytest.mark.parametrize("M,ctx", [(1, 20000), (2, 700)])
def test_decode_splits_around_a_set(native, oracle, M, ctx, S):
    """20,000 keys use every split (two tiles each), 700 leave most of them without a row."""
    q, k, v, kn, vn, _ = oracle.make_inputs(9100 + S, ctx, M)
    cap = (ctx + M + 255) // 256 * 256
    oc = oracle.Cache(cap)
    oc.append(k, v, 0)
    with native.KvCache(max_ctx=cap) as kv:
        kv.import_rows(0, 0, oc.kc[:, :ctx], oc.ks[:, :ctx], oc.vc[:, :ctx], oc.vs[:, :ctx])
        kv.poison_workspace()                                   # rows of splits that are not in use hold NaN
        kv.set_opt(1, S)
        out = kv.layer_call(0, q, kn, vn, ctx)
        oc.append(kn, vn, ctx)
        ref = oc.attend_f32(q, ctx, threads=8, want_f32=True)[1]
        assert_attn_close(out, ref, f"{S} splits")
        kv.set_opt(4, 1)
        back = kv.layer_call(0, q, None, None, ctx)
    # option key 4: 128-point Hadamard transform, 1/16, signs.  A scaled orthogonal map keeps the relative L2 error of the result it
    # is given (at most 1e-3); the rounding to fp16 behind it adds half a spacing a value, 2^-11 at most
    h = np.array([[1.0]])
    for _ in range(7):
        h = np.block([[h, h], [h, -h]])
    want = np.asarray(ref, np.float64) @ h / 16.0 * yko.kvx_signs()[:128]
    assert np.linalg.norm(back - want) <= (1e-3 + 2.0 ** -11) * np.linalg.norm(want)


def _slice_splits(kvh, M, ctx, capacity):
    """Splits the device uses for a slice: chunk_splits of the host, chunk_price of the device, in Python."""
    base = kvh * ((6 * M + 127) // 128)

    def launched(m):
        b = kvh * ((6 * m + 127) // 128)
        fill = lambda s: b * s / (256.0 * ((b * s + 255) // 256)) - 0.005 * s
        return max(range(1, max(1, min(32, 12288 // m, capacity // 256, 2048 // b)) + 1), key=lambda s: (fill(s), -s))

    def price(s):
        lo, hi = ((ctx + min(M, 22) + 31) // 32 * 16 // s + 288), ((ctx + M + 31) // 32 * 16 // s + 288)
        n = base * s
        idle = (256 - (n & 255)) & 255
        t = max(hi, (n >> 1) * (lo + hi) // 256 + lo * idle // 256)
        return t + 96 + M * s // 13 if s > 1 else t

    return min(range(1, launched(M) + 1), key=lambda s: (price(s), s))


@pytest.mark.parametrize("kvh,M,ctx,splits", [(1, 301, 200, 3), (1, 200, 300, 4), (1, 100, 300, 5), (1, 65, 500, 7), (1, 65, 600, 8), (1, 65, 700, 9),
                                              (1, 65, 1000, 10), (1, 129, 5200, 16), (1, 65, 2700, 17), (1, 65, 8000, 27),
                                              (2, 1000, 100, 2), (1, 682, 1000, 4), (1, 683, 600, 4), (1, 683, 1400, 5),
                                              (3, 1820, 2700, 2), (3, 1821, 2700, 2)])
def test_slice_splits_of_every_size(native, oracle, kvh, M, ctx, splits):
    """Slices of 2 to 27 splits: a split lane of the combiner takes 1, 2, 4 or 8 partials, both sides of every line.  Then rows
    for less and more than the 4,096 waves launched (4,092, 4,098, 12,000), and for one and for eight rows a step (32,760 and 32,778, 2 at
    the end)."""
    assert _slice_splits(kvh, M, ctx, 8192) == splits
    q, k, v, kn, vn, _ = oracle.make_inputs(9300 + splits, ctx, M, 6 * kvh, kvh)
    oc = oracle.Cache(8192, 6 * kvh, kvh)
    oc.append(k, v, 0)
    with native.KvCache(max_ctx=8192, n_heads=6 * kvh, n_kv_heads=kvh, max_rows=M) as kv:
        kv.import_rows(0, 0, oc.kc[:, :ctx], oc.ks[:, :ctx], oc.vc[:, :ctx], oc.vs[:, :ctx])
        kv.poison_workspace()
        out = kv.layer_call(0, q, kn, vn, ctx)
    oc.append(kn, vn, ctx)
    assert_attn_close(out, oc.attend_f32(q, ctx, threads=8, want_f32=True)[1], f"{splits} splits")


def test_stream_whose_share_spans_sets(native, oracle):
    lens = [9000, 40]
    with native.KvCache(n_layers=2, max_ctx=9216, max_rows=2) as kv:
        refs = []
        for s, n in enumerate(lens):
            _, k, v, _, _, _ = oracle.make_inputs(9200 + s, n, 1)
            oc = oracle.Cache(9216)
            oc.append(k, v, 0)
            kv.import_rows(s, 0, oc.kc[:, :n], oc.ks[:, :n], oc.vc[:, :n], oc.vs[:, :n])
            refs.append(oc)
        rng = np.random.default_rng(9)
        q, k, v = (rng.standard_normal((2, h, 128)).astype(np.float16) for h in (24, 4, 4))
        kv.poison_workspace()
        out = kv.ms_call(q, k, v, np.array(lens, np.int32), np.array([0, 1], np.int32))
        for t, n in enumerate(lens):
            refs[t].append(k[t:t + 1], v[t:t + 1], n)
            assert_attn_close(out[t:t + 1], refs[t].attend_f32(q[t:t + 1], n, want_f32=True)[1], f"stream of {n}")


@pytest.mark.parametrize("M", [1, 2, 5])
@pytest.mark.parametrize("unrot", [0, 1])
def test_row_without_a_softmax_is_zero(native, oracle, M, unrot):
    """A cached key whose scale is infinite leaves query heads that score it above everything without a softmax: their rows are zeros,
    with and without the inverse rotation, and the other KV heads' rows keep their bits."""
    ctx = 3000
    q, k, v, _, _, _ = oracle.make_inputs(9400 + M, ctx, M)
    q[:, :6] = 1.0
    k[77, 0] = 1.0                                              # codes 7 in every channel: the score of key 77 is +inf below
    oc = oracle.Cache(3072)
    oc.append(k, v, 0)
    outs = []
    for bits in (oc.ks[0, 77, 0], 0x7c00):
        ks = oc.ks.copy()
        ks[0, 77, 0] = bits
        with native.KvCache(max_ctx=3072) as kv:
            kv.set_opt(4, unrot)
            kv.import_rows(0, 0, oc.kc[:, :ctx], ks[:, :ctx], oc.vc[:, :ctx], oc.vs[:, :ctx])
            outs.append(kv.layer_call(0, q, None, None, ctx - M).view(np.uint16))
    assert np.array_equal(outs[0][:, 6:], outs[1][:, 6:])
    assert outs[0][:, :6].any() and not (outs[1][:, :6] & 0x7fff).any()
