"""Queries over 128-channel rows: a power of two moved from the queries into the cached keys changes no bit of the result.  Windows and prefill
slices take the whole fp16 range, down to subnormals and up to the largest finite values; decode passes (1 and 2 rows, streams) take
queries up to a quarter of it and, on the odd channels, lose what lies below 2^-22."""
import numpy as np
import pytest

from tests.tolerances import assert_attn_close

pytestmark = pytest.mark.gpu

CTX = 500


def _rows(M, s):
    """q, k, v so that q * 2^s and k * 2^-s are fp16 values, and so are the scales of the keys' groups (normal ones: the codes stay)."""
    rng = np.random.default_rng(700 + M)
    if s < 0:                                                   # multiples of 2^-7 below 4: of 2^-24 once scaled by 2^-17, of 2^-22 by 2^-15
        q = np.clip(np.round(rng.standard_normal((M, 24, 128)) * 128), -511, 511) / 128
        k = np.clip(rng.standard_normal((CTX + M, 4, 128)), -4, 4) / 16
    else:                                                       # up to 3.99, 65,372 once scaled by 2^14 (16,343 by 2^12); every group of k reaches 8, values are multiples of 2^-9
        q = rng.choice([-1.0, 1.0], (M, 24, 128)) * rng.uniform(0.25, 3.99, (M, 24, 128))
        k = np.round(np.clip(rng.standard_normal((CTX + M, 4, 128)), -2, 2) * 512) / 512
        k[:, :, ::32] = 8.0
    return q.astype(np.float16), k.astype(np.float16), rng.standard_normal((CTX + M, 4, 128)).astype(np.float16)


@pytest.mark.parametrize("s", [-17, 14])
@pytest.mark.parametrize("M,mid", [(3, 8), (8, 8), (9, 8), (10, 16), (16, 8), (22, 8), (64, 8), (130, 8)])
def test_a_power_of_two_moves_from_query_to_key(native, oracle, M, mid, s):
    q, k, v = _rows(M, s)
    qs, ks = (np.ldexp(q.astype(np.float64), s), np.ldexp(k.astype(np.float64), -s))
    assert np.array_equal(qs, qs.astype(np.float16)) and np.array_equal(ks, ks.astype(np.float16))
    outs = []
    for qq, kk in ((q, k), (qs.astype(np.float16), ks.astype(np.float16))):
        with native.KvCache(max_ctx=768, max_rows=max(M, 64)) as kv:
            kv.set_opt(8, mid)
            kv.append_host(0, kk[:CTX], v[:CTX], 0)
            outs.append((kv.layer_call(0, qq, kk[CTX:], v[CTX:], CTX), kv.export_rows(0, 0, CTX + M)[0]))
    assert np.array_equal(outs[0][1], outs[1][1])               # the keys' codes
    oc = oracle.Cache(768)
    oc.append(k, v, 0)
    assert_attn_close(outs[0][0], oc.attend_f32(q, CTX, threads=8, want_f32=True)[1], f"M={M}", two_spacings=True)
    assert np.array_equal(outs[0][0].view(np.uint16), outs[1][0].view(np.uint16))


@pytest.mark.parametrize("s", [-15, 12])
@pytest.mark.parametrize("M,streams", [(1, False), (2, False), (5, True)])
def test_decode_within_its_range(native, oracle, M, streams, s):
    q, k, v = _rows(M, s)
    outs = []
    for qq, kk in ((q, k), (np.ldexp(q.astype(np.float64), s).astype(np.float16), np.ldexp(k.astype(np.float64), -s).astype(np.float16))):
        with native.KvCache(n_layers=M if streams else 1, max_ctx=768) as kv:
            for layer in range(M if streams else 1):
                kv.append_host(layer, kk[:CTX], v[:CTX], 0)
            outs.append(kv.ms_call(qq, kk[CTX:], v[CTX:], [CTX] * M, list(range(M))) if streams else kv.layer_call(0, qq, kk[CTX:], v[CTX:], CTX))
    for t in range(M) if streams else [slice(0, M)]:
        new = slice(CTX + t, CTX + t + 1) if streams else slice(CTX, CTX + M)
        oc = oracle.Cache(768)
        oc.append(np.concatenate([k[:CTX], k[new]]), np.concatenate([v[:CTX], v[new]]), 0)
        rows = slice(t, t + 1) if streams else t
        assert_attn_close(outs[0][rows], oc.attend_f32(q[rows], CTX, want_f32=True)[1], f"rows {rows}", two_spacings=True)
    assert np.array_equal(outs[0].view(np.uint16), outs[1].view(np.uint16))
