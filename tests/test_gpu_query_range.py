"""Windows and prefill slices over 128-channel rows take queries over the whole fp16 range: a power of two moved from the queries into the
cached keys changes no bit of the result, down to queries that are fp16 subnormals and up to the largest finite ones."""
import numpy as np
import pytest

from tests.tolerances import assert_attn_close

pytestmark = pytest.mark.gpu

CTX = 500


def _rows(M, s):
    """q, k, v so that q * 2^s and k * 2^-s are fp16 values, and so are the scales of the keys' groups (normal ones: the codes stay)."""
    rng = np.random.default_rng(700 + M)
    if s < 0:                                                   # multiples of 2^-7 below 4: of 2^-24 once scaled by 2^-17
        q = np.clip(np.round(rng.standard_normal((M, 24, 128)) * 128), -511, 511) / 128
        k = np.clip(rng.standard_normal((CTX + M, 4, 128)), -4, 4) / 16
    else:                                                       # up to 3.99, 65,372 once scaled by 2^14; every group of k reaches 8, values are multiples of 2^-9
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
