"""Multi-stream passes (batched decode): every row of a pass names its own KV container and position.  Checked against the
oracle run stream by stream on the same rows."""
import numpy as np
import pytest

from tolerances import assert_attn_close

pytestmark = pytest.mark.gpu

CTX = 1024
LENS = [300, 17, 900, 512, 0]                             # cached tokens per stream; the last stream is empty


def _streams(native, oracle, paged, seed=3):
    rng = np.random.default_rng(seed)
    kv = native.KvCache(n_layers=len(LENS), max_ctx=CTX, max_rows=64, paged=paged)
    if paged:
        for s in range(len(LENS)):
            kv.set_page_table(rng.permutation(CTX // 256).astype(np.int32), layer=s)
    refs = []
    for s, n in enumerate(LENS):
        ref = oracle.Cache(CTX)
        if n:
            _, k, v, _, _, _ = oracle.make_inputs(seed * 100 + s, n, 1)
            kv.append_host(s, k, v, 0)
            ref.append(k, v, 0)
        refs.append(ref)
    return kv, refs, rng


def _rows(rng, M):
    q = rng.standard_normal((M, 24, 128)).astype(np.float16)
    k = rng.standard_normal((M, 4, 128)).astype(np.float16)
    v = rng.standard_normal((M, 4, 128)).astype(np.float16)
    return q, k, v


@pytest.mark.parametrize("paged", [False, True])
def test_one_row_per_stream(native, oracle, paged):
    kv, refs, rng = _streams(native, oracle, paged)
    with kv:
        slots = np.array([2, 0, 4, 1, 3], np.int32)       # any order
        pos = np.array([LENS[s] for s in slots], np.int32)
        q, k, v = _rows(rng, len(slots))
        out = kv.ms_call(q, k, v, pos, slots)
        for t, s in enumerate(slots):
            refs[s].append(k[t:t + 1], v[t:t + 1], int(pos[t]))
            expect = refs[s].attend_f32(q[t:t + 1], int(pos[t]))
            assert_attn_close(out[t:t + 1], expect, f"row {t} stream {s}")
            # the appended row is what the single-stream append stores
            got = kv.export_rows(int(s), int(pos[t]), 1)
            assert np.array_equal(got[0], refs[s].kc[:, pos[t]:pos[t] + 1]) and np.array_equal(got[3], refs[s].vs[:, pos[t]:pos[t] + 1])


def test_rows_of_one_stream_follow_each_other(native, oracle):
    kv, refs, rng = _streams(native, oracle, False)
    with kv:
        # stream 0: its last token and two draft tokens; stream 2: one row; stream 0 rows see each other's keys
        slots = np.array([0, 0, 0, 2], np.int32)
        pos = np.array([300, 301, 302, 900], np.int32)
        q, k, v = _rows(rng, 4)
        out = kv.ms_call(q, k, v, pos, slots)
        refs[0].append(k[0:3], v[0:3], 300)
        assert_attn_close(out[0:3], refs[0].attend_f32(q[0:3], 300), "stream 0 window")     # row t sees keys [0, 300 + t]
        refs[2].append(k[3:4], v[3:4], 900)
        assert_attn_close(out[3:4], refs[2].attend_f32(q[3:4], 900), "stream 2")


@pytest.mark.parametrize("merge_in_launch", [0, 1])
def test_more_rows_than_sixteen_and_attend_only(native, oracle, merge_in_launch):
    kv, refs, rng = _streams(native, oracle, False)
    with kv:
        kv.set_opt(7, merge_in_launch)
        M = 24
        slots = (np.arange(M) % 4).astype(np.int32)
        pos = np.array([LENS[s] - 1 - (t // 4) for t, s in enumerate(slots)], np.int32)     # positions inside the cached part
        q, _, _ = _rows(rng, M)
        out = kv.ms_call(q, None, None, pos, slots)
        for t, s in enumerate(slots):
            assert_attn_close(out[t:t + 1], refs[s].attend_f32(q[t:t + 1], int(pos[t])), f"row {t}")


@pytest.mark.parametrize("merge_in_launch", [0, 1])
def test_rejected_rows_yield_zeros_and_touch_nothing(native, oracle, merge_in_launch):
    kv, refs, rng = _streams(native, oracle, False)
    with kv:
        kv.set_opt(7, merge_in_launch)                    # the last workgroup of a column merges the splits / the combiner launch does
        slots = np.array([1, 9, 3, -1, 2], np.int32)
        pos = np.array([17, 5, -4, 5, CTX], np.int32)     # only row 0 is valid
        q, k, v = _rows(rng, 5)
        before = kv.export_rows(2, 0, CTX)
        out = kv.ms_call(q, k, v, pos, slots)
        assert not np.any(out[1:].view(np.uint16) & 0x7fff)
        refs[1].append(k[0:1], v[0:1], 17)
        assert_attn_close(out[0:1], refs[1].attend_f32(q[0:1], 17), "valid row")
        after = kv.export_rows(2, 0, CTX)
        for a, b in zip(before, after):
            assert np.array_equal(a, b)
        with pytest.raises(native.YkaError):
            kv.ms_call(q, k, None, pos, slots)


# ---- the same passes over the reference's own 256-channel rows (handles opened with head_dim = 256) ----

def _streams256(native, oracle, paged, seed=5):
    rng = np.random.default_rng(seed)
    kv = native.KvCache(n_layers=len(LENS), head_dim=256, max_ctx=CTX, max_rows=64, paged=paged)
    if paged:
        for s in range(len(LENS)):
            kv.set_page_table(rng.permutation(CTX // 256).astype(np.int32), layer=s)
    refs = []
    for s, n in enumerate(LENS):
        ref = oracle.Cache(CTX, 24, 4, 256)
        if n:
            k = rng.standard_normal((n, 4, 256)).astype(np.float16)
            k[:, :, [5, 77, 130, 201]] *= 8
            v = rng.standard_normal((n, 4, 256)).astype(np.float16)
            for p in range(0, n, 64):
                kv.append_host(s, k[p:p + 64], v[p:p + 64], p)
            ref.append(k, v, 0)
        refs.append(ref)
    return kv, refs, rng


def _rows256(rng, M):
    return tuple(rng.standard_normal((M, h, 256)).astype(np.float16) for h in (24, 4, 4))


@pytest.mark.parametrize("paged", [False, True])
def test_one_row_per_stream_256(native, oracle, paged):
    kv, refs, rng = _streams256(native, oracle, paged)
    with kv:
        slots = np.array([2, 0, 4, 1, 3], np.int32)
        pos = np.array([LENS[s] for s in slots], np.int32)
        q, k, v = _rows256(rng, len(slots))
        out = kv.ms_call(q, k, v, pos, slots)
        for t, s in enumerate(slots):
            refs[s].append(k[t:t + 1], v[t:t + 1], int(pos[t]))
            assert_attn_close(out[t:t + 1], refs[s].attend_f32(q[t:t + 1], int(pos[t])), f"row {t} stream {s}")
            got = kv.export_rows(int(s), int(pos[t]), 1)
            assert np.array_equal(got[0], refs[s].kc[:, pos[t]:pos[t] + 1]) and np.array_equal(got[2], refs[s].vc[:, pos[t]:pos[t] + 1])
            assert np.array_equal(got[1].view(np.uint32), refs[s].ks[:, pos[t]:pos[t] + 1].view(np.uint32))
            assert np.array_equal(got[3].view(np.uint32), refs[s].vs[:, pos[t]:pos[t] + 1].view(np.uint32))


def test_rows_of_one_stream_and_bad_rows_256(native, oracle):
    kv, refs, rng = _streams256(native, oracle, False)
    with kv:
        # stream 0: its last token and two draft tokens (they see each other's keys); stream 2: one row; a row whose slot
        # does not exist and one whose position lies outside its container yield zeros and write nothing
        slots = np.array([0, 0, 0, 2, 9, 1], np.int32)
        pos = np.array([300, 301, 302, 900, 5, CTX], np.int32)
        q, k, v = _rows256(rng, 6)
        out = kv.ms_call(q, k, v, pos, slots)
        refs[0].append(k[0:3], v[0:3], 300)
        assert_attn_close(out[0:3], refs[0].attend_f32(q[0:3], 300), "stream 0 window")
        refs[2].append(k[3:4], v[3:4], 900)
        assert_attn_close(out[3:4], refs[2].attend_f32(q[3:4], 900), "stream 2")
        assert not out[4:6].view(np.uint16).any()
        # attend only, more rows than the reference's 16-row cap
        M = 20
        slots = np.array([s % 4 for s in range(M)], np.int32)
        pos = np.array([max(0, LENS[s] - 1 - t) for t, s in enumerate(slots)], np.int32)
        q = rng.standard_normal((M, 24, 256)).astype(np.float16)
        out = kv.ms_call(q, None, None, pos, slots)
        for t, s in enumerate(slots):
            if LENS[s] + (3 if s == 0 else 1 if s == 2 else 0) > pos[t]:
                assert_attn_close(out[t:t + 1], refs[s].attend_f32(q[t:t + 1], int(pos[t])), f"attend-only row {t}")


# The workgroups of a pass are shared out by the streams' lengths: one long stream beside many short ones, every number of
# rows a slice can have (1, 2, a full slice of 64, a second slice), rows that name nothing between them.  The reference is
# one-row passes over the same containers.
@pytest.mark.parametrize("M", [1, 2, 3, 33, 64, 65])
@pytest.mark.parametrize("dim", [128, 256])
def test_streams_of_very_different_lengths(native, dim, M):
    rng = np.random.default_rng(M + dim)
    ctx = 9216
    lens = [9000] + [int(x) for x in rng.integers(1, 200, M - 1)] if M % 2 else [int(x) for x in rng.integers(1, 700, M)]

    def rows(n, heads):
        return rng.standard_normal((n, heads, dim)).astype(np.float16)

    with native.KvCache(n_layers=M, head_dim=dim, max_ctx=ctx, max_rows=max(M, 1024)) as kv:
        for s, n in enumerate(lens):
            for p in range(0, n, 1024):
                kv.append_host(s, rows(min(1024, n - p), 4), rows(min(1024, n - p), 4), p)
        slots = rng.permutation(M).astype(np.int32)
        pos = np.array([lens[s] for s in slots], np.int32)
        bad = [t for t in range(M) if M > 3 and t % 11 == 5]
        pos[bad] = ctx
        q, k, v = rows(M, 24), rows(M, 4), rows(M, 4)
        kv.poison_workspace()
        out = kv.ms_call(q, k, v, pos, slots)
        good = [t for t in range(M) if t not in bad]
        stored = {t: kv.export_rows(int(slots[t]), int(pos[t]), 1) for t in good}
        for t in range(M):
            if t in bad:
                assert not (out[t].view(np.uint16) & 0x7fff).any()
                continue
            ref = kv.layer_call(int(slots[t]), q[t:t + 1], k[t:t + 1], v[t:t + 1], int(pos[t])).astype(np.float32)[0]
            # the same kernel arithmetic with another split count: fp16 partials and outputs, 2^-11 each, summed in fp32
            assert np.linalg.norm(out[t].astype(np.float32) - ref) <= 1e-3 * np.linalg.norm(ref), f"row {t}: stream of {pos[t]} tokens"
        for t in good:                                    # the rows the pass stored are the rows one-row calls have stored since
            assert stored[t][0].any()
            for a, b in zip(stored[t], kv.export_rows(int(slots[t]), int(pos[t]), 1)):
                assert np.array_equal(a.view(np.uint8), b.view(np.uint8)), f"row {t}"


# 128-channel rows, numbers of streams whose whole splits leave a round of workgroups unfilled: long streams (48 tiles for each
# workgroup of one round) use the second number of workgroups, short ones the first; both sides of that line, for 26 rows
# (104 and 182 workgroups a kv head), 33 (99, 231), 48 (96, 192) and 51 (102, 255)
@pytest.mark.parametrize("M,per_round", [(26, 104), (33, 99), (48, 96), (51, 102)])
@pytest.mark.parametrize("more", [0, 1])
def test_the_line_between_short_and_long_streams(native, M, per_round, more):
    rng = np.random.default_rng(M)
    total = 48 * per_round - 1 + more                     # together 48 tiles a workgroup, or one tile less
    tiles = np.full(M, total // M) + (np.arange(M) < total % M)
    lens = tiles * 32 - rng.integers(1, 33, M)            # a row at position p has (p + 32) / 32 tiles
    half = lambda n, heads: rng.standard_normal((n, heads, 128)).astype(np.float16)    # noqa: E731
    pool_k, pool_v = half(6400, 4), half(6400, 4)
    with native.KvCache(n_layers=M, max_ctx=8192, max_rows=6400) as kv:
        for s in range(M):
            n = int(lens[s])
            kv.append_host(s, np.roll(pool_k, s, axis=0)[:n], np.roll(pool_v, 7 * s, axis=0)[:n], 0)
        slots = rng.permutation(M).astype(np.int32)
        pos = lens[slots].astype(np.int32)
        q, k, v = half(M, 24), half(M, 4), half(M, 4)
        kv.poison_workspace()
        out = kv.ms_call(q, k, v, pos, slots).astype(np.float32)
        for t in range(M):
            ref = kv.layer_call(int(slots[t]), q[t:t + 1], k[t:t + 1], v[t:t + 1], int(pos[t])).astype(np.float32)[0]
            assert np.linalg.norm(out[t] - ref) <= 1e-3 * np.linalg.norm(ref), f"row {t}: stream of {pos[t]} tokens"    # as above


# A pass that stores its rows inside the attention launch, with many consecutive rows of one stream: they lie in several tiles, on
# both sides of a split boundary and of a 256-token page, and every workgroup stores those it reads.  Short streams and rows
# that name nothing between them, the rows in any order.  Stored bytes and outputs against the oracle.
@pytest.mark.parametrize("dim", [128, 256])
@pytest.mark.parametrize("paged", [False, True])
@pytest.mark.parametrize("first,n", [(236, 58), (200, 40), (505, 56), (0, 60)])
def test_many_rows_of_one_stream_in_one_pass(native, oracle, dim, paged, first, n):
    rng = np.random.default_rng(first + n + dim)
    half = lambda m, heads: rng.standard_normal((m, heads, dim)).astype(np.float16)    # noqa: E731
    lens = [first, 3, 0, 65]
    with native.KvCache(n_layers=4, head_dim=dim, max_ctx=CTX, max_rows=512, paged=paged) as kv:
        refs = []
        for s, m in enumerate(lens):
            if paged:
                kv.set_page_table(rng.permutation(CTX // 256).astype(np.int32), layer=s)
            refs.append(oracle.Cache(CTX, 24, 4, dim))
            if m:
                k, v = half(m, 4), half(m, 4)
                for p in range(0, m, 512):
                    kv.append_host(s, k[p:p + 512], v[p:p + 512], p)
                refs[s].append(k, v, 0)
        slots = np.array([0] * n + [1, 2, 3, 7], np.int32)
        pos = np.array(list(range(first, first + n)) + [3, 0, 65, 9], np.int32)
        order = rng.permutation(n + 4)
        slots, pos = slots[order], pos[order]
        q, k, v = half(n + 4, 24), half(n + 4, 4), half(n + 4, 4)
        kv.poison_workspace()
        out = kv.ms_call(q, k, v, pos, slots)
        for t in np.argsort(pos, kind="stable"):
            if slots[t] < 4:
                refs[slots[t]].append(k[t:t + 1], v[t:t + 1], int(pos[t]))
        for t, s in enumerate(slots):
            if s == 7:
                assert not (out[t].view(np.uint16) & 0x7fff).any()
            else:                                         # first keys of a stream: two fp16 spacings on values in [2, 4] (tolerances.py)
                assert_attn_close(out[t:t + 1], refs[s].attend_f32(q[t:t + 1], int(pos[t]), want_f32=True)[1], f"row {t} stream {s}", two_spacings=pos[t] < 64)
        for s in range(4):
            held = lens[s] + (n if s == 0 else 1)
            for a, b in zip(kv.export_rows(s, 0, CTX), (refs[s].kc, refs[s].ks, refs[s].vc, refs[s].vs)):
                a, b = a[:, :held].copy().view(np.uint8), b[:, :held].copy().view(np.uint8)
                assert np.array_equal(a, b), f"rows of stream {s}"
