"""What this library is timed on: layer calls of the attention path over a quantized KV cache, as an engine issues them.

A pass is one step of a model: one layer call per attention layer (16 of them in the 64-layer model the shapes come from;
fewer where one layer is large), every layer with its own container, projections and outputs.  24 query heads on 4 KV
heads throughout.  What varies:

  format   flat128   int4 codes, one fp16 scale per 32 channels, head_dim 128
           flat256   int4 codes, one fp32 scale per row, head_dim 256
           kv5, kv4  trellis-coded rows of 5 / 4 bits an element, head_dim 256
  call     layer     append_attend: new K / V rows are quantized into the cache, then attention over it
           post      attn_post, then attend: norm, rotary and rotation of fp32 projections in front of the cache
           streams   append_attend_ms: one row for each of `rows` streams of different lengths
  rows     1 decode, 2 .. 64 a window of draft tokens to verify, more: a chunk of a prompt
  ctx      tokens in the cache before the call (streams: of the longest; the others spread down to a sixteenth of it)
  capacity tokens the containers hold; an engine opens them for the longest context it will serve
  bf16     type of the 16-bit rows at the boundary: bf16 (option key 11) or fp16
  paged    containers in shuffled 256-token pages
  tree     the window is a tree of drafts: a depth table instead of consecutive positions
  graph    the layer calls are replayed from a captured graph (small passes) or issued one by one

Ranges: ctx 0 .. 262,144, capacity up to 16 times the context, 1 .. 2,048 rows, 2 .. 32 streams, every combination of
the rest that the library takes.
"""
import math

import torch

from yasakani_amd import kvqp, native

HEADS, KV_HEADS = 24, 4
LAYERS = 16
FILL = 2048                      # rows per call while a cache is filled
BITS = {"flat128": 0, "flat256": 0, "kv5": 5, "kv4": 4}
MAX_BYTES = 6.5e8                # what a drawn case may read at most: the largest listed one (decode-262k)
MAX_FLOPS = 6.6e12               # and compute at most: prefill-2048-deep


def _case(name=None, format="flat128", call="layer", rows=1, ctx=4096, capacity=0, layers=LAYERS, bf16=False, paged=False, tree=False, graph=True):
    room = -(-max(capacity, ctx + rows) // 256) * 256
    c = dict(format=format, call=call, rows=rows, ctx=ctx, capacity=room, layers=layers, bf16=bf16, paged=paged, tree=tree, graph=graph)
    return c if name is None else dict(name=name, **c)


def listed():
    return [
        # a chat's first turns: one token on a short context, in containers opened for a long one; launches and latency count
        _case("decode-1k", ctx=1003, capacity=32768, bf16=True),
        # one token on a long context: the KV stream
        _case("decode-32k", ctx=32741, capacity=32768),
        # one token on the longest context, paged
        _case("decode-262k", ctx=262100, layers=4, paged=True),
        # a server's step: one token for each of 16 conversations of different lengths
        _case("streams-16", call="streams", rows=16, ctx=32000, capacity=32768, layers=1, bf16=True, graph=False),
        # a small draft tree is verified
        _case("verify-8-tree", rows=8, ctx=12037, capacity=32768, bf16=True, tree=True),
        # the widest window of drafts on a long context
        _case("verify-64", rows=64, ctx=32768, graph=False),
        # a prompt read into an empty cache
        _case("prefill-1500-first", rows=1500, ctx=0, capacity=8192, bf16=True, graph=False),
        # a chunk of a long prompt far into it
        _case("prefill-2048-deep", rows=2048, ctx=131072, layers=2, graph=False),
        # the 256-channel rows: one token, from the projections on
        _case("r256-decode", format="flat256", call="post", ctx=20011, capacity=32768),
        # and a window of drafts
        _case("r256-verify-24", format="flat256", rows=24, ctx=9001, capacity=16384, bf16=True, graph=False),
        # trellis-coded rows: one token, and a window
        _case("kv5-decode", format="kv5", ctx=16001, capacity=32768),
        _case("kv5-verify-16", format="kv5", rows=16, ctx=16384, capacity=16640, graph=False),
    ]


def _log_between(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    while True:
        format = rng.choice(["flat128"] * 6 + ["flat256"] * 2 + ["kv5", "kv5", "kv4"])
        kind = rng.choice(["decode", "decode", "verify", "verify", "verify", "streams", "prefill"])
        ctx = _log_between(rng, 500, 262000)
        capacity = int(ctx * rng.choice([1, 1.3, 2, 4, 16]))
        bf16, paged = rng.random() < 0.5, format[:4] == "flat" and rng.random() < 0.25
        layers, call, tree, graph = LAYERS, "layer", False, rng.random() < 0.7
        if kind == "decode":
            rows = rng.choice([1, 1, 1, 2])
            call = rng.choice(["layer", "layer", "post"])
        elif kind == "verify":
            rows, tree = _log_between(rng, 3, 64), rng.random() < 0.3
        elif kind == "streams":
            rows, call, layers, graph = _log_between(rng, 2, 32), "streams", 1, False
            ctx, capacity = min(ctx, 65536), min(capacity, 65536)
        else:
            rows, graph, ctx = _log_between(rng, 65, 2048), False, rng.choice([0, ctx])
        if BITS[format] and ctx * layers > 300000:
            layers = max(1, 300000 // ctx)           # the trellis encoder fills a cache at about 2 us a token
        while layers > 1 and layers * max(capacity, ctx + rows) > 1100000:
            layers //= 2
        case = _case(None, format, call, rows, ctx, min(capacity, 262144), layers, bf16, paged, tree, graph)
        w = work(case)
        if w["bytes"] <= MAX_BYTES and w["flops"] <= MAX_FLOPS:
            return case


def _dim(case):
    return 128 if case["format"] == "flat128" else 256


def _token_bytes(case):
    """Bytes of one token's K and V rows in the cache of one layer."""
    if case["format"] == "flat128":
        return KV_HEADS * 2 * (64 + 2 * 4)
    return KV_HEADS * 2 * (32 * (BITS[case["format"]] or 4) + 4)


def _lengths(case):
    """Keys a stream holds before the pass: from ctx down to a sixteenth of it, evenly on a logarithmic scale."""
    m = case["rows"]
    return [max(1, int(case["ctx"] * 16.0 ** (-t / max(1, m - 1)))) for t in range(m)]


def work(case):
    m, d, layers = case["rows"], _dim(case), case["layers"]
    cached = sum(_lengths(case)) if case["call"] == "streams" else case["ctx"]
    keys = cached + m if case["call"] == "streams" else sum(case["ctx"] + t + 1 for t in range(m))
    width = 4 if case["call"] == "post" else 2                      # bytes of a projected value
    rows = m * d * (width * (HEADS + 2 * KV_HEADS) + 2 * HEADS) + m * _token_bytes(case)
    return {"bytes": layers * (cached * _token_bytes(case) + rows), "flops": 4.0 * layers * HEADS * d * keys}


def tolerance(case):
    # 16-bit outputs of fp32 sums over probabilities and values that were rounded to fp16.  The same path with its sums in
    # another order (other split counts, another kernel): fp16 rows differ by 4.0e-4 .. 5.0e-4, single values by up to
    # 1.1e-2 of the output's rms (2,048 rows at 131,072 tokens); bf16 rows by 1.0e-3 .. 1.3e-3 and 1.0e-2.  Four times that.
    return {"rel": 5e-3, "max": 0.04} if case["bf16"] else {"rel": 1.9e-3, "max": 0.04}


def _rows(gen, n, case, dtype, outliers=None):
    """n K or V rows: normal values; four channels of K are eight times as large, as key channels are in practice."""
    x = torch.randn(n, KV_HEADS, _dim(case), generator=gen, device="cuda")
    if outliers is not None:
        x[:, :, outliers] *= 8.0
    return x.to(dtype)


class _State:
    """What a program holds between its calls: the cache, the buffers of one step and, if it replays them, the graph."""

    def __init__(self, case, seed):
        self.case = case
        gen = torch.Generator(device="cuda").manual_seed(seed)
        m, d, streams = case["rows"], _dim(case), case["call"] == "streams"
        containers = m if streams else case["layers"]
        self.kv = kv = native.KvCache(n_layers=containers, n_heads=HEADS, n_kv_heads=KV_HEADS, head_dim=d, max_ctx=case["capacity"],
                                      max_rows=max(m, FILL), paged=case["paged"])
        if BITS[case["format"]]:
            kv.set_profile(kvqp.synthetic(layers=containers, kk=BITS[case["format"]], seed=7))
        if case["bf16"]:
            kv.set_opt(11, 1)
        if case["paged"]:
            kv.set_page_table(torch.randperm(case["capacity"] // 256, generator=gen, device="cuda").cpu().numpy())
        dtype = torch.bfloat16 if case["bf16"] else torch.float16
        outliers = torch.randperm(d, generator=gen, device="cuda")[:4]
        shape = (m,) if streams else (case["layers"], m)
        if case["call"] == "post":
            self._post_parameters(gen, d)
            kv.set_opt(4, 1)                              # outputs leave the rotated space
        for layer in range(containers):
            self._fill(gen, layer, _lengths(case)[layer] if streams else case["ctx"], dtype, outliers)
        new = torch.float32 if case["call"] == "post" else dtype
        self.q = torch.randn(*shape, HEADS, d, generator=gen, device="cuda").to(new)
        n = m if streams else case["layers"] * m
        self.k = _rows(gen, n, case, new, outliers).view(*shape, KV_HEADS, d)
        self.v = _rows(gen, n, case, new).view(*shape, KV_HEADS, d)
        self.q16 = torch.empty(*shape, HEADS, d, dtype=dtype, device="cuda") if case["call"] == "post" else None
        self.out = torch.zeros(*shape, HEADS, d, dtype=dtype, device="cuda")
        self.pos = torch.tensor([case["ctx"]], dtype=torch.int32, device="cuda")
        self.depth = self._tree(gen, m) if case["tree"] else None
        if streams:
            self.row_slot = torch.randperm(m, generator=gen, device="cuda").to(torch.int32)
            self.row_pos = torch.tensor(_lengths(case), dtype=torch.int32, device="cuda")[self.row_slot.long()].contiguous()
        self.graph = None
        if case["graph"]:
            torch.cuda.synchronize()
            self.graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(self.graph):
                self.step()
        torch.cuda.synchronize()

    def _post_parameters(self, gen, d):
        rope_dims = d // 4
        angle = torch.arange(self.case["capacity"], device="cuda", dtype=torch.float64)[:, None] \
            * (1e6 ** (-2.0 * torch.arange(rope_dims // 2, device="cuda", dtype=torch.float64) / rope_dims))[None, :]
        self.rope = torch.stack([torch.cos(angle), torch.sin(angle)], dim=-1).float().contiguous()
        self.norm_q, self.norm_k = ((torch.randn(d, generator=gen, device="cuda") * 0.1).half() for _ in range(2))
        self.post = native.PostParams(self.norm_q.data_ptr(), self.norm_k.data_ptr(), 1e-6, self.rope.data_ptr(), rope_dims, self.case["capacity"], 1)

    @staticmethod
    def _tree(gen, m):
        """Depth of every draft in a tree whose node t hangs on one of the nodes before it."""
        u, depth = torch.rand(m, generator=gen, device="cuda").tolist(), [0]
        for t in range(1, m):
            depth.append(depth[max(0, t - 1 - int(3 * u[t]))] + 1)
        return torch.tensor(depth, dtype=torch.uint8, device="cuda")

    def _fill(self, gen, layer, n, dtype, outliers):
        stream = torch.cuda.current_stream().cuda_stream
        if self.case["call"] == "post":
            q = torch.randn(min(n, FILL), HEADS, _dim(self.case), generator=gen, device="cuda")
            q16 = torch.empty(q.shape, dtype=torch.float16, device="cuda")
        for at in range(0, n, FILL):
            rows = min(FILL, n - at)
            pos = torch.tensor([at], dtype=torch.int32, device="cuda")
            if self.case["call"] == "post":
                k, v = _rows(gen, rows, self.case, torch.float32, outliers), _rows(gen, rows, self.case, torch.float32)
                self.kv.attn_post(layer, q.data_ptr(), k.data_ptr(), v.data_ptr(), rows, pos.data_ptr(), self.post, q16.data_ptr(), stream)
            else:
                k, v = _rows(gen, rows, self.case, dtype, outliers), _rows(gen, rows, self.case, dtype)
                self.kv.append(layer, k.data_ptr(), v.data_ptr(), rows, pos.data_ptr(), stream)

    def step(self):
        """One model step: the layer calls of every layer, in order, on the current stream."""
        m, kv, call, stream = self.case["rows"], self.kv, self.case["call"], torch.cuda.current_stream().cuda_stream
        if call == "streams":
            kv.append_attend_ms(self.q.data_ptr(), self.k.data_ptr(), self.v.data_ptr(), m, self.row_pos.data_ptr(), self.row_slot.data_ptr(),
                                self.out.data_ptr(), stream)
            return
        pos, depth = self.pos.data_ptr(), None if self.depth is None else self.depth.data_ptr()
        for layer in range(self.case["layers"]):
            q, k, v, out = (x[layer].data_ptr() for x in (self.q, self.k, self.v, self.out))
            if call == "post":
                q16 = self.q16[layer].data_ptr()
                kv.attn_post(layer, q, k, v, m, pos, self.post, q16, stream)
                kv.attend(layer, q16, m, pos, out, depth, stream)
            else:
                kv.append_attend(layer, q, k, v, m, pos, out, depth, stream)


def prepare(case, seed):
    return _State(case, seed)


def run(state):
    if state.graph is not None:
        state.graph.replay()
    else:
        state.step()
    return state.out if state.q16 is None else [state.out, state.q16]
