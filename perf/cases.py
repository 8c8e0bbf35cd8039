"""The work that users of this library have it do, as measurable cases.

A case is a dict of plain values; `prepare` builds what a program holds before the call (weights in GGUF block
layout, inputs, scratch objects), `run` is one pass through the public C ABI.  Five kinds:

  stack   one decode step through a stack of MoE layers in one call (wd_moe_stack_f32), the routed ids chosen by the
          router or replayed from a trace
  layers  the MoE layers of one decode step called one by one, as a decoder with attention between them does
          (wd_moe_layer_f32, or wd_moe_layer_hc_f32 where the residual is a set of hyper-connection streams)
  tokens  a speculative-verify batch of 2..8 tokens through every layer (wd_moe_layer_tokens_f32)
  cached  decode with the routed experts in pinned host memory behind an LRU pool in HBM (wd_moe_stack_cached_f32)
  dense   the quantised matrix-vector products of the dense blocks and of the output head
          (activation quantisers, wd_gemv_*)
"""
import ctypes as C
import math

import numpy as np
import torch

from warpdecode_amd import capi, synth

TYPES = {"q4_0": synth.Q4_0, "q8_0": synth.Q8_0, "iq4_nl": synth.IQ4_NL, "iq3_s": synth.IQ3_S, "iq2_s": synth.IQ2_S,
         "q6_k": synth.Q6_K}
K_TYPES = ("iq3_s", "iq2_s", "q6_k")   # blocks of 256 weights, activations in Q8_K; the others take Q8_0 activations
# fp16 block scales |N(0, sigma)| such that the weights are of the order of 0.01..0.02
SIGMA = {"q4_0": 0.02 / 8, "q8_0": 0.02 / 127, "iq4_nl": 0.02 / 127, "iq3_s": 2e-4, "iq2_s": 5e-4, "q6_k": 0.02 / 2048}
RESIDUAL_SCALE = 0.05   # keeps the input of every layer of a stack near unit RMS
# share of the common direction in the tokens of one batch, and in consecutive tokens: about half of the selected
# experts are the same
TOKEN_MIX = 0.55


def _moe(name, kind, hidden, ffn, experts, top_k, gate, down, shared, layers, **more):
    c = dict(name=name, kind=kind, hidden=hidden, ffn=ffn, experts=experts, top_k=top_k, gate=gate, down=down,
             shared=shared, layers=layers)
    c.update(more)
    return c


def listed():
    return [
        # one decode step of the 48-layer, 512-expert model this library is built around; the router chooses
        _moe("stack_routed", "stack", 2048, 512, 512, 10, "iq3_s", "q8_0", True, 48, trace=False),
        # the same step with a recorded routing trace (Zipf-distributed ids): the headline benchmark
        _moe("stack_trace", "stack", 2048, 512, 512, 10, "iq3_s", "q8_0", True, 48, trace=True),
        # a small mixture without shared expert, everything in Q8_0
        _moe("stack_q8", "stack", 2048, 512, 64, 8, "q8_0", "q8_0", False, 48, trace=False),
        # the layer at the shapes and types of the target model, called between attention blocks, combine included
        _moe("layers_model", "layers", 2560, 640, 512, 10, "iq2_s", "iq4_nl", True, 16, hc=4),
        # wide experts, 128 of them, no shared expert: the other common proportions of a mixture
        _moe("layers_wide", "layers", 4096, 1536, 128, 8, "iq3_s", "q8_0", False, 8, hc=0),
        # a single small layer: the latency of one call
        _moe("layer_small", "layers", 1024, 256, 64, 6, "iq3_s", "q8_0", True, 1, hc=0),
        # speculative verify: one committed and three draft tokens through the 512-expert layer
        _moe("tokens_4", "tokens", 2048, 512, 512, 10, "iq3_s", "q8_0", True, 8, tokens=4),
        # experts that do not fit in HBM: host memory behind a pool of half their number, the router decides per layer
        _moe("cached_routed", "cached", 2048, 512, 128, 10, "iq3_s", "q8_0", True, 8, trace=False, pool=0.5),
        # a dense 1B model in Q4_0: every projection of 16 blocks and the 128256-row head
        dict(name="dense_q4", kind="dense", type="q4_0", hidden=2048, kv=512, inner=8192, vocab=128256, blocks=16),
        # the Q8_0 projections around the MoE layers of the target model (no dense head)
        dict(name="dense_q8", kind="dense", type="q8_0", hidden=2560, kv=512, inner=2560, vocab=0, blocks=24),
        # the Q6_K output head alone
        dict(name="head_q6k", kind="dense", type="q6_k", hidden=2048, kv=0, inner=0, vocab=151936, blocks=0),
        # one small projection alone: the latency of quantise + matrix-vector product, an odd number of rows
        dict(name="gemv_small", kind="dense", type="q8_0", hidden=2048, kv=0, inner=0, vocab=1001, blocks=0),
    ]


def _log(rng, lo, hi, step=1):
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(step, int(round(v / step)) * step)


def draw(rng):
    c = _draw(rng)
    # fewer layers or blocks where a pass would read more than the largest listed one
    n = "blocks" if c["kind"] == "dense" else "layers"
    while work(c)["bytes"] > 1.2e9 and c[n] > 1:
        c[n] -= 1
    return c


def _draw(rng):
    kind = rng.choice(["stack", "stack", "layers", "layers", "layers", "tokens", "tokens", "cached", "dense", "dense", "dense"])
    if kind == "dense":
        t = rng.choice(sorted(TYPES))
        # any row length of whole blocks; the K types' blocks are 256 wide
        step = 256 if t in K_TYPES else 32
        if rng.random() < 0.5:   # a single matrix: a head, or one projection
            c = dict(kind=kind, type=t, hidden=_log(rng, 512, 16384, step), kv=0, inner=0, vocab=_log(rng, 64, 160000), blocks=0)
            c["vocab"] = max(64, min(c["vocab"], (1 << 29) // c["hidden"]))
            return c
        h = _log(rng, 768, 5120, step)
        return dict(kind=kind, type=t, hidden=h, kv=_log(rng, 128, 1024, 64), inner=_log(rng, 512, 12288, step),
                    vocab=rng.choice([0, _log(rng, 16000, 100000)]), blocks=_log(rng, 1, 16))
    gate = rng.choice(["iq3_s", "iq3_s", "iq2_s", "iq2_s", "q8_0", "iq4_nl"])
    c = dict(kind=kind, hidden=_log(rng, 1024, 4096, 256), ffn=_log(rng, 128, 1536, 32), experts=_log(rng, 16, 512, 8),
             top_k=rng.randint(2, 10), gate=gate, down=rng.choice(["q8_0", "iq4_nl"]), shared=rng.random() < 0.5)
    if kind == "stack":
        c.update(layers=_log(rng, 2, 48), trace=rng.random() < 0.3)
    elif kind == "layers":
        c.update(layers=_log(rng, 1, 24), hc=rng.choice([0, 0, 4]))
    elif kind == "tokens":
        c.update(layers=_log(rng, 1, 8), tokens=rng.randint(2, 8))
    else:
        c.update(layers=_log(rng, 2, 8), trace=rng.random() < 0.5, pool=0.5)
        c["experts"] = max(32, min(c["experts"], 128))
    most = 1.5e9 if kind == "cached" else 6e9   # bytes of routed weights
    c["layers"] = max(1, min(c["layers"], int(most / (c["experts"] * _expert_bytes(c)))))
    if kind == "cached":
        c["experts"] = max(32, min(c["experts"], int(most / (c["layers"] * _expert_bytes(c))) // 8 * 8))
    return c


# ---- inputs ---------------------------------------------------------------------------------------------------
def _expert_bytes(c):
    return 2 * c["ffn"] * _row(c["gate"], c["hidden"]) + c["hidden"] * _row(c["down"], c["ffn"])


def _row(t, cols):
    return synth.row_bytes(TYPES[t], cols)


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _matrix(g, t, rows, cols):
    """Random blocks of type `t` on the GPU: uniform codes, scales |N(0, sigma)|."""
    size, block = rows * _row(t, cols), synth.BLOCK_BYTES[TYPES[t]]
    w = torch.empty((size + 3) // 4, dtype=torch.int32, device="cuda").random_(-2 ** 31, 2 ** 31 - 1, generator=g).view(torch.uint8)[:size]
    if t == "q8_0":
        w.view(torch.int8).clamp_(min=-127)   # the quantiser's range
    blocks = w.view(-1, block)
    if t == "q6_k":
        blocks[:, 192:208].bitwise_and_(0x3f)  # sub-block scales
    d = torch.randn(blocks.shape[0], device="cuda", generator=g).abs_().mul_(SIGMA[t]).half()
    at = block - 2 if t == "q6_k" else 0
    blocks[:, at:at + 2] = d.view(torch.uint8).view(-1, 2)
    return w


def _normed(g, *shape):
    x = torch.randn(*shape, device="cuda", generator=g)
    return x / x.square().mean(-1, keepdim=True).sqrt()


def _correlated(g, n, hidden):
    """n unit-RMS inputs around a common direction."""
    x = TOKEN_MIX * torch.randn(hidden, device="cuda", generator=g) + (1 - TOKEN_MIX) * torch.randn(n, hidden, device="cuda", generator=g)
    return x / x.square().mean(-1, keepdim=True).sqrt()


def _p(t):
    return C.c_void_p(t.data_ptr())


def _stream():
    return C.c_void_p(torch.cuda.current_stream().cuda_stream)


class _State:
    """Inputs, weights and the library objects of one case; the objects go with it."""

    def __init__(self, case):
        capi.call("wd_init", 0)
        self.case, self.keep, self.owned = case, [], []

    def scratch(self, c):
        h = C.c_void_p()
        capi.call("wd_moe_scratch_create", C.byref(h), c["hidden"], c["ffn"], c["experts"], c["top_k"])
        self.owned.append(("wd_moe_scratch_destroy", h))
        return h

    def pinned(self, tensor):
        h = C.c_void_p()
        capi.call("wd_malloc_host", C.byref(h), tensor.numel())
        self.owned.append(("wd_free_host", h))
        capi.call("wd_memcpy_d2h", h, _p(tensor), tensor.numel(), None)
        return h

    def __del__(self):
        if self.owned:
            torch.cuda.synchronize()
        for name, h in reversed(self.owned):
            getattr(capi.load(), name)(h)
        self.owned = []


def _layers(s, c, g, on_host=False):
    """The stack's descriptors; with `on_host` the routed tensors go to pinned host memory (returned per layer)."""
    H, F, E = c["hidden"], c["ffn"], c["experts"]
    arr, host = (capi.MoeLayer * c["layers"])(), []
    for d in arr:
        t = dict(router=torch.randn(E, H, device="cuda", generator=g) / math.sqrt(H), gate=_matrix(g, c["gate"], E * F, H),
                 up=_matrix(g, c["gate"], E * F, H), down=_matrix(g, c["down"], E * H, F))
        if c["shared"]:
            t.update(shared_gate_inp=torch.randn(H, device="cuda", generator=g) * 0.02, shared_gate=_matrix(g, "q8_0", F, H),
                     shared_up=_matrix(g, "q8_0", F, H), shared_down=_matrix(g, "q8_0", H, F))
        if on_host:
            host.append([s.pinned(t.pop(n)) for n in ("gate", "up", "down")])
        s.keep.append(t)
        d.hidden, d.expert_ffn, d.n_experts, d.top_k, d.expert_scale = H, F, E, c["top_k"], 1.0
        d.gate_type = d.up_type = TYPES[c["gate"]]
        d.down_type = TYPES[c["down"]]
        for name, tensor in t.items():
            setattr(d, name, tensor.data_ptr())
        d.gate_stride = d.up_stride = F * _row(c["gate"], H)
        d.down_stride = H * _row(c["down"], F)
    return arr, host


def _traces(seed, c, tokens):
    """Zipf(1.1)-distributed ids over a permutation of each layer's experts."""
    rng = np.random.default_rng(seed)
    perms = [rng.permutation(c["experts"]) for _ in range(c["layers"])]
    return np.stack([np.stack([synth.zipf_ids(rng, c["experts"], c["top_k"], 1.1, p) for p in perms]) for _ in range(tokens)])


def prepare(case, seed):
    c = case
    s, g = _State(c), _gen(seed)
    if c["kind"] == "dense":
        return _prepare_dense(s, c, g)
    H, NL = c["hidden"], c["layers"]
    s.layers, host = _layers(s, c, g, on_host=c["kind"] == "cached")
    if c["kind"] in ("stack", "cached"):
        s.scratch_h = s.scratch(c)
        s.x, s.out = torch.empty(H, device="cuda"), torch.empty(H, device="cuda")
        # a cached decode runs through a text: 32 consecutive tokens; a stack takes one
        n = 32 if c["kind"] == "cached" else 1
        s.xs = _correlated(g, n, H) if n > 1 else _normed(g, n, H)
        s.token = 0
        s.trace_h = s.trace_d = None
        if c["trace"]:
            s.trace_h = np.ascontiguousarray(_traces(seed, c, n), np.int32)
            s.trace_d = torch.from_numpy(s.trace_h).cuda()
    if c["kind"] == "cached":
        gate, down = c["ffn"] * _row(c["gate"], H), H * _row(c["down"], c["ffn"])
        slots = max(int(c["pool"] * c["experts"] * NL), 2 * c["top_k"])
        s.cache = C.c_void_p()
        capi.call("wd_expert_cache_create", C.byref(s.cache), slots * (2 * gate + down), gate, gate, down, NL, c["experts"], 0)
        s.owned.append(("wd_expert_cache_destroy", s.cache))
        for l, h in enumerate(host):
            capi.call("wd_expert_cache_register_layer", s.cache, l, *h)
    elif c["kind"] == "layers":
        s.scratch_h = s.scratch(c)
        s.x, s.out = _normed(g, NL, H), torch.empty(NL, H, device="cuda")
        if c["hc"]:
            s.residual0 = torch.randn(c["hc"], H, device="cuda", generator=g)
            s.residual = torch.empty_like(s.residual0)
            s.inject = torch.randn(NL, c["hc"], device="cuda", generator=g)
    elif c["kind"] == "tokens":
        s.scratches = (C.c_void_p * c["tokens"])(*[s.scratch(c).value for _ in range(c["tokens"])])
        s.x = torch.stack([_correlated(g, c["tokens"], H) for _ in range(NL)])
        s.out = torch.empty_like(s.x)
    return s


def _prepare_dense(s, c, g):
    """`blocks` dense blocks (query, key, value, output, gate, up, down) and a head of `vocab` rows, each where its size
    is not zero.  The inputs of a block's projections (what norm and attention hand over) are given."""
    H, I, KV, t = c["hidden"], c["inner"], c["kv"], c["type"]
    s.blocks = []
    for _ in range(c["blocks"]):
        s.blocks.append({n: (_matrix(g, t, r, k), r, k) for n, r, k in
                         (("q", H, H), ("k", KV, H), ("v", KV, H), ("o", H, H), ("gate", I, H), ("up", I, H), ("down", H, I))})
    s.head = (_matrix(g, t, c["vocab"], H), c["vocab"], H) if c["vocab"] else None
    s.inputs = _normed(g, c["blocks"], 3, H)      # of q/k/v, of o, of gate/up
    s.final = _normed(g, H)
    s.qkv = torch.empty(c["blocks"], H + 2 * KV, device="cuda")
    s.attn = torch.empty(c["blocks"], H, device="cuda")
    s.gate_up = torch.empty(c["blocks"], 2, I, device="cuda")
    s.act = torch.empty(I, device="cuda")
    s.mlp = torch.empty(c["blocks"], H, device="cuda")
    s.logits = torch.empty(c["vocab"], device="cuda")
    n = max(H, I)
    s.qs = torch.empty(n, dtype=torch.int8, device="cuda")
    s.scales = torch.empty(n // 32 * 2, dtype=torch.int16, device="cuda")     # f16 per 32 values, or f32 per 256
    s.bsums = torch.empty(max(n // 16, 1), dtype=torch.int16, device="cuda")
    return s


# ---- one pass ---------------------------------------------------------------------------------------------------
def run(s):
    c = s.case
    return {"stack": _run_stack, "cached": _run_cached, "layers": _run_layers, "tokens": _run_tokens, "dense": _run_dense}[c["kind"]](s, c)


def _run_stack(s, c):
    s.x.copy_(s.xs[0])      # the token's input comes in; the call updates it in place
    capi.call("wd_moe_stack_f32", s.layers, c["layers"], _p(s.x), _p(s.out), s.scratch_h,
              _p(s.trace_d) if c["trace"] else None, RESIDUAL_SCALE, 0, _stream())
    return {"x": s.x, "out": s.out}


def _run_cached(s, c):
    i = s.token % len(s.xs)
    s.token += 1
    s.x.copy_(s.xs[i])
    trace = (s.trace_h[i].ctypes.data_as(C.c_void_p), _p(s.trace_d[i])) if c["trace"] else (None, None)
    capi.call("wd_moe_stack_cached_f32", s.layers, c["layers"], s.cache, _p(s.x), _p(s.out), s.scratch_h, *trace, RESIDUAL_SCALE, 0, _stream())
    return {"x": s.x, "out": s.out}


def _run_layers(s, c):
    st, x, out, step = _stream(), s.x.data_ptr(), s.out.data_ptr(), 4 * c["hidden"]
    if not c["hc"]:
        for l in range(c["layers"]):
            capi.call("wd_moe_layer_f32", C.byref(s.layers[l]), x + l * step, out + l * step, s.scratch_h, 0, st)
        return {"out": s.out}
    s.residual.copy_(s.residual0)
    res, inject = s.residual.data_ptr(), s.inject.data_ptr()
    for l in range(c["layers"]):
        capi.call("wd_moe_layer_hc_f32", C.byref(s.layers[l]), x + l * step, out + l * step, res, inject + l * 4 * c["hc"], c["hc"], 0,
                  s.scratch_h, 0, st)
    return {"out": s.out, "residual": s.residual}


def _run_tokens(s, c):
    st, x, out, step = _stream(), s.x.data_ptr(), s.out.data_ptr(), 4 * c["hidden"] * c["tokens"]
    for l in range(c["layers"]):
        capi.call("wd_moe_layer_tokens_f32", C.byref(s.layers[l]), x + l * step, out + l * step, c["tokens"], s.scratches, 0, st)
    return {"out": s.out}


def _quantise(s, t, x, n, st):
    if t in K_TYPES:
        capi.call("wd_q8_k_quantize_f32", x, n, _p(s.qs), _p(s.scales), _p(s.bsums), st)
    else:
        capi.call("wd_q8_0_quantize_f32", x, n, _p(s.qs), _p(s.scales), st)


def _products(s, t, mats, outs, st):
    """Matrices of one row length on the quantised activation."""
    cols = mats[0][2]
    if t in ("q8_0", "q4_0") and len(mats) > 1:
        items = (capi.GemvItem * len(mats))(*[(w.data_ptr(), rows, s.qs.data_ptr(), s.scales.data_ptr(), o) for (w, rows, _), o in zip(mats, outs)])
        capi.call("wd_gemv_q8_0_batch_f32", TYPES[t], items, len(mats), cols, st)
        return
    for (w, rows, _), o in zip(mats, outs):
        if t == "q6_k":
            capi.call("wd_gemv_q6_k_q8_k_f32", _p(w), rows, cols, _p(s.qs), _p(s.scales), _p(s.bsums), o, None, st)
        else:
            capi.call("wd_gemv_q8_k_f32" if t in K_TYPES else "wd_gemv_q8_0_f32", TYPES[t], _p(w), rows, cols, _p(s.qs), _p(s.scales), o, None, st)


def _run_dense(s, c):
    st, t, H, I, KV = _stream(), c["type"], c["hidden"], c["inner"], c["kv"]
    for b, m in enumerate(s.blocks):
        x, qkv, gu = s.inputs[b].data_ptr(), s.qkv[b].data_ptr(), s.gate_up[b].data_ptr()
        _quantise(s, t, x, H, st)
        _products(s, t, [m["q"], m["k"], m["v"]], [qkv, qkv + 4 * H, qkv + 4 * (H + KV)], st)
        _quantise(s, t, x + 4 * H, H, st)
        _products(s, t, [m["o"]], [s.attn[b].data_ptr()], st)
        _quantise(s, t, x + 8 * H, H, st)
        _products(s, t, [m["gate"], m["up"]], [gu, gu + 4 * I], st)
        capi.call("wd_silu_mul_experts_f32", gu, _p(s.act), I, 1, st)
        _quantise(s, t, _p(s.act), I, st)
        _products(s, t, [m["down"]], [s.mlp[b].data_ptr()], st)
    if s.head is not None:
        _quantise(s, t, _p(s.final), H, st)
        _products(s, t, [s.head], [s.logits.data_ptr()], st)
    return {"qkv": s.qkv, "attn": s.attn, "gate_up": s.gate_up, "mlp": s.mlp, "logits": s.logits}


# ---- what a pass cannot do without --------------------------------------------------------------------------------
def work(case):
    """Every weight that a pass uses, read once (of a batch of tokens: the experts of the union of their selections, about
    half of which coincide), inputs and outputs once; two operations per weight and token that uses it."""
    c = case
    if c["kind"] == "dense":
        H, I, KV, V, n, t = c["hidden"], c["inner"], c["kv"], c["vocab"], c["blocks"], c["type"]
        weights = n * (2 * H * H + 2 * KV * H + 3 * H * I) + V * H
        size = n * ((2 * H + 2 * KV + 2 * I) * _row(t, H) + (H * _row(t, I) if I else 0)) + V * _row(t, H)
        return {"bytes": size + 4 * (n * (5 * H + 2 * KV + 2 * I) + H + V), "flops": 2 * weights}
    H, F, E, k, NL, T = c["hidden"], c["ffn"], c["experts"], c["top_k"], c["layers"], c.get("tokens", 1)
    union = min(E, k * (T + 1) / 2)
    size = 4 * E * H + union * _expert_bytes(c)
    weights = E * H + 3 * k * H * F
    if c["shared"]:
        size += 4 * H + 2 * F * _row("q8_0", H) + H * _row("q8_0", F)
        weights += H + 3 * H * F
    vectors = 2 * T * NL if c["kind"] in ("layers", "tokens") else 3
    return {"bytes": NL * size + 4 * H * (vectors + 2 * c.get("hc", 0)), "flops": 2 * NL * T * weights}


def tolerance(case):
    """Order and rounding of every sum are part of the contract (results bit for bit those of the CPU path), except for
    Q4_0: its sums of 32-bit floats have no fixed order (about 1e-6), and where such a sum is quantised to 8 bits for the
    next product a value next to a rounding boundary may land on the other side (one step of 127 in a few of thousands)."""
    if case["kind"] == "dense" and case["type"] == "q4_0":
        return {"rel": 1e-5} if not case["blocks"] else {"rel": 1e-3, "max": 2e-2}
    return "exact"
