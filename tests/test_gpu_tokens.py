"""M tokens through one layer (speculative-verify batch): every selected expert is read once for all
tokens that routed to it, and each token's result is bit-identical to its own one-token pass and to
the CPU oracle."""
import ctypes as C

import numpy as np
import pytest

from warpdecode_amd import capi, synth

pytestmark = pytest.mark.gpu
SEED = 20261014


@pytest.fixture(scope="module")
def g():
    import gpu_util
    gpu_util.init()
    return gpu_util


def correlated_tokens(H, T, seed, mix=0.6):
    rng = synth.rng_for(SEED, 71, seed)
    base = rng.normal(0, 1, H)
    xs = []
    for _ in range(T):
        v = mix * base + (1 - mix) * rng.normal(0, 1, H)
        xs.append((v / np.sqrt(np.mean(v ** 2))).astype(np.float32))
    return np.stack(xs)


def run_tokens(g, dl, L, xs, flags=0, ids=None, weights=None):
    H, F, E, k = L["hidden"], L["expert_ffn"], L["n_experts"], L["top_k"]
    T = xs.shape[0]
    scs = [g.Scratch(H, F, E, k) for _ in range(T)]
    if ids is not None:
        for t in range(T):
            capi.call("wd_memcpy_h2d", C.c_void_p(scs[t].raw("ids")), np.ascontiguousarray(ids[t], np.int32).ctypes.data_as(C.c_void_p), 4 * k, None)
            capi.call("wd_memcpy_h2d", C.c_void_p(scs[t].raw("weights")), np.ascontiguousarray(weights[t], np.float32).ctypes.data_as(C.c_void_p), 4 * k, None)
    arr = (C.c_void_p * T)(*[s.h for s in scs])
    dx, out = g.dev(xs), g.empty((T, H), np.float32)
    capi.call("wd_moe_layer_tokens_f32", C.byref(dl.desc), g.ptr(dx), g.ptr(out), T, arr, flags, g.stream())
    g.sync()
    res = dict(out=g.host(out), ids=np.stack([s.get("ids", k, np.int32) for s in scs]),
               weights=np.stack([s.get("weights", k, np.float32) for s in scs]),
               accum=np.stack([s.get("accum", H, np.float32) for s in scs]),
               act=np.stack([s.get("act", (k + 1) * F, np.float32).reshape(k + 1, F) for s in scs]))
    for s in scs:
        s.close()
    return res


def run_single(g, dl, L, x, flags=0, ids=None, weights=None):
    r = run_tokens(g, dl, L, x[None, :], flags, None if ids is None else ids[None], None if weights is None else weights[None])
    return {n: v[0] for n, v in r.items()}


@pytest.mark.parametrize("T", [1, 4, 8])
def test_c4_tokens(g, oracle, T):
    """Workload C4: T tokens through the 512-expert top-10 IQ3_S/Q8_0 layer with overlapping routing."""
    L = synth.make_c2()
    dl = g.DeviceLayer(L)
    xs = correlated_tokens(2048, T, T)
    got = run_tokens(g, dl, L, xs)
    union = set(got["ids"].ravel().tolist())
    if T == 4:
        assert 10 < len(union) < 40        # the sets overlap but are not identical
    for t in range(T):
        want, d = oracle.moe_layer(L, xs[t])
        assert np.array_equal(got["ids"][t], d["ids"])
        assert g.same_bits(got["weights"][t], d["weights"])
        assert g.same_bits(got["act"][t][:10], d["act"])
        assert g.same_bits(got["accum"][t], d["routed"])
        assert g.same_bits(got["out"][t], want)
    one = run_tokens(g, dl, L, xs[:1])
    assert g.same_bits(one["out"][0], got["out"][0])


@pytest.mark.parametrize("gate_t,down_t,shared,H,F,E,k", [
    (synth.IQ2_S, synth.Q8_0, True, 512, 64, 16, 4),
    (synth.IQ3_S, synth.Q8_0, False, 768, 96, 8, 8),
    (synth.Q8_0, synth.Q8_0, False, 512, 64, 8, 2),         # not on the union path: one pass per token
    (synth.IQ3_S, synth.IQ4_NL, True, 512, 64, 8, 2),       # union pass for gate/up, the one-token down dispatch per token
    (synth.IQ2_S, synth.IQ4_NL, True, 2560, 640, 32, 10),   # the model's own types and shapes: the aligned multi-token down dispatch
    (synth.IQ3_S, synth.Q8_0, True, 2560, 640, 16, 4),      # 20-block Q8_0 down rows: the aligned multi-token down dispatch
    (synth.IQ3_S, synth.IQ4_NL, True, 2048, 512, 16, 4),    # 16-block IQ4_NL down rows, idem
    (synth.IQ2_S, synth.IQ4_NL, False, 2560, 640, 16, 8),   # idem without a shared expert
])
def test_tokens_equal_single_passes(g, oracle, gate_t, down_t, shared, H, F, E, k):
    L = synth.make_layer(H, F, E, k, gate_t, down_t, shared, seed=SEED, layer=7, router_sigma=1.0 / np.sqrt(H))
    dl = g.DeviceLayer(L)
    xs = correlated_tokens(H, 5, H)
    got = run_tokens(g, dl, L, xs)
    for t in range(5):
        one = run_single(g, dl, L, xs[t])
        assert np.array_equal(got["ids"][t], one["ids"])
        assert g.same_bits(got["out"][t], one["out"]) and g.same_bits(got["accum"][t], one["accum"])
        want, _ = oracle.moe_layer(L, xs[t])
        assert g.same_bits(got["out"][t], want)


@pytest.mark.parametrize("T,F", [(2, 32), (3, 640), (4, 96)])
def test_up_to_four_tokens_on_ten_super_blocks_of_iq2_s(g, oracle, T, F):
    """The kernel of up to four tokens whose look-ups are made half a block at a time."""
    H, E, k = 2560, 16, 6
    L = synth.make_layer(H, F, E, k, synth.IQ2_S, synth.IQ4_NL, True, seed=SEED, layer=17 + T, router_sigma=1.0 / np.sqrt(H))
    xs = correlated_tokens(H, T, H + T)
    got = run_tokens(g, g.DeviceLayer(L), L, xs)
    for t in range(T):
        want, d = oracle.moe_layer(L, xs[t])
        assert np.array_equal(got["ids"][t], d["ids"]) and g.same_bits(got["accum"][t], d["routed"]) and g.same_bits(got["out"][t], want)


def test_tokens_preselected_full_overlap(g, oracle):
    """All tokens name the same experts in different orders: one union entry per expert."""
    L = synth.make_c2(n_experts=32)
    dl = g.DeviceLayer(L)
    T, k = 4, 10
    xs = correlated_tokens(2048, T, 3)
    rng = np.random.default_rng(SEED)
    base = rng.choice(32, size=k, replace=False)
    ids = np.stack([rng.permutation(base) for _ in range(T)]).astype(np.int32)
    wts = rng.uniform(0.05, 0.15, (T, k)).astype(np.float32)
    got = run_tokens(g, dl, L, xs, flags=capi.MOE_PRESELECTED, ids=ids, weights=wts)
    for t in range(T):
        want, _ = oracle.moe_layer(L, xs[t], ids=ids[t], weights=wts[t])
        assert g.same_bits(got["out"][t], want)


def test_tokens_errors(g):
    L = synth.make_layer(512, 64, 8, 2, synth.IQ3_S, synth.Q8_0, False)
    dl = g.DeviceLayer(L)
    sc = g.Scratch(512, 64, 8, 2)
    arr = (C.c_void_p * 2)(sc.h, sc.h)
    x = g.empty((2, 512), np.float32)
    lib = capi.load()
    assert lib.wd_moe_layer_tokens_f32(C.byref(dl.desc), g.ptr(x), g.ptr(x), 2, arr, 0, None) == -1   # shared scratch
    assert lib.wd_moe_layer_tokens_f32(C.byref(dl.desc), g.ptr(x), g.ptr(x), 9, arr, 0, None) == -1
    sc.close()


@pytest.mark.parametrize("shape", ["c2", "model", "small-unaligned"])
def test_tokens_on_a_table_of_expert_views(g, oracle, shape):
    """wd_moe_layer_tokens_pairs_f32: the pass over (gate, up, down) views given expert by expert - the form in which the
    reference's token batch receives acquired experts (src/qwen38_moe.cuh:2907-3109) - with entry numbers as ids.  The
    views here point into resident tensors, in a shuffled order with a few entries nobody selects; every token must
    come out as from the pass over the tensors themselves, i.e. as from the oracle."""
    if shape == "c2":
        L, T = synth.make_c2(n_experts=64), 4
    elif shape == "model":
        L, T = synth.make_layer(2560, 640, 32, 8, synth.IQ2_S, synth.IQ4_NL, shared=True, seed=SEED + 3), 3
    else:
        L, T = synth.make_layer(512, 64, 16, 4, synth.IQ3_S, synth.Q8_0, shared=False, seed=SEED + 4), 5
    H, F, E, k = L["hidden"], L["expert_ffn"], L["n_experts"], L["top_k"]
    dl = g.DeviceLayer(L)
    if shape == "small-unaligned":     # views that are only 2-byte aligned: the tensors copied to an odd-word offset
        for name in ("gate", "up", "down"):
            raw = np.concatenate([np.zeros(2, np.uint8), np.ascontiguousarray(L[name]).reshape(-1)])
            dl.keep[name + "_shifted"] = g.dev(raw)
            setattr(dl.desc, name, dl.keep[name + "_shifted"].data_ptr() + 2)
    xs = correlated_tokens(H, T, 31 + T)
    ref = run_tokens(g, dl, L, xs)
    rng = np.random.default_rng(SEED + 55)
    union = sorted(set(ref["ids"].ravel().tolist()))
    entries = union + [e for e in range(E) if e not in union][:3]
    order = rng.permutation(len(entries))
    entries = [entries[i] for i in order]
    entry_of = {e: i for i, e in enumerate(entries)}
    d = dl.desc
    P = C.c_void_p * len(entries)
    hg = P(*[d.gate + e * d.gate_stride for e in entries])
    hu = P(*[d.up + e * d.up_stride for e in entries])
    hd = P(*[d.down + e * d.down_stride for e in entries])
    scs = [g.Scratch(H, F, E, k) for _ in range(T)]
    for t in range(T):
        vids = np.array([entry_of[e] for e in ref["ids"][t]], np.int32)
        capi.call("wd_memcpy_h2d", C.c_void_p(scs[t].raw("ids")), vids.ctypes.data_as(C.c_void_p), 4 * k, None)
        capi.call("wd_memcpy_h2d", C.c_void_p(scs[t].raw("weights")), np.ascontiguousarray(ref["weights"][t]).ctypes.data_as(C.c_void_p), 4 * k, None)
    arr = (C.c_void_p * T)(*[s.h for s in scs])
    dx, out = g.dev(xs), g.empty((T, H), np.float32)
    lib = capi.load()
    for rep in range(6):       # more calls than the ring of pointer tables has entries
        capi.call("wd_moe_layer_tokens_pairs_f32", C.byref(d), hg, hu, hd, len(entries), g.ptr(dx), g.ptr(out), T, arr,
                  capi.MOE_PRESELECTED, g.stream())
    g.sync()
    got = g.host(out)
    for t in range(T):
        want, dump = oracle.moe_layer(L, xs[t])
        assert g.same_bits(got[t], want), (shape, t)
        assert g.same_bits(scs[t].get("accum", H, np.float32), dump["routed"]), (shape, t)
        assert g.same_bits(got[t], ref["out"][t])
    assert lib.wd_moe_layer_tokens_pairs_f32(C.byref(d), hg, hu, hd, len(entries), g.ptr(dx), g.ptr(out), T, arr, 0, g.stream()) == -1
    assert lib.wd_moe_layer_tokens_pairs_f32(C.byref(d), hg, hu, hd, 129, g.ptr(dx), g.ptr(out), T, arr, capi.MOE_PRESELECTED, g.stream()) == -1
    for s in scs:
        s.close()


@pytest.mark.parametrize("H,T", [(17920, 8), (24064, 6), (35840, 1)])
def test_the_longest_rows_of_a_token_batch(g, oracle, H, T):
    """Rows whose inputs fill the LDS: T of them in Q8_K beside the codebooks and the union (162128 of 163840 bytes at 17920 and eight
    tokens), or one in f32 beside the selection's work area."""
    F, E, k = 32, 8, 2
    L = synth.make_layer(H, F, E, k, synth.IQ2_S, synth.Q8_0, True, seed=SEED, layer=37, router_sigma=1.0 / np.sqrt(H))
    xs = correlated_tokens(H, T, 13)
    dl = g.DeviceLayer(L)
    r = run_tokens(g, dl, L, xs)
    for t in range(T):
        assert g.same_bits(r["out"][t], oracle.moe_layer(L, xs[t])[0]), t


def test_a_refused_table_of_expert_views_runs_nothing(g, oracle):
    """Down rows of more than 48 blocks have no dispatch for a pointer table: the call is refused before anything is launched (the
    scratches' activations stay as they are), and a preselected and a routed batch on the same scratches are the oracle's."""
    H, F, E, k, T = 512, 1568, 16, 4, 3
    L = synth.make_layer(H, F, E, k, synth.IQ3_S, synth.Q8_0, True, seed=SEED, layer=36, router_sigma=1.0 / np.sqrt(H))
    xs = correlated_tokens(H, 2 * T, 12)
    dl, scr = g.DeviceLayer(L), [g.Scratch(H, F, E, k) for _ in range(T)]
    arr = (C.c_void_p * T)(*[s.h for s in scr])
    ids, wts = np.arange(k, dtype=np.int32), np.full(k, 0.25, np.float32)
    for s in scr:
        capi.call("wd_memcpy_h2d", C.c_void_p(s.raw("ids")), ids.ctypes.data_as(C.c_void_p), 4 * k, None)
        capi.call("wd_memcpy_h2d", C.c_void_p(s.raw("weights")), wts.ctypes.data_as(C.c_void_p), 4 * k, None)
    d, P, lib = dl.desc, C.c_void_p * E, capi.load()
    table = [P(*[base + e * stride for e in range(E)]) for base, stride in ((d.gate, d.gate_stride), (d.up, d.up_stride), (d.down, d.down_stride))]
    dx, out = g.dev(xs), g.empty((T, H), np.float32)
    for flags in (capi.MOE_PRESELECTED, 0):
        before = [s.get("act", (k + 1) * F, np.float32) for s in scr]
        rc = lib.wd_moe_layer_tokens_pairs_f32(C.byref(d), *table, E, C.c_void_p(dx.data_ptr() + 4 * H * T), g.ptr(out), T, arr, capi.MOE_PRESELECTED, g.stream())
        assert rc == -1 and "no multi-token dispatch" in lib.wd_last_error().decode()
        g.sync()
        for s, a in zip(scr, before):
            assert g.same_bits(s.get("act", (k + 1) * F, np.float32), a)
        capi.call("wd_moe_layer_tokens_f32", C.byref(d), g.ptr(dx), g.ptr(out), T, arr, flags, g.stream())
        g.sync()
        for t in range(T):
            want = oracle.moe_layer(L, xs[t], ids=ids, weights=wts)[0] if flags else oracle.moe_layer(L, xs[t])[0]
            assert g.same_bits(g.host(out)[t], want), (flags, t)
    assert [lib.wd_moe_scratch_status(s.h) for s in scr] == [0] * T
    for s in scr:
        s.close()


@pytest.mark.parametrize("gate,F", [(synth.IQ3_S, 64), (synth.Q8_0, 64), (synth.IQ2_S, 1568)])
def test_bounded_wait_of_a_token_batch(g, oracle, gate, F):
    """With a wait limit of one poll the routed workgroups give up before the ids are published: every token's status word and
    data say so; with the default limit the same scratches give the oracle's results, in one launch and in two."""
    H, E, k, T = 512, 64, 6, 3
    L = synth.make_layer(H, F, E, k, gate, synth.Q8_0, True, seed=SEED, layer=33, router_sigma=1.0 / np.sqrt(H))
    xs = correlated_tokens(H, T, 9)
    dl, scr = g.DeviceLayer(L), [g.Scratch(H, F, E, k) for _ in range(T)]
    arr = (C.c_void_p * T)(*[s.h for s in scr])
    dx, out = g.dev(xs), g.empty((T, H), np.float32)
    lib = capi.load()
    capi.call("wd_moe_scratch_set_wait_limit", scr[0].h, 1)
    capi.call("wd_moe_layer_tokens_f32", C.byref(dl.desc), g.ptr(dx), g.ptr(out), T, arr, 0, g.stream())
    g.sync()
    assert [lib.wd_moe_scratch_status(s.h) for s in scr] == [1] * T
    assert np.isnan(g.host(out)).all()
    for s in scr:
        capi.call("wd_moe_scratch_set_wait_limit", s.h, 0)
    for flags in (0, capi.MOE_SPLIT_AB, 0):
        capi.call("wd_moe_layer_tokens_f32", C.byref(dl.desc), g.ptr(dx), g.ptr(out), T, arr, flags, g.stream())
        g.sync()
        for t in range(T):
            want, d = oracle.moe_layer(L, xs[t])
            assert np.array_equal(scr[t].get("ids", k, np.int32), d["ids"]) and g.same_bits(g.host(out)[t], want), (flags, t)
    assert [lib.wd_moe_scratch_status(s.h) for s in scr] == [0] * T
    for s in scr:
        s.close()


@pytest.mark.parametrize("E,k", [(64, 6), (512, 10), (640, 10)])
@pytest.mark.parametrize("form", ["one launch", "split", "preselected"])
def test_logits_that_are_late_are_reported(g, oracle, E, k, form):
    """With a wait limit of one poll the workgroup that selects a token's experts may find logits missing, and those that wait for the ids the
    ids: a token's results are then NaN with its status word set, and the oracle's where it is clear.  Where nobody in the dispatch
    waits for the ids - the routed part is a launch of its own, or the ids are given - nothing is ever late."""
    preselected = form == "preselected"
    H, F, T = 512, 64, 5
    L = synth.make_layer(H, F, E, k, synth.IQ3_S, synth.Q8_0, True, seed=SEED, layer=34, router_sigma=1.0 / np.sqrt(H))
    xs = correlated_tokens(H, T, 10)
    dl, scr = g.DeviceLayer(L), [g.Scratch(H, F, E, k) for _ in range(T)]
    arr = (C.c_void_p * T)(*[s.h for s in scr])
    dx, out = g.dev(xs), g.empty((T, H), np.float32)
    lib = capi.load()
    ids, wts = np.arange(k, dtype=np.int32), np.full(k, 0.125, np.float32)
    flags = {"one launch": 0, "split": capi.MOE_SPLIT_AB, "preselected": capi.MOE_PRESELECTED}[form]
    want = [oracle.moe_layer(L, x, ids=ids, weights=wts)[0] if preselected else oracle.moe_layer(L, x)[0] for x in xs]
    for limit in (1,) * 12 + (0,):
        for s in scr:
            capi.call("wd_moe_scratch_set_wait_limit", s.h, limit)
            if preselected:
                capi.call("wd_memcpy_h2d", C.c_void_p(s.raw("ids")), ids.ctypes.data_as(C.c_void_p), 4 * k, g.stream())
                capi.call("wd_memcpy_h2d", C.c_void_p(s.raw("weights")), wts.ctypes.data_as(C.c_void_p), 4 * k, g.stream())
        out.zero_()
        capi.call("wd_moe_layer_tokens_f32", C.byref(dl.desc), g.ptr(dx), g.ptr(out), T, arr, flags, g.stream())
        g.sync()
        for t, s in enumerate(scr):
            late = lib.wd_moe_scratch_status(s.h)
            assert late in ((0, 1) if limit and form == "one launch" else (0,))
            assert np.isnan(g.host(out)[t]).all() if late else g.same_bits(g.host(out)[t], want[t]), (limit, t)
    for s in scr:
        s.close()


@pytest.mark.parametrize("E,k", [(64, 6), (2048, 4), (2056, 4)])
def test_scratches_at_many_addresses(g, oracle, E, k):
    """What workgroups hand on lies in pieces of the scratch chosen by where the scratch happens to be (and the logits outside of them where
    they do not fit one): scratches of different sizes, used one by one and as a batch, give the oracle's results, twice."""
    H, F, T = 512, 64, 8
    L = synth.make_layer(H, F, 64, k, synth.IQ3_S, synth.Q8_0, True, seed=SEED, layer=39, router_sigma=1.0 / np.sqrt(H))
    xs = correlated_tokens(H, T, 13)
    want = [oracle.moe_layer(L, x)[0] for x in xs]
    dl = g.DeviceLayer(L)
    scr = [g.Scratch(H, F, E, k + t) for t in range(T)]
    arr = (C.c_void_p * T)(*[s.h for s in scr])
    dx, out = g.dev(xs), g.empty((T, H), np.float32)
    for turn in range(2):
        for t, s in enumerate(scr):
            row = C.c_void_p(dx.data_ptr() + 4 * H * t), C.c_void_p(out.data_ptr() + 4 * H * t)
            capi.call("wd_moe_layer_f32", C.byref(dl.desc), *row, s.h, 0, g.stream())
        g.sync()
        assert g.same_bits(g.host(out), np.stack(want)), ("layers", turn)
        out.zero_()
        capi.call("wd_moe_layer_tokens_f32", C.byref(dl.desc), g.ptr(dx), g.ptr(out), T, arr, 0, g.stream())
        g.sync()
        assert g.same_bits(g.host(out), np.stack(want)), ("batch", turn)
    stack = (capi.MoeLayer * 35)(*[dl.desc] * 35)    # records of published ids beyond the first piece's
    x0, o0 = g.dev(xs[0]), g.empty(H, np.float32)
    for flags in (0, capi.MOE_SPLIT_AB):
        xc = g.dev(xs[0])
        capi.call("wd_moe_stack_f32", stack, 35, g.ptr(xc), g.ptr(out), scr[0].h, None, 0.0, flags, g.stream())
        capi.call("wd_moe_layer_f32", C.byref(dl.desc), g.ptr(x0), g.ptr(o0), scr[0].h, 0, g.stream())
        g.sync()
        assert g.same_bits(g.host(out)[0], want[0]) and g.same_bits(g.host(o0), want[0]), flags
    assert [capi.load().wd_moe_scratch_status(s.h) for s in scr] == [0] * T
    for s in scr:
        s.close()


@pytest.mark.parametrize("shape", ["eight-blocks", "q8_0", "ids-by-the-block-form"])
def test_passes_that_end_before_the_down_projections(g, oracle, shape):
    """Calls of dispatch A or of A and B without C, on one input, leave nothing on the scratch that a pass of another kind takes
    for its own: one-token layers, token batches and the dispatches one by one, on other inputs, give the oracle's results."""
    H, F, E, k, gate, shared = {"eight-blocks": (2048, 64, 64, 6, synth.IQ3_S, True), "q8_0": (512, 96, 24, 4, synth.Q8_0, False),
                                "ids-by-the-block-form": (512, 64, 640, 10, synth.IQ2_S, True)}[shape]
    T = 3
    L = synth.make_layer(H, F, E, k, gate, synth.Q8_0, shared, seed=SEED, layer=35, router_sigma=1.0 / np.sqrt(H))
    xs = correlated_tokens(H, 2 * T, 11, mix=0.2)
    dl, scr = g.DeviceLayer(L), [g.Scratch(H, F, E, k) for _ in range(T)]
    arr = (C.c_void_p * T)(*[s.h for s in scr])
    stack = (capi.MoeLayer * 3)(dl.desc, dl.desc, dl.desc)
    dx, out = g.dev(xs), g.empty((T, H), np.float32)
    want = [oracle.moe_layer(L, x)[0] for x in xs]
    A, B, CC = capi.MOE_ONLY_A, capi.MOE_ONLY_B, capi.MOE_ONLY_C
    row = lambda b, t: C.c_void_p(b.data_ptr() + 4 * H * t)

    def layer(t, x, flags):
        capi.call("wd_moe_layer_f32", C.byref(dl.desc), row(dx, x), row(out, t), scr[t].h, flags, g.stream())

    def one_by_one(t, x):
        layer(t, x, A)
        layer(t, x, B | capi.MOE_PRESELECTED)
        layer(t, x, CC | capi.MOE_PRESELECTED)

    before = {"A": lambda: [layer(t, T + t, A) for t in range(T)],
              "A and B": lambda: [layer(t, T + t, A | B) for t in range(T)],
              "A and B apart": lambda: [layer(t, T + t, A | B | capi.MOE_SPLIT_AB) for t in range(T)],
              "a batch's A and B": lambda: capi.call("wd_moe_layer_tokens_f32", C.byref(dl.desc), row(dx, T), g.ptr(out), T, arr, A | B, g.stream()),
              "a stack's A and B": lambda: [capi.call("wd_moe_stack_f32", stack, 3, row(dx, T), row(out, 0), s.h, None, 0.0, A | B, g.stream()) for s in scr]}
    passes = {"batch": lambda: capi.call("wd_moe_layer_tokens_f32", C.byref(dl.desc), row(dx, 0), g.ptr(out), T, arr, 0, g.stream()),
              "batch in two": lambda: capi.call("wd_moe_layer_tokens_f32", C.byref(dl.desc), row(dx, 0), g.ptr(out), T, arr, capi.MOE_SPLIT_AB, g.stream()),
              "layer": lambda: [layer(t, t, 0) for t in range(T)], "one by one": lambda: [one_by_one(t, t) for t in range(T)]}
    for first, ends_early in before.items():
        for second, whole in passes.items():
            ends_early()
            ends_early()
            out.zero_()
            whole()
            g.sync()
            for t in range(T):
                assert g.same_bits(g.host(out)[t], want[t]), (first, second, t)
    assert [capi.load().wd_moe_scratch_status(s.h) for s in scr] == [0] * T
    for s in scr:
        s.close()


@pytest.mark.parametrize("E,k", [(64, 6), (640, 10)])
def test_logits_of_the_reserved_nan(g, E, k):
    """A router row, then the shared expert's gate row, whose logit is the NaN that stands for "not handed on yet": one-token layers and
    token batches end with the status word clear and with what any other NaN there gives.  (A NaN among the logits leaves k times the
    same id with infinite weights, so only the selection and the staged dispatches' results, which hand nothing on, are compared.)"""
    H, F, T = 512, 64, 3
    L = synth.make_layer(H, F, E, k, synth.IQ3_S, synth.Q8_0, True, seed=SEED, layer=38, router_sigma=1.0 / np.sqrt(H))
    xs = correlated_tokens(H, T, 14)
    clean = run_tokens(g, g.DeviceLayer(L), L, xs)
    late = int(clean["ids"][0][k - 1])
    lib = capi.load()
    for name, row in (("router", late), ("router", E - 1), ("shared_gate_inp", 0)):
        seen = []
        for bits in (0xffffffff, 0x7fc00000):
            bad = dict(L)
            bad[name] = np.array(L[name], np.float32)
            bad[name].reshape(-1, H)[row, 5] = np.array([bits], np.uint32).view(np.float32)[0]
            dl, scr = g.DeviceLayer(bad), [g.Scratch(H, F, E, k) for _ in range(T)]
            arr = (C.c_void_p * T)(*[s.h for s in scr])
            dx = g.dev(xs)
            for how in ("batch", "batch in two", "layer", "staged"):
                out = g.empty((T, H), np.float32)
                if how.startswith("batch"):
                    capi.call("wd_moe_layer_tokens_f32", C.byref(dl.desc), g.ptr(dx), g.ptr(out), T, arr, 0 if how == "batch" else capi.MOE_SPLIT_AB, g.stream())
                else:
                    for t, s in enumerate(scr):
                        capi.call("wd_moe_layer_f32", C.byref(dl.desc), C.c_void_p(dx.data_ptr() + 4 * H * t), C.c_void_p(out.data_ptr() + 4 * H * t), s.h,
                                  capi.MOE_STAGED if how == "staged" else 0, g.stream())
                g.sync()
                assert [lib.wd_moe_scratch_status(s.h) for s in scr] == [0] * T, (name, row, how)
                if name == "router":  # (the logits as the caller sees them: the word is the reserved one)
                    assert [int(s.get("logits", E, np.float32).view(np.uint32)[row]) for s in scr] == [bits] * T, how
                ids, weights, accum = (np.stack([s.get(n, w, d) for s in scr]) for n, w, d in (("ids", k, np.int32), ("weights", k, np.float32), ("accum", H, np.float32)))
                seen.append((how, ids, weights, accum, g.host(out)))
            for s in scr:
                s.close()
        _, ids, *staged = seen[-1]
        for how, ids_h, *values in seen:
            assert np.array_equal(ids_h, ids), (name, row, how)
            for a, b in list(zip(values, staged))[:1 if how.startswith("batch") and name == "router" else 3]:
                assert np.array_equal(np.isnan(a), np.isnan(b)) and g.same_bits(a[~np.isnan(a)], b[~np.isnan(b)]), (name, row, how)
            if name == "shared_gate_inp":
                assert np.array_equal(ids_h, clean["ids"]) and g.same_bits(values[1], clean["accum"]) and np.isnan(values[2]).all(), how
