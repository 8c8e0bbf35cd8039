"""The layer dispatches at the sizes where the choice of a kernel or the end of a tile changes: super-blocks per gate/up row
around the passes of eight and the two fetches, down rows around the 16-block passes, router rows of one and two waves,
experts around the 64-logit registers of the selection, tensors that are only 2-byte aligned."""
import numpy as np
import pytest

from warpdecode_amd import synth
from test_gpu_layer import SEED, check_layer

pytestmark = pytest.mark.gpu
IQ3, IQ2, Q8, IQ4 = synth.IQ3_S, synth.IQ2_S, synth.Q8_0, synth.IQ4_NL


@pytest.fixture(scope="module")
def g():
    import gpu_util
    gpu_util.init()
    return gpu_util


SHAPES = [
    (256, 64, 8, 8, IQ3, IQ4, True),         # one super-block, every expert selected
    (1792, 1536, 136, 10, IQ2, Q8, False),   # a last pass of seven, down rows of 48 blocks
    (2304, 544, 72, 9, IQ3, IQ4, True),      # nine super-blocks (a pass of one), an unpaired 17th down block
    (2304, 800, 64, 8, IQ4, IQ4, True),      # 72 gate blocks: a second pass of eight
    (2816, 1568, 264, 5, IQ4, IQ4, False),   # 49 down blocks: beyond what is held in flight
    (3328, 160, 200, 7, Q8, Q8, True),       # five down blocks
    (4096, 1056, 24, 3, IQ2, Q8, True),      # sixteen super-blocks, 33 down blocks
    (4352, 64, 520, 2, IQ3, Q8, True),       # beyond the aligned fetch and the paired router rows
    (4352, 1024, 8, 6, IQ3, Q8, True),       # rows taken field by field, in a loop: of every type
    (4352, 1024, 8, 7, IQ2, IQ4, False),
    (4608, 1024, 8, 6, Q8, Q8, True),
    (4352, 1024, 8, 6, IQ4, IQ4, True),
    (4352, 544, 8, 4, Q8, IQ4, False),       # field by field, an item per workgroup
    (4352, 96, 16, 5, IQ2, Q8, True),
    (4608, 64, 8, 3, IQ4, Q8, True),
    (1024, 96, 128, 15, IQ4, Q8, True),      # the largest selection of one wave
    (512, 64, 136, 16, IQ3, Q8, False),      # top-16: the selection by a whole workgroup, more candidates than it ranks
    (512, 64, 512, 16, IQ3, Q8, True),
    (256, 288, 16, 16, IQ3, Q8, True),       # seventeen down matrices: two per wave, rows of 9, 16 and 24 blocks
    (512, 512, 16, 16, IQ2, IQ4, True),
    (256, 768, 16, 16, Q8, IQ4, True),
    (512, 544, 16, 16, IQ4, Q8, True),
    (512, 256, 16, 16, IQ3, IQ4, True),      # eight blocks: the four-row form
    (4096, 800, 16, 12, IQ3, Q8, True),      # 32 MB and more of down rows: as aligned words; 25, 32, 33 and 48 blocks
    (4096, 1024, 16, 9, IQ2, Q8, True),
    (4096, 1056, 16, 9, IQ3, Q8, True),
    (4096, 1536, 8, 8, IQ2, Q8, False),
    (4608, 1024, 16, 15, IQ3, IQ4, True),    # (as blocks)
    (4096, 1536, 16, 12, IQ2, IQ4, False),
    (3072, 1536, 16, 16, IQ3, IQ4, True),    # items beyond the device, 17 matrices
]


@pytest.mark.parametrize("H,F,E,k,gate,down,shared", SHAPES)
def test_layer_shapes(g, oracle, H, F, E, k, gate, down, shared):
    L = synth.make_layer(H, F, E, k, gate, down, shared, seed=SEED, layer=H + F, router_sigma=1.0 / np.sqrt(H))
    x = synth.rms_normed(synth.rng_for(SEED, 61, H + F), H)
    check_layer(g, oracle, L, x)
    ids = synth.rng_for(SEED, 62, H + F).permutation(E)[:k].astype(np.int32)   # known before the launch
    check_layer(g, oracle, L, x, ids=ids, weights=np.linspace(0.3, 0.05, k).astype(np.float32), flags=1)


@pytest.mark.parametrize("H,nb,k,down,shared", [
    (256, 1, 2, IQ4, False),      # one row per workgroup, fewer matrices than waves that fold
    (512, 16, 3, Q8, False), (768, 17, 6, IQ4, True), (1024, 33, 1, Q8, True), (1024, 48, 8, IQ4, True),
    (1280, 12, 5, Q8, True), (1280, 13, 3, IQ4, False), (1280, 25, 15, IQ4, True), (1280, 37, 4, Q8, False),
    (1536, 10, 4, Q8, True), (1536, 9, 4, IQ4, True), (1536, 17, 7, IQ4, False), (1536, 41, 2, IQ4, True),
    (2304, 13, 6, IQ4, True), (2304, 24, 5, Q8, False), (2304, 36, 8, Q8, True), (2560, 12, 4, IQ4, True), (2560, 37, 6, IQ4, False),
    (2816, 11, 5, IQ4, False), (2816, 40, 7, Q8, True), (3072, 10, 4, Q8, True), (3072, 31, 5, IQ4, True), (3072, 41, 5, IQ4, False),
    (3328, 9, 6, IQ4, True), (3328, 27, 5, IQ4, True), (3328, 45, 6, IQ4, False), (3584, 19, 6, IQ4, True), (3584, 37, 7, Q8, False),
    (3840, 8, 6, Q8, False), (3840, 17, 5, IQ4, True), (4096, 7, 15, IQ4, True), (4096, 33, 6, IQ4, False)])
def test_rows_per_compute_unit(g, oracle, H, nb, k, down, shared):
    """Down rows of nb blocks, hidden / 256 rows per workgroup: passes that end on a row's last block, one before and one
    behind it, an unpaired last IQ4_NL block in passes of even and odd length, rows in one group and in two of equal and unequal size."""
    F, E = 32 * nb, 16
    L = synth.make_layer(H, F, E, k, IQ3, down, shared, seed=SEED, layer=H + nb, router_sigma=1.0 / np.sqrt(H))
    check_layer(g, oracle, L, synth.rms_normed(synth.rng_for(SEED, 67, H + nb), H))


@pytest.mark.parametrize("gate", [Q8, IQ4])
@pytest.mark.parametrize("H", [256, 768, 1024, 1280, 1536, 2048, 2304, 3072, 3328, 4096, 4352, 6400])
def test_row_pairs_of_blocks(g, oracle, H, gate):
    """Gate and up rows (and the shared expert's) of 8 to 200 blocks: passes that end in the first or the second half of the
    tile, on a whole one, and rows of one, two and more passes."""
    F, E, k = 96, 16, 3
    L = synth.make_layer(H, F, E, k, gate, Q8, True, seed=SEED, layer=H, router_sigma=1.0 / np.sqrt(H))
    check_layer(g, oracle, L, synth.rms_normed(synth.rng_for(SEED, 66, H), H))


@pytest.mark.parametrize("H,F,E", [(256, 32, 64), (256, 32, 128), (256, 32, 256), (256, 32, 512), (2048, 512, 64)])
def test_near_tie_at_the_end_of_a_key_cell(g, oracle, H, F, E):
    """Router rows whose logits are the near-tie row: the layer, a token batch and a stack of one layer (one launch at
    2048 / 512) take the expert with the lower id of two equal probabilities."""
    import ctypes as C

    from test_selection_margin import near_tie_row
    from warpdecode_amd import capi
    k, T = 6, 2
    L = synth.make_layer(H, F, E, k, IQ3, Q8, True, seed=SEED, layer=E, router_sigma=1.0)
    L["router"] = np.ascontiguousarray(L["router"], np.float32).reshape(E, H).copy()
    L["router"][:, 0] = near_tie_row(E)
    x = np.zeros(H, np.float32)
    x[0] = 1.0
    got = check_layer(g, oracle, L, x)
    assert got["ids"][-1] == 30
    want, _ = oracle.moe_layer(L, x)
    dl, scr = g.DeviceLayer(L), [g.Scratch(H, F, E, k) for _ in range(T)]
    dx, out = g.dev(np.stack([x] * T)), g.empty((T, H), np.float32)
    capi.call("wd_moe_layer_tokens_f32", C.byref(dl.desc), g.ptr(dx), g.ptr(out), T, (C.c_void_p * T)(*[s.h.value for s in scr]), 0, g.stream())
    g.sync()
    assert all(g.same_bits(g.host(out)[t], want) for t in range(T))
    dx, out = g.dev(x), g.empty(H, np.float32)
    capi.call("wd_moe_stack_f32", (capi.MoeLayer * 1)(dl.desc), 1, g.ptr(dx), g.ptr(out), scr[0].h, None, 0.05, 0, g.stream())
    g.sync()
    assert g.same_bits(g.host(out), want)
    for s in scr:
        s.close()


@pytest.mark.parametrize("H,F,k", [(2048, 512, 16), (2560, 640, 4), (3072, 96, 3)])
def test_tensors_on_two_byte_boundaries(g, oracle, monkeypatch, H, F, k):
    import torch
    E = 16
    L = synth.make_layer(H, F, E, k, IQ3, Q8, True, seed=SEED, layer=H + 1, router_sigma=1.0 / np.sqrt(H))
    x = synth.rms_normed(synth.rng_for(SEED, 63, H), H)
    aligned = g.dev

    def dev(a):
        if a.dtype != np.uint8:
            return aligned(a)
        t = torch.empty(a.size + 16, dtype=torch.uint8, device="cuda")[2:2 + a.size]
        t.copy_(torch.from_numpy(np.ascontiguousarray(a).reshape(-1)))
        return t

    monkeypatch.setattr(g, "dev", dev)
    check_layer(g, oracle, L, x)


@pytest.mark.parametrize("H,F,E,k,gate,down,shared,T", [
    (256, 32, 8, 2, Q8, Q8, False, 2),           # one block per lane row, one down block
    (2048, 544, 24, 6, Q8, IQ4, True, 5),        # 64 gate blocks, an unpaired 17th down block
    (2304, 768, 16, 4, IQ4, Q8, True, 8),        # 72 gate blocks: a second pass of eight; 24 down blocks
    (1792, 512, 32, 5, IQ3, IQ4, False, 3),      # a pass of seven super-blocks
    (2304, 640, 16, 3, IQ2, IQ4, True, 4),       # nine
    (4096, 1056, 16, 3, IQ3, Q8, True, 7),       # sixteen, 33 down blocks
    (512, 800, 16, 4, IQ3, Q8, True, 5),         # 25 and 32 down blocks
    (768, 1024, 16, 3, IQ2, IQ4, False, 8),
    (3072, 1536, 16, 10, IQ4, IQ4, True, 2),     # 48 down blocks
    (256, 288, 16, 3, IQ3, IQ4, True, 4),        # hidden / 256 rows per workgroup: nine blocks
    (768, 1440, 16, 6, IQ3, Q8, True, 7),
    (1024, 512, 16, 4, IQ2, IQ4, False, 5),
    (1280, 1184, 16, 5, IQ3, IQ4, True, 8),      # 37
    (1536, 1312, 16, 10, IQ2, Q8, True, 3),      # 41
    (2304, 800, 16, 3, IQ3, IQ4, True, 5),       # two groups of five and four rows, 25 blocks
    (2560, 1152, 16, 6, IQ2, Q8, False, 2),
    (2816, 1312, 16, 2, IQ3, IQ4, True, 6),      # six and five rows, 41 blocks
    (3072, 1216, 16, 4, IQ2, Q8, True, 8),
    (1024, 1568, 16, 2, IQ2, Q8, True, 6)])      # 49: the one-token dispatch per token
def test_token_batch_shapes(g, oracle, H, F, E, k, gate, down, shared, T):
    import ctypes as C

    from warpdecode_amd import capi
    L = synth.make_layer(H, F, E, k, gate, down, shared, seed=SEED, layer=H + T, router_sigma=1.0 / np.sqrt(H))
    base = synth.rng_for(SEED, 64, H + T).normal(0, 1, H)
    xs = np.stack([synth.rms_normed(synth.rng_for(SEED, 65, H + T, t), H) + base for t in range(T)]).astype(np.float32)
    dl, scr = g.DeviceLayer(L), [g.Scratch(H, F, E, k) for _ in range(T)]
    dx, out = g.dev(xs), g.empty((T, H), np.float32)
    arr = (C.c_void_p * T)(*[s.h.value for s in scr])
    capi.call("wd_moe_layer_tokens_f32", C.byref(dl.desc), g.ptr(dx), g.ptr(out), T, arr, 0, g.stream())
    g.sync()
    got = g.host(out)
    for t in range(T):
        want, d = oracle.moe_layer(L, xs[t])
        assert np.array_equal(scr[t].get("ids", k, np.int32), d["ids"])
        assert g.same_bits(got[t], want), t
    for s in scr:
        s.close()
