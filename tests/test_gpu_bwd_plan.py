"""The backward's work division (bwd_plan, csrc/fa_launch.hip): phases apart,
key tiles shared by several workgroups, two workgroups per CU and one item per
tile, each at shapes whose plan takes it (asserted: fa_bwd_plan), with ragged
edges, against the float64 oracle at the suite's bars. No counterpart in the
reference, which has one backward grid (flash_bwd.cuh:475-483)."""
import ctypes

import numpy as np
import pytest
import torch

from helpers import (FWD_MAX_ABS, GRAD_REL_L2, REF_REL, bwd_plan, load_capi, make_inputs,
                     np64)
from oracle import attention as ora

pytestmark = pytest.mark.gpu

DEV = "cuda"

# B, Hq, Hkv, N, D, causal: apart, parts, two workgroups per CU (bwd_plan)
CASES = [
    ((1, 4, 4, 256, 64, True), (True, 1, False)),
    ((1, 16, 1, 385, 64, True), (True, 16, False)),   # one kv head, a ragged last tile
    ((1, 16, 1, 511, 128, False), (True, 16, False)),  # keys past N masked once
    ((1, 6, 2, 129, 128, True), (True, 3, False)),    # a tile of one row; more parts than steps
    ((2, 4, 2, 300, 256, True), (True, 4, False)),
    ((1, 8, 2, 300, 96, True), (True, 8, False)),
    ((1, 8, 2, 200, 40, False), (True, 6, False)),    # a head dim below its width
    ((3, 12, 12, 700, 64, False), (True, 1, True)),
    ((5, 8, 2, 774, 64, True), (True, 3, True)),
    ((11, 4, 1, 387, 64, False), (True, 3, True)),
    ((9, 8, 8, 537, 128, True), (True, 1, False)),    # over one round of one item per tile
    ((10, 12, 12, 394, 64, True), (False, 1, True)),
    ((9, 4, 4, 778, 64, True), (False, 1, False)),    # tiles split in pairs, an odd number
    ((10, 12, 12, 167, 128, False), (False, 1, False)),
    ((9, 12, 12, 161, 256, False), (False, 1, False)),
    ((1, 1, 1, 2, 128, True), (True, 1, False)),  # two rows (with one, dQ and dK are zero up to rounding)
]


@pytest.mark.parametrize("shape,plan", CASES)
def test_plans_match_oracle(shape, plan):
    import fa_p100
    assert bwd_plan(*shape) == plan
    B, Hq, Hkv, N, D, causal = shape
    q, k, v, do = make_inputs(B, Hq, Hkv, N, D, seed=N + D)
    qg, kg, vg = (t.to(DEV).requires_grad_(True) for t in (q, k, v))
    o = fa_p100.flash_attn(qg, kg, vg, causal)
    grads = torch.autograd.grad(o, (qg, kg, vg), do.to(DEV), retain_graph=True)
    again = torch.autograd.grad(o, (qg, kg, vg), do.to(DEV))
    G = Hq // Hkv
    b = B - 1  # one batch entry and its last kv head's group
    sq, sk = (slice(b, B), slice(Hq - G, Hq)), (slice(b, B), slice(Hkv - 1, Hkv))
    args = [np64(t) for t in (q[sq], k[sk], v[sk])]
    ref = ora.attention_bwd(*args, np64(do[sq]), causal)
    assert ora.max_abs(np64(o[sq]), ora.attention_fwd(*args, causal)[0]) <= FWD_MAX_ABS
    for name, g, r, s in zip(("dQ", "dK", "dV"), grads, ref, (sq, sk, sk)):
        g = np64(g[s])
        assert np.isfinite(g).all(), name
        assert ora.rel_max_rms(g, r) < REF_REL if np.any(r) else not np.any(g), name
        if np.any(r):
            assert ora.rel_l2(g, r) <= GRAD_REL_L2, name
    for g, h in zip(grads, again):  # the parts are added in one order
        assert torch.equal(g, h)


def test_key_tiles_past_every_key_length_have_zero_gradients():
    """Key tiles wholly past an entry's key length run no step; their dK, dV
    are written as zeros, in every plan."""
    import fa_p100
    B, H, N, D = 2, 2, 640, 64
    q, k, v, do = (t.to(DEV) for t in make_inputs(B, H, H, N, D, seed=3))
    kv_len = torch.tensor([130, 640], dtype=torch.int32, device=DEV)
    for causal in (False, True):
        leaves = [t.clone().requires_grad_(True) for t in (q, k, v)]
        fa_p100.flash_attn(*leaves, causal, kv_len=kv_len).backward(do)
        for g in (leaves[1].grad, leaves[2].grad):
            assert torch.isfinite(g).all() and not g[0, :, 130:].any()
            assert g[0, :, :130].any() and g[1, :, 512:].any()


@pytest.mark.parametrize("shape,plan", CASES)
def test_nothing_unwritten_is_read(shape, plan):
    """Workspace and outputs full of NaN before the call: the results of zeros
    there, bit for bit, so that every value read was written and every element
    of the outputs is."""
    lib = load_capi()
    B, Hq, Hkv, N, D, causal = shape
    q, k, v, do = (t.to(DEV) for t in make_inputs(B, Hq, Hkv, N, D, seed=4))
    o, lse = torch.empty_like(q), torch.empty(B, Hq, N, device=DEV)
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    args = (B, Hq, Hkv, N, D, int(causal))
    assert lib.fa_fwd(*map(p, (q, k, v, o, lse)), *args, 0, s) == 0
    size = lib.fa_bwd_workspace_bytes(*args[:5])
    results = []
    for fill in (0.0, float("nan")):
        ws = torch.full((size // 4,), fill, device=DEV)
        out = [torch.full_like(t, fill) for t in (q, k, v)]
        assert lib.fa_bwd_half_dq(*map(p, (q, k, v, do, o, lse, *out, ws)), size, *args, s) == 0
        results.append(out)
    for a, b in zip(*results):
        assert torch.isfinite(b).all() and torch.equal(a, b)


@pytest.mark.parametrize("Hq,Hkv,N,D,causal", [
    (16, 1, 500, 64, True), (16, 1, 900, 128, False), (4, 2, 300, 256, True),
    (32, 4, 1024, 64, True)])
def test_a_workspace_of_the_pairs_slots_is_enough(Hq, Hkv, N, D, causal):
    """A workspace that ends after two slots per pair of key tiles is taken: the
    same gradients up to the order of their sums, no byte past it touched; one
    byte less is refused."""
    lib = load_capi()
    q, k, v, do = (t.to(DEV) for t in make_inputs(1, Hq, Hkv, N, D, seed=7))
    o, lse = torch.empty_like(q), torch.empty(1, Hq, N, device=DEV)
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    shape = (1, Hq, Hkv, N, D, int(causal))
    assert lib.fa_fwd(*map(p, (q, k, v, o, lse)), *shape, 0, s) == 0
    a256 = lambda n: (n + 255) // 256 * 256
    pairs = -(-N // 128) // 2
    width = next(w for w in (32, 64, 96, 128, 256) if D <= w)
    small = 2 * a256(Hq * N * 4) + a256(Hq * pairs * 4) + Hkv * pairs * 2 * 128 * width * 2 * 4
    full = lib.fa_bwd_workspace_bytes(*shape[:5])
    assert small < full
    grads = []
    for size in (full, small):
        ws = torch.full((full // 4 + 64,), float("nan"), device=DEV)
        out = [torch.full_like(t, float("nan")) for t in (q, k, v)]
        args = [*map(p, (q, k, v, do, o, lse, *out)), p(ws)]
        assert lib.fa_bwd_half_dq(*args, size, *shape, s) == 0
        assert torch.isnan(ws[size // 4:]).all()
        grads.append(out)
    assert lib.fa_bwd_half_dq(*args, small - 1, *shape, s) == 10006
    for x, y in zip(*grads):
        assert torch.isfinite(x).all()
        # (fp32 sums in another order, rounded to 16 bits: an ulp here and there)
        assert ((x.float() - y.float()).norm() / x.float().norm()).item() <= 2 ** -11
