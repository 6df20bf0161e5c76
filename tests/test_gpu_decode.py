"""The forward over few query rows (csrc/fa_dec.hip): row tiles that hold the
rows of several query heads, keys shared by several workgroups, every width,
both layouts and formats, key lengths, windows and ALiBi, at the edges of the
32-row tiles and 32-key blocks, against the float64 oracle; and the C ABI's
fa_fwd_ws. No counterpart in the reference (fa_p100.py:48-55 has one row count)."""
import ctypes

import numpy as np
import pytest
import torch

from helpers import FWD_MAX_ABS, LSE_MAX_ABS, fa_opts, fwd_plan, load_capi, np64
from oracle import attention as ora

pytestmark = pytest.mark.gpu

DEV = "cuda"

# B, Hq, Hkv, N, Nk, D, causal: parts (fwd_plan)
CASES = [
    ((1, 16, 8, 1, 1021, 128, True), 1),
    ((1, 8, 2, 1, 4097, 128, True), 24),    # a block of one key
    ((2, 8, 1, 4, 3000, 64, True), 12),     # 32 rows of eight heads
    ((1, 8, 1, 5, 2049, 64, False), 12),    # 40 rows: a head across two tiles
    ((1, 4, 4, 33, 1500, 96, True), 6),     # 33 rows of one head
    ((2, 4, 2, 3, 2500, 256, True), 12),    # four waves
    ((1, 2, 1, 2, 1100, 40, True), 1),      # a head dim below its width
    ((3, 1, 1, 1, 2, 128, True), 1),        # two keys: most waves have no block
    ((1, 2, 2, 1, 700, 32, False), 1),
]


def inputs(B, Hq, Hkv, N, Nk, D, seed, dtype=torch.half):
    g = torch.Generator().manual_seed(seed)
    shapes = ((B, Hq, N, D), (B, Hkv, Nk, D), (B, Hkv, Nk, D))
    return [torch.randn(s, generator=g).to(dtype) for s in shapes]


def check(o, lse, ref, bf16=False):
    ref_o, ref_lse = ref
    assert ora.max_abs(np64(o), ref_o) <= (2.5e-2 if bf16 else FWD_MAX_ABS)
    lse, fin = np64(lse), np.isfinite(ref_lse)
    assert np.array_equal(np.isfinite(lse), fin)
    assert ora.max_abs(lse[fin], ref_lse[fin]) <= LSE_MAX_ABS


@pytest.mark.parametrize("dtype", [torch.half, torch.bfloat16])
@pytest.mark.parametrize("shape,parts", CASES)
def test_decode_matches_oracle(shape, parts, dtype):
    import fa_p100
    assert fwd_plan(*shape) == ("dec", 0, False, parts)
    B, Hq, Hkv, N, Nk, D, causal = shape
    q, k, v = inputs(B, Hq, Hkv, N, Nk, D, seed=N + Nk, dtype=dtype)
    ref = ora.attention_fwd(*(t.double().numpy() for t in (q, k, v)), causal)
    dense = [t.to(DEV) for t in (q, k, v)]
    o, lse = fa_p100._ext.forward_dt(*dense, causal)
    check(o, lse, ref, dtype == torch.bfloat16)
    views = [t.transpose(1, 2).contiguous() for t in dense]
    ob, lse_b = fa_p100._ext.forward_bnhd(*views, causal)
    assert torch.equal(ob.transpose(1, 2), o) and torch.equal(lse_b, lse)


@pytest.mark.parametrize("N,Nk,window,parts", [
    (1, 2000, 0, 8), (1, 2000, 300, 1), (6, 1537, 70, 1), (1, 9000, 5000, 12), (6, 9001, 4000, 16)])
def test_decode_with_key_lengths_window_and_alibi(N, Nk, window, parts):
    """Lengths from one key to all; with a window some rows see no key (o = 0,
    lse = +inf); parts past an entry's keys are empty."""
    import fa_p100
    B, Hq, Hkv, D = 4, 8, 2, 64
    assert fwd_plan(B, Hq, Hkv, N, Nk, D, True, kv_len=1, window=window,
                    alibi_slopes=1) == ("dec", 0, False, parts)
    q, k, v = inputs(B, Hq, Hkv, N, Nk, D, seed=Nk)
    lens = [1, 260, Nk - 3, Nk]
    slopes = torch.tensor([2.0 ** (-h - 1) for h in range(Hq)])
    ref = ora.attention_fwd(*(t.double().numpy() for t in (q, k, v)), True, kv_len=lens,
                            window=window or None, alibi=slopes.double().numpy())
    o, lse = fa_p100._ext.forward_dt(
        *(t.to(DEV) for t in (q, k, v)), True,
        torch.tensor(lens, dtype=torch.int32, device=DEV), window, slopes.to(DEV))
    check(o, lse, ref)


def test_capi_workspace():
    """fa_fwd_ws with fa_fwd_workspace_bytes (NaN-filled) equals the op, and
    refuses a smaller one; without one, fa_fwd_ex's result."""
    import fa_p100
    lib = load_capi()
    vp = ctypes.c_void_p
    B, Hq, Hkv, N, Nk, D = 1, 8, 2, 1, 6000, 128
    q, k, v = (t.to(DEV) for t in inputs(B, Hq, Hkv, N, Nk, D, seed=2))
    op = fa_opts(kv_rows=Nk)
    args = (B, Hq, Hkv, N, D, 1)
    size = lib.fa_fwd_workspace_bytes(*args, op)
    assert size > 0 and lib.fa_fwd_workspace_bytes(B, Hq, Hkv, N, D, 1, None) == 0
    ws = torch.full((size // 4,), float("nan"), device=DEV)
    o, lse = torch.empty_like(q), torch.empty(B, Hq, N, device=DEV)
    s = vp(torch.cuda.current_stream().cuda_stream)
    ptrs = [vp(t.data_ptr()) for t in (q, k, v, o, lse)]
    assert lib.fa_fwd_ws(*ptrs, vp(ws.data_ptr()), size - 1, *args, op, s) == 10006
    assert lib.fa_fwd_ws(*ptrs, vp(ws.data_ptr()), size, *args, op, s) == 0
    want, want_lse = fa_p100._ext.forward_dt(q, k, v, True)
    assert torch.equal(o, want) and torch.equal(lse, want_lse)
    assert lib.fa_fwd_ws(*ptrs, None, 0, *args, op, s) == 0
    plain, plain_lse = torch.empty_like(q), torch.empty_like(lse)
    assert lib.fa_fwd_ex(*ptrs[:3], vp(plain.data_ptr()), vp(plain_lse.data_ptr()), *args, op,
                         s) == 0
    assert torch.equal(o, plain) and torch.equal(lse, plain_lse)


def test_decode_under_graph_capture():
    """Captured with its workspace and replayed on new inputs."""
    import fa_p100
    q, k, v = (t.to(DEV) for t in inputs(1, 8, 2, 1, 5000, 128, seed=6))
    fa_p100.flash_attn(q, k, v, True)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        o = fa_p100.flash_attn(q, k, v, True)
    for seed in range(3):
        for t, new in zip((q, k, v), inputs(1, 8, 2, 1, 5000, 128, seed=seed)):
            t.copy_(new)
        graph.replay()
        assert torch.equal(o, fa_p100.flash_attn(q, k, v, True))
