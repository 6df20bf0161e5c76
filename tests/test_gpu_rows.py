"""The forward whose waves own 32 rows each (csrc/fa_rows.hip): 4 and 8 waves,
long and short causal tiles paired, key ranges shared by workgroups, each at
shapes whose plan takes it (fwd_plan, csrc/fa_launch.hip), with ragged tiles,
key lengths, windows and packed sequences; one (batch, head) slice against the
float64 oracle (flash_fwd.cuh:321-339 is the result it restates)."""
import numpy as np
import pytest
import torch

from helpers import FWD_MAX_ABS, LSE_MAX_ABS, np64
from oracle import attention as ora

pytestmark = pytest.mark.gpu

DEV = "cuda"

CASES = [
    # B, Hq, Hkv, N, Nk, D, causal
    (2, 4, 2, 264, 264, 80, True),      # 4 waves, a last tile of 8 rows
    (8, 4, 1, 257, 257, 256, True),     # ... of one row
    (10, 8, 2, 145, 145, 128, False),   # keys past N masked
    (14, 12, 12, 189, 189, 64, True),
    (12, 8, 2, 321, 321, 32, True),
    (7, 12, 12, 589, 589, 128, False),  # 8 waves
    (6, 8, 8, 1114, 1114, 256, True),   # 8 waves
    (4, 8, 8, 3634, 3634, 64, True),    # paired tiles, an odd number of them
    (8, 4, 4, 3032, 3032, 128, True),   # paired tiles
    (1, 8, 1, 1188, 5122, 128, True),   # parts
    (1, 4, 1, 1474, 3529, 256, True),   # parts
]


def make(B, Hq, Hkv, N, Nk, D, seed, dtype=torch.half):
    g = torch.Generator().manual_seed(seed)
    shapes = ((B, Hq, N, D), (B, Hkv, Nk, D), (B, Hkv, Nk, D))
    return [torch.randn(s, generator=g).to(dtype) for s in shapes]


def check(o, lse, q, k, v, causal, b, h, bf16=False, **kw):
    Hq, Hkv = q.size(1), k.size(1)
    g = h // (Hq // Hkv)
    args = [np64(t[b:b + 1, i:i + 1]) for t, i in ((q, h), (k, g), (v, g))]
    ref_o, ref_lse = ora.attention_fwd(*args, causal, **kw)
    assert ora.max_abs(np64(o[b:b + 1, h:h + 1]), ref_o) <= (2.5e-2 if bf16 else FWD_MAX_ABS)
    got, fin = np64(lse[b:b + 1, h:h + 1]), np.isfinite(ref_lse)
    assert np.array_equal(np.isfinite(got), fin)
    assert ora.max_abs(got[fin], ref_lse[fin]) <= LSE_MAX_ABS


@pytest.mark.parametrize("dtype", [torch.half, torch.bfloat16])
@pytest.mark.parametrize("B,Hq,Hkv,N,Nk,D,causal", CASES)
def test_rows_match_oracle(B, Hq, Hkv, N, Nk, D, causal, dtype):
    import fa_p100
    q, k, v = make(B, Hq, Hkv, N, Nk, D, seed=N + D, dtype=dtype)
    dense = [t.to(DEV) for t in (q, k, v)]
    o, lse = fa_p100._ext.forward_dt(*dense, causal)
    assert torch.isfinite(o).all() and torch.isfinite(lse).all()
    for b, h in ((0, 0), (B - 1, Hq - 1)):
        check(o, lse, q, k, v, causal, b, h, dtype == torch.bfloat16)
    ob, lse_b = fa_p100._ext.forward_bnhd(*(t.transpose(1, 2).contiguous() for t in dense), causal)
    assert torch.equal(ob.transpose(1, 2), o) and torch.equal(lse_b, lse)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("option", ["kv_len", "window", "segments"])
def test_rows_bounds(option, causal):
    """Lengths of one key and up; windows narrower than a stage; sequences of
    one token, at a stage's edge and over several tiles."""
    import fa_p100
    B, Hq, Hkv, N, D = 3, 8, 2, 517, 64
    q, k, v = make(B, Hq, Hkv, N, N, D, seed=8)
    kw, okw = {}, {}
    if option == "kv_len":
        lens = [1, 64, 300]
        kw["kv_len"] = torch.tensor(lens, dtype=torch.int32, device=DEV)
        okw = [dict(kv_len=[n]) for n in lens]
    elif option == "window":
        if not causal:
            pytest.skip("windows need causal masking")
        kw["window"] = 37
        okw = [dict(window=37)] * B
    else:
        cuts = [[1, 64, 192, 200, 517], [517], [130, 131, 400, 517]]
        ids = torch.tensor([[sum(i >= c for c in cs) for i in range(N)] for cs in cuts])
        kw["seg_start"], kw["seg_end"] = fa_p100.segment_bounds(ids.to(DEV))
        okw = [dict(segments=ids[b:b + 1].numpy()) for b in range(B)]
    o, lse = fa_p100._ext.forward_dt(*(t.to(DEV) for t in (q, k, v)), causal, **kw)
    for b in range(B):
        check(o, lse, q, k, v, causal, b, Hq - 1, **okw[b])
