"""The forward whose waves own 32 rows each (csrc/fa_rows.hip): 4 and 8 waves,
long and short causal tiles paired, key ranges shared by workgroups, each at
shapes whose plan takes it (asserted: fa_fwd_plan), with ragged tiles,
key lengths, windows and packed sequences; one (batch, head) slice against the
float64 oracle (flash_fwd.cuh:321-339 is the result it restates)."""
import numpy as np
import pytest
import torch

from helpers import FWD_MAX_ABS, LSE_MAX_ABS, fwd_plan, np64
from oracle import attention as ora

pytestmark = pytest.mark.gpu

DEV = "cuda"

# B, Hq, Hkv, N, Nk, D, causal: waves, paired, parts (fwd_plan)
CASES = [
    ((2, 4, 2, 264, 264, 80, True), (4, False, 1)),  # a last tile of 8 rows
    ((8, 4, 1, 257, 257, 256, True), (4, False, 1)),  # ... of one row
    ((10, 8, 2, 145, 145, 128, False), (4, False, 1)),  # keys past N masked
    ((7, 12, 12, 589, 589, 128, False), (4, False, 1)),
    ((1, 2, 2, 138, 138, 256, False), (4, False, 1)),
    ((14, 12, 12, 189, 189, 64, True), (8, False, 1)),
    ((12, 8, 2, 321, 321, 32, True), (8, False, 1)),
    ((11, 12, 12, 398, 398, 80, True), (8, False, 1)),
    ((16, 16, 8, 169, 169, 128, True), (8, False, 1)),
    ((11, 16, 8, 132, 132, 256, True), (8, False, 1)),
    ((12, 12, 12, 133, 133, 32, False), (8, False, 1)),
    ((3, 48, 12, 130, 130, 64, False), (8, False, 1)),
    ((13, 12, 12, 129, 129, 256, False), (8, False, 1)),
    ((10, 12, 12, 340, 340, 32, True), (4, True, 1)),
    ((4, 8, 8, 3634, 3634, 64, True), (4, True, 1)),  # an odd number of tiles
    ((13, 4, 2, 514, 514, 96, True), (4, True, 1)),
    ((9, 48, 12, 136, 136, 128, True), (4, True, 1)),
    ((6, 8, 8, 1114, 1114, 256, True), (4, True, 1)),
    ((1, 8, 1, 1188, 5122, 128, True), (4, False, 3)),
    ((3, 1, 1, 968, 4668, 96, False), (4, False, 8)),
    ((6, 4, 4, 680, 3570, 64, False), (8, False, 3)),
    ((3, 16, 8, 188, 4334, 80, True), (8, False, 4)),
    ((1, 8, 2, 1474, 6000, 256, True), (8, False, 4)),
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
@pytest.mark.parametrize("shape,plan", CASES)
def test_rows_match_oracle(shape, plan, dtype):
    import fa_p100
    assert fwd_plan(*shape) == ("rows", *plan)
    B, Hq, Hkv, N, Nk, D, causal = shape
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
@pytest.mark.parametrize("B,Hq,Hkv,N,D,waves", [
    (4, 8, 2, 517, 64, 4), (3, 48, 12, 136, 64, 8), (12, 16, 4, 140, 256, 8)])
def test_rows_bounds(B, Hq, Hkv, N, D, waves, option, causal):
    """Lengths of one key and up; windows narrower than a stage; sequences of
    one token, at a stage's edge and over several tiles."""
    import fa_p100
    q, k, v = make(B, Hq, Hkv, N, N, D, seed=8)
    kw, okw = {}, {}
    if option == "kv_len":
        lens = [min(N, n) for n in ([1, 64, 300, 129] * B)[:B]]
        kw["kv_len"] = torch.tensor(lens, dtype=torch.int32, device=DEV)
        okw = [dict(kv_len=[n]) for n in lens]
    elif option == "window":
        if not causal:
            pytest.skip("windows need causal masking")
        kw["window"] = 37
        okw = [dict(window=37)] * B
    else:
        cuts = [[1, 64, 192, 200], [], [130, 131, 400]]
        ids = torch.tensor([[sum(i >= c for c in cuts[b % 3]) for i in range(N)] for b in range(B)])
        kw["seg_start"], kw["seg_end"] = fa_p100.segment_bounds(ids.to(DEV))
        okw = [dict(segments=ids[b:b + 1].numpy()) for b in range(B)]
    assert fwd_plan(B, Hq, Hkv, N, N, D, causal, **kw) == ("rows", waves, False, 1)
    o, lse = fa_p100._ext.forward_dt(*(t.to(DEV) for t in (q, k, v)), causal, **kw)
    for b in range(min(B, 4)):
        check(o, lse, q, k, v, causal, b, Hq - 1, **okw[b])


FEAT_CASES = [
    # B, H, N, D, causal: N a multiple of 4 (the bias rows' 16-byte loads), ragged
    # against stages of 64 keys and tiles of 128 rows
    (8, 12, 516, 64, False),
    (8, 12, 516, 64, True),
    (3, 16, 260, 96, True),
    (2, 32, 388, 128, True),
    (12, 8, 132, 32, False),
    (4, 16, 1284, 64, True),  # paired tiles
]


@pytest.mark.parametrize("feature", ["bias", "bias_shared", "dropout", "kv_len"])
@pytest.mark.parametrize("B,H,N,D,causal", FEAT_CASES)
def test_rows_bias_and_dropout(B, H, N, D, causal, feature):
    """A bias per head and one shared by all (rows of one plane through every
    head's loads), -inf and the type's lowest value in it, dropout's keep bits,
    and a bias with key lengths."""
    import fa_p100
    given = dict(drop=1, drop_scale=1.25) if feature == "dropout" else dict(bias=16)
    assert fwd_plan(B, H, H, N, N, D, causal, **given) == ("rows", 4, N == 1284, 1)
    q, k, v = make(B, H, H, N, N, D, seed=N)
    dev = [t.to(DEV) for t in (q, k, v)]
    g = torch.Generator().manual_seed(1)
    slices = ((0, 0), (B - 1, H - 1))
    if feature == "dropout":
        z, _, zs = fa_p100.dropout_bits(77, 0.2, B, H, N, DEV, causal=causal)
        o, lse = fa_p100._ext.forward_dt(*dev, causal, drop=z, drop_scale=zs)
        for b, h in slices:
            words = z[b, h].cpu().numpy().view(np.uint32)
            keep = ((words[:, :, None] >> np.arange(32, dtype=np.uint32)) & 1).astype(bool)
            keep = keep.reshape(N, -1)[None, None, :, :N]
            # (P / (1 - p): the bar scales with it)
            check_drop(o, lse, q, k, v, causal, b, h, (keep, zs))
        return
    shape = (1, 1, N, N) if feature == "bias_shared" else (1, H, N, N)
    bias = torch.randn(shape, generator=g)
    bias[..., 3::7] = -float("inf")  # hidden keys
    bias[..., 1, :] = torch.finfo(torch.float32).min  # a row of the lowest value
    bias[..., 1, 0] = 0.0
    kw, lens = {}, [N] * B
    if feature == "kv_len":
        lens = [max(1, N - 37 * b) for b in range(B)]
        kw["kv_len"] = torch.tensor(lens, dtype=torch.int32, device=DEV)
    o, lse = fa_p100._ext.forward_dt(*dev, causal, bias=bias.to(DEV), **kw)
    for b, h in slices:
        plane = bias[:, h:h + 1] if shape[1] > 1 else bias
        check(o, lse, q, k, v, causal, b, h, bias=np64(plane), kv_len=[lens[b]])


def check_drop(o, lse, q, k, v, causal, b, h, dropout):
    args = [np64(t[b:b + 1, h:h + 1]) for t in (q, k, v)]
    ref_o, ref_lse = ora.attention_fwd(*args, causal, dropout=dropout)
    assert ora.max_abs(np64(o[b:b + 1, h:h + 1]), ref_o) <= FWD_MAX_ABS * dropout[1] ** 2
    assert ora.max_abs(np64(lse[b:b + 1, h:h + 1]), ref_lse) <= LSE_MAX_ABS


@pytest.mark.parametrize("layout", ["bhnd", "bnhd"])
@pytest.mark.parametrize("N", [130, 256])
def test_bias_gradient_is_written_whole(N, layout):
    """Without causal masking, lengths or sequences the backward writes every
    element of the bias's gradient: a buffer of NaN comes back finite."""
    import fa_p100
    q, k, v, do = (torch.randn(2, 4, N, 64, device=DEV).half() for _ in range(4))
    bias = torch.randn(1, 4, N, N, device=DEV)
    dbias = torch.full((2, 4, N, N), float("nan"), device=DEV)
    forward, backward = fa_p100._ext.forward_dt, fa_p100._ext.backward_dt
    args = [q, k, v, do]
    if layout == "bnhd":
        forward, backward = fa_p100._ext.forward_bnhd, fa_p100._ext.backward_bnhd
        args = [t.transpose(1, 2).contiguous() for t in args]
    o, lse = forward(*args[:3], False, bias=bias)
    backward(*args, o, lse, False, bias=bias, dbias=dbias)
    assert torch.isfinite(dbias).all()
    s = (q.float() @ k.float().transpose(-1, -2).contiguous() / 8 + bias)
    p = s.softmax(-1)
    dp = do.float() @ v.float().transpose(-1, -2).contiguous()
    ref = p * (dp - (dp * p).sum(-1, keepdim=True))
    assert ((dbias - ref).norm() / ref.norm()).item() <= 5e-3


@pytest.mark.parametrize("B,H,N,Nk,D,causal,plan", [
    (8, 12, 516, 516, 64, False, (4, False, 1)),
    (8, 12, 517, 517, 128, True, (4, False, 1)),
    (4, 16, 1285, 1285, 64, True, (4, True, 1)),
    (3, 16, 261, 261, 256, True, (4, False, 1)),
    (1, 8, 1188, 5122, 96, True, (4, False, 3)),  # distances from the last key's diagonal
])
def test_rows_alibi(B, H, N, Nk, D, causal, plan):
    import fa_p100
    assert fwd_plan(B, H, H, N, Nk, D, causal, alibi_slopes=1) == ("rows", *plan)
    q, k, v = make(B, H, H, N, Nk, D, seed=N)
    slopes = torch.tensor([2.0 ** (-8.0 * (h + 1) / H) for h in range(H)])
    o, lse = fa_p100._ext.forward_dt(*(t.to(DEV) for t in (q, k, v)), causal,
                                     alibi_slopes=slopes.to(DEV))
    for b, h in ((0, 0), (B - 1, H - 1)):
        check(o, lse, q, k, v, causal, b, h, alibi=slopes[h:h + 1].double().numpy())
