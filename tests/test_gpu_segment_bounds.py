"""segment_bounds' HIP kernel (fa_segment_bounds) against its torch scans, which
CPU ids take: rows around a thread's 4 ids, a wave's 256 and a workgroup's
4096, both id types, ids that are not dense. No counterpart in the reference."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("N", [1, 2, 3, 4, 5, 255, 256, 257, 1024, 4095, 4096, 4097, 9000])
def test_kernel_equals_torch_scans(N, dtype):
    import fa_p100
    g = torch.Generator().manual_seed(N)
    rows = [torch.zeros(N), torch.arange(N)]
    for p in (0.5, 0.01, 0.0003):  # runs of about two, a hundred, thousands
        rows.append((torch.rand(N, generator=g) < p).cumsum(0))
    rows.append(torch.randint(0, 2, (N,), generator=g))  # ids that come again
    ids = torch.stack([r.to(torch.int64) for r in rows])
    if dtype == torch.int64:
        ids = ids * (1 << 32) + 5  # equal low halves are not equal ids
    ids = ids.to(dtype)
    want = fa_p100.segment_bounds(ids)
    strided = ids.t().contiguous().cuda().t()
    for got in (fa_p100.segment_bounds(ids.cuda()), fa_p100.segment_bounds(strided),
                fa_p100.segment_bounds(ids[:1].cuda().expand(3, N))):
        for a, b in zip(got, want):
            rows_b = b if a.size(0) == b.size(0) else b[:1].expand(3, N)
            assert a.dtype == torch.int32 and a.is_contiguous()
            assert torch.equal(a.cpu(), rows_b)


@pytest.mark.parametrize("how", ["jit.trace", "make_fx", "make_fx pre_dispatch", "compile"])
def test_recorded_and_compiled_calls_stay_torch_operators(how):
    """A graph recorded over one packing computes another's bounds; a compiled
    call stays whole."""
    import fa_p100
    from torch.fx.experimental.proxy_tensor import make_fx
    first = (torch.arange(130, device="cuda") // 50).expand(2, 130).contiguous()
    ids = (torch.arange(130, device="cuda") // 30).expand(2, 130).contiguous()
    want = fa_p100.segment_bounds(ids)
    if how == "jit.trace":
        got = torch.jit.trace(fa_p100.segment_bounds, (first,), check_trace=False)(ids)
    elif how == "compile":
        got = torch.compile(fa_p100.segment_bounds, backend="eager", fullgraph=True)(ids)
    else:
        got = make_fx(fa_p100.segment_bounds, pre_dispatch=how.endswith("dispatch"))(first)(ids)
    for a, b in zip(got, want):
        assert torch.equal(a, b)
