"""flash_attn's autograd Function in C++ (fa_p100_ext.flash_attn) against the
Python one it stands in for (fa_p100.py:31-45): the same outputs and gradients
bit for bit in both layouts, the same saved tensors seen by saved-tensor hooks,
and the same refusals under functorch and forward-mode differentiation."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


def leaves(layout, dtype=torch.half, B=2, Hq=4, Hkv=2, N=130, D=64, seed=0):
    g = torch.Generator().manual_seed(seed)
    out = []
    for h in (Hq, Hkv, Hkv, Hq):
        t = torch.randn(B, N, h, D, generator=g).to(dtype).to(DEV).transpose(1, 2)
        out.append(t if layout == "bnhd" else t.contiguous())
    return [t.detach().requires_grad_(i < 3) for i, t in enumerate(out)]


OPTIONS = {
    "plain": {},
    "kv_len": dict(kv_len=torch.tensor([100, 130], dtype=torch.int32)),
    "window": dict(window=40),
    "alibi": dict(alibi=torch.tensor([0.5, 0.25, 0.125, 0.06])),
    "scale": dict(scale=0.2),
}


@pytest.mark.parametrize("dtype", [torch.half, torch.bfloat16])
@pytest.mark.parametrize("layout", ["bhnd", "bnhd", "mixed"])
@pytest.mark.parametrize("option", list(OPTIONS) + ["segments"])
def test_equals_the_python_function(option, layout, dtype):
    import fa_p100
    q, k, v, do = leaves("bnhd" if layout == "mixed" else layout, dtype)
    if layout == "mixed":  # q a view, k dense: the dense path's copies
        k = k.detach().contiguous().requires_grad_()
    if option == "segments":
        ids = (torch.arange(130) // 50).expand(2, 130).to(DEV)
        public = dict(segment_ids=ids)
        args = dict(segs=fa_p100.segment_bounds(ids))
    else:
        args = {n: t.to(DEV) if torch.is_tensor(t) else t for n, t in OPTIONS[option].items()}
        names = dict(kv_len="kv_len", window="sliding_window", alibi="alibi_slopes",
                     scale="softmax_scale")
        public = {names[n]: t for n, t in args.items()}
    o = fa_p100.flash_attn(q, k, v, True, **public)
    a = [args.get(n, d) for n, d in (("kv_len", None), ("window", 0), ("alibi", None),
                                     ("segs", None), ("scale", 0.0))]
    o_py = fa_p100._FlashAttnP100.apply(q, k, v, True, False, *a, None, None, None, None)
    assert torch.equal(o, o_py) and o.stride() == o_py.stride()
    for x, y in zip(torch.autograd.grad(o, (q, k, v), do),
                    torch.autograd.grad(o_py, (q, k, v), do)):
        assert torch.equal(x, y) and x.stride() == y.stride() and x.dtype == y.dtype


@pytest.mark.parametrize("layout", ["bhnd", "bnhd"])
def test_saved_tensor_hooks_see_what_is_saved(layout):
    import fa_p100
    q, k, v, do = leaves(layout)
    packed = []

    def pack(t):
        packed.append((tuple(t.shape), t.dtype))
        return t.cpu()

    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.to(DEV)):
        o = fa_p100.flash_attn(q, k, v, True)
    first, packed = packed, []
    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.to(DEV)):
        o_py = fa_p100._FlashAttnP100.apply(q, k, v, True, False)
    assert first == packed and len(first) == 5
    for x, y in zip(torch.autograd.grad(o, (q, k, v), do),
                    torch.autograd.grad(o_py, (q, k, v), do)):
        assert torch.equal(x, y)


def test_refusals_and_modes():
    import fa_p100
    q, k, v, do = leaves("bhnd")
    with pytest.raises(RuntimeError):
        torch.func.vmap(lambda x: fa_p100.flash_attn(x, k, v, True))(q[None])
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda x: fa_p100.flash_attn(x, k, v, True).float().sum())(q)
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(q.detach(), torch.ones_like(q))
        with pytest.raises(RuntimeError):
            fa_p100.flash_attn(dual, k, v, True)
    with torch.no_grad():
        assert not fa_p100.flash_attn(q, k, v, True).requires_grad
    o = fa_p100.flash_attn(q, k.detach(), v.detach(), True)  # only q needs a gradient
    (dq,) = torch.autograd.grad(o, q, do, retain_graph=True)
    assert torch.equal(dq, torch.autograd.grad(o, q, do)[0])
    o = fa_p100.flash_attn(q, k, v, True)
    grads = torch.autograd.grad(o, (q, k, v), do, create_graph=True)
    assert not any(g.requires_grad for g in grads)  # as the Python Function's
    with torch.no_grad():
        k.add_(1)  # saved for the backward
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        torch.autograd.grad(fa_p100_out(q, k, v), (q,), do)


def fa_p100_out(q, k, v):
    import fa_p100
    o = fa_p100.flash_attn(q, k, v, True)
    with torch.no_grad():
        k.add_(1)
    return o


@pytest.mark.parametrize("layout", ["bhnd", "bnhd"])
def test_a_traced_call_runs_again_on_new_inputs(layout):
    """torch.jit.trace records the Python Function as a node: the traced module
    computes new inputs' outputs and their gradients."""
    import fa_p100
    first, (q, k, v, do) = leaves(layout, seed=1), leaves(layout, seed=2)
    traced = torch.jit.trace(lambda q, k, v: fa_p100.flash_attn(q, k, v, True),
                             tuple(t.detach() for t in first[:3]), check_trace=False)
    o, want = traced(q, k, v), fa_p100.flash_attn(q, k, v, True)
    assert torch.equal(o, want)
    for x, y in zip(torch.autograd.grad(o, (q, k, v), do),
                    torch.autograd.grad(want, (q, k, v), do)):
        assert torch.equal(x, y)


def test_gradients_on_a_side_stream_and_from_threads():
    import threading

    import fa_p100
    q, k, v, do = leaves("bhnd", N=700)
    want = torch.autograd.grad(fa_p100.flash_attn(q, k, v, True), (q, k, v), do)
    torch.cuda.synchronize()
    results = [None] * 4

    def work(i):
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            for _ in range(3):
                results[i] = torch.autograd.grad(fa_p100.flash_attn(q, k, v, True), (q, k, v), do)
        s.synchronize()

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for r in results:
        for x, y in zip(r, want):
            assert torch.equal(x, y)
