"""The native host path (csrc/torch_front.cpp) against the Python autograd Functions it stands in for: same library calls,
so every result is bit for bit the same; and the calls it leaves to them."""
import pytest
import torch
import torch.utils.checkpoint

from flash_trittention import TrittentionTriton, _lib, flash_trittention
from flash_trittention.dot_product_sum.trittention_triton import TrittentionTritonFunction
from flash_trittention.triple_dot_product.flash_trittention import FlashTrittention

pytestmark = pytest.mark.gpu


def make(dtype, fused, B=2, H=3, T=70, D=32):
    g = torch.Generator(device="cuda").manual_seed(3)
    if fused:
        x = torch.randn(B, T, 6, H, D, generator=g, device="cuda").to(dtype)
        return [x[:, :, i].transpose(1, 2) for i in range(6)]
    return [torch.randn(B, H, T, D, generator=g, device="cuda").to(dtype) for _ in range(6)]


def leaves(tensors, wanted):
    return [t.detach().requires_grad_(bool(w)) for t, w in zip(tensors, wanted)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("convert", [False, True])
@pytest.mark.parametrize("wanted", [(1, 1, 1, 1, 1), (0, 1, 0, 0, 1)])
def test_native_path_equals_the_functions(dtype, fused, convert, wanted):
    print(f"case native {dtype} fused={fused} convert={convert} {wanted}", flush=True)
    *ins, grad = make(dtype, fused)
    a, b = leaves(ins, wanted), leaves(ins, wanted)
    window = (24, None, 9, 2**40)  # k1_window, k2_window, kk_left, kk_right
    out = flash_trittention(*a, softmax_scale=0.2, k1_window=window[0], k2_window=window[1], kk_left=window[2],
                            kk_right=window[3], convert_to_float32=convert)
    assert "Flash" not in type(out.grad_fn).__name__  # not the Python Function's node
    ref = FlashTrittention.apply(*b, 0.2, window[2], window[3], window[0], window[1], True, convert)
    assert torch.equal(out, ref)
    pick = lambda ts: [t for t in ts if t.requires_grad]
    for x, y in zip(torch.autograd.grad(out, pick(a), grad), torch.autograd.grad(ref, pick(b), grad)):
        assert torch.equal(x, y)

    a, b = leaves(ins, wanted), leaves(ins, wanted)
    out, m = TrittentionTriton(softmax_scale=0.2, k_diff=40, convert_to_float32=convert)(*a)
    ref, m_ref = TrittentionTritonFunction.apply(*b, True, 0.2, 40, convert)
    assert torch.equal(out, ref) and torch.equal(m, m_ref) and not m.requires_grad
    for x, y in zip(torch.autograd.grad(out, pick(a), grad), torch.autograd.grad(ref, pick(b), grad)):
        assert torch.equal(x, y)


def test_native_path_without_a_graph_and_on_another_stream():
    *ins, _ = make(torch.bfloat16, False)
    with torch.no_grad():
        want = flash_trittention(*leaves(ins, (1,) * 5), k1_window=None, k2_window=None, kk_left=None, kk_right=None)
    assert not want.requires_grad
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        got = flash_trittention(*ins, k1_window=None, k2_window=None, kk_left=None, kk_right=None)
    torch.cuda.current_stream().wait_stream(side)
    assert torch.equal(want, got)


def test_calls_the_native_path_leaves_to_the_functions():
    *ins, grad = make(torch.bfloat16, False)
    native = _lib.native()
    none = (None,) * 4
    assert native.tdp(*(t.cpu() for t in ins), 0.1, *none, True, False) is None
    assert native.tdp(*ins[:4], ins[4][:, :, 1:], 0.1, *none, True, False) is None
    assert native.tdp(*ins[:4], ins[4].float(), 0.1, *none, True, False) is None
    assert native.tdp(*ins, 0.1, None, None, None, -1, True, False) is None
    assert native.dps(*ins, True, 0.1, -3, False) is None
    with pytest.raises(ValueError):
        flash_trittention(*ins, k2_window=-1)
    with pytest.raises(ValueError):
        flash_trittention(*ins[:4], ins[4].float())
    # a view the library cannot read (strided last dimension) is copied, as the Functions do
    odd = [torch.stack((t, t), -1)[..., 0] for t in ins]
    full = dict(k1_window=None, k2_window=None, kk_left=None, kk_right=None)
    assert torch.equal(flash_trittention(*odd, **full), flash_trittention(*ins, **full))


def test_native_backward_takes_another_dtype_and_refuses_changed_inputs():
    *ins, grad = make(torch.bfloat16, False)
    a = leaves(ins, (1,) * 5)
    full = dict(k1_window=None, k2_window=None, kk_left=None, kk_right=None)
    out = flash_trittention(*a, **full)
    want = torch.autograd.grad(out, a, grad, retain_graph=True)
    assert all(torch.equal(x, y) for x, y in zip(want, torch.autograd.grad(out, a, grad, retain_graph=True)))
    with torch.no_grad():
        a[1].add_(1)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        torch.autograd.grad(out, a, grad)


FULL = dict(k1_window=None, k2_window=None, kk_left=None, kk_right=None)


def test_native_path_leaves_transforms_traces_and_tangents_to_the_functions():
    *ins, _ = make(torch.float32, False)
    native = _lib.native()
    call = lambda *t: native.tdp(*t, 0.1, None, None, None, None, True, False)
    assert call(*ins) is not None

    class Tagged(torch.Tensor):
        pass

    assert call(ins[0].as_subclass(Tagged), *ins[1:]) is None
    assert call(torch.nn.Parameter(ins[0]), *ins[1:]) is not None
    seen = []

    def under(x):  # nothing of the call is wrapped, the transform is active all the same
        seen.append(call(*ins))
        return x

    torch.func.vmap(under)(torch.zeros(3))
    assert seen == [None]
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(ins[0], torch.ones_like(ins[0]))
        assert call(dual, *ins[1:]) is None
    traced = torch.jit.trace(lambda *t: flash_trittention(*t, **FULL), tuple(ins), check_trace=False)
    other = [t.flip(2).contiguous() for t in ins]
    assert torch.equal(traced(*other), flash_trittention(*other, **FULL))  # recorded, not a constant


def test_native_path_under_saved_tensor_hooks():
    """Hooks that move the saved tensors away and back, one that brings them back in another layout, and recomputation
    (checkpoint stops it with an exception out of a hook)."""
    *ins, grad = make(torch.bfloat16, False)
    a = leaves(ins, (1,) * 5)
    want = torch.autograd.grad(flash_trittention(*a, **FULL), a, grad)

    def other_layout(t):
        big = torch.empty(t.numel() * 2 + 1, dtype=t.dtype, device=t.device)[1:]
        wide = big.view(*t.shape, 2)[..., 0]
        wide.copy_(t)
        return wide

    for pack, unpack in ((lambda t: t.cpu(), lambda t: t.cuda()), (other_layout, lambda t: t)):
        with torch.autograd.graph.saved_tensors_hooks(pack, unpack):
            out = flash_trittention(*a, **FULL)
            o2, _ = TrittentionTriton(softmax_scale=0.2, k_diff=40)(*a)
        assert all(torch.equal(x, y) for x, y in zip(want, torch.autograd.grad(out, a, grad)))
        ref, _ = TrittentionTriton(softmax_scale=0.2, k_diff=40)(*a)
        assert all(torch.equal(x, y) for x, y in
                   zip(torch.autograd.grad(o2, a, grad), torch.autograd.grad(ref, a, grad)))
    out = torch.utils.checkpoint.checkpoint(lambda *t: flash_trittention(*t, **FULL) * 1, *a, use_reentrant=False)
    assert all(torch.equal(x, y) for x, y in zip(want, torch.autograd.grad(out, a, grad)))

    class Stop(Exception):
        pass

    def stop(t):
        raise Stop

    with pytest.raises(Stop), torch.autograd.graph.saved_tensors_hooks(stop, lambda t: t):
        flash_trittention(*a, **FULL)


def test_native_path_arguments_without_a_truth_value():
    *ins, _ = make(torch.bfloat16, False)
    with pytest.raises(RuntimeError, match="ambiguous"):
        flash_trittention(*ins, causal=torch.ones(2), **FULL)
    with pytest.raises(RuntimeError, match="ambiguous"):
        flash_trittention(*ins, convert_to_float32=torch.ones(2), **FULL)


def test_kernels_switched_between_a_keeping_forward_and_its_backward(tune):
    *ins, grad = make(torch.float32, False)
    a = leaves(ins, (1,) * 5)
    out, _ = TrittentionTriton(softmax_scale=0.2, k_diff=40)(*a)
    want = torch.autograd.grad(out, a, grad, retain_graph=True)
    tune(_lib.TUNE_F32_VALU, 1)
    for x, y in zip(torch.autograd.grad(out, a, grad), want):
        torch.testing.assert_close(x, y, rtol=1e-4, atol=2e-5)
