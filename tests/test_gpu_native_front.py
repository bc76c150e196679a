"""The native host path (csrc/torch_front.cpp) against the Python autograd Functions it stands in for: same library calls,
so every result is bit for bit the same; and the calls it leaves to them."""
import pytest
import torch

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
