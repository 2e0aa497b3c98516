"""_ops.run_function: a Function's forward alone where gradients are off, and
apply wherever something records, transforms or refuses the call."""
import pytest
import torch
from torch.autograd import forward_ad

from uttt_amd._ops import run_function

CTX = []


class _Double(torch.autograd.Function):
    @staticmethod
    @torch.amp.custom_fwd(cast_inputs=torch.bfloat16, device_type="cpu")
    def forward(ctx, x, n):
        CTX.append(type(ctx).__name__)
        ctx.save_for_backward(x)
        ctx.n = n
        ctx.mark_non_differentiable(n)
        return x * 2, n

    @staticmethod
    def backward(ctx, g, _):
        assert ctx.saved_tensors[0].shape == g.shape
        return g * 2, None


def _run(x):
    CTX.clear()
    out, n = run_function(_Double, x, torch.zeros(1, dtype=torch.int32))
    return out, CTX[0]


def test_routes():
    x = torch.randn(3, requires_grad=True)
    out, ctx = _run(x)
    assert ctx == "_DoubleBackward" and torch.autograd.grad(out.sum(), x)[0].eq(2).all()
    with torch.no_grad():
        out, ctx = _run(x)
        assert ctx == "_NoGraph" and not out.requires_grad and torch.equal(out, x.detach() * 2)
        with torch.autocast("cpu", dtype=torch.bfloat16):
            out, ctx = _run(x)
            assert ctx == "_NoGraph" and out.dtype == torch.bfloat16
        out = torch.jit.trace(lambda t: run_function(_Double, t, torch.zeros(1))[0], x,
                              check_trace=False)
        assert "Double" in str(out.graph)
    with torch.inference_mode():
        assert _run(x)[1] == "_NoGraph"


@pytest.mark.parametrize("grad", [False, True])
def test_a_given_row_map_comes_out_as_an_alias(grad, monkeypatch):
    """As Function.apply returns it: metadata of its own, the same storage."""
    from uttt_amd.lact_moe_triton import triton_permute as tp

    monkeypatch.setattr(tp, "triton_permute_with_mask_map",
                        lambda x, *a: (x.repeat(1, 2, 1), None))
    x, mask = torch.randn(1, 4, 8, requires_grad=True), torch.ones(1, 2, 4, dtype=torch.bool)
    rm = torch.zeros(1, 4, 5, dtype=torch.int32)
    with torch.set_grad_enabled(grad):
        out = tp.permute_with_expert_mask(x, mask, None, 2, rm)[2]
    assert out is not rm and out.data_ptr() == rm.data_ptr()
    out.unsqueeze_(0)
    assert rm.shape == (1, 4, 5)


class _Address(torch.autograd.Function):
    """Takes the storage's address, as every C call does."""

    @staticmethod
    def forward(ctx, x):
        return x + (0 if x.data_ptr() else 1)

    @staticmethod
    def backward(ctx, g):
        return g


def test_a_tensor_that_outlived_its_transform():
    kept = []

    def loss(x):
        kept.append(x * 2)
        return kept[0].sum()

    x = torch.randn(3)
    torch.func.grad(loss)(x)
    with torch.no_grad():
        assert torch.equal(run_function(_Address, kept[0]), x * 2)


def test_transforms_take_apply():
    with torch.no_grad():
        with pytest.raises(RuntimeError, match="setup_context|vmap"):
            torch.vmap(lambda t: _run(t)[0])(torch.randn(2, 3))
        with forward_ad.dual_level():
            x = forward_ad.make_dual(torch.randn(3), torch.randn(3))
            CTX.clear()
            with torch.autograd.forward_ad._set_fwd_grad_enabled(True):
                with pytest.raises(RuntimeError, match="jvp|forward"):
                    run_function(_Double, x, torch.zeros(1, dtype=torch.int32))
            assert CTX == ["_DoubleBackward"]
