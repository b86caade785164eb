"""Calls that something else watches -- forward-mode derivatives, function transforms, tracers -- do not take the short ways
that go to the kernels behind torch's back."""
import pytest
import torch
import torch.autograd.forward_ad as fwd_ad
from torch.utils._python_dispatch import TorchDispatchMode

from analog_moe_amd import ffn, moe_layer
from tests import util
from tests.test_emu_kernels import emu_ops  # noqa: F401


def call(pr, x):
    return ffn.moe_ffn(x, pr["keys"], pr["values"], None, pr["gate"], pr["idx"], ffn.FFNConfig(inp_res=-1.0))


@pytest.fixture
def pr():
    return util.make_problem(7, T=10, D=32, E=3, F=24, k=2)


def test_forward_mode_derivative_is_refused_not_dropped(emu_ops, pr):
    with torch.no_grad(), fwd_ad.dual_level():
        with pytest.raises(NotImplementedError):
            call(pr, fwd_ad.make_dual(pr["x"], torch.ones_like(pr["x"])))
    with torch.no_grad():
        assert torch.equal(call(pr, pr["x"]), ffn.ffn_forward(pr["x"], pr["keys"], pr["values"], None, pr["gate"], pr["idx"],
                                                             ffn.FFNConfig(inp_res=-1.0))[0])


def test_function_transforms_are_refused(emu_ops, pr):
    with torch.no_grad(), pytest.raises(RuntimeError):
        torch.func.vmap(lambda x: call(pr, x))(pr["x"][None])


def test_a_trace_computes_anew(emu_ops, pr):
    with torch.no_grad():
        traced = torch.jit.trace(lambda x: call(pr, x), (pr["x"],), check_trace=False)
        other = pr["x"].flip(0).contiguous()
        assert torch.equal(traced(other), call(pr, other))


def test_the_router_sees_who_watches():
    x = torch.zeros(2, 3)
    seen = []
    assert moe_layer._plain(x) and not moe_layer._plain(x.as_subclass(type("Sub", (torch.Tensor,), {})))
    with fwd_ad.dual_level():
        assert not moe_layer._plain(x)
    torch.func.vmap(lambda t: (seen.append(moe_layer._plain(t)), t)[1])(x)
    torch.jit.trace(lambda t: (seen.append(moe_layer._plain(t)), t + 1)[1], (x,), check_trace=False)

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))
    with Mode():
        seen.append(moe_layer._plain(x))
    assert seen == [False, False, False]


@pytest.mark.gpu
def test_layer_in_eval_mode_refuses_a_dual_tensor():
    from analog_moe_amd import config as rpu
    with torch.device("cuda"):
        layer = moe_layer.AnalogSigmaMoELayer(rpu.TorchInferenceRPUConfig(), d_model=64, n_experts=4, expert_size=64, k=2).eval()
    x = torch.randn(1, 9, 64, device="cuda")
    with torch.no_grad(), fwd_ad.dual_level(), pytest.raises(NotImplementedError):
        layer(fwd_ad.make_dual(x, torch.ones_like(x)))
