"""flash_attn_func under torch's own machinery around an autograd function; its node lives in the extension."""
import pytest
import torch
import torch.utils.checkpoint
from torch.autograd import forward_ad

import abi  # noqa: F401  (puts the package on sys.path)
from oracle import attention_oracle as ao


def test_trace_takes_the_recordable_node(monkeypatch):
    """On the CPU, with the extension's functions replaced: a trace holds a call, not a constant."""
    from flash_attn_v100 import flash_attn_interface as interface

    class Stub:
        fwd = staticmethod(lambda q, k, v, out, scale, causal: (torch.from_numpy(q.detach().numpy() * 2), None))
        attention = staticmethod(lambda q, k, v, scale, causal: torch.from_numpy(q.detach().numpy() * 2))

    monkeypatch.setattr(interface, "flash_attn_cuda", Stub)
    q, k, v, _ = ao.make_inputs(1, 8, 1, 64, seed=1)
    traced = torch.jit.trace(lambda a, b, c: interface.flash_attn_func(a, b, c), (q, k, v), check_trace=False)
    assert "FlashAttnFunc" in str(traced.graph)
    assert torch.equal(traced(-q, k, v), q * -2)


@pytest.mark.parametrize("of", ["softmax_scale", "causal"])
def test_trace_keeps_the_inputs_that_options_are(monkeypatch, of):
    """On the CPU, with the extension's functions replaced: a scale or a mask that is an input of the traced function stays
    one, so that a replay takes the new value."""
    from flash_attn_v100 import flash_attn_interface as interface

    class Stub:
        @staticmethod
        def fwd(q, k, v, out, scale, causal):
            return torch.from_numpy(q.detach().numpy() * (float(scale) + 10 * bool(causal))), None

    monkeypatch.setattr(interface, "flash_attn_cuda", Stub)
    q, k, v, _ = ao.make_inputs(1, 8, 1, 64, seed=1)
    q = q.clamp(-1, 1)
    if of == "softmax_scale":
        call, first, then = lambda a, b, c, s: interface.flash_attn_func(a, b, c, s), torch.tensor(2.0), torch.tensor(3.0)
    else:
        call, first, then = lambda a, b, c, s: interface.flash_attn_func(a, b, c, 2.0, s), torch.tensor(False), torch.tensor(True)
    traced = torch.jit.trace(call, (q, k, v, first), check_trace=False)
    assert torch.equal(traced(q, k, v, first), q * 2)
    assert torch.equal(traced(q, k, v, then), q * (3 if of == "softmax_scale" else 12))


def test_the_extension_has_no_function_without_a_caller():
    import flash_attn_v100_cuda

    assert {name for name in dir(flash_attn_v100_cuda) if not name.startswith("_")} == {"attention", "fwd", "bwd"}


@pytest.mark.gpu
def test_trace_of_the_extension():
    from flash_attn_v100 import flash_attn_func

    q, k, v, _ = (t.cuda() for t in ao.make_inputs(1, 70, 2, 64, seed=1))
    with torch.no_grad():
        traced = torch.jit.trace(lambda a, b, c: flash_attn_func(a, b, c, None, True), (q, k, v), check_trace=False)
        assert torch.equal(traced(k, v, q), flash_attn_func(k, v, q, None, True))


@pytest.mark.gpu
@pytest.mark.parametrize("grad_mode", [False, True])
def test_forward_mode_is_refused(grad_mode):
    """There is no derivative in forward mode: a tangent is refused and not dropped, with and without grad mode."""
    from flash_attn_v100 import flash_attn_func

    q, k, v, _ = (t.cuda() for t in ao.make_inputs(1, 33, 2, 64, seed=2))
    with torch.set_grad_enabled(grad_mode), forward_ad.dual_level():
        for which in range(3):
            args = [q, k, v]
            args[which] = forward_ad.make_dual(args[which], torch.ones_like(args[which]))
            with pytest.raises(RuntimeError):
                flash_attn_func(*args)


@pytest.mark.gpu
def test_saved_tensor_hooks_and_checkpoint():
    from flash_attn_v100 import flash_attn_func

    q, k, v, do = (t.cuda() for t in ao.make_inputs(2, 130, 3, 128, seed=3))
    leaves = [t.clone().requires_grad_() for t in (q, k, v)]
    want = torch.autograd.grad(flash_attn_func(*leaves), leaves, do)
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t.shape) or t.cpu(), lambda t: t.cuda()):
        out = flash_attn_func(*leaves)
    assert len(packed) == 5  # q, k, v, out and the logsumexp
    for a, b in zip(torch.autograd.grad(out, leaves, do), want):
        assert torch.equal(a, b)
    out = torch.utils.checkpoint.checkpoint(flash_attn_func, *leaves, use_reentrant=False)
    for a, b in zip(torch.autograd.grad(out, leaves, do), want):
        assert torch.equal(a, b)
