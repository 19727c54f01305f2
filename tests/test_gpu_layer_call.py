"""The layers' one-call path (autograd in C++) against the Python Functions on the same tensors."""
import pytest
import torch

from common import cast_case, make_case

pytestmark = pytest.mark.gpu


def _leaves(dtype, names):
    case = cast_case(make_case(5, 2, 64, 48, 9, 11), dtype, 'cuda')
    t = {k: case[k].clone() for k in ('input', 'offset', 'mask', 'weight', 'bias')}
    for k in names:
        t[k].requires_grad_(True)
    return t


@pytest.mark.parametrize('names', [('input',), ('weight',), ('bias',), ('offset', 'bias'), ('mask', 'weight'),
                                   ('input', 'offset', 'mask', 'weight', 'bias')], ids='-'.join)
def test_gradients_that_are_asked_for(names):
    from mmcv_amd.ops import ModulatedDeformConv2dFunction, modulated_deform_conv2d
    args = ('input', 'offset', 'mask', 'weight', 'bias')
    got = []
    for fn in (modulated_deform_conv2d, ModulatedDeformConv2dFunction.apply):
        t = _leaves(torch.float32, names)
        y = fn(*[t[k] for k in args], 1, 1, 1, 1, 1)
        got.append((y.detach(),) + torch.autograd.grad(y.square().sum(), [t[k] for k in names]))
    assert torch.equal(got[0][0], got[1][0])
    for a, b in zip(*got):  # (grad_input is summed by atomics: the last bits vary)
        assert a.dtype == b.dtype and a.shape == b.shape
        assert float((a - b).abs().max()) <= 1e-5 * float(b.abs().max())


def test_unmodulated_gradients_and_mixed_types():
    from mmcv_amd.ops import DeformConv2dFunction, deform_conv2d
    got = []
    for fn in (deform_conv2d, DeformConv2dFunction.apply):
        t = _leaves(torch.float32, ('input', 'weight'))
        y = fn(t['input'], t['offset'].half(), t['weight'], 1, 1)  # offset's type decides
        assert y.dtype == torch.float16
        grads = torch.autograd.grad(y.float().sum(), [t['input'], t['weight']])
        assert all(g.dtype == torch.float32 for g in grads)
        got.append((y.detach(),) + grads)
    for a, b in zip(*got):
        assert float((a.float() - b.float()).abs().max()) <= 2e-3 * float(b.float().abs().max())


def test_second_derivative_raises():
    from mmcv_amd.ops import modulated_deform_conv2d
    t = _leaves(torch.float32, ('input',))
    y = modulated_deform_conv2d(*[t[k] for k in ('input', 'offset', 'mask', 'weight', 'bias')], 1, 1)
    (g,) = torch.autograd.grad(y.square().sum(), t['input'], create_graph=True)
    with pytest.raises(RuntimeError, match='once_differentiable'):
        g.sum().backward()


def test_too_small_input_is_a_value_error():
    from mmcv_amd.ops import modulated_deform_conv2d
    z = lambda *s: torch.zeros(*s, device='cuda')
    with pytest.raises(ValueError, match='too small'):
        modulated_deform_conv2d(z(1, 4, 2, 2), z(1, 18, 1, 1), z(1, 9, 1, 1), z(4, 4, 3, 3), None)


def test_function_transforms_and_forward_mode_are_refused():
    """A Function without setup_context, vmap rule and jvp refuses them; so does the one call."""
    from mmcv_amd.ops import modulated_deform_conv2d
    t = _leaves(torch.float32, ())
    rest = [t[k] for k in ('offset', 'mask', 'weight', 'bias')]
    with pytest.raises(RuntimeError):
        torch.func.vmap(lambda x: modulated_deform_conv2d(x, *rest, 1, 1))(t['input'][None])
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda x: modulated_deform_conv2d(x, *rest, 1, 1).sum())(t['input'])
    with torch.autograd.forward_ad.dual_level(), pytest.raises(RuntimeError):
        x = torch.autograd.forward_ad.make_dual(t['input'], torch.ones_like(t['input']))
        modulated_deform_conv2d(x, *rest, 1, 1)
