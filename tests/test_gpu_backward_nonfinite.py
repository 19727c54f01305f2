"""16-bit gradients of what is not finite: an infinity or NaN in grad_output or the mask, and a column gradient beyond
fp16, reach the gradients they belong to and nothing else, against the kernels without a window."""
import pytest
import torch

from mmcv_amd import capi
from common import capi_backward, cast_case, make_case

pytestmark = pytest.mark.gpu

NAMES = ('grad_input', 'grad_offset', 'grad_mask', 'grad_weight', 'grad_bias')
#: 2-norm of a 16-bit result's error: one rounding of each intermediate tensor and of the result
REL = {torch.bfloat16: 1e-2, torch.float16: 2e-3}
SHAPES = {
    'whole_slabs': (dict(N=1, Cin=128, Cout=128, H=18, W=37, sigma=0.7), capi.PATH_FUSED),
    'whole_slabs_dg2': (dict(N=2, Cin=128, Cout=64, H=9, W=33, deform_groups=2, sigma=3.0), capi.PATH_FUSED),
    'few_tiles': (dict(N=1, Cin=64, Cout=64, H=12, W=20), capi.PATH_AUTO),
    'padded': (dict(N=2, Cin=20, Cout=12, H=11, W=35), capi.PATH_AUTO),
    'uneven': (dict(N=2, Cin=96, Cout=72, H=13, W=17, deform_groups=2), capi.PATH_AUTO),
}


def _case(shape, dtype, seed):
    kw, path = SHAPES[shape]
    case = make_case(seed, **kw)
    # never on a pixel: a corner of weight zero makes NaN of an infinity in both, but not for the same reason
    case['offset'] = torch.floor(case['offset']) + torch.randint(1, 4, case['offset'].shape,
                                                                generator=torch.Generator().manual_seed(seed)) / 4
    gy = torch.randn(kw['N'], kw['Cout'], *case['offset'].shape[2:], generator=torch.Generator().manual_seed(seed + 1))
    return cast_case(case, dtype, 'cuda'), gy.to(dtype), path


def _check(got, ref, dtype, same):
    for nm, a, b in zip(NAMES, got, ref):
        a, b = a.double(), b.double()
        if same:
            assert torch.equal(a.isfinite(), b.isfinite()), (nm, int(a.isfinite().sum()), int(b.isfinite().sum()))
        else:
            assert not bool((a.isfinite() & ~b.isfinite()).any()), nm
        ok = a.isfinite() & b.isfinite()
        assert float((a[ok] - b[ok]).norm()) <= REL[dtype] * max(float(b[ok].norm()), 1e-30), nm


@pytest.mark.parametrize('value', ['inf', '-inf', 'nan'])
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16], ids=['bf16', 'f16'])
@pytest.mark.parametrize('shape', sorted(SHAPES))
def test_grad_output(shape, dtype, value):
    print(f'case={shape} {dtype} {value}', flush=True)
    dev, gy, path = _case(shape, dtype, 61)
    gy[0, 3, 4, 6] = float(value)
    got, ref = capi_backward(dev, gy.cuda(), path=path), capi_backward(dev, gy.cuda(), path=capi.PATH_DIRECT)
    assert 0 < int((~ref[0].isfinite()).sum()) < ref[0].numel() // 2
    _check(got, ref, dtype, same=True)


@pytest.mark.parametrize('value', ['inf', 'nan'])
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16], ids=['bf16', 'f16'])
@pytest.mark.parametrize('shape', sorted(SHAPES))
def test_mask(shape, dtype, value):
    print(f'case={shape} {dtype} {value}', flush=True)
    dev, gy, path = _case(shape, dtype, 62)
    dev['mask'][0, 4, 4, 6] = float(value)
    got, ref = capi_backward(dev, gy.cuda(), path=path), capi_backward(dev, gy.cuda(), path=capi.PATH_DIRECT)
    assert 0 < int((~ref[0].isfinite()).sum()) < ref[0].numel() // 2
    _check(got, ref, dtype, same=True)


@pytest.mark.parametrize('shape', sorted(SHAPES))
def test_column_gradient_beyond_fp16(shape):
    """Where the column gradient is held in fp16 it overflows before the result does: it may be infinite then, but is no
    other number than the true one."""
    print(f'case={shape}', flush=True)
    dev, gy, path = _case(shape, torch.float16, 63)
    dev['weight'] = dev['weight'].abs() + 0.25
    gy[0, :, 4, 6] = 60000.0
    got, ref = capi_backward(dev, gy.cuda(), path=path), capi_backward(dev, gy.cuda(), path=capi.PATH_DIRECT)
    assert int((~ref[0].isfinite()).sum()) > 0
    _check(got, ref, torch.float16, same=False)


@pytest.mark.parametrize('scale', [1e-36, 1e-30, 1e30])
def test_magnitudes(scale):
    """bf16 gradients of any size, through the window or past it."""
    print(f'scale={scale}', flush=True)
    for shape in ('whole_slabs', 'padded'):
        dev, gy, path = _case(shape, torch.bfloat16, 64)
        gy = (gy.float() * scale).bfloat16()
        got, ref = capi_backward(dev, gy.cuda(), path=path), capi_backward(dev, gy.cuda(), path=capi.PATH_DIRECT)
        _check(got, ref, torch.bfloat16, same=True)
