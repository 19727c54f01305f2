"""Calls of few tiles: which kernel takes them, at the edges of the rule, and tiles cut into as many parts as there are."""
import ctypes

import pytest
import torch

from common import TOL, capi, capi_forward, cast_case, make_case, oracle_forward, rel_err

pytestmark = pytest.mark.gpu


def _kernels(case, dtype, **over):
    n, cin, h, w = case['input'].shape
    code = {torch.float32: capi.MDCN_F32, torch.bfloat16: capi.MDCN_BF16, torch.float16: capi.MDCN_F16}[dtype]
    p = capi.make_params(code, n, cin, h, w, case['weight'].shape[0], 3, 3, case['stride'], case['padding'],
                         case['dilation'], case['groups'], case['deform_groups'], over.pop('path', capi.PATH_AUTO))
    for k, v in over.items():
        setattr(p, k, v)
    return capi.load().mdcn_forward_kernels(ctypes.byref(p)).decode()


@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16, torch.float16], ids=['f32', 'bf16', 'f16'])
@pytest.mark.parametrize('kw,segment', [
    (dict(N=1, Cin=64, Cout=64, H=9, W=7), True),
    (dict(N=3, Cin=64, Cout=33, H=13, W=11, stride=2), True),
    (dict(N=1, Cin=64, Cout=64, H=12, W=12, deform_groups=1, groups=2), None),
    (dict(N=1, Cin=64, Cout=65, H=9, W=7), False),    # three blocks of output channels
    (dict(N=1, Cin=192, Cout=64, H=9, W=7), False),   # more than 18 iterations
], ids=lambda v: '-'.join(f'{k}{x}' for k, x in v.items()) if isinstance(v, dict) else None)
def test_small_calls(kw, segment, dtype):
    case = cast_case(make_case(41, **kw), dtype)
    dev = cast_case(case, dtype, 'cuda')
    if segment is not None:
        assert ('segment' in _kernels(case, dtype)) == segment
    assert 'segment' not in _kernels(case, dtype, path=capi.PATH_FUSED)
    assert 'segment' not in _kernels(case, dtype, input_nhwc=1)
    ref = oracle_forward(case)
    assert rel_err(capi_forward(dev).float().cpu().numpy(), ref) <= TOL[dtype]
    # unmodulated, and without a split of K
    unmod = dict(dev, mask=None, bias=None)
    ref1 = oracle_forward(dict(case, mask=torch.ones_like(case['mask']), bias=None))
    assert rel_err(capi_forward(unmod, unsplit=True).float().cpu().numpy(), ref1) <= TOL[dtype]


@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16], ids=['f32', 'bf16'])
def test_where_the_segment_kernel_ends(dtype):
    """768 waves of 32 pixels and one more: the two kernels agree on what is the same but for the last row."""
    a = cast_case(make_case(42, N=1, Cin=64, Cout=64, H=128, W=192), dtype, 'cuda')
    b = cast_case(make_case(43, N=1, Cin=64, Cout=64, H=129, W=192), dtype, 'cuda')
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert 'segment' in _kernels(a, dtype) and 'segment' not in _kernels(b, dtype)
    for dev in (a, b):
        ref = capi_forward(dev, path=capi.PATH_DIRECT).float().cpu().numpy()
        assert rel_err(capi_forward(dev).float().cpu().numpy(), ref) <= TOL[dtype]


@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16], ids=['f32', 'bf16'])
@pytest.mark.parametrize('kw', [
    dict(N=1, Cin=512, Cout=512, H=13, W=13), dict(N=1, Cin=256, Cout=200, H=30, W=31),
    dict(N=1, Cin=512, Cout=256, H=12, W=19, deform_groups=4), dict(N=2, Cin=256, Cout=256, H=28, W=28, deform_groups=2),
    dict(N=1, Cin=256, Cout=256, H=64, W=128), dict(N=1, Cin=256, Cout=256, H=64, W=130),
], ids=lambda v: '-'.join(f'{k}{x}' for k, x in v.items()))
def test_narrow_tiles_and_many_parts(kw, dtype):
    dev = cast_case(make_case(44, **kw), dtype, 'cuda')
    ref = capi_forward(dev, path=capi.PATH_DIRECT).float().cpu().numpy()
    y = capi_forward(dev)
    assert rel_err(y.float().cpu().numpy(), ref) <= TOL[dtype]
    # the sum does not depend on which part came last, and the counters are left as they were found
    for _ in range(3):
        assert torch.equal(capi_forward(dev), y)
    assert rel_err(capi_forward(dev, unsplit=True).float().cpu().numpy(), ref) <= TOL[dtype]


@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16, torch.float16], ids=['f32', 'bf16', 'f16'])
@pytest.mark.parametrize('kw', [dict(N=1, Cin=128, Cout=72, H=9, W=11), dict(N=1, Cin=128, Cout=264, H=8, W=9),
                                dict(N=1, Cin=256, Cout=70, H=7, W=9, groups=2)],
                         ids=['tail', 'two_tiles', 'groups'])
def test_weights_that_start_anywhere(kw, dtype):
    """3x3 weights are repacked nine taps at a time where they start 16-byte aligned, one by one elsewhere."""
    dev = cast_case(make_case(45, **kw), dtype, 'cuda')
    y = capi_forward(dev, path=capi.PATH_FUSED)
    flat = torch.empty(dev['weight'].numel() + 1, dtype=dtype, device='cuda')
    flat[1:] = dev['weight'].flatten()
    shifted = dict(dev, weight=flat[1:].view(dev['weight'].shape))
    assert shifted['weight'].data_ptr() % 16 != 0 and dev['weight'].data_ptr() % 16 == 0
    assert torch.equal(capi_forward(shifted, path=capi.PATH_FUSED), y)
    assert rel_err(y.float().cpu().numpy(), oracle_forward(cast_case(make_case(45, **kw), dtype))) <= TOL[dtype]
