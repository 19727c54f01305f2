"""The segment kernel (channel counts that do not fill 128-byte slabs of one deformable group) against the
CPU oracle, through the C ABI with the scratch of mdcn_workspace_wanted()."""
import ctypes

import pytest
import torch

from mmcv_amd import capi
from common import DT, TOL, capi_forward, cast_case, make_case, oracle_forward, rel_err

pytestmark = pytest.mark.gpu

CASES = {
    # 16-byte chunks per segment: below one, one and a rest, chunk groups of 1, 2 and 4 with padding
    'seg1': dict(N=1, Cin=4, Cout=5, H=7, W=9, deform_groups=4),
    'seg3': dict(N=2, Cin=3, Cout=1, H=11, W=13),
    'seg4_dg16': dict(N=1, Cin=64, Cout=64, H=12, W=17, deform_groups=16),
    'seg8_dg8': dict(N=2, Cin=64, Cout=64, H=19, W=23, deform_groups=8),
    'seg24': dict(N=1, Cin=24, Cout=40, H=16, W=15),
    'seg40_groups': dict(N=1, Cin=80, Cout=144, H=10, W=21, groups=2, stride=2),
    'seg48': dict(N=2, Cin=96, Cout=72, H=13, W=11, deform_groups=2, sigma=5.0),
    # groups and deformable groups that do not divide each other
    'gcd': dict(N=1, Cin=48, Cout=66, H=9, W=10, groups=2, deform_groups=3),
    # an odd number of pairs, one pair, a 5 x 5 kernel
    'pairs1': dict(N=3, Cin=8, Cout=32, H=5, W=7, k=1, padding=0),
    'k5': dict(N=1, Cin=20, Cout=33, H=12, W=12, k=5, padding=2),
    # output channels: three blocks, more than one tile of 256, blocks rounded up to a kernel's
    'cout320': dict(N=1, Cin=56, Cout=320, H=9, W=9),
    'cout150': dict(N=1, Cin=120, Cout=150, H=8, W=9, dilation=2, padding=2),
    'cout250': dict(N=1, Cin=16, Cout=250, H=12, W=11),
    # enough pixels that no wave shares its K range
    'large': dict(N=4, Cin=24, Cout=20, H=140, W=131),
}


def segment_forward(case, unsplit=False, short=False):
    lib = capi.load()
    x, off, msk, w, b = (case[k] for k in ('input', 'offset', 'mask', 'weight', 'bias'))
    N, Cin, H, W = x.shape
    Cout, _, kh, kw = w.shape
    p = capi.make_params(DT[x.dtype], N, Cin, H, W, Cout, kh, kw, case['stride'], case['padding'],
                         case['dilation'], case['groups'], case['deform_groups'])
    p.no_k_split = 1 if unsplit else 0
    assert lib.mdcn_forward_kernels(ctypes.byref(p)) == b'segment_kernel'
    rc, Ho, Wo = capi.output_size(p)
    assert rc == 0
    out = torch.full((N, Cout, Ho, Wo), 7.0, dtype=x.dtype, device=x.device)
    need = lib.mdcn_workspace_wanted(ctypes.byref(p))
    assert need > 0 and lib.mdcn_workspace_bytes(ctypes.byref(p)) == 0
    ws = torch.full((need,), 255, dtype=torch.uint8, device=x.device)  # NaNs where nothing writes
    p.input, p.offset, p.weight, p.output = (t.data_ptr() for t in (x, off, w, out))
    p.mask = msk.data_ptr() if msk is not None else None
    p.bias = b.data_ptr() if b is not None else None
    p.workspace, p.workspace_bytes = ws.data_ptr(), need - (1 if short else 0)
    rc = lib.mdcn_forward(ctypes.byref(p), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, capi.status_string(rc)
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize('name', sorted(CASES))
def test_segment_kernel(name, dtype):
    print(f'case={name} dtype={dtype}', flush=True)
    case = cast_case(make_case(31, **CASES[name]), dtype)
    dev = cast_case(case, dtype, 'cuda')
    if name == 'large':  # (the scalar oracle is slow at this size: the one-thread-per-output kernel stands in)
        ref = capi_forward(dev, path=capi.PATH_DIRECT).float().cpu().numpy()
    else:
        ref = oracle_forward(case)
    y = segment_forward(dev)
    assert rel_err(y.float().cpu().numpy(), ref) <= TOL[dtype]
    y1 = segment_forward(dev, unsplit=True)
    assert rel_err(y1.float().cpu().numpy(), ref) <= TOL[dtype]
    if name in ('seg8_dg8', 'seg48'):
        unmod = dict(dev, mask=None, bias=None)
        ref1 = oracle_forward(dict(case, mask=torch.ones_like(case['mask']), bias=None))
        assert rel_err(segment_forward(unmod).float().cpu().numpy(), ref1) <= TOL[dtype]
        # images in passes of one
        lib = capi.load()
        lib.mdcn_set_pass_limits(1, 0)
        try:
            yp = segment_forward(dev)
        finally:
            lib.mdcn_set_pass_limits(0, 0)
        assert rel_err(yp.float().cpu().numpy(), ref) <= TOL[dtype]
        # a workspace one byte short: the kernel that needs none
        assert torch.equal(segment_forward(dev, short=True), capi_forward(dev, path=capi.PATH_DIRECT))


def test_segment_path_on_a_shape_of_the_fused_kernels():
    dev = cast_case(make_case(32, N=1, Cin=64, Cout=96, H=14, W=15), torch.bfloat16, 'cuda')
    lib = capi.load()
    p = capi.make_params(capi.MDCN_BF16, 1, 64, 14, 15, 96, 3, 3, (1, 1), (1, 1), (1, 1), 1, 1, capi.PATH_SEGMENT)
    assert lib.mdcn_forward_kernels(ctypes.byref(p)) == b'segment_kernel'
    ref = capi_forward(dev, path=capi.PATH_FUSED).float()
    out = torch.empty(1, 96, 14, 15, dtype=torch.bfloat16, device='cuda')
    ws = torch.empty(lib.mdcn_workspace_wanted(ctypes.byref(p)), dtype=torch.uint8, device='cuda')
    p.input, p.offset, p.mask, p.weight, p.bias = (dev[k].data_ptr() for k in ('input', 'offset', 'mask', 'weight', 'bias'))
    p.output, p.workspace, p.workspace_bytes = out.data_ptr(), ws.data_ptr(), ws.numel()
    assert lib.mdcn_forward(ctypes.byref(p), None) == 0
    torch.cuda.synchronize()
    assert float((out.float() - ref).abs().max() / ref.abs().max()) <= TOL[torch.bfloat16]


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16], ids=['bf16', 'f16'])
@pytest.mark.parametrize('name', ['seg1', 'seg3', 'seg8_dg8', 'seg24', 'seg40_groups', 'seg48', 'gcd', 'k5', 'cout150', 'cout250'])
def test_16bit_results_are_rounded_once(name, dtype):
    """Samples, products and sums of 16-bit tensors are those of fp32: every output is the true one, rounded once."""
    print(f'case={name} dtype={dtype}', flush=True)
    case = make_case(33, **CASES[name])
    case['offset'] = torch.round(case['offset'] * 4) / 4   # exact positions and corner weights
    dev = cast_case(case, dtype, 'cuda')
    ref = capi_forward({k: v.double() if torch.is_tensor(v) else v for k, v in dev.items()})
    y = segment_forward(dev).double()
    half_ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    # an fp32 sum of (channel, tap) products of terms no larger than some 4 in all: 2^-24 each
    terms = case['weight'][0].numel()
    bound = ref.abs() * half_ulp + 2.0 ** -25 + terms * 2.0 ** -24 * 4
    worst = float(((y - ref).abs() / bound).max())
    assert worst <= 1.0, worst


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16], ids=['bf16', 'f16'])
def test_16bit_infinities(dtype):
    g = torch.Generator().manual_seed(12)
    case = make_case(34, N=2, Cin=24, Cout=40, H=14, W=15, sigma=0.3, padding=0)
    case['offset'] = torch.rand(case['offset'].shape, generator=g) * 0.4 + 0.3
    case['input'][0, 3, 5, 5], case['input'][0, 4, 9, 9] = float('inf'), float('nan')
    case['weight'][5, 3], case['weight'][6, 3], case['weight'][7, 9] = float('inf'), -float('inf'), float('nan')
    dev = cast_case(case, dtype, 'cuda')
    got, ref = segment_forward(dev), capi_forward(dev, path=capi.PATH_DIRECT)
    assert torch.equal(got.isnan(), ref.isnan()) and torch.equal(got.isinf(), ref.isinf())
    ok = ref.isfinite()
    assert 0 < int(ok.sum()) < ok.numel()
    assert float((got[ok] - ref[ok]).abs().max()) <= 2.0 ** (-7 if dtype == torch.bfloat16 else -10) * float(ref[ok].abs().max())
