"""Tiles cut along K: workspaces that do not hold what their parts meet in."""
import ctypes

import pytest
import torch

from common import DT, capi_forward, cast_case, make_case
from mmcv_amd import capi

pytestmark = pytest.mark.gpu


def _forward(case, bytes_off):
    """The call with `bytes_off` bytes less than it asks for."""
    lib = capi.load()
    x, w = case['input'], case['weight']
    p = capi.make_params(DT[x.dtype], *x.shape, w.shape[0], *w.shape[2:], case['stride'], case['padding'], case['dilation'],
                         case['groups'], case['deform_groups'], capi.PATH_FUSED)
    _, Ho, Wo = capi.output_size(p)
    out = torch.empty(x.shape[0], w.shape[0], Ho, Wo, dtype=x.dtype, device=x.device)
    p.input, p.offset, p.mask, p.weight, p.bias = (case[k].data_ptr() for k in ('input', 'offset', 'mask', 'weight', 'bias'))
    p.output = out.data_ptr()
    p.workspace_bytes = lib.mdcn_workspace_bytes(ctypes.byref(p)) - bytes_off
    ws = torch.empty(p.workspace_bytes, dtype=torch.uint8, device=x.device)
    p.workspace = ws.data_ptr()
    assert lib.mdcn_forward(ctypes.byref(p), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    torch.cuda.synchronize()
    return out


# 17 tiles an XCD of 32 workgroups, 72 steps: even shares of tiles that equal parts leave whole; 11 tiles of 144: in the place of two parts
@pytest.mark.parametrize('cin,plane', [(256, (128, 136)), (512, (88, 128))], ids=str)
def test_without_room_for_shares(cin, plane):
    """Shares have two buffers of 128 KiB a workgroup, equal parts one: less room is the other schedule, or whole tiles."""
    print(f'case={cin} {plane}', flush=True)
    case = cast_case(make_case(31, 1, cin, 256, *plane, sigma=2.0), torch.float32, torch.device('cuda:0'))
    whole = capi_forward(case, path=capi.PATH_FUSED, unsplit=True).double()
    for bytes_off in (0, 256, 40 << 20):
        err = float((_forward(case, bytes_off).double() - whole).norm() / whole.norm())
        assert err <= 2 * (9 * cin) ** 0.5 * 2.0 ** -24, (bytes_off, err)   # fp32 sums of 9 cin terms in two orders
