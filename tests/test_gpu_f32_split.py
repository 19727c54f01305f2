"""fp32 tensors on the bf16 matrix pipe (three bf16 planes per operand): the error of fp32 arithmetic, whatever
the magnitudes."""
import pytest
import torch

from common import capi_forward
from mmcv_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('cout', [48, 96, 200], ids=['tile64', 'tile128', 'tile256'])
@pytest.mark.parametrize('scale_x,scale_w', [(1.0, 1.0), (1e18, 1e-15), (3e-17, 1e12), (1e-25, 1e-5)])
def test_split_products_are_fp32(cout, scale_x, scale_w):
    g = torch.Generator().manual_seed(cout)
    n, cin, h, w = 2, 96, 15, 18
    # quarter-pixel offsets and mask values of 8 bits: positions and corner weights are exact in fp32, so that what
    # is left is the rounding of products and sums
    off = torch.round(torch.randn(n, 18, h, w, generator=g) * 8) / 4
    mask = torch.round(torch.rand(n, 9, h, w, generator=g) * 256) / 256
    # magnitudes of one tensor spread over six decades
    spread = 10.0 ** (torch.rand(n, cin, h, w, generator=g) * 6 - 3)
    case = dict(input=torch.randn(n, cin, h, w, generator=g) * spread * scale_x, offset=off, mask=mask,
                weight=torch.randn(cout, cin, 3, 3, generator=g) * scale_w, bias=None, stride=(1, 1), padding=(1, 1),
                dilation=(1, 1), groups=1, deform_groups=1)
    dev = {k: v.cuda() if torch.is_tensor(v) else v for k, v in case.items()}
    y = capi_forward(dev, path=capi.PATH_FUSED).double()
    wide = {k: v.double() if torch.is_tensor(v) else v for k, v in dev.items()}
    ref = capi_forward(wide)
    # sums of 864 products by fp32 adds: sqrt(864) * 2^-24 = 1.8e-6 of the terms' 2-norm for random roundings
    assert float((y - ref).norm() / ref.norm()) <= 1.8e-6
