"""fp32 forward as fp16 pairs: exponents of the rows of either operand, where they can go wrong."""
import pytest
import torch

from common import capi_forward
from mmcv_amd import capi

pytestmark = pytest.mark.gpu


def _case(seed, n, cin, cout, h, w, kernel=(3, 3), groups=1, dgroups=1, stride=1, scale_x=None, scale_w=None, mask=None):
    g = torch.Generator().manual_seed(seed)
    kh, kw = kernel
    ho, wo = (h + 2 - kh) // stride + 1, (w + 2 - kw) // stride + 1
    # quarter-pixel offsets and mask values of 8 bits: positions and corner weights are exact in fp32
    off = torch.round(torch.randn(n, 2 * dgroups * kh * kw, ho, wo, generator=g) * 8) / 4
    m = torch.round(torch.rand(n, dgroups * kh * kw, ho, wo, generator=g) * 255 + 1) / 256
    x, wt = torch.randn(n, cin, h, w, generator=g), torch.randn(cout, cin // groups, kh, kw, generator=g)
    if scale_x is not None:
        x *= scale_x
    if scale_w is not None:
        wt *= scale_w
    if mask is not None:
        m *= mask
    case = dict(input=x, offset=off, mask=m, weight=wt, bias=None, stride=(stride, stride), padding=(1, 1), dilation=(1, 1),
                groups=groups, deform_groups=dgroups)
    return {k: v.cuda() if torch.is_tensor(v) else v for k, v in case.items()}


def _errors(dev, **kw):
    """Relative error (2-norm) against double precision, by (image, output channel) and by (image, pixel)."""
    y = capi_forward(dev, path=capi.PATH_FUSED, **kw).double()
    ref = capi_forward({k: v.double() if torch.is_tensor(v) else v for k, v in dev.items()})
    d = y - ref
    rel = lambda a, b: float((a / b.clamp(min=1e-300)).max())
    return rel(d.flatten(2).norm(dim=2), ref.flatten(2).norm(dim=2)), rel(d.norm(dim=1), ref.norm(dim=1))


SHAPES = [dict(n=2, cin=64, cout=200, h=33, w=37),                       # units of two slabs, 256-channel tiles, a rest of channels
          dict(n=1, cin=96, cout=130, h=21, w=50),                      # of three (read one by one)
          dict(n=1, cin=256, cout=256, h=19, w=23),                     # of eight
          dict(n=2, cin=192, cout=256, h=24, w=30, groups=2, dgroups=3),   # deformable groups that straddle groups: units of one
          dict(n=1, cin=256, cout=160, h=26, w=31, dgroups=2, stride=2),   # units of four
          dict(n=1, cin=64, cout=136, h=40, w=33, kernel=(5, 5)),       # the large table
          dict(n=3, cin=64, cout=144, h=40, w=1),                       # an image one pixel wide
          dict(n=3, cin=64, cout=144, h=1, w=47, kernel=(1, 3)),
          dict(n=3, cin=64, cout=144, h=2, w=2)]


@pytest.mark.parametrize('shape', SHAPES, ids=lambda s: '_'.join(str(v) for v in s.values()))
@pytest.mark.parametrize('unsplit', [False, True], ids=['cut', 'whole'])
def test_error_is_that_of_fp32(shape, unsplit):
    print(f'case={shape}', flush=True)
    g = torch.Generator().manual_seed(3)
    # images, output channels and pixels of very different magnitudes, each of which has an exponent of its own
    images = 10.0 ** (torch.rand(shape['n'], 1, shape['h'], shape['w'], generator=g) * 8 - 4)
    rows = 10.0 ** (torch.rand(shape['cout'], 1, 1, 1, generator=g) * 30 - 15)
    dev = _case(5, scale_x=images, scale_w=rows, **shape)
    by_channel, by_pixel = _errors(dict(dev, weight=dev['weight'] / rows.cuda()), unsplit=unsplit)
    # sums of K products, each off by at most 2^-24 for either operand's rest beyond two fp16 numbers and 2^-22 / 3 for the product of the two
    # rests, added in fp32: sqrt(K) * 2^-24 for random roundings.  By pixel: the worst of thousands, twice that
    K = shape['cin'] // shape.get('groups', 1) * shape.get('kernel', (3, 3))[0] * shape.get('kernel', (3, 3))[1]
    bound = (K ** 0.5 + 4) * 2.0 ** -24
    # (the bound is on the error over the 2-norm of the terms; an output that the terms cancel in is smaller than that, and with four pixels, of
    # which the magnitudes leave one, a channel is a single output: there only pixels, which have 144 channels, are compared)
    few = shape['h'] * shape['w'] < 32
    assert (few or by_channel <= bound) and by_pixel <= 2 * bound, (by_channel, by_pixel)
    by_channel, _ = _errors(dev, unsplit=unsplit)
    assert few or by_channel <= bound, by_channel


@pytest.mark.parametrize('mask', [2.0 ** -100, 2.0 ** 20, 2.0 ** 90], ids=['tiny', 'large', 'huge'])
def test_masks_of_any_magnitude(mask):
    print(f'mask={mask}', flush=True)
    dev = _case(7, n=1, cin=64, cout=160, h=20, w=24, mask=mask, scale_x=2.0 ** -60 if mask > 1 else 1.0)
    by_channel, by_pixel = _errors(dev)
    assert by_channel <= (576 ** 0.5 + 4) * 2.0 ** -24 and by_pixel <= 2 * (576 ** 0.5 + 4) * 2.0 ** -24


def test_without_room_for_exponents():
    """A workspace that ends behind the copies gives the same call as bf16 triples, a smaller one is refused."""
    import ctypes
    dev = _case(8, n=2, cin=64, cout=200, h=33, w=37)
    y = capi_forward(dev, path=capi.PATH_FUSED)
    lib = capi.load()
    p = capi.make_params(capi.MDCN_F32, 2, 64, 33, 37, 200, 3, 3, (1, 1), (1, 1), (1, 1), 1, 1, capi.PATH_FUSED)
    out = torch.empty_like(y)
    p.input, p.offset, p.mask, p.weight = (dev[k].data_ptr() for k in ('input', 'offset', 'mask', 'weight'))
    p.output = out.data_ptr()
    copies = 2 * 35 * 39 * 64 * 4, 256 * 576 * 6
    need = sum((v + 255) // 256 * 256 for v in copies)
    assert need < lib.mdcn_workspace_bytes(ctypes.byref(p))
    ws = torch.empty(need, dtype=torch.uint8, device='cuda')
    p.workspace, p.workspace_bytes = ws.data_ptr(), need
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert lib.mdcn_forward(ctypes.byref(p), stream) == 0
    torch.cuda.synchronize()
    assert not torch.equal(out, y)
    assert float((out - y).norm() / y.norm()) <= 2 * (576 ** 0.5 + 4) * 2.0 ** -24
    p.workspace_bytes = need - 256
    assert lib.mdcn_forward(ctypes.byref(p), stream) == -4
