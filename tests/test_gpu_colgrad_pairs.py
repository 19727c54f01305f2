"""fp32 column gradient as fp16 pairs: exponents of the rows of either operand, where they can go wrong."""
import ctypes

import pytest
import torch

from common import capi_backward
from mmcv_amd import capi

pytestmark = pytest.mark.gpu


def _case(seed, n, cin, cout, h, w, kernel=(3, 3), groups=1, dgroups=1, stride=1):
    g = torch.Generator().manual_seed(seed)
    kh, kw = kernel
    ho, wo = (h + 2 - kh) // stride + 1, (w + 2 - kw) // stride + 1
    # quarter-pixel offsets and mask values of 8 bits: positions and corner weights are exact in fp32
    case = dict(input=torch.randn(n, cin, h, w, generator=g),
                offset=torch.round(torch.randn(n, 2 * dgroups * kh * kw, ho, wo, generator=g) * 6) / 4,
                mask=torch.round(torch.rand(n, dgroups * kh * kw, ho, wo, generator=g) * 255 + 1) / 256,
                weight=torch.randn(cout, cin // groups, kh, kw, generator=g), bias=None, stride=(stride, stride), padding=(1, 1),
                dilation=(1, 1), groups=groups, deform_groups=dgroups)
    return {k: v.cuda() if torch.is_tensor(v) else v for k, v in case.items()}, torch.randn(n, cout, ho, wo, generator=g).cuda()


SHAPES = [dict(n=2, cin=64, cout=96, h=33, w=37),                     # planes and rows that no tile divides
          dict(n=1, cin=32, cout=72, h=20, w=31),                     # most of the last K step is padding
          dict(n=1, cin=96, cout=130, h=21, w=50),                    # five K steps, padding in the last
          dict(n=2, cin=64, cout=256, h=24, w=30, groups=2, dgroups=2),
          dict(n=1, cin=64, cout=512, h=26, w=31, stride=2),          # sixteen
          dict(n=1, cin=64, cout=128, h=24, w=33, kernel=(1, 3)),
          dict(n=8, cin=512, cout=256, h=36, w=50)]                   # tiles of 256


@pytest.mark.parametrize('shape', SHAPES, ids=lambda s: '_'.join(str(v) for v in s.values()))
def test_error_is_that_of_fp32(shape):
    print(f'case={shape}', flush=True)
    dev, go = _case(5, **shape)
    g = torch.Generator().manual_seed(3)
    # pixels of grad_output, and input channels of the weights, of very different magnitudes: each has an exponent of its own
    go = go * (10.0 ** (torch.rand(go.shape[0], 1, *go.shape[2:], generator=g) * 8 - 4)).cuda()
    rows = (10.0 ** (torch.rand(1, dev['weight'].shape[1], 1, 1, generator=g) * 16 - 8)).cuda()
    double = lambda d: {k: v.double() if torch.is_tensor(v) else v for k, v in d.items()}
    K, C = shape['cout'] // shape.get('groups', 1), shape['cin']
    # sums of K products, each off by at most 2^-24 for either operand's rest beyond two fp16 numbers and 2^-22 / 3 for the product of the two
    # rests, added in fp32: sqrt(K) * 2^-24 for random roundings.
    bound = (K ** 0.5 + 4) * 2.0 ** -24

    def error(y, ref, dims):
        norm = lambda t: torch.linalg.vector_norm(t, dim=dims)
        return float((norm(y.double() - ref) / norm(ref).clamp(min=1e-300)).max())

    wide = dict(dev, weight=dev['weight'] * rows)
    gin = capi_backward(wide, go, path=capi.PATH_FUSED)[0]
    ref = capi_backward(double(wide), go.double())[0]
    by_channel = error(gin, ref, (0, 2, 3))
    assert by_channel <= bound, by_channel
    # by pixel: the worst of thousands, and a sum over channels behind it
    gmask = capi_backward(dev, go, path=capi.PATH_FUSED)[2]
    by_pixel = error(gmask, capi_backward(double(dev), go.double())[2], (1,))
    few = shape.get('dgroups', 1) * 9
    assert by_pixel <= 2 * ((K + C) ** 0.5 + 4) * 2.0 ** -24 * (16 if few < 10 else 8), by_pixel


def _as_triples(dev, go):
    """The gradients of input, offset and mask with a workspace that ends in front of the magnitudes."""
    lib = capi.load()
    bp = capi.MdcnBwdParams()
    bp.conv = capi.make_params(capi.MDCN_F32, 2, 64, 33, 37, 128, 3, 3, (1, 1), (1, 1), (1, 1), 1, 1)
    p = bp.conv
    p.path = capi.PATH_FUSED
    out = [torch.empty_like(dev[k]) for k in ('input', 'offset', 'mask')]
    p.input, p.offset, p.mask, p.weight = (dev[k].data_ptr() for k in ('input', 'offset', 'mask', 'weight'))
    bp.grad_output = go.data_ptr()
    bp.grad_input, bp.grad_offset, bp.grad_mask = (t.data_ptr() for t in out)
    up = lambda v: (v + 255) // 256 * 256
    need = lib.mdcn_backward_workspace_bytes(ctypes.byref(bp)) - up(2 * 4 * 33 * 37 * 2) - up(640 * 4) - up(640 * 128 * 4)
    ws = torch.empty(need, dtype=torch.uint8, device='cuda')
    p.workspace, p.workspace_bytes = ws.data_ptr(), need
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert lib.mdcn_backward(ctypes.byref(bp), stream) == 0
    torch.cuda.synchronize()
    p.workspace_bytes = need - 256
    assert lib.mdcn_backward(ctypes.byref(bp), stream) == -4
    return out


def test_without_room_for_magnitudes():
    """Such a workspace gives the same call as bf16 triples, a smaller one is refused."""
    dev, go = _case(8, 2, 64, 128, 33, 37)
    y = capi_backward(dev, go, path=capi.PATH_FUSED)[0]
    gin = _as_triples(dev, go)[0]
    assert not torch.equal(gin, y)
    assert float((gin - y).norm() / y.norm()) <= 2 * (128 ** 0.5 + 4) * 2.0 ** -24


@pytest.mark.parametrize('where', ['weight', 'grad_output'])
@pytest.mark.parametrize('value', [float('inf'), float('nan'), 3e38])
def test_not_finite(where, value):
    """One number that fp16 pairs cannot hold, or whose row overflows: what is finite, and its value, as with bf16 triples."""
    print(f'case={where} {value}', flush=True)
    dev, go = _case(9, 2, 64, 128, 33, 37)
    dev['weight'][:, 7] *= 1e6   # a row whose other numbers fp16 does not hold unscaled
    (dev['weight'] if where == 'weight' else go)[1, 7, 1, 1] = value
    for y, ref in zip(capi_backward(dev, go, path=capi.PATH_FUSED)[:3], _as_triples(dev, go)):
        assert torch.equal(y.isnan(), ref.isnan()) and torch.equal(y.isinf(), ref.isinf())
        ok = ref.isfinite()
        d, r = (y - ref)[ok].double(), ref[ok].double()
        assert float(d.norm() / r.norm()) <= 4 * (128 ** 0.5 + 4) * 2.0 ** -24
