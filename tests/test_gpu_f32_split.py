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


def test_what_is_not_finite_stays_what_it_is():
    """Infinities, NaN and the largest numbers, in either operand, against one thread per output."""
    g = torch.Generator().manual_seed(9)
    n, c, h, w = 1, 64, 12, 14
    x, wt = torch.randn(n, c, h, w, generator=g), torch.randn(96, c, 3, 3, generator=g)
    # some weights are bf16 numbers, whose lower planes are zero
    wt[:, ::2] = wt[:, ::2].bfloat16().float()
    big = torch.finfo(torch.float32).max
    x[0, 3, 2, 2], x[0, 4, 5, 9], x[0, 5, 9, 3] = float('inf'), -float('inf'), float('nan')
    x[0, 6, 10, 11], x[0, 7, 10, 2] = big, -big
    wt *= 1e-3
    wt[5, 8, 1, 1], wt[6, 9, 0, 2], wt[7, 10, 2, 0] = float('inf'), float('nan'), big
    # no position on a pixel (no corner has weight zero) and none outside (where one path multiplies zeros, the other nothing)
    off = torch.rand(n, 18, h - 2, w - 2, generator=g) * 0.4 + 0.3
    case = dict(input=x, offset=off, mask=torch.rand(n, 9, h - 2, w - 2, generator=g) * 0.5 + 0.1, weight=wt,
                bias=None, stride=(1, 1), padding=(0, 0), dilation=(1, 1), groups=1, deform_groups=1)
    dev = {k: v.cuda() if torch.is_tensor(v) else v for k, v in case.items()}
    got, ref = capi_forward(dev, path=capi.PATH_FUSED), capi_forward(dev, path=capi.PATH_DIRECT)
    assert torch.equal(got.isnan(), ref.isnan()), (int(got.isnan().sum()), int(ref.isnan().sum()))
    assert torch.equal(got == float('inf'), ref == float('inf'))
    assert torch.equal(got == -float('inf'), ref == -float('inf'))
    ok = ref.isfinite()
    assert 0 < int(ok.sum()) < ok.numel() and int((ref.abs() == float('inf')).sum()) > 100
    # (sums that hold a product with the largest numbers are as coarse as those)
    small = ok & (ref.abs() < 1e30)
    assert float((got[small] - ref[small]).norm() / ref[small].norm()) <= 1e-6
    large = ok & (ref.abs() >= 1e30)
    assert int(large.sum()) > 100 and float(((got[large] - ref[large]) / ref[large]).abs().max()) <= 1e-5


def _backward_case(seed, n, cin, cout, h, w):
    g = torch.Generator().manual_seed(seed)
    off = torch.round(torch.randn(n, 18, h, w, generator=g) * 8) / 4 + 0.125   # exact, and never on a pixel
    case = dict(input=torch.randn(n, cin, h, w, generator=g), offset=off,
                mask=torch.round(torch.rand(n, 9, h, w, generator=g) * 255 + 1) / 256,
                weight=torch.randn(cout, cin, 3, 3, generator=g) * 0.05, bias=None, stride=(1, 1), padding=(1, 1),
                dilation=(1, 1), groups=1, deform_groups=1)
    gy = torch.randn(n, cout, h, w, generator=g) * 10.0 ** (torch.rand(n, cout, h, w, generator=g) * 4 - 2)
    return {k: v.cuda() if torch.is_tensor(v) else v for k, v in case.items()}, gy.cuda()


@pytest.mark.parametrize('cin,cout', [(64, 64), (256, 200), (40, 256)], ids=['narrow', 'wide', 'padded'])
def test_gradients_are_fp32(cin, cout):
    from common import capi_backward
    dev, gy = _backward_case(cin, 2, cin, cout, 17, 21)
    got = capi_backward(dev, gy, path=capi.PATH_FUSED)
    ref = capi_backward({k: v.double() if torch.is_tensor(v) else v for k, v in dev.items()}, gy.double())
    # grad_input, grad_offset, grad_mask: sums over cout and then over some 9 cin at most; grad_weight: over 714 pixels.
    # Roundings of 2^-24 each, at random: sqrt(terms) of them.  grad_bias aside (float sums of grad_output).
    for name, a, b in zip(('input', 'offset', 'mask', 'weight'), got, ref):
        terms = 714 if name == 'weight' else cout + 9 * cin
        assert float((a.double() - b).norm() / b.norm()) <= terms ** 0.5 * 2.0 ** -24, name


@pytest.mark.parametrize('cin,cout', [(64, 64), (256, 256)], ids=['narrow', 'wide'])
def test_gradients_of_what_is_not_finite(cin, cout):
    """An infinity, a NaN and the largest number in grad_output stay in the gradients they belong to."""
    from common import capi_backward
    dev, gy = _backward_case(cin + 1, 1, cin, cout, 16, 18)
    big = torch.finfo(torch.float32).max
    dev['weight'] *= 1e-3
    gy[0, 3, 4, 5], gy[0, 9, 12, 7], gy[0, 11, 9, 9] = float('inf'), float('nan'), big
    got = capi_backward(dev, gy, path=capi.PATH_FUSED)
    ref = capi_backward(dev, gy, path=capi.PATH_DIRECT)
    assert torch.equal(got[3].isnan(), ref[3].isnan()) and torch.equal(got[3].isinf(), ref[3].isinf())
    for name, a, b in zip(('input', 'offset', 'mask', 'weight'), got, ref):
        assert torch.equal(a.isfinite(), b.isfinite()), name
        small = b.isfinite() & (b.abs() < 1e28)
        assert 0 < int(small.sum()) < small.numel(), name
        assert float((a[small] - b[small]).norm() / b[small].norm()) <= 1e-5, name


# Calls that run in tiles of 256: the column gradient of 9 x 113 and 8 x 96 tiles (four and three rounds of the chip, full), the weight
# gradient of 6 144 K steps (2 560 and more) with an uneven last tile of rows (9 x 224 = 7.875 x 256).
LARGE = [(113, 256, 32), (96, 224, 256)]


@pytest.mark.parametrize('n,cin,cout', LARGE, ids=['column', 'column_weight'])
def test_gradients_in_tiles_of_256(n, cin, cout):
    from common import capi_backward
    print(f'n={n}', flush=True)
    dev, gy = _backward_case(cin + 2, n, cin, cout, 16, 16)
    got = capi_backward(dev, gy, path=capi.PATH_FUSED)
    ref = capi_backward({k: v.double() if torch.is_tensor(v) else v for k, v in dev.items()}, gy.double())
    for name, a, b in zip(('input', 'offset', 'mask', 'weight'), got, ref):   # (bounds: above)
        terms = 256 * n if name == 'weight' else cout + 9 * cin
        assert float((a.double() - b).norm() / b.norm()) <= terms ** 0.5 * 2.0 ** -24, name


@pytest.mark.parametrize('n,cin,cout', LARGE, ids=['column', 'column_weight'])
def test_tiles_of_256_of_what_is_not_finite(n, cin, cout):
    """A workgroup whose sums are not finite makes its tile again: in the first tile, in the uneven last one, and nowhere else."""
    from common import capi_backward
    print(f'n={n}', flush=True)
    dev, gy = _backward_case(cin + 3, n, cin, cout, 16, 16)
    big = torch.finfo(torch.float32).max
    dev['weight'] *= 1e-3
    dev['input'][3, cin - 1, 6, 6] = float('inf')
    gy[0, 3, 4, 5], gy[n - 1, 9, 12, 7], gy[n // 2, 11, 9, 9] = float('inf'), float('nan'), big
    got = capi_backward(dev, gy, path=capi.PATH_FUSED)
    ref = capi_backward(dev, gy, path=capi.PATH_DIRECT)
    assert torch.equal(got[3].isnan(), ref[3].isnan()) and torch.equal(got[3].isinf(), ref[3].isinf())
    for name, a, b in zip(('input', 'offset', 'mask', 'weight'), got, ref):
        assert torch.equal(a.isfinite(), b.isfinite()), name
        small = b.isfinite() & (b.abs() < 1e28)
        assert 0 < int(small.sum()) < small.numel(), name
        assert float((a[small] - b[small]).norm() / b[small].norm()) <= 1e-5, name


@pytest.mark.parametrize('shape', ['fused', 'fused_cut', 'nhwc', 'segment', 'segment_shared'])
def test_infinity_times_infinity(shape):
    """... is infinite, with the sign of the product, and so is a sum that only leaves fp32 at its end."""
    print(f'case={shape}', flush=True)
    g = torch.Generator().manual_seed(10)
    n, c, cout, h, w = (1, 256, 64, 9, 10) if shape == 'fused_cut' else (2, 24, 40, 70, 80) if shape == 'segment' else \
        (1, 24, 40, 12, 14) if shape == 'segment_shared' else (2, 64, 96, 12, 14)
    x, wt = torch.rand(n, c, h, w, generator=g) + 0.1, torch.randn(cout, c, 3, 3, generator=g)
    x[0, 3, 2, 2], x[0, 4, 5, 9] = float('inf'), -float('inf')
    wt[5, 3], wt[6, 3], wt[7, 4] = float('inf'), -float('inf'), -float('inf')
    wt[8, 5] = torch.finfo(torch.float32).max   # samples of this channel reach 1: products of up to fp32's largest, sums beyond
    x[n - 1, 5] = 2.0
    off = torch.rand(n, 18, h - 2, w - 2, generator=g) * 0.4 + 0.3
    case = dict(input=x, offset=off, mask=torch.rand(n, 9, h - 2, w - 2, generator=g) * 0.5 + 0.4, weight=wt,
                bias=None, stride=(1, 1), padding=(0, 0), dilation=(1, 1), groups=1, deform_groups=1)
    dev = {k: v.cuda() if torch.is_tensor(v) else v for k, v in case.items()}
    ref = capi_forward(dev, path=capi.PATH_DIRECT)
    if shape.startswith('segment'):
        from test_gpu_segment import segment_forward
        got = segment_forward(dev)
    else:
        got = capi_forward(dict(dev, input_nhwc=shape == 'nhwc'), path=capi.PATH_FUSED)
    assert int((ref[0, 5] == float('inf')).sum()) > 4 and int((ref[0, 6] == -float('inf')).sum()) > 4
    assert int((ref[n - 1, 8] == float('inf')).sum()) > 4
    assert torch.equal(got.isnan(), ref.isnan())
    assert torch.equal(got == float('inf'), ref == float('inf')) and torch.equal(got == -float('inf'), ref == -float('inf'))
    # what is finite: sums of up to 2304 products by fp32 adds on either side, sqrt(2304) * 2^-24 = 2.9e-6 each for random
    # roundings; by channel, since those of the largest numbers are as coarse as these
    for co in range(cout):
        ok = ref[:, co].isfinite()
        a, b = got[:, co][ok].double(), ref[:, co][ok].double()
        assert float((a - b).norm()) <= 6e-6 * float(b.norm()), co


TINY = [(2.0 ** -117, 1.0, 1.0), (1.0, 2.0 ** -117, 1.0), (2.0 ** 60, 2.0 ** -118, 1.0), (2.0 ** -30, 1.0, 2.0 ** -88)]


@pytest.mark.parametrize('kernel', ['fused', 'segment'])
@pytest.mark.parametrize('scale_x,scale_w,scale_m', TINY, ids=['x', 'w', 'w_large_x', 'mask'])
def test_smallest_numbers_keep_their_bits(kernel, scale_x, scale_w, scale_m):
    """Operands near the end of fp32's range: a number's lower bf16 planes lie below it."""
    print(f'case={kernel} {scale_x} {scale_w} {scale_m}', flush=True)
    g = torch.Generator().manual_seed(11)
    n, cin, cout, h, w = 2, 64 if kernel == 'fused' else 40, 72, 13, 15
    off = torch.round(torch.randn(n, 18, h, w, generator=g) * 8) / 4   # exact positions and corner weights
    mask = torch.round(torch.rand(n, 9, h, w, generator=g) * 255 + 1) / 256 * scale_m
    # (magnitudes of 1 to 2 times a factor: every operand stays a normal number, and the sums do)
    sign = lambda *s: torch.randint(0, 2, s, generator=g) * 2.0 - 1.0
    x = (1 + torch.rand(n, cin, h, w, generator=g)) * sign(n, cin, h, w) * scale_x
    wt = (1 + torch.rand(cout, cin, 3, 3, generator=g)) * sign(cout, cin, 3, 3) * scale_w
    case = dict(input=x, offset=off, mask=mask, weight=wt, bias=None, stride=(1, 1), padding=(1, 1),
                dilation=(1, 1), groups=1, deform_groups=1)
    dev = {k: v.cuda() if torch.is_tensor(v) else v for k, v in case.items()}
    ref = capi_forward({k: v.double() if torch.is_tensor(v) else v for k, v in dev.items()})
    if kernel == 'segment':
        from test_gpu_segment import segment_forward
        y = segment_forward(dev).double()
    else:
        y = capi_forward(dev, path=capi.PATH_FUSED).double()
    # sums of up to 576 products: 1.8e-6 as above, and outputs of some 2^-114 at least, so that nothing is subnormal
    assert float((y - ref).norm() / ref.norm()) <= 1.8e-6


@pytest.mark.parametrize('scale_x,scale_w,scale_g', [(1.0, 1.0, 2.0 ** -119), (1.0, 2.0 ** -119, 1.0), (2.0 ** -119, 1.0, 1.0),
                                                     (2.0 ** 40, 2.0 ** -119, 2.0 ** 40)], ids=['g', 'w', 'x', 'w_large_g'])
def test_gradients_of_the_smallest_numbers(scale_x, scale_w, scale_g):
    from common import capi_backward
    print(f'case={scale_x} {scale_w} {scale_g}', flush=True)
    dev, gy = _backward_case(12, 2, 64, 64, 11, 14)
    sign = lambda t: torch.where(t < 0, -1.0, 1.0)
    dev['input'] = sign(dev['input']) * (1 + dev['input'].abs().clamp(max=1)) * scale_x
    dev['weight'] = sign(dev['weight']) * (1 + (20 * dev['weight']).abs().clamp(max=1)) * scale_w
    gy = sign(gy) * (1 + gy.abs().clamp(max=1)) * scale_g
    got = capi_backward(dev, gy, path=capi.PATH_FUSED)
    ref = capi_backward({k: v.double() if torch.is_tensor(v) else v for k, v in dev.items()}, gy.double())
    for name, a, b in zip(('input', 'offset', 'mask', 'weight'), got, ref):
        # (a gradient below fp32's normal numbers has lost bits by itself)
        if float(b.abs().max()) < 2.0 ** -120:
            continue
        terms = 308 if name == 'weight' else 64 + 9 * 64
        assert float((a.double() - b).norm() / b.norm()) <= terms ** 0.5 * 2.0 ** -24, name
