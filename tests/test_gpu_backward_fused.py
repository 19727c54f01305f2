"""The 16-bit backward in one kernel (bwd_fused_kernel) where it can go wrong: edges of its tiles, chunks of output channels
that are not full, eight channels a pass, odd numbers of taps, cut tiles beside whole rounds of them, offsets beyond either
window; all gradients against the same call in double precision."""
import pytest
import torch

from mmcv_amd import capi
from common import capi_backward, cast_case, make_case

pytestmark = pytest.mark.gpu

CASES = [
    ('one_tile', dict(N=1, Cin=64, Cout=64, H=16, W=16)),
    ('edges_w32', dict(N=2, Cin=64, Cout=128, H=7, W=65)),
    ('edges_w16', dict(N=1, Cin=128, Cout=64, H=17, W=33)),
    ('k192', dict(N=1, Cin=64, Cout=192, H=15, W=18)),
    ('k320', dict(N=1, Cin=64, Cout=320, H=9, W=31)),
    ('k448', dict(N=1, Cin=64, Cout=448, H=10, W=37)),
    ('k512', dict(N=1, Cin=128, Cout=512, H=13, W=21)),
    ('k640_8ch', dict(N=1, Cin=64, Cout=640, H=11, W=20, deform_groups=8)),
    ('8ch', dict(N=1, Cin=192, Cout=64, H=18, W=17, deform_groups=8)),
    ('groups', dict(N=2, Cin=128, Cout=256, H=12, W=34, groups=2, deform_groups=2)),
    ('group_in_dg', dict(N=1, Cin=128, Cout=128, H=12, W=20, groups=2)),
    ('k1x1', dict(N=1, Cin=64, Cout=64, H=20, W=20, k=(1, 1), padding=0)),
    ('k1x3', dict(N=1, Cin=64, Cout=64, H=9, W=40, k=(1, 3), padding=(0, 1))),
    ('k2x2', dict(N=1, Cin=64, Cout=64, H=19, W=23, k=(2, 2))),
    ('s2', dict(N=2, Cin=64, Cout=64, H=37, W=69, stride=2)),
    ('dil3', dict(N=1, Cin=64, Cout=64, H=24, W=26, dilation=3, padding=3)),
    ('far', dict(N=1, Cin=64, Cout=64, H=40, W=45, sigma=6.0)),
    ('far_s2', dict(N=1, Cin=128, Cout=64, H=60, W=75, stride=2, sigma=9.0)),
    ('past_far', dict(N=1, Cin=64, Cout=64, H=50, W=55, sigma=20.0)),
    # (more than 128 output channels: up to a share of 1/11 beyond the margin of 7 or 8 the first window is used)
    ('k256_first_window', dict(N=1, Cin=64, Cout=256, H=40, W=45, sigma=4.0)),
    ('k256_far', dict(N=1, Cin=64, Cout=256, H=40, W=45, sigma=5.5)),
    ('rounds', dict(N=2, Cin=64, Cout=64, H=190, W=194, sigma=1.5)),   # 36 or 37 tiles per XCD: a round, and cut ones
]
NAMES = ('grad_input', 'grad_offset', 'grad_mask', 'grad_weight', 'grad_bias')
#: Unit roundoff: the largest relative error of one rounding.  Over many values its root mean square is 0.42 of that (an error
#: uniform within a last place, values spread over their binade), and two independent ones -- the columns are rounded before they
#: are summed -- add up to 0.6; 0.5 and 0.7 leave room for what else there is, and not for another rounding.  grad_bias has too few
#: values for a mean.
U = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}
SHARE = dict(grad_input=0.5, grad_offset=0.5, grad_mask=0.5, grad_weight=0.7, grad_bias=1.0)


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16], ids=['bf16', 'f16'])
@pytest.mark.parametrize('name,kw', CASES, ids=[c[0] for c in CASES])
def test_fused_backward(name, kw, dtype):
    print(f'case={name} dtype={dtype}', flush=True)
    dev = cast_case(make_case(71, **kw), dtype, 'cuda')
    Ho, Wo = dev['offset'].shape[2:]
    gy = torch.randn(kw['N'], kw['Cout'], Ho, Wo, generator=torch.Generator().manual_seed(4)).to(dtype).cuda()
    for modulated in (True, False):
        case = dict(dev) if modulated else dict(dev, mask=None)
        ref = capi_backward({k: v.double() if torch.is_tensor(v) else v for k, v in case.items()}, gy.double())
        for want in (dict(), dict(want_weight=False)):
            got = capi_backward(case, gy, path=capi.PATH_FUSED, **want)
            for nm, r, o in zip(NAMES, ref, got):
                if o is None or (nm == 'grad_weight' and not want.get('want_weight', True)):
                    continue
                err = float((o.double() - r).norm() / r.norm())
                assert err <= U[dtype] * SHARE[nm], (nm, modulated, want, err)
    # the shares of a tile are added up in a fixed order, and integers in any: two runs differ by the order of the adds to memory
    # alone, which is grad_input's
    again = capi_backward(dev, gy, path=capi.PATH_FUSED)
    first = capi_backward(dev, gy, path=capi.PATH_FUSED)
    for nm, a, b in zip(NAMES[1:], again[1:], first[1:]):
        assert torch.equal(a, b), nm


# Output channels whose weights and gradients differ in magnitude: (how many, weight's factor, gradient's factor).  A filter that
# has died in front of a normalisation layer has weights of zero and a gradient hundreds of times the others'.
UNEVEN = [
    ('one_dead_100', 1, 0.0, 100.0),
    ('one_dead_300', 1, 0.0, 300.0),
    ('four_dead_300', 4, 0.0, 300.0),
    ('one_small', 1, 2.0 ** -9, 300.0),
    ('one_large', 1, 300.0, 2.0 ** -9),
    ('most_dead', 250, 0.0, 300.0),
    ('powers', 256, 1.0, 1.0),   # each channel's weights by a power of two, its gradient by the inverse
]


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16], ids=['bf16', 'f16'])
@pytest.mark.parametrize('name,count,fw,fg', UNEVEN, ids=[c[0] for c in UNEVEN])
def test_uneven_channels(name, count, fw, fg, dtype):
    """The window's quantum goes by the column gradient itself: grad_input stays within its one rounding whatever
    the parts of grad_output that the weights do not carry into it are."""
    print(f'case={name} dtype={dtype}', flush=True)
    case = make_case(73, N=1, Cin=64, Cout=256, H=33, W=40)
    gy = torch.randn(1, 256, 33, 40, generator=torch.Generator().manual_seed(6))
    case['weight'][:count] *= fw
    gy[:, :count] *= fg
    if name == 'powers':
        by = 2.0 ** torch.randint(-6, 7, (count, 1, 1, 1), generator=torch.Generator().manual_seed(7))
        case['weight'] *= by
        gy /= by.transpose(0, 1)
    dev, gy = cast_case(case, dtype, 'cuda'), gy.to(dtype).cuda()
    for modulated in (True, False):
        call = dict(dev) if modulated else dict(dev, mask=None)
        ref = capi_backward({k: v.double() if torch.is_tensor(v) else v for k, v in call.items()}, gy.double())
        got = capi_backward(call, gy, path=capi.PATH_FUSED)
        for nm, r, o in zip(NAMES, ref, got):
            if o is not None:
                err = float((o.double() - r).norm() / r.norm())
                print(nm, modulated, err, flush=True)
                assert err <= U[dtype] * SHARE[nm], (nm, modulated, err)


# Pixels whose gradients are large where their mask is next to nothing: (how many, gradient's factor, mask there).
CLOSED = [('one_1e3_zero', 1, 1e3, 0.0), ('one_8e3_2^-10', 1, 8e3, 2.0 ** -10), ('row_300_zero', 40, 300.0, 0.0),
          ('one_1e2_negative', 1, 1e2, -2.0 ** -9)]


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16], ids=['bf16', 'f16'])
@pytest.mark.parametrize('name,count,fg,mask', CLOSED, ids=[c[0] for c in CLOSED])
def test_closed_gates(name, count, fg, mask, dtype):
    """The window's quantum goes by what is added to it, the column gradient times the mask of the same sample: a large gradient
    under a small mask, or where nothing is sampled, takes no bits from the tile's other pixels."""
    print(f'case={name} dtype={dtype}', flush=True)
    case = make_case(75, N=1, Cin=64, Cout=128, H=33, W=40)
    gy = torch.randn(1, 128, 33, 40, generator=torch.Generator().manual_seed(9))
    gy[:, :, 20, :count] *= fg
    case['mask'][:, :, 20, :count] = mask
    gy[:, :, 9, 7] *= fg   # (all of its samples beyond the image)
    case['offset'][:, :, 9, 7] = 1e4
    dev, gy = cast_case(case, dtype, 'cuda'), gy.to(dtype).cuda()
    ref = capi_backward({k: v.double() if torch.is_tensor(v) else v for k, v in dev.items()}, gy.double())[0]
    got = capi_backward(dev, gy, path=capi.PATH_FUSED)[0].double()
    err = float((got - ref).norm() / ref.norm())
    print(err, flush=True)
    assert err <= U[dtype] * SHARE['grad_input'], err


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16], ids=['bf16', 'f16'])
@pytest.mark.parametrize('mask,e', [(0.25, 20), (2.0 ** -4, 24)], ids=['within_3_bits', 'beyond'])
def test_quantum(mask, e, dtype):
    """The window's quantum, bit for bit: 2^-20 of the largest |d| times the largest mask, wherever each of them is, and of the largest
    product of the two only where that gives three bits or more."""
    print(f'mask={mask} dtype={dtype}', flush=True)
    # 1x1 kernel, weights of one, integer positions: the column gradient is grad_output, a pixel has one contribution
    case = make_case(77, N=1, Cin=64, Cout=64, H=16, W=16, k=(1, 1), padding=0)
    case['weight'] = torch.eye(64).reshape(64, 64, 1, 1)
    case['offset'].zero_()
    case['mask'].fill_(0.25)
    case['mask'][0, 0, 5, 6], case['mask'][0, 0, 11, 3] = 1.0, mask
    gy = torch.randn(1, 64, 16, 16, generator=torch.Generator().manual_seed(11)) * 2.0 ** -14
    gy[0, ::8, 11, 3] = 1.0   # (in every pass's channels)
    dev, gy = cast_case(case, dtype, 'cuda'), gy.to(dtype).cuda()
    got = capi_backward(dev, gy, path=capi.PATH_FUSED)[0]
    ref = torch.round(gy.double() * dev['mask'].double() * 2.0 ** e) * 2.0 ** -e
    assert torch.equal(got, ref.to(dtype)), float((got.double() - ref).abs().max() * 2.0 ** e)


@pytest.mark.parametrize('groups', [1, 8], ids=['16ch', '8ch'])
def test_large_gradients_where_nothing_is_sampled(groups):
    """A sample beyond the image has gradients of zero, whatever the column gradient there times a corner of the image is."""
    print(f'groups={groups}', flush=True)
    case = make_case(76, N=1, Cin=64, Cout=64, H=33, W=40, deform_groups=groups)
    gy = torch.randn(1, 64, 33, 40, generator=torch.Generator().manual_seed(10))
    gy[:, :, 9, 7] *= 1e37
    case['offset'][:, :, 9, 7] = 1e4
    case['input'][:, :, :2, :2] *= 1e3
    dev, gy = cast_case(case, torch.bfloat16, 'cuda'), gy.bfloat16().cuda()
    ref = capi_backward({k: v.double() if torch.is_tensor(v) else v for k, v in dev.items()}, gy.double())
    got = capi_backward(dev, gy, path=capi.PATH_FUSED)
    for nm, r, o in zip(NAMES[:4], ref, got):   # (grad_bias: a sum of gradients up to 1e38)
        assert bool(o.isfinite().all()), nm
        err = float((o.double() - r).norm() / r.norm())
        assert err <= U[torch.bfloat16] * SHARE[nm], (nm, err)
    assert not bool(got[1][:, :, 9, 7].any()) and not bool(got[2][:, :, 9, 7].any())


@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16, torch.float16], ids=['f32', 'bf16', 'f16'])
@pytest.mark.parametrize('cin,path', [(64, capi.PATH_FUSED), (40, capi.PATH_AUTO)], ids=['whole', 'uneven'])
def test_corner_pixel_that_nobody_samples(cin, path, dtype):
    """An infinity in the image's first pixel, and samples beyond the image, but none of that pixel: no gradient has it."""
    print(f'cin={cin} dtype={dtype}', flush=True)
    case = make_case(78, N=2, Cin=cin, Cout=64, H=17, W=40)
    case['offset'] = 3.0 + torch.randint(1, 4, case['offset'].shape, generator=torch.Generator().manual_seed(12)) / 4
    case['offset'][:, :, 9, 7] = 1e4
    gy = torch.randn(2, 64, 17, 40, generator=torch.Generator().manual_seed(13))
    dev, gy = cast_case(case, dtype, 'cuda'), gy.to(dtype).cuda()
    bad = dict(dev, input=dev['input'].clone())
    bad['input'][:, :, 0, 0] = float('inf')
    for want in (dict(), dict(want_data=False)):
        ref, got = capi_backward(dev, gy, path=path, **want), capi_backward(bad, gy, path=path, **want)
        for nm, a, b in zip(NAMES[1:], got[1:], ref[1:]):   # (grad_input is summed in no order, and the image has no part in it)
            assert torch.equal(a, b), (nm, want)


def test_passes_of_images():
    """Cut tiles of several passes of images, the last one of another size, have places of their own for their shares."""
    kw = dict(N=5, Cin=64, Cout=64, H=33, W=47)
    dev = cast_case(make_case(72, **kw), torch.bfloat16, 'cuda')
    gy = torch.randn(5, 64, 33, 47, generator=torch.Generator().manual_seed(5)).bfloat16().cuda()
    whole = capi_backward(dev, gy, path=capi.PATH_FUSED)
    lib = capi.load()
    lib.mdcn_set_pass_limits(0, 2 * 9 * 64 * 33 * 47 * 2)   # two images' columns
    try:
        parts = capi_backward(dev, gy, path=capi.PATH_FUSED)
    finally:
        lib.mdcn_set_pass_limits(0, 0)
    # the offsets' sums are cut at other channels: fp32 sums in another order, which round to a neighbour now and then
    for nm, a, b in zip(NAMES, whole, parts):
        assert float((a.double() - b.double()).norm() / a.double().norm()) <= 0.1 * U[torch.bfloat16], nm


# 5 to 8 taps: as few loads behind the copies of the next pass's weights as there are where items are skipped.
FEW_TAPS = [
    ('k1x5', dict(k=(1, 5), padding=(0, 2))),
    ('k2x3', dict(k=(2, 3), padding=1)),
    ('k1x7', dict(k=(1, 7), padding=(0, 3))),
    ('k2x4', dict(k=(2, 4), padding=1)),
]


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16], ids=['bf16', 'f16'])
@pytest.mark.parametrize('ch', [16, 8])
@pytest.mark.parametrize('cout', [64, 128])
@pytest.mark.parametrize('name,kw', FEW_TAPS, ids=[c[0] for c in FEW_TAPS])
def test_five_to_eight_taps(name, kw, cout, ch, dtype):
    """Many passes of few taps, 16 and 8 channels a pass, with columns and without."""
    print(f'case={name} cout={cout} ch={ch} dtype={dtype}', flush=True)
    # (segments of 24 channels make passes of 8)
    shape = dict(N=1, Cin=128 if ch == 16 else 192, Cout=cout, H=21, W=37, deform_groups=1 if ch == 16 else 8)
    dev = cast_case(make_case(74, **shape, **kw), dtype, 'cuda')
    gy = torch.randn(1, cout, *dev['offset'].shape[2:], generator=torch.Generator().manual_seed(8)).to(dtype).cuda()
    ref = capi_backward({k: v.double() if torch.is_tensor(v) else v for k, v in dev.items()}, gy.double())
    for want in (dict(), dict(want_weight=False)):
        got = capi_backward(dev, gy, path=capi.PATH_FUSED, **want)
        for nm, r, o in zip(NAMES, ref, got):
            if o is None or (nm == 'grad_weight' and not want.get('want_weight', True)):
                continue
            err = float((o.double() - r).norm() / r.norm())
            assert err <= U[dtype] * SHARE[nm], (nm, want, err)
