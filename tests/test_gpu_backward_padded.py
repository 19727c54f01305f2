"""The matrix-core backward where channels are padded: segments that are no whole pass of the scatter kernel,
groups that are no multiple of 32 channels, output channels that are no multiple of 128 bytes, few tiles; all
five gradients, and the weight or data gradients alone, against the CPU oracle."""
import pytest
import torch

import oracle
from mmcv_amd import capi
from common import TOL, capi_backward, cast_case, make_case, rel_err

pytestmark = pytest.mark.gpu

CASES = [
    ('seg1_dg3', dict(N=1, Cin=3, Cout=2, H=9, W=7, deform_groups=3)),
    ('seg4_dg8', dict(N=2, Cin=32, Cout=32, H=11, W=35, deform_groups=8)),
    ('seg8_dg8', dict(N=1, Cin=64, Cout=64, H=17, W=33, deform_groups=8)),
    ('seg20', dict(N=1, Cin=20, Cout=33, H=8, W=32)),
    ('seg48_dg2', dict(N=2, Cin=96, Cout=72, H=13, W=19, deform_groups=2)),
    ('gcd', dict(N=1, Cin=48, Cout=34, H=9, W=12, groups=2, deform_groups=3)),
    ('groups_finer', dict(N=1, Cin=40, Cout=20, H=10, W=9, groups=2)),
    ('s2', dict(N=2, Cin=24, Cout=40, H=19, W=23, stride=2)),
    ('dil2_co200', dict(N=1, Cin=40, Cout=200, H=12, W=11, dilation=2, padding=2)),
    # offsets beyond the scatter kernel's window: the window for far offsets, and past that one too
    ('far', dict(N=1, Cin=64, Cout=32, H=21, W=39, sigma=6.0)),
    ('far_s2', dict(N=1, Cin=64, Cout=32, H=37, W=69, stride=2, sigma=7.0)),
    ('one_pixel', dict(N=1, Cin=8, Cout=8, H=3, W=3, padding=0)),
]
NAMES = ('grad_input', 'grad_offset', 'grad_mask', 'grad_weight', 'grad_bias')


@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16, torch.float16], ids=['f32', 'bf16', 'f16'])
@pytest.mark.parametrize('name,kw', CASES, ids=[c[0] for c in CASES])
def test_padded_backward(name, kw, dtype):
    print(f'case={name} dtype={dtype}', flush=True)
    case = cast_case(make_case(51, **kw), dtype)
    Ho, Wo = case['offset'].shape[2:]
    gy = torch.randn(kw['N'], kw['Cout'], Ho, Wo, generator=torch.Generator().manual_seed(3)).to(dtype)
    geo = dict(stride=case['stride'], padding=case['padding'], dilation=case['dilation'],
               groups=case['groups'], deform_groups=case['deform_groups'])
    ref = oracle.backward(*[case[k].float().numpy() for k in ('input', 'offset', 'mask', 'weight')],
                          gy.float().numpy(), True, **geo)
    dev, gyd = cast_case(case, dtype, 'cuda'), gy.cuda()
    for want in (dict(), dict(want_data=False, want_bias=False), dict(want_weight=False)):
        got = capi_backward(dev, gyd, **want)
        for nm, r, o in zip(NAMES, ref, got):
            if o is None or (nm == 'grad_weight' and want.get('want_weight') is False) or (
                    nm in NAMES[:3] and want.get('want_data') is False):
                continue
            err = rel_err(o.float().cpu().numpy(), r)
            assert err <= TOL[dtype], (nm, want, err)
    # images in passes of one: the weight gradient is summed over the passes
    lib = capi.load()
    lib.mdcn_set_pass_limits(0, 1)
    try:
        got = capi_backward(dev, gyd)
    finally:
        lib.mdcn_set_pass_limits(0, 0)
    for nm, r, o in zip(NAMES, ref, got):
        assert rel_err(o.float().cpu().numpy(), r) <= TOL[dtype], nm


@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16], ids=['f32', 'bf16'])
@pytest.mark.parametrize('cin,dg,h', [(24, 1, 9), (40, 1, 9), (96, 2, 9), (200, 1, 17), (504, 1, 5), (520, 1, 9)])
def test_shares_of_passes(cin, dg, h, dtype):
    """A tile's 3, 5, 6, 25, 63 and 65 passes over the window among as many workgroups, or 32 of them: every pass is somebody's."""
    print(f'cin={cin} dg={dg} h={h} dtype={dtype}', flush=True)
    case = cast_case(make_case(55, N=1, Cin=cin, Cout=36, H=h, W=37, deform_groups=dg), dtype)
    gy = torch.randn(1, 36, h, 37, generator=torch.Generator().manual_seed(7)).to(dtype)
    geo = dict(stride=1, padding=1, dilation=1, groups=1, deform_groups=dg)
    ref = oracle.backward(*[case[k].float().numpy() for k in ('input', 'offset', 'mask', 'weight')],
                          gy.float().numpy(), True, **geo)
    for nm, r, o in zip(NAMES, ref, capi_backward(cast_case(case, dtype, 'cuda'), gy.cuda())):
        err = rel_err(o.float().cpu().numpy(), r)
        assert err <= TOL[dtype], (nm, err)


def test_padding_channels_have_no_gradient():
    """An infinity of grad_output leaves NaN in the column gradient of the padding channels (zero weights times
    infinity): what follows a segment's planes in grad_input -- here the other image's -- has none of it."""
    print('padding, not finite', flush=True)
    case = make_case(52, N=2, Cin=6, Cout=10, H=9, W=11, sigma=0.5)
    gy = torch.randn(2, 10, 9, 11, generator=torch.Generator().manual_seed(4))
    gy[0, 3, 4, 5] = float('inf')
    dev, gyd = cast_case(case, torch.float32, 'cuda'), gy.cuda()
    got, ref = capi_backward(dev, gyd), capi_backward(dev, gyd, path=capi.PATH_DIRECT)
    assert not bool(ref[0][0].isfinite().all()) and bool(ref[0][1].isfinite().all())
    for nm, a, b in zip(NAMES[:3], got, ref):
        assert torch.equal(a.isfinite(), b.isfinite()), nm
        ok = b.isfinite()
        assert float((a[ok] - b[ok]).abs().max() / b[ok].abs().max()) <= TOL[torch.float32], nm


@pytest.mark.parametrize('cin', [64, 12], ids=['whole', 'padded'])
def test_far_samples_of_what_is_not_finite(cin):
    """Samples beyond the scatter kernel's window of a pixel whose grad_output is infinite: their gradient goes to the
    corners they sample, and NaN to nobody else's."""
    print('far, not finite', flush=True)
    case = make_case(53, N=1, Cin=cin, Cout=16, H=32, W=96, sigma=0.5)
    # one output pixel samples 40 columns to the right of itself: beyond the margin of either window
    case['offset'][0, 1::2, 20, 20] += 40.0
    gy = torch.randn(1, 16, 32, 96, generator=torch.Generator().manual_seed(5))
    gy[0, 3, 20, 20] = float('inf')
    dev, gyd = cast_case(case, torch.float32, 'cuda'), gy.cuda()
    got, ref = capi_backward(dev, gyd), capi_backward(dev, gyd, path=capi.PATH_DIRECT)
    assert not bool(ref[0].isfinite().all()) and bool(ref[0][..., :40].isfinite().all())
    for nm, a, b in zip(NAMES[:3], got, ref):
        assert torch.equal(a.isfinite(), b.isfinite()), nm
        ok = b.isfinite()
        assert float((a[ok] - b[ok]).abs().max() / b[ok].abs().max()) <= TOL[torch.float32], nm


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16], ids=['bf16', 'f16'])
@pytest.mark.parametrize('name', ['few_tiles', 'seg4_dg8', 'seg20', 'seg48_dg2', 'gcd', 's2', 'far', 'far_s2', 'one_pixel'])
def test_small_16bit_gradients_are_rounded_once(name, dtype):
    """Calls of few tiles or uneven channels keep the column gradient and the sums of grad_input, grad_offset and
    grad_mask in fp32: every element is the true one, rounded once -- also in an image whose gradients are small."""
    print(f'case={name} dtype={dtype}', flush=True)
    kw = dict(CASES).get(name, dict(N=2, Cin=128, Cout=64, H=14, W=30))
    case = make_case(54, **kw)
    # quarter pixels, never on one: exact positions, and no jump of the offsets' gradient
    frac = torch.randint(1, 4, case['offset'].shape, generator=torch.Generator().manual_seed(1)) / 4
    case['offset'] = torch.floor(case['offset']) + frac
    gy = torch.randn(kw['N'], kw['Cout'], *case['offset'].shape[2:], generator=torch.Generator().manual_seed(6))
    gy[0] *= 1e-3
    dev, gyd = cast_case(case, dtype, 'cuda'), gy.to(dtype).cuda()
    got = capi_backward(dev, gyd)
    wide = {k: v.double() if torch.is_tensor(v) else v for k, v in dev.items()}
    ref = capi_backward(wide, gyd.double())
    half_ulp, tiny = (2.0 ** -8, 0.0) if dtype == torch.bfloat16 else (2.0 ** -11, 2.0 ** -25)
    for nm, a, b in zip(NAMES[:3], got, ref):
        for n in range(kw['N']):
            # (sums of cout and then up to 9 cin fp32 products: 2^-24 each of terms no larger than the image's largest sum)
            bound = b[n].abs() * half_ulp + tiny + (kw['Cout'] + 9 * kw['Cin']) * 2.0 ** -24 * b[n].abs().max()
            worst = float(((a[n].double() - b[n]).abs() / bound).max())
            assert worst <= 1.0, (nm, n, worst)


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16], ids=['bf16', 'f16'])
@pytest.mark.parametrize('name', ['few_tiles', 'one_tile', 'seg20', 's2'])
def test_small_16bit_gradients_beside_a_large_one(name, dtype):
    """... and in a tile of which one pixel, its mask open, has 1e5 times the gradient of the others: what that pixel does not reach
    keeps the bits it has by itself."""
    print(f'case={name} dtype={dtype}', flush=True)
    kw = dict(CASES + [('few_tiles', dict(N=2, Cin=128, Cout=64, H=14, W=30)), ('one_tile', dict(N=1, Cin=64, Cout=128, H=8, W=17))])[name]
    case = make_case(58, **kw)
    frac = torch.randint(1, 4, case['offset'].shape, generator=torch.Generator().manual_seed(1)) / 4
    case['offset'] = torch.floor(case['offset']) + frac
    gy = torch.randn(kw['N'], kw['Cout'], *case['offset'].shape[2:], generator=torch.Generator().manual_seed(6)) / 64
    case['mask'][0, :, 4, 4] = 1.0
    even = gy.clone()
    even[0, :, 4, 4] = 0.0
    gy[0, :, 4, 4] *= 1e5
    dev, gyd = cast_case(case, dtype, 'cuda'), gy.to(dtype).cuda()
    got = capi_backward(dev, gyd)[0].double()
    wide = {k: v.double() if torch.is_tensor(v) else v for k, v in dev.items()}
    ref, alone = (capi_backward(wide, v.to(dtype).double().cuda())[0] for v in (gy, even))
    far = ref == alone   # elements that the pixel does not reach
    assert far.sum() > far.numel() // 2
    half_ulp, tiny = (2.0 ** -8, 0.0) if dtype == torch.bfloat16 else (2.0 ** -11, 2.0 ** -25)
    # (sums of cout fp32 products: 2^-24 each of terms no larger than the largest of these sums)
    bound = ref.abs() * half_ulp + tiny + (kw['Cout'] + 9 * kw['Cin']) * 2.0 ** -24 * ref[far].abs().max()
    worst = float(((got - ref).abs() / bound)[far].max())
    print(worst, flush=True)
    assert worst <= 1.0, worst


@pytest.mark.parametrize('cin,groups', [(40, 1), (24, 2), (6, 1)])
def test_stale_workspace(cin, groups):
    """Nothing depends on what the workspace held: not the results, and not the way they are computed either (fp32 sums
    that meet a NaN are computed again with other roundings)."""
    print(f'cin={cin} groups={groups}', flush=True)
    dev = cast_case(make_case(55, N=2, Cin=cin, Cout=20, H=13, W=18, groups=groups), torch.float32, 'cuda')
    gy = torch.randn(2, 20, 13, 18, generator=torch.Generator().manual_seed(8)).cuda()
    zeros, nans = capi_backward(dev, gy, ws_fill=0), capi_backward(dev, gy, ws_fill=255)
    assert torch.equal(zeros[3], nans[3]) and bool(nans[3].isfinite().all())
    for a, b in zip(zeros[1:3], nans[1:3]):
        assert torch.equal(a, b)


@pytest.mark.parametrize('count', [1, 2, 3, 5, 8, 9, 17, 63, 64])
@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16], ids=['f32', 'bf16'])
@pytest.mark.parametrize('name,kw', [
    ('8ch', dict(Cin=64)),
    ('8ch_padded', dict(Cin=20)),
    ('4ch', dict(Cin=64, stride=2)),
    ('4ch_padded', dict(Cin=6, deform_groups=1)),
], ids=['8ch', '8ch_padded', '4ch', '4ch_padded'])
def test_samples_beyond_the_window(name, kw, dtype, count):
    """`count` of the 64 pixels of every second wavefront's two rows sample 40 columns away, beyond either window: groups of samples
    that go to memory together, full and not, and many enough of them that the window for far offsets is used."""
    print(f'case={name} dtype={dtype} count={count}', flush=True)
    s = kw.get('stride', 1)
    case = make_case(55, N=1, Cout=24, H=15 * s + 1, W=95 * s + 1, sigma=0.0, **{k: v for k, v in kw.items()})
    off = case['offset']
    off += 0.25
    px = torch.randperm(64, generator=torch.Generator().manual_seed(count))[:count]
    for y0 in range(0, off.shape[2] - 1, 4):
        off[0, 1::2, y0 + px // 32, px % 32] += 40.0
    gy = torch.randn(1, 24, *off.shape[2:], generator=torch.Generator().manual_seed(7))
    dev, gyd = cast_case(case, dtype, 'cuda'), gy.to(dtype).cuda()
    ref = capi_backward({k: v.double() if torch.is_tensor(v) else v for k, v in dev.items()}, gyd.double())
    got = capi_backward(dev, gyd)
    # 16 bits: one rounding, of root mean square 0.42 of the unit roundoff; fp32: products of 24 terms and sums of some tens of them,
    # each rounded, 2^-24 sqrt(100)
    limit = 10 * 2.0 ** -24 if dtype == torch.float32 else 0.5 * 2.0 ** -8
    for nm, r, o in zip(NAMES[:3], ref, got):
        err = float((o.double() - r).norm() / r.norm())
        assert err <= limit, (nm, err)


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16], ids=['bf16', 'f16'])
def test_large_plane_of_uneven_channels(dtype):
    """An image whose fp32 column gradient is larger than its columns may be (1.5 GiB) has the matrix cores all the same."""
    print(f'large plane dtype={dtype}', flush=True)
    case = make_case(56, N=1, Cin=96, Cout=16, H=720, W=1280)
    frac = torch.randint(1, 4, case['offset'].shape, generator=torch.Generator().manual_seed(1)) / 4
    case['offset'] = torch.floor(case['offset']) + frac   # quarter pixels: exact positions in either type
    gy = torch.randn(1, 16, 720, 1280, generator=torch.Generator().manual_seed(9))
    dev, gyd = cast_case(case, dtype, 'cuda'), gy.to(dtype).cuda()
    got = capi_backward(dev, gyd)
    ref = capi_backward({k: v.double() if torch.is_tensor(v) else v for k, v in dev.items()}, gyd.double())
    u = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    # root mean square of one rounding: 0.42 of the unit roundoff; of two -- grad_weight's columns are rounded -- 0.6
    for nm, r, o, share in zip(NAMES, ref, got, (0.5, 0.5, 0.5, 0.7, 1.0)):
        err = float((o.double() - r).norm() / r.norm())
        assert err <= share * u, (nm, err)


@pytest.mark.parametrize('dtype,n,h,w', [(torch.float32, 1, 100, 103), (torch.bfloat16, 4, 92, 100), (torch.float16, 2, 90, 100)],
                         ids=['f32', 'bf16', 'f16'])
def test_large_products(dtype, n, h, w):
    """Just above the sizes from which the products run in tiles of 256 (2 898 and 5 184 K steps for the weight gradient of fp32 and
    bf16, 648 tiles of the fp16 column gradient), channels uneven.  fp32 sums of up to 10 300 products: 1e-5 of the norm; 16 bits: one
    rounding of the result and one of the columns."""
    print(f'dtype={dtype} n={n}', flush=True)
    dev = cast_case(make_case(57, N=n, Cin=232, Cout=200, H=h, W=w), dtype, 'cuda')
    gy = torch.randn(n, 200, h, w, generator=torch.Generator().manual_seed(9)).to(dtype).cuda()
    ref = capi_backward({k: v.double() if torch.is_tensor(v) else v for k, v in dev.items()}, gy.double())
    for nm, r, o in zip(NAMES, ref, capi_backward(dev, gy)):
        err = float((o.double() - r).norm() / r.norm())
        assert err <= {torch.float32: 1e-5, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype], (nm, err)


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16], ids=['bf16', 'f16'])
def test_large_products_of_uneven_rows(dtype):
    """The same with rows of the products that fill the last tile of 256 to seven eighths (9 x 224): 5 760 K steps and 1 440 tiles."""
    print(f'dtype={dtype}', flush=True)
    dev = cast_case(make_case(59, N=5, Cin=224, Cout=200, H=92, W=100), dtype, 'cuda')
    gy = torch.randn(5, 200, 92, 100, generator=torch.Generator().manual_seed(10)).to(dtype).cuda()
    ref = capi_backward({k: v.double() if torch.is_tensor(v) else v for k, v in dev.items()}, gy.double())
    for nm, r, o in zip(NAMES, ref, capi_backward(dev, gy)):
        err = float((o.double() - r).norm() / r.norm())
        assert err <= {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype], (nm, err)
