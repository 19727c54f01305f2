"""conv_offset inside the library: the tiled kernel's forms, at the edges of its tiles, stages and weight ring."""
import pytest
import torch

from common import capi_pack_forward, cast_pack_case, make_pack_case

pytestmark = pytest.mark.gpu

# (N, Cin, H, W, options): several rows per workgroup (a call that fills the chip) and one, one slab at a time and
# several, a last stage that is not full, 27 to 108 channels, rings of 9 and 3 taps with remainders
CASES = {
    'rows4': (8, 64, 126, 97, {}),
    'rows4_two_slabs': (9, 128, 125, 96, {}),
    'rows4_stride2': (9, 64, 250, 190, dict(stride=2)),
    'rows2_36ch': (8, 128, 67, 129, dict(deform_groups=2)),
    'rows2_108ch': (8, 256, 66, 70, dict(deform_groups=4)),
    'row1_stages': (1, 1024, 33, 33, {}),
    'row1_two_per_cu': (5, 512, 34, 65, {}),
    'row1_5x5': (1, 320, 20, 31, dict(k=5, padding=2)),
    'row1_108ch_stride2': (2, 512, 31, 35, dict(deform_groups=4, stride=2)),
    'row1_1x4_dil3': (1, 128, 9, 40, dict(k=(1, 4), padding=(0, 5), dilation=3)),
}


@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16, torch.float16], ids=['f32', 'bf16', 'f16'])
@pytest.mark.parametrize('name', CASES)
def test_conv_offset_alone(name, dtype):
    n, cin, h, w, kw = CASES[name]
    case = cast_pack_case(make_pack_case(31, N=n, Cin=cin, Cout=64, H=h, W=w, **kw), dtype)
    _, raw = capi_pack_forward(cast_pack_case(case, dtype, 'cuda'), own_conv=True, want_raw=True)
    ref = torch.nn.functional.conv2d(case['input'].double(), case['offset_weight'].double(),
                                     case['offset_bias'].double(), case['stride'], case['padding'], case['dilation'])
    err = (raw.cpu().double() - ref).abs().max() / ref.abs().max()
    # one rounding of the result (8, 11 or 24 bits of a value in [1, 2): half of the last), and fp32 sums: 2^-24 each,
    # sqrt(terms) of them, five of their deviations
    terms = cin * case['offset_weight'].shape[2] * case['offset_weight'].shape[3]
    rounding = 2.0 ** {torch.float32: -24, torch.bfloat16: -8, torch.float16: -11}[dtype]
    assert float(err) <= rounding + 5 * terms ** 0.5 * 2.0 ** -24
