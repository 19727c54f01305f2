"""The Pack layers in training, conv_offset's backward inside the library, against that backward in torch in double precision
and the same deformable convolution."""
import pytest
import torch
import torch.nn as nn

pytestmark = pytest.mark.gpu

# unit roundoff of the element type
ROUND = {torch.float32: 2.0**-24, torch.float16: 2.0**-11, torch.bfloat16: 2.0**-8}

# (N, Cin, Cout, H, W, kernel, stride, padding, dilation, deformable groups)
SHAPES = [
    (2, 64, 64, 9, 33, 3, 1, 1, 1, 1),      # one pixel past a run of 32 columns, one row past a tile
    (1, 64, 32, 5, 5, 3, 1, 1, 1, 1),       # smaller than a tile
    (3, 128, 64, 16, 64, 3, 1, 1, 1, 1),    # whole tiles
    (2, 64, 64, 19, 41, 3, 2, 1, 1, 1),     # stride: odd sizes, rows and columns that no tap meets
    (1, 64, 64, 14, 37, 3, 3, 0, 1, 1),
    (1, 64, 64, 23, 29, 3, 1, 4, 4, 1),     # dilation
    (1, 192, 64, 7, 35, 1, 1, 0, 1, 1),     # one tap, three blocks a workgroup
    (1, 64, 64, 12, 34, 5, 1, 2, 1, 1),     # 25 taps: three groups of them
    (2, 256, 64, 10, 21, 3, 1, 1, 1, 4),    # 108 channels of conv_offset
    (8, 128, 128, 64, 96, 3, 1, 1, 1, 1),   # eight rows a workgroup in the data kernel
    (8, 128, 128, 64, 96, 3, 2, 1, 1, 2),
]


def _layer(cls, shape, dtype):
    n, ci, co, h, w, k, s, p, d, dg = shape
    torch.manual_seed(7)
    layer = cls(ci, co, k, stride=s, padding=p, dilation=d, deform_groups=dg, bias=False).cuda()
    with torch.no_grad():
        layer.conv_offset.weight.normal_(0, 0.5 / (ci * k * k)**0.5)
        layer.conv_offset.bias.uniform_(-0.5, 0.5)
    x = torch.randn(n, ci, h, w, device='cuda')
    return layer.to(dtype), x.to(dtype)


def _step(layer, x, go=None, **kw):
    x = x.detach().requires_grad_(True)
    y = layer(x)
    if go is None:
        go = torch.randn_like(y)
    names = [x] + list(layer.parameters())
    return y.detach(), go, torch.autograd.grad(y, names, go)


@pytest.mark.parametrize('dtype', ROUND, ids=lambda d: str(d)[6:])
@pytest.mark.parametrize('shape', SHAPES, ids=lambda s: 'x'.join(map(str, s)))
@pytest.mark.parametrize('modulated', [True, False], ids=['dcnv2', 'dcnv1'])
def test_against_torch_convolution(monkeypatch, modulated, shape, dtype):
    from mmcv_amd.ops import DeformConv2dPack, ModulatedDeformConv2dPack
    import mmcv_amd.ops.modulated_deform_conv as mdc
    monkeypatch.setattr(torch.backends.cudnn, 'deterministic', True)  # conv_offset's forward runs twice
    layer, x = _layer(ModulatedDeformConv2dPack if modulated else DeformConv2dPack, shape, dtype)
    calls = []
    real = mdc.ext_module.pack_train_call

    class Spy:
        def __getattr__(self, name):
            return getattr(ext, name)

        def pack_train_call(self, *a):
            out = real(*a)
            calls.append(out is not None)
            return out

    ext = mdc.ext_module
    import mmcv_amd.ops.deform_conv as dc
    monkeypatch.setattr(mdc, 'ext_module', Spy())
    monkeypatch.setattr(dc, 'ext_module', Spy())
    y, go, got = _step(layer, x)
    assert calls == [True]

    # The same layer step by step: offset and mask from the same conv_offset, their gradients as tensors of the type, the
    # gradients that these give conv_offset in double precision
    weight = layer.weight.detach().requires_grad_(True)
    x0 = x.detach().requires_grad_(True)
    raw = layer.conv_offset(x).detach()
    n_off = raw.shape[1] * 2 // 3 if modulated else raw.shape[1]
    off = raw[:, :n_off].contiguous().requires_grad_(True)
    geo = (layer.stride, layer.padding, layer.dilation, layer.groups, layer.deform_groups)
    if modulated:
        mask = torch.sigmoid(raw[:, n_off:]).requires_grad_(True)
        y0 = mdc.modulated_deform_conv2d(x0, off, mask, weight, None, *geo)
        gx, goff, gmask, gw = torch.autograd.grad(y0, (x0, off, mask, weight), go)
        m = mask.detach()
        graw = torch.cat([goff, (gmask.float() * (1 - m.float()) * m.float()).to(dtype)], 1).double()
    else:
        y0 = dc.deform_conv2d(x0, off, weight, *geo)
        gx, goff, gw = torch.autograd.grad(y0, (x0, off, weight), go)
        graw = goff.double()
    assert torch.equal(y, y0)

    def conv_grads(x, w, g):
        """(of input, weight, bias; the bias' value does not matter)"""
        leaves = [t.detach().requires_grad_(True) for t in (x, w, w.new_zeros(w.shape[0]))]
        out = torch.nn.functional.conv2d(*leaves, layer.conv_offset.stride, layer.conv_offset.padding,
                                         layer.conv_offset.dilation)
        return torch.autograd.grad(out, leaves, g)

    x64, w64 = x.double(), layer.conv_offset.weight.detach().double()
    want = conv_grads(x64, w64, graw)
    scale = conv_grads(x64.abs(), w64.abs(), graw.abs())  # of each sum: that of its terms' absolute values
    names = dict(zip(['x'] + [n for n, _ in layer.named_parameters()], got))
    gx, u32 = gx.double(), 2.0**-24

    # A sum of K products in fp32 is off by K u32 of its scale at most (of four pixels' sums of a bias more than that is
    # never reached), its rounding to the type by one rounding of itself.  The input's gradient also has the convolution's, which
    # comes rounded once and, a sum of atomics, differs by 1e-5 of its largest between two runs: one rounding more.
    def close(a, want, bound, what):
        err = (a.double() - want).abs()
        assert torch.isfinite(a).all() and bool((err <= bound).all()), (what, float((err / bound).max()))

    px = raw.shape[0] * raw.shape[2] * raw.shape[3]
    kx = raw.shape[1] * layer.weight.shape[2] * layer.weight.shape[3]
    u = ROUND[dtype]
    tiny = 2.0**-24 if dtype == torch.float16 else 1e-30  # (below the normal numbers)
    close(names['conv_offset.weight'], want[1], u * want[1].abs() + px * u32 * scale[1] + tiny, 'conv_offset.weight')
    close(names['conv_offset.bias'], want[2], u * want[2].abs() + px * u32 * scale[2] + tiny, 'conv_offset.bias')
    total = gx + want[0]
    close(names['x'], total, u * (2 * gx.abs() + 1.01 * total.abs()) + kx * u32 * scale[0] + 1e-5 * gx.abs().max() + tiny, 'x')
    close(names['weight'], gw.double(), 2 * u * gw.double().abs() + 1e-5 * gw.double().abs().max(), 'weight')


def test_gradients_that_are_asked_for():
    """Every subset gives what the whole gives (sums of atomics aside)."""
    from mmcv_amd.ops import ModulatedDeformConv2dPack
    layer, x = _layer(ModulatedDeformConv2dPack, SHAPES[0], torch.float32)
    _, go, want = _step(layer, x)
    names = ['x'] + [n for n, _ in layer.named_parameters()]
    want = dict(zip(names, want))
    for take in (['x'], ['weight'], ['conv_offset.weight'], ['conv_offset.bias'], ['x', 'conv_offset.bias'],
                 ['weight', 'conv_offset.weight']):
        x1 = x.detach().requires_grad_('x' in take)
        for n, p in layer.named_parameters():
            p.requires_grad_(n in take)
        leaves = [x1 if n == 'x' else dict(layer.named_parameters())[n] for n in take]
        for n, g in zip(take, torch.autograd.grad(layer(x1), leaves, go)):
            assert float((g - want[n]).abs().max()) <= 1e-5 * float(want[n].abs().max()), (take, n)


@pytest.mark.parametrize('form', ['channels_last', 'weights_channels_last', 'slice', 'transposed', 'gradient_expanded',
                                  'gradient_transposed', 'unaligned', 'saved_on_cpu', 'no_offset_bias', 'other_stream'])
def test_forms(monkeypatch, form):
    """Orders and strides of what a call is given, against the layer's own sequence of operations."""
    import contextlib
    from mmcv_amd.ops import ModulatedDeformConv2dPack
    monkeypatch.setattr(torch.backends.cudnn, 'deterministic', True)
    layer, x = _layer(ModulatedDeformConv2dPack, (2, 64, 48, 11, 13, 3, 1, 1, 1, 1), torch.float32)
    go = torch.randn(2, 48, 11, 13, device='cuda')
    if form == 'channels_last':
        x = x.to(memory_format=torch.channels_last)
    elif form == 'weights_channels_last':
        layer = layer.to(memory_format=torch.channels_last)
    elif form == 'slice':
        x = torch.randn(2, 70, 14, 13, device='cuda')[:, 3:67, 2:13]
    elif form == 'transposed':
        x = x.transpose(2, 3).contiguous().transpose(2, 3)
    elif form == 'gradient_expanded':
        go = torch.randn(1, 48, 1, 1, device='cuda').expand(2, 48, 11, 13)
    elif form == 'gradient_transposed':
        go = go.transpose(2, 3).contiguous().transpose(2, 3)
    elif form == 'unaligned':
        x = torch.randn(x.numel() + 1, device='cuda')[1:].view(x.shape)
    elif form == 'no_offset_bias':
        layer.conv_offset.bias = None
    assert form != 'slice' or not x.is_contiguous()
    got = []
    for fuse in ('none', 'full'):
        layer.fuse = fuse
        stream = torch.cuda.Stream() if form == 'other_stream' else torch.cuda.current_stream()
        stream.wait_stream(torch.cuda.current_stream())
        hooks = torch.autograd.graph.save_on_cpu() if form == 'saved_on_cpu' else contextlib.nullcontext()
        with torch.cuda.stream(stream), hooks:
            x1 = x.detach().requires_grad_(True)
            y = layer(x1)
            names = [x1] + list(layer.parameters())
            grads = torch.autograd.grad(y, names, go)
        torch.cuda.synchronize()
        got.append((y.detach(),) + grads)
    assert torch.equal(got[0][0], got[1][0])
    for a, b in zip(*got):  # (sums in fp32 of up to 1 728 terms, in other orders)
        assert a.shape == b.shape and float((a - b).abs().max()) <= 1e-5 * float(a.abs().max())


def test_second_derivative_raises():
    from mmcv_amd.ops import ModulatedDeformConv2dPack
    layer, x = _layer(ModulatedDeformConv2dPack, SHAPES[0], torch.float32)
    x = x.requires_grad_(True)
    (g,) = torch.autograd.grad(layer(x).square().sum(), x, create_graph=True)
    with pytest.raises(RuntimeError, match='once_differentiable'):
        g.sum().backward()


def test_calls_that_keep_the_module():
    """Whoever watches, wraps or replaces conv_offset still gets every call of it."""
    from mmcv_amd.ops import ModulatedDeformConv2dPack
    seen = []

    def fresh():
        layer, x = _layer(ModulatedDeformConv2dPack, SHAPES[0], torch.float32)
        return layer, x.requires_grad_(True)

    layer, x = fresh()
    y = layer(x)
    for hook in ('register_forward_hook', 'register_forward_pre_hook'):
        layer, x = fresh()
        getattr(layer.conv_offset, hook)(lambda *a: seen.append(hook))
        assert float((layer(x) - y).abs().max()) < 1e-3
        assert seen.pop() == hook
    layer, x = fresh()
    layer.conv_offset.register_full_backward_hook(lambda *a: seen.append('backward'))
    layer(x).sum().backward()
    assert seen.pop() == 'backward'
    layer, x = fresh()
    nn.utils.parametrizations.weight_norm(layer.conv_offset)
    layer(x).sum().backward()
    assert all(p.grad is not None for p in layer.conv_offset.parameters())
    layer, x = fresh()
    inner = layer.conv_offset._conv_forward
    layer.conv_offset._conv_forward = lambda *a: (seen.append('inner'), inner(*a))[1]
    layer(x)
    assert seen.pop() == 'inner'
    layer, x = fresh()
    with torch.autocast('cuda', dtype=torch.bfloat16):
        assert layer(x).dtype == torch.bfloat16
    layer, x = fresh()
    with torch.autograd.forward_ad.dual_level(), pytest.raises(NotImplementedError):
        layer(torch.autograd.forward_ad.make_dual(x, torch.ones_like(x)))


@pytest.mark.parametrize('modulated', [True, False], ids=['dcnv2', 'dcnv1'])
def test_function_modes(monkeypatch, modulated):
    """A function mode sees the operations of a training call; the one that places new tensors does not ask for them."""
    from mmcv_amd.ops import DeformConv2dPack, ModulatedDeformConv2dPack
    import mmcv_amd.ops.deform_conv as dc
    import mmcv_amd.ops.modulated_deform_conv as mdc
    seen = []

    class Watch(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(getattr(func, '__name__', str(func)))
            return func(*args, **(kwargs or {}))

    layer, x = _layer(ModulatedDeformConv2dPack if modulated else DeformConv2dPack, SHAPES[0], torch.float32)
    x.requires_grad_(True)
    with Watch():
        layer(x)
    assert {'conv2d', 'chunk', 'cat', 'sigmoid'} <= set(seen) if modulated else 'conv2d' in seen
    module, calls = mdc if modulated else dc, []
    ext = module.ext_module

    class Spy:
        def __getattr__(self, name):
            calls.append(name)
            return getattr(ext, name)

    monkeypatch.setattr(module, 'ext_module', Spy())
    with torch.device('cuda'):
        layer(x)
    assert calls == ['pack_train_call']


@pytest.mark.parametrize('dtype,channels', [(torch.float32, 48), (torch.bfloat16, 96), (torch.float64, 64)], ids=['f32', 'bf16', 'f64'])
@pytest.mark.parametrize('modulated', [True, False], ids=['dcnv2', 'dcnv1'])
def test_uneven_channels_do_not_ask(monkeypatch, modulated, dtype, channels):
    """Channels that conv_offset's backward in the library does not cover go to the sequence of operations without a call into it.
    (Double precision is asked for and refused.)"""
    from mmcv_amd.ops import DeformConv2dPack, ModulatedDeformConv2dPack
    import mmcv_amd.ops.deform_conv as dc
    import mmcv_amd.ops.modulated_deform_conv as mdc
    module, calls = mdc if modulated else dc, []
    ext = module.ext_module

    class Spy:
        def __getattr__(self, name):
            calls.append(name)
            return getattr(ext, name)

    shape = (1, channels, 32, 9, 17, 3, 1, 1, 1, 1)
    layer, x = _layer(ModulatedDeformConv2dPack if modulated else DeformConv2dPack, shape, dtype)
    monkeypatch.setattr(module, 'ext_module', Spy())
    y, _, grads = _step(layer, x)
    assert ('pack_train_call' in calls) == (dtype == torch.float64)
    assert y.shape == (1, 32, 9, 17) and all(bool(g.isfinite().all()) for g in grads)


@pytest.mark.parametrize('which', ['weight', 'bias'])
@pytest.mark.parametrize('modulated', [True, False], ids=['dcnv2', 'dcnv1'])
def test_parameter_subclasses(modulated, which):
    """A subclass of Parameter sees the convolution it is a parameter of."""
    from mmcv_amd.ops import DeformConv2dPack, ModulatedDeformConv2dPack
    seen = []

    class Watched(nn.Parameter):
        @classmethod
        def __torch_function__(cls, func, types, args=(), kwargs=None):
            seen.append(getattr(func, '__name__', str(func)))
            with torch._C.DisableTorchFunctionSubclass():
                return func(*args, **(kwargs or {}))

    layer, x = _layer(ModulatedDeformConv2dPack if modulated else DeformConv2dPack, SHAPES[0], torch.float32)
    setattr(layer.conv_offset, which, Watched(getattr(layer.conv_offset, which).detach()))
    layer(x.requires_grad_(True)).sum().backward()
    assert 'conv2d' in seen


def test_captured_step():
    """A training step in a graph, replayed on new input."""
    from mmcv_amd.ops import ModulatedDeformConv2dPack
    layer, x = _layer(ModulatedDeformConv2dPack, SHAPES[3], torch.bfloat16)
    static = x.clone()
    _, go, _ = _step(layer, static)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        _step(layer, static, go)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y, _, grads = _step(layer, static, go)
    for seed in range(3):
        torch.manual_seed(seed)
        static.copy_(torch.randn_like(x))
        graph.replay()
        torch.cuda.synchronize()
        want_y, _, want = _step(layer, static, go)
        assert torch.equal(y, want_y)
        for a, b in zip(grads, want):  # (grad_input is summed by atomics, then rounded)
            assert float((a.float() - b.float()).abs().max()) <= 2.0**-7 * float(b.float().abs().max())
