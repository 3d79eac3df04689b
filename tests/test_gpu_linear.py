"""The weight gradient kernel of linear layers, and what decides whether a layer takes it."""
import pytest
import torch
from torch import nn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('rows,out_features,in_features', [
    (1, 128, 128),             # less than one tile
    (32, 128, 128),
    (33, 128, 128),            # one row in the last tile
    (95, 128, 256),
    (64, 128, 256),            # two tiles: the three buffers are not all used
    (96, 256, 128),
    (16 * 32 * 5 + 32, 128, 384),      # shares of unequal length
    (8192, 512, 256),
    (8191, 256, 128),          # several shares, a ragged last tile
    (16384, 1536, 512),
])
def test_kernel_against_fp64(rows, out_features, in_features):
    from simplicial_attention_amd import _native
    lib = _native.load()
    print(f'\ncase rows={rows} out={out_features} in={in_features}', flush=True)
    g = torch.Generator(device='cuda').manual_seed(rows + out_features)
    # (rows inside wider ones: strides of their own)
    dy = torch.randn(rows, out_features + 8, generator=g, device='cuda').bfloat16()[:, :out_features]
    x = torch.randn(rows, in_features + 16, generator=g, device='cuda').bfloat16()[:, :in_features]
    dw = torch.full((out_features, in_features), float('nan'), device='cuda', dtype=torch.bfloat16)
    size = lib.sa2_wgrad_workspace_bytes(rows, out_features, in_features)
    ws = torch.full((size,), 255, dtype=torch.uint8, device='cuda')
    _native.check(lib.sa2_wgrad(dy.data_ptr(), dy.stride(0), x.data_ptr(), x.stride(0), rows, out_features, in_features, dw.data_ptr(), ws.data_ptr(), size,
                                torch.cuda.current_stream().cuda_stream))
    want = dy.double().t() @ x.double()
    # one rounding to bf16 (2^-9 of the value at most) of fp32 sums (error about 1e-6 of the terms' norm, sqrt(rows))
    assert bool(((dw.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-5 * rows ** 0.5).all())


def test_sizes_that_do_not_fit_are_refused():
    from simplicial_attention_amd import _native
    lib = _native.load()
    for sizes in ((32, 64, 128), (32, 128, 192), (0, 128, 128)):
        assert lib.sa2_wgrad_workspace_bytes(*sizes) == -1


def _layer(bias=True):
    torch.manual_seed(0)
    return nn.Linear(128, 256, bias=bias).cuda().bfloat16(), torch.randn(4, 2048, 128, device='cuda').bfloat16().requires_grad_()


@pytest.mark.parametrize('bias', [True, False])
def test_layer_gradients_match_torch(bias):
    from simplicial_attention_amd.linear import apply_linear
    layer, x = _layer(bias)
    dout = torch.randn(4, 2048, 256, device='cuda').bfloat16()
    params = [x, *layer.parameters()]
    got_out, want_out = apply_linear(layer, x), layer(x)
    assert torch.equal(got_out, want_out) and got_out.grad_fn.name() != want_out.grad_fn.name()
    got = torch.autograd.grad(got_out, params, dout.transpose(0, 1).contiguous().transpose(0, 1))
    for a, b in zip(got, torch.autograd.grad(want_out, params, dout)):
        assert float((a.float() - b.float()).norm() / b.float().norm()) <= 2.0 ** -8        # (two bf16 roundings of the same sums)


def test_second_derivatives_and_tangents_stay():
    import torch.autograd.forward_ad as fwAD
    from simplicial_attention_amd.linear import apply_linear
    layer, x = _layer()
    second = []
    for f in (apply_linear, lambda m, t: m(t)):
        gx, gw = torch.autograd.grad(f(layer, x).float().pow(2).sum(), [x, layer.weight], create_graph=True)
        second.append(torch.autograd.grad(gx.float().pow(2).sum() + gw.float().sum(), [x, layer.weight]))
    for a, b in zip(*second):
        assert float((a.float() - b.float()).norm() / b.float().norm()) <= 1e-2
    with fwAD.dual_level():
        out = apply_linear(layer, fwAD.make_dual(x.detach(), torch.ones_like(x)))
        assert fwAD.unpack_dual(out).tangent is not None


def test_hooks_see_the_layer():
    from simplicial_attention_amd.linear import apply_linear
    layer, x = _layer()
    seen = []
    handle = layer.register_forward_hook(lambda m, args, out: seen.append(out.shape))
    apply_linear(layer, x)
    handle.remove()
    assert seen == [(4, 2048, 256)]


@pytest.mark.parametrize('owner,name', [(nn.Linear, 'forward'), (nn.Module, '__call__'), (nn.Module, '_call_impl'), (nn.functional, 'linear')])
def test_replaced_functions_see_the_layer(owner, name, monkeypatch):
    """Replacements for all linear layers: the class's forward, a module's call, the function behind them."""
    from simplicial_attention_amd.linear import apply_linear
    layer, x = _layer()
    seen, original = [], getattr(owner, name)

    def replacement(*args, **kwargs):
        seen.append(name)
        return original(*args, **kwargs)

    monkeypatch.setattr(owner, name, replacement)
    apply_linear(layer, x)
    assert seen


def test_a_compiled_layer_is_called():
    from simplicial_attention_amd.linear import apply_linear
    layer, x = _layer()
    seen = []
    layer._compiled_call_impl = lambda *args: seen.append(args) or layer._call_impl(*args)      # (what nn.Module.compile sets)
    apply_linear(layer, x)
    assert seen


@pytest.mark.parametrize('bias', [True, False])
def test_batched_output_gradients(bias):
    """``is_grads_batched``: the node meets a batched tensor in its backward only."""
    from simplicial_attention_amd.linear import apply_linear
    layer, x = _layer(bias)
    douts = torch.randn(3, 4, 2048, 256, device='cuda').bfloat16()
    params = [x, *layer.parameters()]
    out = apply_linear(layer, x)
    got = torch.autograd.grad(out, params, douts, retain_graph=True, is_grads_batched=True)
    for n in range(3):
        for a, b in zip(got, torch.autograd.grad(out, params, douts[n], retain_graph=True)):
            assert float((a[n].float() - b.float()).norm() / b.float().norm()) <= 2.0 ** -8      # (two bf16 roundings of the same sums)


def test_tangents_of_output_gradients_stay():
    """Forward over reverse: the layer's own inputs are plain, the gradient that comes back carries a tangent."""
    import torch.autograd.forward_ad as fwAD
    from simplicial_attention_amd.linear import apply_linear
    layer, x = _layer()
    out = apply_linear(layer, x)
    dout, tangent = torch.randn_like(out), torch.randn_like(out)
    with fwAD.dual_level():
        got = torch.autograd.grad(out, layer.weight, fwAD.make_dual(dout, tangent), retain_graph=True)[0]
        got = fwAD.unpack_dual(got).tangent
    want = torch.autograd.grad(out, layer.weight, tangent)[0]
    assert got is not None and float((got.float() - want.float()).norm() / want.float().norm()) <= 2.0 ** -8


def test_a_weight_that_no_gradient_needs_may_change():
    """As with torch's node: an input without a gradient leaves the weight free between forward and backward; one with a gradient does not."""
    from simplicial_attention_amd.linear import apply_linear
    layer, x = _layer()
    dout = torch.randn(4, 2048, 256, device='cuda').bfloat16()
    want = torch.autograd.grad(apply_linear(layer, x.detach()), layer.weight, dout)[0]
    out, with_x = apply_linear(layer, x.detach()), apply_linear(layer, x)
    with torch.no_grad():
        layer.weight.mul_(2)
    assert torch.equal(torch.autograd.grad(out, layer.weight, dout)[0], want)
    with pytest.raises(RuntimeError, match='modified by an inplace operation'):
        torch.autograd.grad(with_x, layer.weight, dout)
