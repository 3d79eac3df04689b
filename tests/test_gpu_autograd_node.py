"""What goes through autograd stays visible to it: tangents, tracers and saved-tensor hooks."""
import pytest
import torch
import torch.autograd.forward_ad as fwAD

pytestmark = pytest.mark.gpu


def _inputs(d=64, dtype=torch.bfloat16, grad=False):
    g = torch.Generator().manual_seed(3)
    return [torch.randn(1, 96, h, d, generator=g).to('cuda', dtype).requires_grad_(grad) for h in (2, 1, 1, 1, 1)]


def _attend(q, k1, k2, v1, v2):
    from simplicial_attention_amd import sliding_two_simplicial_attn
    return sliding_two_simplicial_attn(q, (k1, k2), (v1, v2), w1=40, w2=9)


@pytest.mark.parametrize('grad_mode', [True, False])
def test_forward_mode_is_refused(grad_mode):
    """There is no forward derivative: a tangent is refused, not dropped, whether or not a graph is being built."""
    from simplicial_attention_amd.qkv_norm import FusedQKVNorm
    ts = _inputs()
    qkv = torch.randn(1, 32, 6 * 64, device='cuda').bfloat16()
    with torch.set_grad_enabled(grad_mode), fwAD.dual_level():
        dual = fwAD.make_dual(ts[0], torch.ones_like(ts[0]))
        with pytest.raises(RuntimeError):
            _attend(dual, *ts[1:])
        with pytest.raises(RuntimeError):
            FusedQKVNorm.apply(fwAD.make_dual(qkv, torch.ones_like(qkv)), None, None, None, None, None, 2, 1, 64, 1e-6)


@pytest.mark.parametrize('d,dtype', [(64, torch.bfloat16), (48, torch.float32)])
def test_traced_calls_run_the_kernels(d, dtype):
    ts = _inputs(d, dtype)
    traced = torch.jit.trace(_attend, tuple(ts), check_trace=False)
    others = [t.flip(1).contiguous() for t in ts]
    assert torch.equal(traced(*others), _attend(*others))


def test_traced_module_runs_the_kernels():
    from simplicial_attention_amd import SlidingWindowTwoSimplicialMHA
    torch.manual_seed(0)
    module = SlidingWindowTwoSimplicialMHA(64, dim_head=64, heads=2, key_value_heads=1, w1=40, w2=9).cuda().bfloat16()
    x = torch.randn(1, 96, 64, device='cuda').bfloat16()
    with torch.no_grad():
        traced = torch.jit.trace(module, x, check_trace=False)
        assert torch.equal(traced(x.flip(1)), module(x.flip(1)))


def test_saved_tensor_hooks_see_the_saved_tensors():
    ts = _inputs(grad=True)
    dout = torch.randn(1, 96, 2, 64, device='cuda').bfloat16()
    plain = torch.autograd.grad(_attend(*ts), ts, dout)
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t) or t.cpu(), lambda t: t.cuda()):
        out = _attend(*ts)
    assert len(packed) >= 7
    for a, b in zip(plain, torch.autograd.grad(out, ts, dout)):
        assert torch.equal(a, b)


def test_the_python_form_of_the_nodes_gives_the_same_gradients():
    from simplicial_attention_amd import _native
    from simplicial_attention_amd.two_simplicial_attention import partials_budget
    ts = _inputs(grad=True)
    dout = torch.randn(1, 96, 2, 64, device='cuda').bfloat16()
    want_out = _attend(*ts)
    want = torch.autograd.grad(want_out, ts, dout)
    with torch.no_grad():
        ext = _native.torch_ext()
        out, saved, sizes, scale = ext.attend_forward(*ts, 40, 9, None, True, partials_budget.admit)
        grads = ext.attend_backward(saved, sizes, scale, dout)
    assert torch.equal(out, want_out)
    assert all(torch.equal(a, b) for a, b in zip(grads, want))


@pytest.mark.parametrize('python_form', [False, True])
def test_a_forward_that_fails_leaves_the_budget_of_saved_partials_whole(python_form):
    """An allocation that fails (the device's share for this process is taken up to a few MiB): the bytes admitted for partials are
    given back, or were not admitted yet."""
    from simplicial_attention_amd import _native
    from simplicial_attention_amd.two_simplicial_attention import partials_budget, sliding_two_simplicial_attn
    n = 4096                           # q: 8 MiB of bf16
    ts = [torch.randn(1, n, h, 128, device='cuda', dtype=torch.bfloat16).requires_grad_() for h in (8, 8, 8, 8, 8)]
    live = lambda: partials_budget.live.get(0, 0) - _native.torch_ext().released_bytes(0)
    out = sliding_two_simplicial_attn(ts[0], (ts[1], ts[2]), (ts[3], ts[4]), w1=32, w2=2)
    del out
    before = live()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    try:
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (4 << 20)) / total)
        with pytest.raises(torch.OutOfMemoryError):
            if python_form:
                _native.torch_ext().attend_forward(*ts, 32, 2, None, True, partials_budget.admit)
            else:
                sliding_two_simplicial_attn(ts[0], (ts[1], ts[2]), (ts[3], ts[4]), w1=32, w2=2)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert live() == before
