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


def test_saved_partials_outlive_their_use_on_another_stream():
    """A saved-tensor hook that copies on a stream of its own and calls record_stream: the allocator hands the memory out again only
    when that stream has got there."""
    ts = [torch.randn(1, 512, h, 64, device='cuda', dtype=torch.bfloat16).requires_grad_() for h in (2, 2, 2, 2, 2)]
    side, taken = torch.cuda.Stream(), []

    def pack(t):
        with torch.cuda.stream(side):
            torch.cuda._sleep(50_000_000)      # (tens of milliseconds: the stream is behind for the rest of the test)
        t.record_stream(side)
        taken.append((t.data_ptr(), t.untyped_storage().nbytes()))
        return t.shape

    with torch.autograd.graph.saved_tensors_hooks(pack, lambda shape: None):
        out = _attend(*ts)
    largest = max(size for _, size in taken)
    places = {ptr for ptr, size in taken if size == largest}       # (the partials: w2 times the size of q)
    del out
    again = [torch.empty(largest, dtype=torch.uint8, device='cuda') for _ in range(3)]
    assert not side.query()
    assert not places & {t.data_ptr() for t in again}
    torch.cuda.synchronize()


def test_partials_are_counted_while_they_are_saved():
    from simplicial_attention_amd import _native
    from simplicial_attention_amd.two_simplicial_attention import partials_budget
    live = lambda: partials_budget.live.get(0, 0) - _native.torch_ext().released_bytes(0)
    ts = _inputs(grad=True)
    before = live()
    out = _attend(*ts)
    assert live() - before == 2 * 9 * 96 * (64 * 2 + 4)            # heads, offsets, rows of 64 bf16 values and a reference each
    torch.autograd.grad(out.sum(), ts, retain_graph=True)
    assert live() > before
    torch.autograd.grad(out.sum(), ts)
    assert live() == before
    out = _attend(*ts)
    del out
    assert live() == before
