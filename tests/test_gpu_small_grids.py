"""Work shared by several workgroups against the same work in one, and the conversions around the kernels."""
import pytest
import torch

from tests import parity_util as U

pytestmark = pytest.mark.gpu

SHAPES = [
    # b, n, hq, hk, w1, w2
    (1, 40, 1, 1, 16, 33),         # two query tiles of several rounds
    (1, 333, 2, 1, 512, 32),
    (1, 700, 2, 2, 300, 20),
]


@pytest.mark.parametrize('d', [32, 64, 128])
@pytest.mark.parametrize('b,n,h,hk,w1,w2', SHAPES)
def test_forward_in_shares(b, n, h, hk, w1, w2, d):
    """fp32 partial rows merged once: out and lse agree to one bf16 rounding and to fp32 sums."""
    from simplicial_attention_amd import _native
    lib = _native.load()
    print(f'\ncase b={b} n={n} h={h} hk={hk} d={d} w1={w1} w2={w2}', flush=True)
    ins = [t.cuda() for t in U.make_inputs(b, n, h, hk, d, seed=n + d)][:5]
    prob = _native.problem(b, n, h, hk, d, w1, w2, True, d ** -0.5)
    size = lib.sa2_fwd_workspace_bytes(prob)
    assert size > 0, 'the grid is not small enough to be shared out'
    arg, stream = _native.tensor_arg, torch.cuda.current_stream().cuda_stream
    results = []
    for ws in (None, torch.full((size,), 255, dtype=torch.uint8, device='cuda')):
        out, lse = torch.full_like(ins[0], float('nan')), torch.full((b, h, n), float('nan'), device='cuda')
        _native.check(lib.sa2_fwd_ws(prob, *(arg(t) for t in ins), arg(out), None, lse.data_ptr(), None, None if ws is None else ws.data_ptr(),
                                     0 if ws is None else size, stream))
        torch.cuda.synchronize()
        results.append((out.float(), lse))
    (o0, l0), (o1, l1) = results
    assert float((l0 - l1).abs().max()) <= 1e-4 * max(1.0, float(l0.abs().max()))
    # (the saved maximum of a share differs, so weights round to bf16 at other places: 2^-9 each, averaged over the row)
    assert float((o0 - o1).norm() / o0.norm()) <= 2.0 ** -8


@pytest.mark.parametrize('d', [32, 64, 128])
@pytest.mark.parametrize('shared', [True, False], ids=['shared', 'unshared'])
@pytest.mark.parametrize('b,n,h,hk,w1,w2', [
    (1, 1, 1, 1, 4, 3), (1, 33, 3, 1, 16, 9), (1, 70, 4, 2, 70, 33), (1, 257, 2, 2, 40, 128),
    (1, 70, 2, 1, 33, 16), (1, 70, 2, 1, 33, 17), (1, 113, 2, 2, 33, 49),      # eight offsets per group and one more, in either block of 32
    (8, 33, 32, 32, 8, 5),         # 512 blocks of dV2 rows: the last grid that takes one launch
    (8, 33, 33, 33, 8, 5),         # 528: the first that takes two
])
def test_second_set_gradients_of_small_grids(b, n, h, hk, w1, w2, d, shared):
    """dV2, dK2 and dQ merged in one launch: single rows, remainders of tiles, groups, offsets beyond one block of 32."""
    print(f'\ncase b={b} n={n} h={h} hk={hk} d={d} w1={w1} w2={w2} shared={shared}', flush=True)
    ins = U.make_inputs(b, n, h, hk, d, seed=7 * n + d, std=d ** -0.5)
    ref_out, _, ref_grads = U.oracle_fwd_bwd(*ins, w1, w2)
    if shared:
        out, grads = U.hip_fwd_bwd(*ins, w1, w2)
    else:
        out, _, grads = U.hip_unshared_fwd_bwd(*ins, w1, w2, use_saved=True)
    U.check_all(out, grads, ref_out, ref_grads)


@pytest.mark.parametrize('d', [32, 64, 128])
@pytest.mark.parametrize('shared', [True, False], ids=['shared', 'unshared'])
@pytest.mark.parametrize('b,n,h,hk,w1,w2', [(1, 70, 4, 2, 70, 33), (1, 257, 2, 2, 40, 128), (1, 300, 8, 2, 64, 20)])
def test_partials_do_not_reach_the_other_gradients(b, n, h, hk, w1, w2, d, shared):
    """Whether partials are saved decides how dV2 is formed and nothing else: the other gradients have the same bits."""
    print(f'\ncase b={b} n={n} h={h} hk={hk} d={d} w1={w1} w2={w2} shared={shared}', flush=True)
    ins = U.make_inputs(b, n, h, hk, d, seed=n + d, std=1.0)
    with_saved, without = (U.hip_abi_fwd_bwd(*ins, w1, w2, use_saved, shared=shared)[2] for use_saved in (True, False))
    for name, x, y in zip(('dq', 'dk1', 'dk2', 'dv1'), with_saved, without):
        assert bool(torch.isfinite(x).all()) and torch.equal(x, y), name


@pytest.mark.parametrize('d', [65, 80, 96, 97])
@pytest.mark.parametrize('b,n,h,hk,w1,w2', [(1, 1, 1, 1, 4, 3), (1, 75, 4, 2, 40, 41),
                                            (8, 40, 66, 33, 16, 9),      # more query tiles than are shared out
                                            (1, 200, 4, 2, 100, 12),     # lower edge, interior and diagonal tiles: shared out,
                                            (8, 200, 20, 10, 100, 3)])   # and in undivided walks
def test_narrow_heads_on_the_kernels_of_wide_ones(b, n, h, hk, w1, w2, d):
    """Up to 96 channels padded to 128 leave the products over the last 32 out; 97 takes them all."""
    print(f'\ncase b={b} n={n} h={h} hk={hk} d={d} w1={w1} w2={w2}', flush=True)
    ins = U.make_inputs(b, n, h, hk, d, seed=3 * n + d, std=d ** -0.5)
    ref_out, _, ref_grads = U.oracle_fwd_bwd(*ins, w1, w2)
    out, grads = U.hip_fwd_bwd(*ins, w1, w2)
    U.check_all(out, grads, ref_out, ref_grads)


@pytest.mark.parametrize('dtype,dim_qk,dim_v', [(torch.float16, 96, 70), (torch.float16, 65, 96), (torch.float32, 40, 80), (torch.bfloat16, 96, 97)])
@pytest.mark.parametrize('b,n,h,hk,w1,w2', [(1, 200, 4, 2, 100, 12), (8, 200, 20, 10, 100, 3)])
def test_narrow_heads_with_values_of_another_width(b, n, h, hk, w1, w2, dtype, dim_qk, dim_v):
    """The wider of the two head dimensions decides which products are left out.  The output gradients are scaled up by a power of two, as
    float16 training scales its loss, and the gradients back down: the rms of dq is about 1e-6 here, of which the rounding to float16's
    subnormal spacing, 2^-24 / sqrt(12) = 1.7e-8, would alone be more than 1 %."""
    from simplicial_attention_amd import sliding_two_simplicial_attn
    print(f'\ncase b={b} n={n} h={h} hk={hk} dim_qk={dim_qk} dim_v={dim_v} w1={w1} w2={w2} {dtype}', flush=True)
    q, k1, k2 = U.make_inputs(b, n, h, hk, dim_qk, seed=dim_qk, std=dim_qk ** -0.5)[:3]
    _, v1, v2, _, _, dout = U.make_inputs(b, n, h, hk, dim_v, seed=1000 + dim_v, std=dim_v ** -0.5)
    ref_out, _, ref_grads = U.oracle_fwd_bwd(q, k1, k2, v1, v2, dout, w1, w2)
    loss_scale = 2.0 ** 10
    ts = [t.to(dtype).cuda().requires_grad_(True) for t in (q, k1, k2, v1, v2)]
    out = sliding_two_simplicial_attn(ts[0], (ts[1], ts[2]), (ts[3], ts[4]), w1=w1, w2=w2)
    grads = torch.autograd.grad(out, ts, (dout * loss_scale).to(dtype).cuda())
    U.check_all(out, [g.float() / loss_scale for g in grads], ref_out, ref_grads)


@pytest.mark.parametrize('channels', [1, 40, 65, 96, 97])
@pytest.mark.parametrize('use_saved', [True, False], ids=['saved', 'recomputed'])
@pytest.mark.parametrize('b,n,h,hk,w1,w2', [(1, 200, 4, 2, 100, 12), (8, 200, 20, 10, 100, 3)])
def test_products_over_padding_add_nothing(b, n, h, hk, w1, w2, use_saved, channels):
    """sa2_bwd_split_padded on heads of 128 with zero channels: what is left out would have added zeros to fp32 sums, so every gradient
    has the bits of the call that takes all channels."""
    print(f'\ncase b={b} n={n} h={h} hk={hk} channels={channels} w1={w1} w2={w2} saved={use_saved}', flush=True)
    ins = U.make_inputs(b, n, h, hk, 128, seed=channels, std=1.0)
    for t in ins:
        t[..., channels:] = 0
    scale = channels ** -0.5
    few, every = (U.hip_abi_fwd_bwd(*ins, w1, w2, use_saved, scale, shared=True, channels=c)[2] for c in (channels, 128))
    for name, x, y in zip(('dq', 'dk1', 'dk2', 'dv1', 'dv2'), few, every):
        x, y = x[..., :channels], y[..., :channels]
        assert bool(torch.isfinite(x).all()) and torch.equal(x, y), name


@pytest.mark.parametrize('d', [32, 64, 128])
@pytest.mark.parametrize('b,n,h,hk,w1,w2', [(1, 128, 8, 1, 40, 33), (1, 70, 4, 2, 70, 128), (1, 200, 8, 1, 128, 64)])
def test_shares_merged_from_a_poisoned_workspace(b, n, h, hk, w1, w2, d):
    """Shared query tiles with saved partials, every byte of scratch and results NaN before the call: a share's row that is read has been
    written, twice the same bits, and the sums are those of sa2_bwd in another order."""
    from simplicial_attention_amd import _native
    lib = _native.load()
    print(f'\ncase b={b} n={n} h={h} hk={hk} d={d} w1={w1} w2={w2}', flush=True)
    prob = _native.problem(b, n, h, hk, d, w1, w2, True, d ** -0.5)
    # (scatter rows and fp32 dq rows of several shares: the query tiles are shared out)
    sets, rest = divmod(lib.sa2_bwd_split_workspace_bytes(prob, 1), lib.sa2_bwd_workspace_bytes(prob) // 2 + b * h * n * d * 4)
    assert sets > 1 and rest == 0
    ins = U.make_inputs(b, n, h, hk, d, seed=5, std=d ** -0.5)
    one = U.hip_abi_fwd_bwd(*ins, w1, w2, True)[2]
    shares, again = (U.hip_abi_fwd_bwd(*ins, w1, w2, True, shared=True)[2] for _ in range(2))
    for name, x, y, z in zip(('dq', 'dk1', 'dk2', 'dv1', 'dv2'), one, shares, again):
        assert torch.equal(y, z), name
        x, y = x.float(), y.float()
        # bf16 roundings of fp32 sums that agree to about 1e-5: one bf16 step (2^-7) apart at most, 2^-9 on average
        assert bool(torch.isfinite(y).all()) and float((x - y).norm() / x.norm()) <= 2.0 ** -9, name
        assert bool(((x - y).abs() <= 2.0 ** -7 * x.abs() + 1e-5 * float(x.abs().max())).all()), name


@pytest.mark.parametrize('src_type,dst_type', [(torch.float32, torch.bfloat16), (torch.float16, torch.bfloat16), (torch.bfloat16, torch.float32),
                                               (torch.bfloat16, torch.float16), (torch.bfloat16, torch.bfloat16)])
@pytest.mark.parametrize('src_dim,dst_dim,vector', [(96, 128, True), (128, 96, True), (33, 64, False), (64, 33, False), (5, 32, False), (64, 64, True)])
def test_conversions_against_torch(src_type, dst_type, src_dim, dst_dim, vector):
    """Truncated or zero-padded rows; `vector`: whether rows are aligned for 16-byte accesses.  One rounding, as torch's."""
    import ctypes
    from simplicial_attention_amd import _native
    lib = _native.load()
    lib.sa2_convert.restype = ctypes.c_int
    code = {torch.bfloat16: 0, torch.float16: 1, torch.float32: 2}

    class Conversion(ctypes.Structure):
        _fields_ = [('src', _native.TensorArg), ('dst', _native.TensorArg)] + [(f, ctypes.c_int32) for f in
                   ('src_type', 'dst_type', 'src_dim', 'dst_dim', 'batch', 'seq_len', 'heads')]

    b, n, h = 2, 37, 3
    pad = 8 if vector else 3
    src = (torch.randn(b, n, h, src_dim + pad, device='cuda') * 3).to(src_type)[..., :src_dim]
    src[0, 0, 0, :3] = torch.tensor([float('inf'), float('nan'), -0.0], device='cuda').to(src_type)
    dst = torch.full((b, n, h, dst_dim + pad), 7.0, device='cuda').to(dst_type)
    item = Conversion(_native.tensor_arg(src), _native.tensor_arg(dst[..., :dst_dim]), code[src_type], code[dst_type], src_dim, dst_dim, b, n, h)
    _native.check(lib.sa2_convert(ctypes.byref(item), 1, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    want = torch.zeros(b, n, h, dst_dim, device='cuda', dtype=dst_type)
    common = min(src_dim, dst_dim)
    want[..., :common] = src[..., :common].to(dst_type)
    assert torch.equal(torch.nan_to_num(dst[..., :dst_dim], nan=123.0), torch.nan_to_num(want, nan=123.0))
    assert torch.equal(dst[..., :dst_dim].isnan(), want.isnan()) and bool((dst[..., dst_dim:] == 7.0).all())
