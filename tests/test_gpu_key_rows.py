"""The dK1/dV1 kernels of head dimensions 128 and 256 at the edges of their walks: second windows around the chunks and the 48 rows
of the circular buffers (bwd_kvr_kernel, D = 256) and around blocks of 32 offsets (bwd_kv8_kernel, D = 128), first windows around a
tile, ragged last tiles and slabs, several query heads per key/value head, one workgroup per key slab and several."""
import pytest
import torch

from tests import parity_util as U

pytestmark = pytest.mark.gpu

CASES = [
    # b, n, hq, hk, w1, w2
    (1, 33, 1, 1, 33, 1),         # one offset per query tile: every step changes the tile
    (1, 129, 1, 1, 1, 3),         # a first window of one row, one row in the last slab
    (1, 257, 2, 1, 31, 2),
    (2, 127, 2, 2, 32, 47),       # around the circular buffers' 48 rows
    (1, 200, 2, 1, 33, 48),
    (1, 225, 1, 1, 64, 49),
    (1, 300, 4, 1, 129, 97),      # four query heads per key/value head, more than two rounds of the buffers
    (1, 640, 1, 1, 160, 7),       # slabs with query tiles before, inside and behind their own rows
]


@pytest.mark.parametrize('d', [128, 256])
@pytest.mark.parametrize('b,n,hq,hk,w1,w2', CASES)
def test_against_oracle(b, n, hq, hk, w1, w2, d):
    print(f'\ncase b={b} n={n} hq={hq} hk={hk} d={d} w1={w1} w2={w2}', flush=True)
    ins = U.make_inputs(b, n, hq, hk, d, seed=n + w1 + w2, std=d ** -0.5)
    ref_out, _, ref_grads = U.oracle_fwd_bwd(*ins, w1, w2)
    out, grads = U.hip_fwd_bwd(*ins, w1, w2)
    U.check_all(out, grads, ref_out, ref_grads)


@pytest.mark.parametrize('d', [32, 64, 128, 256])
def test_several_workgroups_per_slab_against_one(d):
    """The same sums in shares (all gradients at D = 32 to 128, dK1 and dV1 at 256): fp32 partial sums in another order, rounded to
    bf16 once."""
    from simplicial_attention_amd import _native
    lib = _native.load()
    b, n, h, hk, w1, w2 = 1, 700, 2, 1, 200, 21
    ins = [t.cuda() for t in U.make_inputs(b, n, h, hk, d, seed=5, std=d ** -0.5)]
    q, k1, k2, v1, v2, dout = ins
    prob = _native.problem(b, n, h, hk, d, w1, w2, True, d ** -0.5)
    arg = _native.tensor_arg
    out, lo = torch.empty_like(q), torch.empty_like(q)
    lse, delta = torch.empty(b, h, n, device='cuda'), torch.empty(b, h, n, device='cuda')
    stream = torch.cuda.current_stream().cuda_stream
    _native.check(lib.sa2_fwd(prob, *(arg(t) for t in (q, k1, k2, v1, v2, out)), arg(lo), lse.data_ptr(), None, stream))
    results = []
    for split in (False, True):
        size = lib.sa2_bwd_split_workspace_bytes(prob, 0) if split else lib.sa2_bwd_workspace_bytes(prob)
        ws = torch.full((size,), 255, dtype=torch.uint8, device='cuda')                # (NaN wherever nothing was written)
        grads = [torch.full_like(t, float('nan')) for t in (q, k1, k2, v1, v2)]
        dq, dk1, dk2, dv1, dv2 = grads
        call = lib.sa2_bwd_split if split else lib.sa2_bwd
        _native.check(call(prob, *(arg(t) for t in (q, k1, k2, v1, v2, out)), arg(lo), arg(dout), lse.data_ptr(), None, delta.data_ptr(),
                           *(arg(t) for t in (dq, dk1, dk2, dv1, dv2)), ws.data_ptr(), size, stream))
        torch.cuda.synchronize()
        results.append([t.float() for t in grads])
    for one, shares in zip(*results):
        # both are the bf16 rounding of fp32 sums that agree to about 1e-5: one bf16 step (2^-7) apart at most, 2^-9 on average
        assert bool(torch.isfinite(shares).all())
        assert float((one - shares).norm() / one.norm()) <= 2.0 ** -9
        assert bool(((one - shares).abs() <= 2.0 ** -7 * one.abs() + 1e-5 * float(one.abs().max())).all())
