"""Measured cases of sliding-window 2-simplicial attention.

A case is one pass through a public entry point, as a user's program calls it:

* ``kind='core'``   ``sliding_two_simplicial_attn`` on (b, n, h, d) tensors,
* ``kind='module'`` ``SlidingWindowTwoSimplicialMHA`` on (b, n, dim) tokens,
* ``kind='lm'``     ``TwoSimplicialLM`` with ``return_loss=True`` on byte tokens,

each either forward without a graph (``train=False``: evaluation, prefill) or forward and backward
(``train=True``: outputs and every gradient).

Ranges that the listed cases stand for (``draw`` samples them): batch 1 .. 8, 1 .. 16 heads with 1 .. 4 query heads per
key/value head, 17 .. 32768 rows, head dimensions 32 .. 256 (native and padded ones), first windows 16 .. 1024, second
windows 2 .. 128, bfloat16 (mostly), float16 and float32 tensors.
"""
import math

import torch

from simplicial_attention_amd import SlidingWindowTwoSimplicialMHA, sliding_two_simplicial_attn
from simplicial_attention_amd.two_simplicial_transformer import TwoSimplicialLM

_DTYPES = {'bf16': torch.bfloat16, 'fp16': torch.float16, 'fp32': torch.float32}
_NUM_TOKENS = 256


def _core(name, train, b, n, h, hk, d, w1, w2, dtype='bf16'):
    return {'name': name, 'kind': 'core', 'train': train, 'b': b, 'n': n, 'h': h, 'hk': hk, 'd': d, 'w1': w1, 'w2': w2, 'dtype': dtype}


def _module(name, train, b, n, dim, h, hk, d, w1, w2):
    return {'name': name, 'kind': 'module', 'train': train, 'b': b, 'n': n, 'dim': dim, 'h': h, 'hk': hk, 'd': d, 'w1': w1, 'w2': w2, 'dtype': 'bf16'}


def _lm(name, train, b, n, dim, depth, every, h, hk, d, w1, w2):
    return {'name': name, 'kind': 'lm', 'train': train, 'b': b, 'n': n, 'dim': dim, 'depth': depth, 'every': every, 'h': h, 'hk': hk, 'd': d,
            'w1': w1, 'w2': w2, 'dtype': 'bf16'}


def listed():
    return [
        # the smallest call: the shape of the parity test, evaluated without a graph (latency and launches)
        _core('core_fwd_smallest', False, 2, 128, 4, 4, 64, 64, 32),
        # full causal attention of a toy model in float32 (windows as long as the sequence), trained
        _core('core_train_fp32_full_causal', True, 1, 128, 4, 4, 32, 128, 128, 'fp32'),
        # one ragged sequence with grouped heads, trained: fine-tuning on single documents
        _core('core_train_ragged_n1000', True, 1, 1000, 8, 4, 64, 512, 32),
        # a float16 model whose head dimension is not one of the native ones, odd length, windows off the tile size
        _core('core_train_fp16_d96_odd', True, 2, 2999, 6, 2, 96, 300, 20, 'fp16'),
        # multi-head module, evaluation of a short batch
        _module('module_fwd_b2_n1024', False, 2, 1024, 512, 8, 8, 64, 512, 32),
        # multi-head module, one layer's training step at a training batch
        _module('module_train_b8_n2048', True, 8, 2048, 512, 8, 4, 64, 512, 32),
        # attention core of that layer alone
        _core('core_train_b8_n2048_d64', True, 8, 2048, 8, 4, 64, 512, 32),
        # language model, every second layer simplicial: loss and gradients of a training step
        _lm('lm_train_depth4_b8_n2048', True, 8, 2048, 512, 4, 2, 8, 4, 64, 512, 32),
        # widest heads
        _core('core_train_b2_n4096_d256', True, 2, 4096, 8, 8, 256, 512, 32),
        # the headline shape: prefill (no graph) and training
        _core('core_fwd_b4_n8192_d128', False, 4, 8192, 8, 8, 128, 512, 32),
        _core('core_train_b4_n8192_d128', True, 4, 8192, 8, 8, 128, 512, 32),
        # long context, the largest
        _core('core_train_b1_n32768_d128', True, 1, 32768, 16, 16, 128, 512, 32),
    ]


def _attended_triples(n, w1, w2):
    """sum over rows i of min(i + 1, w1) * min(i + 1, w2)"""
    lo, hi = sorted((min(w1, n), min(w2, n)))
    squares = lo * (lo + 1) * (2 * lo + 1) // 6                       # rows below both windows
    ramp = lo * (hi * (hi + 1) - lo * (lo + 1)) // 2                  # one window full
    return squares + ramp + (n - hi) * lo * hi


def _core_flops(c):
    per_triple = 18 if c['train'] else 4                              # contractions: 2 forward, 7 backward, 2 d flop each
    return per_triple * c['d'] * c['b'] * c['h'] * _attended_triples(c['n'], c['w1'], c['w2'])


def _module_weights(c):
    return c['dim'] * (c['h'] + 4 * c['hk']) * c['d'] + c['h'] * c['d'] * c['dim']


def work(case):
    """Contractions of the attended triples and of the projections; inputs read once, outputs written once."""
    c = case
    passes = 3 if c['train'] else 1                                   # a matrix product and its two gradients
    size = 4 if c['dtype'] == 'fp32' else 2
    rows = c['b'] * c['n']
    if c['kind'] == 'core':
        q, kv = rows * c['h'] * c['d'] * size, rows * c['hk'] * c['d'] * size
        moved = 2 * q + 4 * kv + ((2 * q + 4 * kv) if c['train'] else 0)
        return {'bytes': moved, 'flops': _core_flops(c)}
    if c['kind'] == 'module':
        w = _module_weights(c)
        x = rows * c['dim'] * size
        moved = 2 * x + w * size + ((2 * x + w * size) if c['train'] else 0)
        return {'bytes': moved, 'flops': _core_flops(c) + passes * 2 * rows * w}
    simplicial = c['depth'] // c['every']
    ordinary = c['depth'] - simplicial
    w_attn = c['dim'] * (2 * c['h'] + 2 * c['hk']) * c['d']
    w_ff = 8 * c['dim'] ** 2
    weights = simplicial * _module_weights(c) + ordinary * w_attn + c['depth'] * w_ff + _NUM_TOKENS * c['dim']
    params = weights + (_NUM_TOKENS + c['n']) * c['dim']
    dense = (3.5 if c['train'] else 1) * 2 * c['d'] * c['b'] * c['h'] * c['n'] ** 2
    moved = 8 * c['b'] * (c['n'] + 1) + params * size * (2 if c['train'] else 1) + (0 if c['train'] else rows * _NUM_TOKENS * size)
    return {'bytes': moved, 'flops': simplicial * _core_flops(c) + ordinary * dense + passes * 2 * rows * weights}


def tolerance(case):
    """Operands and packed weights are bfloat16 on every path (float16 and float32 tensors are computed in it too).  Two
    correct forms of the core differ by the rounding of the same products at other places: up to 1e-2.  Around the core
    the projections and norms round to bfloat16 as well, layer after layer."""
    return {'rel': {'core': 1e-2, 'module': 1e-2, 'lm': 2e-2}[case['kind']]}


def prepare(case, seed):
    """Unit-variance q, k and v (what the per-head RMSNorms of the module hand over) and unit-variance output gradients."""
    c = case
    g = torch.Generator(device='cuda').manual_seed(int(seed))
    dtype = _DTYPES[c['dtype']]
    randn = lambda *shape: torch.randn(*shape, generator=g, device='cuda').to(dtype)
    if c['kind'] == 'core':
        q, dout = randn(c['b'], c['n'], c['h'], c['d']), randn(c['b'], c['n'], c['h'], c['d'])
        kv = [randn(c['b'], c['n'], c['hk'], c['d']) for _ in range(4)]
        leaves = [t.requires_grad_(c['train']) for t in (q, *kv)]
        return {'case': c, 'leaves': leaves, 'dout': dout}
    torch.manual_seed(int(seed))
    if c['kind'] == 'module':
        with torch.device('cuda'):
            module = SlidingWindowTwoSimplicialMHA(c['dim'], dim_head=c['d'], heads=c['h'], key_value_heads=c['hk'], w1=c['w1'], w2=c['w2'])
        module = module.to(dtype)
        x = randn(c['b'], c['n'], c['dim']).requires_grad_(c['train'])
        return {'case': c, 'module': module, 'x': x, 'dout': randn(c['b'], c['n'], c['dim']), 'params': list(module.parameters())}
    with torch.device('cuda'):
        lm = TwoSimplicialLM(num_tokens=_NUM_TOKENS, dim=c['dim'], depth=c['depth'], max_seq_len=c['n'], dim_head=c['d'], heads=c['h'],
                             two_simplicial_attn_every=c['every'],
                             transformer_kwargs=dict(key_value_heads=c['hk'], two_simplicial_attn_kwargs=dict(w1=c['w1'], w2=c['w2'])))
    lm = lm.to(dtype)
    tokens = torch.randint(0, _NUM_TOKENS, (c['b'], c['n'] + 1), generator=g, device='cuda')
    return {'case': c, 'module': lm, 'tokens': tokens, 'params': list(lm.parameters())}


def run(state):
    c = state['case']
    if c['kind'] == 'core':
        q, k1, k2, v1, v2 = state['leaves']
        if not c['train']:
            with torch.no_grad():
                return sliding_two_simplicial_attn(q, (k1, k2), (v1, v2), w1=c['w1'], w2=c['w2'])
        out = sliding_two_simplicial_attn(q, (k1, k2), (v1, v2), w1=c['w1'], w2=c['w2'])
        return [out.detach(), *torch.autograd.grad(out, state['leaves'], state['dout'])]
    if c['kind'] == 'module':
        if not c['train']:
            with torch.no_grad():
                return state['module'](state['x'])
        out = state['module'](state['x'])
        return [out.detach(), *torch.autograd.grad(out, [state['x'], *state['params']], state['dout'])]
    if not c['train']:
        with torch.no_grad():
            return state['module'](state['tokens'][:, :-1])
    loss = state['module'](state['tokens'], return_loss=True)
    return [loss.detach(), *torch.autograd.grad(loss, state['params'])]


# a drawn case costs at most what these pay for (flop): the long-context case at its head dimensions; wider heads run on
# kernels of a lower rate and get the budget of their own listed case
_BUDGET = 18 * 128 * 16 * _attended_triples(32768, 512, 32)
_BUDGET_WIDE = 18 * 256 * 2 * 8 * _attended_triples(4096, 512, 32)


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        kind = rng.choice(['core'] * 7 + ['module'] * 2 + ['lm'])
        train = rng.random() < 0.65
        hk = rng.choice([1, 2, 4, 8])
        h = hk * rng.choice([g for g in (1, 2, 4) if hk * g <= 16])
        b = rng.randint(1, 8)
        w1, w2 = _log_uniform(rng, 16, 1024), _log_uniform(rng, 2, 128)
        if kind == 'core':
            d = rng.choice([32, 64, 64, 64, 128, 128, 128, 256, 48, 80, 96])
            dtype = rng.choice(['bf16'] * 6 + ['fp16', 'fp32'])
            case = _core('', train, b, _log_uniform(rng, 17, 32768), h, hk, d, w1, w2, dtype)
        elif kind == 'module':
            case = _module('', train, b, _log_uniform(rng, 64, 8192), rng.choice([128, 256, 384, 512, 768, 1024]), h, hk,
                           rng.choice([32, 64, 128]), w1, w2)
        else:
            every = rng.choice([1, 2, 4])
            case = _lm('', train, b, _log_uniform(rng, 64, 4096), rng.choice([128, 256, 512]), every * rng.choice([1, 4 // every]), every, h, hk,
                       rng.choice([32, 64]), w1, w2)
        del case['name']
        # (narrow heads do as much elementwise work per triple as wide ones: counted as if 128 wide)
        cost = work(case)['flops'] * max(1.0, 128 / case['d'])
        if cost <= (_BUDGET_WIDE if case['d'] > 128 else _BUDGET):
            return case
