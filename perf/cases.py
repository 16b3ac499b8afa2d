"""Performance cases of the block-scaled GEMM family: the calls that a serving or training program makes.

Every case runs ONE call of a public entry point of ``deep_gemm`` on operands that lie on the GPU as such a
program holds them: activations and weights quantised to e4m3 (1x128 and 128x128 UE8M0 blocks), weights in e2m1
(1x32 blocks), or bf16.  Weight scale factors are in the kernels' layout (a program lays them out once);
activation scale factors are in that layout too (``sf="packed"``: a quantiser that writes it) or as the fp32
tensor of a plain quantiser (``sf="fp32"``, converted inside the call).

The sizes are those of this repository's configurations, tests and benchmark: N x K of 2112x7168, 24576x1536,
7168x16384, 4096x7168 and 7168x2048, expert shapes 4096x7168, 7168x2048 and 4096x2048, 8192 routed tokens with 32
local experts, and the h=8, r=4096, d=1024 head contraction.
"""
import math
import os
import random
import sys

import torch

sys.path.insert(1, os.path.abspath('deepgemm-ascend_amd'))

import deep_gemm  # noqa: E402

E4M3_MAX, E2M1_MAX = 448.0, 6.0
E2M1_VALUES = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)
E2M1_BOUNDS = (0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0)


def listed():
    return [
        # One token of one sequence through a projection: the smallest call, latency and the read of the weights.
        dict(name='decode_1', op='dense', kind='fp8', form='nt', m=1, n=2112, k=7168, sf='packed'),
        # One decode step of a batch of 128 sequences, with the quantiser's fp32 activation scales.
        dict(name='decode_128', op='dense', kind='fp8', form='nt', m=128, n=7168, k=2048, sf='fp32'),
        # The last chunk of a prompt: an odd number of tokens.
        dict(name='chunk_odd', op='dense', kind='fp8', form='nt', m=1237, n=2112, k=7168, sf='fp32'),
        # A prefill step (the benchmark's headline shape).
        dict(name='prefill', op='dense', kind='fp8', form='nt', m=4096, n=7168, k=2048, sf='packed'),
        # The longest dense contraction (an MLP's or output projection's down direction).
        dict(name='prefill_long', op='dense', kind='fp8', form='nt', m=4096, n=7168, k=16384, sf='packed'),
        # Layers kept in bf16: forward ...
        dict(name='bf16_forward', op='dense', kind='bf16', form='nt', m=4096, n=4096, k=7168, sf='none'),
        # ... and backward, the weight gradient (both operands contiguous along their tokens' features), in fp32.
        dict(name='bf16_wgrad', op='dense', kind='bf16', form='tn', m=2112, n=7168, k=4096, sf='none', out='fp32'),
        # Mixture of experts, prefill: tokens routed to 32 local experts, rows padded to 128, e4m3 weights.
        dict(name='moe_prefill', op='contiguous', kind='fp8', form='nt', groups=32, tokens=8192, align=128, n=4096,
             k=7168, layout='psum', sf='fp32'),
        # The same with e2m1 weights and long groups.
        dict(name='moe_prefill_fp4', op='contiguous', kind='fp8fp4', form='nt', groups=8, tokens=32768, align=256,
             n=4096, k=2048, layout='psum', sf='packed'),
        # Mixture of experts, decode: about 32 tokens for each of 32 experts in a fixed buffer of 128 rows.
        dict(name='moe_decode', op='masked', kind='fp8', groups=32, max_m=128, mean_m=32, n=7168, k=2048, sf='packed'),
        # Mixture of experts, training: the weight gradient of four experts, contracted over their tokens.
        dict(name='moe_wgrad', op='kgrouped', kind='fp8', groups=4, tokens=32768, m=7168, n=2048, sf='fp32'),
        # Per-head contraction of the attention output (batched over the heads).
        dict(name='heads', op='einsum', kind='fp8', b=4096, h=8, r=4096, d=1024, sf='fp32'),
    ]


def _log_int(rng, lo, hi, multiple=1):
    return max(multiple, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / multiple)) * multiple)


def draw(rng):
    op = rng.choice(['dense'] * 6 + ['contiguous'] * 2 + ['masked', 'kgrouped', 'einsum'])
    if op == 'dense':
        kind = rng.choice(['fp8', 'fp8', 'fp8', 'bf16', 'bf16', 'fp8fp4'])
        form = rng.choice(['nt', 'nt', 'nt', 'nn', 'tn']) if kind != 'fp8fp4' else 'nt'
        while True:
            m = _log_int(rng, 1, 8192) if form != 'tn' else _log_int(rng, 512, 8192, 16)
            n = _log_int(rng, 512, 24576, rng.choice([1, 32, 64, 128]) if form == 'nt' else 16)
            k = _log_int(rng, 512, 16384, rng.choice([32, 128, 128, 128]))
            if 2.0 * m * n * k <= 4.8e11:
                break
        return dict(op=op, kind=kind, form=form, m=m, n=n, k=k,
                    sf='none' if kind == 'bf16' else rng.choice(['packed', 'fp32']) if form == 'nt' else 'fp32',
                    out='fp32' if form == 'tn' else 'bf16')
    if op == 'contiguous':
        kind = rng.choice(['fp8', 'fp8', 'fp8fp4', 'bf16'])
        while True:
            groups, tokens = rng.choice([4, 8, 16, 32, 48]), _log_int(rng, 512, 32768)
            n, k = _log_int(rng, 1024, 8192, 64), _log_int(rng, 1024, 8192, 128)
            if 2.0 * tokens * n * k <= 4.8e11 and groups * n * k <= 1 << 30:
                break
        return dict(op=op, kind=kind, form=rng.choice(['nt', 'nt', 'nn']) if kind != 'fp8fp4' else 'nt', groups=groups,
                    tokens=tokens, align=rng.choice([128, 128, 256]), n=n, k=k, layout=rng.choice(['psum', 'indices']),
                    sf='none' if kind == 'bf16' else rng.choice(['packed', 'fp32']))
    if op == 'masked':
        max_m = rng.choice([16, 32, 64, 128, 256, 512, 1024])
        groups = rng.choice([8, 16, 32])
        return dict(op=op, kind=rng.choice(['fp8', 'fp8', 'bf16']), groups=groups, max_m=max_m,
                    mean_m=_log_int(rng, 4, 0.75 * max_m), n=_log_int(rng, 1024, 8192, 64),
                    k=_log_int(rng, 1024, 8192, 128), sf='packed')
    if op == 'kgrouped':
        while True:
            groups, tokens = rng.choice([2, 4, 8, 16]), _log_int(rng, 2048, 32768)
            m, n = _log_int(rng, 1024, 8192, 64), _log_int(rng, 1024, 8192, 64)
            if 2.0 * m * n * tokens <= 4.8e11 and groups * m * n <= 1 << 28:
                break
        return dict(op=op, kind=rng.choice(['fp8', 'bf16']), groups=groups, tokens=tokens, m=m, n=n, sf='fp32')
    while True:
        b, h = _log_int(rng, 16, 8192), rng.choice([4, 8, 16, 32])
        r, d = _log_int(rng, 512, 4096, 128), _log_int(rng, 128, 2048, 128)
        if 2.0 * b * h * r * d <= 2.8e11:
            return dict(op='einsum', kind='fp8', b=b, h=h, r=r, d=d, sf='fp32')


# ------------------------------------------------------------------------------------------- inputs
def _pow2_ceil(x):
    bits = x.view(torch.int32)
    e = ((bits >> 23) & 0xff) + ((bits & 0x7fffff) != 0).to(torch.int32)
    return (e.clamp(1, 254) << 23).view(torch.float32)


def _ceil(a, b):
    return -(-a // b)


def _blocks(x, gm, gk):
    """[rows, k] -> ([ceil(rows / gm), ceil(k / gk)] maxima of the blocks' magnitudes, floored)."""
    rows, k = x.shape
    x = torch.nn.functional.pad(x.abs(), (0, _ceil(k, gk) * gk - k, 0, _ceil(rows, gm) * gm - rows))
    return x.view(_ceil(rows, gm), gm, _ceil(k, gk), gk).amax(dim=(1, 3)).clamp(1e-4)


def _spread(sf, gm, gk, rows, k):
    return sf.repeat_interleave(gm, 0)[:rows].repeat_interleave(gk, 1)[:, :k]


def _quantise(x, gm, gk):
    """e4m3 codes and fp32 power-of-two scales of the gm x gk blocks of x [rows, k]."""
    sf = _pow2_ceil(_blocks(x, gm, gk) / E4M3_MAX)
    return (x / _spread(sf, gm, gk, *x.shape)).to(torch.float8_e4m3fn), sf


def _quantise_e2m1(x, gk):
    """e2m1 codes packed two along k (even k in the low nibble) and the scales of 1 x gk blocks."""
    sf = _pow2_ceil(_blocks(x, 1, gk) / E2M1_MAX)
    y = x / _spread(sf, 1, gk, *x.shape)
    code = torch.zeros_like(y, dtype=torch.uint8)
    for bound in E2M1_BOUNDS:
        code += (y.abs() > bound).to(torch.uint8)
    code |= ((y < 0) & (code != 0)).to(torch.uint8) << 3
    return (code[:, ::2] | (code[:, 1::2] << 4)).contiguous().view(torch.int8), sf


def _generator(seed):
    return torch.Generator(device='cuda').manual_seed(seed)


def _normal(gen, rows, k, scale=1.0):
    return torch.randn(rows, k, device='cuda', generator=gen) * scale


def _stack(parts):
    return tuple(torch.stack(t) for t in zip(*parts))


def _packed(sf, mn, k, gran, is_sfa, **more):
    return deep_gemm.transform_sf_into_required_layout(sf, mn, k, gran, is_sfa=is_sfa, **more)


def _sizes(case):
    """Tokens of each group: a routing drawn from the case itself, so a case has one shape whatever the seed."""
    rng = random.Random('%d %d %d' % (case['groups'], case['tokens'], case['n']))
    share = [rng.uniform(0.7, 1.3) for _ in range(case['groups'])]
    sizes = [max(1, int(case['tokens'] * s / sum(share))) for s in share]
    sizes[-1] += max(0, case['tokens'] - sum(sizes))
    return sizes


def _psum(sizes, align):
    total, ends = 0, []
    for s in sizes:
        ends.append(total + s)
        total = _ceil(total + s, align) * align
    return total, ends


def _weights(gen, case, n, k):
    """(data, scale factors) of one weight matrix [n, k]; the scales in the kernels' layout, with its recipe."""
    x = _normal(gen, n, k, 1.0 / math.sqrt(k))
    if case['kind'] == 'bf16':
        return x.to(torch.bfloat16), None
    if case['kind'] == 'fp8fp4':
        return _quantise_e2m1(x, 32)
    return _quantise(x, 128, 128)


def _weight_gran(case):
    return (1, 32) if case['kind'] == 'fp8fp4' else (128, 128)


def _activations(gen, case, rows, k):
    x = _normal(gen, rows, k)
    return (x.to(torch.bfloat16), None) if case['kind'] == 'bf16' else _quantise(x, 1, 128)


def _align_of(case):
    return case.get('align', 256)


def prepare(case, seed):
    return globals()['_prepare_' + case['op']](dict(case), _generator(seed))


def _out_type(case):
    return torch.float32 if case.get('out') == 'fp32' else torch.bfloat16


def _prepare_dense(case, gen):
    m, n, k, form = case['m'], case['n'], case['k'], case['form']
    a, sfa = _activations(gen, case, m, k)
    if form == 'tn' and case['kind'] == 'fp8':
        b, sfb = _activations(gen, case, n, k)   # a weight gradient: both operands are activations
        grans = dict(recipe_a=(1, 128), recipe_b=(1, 128))
    else:
        b, sfb = _weights(gen, case, n, k)
        grans = dict(recipe_a=(1, 128), recipe_b=_weight_gran(case))
    if form[0] == 't':
        a, sfa = a.t().contiguous(), None if sfa is None else sfa.t().contiguous()
    if form[1] == 'n':
        b, sfb = b.t().contiguous(), None if sfb is None else sfb.t().contiguous()
    s = dict(case, d=torch.zeros(m, n, dtype=_out_type(case), device='cuda'))
    if case['kind'] == 'bf16':
        return dict(s, call=getattr(deep_gemm, 'bf16_gemm_' + form), a=a, b=b, keys={})
    if form == 'nt':
        sfb = _packed(sfb, n, k, grans['recipe_b'], False)
        grans['recipe_b'] = (1, 32)
        if case['sf'] == 'packed':
            sfa = _packed(sfa, m, k, grans['recipe_a'], True)
            grans['recipe_a'] = (1, 32)
    name = ('fp8_gemm_' if case['kind'] == 'fp8' else 'fp8_fp4_gemm_') + form
    return dict(s, call=getattr(deep_gemm, name), a=(a, sfa), b=(b, sfb), keys=grans)


def _prepare_contiguous(case, gen):
    groups, n, k, align = case['groups'], case['n'], case['k'], case['align']
    sizes = _sizes(case)
    total, ends = _psum(sizes, align)
    deep_gemm.set_mk_alignment_for_contiguous_layout(align)
    rows = torch.full((total,), -1, dtype=torch.int32)
    for g, (end, size) in enumerate(zip(ends, sizes)):
        rows[end - size:end] = g
    x = _normal(gen, total, k)
    x[(rows < 0).to(x.device)] = 0
    a, sfa = (x.to(torch.bfloat16), None) if case['kind'] == 'bf16' else _quantise(x, 1, 128)
    del x
    b, sfb = None, None
    if case['kind'] == 'bf16':
        b = torch.stack([_weights(gen, case, n, k)[0] for _ in range(groups)])
    else:
        b, sfb = _stack([_weights(gen, case, n, k) for _ in range(groups)])
    psum = case['layout'] == 'psum'
    layout = (torch.tensor(ends, dtype=torch.int32) if psum else rows).to('cuda')
    d = torch.zeros(total, n, dtype=torch.bfloat16, device='cuda')
    keys = dict(use_psum_layout=psum)
    nn = case['form'] == 'nn'
    if nn:
        b = b.transpose(1, 2).contiguous()
    s = dict(case, d=d, layout=layout, keys=keys)
    if case['kind'] == 'bf16':
        return dict(s, call=getattr(deep_gemm, 'm_grouped_bf16_gemm_%s_contiguous' % case['form']), a=a, b=b)
    keys.update(recipe_a=(1, 128), recipe_b=_weight_gran(case))
    sfb = _packed(sfb, n, k, keys['recipe_b'], False, num_groups=groups)
    if nn:
        sfb = sfb.transpose(1, 2)
    keys['recipe_b'] = (1, 32)
    if case['sf'] == 'packed':
        sfa = _packed(sfa, total, k, (1, 128), True, psum_layout=layout if psum else None)
        keys['recipe_a'] = (1, 32)
    name = 'm_grouped_%s_gemm_%s_contiguous' % ('fp8' if case['kind'] == 'fp8' else 'fp8_fp4', case['form'])
    return dict(s, call=getattr(deep_gemm, name), a=(a, sfa), b=(b, sfb))


def _masked_rows(case, gen):
    lo, hi = max(1, case['mean_m'] // 2), min(case['max_m'], case['mean_m'] * 3 // 2)
    return torch.randint(lo, hi + 1, (case['groups'],), device='cuda', generator=gen, dtype=torch.int32)


def _prepare_masked(case, gen):
    groups, max_m, n, k = case['groups'], case['max_m'], case['n'], case['k']
    masked = _masked_rows(case, gen)
    s = dict(case, masked=masked, d=torch.zeros(groups, max_m, n, dtype=torch.bfloat16, device='cuda'))
    if case['kind'] == 'bf16':
        return dict(s, call=deep_gemm.m_grouped_bf16_gemm_nt_masked, keys={},
                    a=torch.stack([_activations(gen, case, max_m, k)[0] for _ in range(groups)]),
                    b=torch.stack([_weights(gen, case, n, k)[0] for _ in range(groups)]))
    a, sfa = _stack([_activations(gen, case, max_m, k) for _ in range(groups)])
    b, sfb = _stack([_weights(gen, case, n, k) for _ in range(groups)])
    return dict(s, call=deep_gemm.m_grouped_fp8_gemm_nt_masked, keys={},
                a=(a, _packed(sfa, max_m, k, (1, 128), True, num_groups=groups)),
                b=(b, _packed(sfb, n, k, (128, 128), False, num_groups=groups)))


def _quantise_columns(x, gk):
    """e4m3 codes of x [k, mn] with one scale per column and gk rows: (codes, scales [k / gk, mn])."""
    q, sf = _quantise(x, gk, 1)
    return q, sf


def _prepare_kgrouped(case, gen):
    m, n = case['m'], case['n']
    sizes = _sizes(case)
    total, ends = _psum(sizes, 256)
    deep_gemm.set_mk_alignment_for_contiguous_layout(256)
    real = torch.zeros(total, 1, device='cuda')
    for end, size in zip(ends, sizes):
        real[end - size:end] = 1
    layout = torch.tensor(ends, dtype=torch.int32, device='cuda')
    d = torch.zeros(case['groups'], m, n, dtype=torch.float32, device='cuda')
    s = dict(case, d=d, layout=layout, sizes=sizes, keys={})
    if case['kind'] == 'bf16':
        return dict(s, call=deep_gemm.k_grouped_bf16_gemm_tn_contiguous, a=(_normal(gen, total, m) * real).to(torch.bfloat16),
                    b=(_normal(gen, total, n) * real).to(torch.bfloat16))
    return dict(s, call=deep_gemm.k_grouped_fp8_gemm_tn_contiguous, a=_quantise_columns(_normal(gen, total, m) * real, 32),
                b=_quantise_columns(_normal(gen, total, n) * real, 32))


def _prepare_einsum(case, gen):
    b, h, r, d = case['b'], case['h'], case['r'], case['d']
    a, sfa = _quantise(_normal(gen, b * h, r), 1, 32)
    w, sfw = _stack([_quantise(_normal(gen, d, r, 1.0 / math.sqrt(r)), 1, 32) for _ in range(h)])
    return dict(case, a=(a.view(b, h, r), sfa.view(b, h, -1)), b=(w, sfw),
                d=torch.zeros(b, h, d, dtype=torch.bfloat16, device='cuda'))


# ------------------------------------------------------------------------------------------- the call
def run(state):
    op, d = state['op'], state['d']
    if op == 'dense':
        state['call'](state['a'], state['b'], d, **state['keys'])
    elif op == 'contiguous':
        state['call'](state['a'], state['b'], d, state['layout'], **state['keys'])
    elif op == 'masked':
        state['call'](state['a'], state['b'], d, state['masked'], state['mean_m'])
    elif op == 'kgrouped':
        state['call'](state['a'], state['b'], d, state['sizes'], state['layout'])
    else:
        deep_gemm.fp8_einsum('bhr,hdr->bhd', state['a'], state['b'], d)
    return d


# ------------------------------------------------------------------------------------------- what it needs
def _operand_bytes(case, rows, k, weight):
    """Bytes of one operand and its scale factors as run() is given them."""
    if case['kind'] == 'bf16':
        return 2 * rows * k
    if weight:
        return rows * k // (2 if case['kind'] == 'fp8fp4' else 1) + rows * _ceil(k, 64) * 2
    return rows * k + (rows * _ceil(k, 64) * 2 if case['sf'] == 'packed' else rows * _ceil(k, 128) * 4)


def work(case):
    op = case['op']
    if op == 'dense':
        m, n, k = case['m'], case['n'], case['k']
        out = m * n * (4 if case.get('out') == 'fp32' else 2)
        return dict(flops=2.0 * m * n * k, bytes=_operand_bytes(case, m, k, False) + _operand_bytes(case, n, k, True) + out)
    if op == 'contiguous':
        sizes, n, k = _sizes(case), case['n'], case['k']
        total, valid = _psum(sizes, case['align'])[0], sum(sizes)
        return dict(flops=2.0 * valid * n * k, bytes=_operand_bytes(case, valid, k, False)
                    + _operand_bytes(case, case['groups'] * n, k, True) + 2 * total * n)
    if op == 'masked':
        lo, hi = max(1, case['mean_m'] // 2), min(case['max_m'], case['mean_m'] * 3 // 2)
        rows, n, k = int(case['groups'] * (lo + hi) / 2), case['n'], case['k']
        return dict(flops=2.0 * rows * n * k, bytes=_operand_bytes(case, rows, k, False)
                    + _operand_bytes(case, case['groups'] * n, k, True) + 2 * rows * n)
    if op == 'kgrouped':
        m, n, k = case['m'], case['n'], sum(_sizes(case))
        per = 2 * k if case['kind'] == 'bf16' else k + _ceil(k, 32) * 4
        return dict(flops=2.0 * m * n * k, bytes=(m + n) * per + 4 * case['groups'] * m * n)
    b, h, r, d = case['b'], case['h'], case['r'], case['d']
    return dict(flops=2.0 * b * h * r * d, bytes=(b * h + h * d) * (r + _ceil(r, 32) * 4) + 2 * b * h * d)


def tolerance(case):
    """What another order of the sums shows.  fp32 results: e4m3 products are off by 1.5e-5 of the result (the
    alignment of the products inside one matrix instruction, largest 1.4e-4), bf16 ones by 5e-7 (largest 5e-6);
    four times that.  bf16 results round the other way in the few places where such a difference decides (0.5e-4
    between K splits of bf16 products, 2.5e-4 expected from 1.5e-5), by one unit, 2^-7 of the value at most."""
    if case['op'] == 'kgrouped' or case.get('out') == 'fp32':
        return dict(rel=2.2e-6, max=2e-5) if case['kind'] == 'bf16' else dict(rel=6e-5, max=6e-4)
    return dict(rel=1e-3, max=0.016)


# ------------------------------------------------------------------------------------------- in 64 bits
def _e4m3(q, sf, gm, gk):
    return q.double() * _spread(sf, gm, gk, *q.shape).double()


def _e2m1(q, sf, gk):
    values = torch.tensor(E2M1_VALUES + tuple(-v for v in E2M1_VALUES), dtype=torch.float64, device='cuda')
    q = q.view(torch.uint8).int()
    x = torch.stack([values[q & 15], values[q >> 4]], dim=-1).flatten(1)
    return x * _spread(sf, 1, gk, *x.shape).double()


def _packed_scale(sf):
    """The fp64 scale of each 32 columns held by a packed scale tensor [mn, k / 64]."""
    x = sf.int() & 0xffff
    e = torch.stack([x & 255, x >> 8], dim=-1).flatten(1)
    return torch.exp2((e - 127).double())


def _values(case, data, sf, gran):
    if sf is None:
        return data.double()
    if sf.dtype == torch.int16:
        sf, gran = _packed_scale(sf), (1, 32)
    if data.dtype == torch.int8:
        return _e2m1(data, sf[:, :_ceil(2 * data.shape[1], 32)], 32)
    return _e4m3(data, sf, *gran)


def _pair(x):
    return x if isinstance(x, tuple) else (x, None)


def _product(a, b):
    return torch.matmul(a, b.t())


def exact(case, seed):
    s = prepare(case, seed)
    op = case['op']
    (a, sfa), (b, sfb) = _pair(s['a']), _pair(s['b'])
    if op == 'dense':
        ga, gb = s['keys'].get('recipe_a'), s['keys'].get('recipe_b')
        if case['form'][0] == 't':
            a, sfa = a.t(), None if sfa is None else sfa.t()
        if case['form'][1] == 'n':
            b, sfb = b.t(), None if sfb is None else sfb.t()
        return _product(_values(case, a, sfa, ga), _values(case, b, sfb, gb))
    if op == 'contiguous':
        out = torch.zeros(s['d'].shape, dtype=torch.float64, device='cuda')
        ends, sizes = _psum(_sizes(case), case['align'])[1], _sizes(case)
        for g, (end, size) in enumerate(zip(ends, sizes)):
            wb, ws = b[g], None if sfb is None else sfb[g]
            if case['form'] == 'nn':
                wb, ws = wb.t(), None if ws is None else ws.t()
            r = slice(end - size, end)
            out[r] = _product(_values(case, a[r], None if sfa is None else sfa[r], (1, 128)), _values(case, wb, ws, (1, 32)))
        return out
    if op == 'masked':
        out = torch.zeros(s['d'].shape, dtype=torch.float64, device='cuda')
        for g, rows in enumerate(s['masked'].tolist()):
            va = _values(case, a[g], None if sfa is None else sfa[g], (1, 32))
            out[g, :rows] = _product(va[:rows], _values(case, b[g], None if sfb is None else sfb[g], (1, 32)))
        return out
    if op == 'kgrouped':
        out = torch.zeros(s['d'].shape, dtype=torch.float64, device='cuda')
        va, vb = (x.double() if f is None else _e4m3(x, f, 32, 1) for x, f in ((a, sfa), (b, sfb)))
        start = 0
        for g, end in enumerate(s['layout'].tolist()):
            out[g] = torch.matmul(va[start:end].t(), vb[start:end])
            start = _ceil(end, 256) * 256
        return out
    out = torch.empty(s['d'].shape, dtype=torch.float64, device='cuda')
    for h in range(case['h']):
        out[:, h] = _product(_e4m3(a[:, h], sfa[:, h], 1, 32), _e4m3(b[h], sfb[h], 1, 32))
    return out
