"""The work a program gives this framework, as cases that can be timed and compared.

Every public operator is here, from one token of a decode step to the largest prefill: the FP8 block-scaled GEMM (from
quantised and from bf16 activations), the 16-bit GEMM in both types, the fp32 GEMM with alpha and beta, both grouped
layouts and both quantisers. `listed` names twelve of them, `draw` gives more from the same ranges.

A case of kind 'decode' is a pass over `layers` weight matrices of one shape, each with activations of its own: what a
decoding step of a model does, whose weights do not fit any cache.
"""
import math

import torch

import yan_amd as yan

DTYPES = {'bf16': torch.bfloat16, 'fp16': torch.half, 'fp32': torch.float32}
BLOCK = 128         # one scale block along K; also the row alignment of a group in the contiguous layout


def listed():
    return [
        # one token against one projection with few outputs: the smallest call, all latency
        {'name': 'fp8_one_token', 'kind': 'decode', 'op': 'fp8', 'm': 1, 'n': 2112, 'k': 7168, 'layers': 1},
        # a decode step of 64 sequences from bf16 activations, quantised on the way, over twelve projections
        {'name': 'fp8_decode_64', 'kind': 'decode', 'op': 'bf16_fp8', 'm': 64, 'n': 4096, 'k': 7168, 'layers': 12},
        # a decode step of an unquantised model with a batch that is no multiple of anything
        {'name': 'bf16_decode_37', 'kind': 'decode', 'op': 'bf16', 'm': 37, 'n': 4096, 'k': 7168, 'layers': 8},
        # a chunk of a prompt with a ragged number of tokens, activation scales as row-major code hands them over
        {'name': 'fp8_chunk_1023', 'kind': 'fp8', 'm': 1023, 'n': 7168, 'k': 4096, 'scales': 'row_major'},
        # prefill of 4096 tokens, the headline shape, scales as the quantiser of this framework writes them
        {'name': 'fp8_prefill_4096', 'kind': 'fp8', 'm': 4096, 'n': 7168, 'k': 7168, 'scales': 'token_contiguous'},
        # fp16 with every dimension ragged: a vocabulary slice, an inner size that is no multiple of 64
        {'name': 'fp16_ragged', 'kind': 'half', 'dtype': 'fp16', 'm': 1111, 'n': 5004, 'k': 2056},
        # a large bf16 layer
        {'name': 'bf16_8192', 'kind': 'half', 'dtype': 'bf16', 'm': 8192, 'n': 8192, 'k': 8192},
        # fp32 with few rows and a long K, accumulated onto what is in c
        {'name': 'fp32_few_rows', 'kind': 'float', 'm': 128, 'n': 2112, 'k': 7168, 'alpha': 1.0, 'beta': 1.0},
        # mixture of experts, prefill: tokens of sixteen experts, as many each as the router sends
        {'name': 'moe_prefill', 'kind': 'contiguous', 'groups': 16, 'rows': 6144, 'n': 4096, 'k': 7168},
        # mixture of experts, decode: 32 experts on this GPU with about eight tokens each in fixed slots of 64
        {'name': 'moe_decode', 'kind': 'masked', 'groups': 32, 'm_max': 64, 'expected_m': 8, 'n': 4096, 'k': 7168},
        # activations on their way into an FP8 GEMM
        {'name': 'quantise_tokens', 'kind': 'per_token', 'dtype': 'bf16', 'm': 4096, 'k': 7168, 'col_major': True},
        # weights at load time or after an update
        {'name': 'quantise_weights', 'kind': 'per_block', 'dtype': 'bf16', 'n': 7168, 'k': 7168},
    ]


MOST_FLOP = 2.0 * 8192 ** 3         # bf16_8192; fp32 runs at a sixteenth of the rate
MOST_BYTES = 1.2e9


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _multiple(rng, low, high, of):
    return min(high, max(low, _log(rng, low, high) // of * of))


def _outputs(rng, low, high):
    """Output features: multiples of 64 as models have them, or, one time in four, a ragged size (n % 4 == 0)."""
    return _multiple(rng, low, high, 4 if rng.random() < 0.25 else 64)


def _candidate(rng):
    kind = rng.choice(['decode', 'decode', 'fp8', 'fp8', 'half', 'half', 'float', 'contiguous', 'masked', 'per_token', 'per_block'])
    if kind == 'decode':
        op = rng.choice(['fp8', 'bf16_fp8', 'bf16', 'fp16'])
        return {'kind': kind, 'op': op, 'm': _log(rng, 1, 128), 'n': _outputs(rng, 1024, 16384), 'k': _multiple(rng, 1024, 16384, 128),
                'layers': _log(rng, 1, 12)}
    if kind == 'fp8':
        return {'kind': kind, 'm': _log(rng, 128, 8192), 'n': _outputs(rng, 1024, 16384), 'k': _multiple(rng, 512, 16384, 128),
                'scales': rng.choice(['row_major', 'token_contiguous'])}
    if kind == 'half':
        k_step = 8 if rng.random() < 0.25 else 64
        return {'kind': kind, 'dtype': rng.choice(['bf16', 'fp16']), 'm': _log(rng, 128, 8192), 'n': _outputs(rng, 1024, 16384),
                'k': _multiple(rng, 512, 16384, k_step)}
    if kind == 'float':
        return {'kind': kind, 'm': _multiple(rng, 128, 4096, 128), 'n': _multiple(rng, 256, 8192, 64), 'k': _log(rng, 256, 8192),
                'alpha': 1.0, 'beta': rng.choice([0.0, 1.0])}
    if kind == 'contiguous':
        groups = _log(rng, 4, 64)
        return {'kind': kind, 'groups': groups, 'rows': _multiple(rng, 1024, 16384, BLOCK), 'n': _multiple(rng, 1024, 7168, 64),
                'k': _multiple(rng, 1024, 7168, 128)}
    if kind == 'masked':
        m_max = rng.choice([64, 128, 256])
        return {'kind': kind, 'groups': _log(rng, 4, 64), 'm_max': m_max, 'expected_m': _log(rng, 1, m_max // 2),
                'n': _multiple(rng, 1024, 7168, 64), 'k': _multiple(rng, 1024, 7168, 128)}
    if kind == 'per_token':
        return {'kind': kind, 'dtype': rng.choice(['bf16', 'fp32']), 'm': _log(rng, 1, 16384), 'k': _multiple(rng, 1024, 16384, 128),
                'col_major': rng.random() < 0.7}
    return {'kind': kind, 'dtype': rng.choice(['bf16', 'fp32']), 'n': _outputs(rng, 1024, 16384), 'k': _multiple(rng, 1024, 16384, 128)}


def draw(rng):
    while True:
        case = _candidate(rng)
        need = work(case)
        if need['bytes'] <= MOST_BYTES and need['flops'] * (16 if case['kind'] == 'float' else 1) <= MOST_FLOP:
            return case


def _activations(gen, *shape, dtype=torch.bfloat16):
    """N(0, 1) with a few features twenty times as large, as hidden states have them."""
    x = torch.randn(*shape, generator=gen, device='cuda', dtype=torch.float32)
    loud = torch.rand(shape[-1], generator=gen, device='cuda') < 0.004
    return torch.where(loud, 20.0 * x, x).to(dtype)


def _weights(gen, n, k, dtype=torch.bfloat16):
    return (torch.randn(n, k, generator=gen, device='cuda', dtype=torch.float32) * k ** -0.5).to(dtype)


def _quantised_weights(gen, groups, n, k):
    q = torch.empty((groups, n, k), dtype=torch.float8_e4m3fn, device='cuda')
    scales = torch.empty((groups, -(-n // BLOCK), k // BLOCK), dtype=torch.float32, device='cuda')
    for g in range(groups):
        q[g], scales[g] = yan.per_block_cast_to_fp8(_weights(gen, n, k))
    return q, scales


def prepare(case, seed):
    gen = torch.Generator(device='cuda')
    gen.manual_seed(seed)
    kind = case['kind']
    bf16 = torch.bfloat16
    state = {'kind': kind}
    if kind == 'decode':
        m, n, k, op = case['m'], case['n'], case['k'], case['op']
        calls = []
        for _ in range(case['layers']):
            x = _activations(gen, m, k, dtype=torch.half if op == 'fp16' else bf16)
            out = torch.zeros((m, n), dtype=x.dtype, device='cuda')
            if op in ('fp8', 'bf16_fp8'):
                w = tuple(t[0] for t in _quantised_weights(gen, 1, n, k))
                calls.append((yan.per_token_cast_to_fp8(x, col_major_scales=True) if op == 'fp8' else x, w, out))
            else:
                calls.append((x, _weights(gen, n, k, x.dtype), out))
        state['fn'] = {'fp8': yan.gemm_fp8_fp8_bf16_nt, 'bf16_fp8': yan.gemm_bf16_fp8_bf16_nt, 'bf16': yan.gemm_bf16_tn,
                       'fp16': yan.gemm_fp16_tn}[op]
        state['calls'] = calls
    elif kind == 'fp8':
        m, n, k = case['m'], case['n'], case['k']
        state['lhs'] = yan.per_token_cast_to_fp8(_activations(gen, m, k), col_major_scales=case['scales'] == 'token_contiguous')
        state['rhs'] = tuple(t[0] for t in _quantised_weights(gen, 1, n, k))
        state['out'] = torch.zeros((m, n), dtype=bf16, device='cuda')
    elif kind == 'half':
        dtype = DTYPES[case['dtype']]
        state['fn'] = yan.gemm_bf16_tn if dtype == bf16 else yan.gemm_fp16_tn
        state['lhs'] = _activations(gen, case['m'], case['k'], dtype=dtype)
        state['rhs'] = _weights(gen, case['n'], case['k'], dtype)
        state['out'] = torch.zeros((case['m'], case['n']), dtype=dtype, device='cuda')
    elif kind == 'float':
        m, n, k = case['m'], case['n'], case['k']
        state['lhs'] = torch.randn(k, m, generator=gen, device='cuda').t()                   # first dimension contiguous
        state['rhs'] = (torch.randn(k, n, generator=gen, device='cuda') * k ** -0.5).t()
        state['start'] = torch.randn(m, n, generator=gen, device='cuda')
        state['out'] = torch.zeros((m, n), device='cuda')
        state['alpha'], state['beta'] = case['alpha'], case['beta']
    elif kind == 'contiguous':
        groups, rows, n, k = case['groups'], case['rows'], case['n'], case['k']
        # the router's choice, block by block: popular experts get more
        popular = torch.rand(groups, generator=gen, device='cuda') + 0.25
        blocks = torch.multinomial(popular, rows // BLOCK, replacement=True, generator=gen).sort().values
        state['indices'] = blocks.to(torch.int32).repeat_interleave(BLOCK)
        state['lhs'] = yan.per_token_cast_to_fp8(_activations(gen, rows, k), col_major_scales=True)
        state['rhs'] = _quantised_weights(gen, groups, n, k)
        state['out'] = torch.zeros((rows, n), dtype=bf16, device='cuda')
    elif kind == 'masked':
        groups, m_max, n, k = case['groups'], case['m_max'], case['n'], case['k']
        rate = torch.full((groups,), float(case['expected_m']), device='cuda')
        state['masked_m'] = torch.poisson(rate, generator=gen).clamp(max=m_max).to(torch.int32)
        state['expected_m'] = case['expected_m']
        q, scales = yan.per_token_cast_to_fp8(_activations(gen, groups * m_max, k))
        state['lhs'] = q.view(groups, m_max, k), yan.get_col_major_tensor(scales.view(groups, m_max, k // BLOCK))
        state['rhs'] = _quantised_weights(gen, groups, n, k)
        state['out'] = torch.zeros((groups, m_max, n), dtype=bf16, device='cuda')
    elif kind == 'per_token':
        state['x'] = _activations(gen, case['m'], case['k'], dtype=DTYPES[case['dtype']])
        state['col_major'] = case['col_major']
    else:
        state['x'] = _weights(gen, case['n'], case['k'], DTYPES[case['dtype']])
    return state


def run(state):
    kind = state['kind']
    if kind == 'decode':
        fn = state['fn']
        for x, w, out in state['calls']:
            fn(x, w, out)
        return [out for _, _, out in state['calls']]
    if kind == 'fp8':
        yan.gemm_fp8_fp8_bf16_nt(state['lhs'], state['rhs'], state['out'])
    elif kind == 'half':
        state['fn'](state['lhs'], state['rhs'], state['out'])
    elif kind == 'float':
        if state['beta'] != 0.0:
            state['out'].copy_(state['start'])          # what the program has accumulated so far
        yan.gemm_float_nt(state['lhs'], state['rhs'], state['out'], state['alpha'], state['beta'])
    elif kind == 'contiguous':
        yan.m_grouped_gemm_fp8_fp8_bf16_nt_contiguous(state['lhs'], state['rhs'], state['out'], state['indices'])
    elif kind == 'masked':
        yan.m_grouped_gemm_fp8_fp8_bf16_nt_masked(state['lhs'], state['rhs'], state['out'], state['masked_m'], state['expected_m'])
    elif kind == 'per_token':
        return yan.per_token_cast_to_fp8(state['x'], col_major_scales=state['col_major'])
    else:
        return yan.per_block_cast_to_fp8(state['x'])
    return state['out']


def work(case):
    kind = case['kind']
    if kind in ('per_token', 'per_block'):
        rows, k = case['m' if kind == 'per_token' else 'n'], case['k']
        groups = rows * (k // BLOCK) if kind == 'per_token' else -(-rows // BLOCK) * (k // BLOCK)
        return {'bytes': rows * k * ((2 if case['dtype'] == 'bf16' else 4) + 1) + 4 * groups, 'flops': 0}
    n, k = case['n'], case['k']
    if kind == 'float':
        m = case['m']
        return {'bytes': 4 * (m * k + n * k + m * n * (3 if case['beta'] else 1)), 'flops': 2 * m * n * k}
    if kind == 'contiguous':
        m, weights = case['rows'], min(case['groups'], case['rows'] // BLOCK)
    elif kind == 'masked':
        m = case['groups'] * case['expected_m']
        weights = case['groups'] * (1 - math.exp(-case['expected_m']))          # experts that got a token at all
    else:
        m, weights = case['m'], 1
    eight_bit = kind in ('fp8', 'contiguous', 'masked') or case.get('op') in ('fp8', 'bf16_fp8')
    if eight_bit:
        x_bytes = 2 * m * k if case.get('op') == 'bf16_fp8' else m * k + 4 * m * (k // BLOCK)
        w_bytes = weights * (n * k + 4 * -(-n // BLOCK) * (k // BLOCK))
    else:
        x_bytes, w_bytes = 2 * m * k, 2 * n * k
    layers = case.get('layers', 1)
    return {'bytes': layers * (x_bytes + w_bytes + 2 * m * n), 'flops': layers * 2 * m * n * k}


def tolerance(case):
    """About four times what each path showed against itself in 64 bits, rounded to the output's type. FP8: rel 4e-4 (the
    matrix core drops product bits inside a block of 128), bf16 4e-5, fp16 1.3e-5, and one step of the output's type at
    the most in a single value; fp32: rel 1.2e-6 and max 1.2e-5 against the same sums in the opposite order."""
    kind = case['kind']
    if kind in ('per_token', 'per_block'):
        return 'exact'
    if kind == 'float':
        return {'rel': 5e-6, 'max': 5e-5}
    dtype = case.get('dtype') or case.get('op')
    if dtype == 'fp16':
        return {'rel': 6e-5, 'max': 4e-3}
    return {'rel': 2e-4 if dtype == 'bf16' else 1.6e-3, 'max': 0.03}
