"""The workloads this framework is timed on, through its public Python entry points.

Six kinds of work, each over the range of sizes it has in use:

    gemm          fp8_gemm on operands that are already quantised (an upstream kernel wrote e4m3 and scales)
    linear        per_token_group_quant_fp8 + fp8_gemm: a block-scaled FP8 linear layer on a 16- or 32-bit activation
    grouped       m_grouped_fp8_gemm_nt_contiguous: expert-contiguous rows (one projection of an MoE prefill)
    masked        m_grouped_fp8_gemm_nt_masked: fixed-capacity expert buffers (one projection of an MoE decode step)
    moe_prefill   fused_moe_v3: the whole expert MLP on the tokens one GPU received
    moe_decode    low_latency_experts on fixed-capacity buffers, then ep_gather back to token order

``draw`` takes sizes from the whole range of the same kinds, odd ones among them.
"""
import math

import torch

from dlblas_amd.kernels.fp8 import per_block_quant_fp8, per_token_group_quant_fp8
from dlblas_amd.kernels.fp8_gemm import fp8_gemm
from dlblas_amd.kernels.fp8_gemm_grouped import m_grouped_fp8_gemm_nt_contiguous, m_grouped_fp8_gemm_nt_masked
from dlblas_amd.kernels.fused_moe_v3 import ep_gather, fused_moe_v3
from dlblas_amd.kernels.moe import low_latency_experts

BLOCK = 128
DTYPES = {'bf16': torch.bfloat16, 'f16': torch.float16, 'f32': torch.float32}
BYTES = {'bf16': 2, 'f16': 2, 'f32': 4}
LARGEST_FLOPS = 2.0 * 4096 * 7168 * 18432  # the largest listed case; a drawn one stays below it
LARGEST_WEIGHT = 36864 * 7168
LARGEST_EXPERTS = 32 * 3 * 2048 * 7168


def _ceil(x, y):
    return -(-x // y)


def listed():
    return [
        # one token of a running sequence against a narrow projection: latency and launches
        dict(name='gemm_1x2112x7168', kind='gemm', m=1, n=2112, k=7168, out='bf16'),
        # a decode step of 16 sequences, quantiser included
        dict(name='linear_16x7168x2048', kind='linear', m=16, n=7168, k=2048, x='bf16', out='bf16'),
        # a decode step of an odd number of sequences against the narrow projection
        dict(name='linear_100x2112x7168', kind='linear', m=100, n=2112, k=7168, x='bf16', out='bf16'),
        # a chunk of a chunked prefill, odd length
        dict(name='gemm_500x4096x7168', kind='gemm', m=500, n=4096, k=7168, out='bf16'),
        # a layer whose sizes are multiples of no tile, with a ragged last K block, fp32 result
        dict(name='gemm_300x1000x1040_f32', kind='gemm', m=300, n=1000, k=1040, out='f32'),
        # prefill, compute-bound: the headline GEMM
        dict(name='gemm_4096x7168x18432', kind='gemm', m=4096, n=7168, k=18432, out='bf16'),
        # prefill with a short K and a wide output, quantiser included
        dict(name='linear_4096x24576x1536', kind='linear', m=4096, n=24576, k=1536, x='bf16', out='bf16'),
        # gate/up projection of 32 local experts on 8192 routed rows
        dict(name='grouped_32x8192_4096x7168', kind='grouped', e=32, tokens=8192, n=4096, k=7168, out='bf16'),
        # down projection of 32 local experts in a decode step, buffers of 256 rows filled to a random height
        dict(name='masked_32x256_7168x2048', kind='masked', e=32, cap=256, n=7168, k=2048, out='bf16'),
        # an expert MLP on a short chunk: about 16 rows per local expert, padded to 128
        dict(name='moe_prefill_500', kind='moe_prefill', tokens=500, e=32, total=256, topk=8, h=7168, i=2048),
        # the same on a full prefill batch
        dict(name='moe_prefill_8192', kind='moe_prefill', tokens=8192, e=32, total=256, topk=8, h=7168, i=2048),
        # an expert MLP in a decode step: 1024 sequences over all GPUs, about 32 rows per local expert
        dict(name='moe_decode_1024', kind='moe_decode', tokens=1024, cap=128, e=32, total=256, topk=8, h=7168, i=2048),
    ]


def _log_int(rng, lo, hi, multiple=1):
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / multiple)) * multiple))


def draw(rng):
    while True:
        kind = rng.choice(['gemm', 'gemm', 'linear', 'linear', 'grouped', 'masked', 'moe_prefill', 'moe_decode'])
        if kind in ('gemm', 'linear'):
            k = _log_int(rng, 512, 18432, 128)
            if kind == 'gemm' and rng.random() < 0.15:
                k = _log_int(rng, 512, 2048, 16)  # ragged last K block
            c = dict(kind=kind, m=_log_int(rng, 1, 4096), n=_log_int(rng, 512, 36864, rng.choice([1, 8, 64, 128])), k=k,
                     out=rng.choice(['bf16', 'bf16', 'bf16', 'f32']))
            if kind == 'linear':
                c['x'] = rng.choice(['bf16', 'bf16', 'f16', 'f32'])
            if c['n'] * c['k'] <= LARGEST_WEIGHT and 2.0 * c['m'] * c['n'] * c['k'] <= LARGEST_FLOPS:
                return c
            continue
        e = rng.choice([8, 16, 32])
        if kind in ('grouped', 'masked'):
            c = dict(kind=kind, e=e, n=_log_int(rng, 512, 7168, 128), k=_log_int(rng, 512, 7168, 128), out=rng.choice(['bf16', 'bf16', 'f32']))
            if kind == 'grouped':
                c['tokens'] = _log_int(rng, 64, 8192)
            else:
                c['cap'] = _log_int(rng, 16, 512, 8)
            return c
        c = dict(kind=kind, e=e, total=8 * e, topk=8, h=_log_int(rng, 1024, 7168, 128), i=_log_int(rng, 256, 2048, 128))
        if kind == 'moe_prefill':
            c['tokens'] = _log_int(rng, 64, 8192)
        else:
            c['tokens'] = _log_int(rng, 16, 2048)
            # capacity of an expert's buffer: well above the mean, as a serving program sizes it
            c['cap'] = max(64, _ceil(4 * c['tokens'] * c['topk'] // c['total'], 64) * 64)
        if 3 * c['e'] * c['h'] * c['i'] <= LARGEST_EXPERTS:
            return c


# --- inputs -------------------------------------------------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device='cuda').manual_seed(seed)


def _act(m, k, g, dtype='bf16'):
    return torch.randn(m, k, device='cuda', generator=g).to(DTYPES[dtype])


def _quantised_act(m, k, g):
    """[m, k] e4m3 codes of N(0, 1) activations and their 1 x 128 scales; a ragged last block has a scale of its own."""
    pad = _ceil(k, BLOCK) * BLOCK
    x = torch.zeros(m, pad, device='cuda', dtype=torch.bfloat16)
    x[:, :k] = _act(m, k, g)
    q, s = per_token_group_quant_fp8(x, BLOCK)
    return q[:, :k].contiguous(), s


def _weight(n, k, g):
    """[n, k] e4m3 codes of N(0, 0.02) weights and their 128 x 128 block scales."""
    return per_block_quant_fp8((torch.randn(n, k, device='cuda', generator=g) * 0.02).to(torch.bfloat16))


def _expert_weights(e, n, k, g):
    q = torch.empty(e, n, k, device='cuda', dtype=torch.float8_e4m3fn)
    s = torch.empty(e, _ceil(n, BLOCK), _ceil(k, BLOCK), device='cuda')
    for j in range(e):
        q[j], s[j] = _weight(n, k, g)
    return q, s


def _routing(tokens, topk, e, total, g):
    """topk distinct experts of `total` per token; the first `e` are local, the others are -1 as a dispatch leaves them."""
    ids = torch.rand(tokens, total, device='cuda', generator=g).topk(topk, dim=1).indices
    ids = torch.where(ids < e, ids, torch.full_like(ids, -1))
    weights = torch.softmax(torch.randn(tokens, topk, device='cuda', generator=g), dim=1)
    return ids, weights


def prepare(case, seed):
    g = _gen(seed)
    kind = case['kind']
    st = {'case': case}
    if kind == 'gemm':
        st['a'], st['a_s'] = _quantised_act(case['m'], case['k'], g)
        st['w'], st['w_s'] = _weight(case['n'], case['k'], g)
    elif kind == 'linear':
        st['x'] = _act(case['m'], case['k'], g, case['x'])
        st['w'], st['w_s'] = _weight(case['n'], case['k'], g)
    elif kind == 'grouped':
        e, n, k = case['e'], case['n'], case['k']
        # how uneven the routing is belongs to the case (the number of padded rows is then the same for every seed), which
        # expert is the busy one to the seed
        expert = torch.randint(0, e, (case['tokens'], ), device='cuda', generator=_gen(20))
        padded = (torch.bincount(expert, minlength=e) + BLOCK - 1) // BLOCK * BLOCK
        padded = padded[torch.randperm(e, device='cuda', generator=g)]
        st['m_indices'] = torch.repeat_interleave(torch.arange(e, device='cuda', dtype=torch.int32), padded)
        rows = st['m_indices'].numel()
        st['a'], st['a_s'] = _quantised_act(rows, k, g)
        st['w'], st['w_s'] = _expert_weights(e, n, k, g)
        st['out'] = torch.zeros(rows, n, device='cuda', dtype=DTYPES[case['out']])
    elif kind == 'masked':
        e, cap, n, k = case['e'], case['cap'], case['n'], case['k']
        st['masked_m'] = torch.randint(0, cap + 1, (e, ), device='cuda', generator=g, dtype=torch.int32)
        st['expected_m'] = int(st['masked_m'].float().mean())
        a, a_s = _quantised_act(e * cap, k, g)
        st['a'], st['a_s'] = a.view(e, cap, k), a_s.view(e, cap, -1)
        st['w'], st['w_s'] = _expert_weights(e, n, k, g)
        st['out'] = torch.zeros(e, cap, n, device='cuda', dtype=DTYPES[case['out']])
    elif kind == 'moe_prefill':
        e, h, i = case['e'], case['h'], case['i']
        st['x'] = _quantised_act(case['tokens'], h, g)
        st['ids'], st['weights'] = _routing(case['tokens'], case['topk'], e, case['total'], g)
        per_expert = torch.bincount(st['ids'][st['ids'] >= 0], minlength=e)
        st['counts'] = ((per_expert + BLOCK - 1) // BLOCK * BLOCK).tolist()
        st['w13'] = _expert_weights(e, 2 * i, h, g)
        st['w2'] = _expert_weights(e, h, i, g)
    else:
        e, cap, h, i = case['e'], case['cap'], case['h'], case['i']
        ids, st['weights'] = _routing(case['tokens'], case['topk'], e, case['total'], g)
        # slot rank inside its expert, in token order; rows beyond the capacity are dropped as a dispatch would
        flat = torch.where(ids < 0, e, ids).flatten()
        one_hot = torch.nn.functional.one_hot(flat, e + 1)[:, :e]
        rank = ((one_hot.cumsum(0) - 1) * one_hot).sum(1)
        keep = (flat < e) & (rank < cap)
        st['ids'] = torch.where(keep, flat, -1).view_as(ids)
        st['index'] = torch.where(keep, flat * cap + rank, 0).view_as(ids)
        st['masked_m'] = torch.bincount(flat[keep], minlength=e).to(torch.int32)
        st['expected_m'] = max(1, _ceil(case['tokens'] * case['topk'], case['total']))
        a, a_s = _quantised_act(e * cap, h, g)
        st['a'] = (a.view(e, cap, h), a_s.view(e, cap, -1))
        st['w13'] = _expert_weights(e, 2 * i, h, g)
        st['w2'] = _expert_weights(e, h, i, g)
        st['out'] = torch.zeros(case['tokens'], h, device='cuda', dtype=torch.bfloat16)
    return st


def _gemm(a, w, a_s, w_s, out):
    default = torch.get_default_dtype()
    torch.set_default_dtype(DTYPES[out])  # the type fp8_gemm returns
    try:
        return fp8_gemm(a, w, a_s, w_s)
    finally:
        torch.set_default_dtype(default)


def run(state):
    case = state['case']
    kind = case['kind']
    if kind == 'gemm':
        return _gemm(state['a'], state['w'], state['a_s'], state['w_s'], case['out'])
    if kind == 'linear':
        q, s = per_token_group_quant_fp8(state['x'], BLOCK)
        return _gemm(q, state['w'], s, state['w_s'], case['out'])
    if kind == 'grouped':
        m_grouped_fp8_gemm_nt_contiguous((state['a'], state['a_s']), (state['w'], state['w_s']), state['out'], state['m_indices'])
        return state['out']
    if kind == 'masked':
        m_grouped_fp8_gemm_nt_masked((state['a'], state['a_s']), (state['w'], state['w_s']), state['out'], state['masked_m'],
                                     state['expected_m'])
        return state['out']
    if kind == 'moe_prefill':
        return fused_moe_v3(state['x'], state['ids'], state['weights'], state['w13'], state['w2'], state['counts'])
    down = low_latency_experts(state['a'], *state['w13'], *state['w2'], state['masked_m'], state['expected_m'])
    ep_gather(down.view(-1, case['h']), state['ids'], state['weights'], state['index'], state['out'])
    return state['out']


# --- what a pass cannot do without --------------------------------------------------------------------------------


def _scales(rows, k):
    return 4 * rows * _ceil(k, BLOCK)


def _weight_bytes(n, k):
    return n * k + 4 * _ceil(n, BLOCK) * _ceil(k, BLOCK)


def _experts_hit(slots, e, total):
    """Expected number of the `e` local experts that at least one of `slots` routed slots lands on."""
    return e * (1.0 - (1.0 - 1.0 / total)**slots)


def work(case):
    kind = case['kind']
    if kind in ('gemm', 'linear'):
        m, n, k = case['m'], case['n'], case['k']
        read = m * k * BYTES[case['x']] if kind == 'linear' else m * k + _scales(m, k)
        return {'bytes': read + _weight_bytes(n, k) + m * n * BYTES[case['out']], 'flops': 2.0 * m * n * k}
    e = case['e']
    if kind == 'grouped':
        rows, n, k = case['tokens'], case['n'], case['k']
        hit = _experts_hit(rows, e, e)
        return {'bytes': rows * k + _scales(rows, k) + hit * _weight_bytes(n, k) + rows * n * BYTES[case['out']] + 4 * rows,
                'flops': 2.0 * rows * n * k}
    if kind == 'masked':
        rows, n, k = e * case['cap'] / 2, case['n'], case['k']
        return {'bytes': rows * k + _scales(rows, k) + e * _weight_bytes(n, k) + rows * n * BYTES[case['out']] + 4 * e,
                'flops': 2.0 * rows * n * k}
    h, i = case['h'], case['i']
    slots = case['tokens'] * case['topk']
    rows = slots * e / case['total']
    hit = _experts_hit(slots, e, case['total'])
    tables = slots * (8 + 4) + 4 * e
    read = case['tokens'] * h + _scales(case['tokens'], h) if kind == 'moe_prefill' else rows * h + _scales(rows, h) + 8 * slots
    return {'bytes': read + tables + hit * (_weight_bytes(2 * i, h) + _weight_bytes(h, i)) + 2 * case['tokens'] * h,
            'flops': 2.0 * rows * 3 * i * h}


def tolerance(case):
    """About four times the error measured against 64-bit sums: 1.4e-5 (largest 9e-5 of the rms) for fp32 results, which is
    the truncation of the e4m3 matrix instructions; 1.7e-3 (one ulp at most) for bf16 results; 2.6e-3 for the expert MLPs,
    where a value next to a rounding boundary of the second quantiser moves by a whole e4m3 step (largest 0.16)."""
    if case['kind'] in ('gemm', 'linear', 'grouped', 'masked'):
        if case['out'] == 'f32':
            return {'rel': 6e-5, 'max': 4e-4}
        return {'rel': 6e-3, 'max': 1.6e-2}
    return {'rel': 1e-2, 'max': 0.6}
