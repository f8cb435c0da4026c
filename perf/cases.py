"""The work that users of this framework have it do, as cases to be timed.

A case is one pass through the public entry points on inputs that are on the GPU already:

  step       one generation step on the packed cache: `PackedKVCache.append` + `attend`
  schedule   a whole scale schedule on the packed cache (one layer of one generation)
  masked     a whole sequence in one call under the block-causal next-scale mask (a key limit per query)
  producer   a step from the qkv projection's output on: `append_from_qkv` + `attend`, tokens-first result
  queries    few queries over a long cache that is there already
  rule       a whole schedule on the drop-in quantizers with the attention over their packed caches: `fused_step`
  dropin     a whole schedule through `VAR_Q.use_var_q`: every step hands out the dequantized cache
  shared     quantize + pack with groups that span tokens, then unpack + dequantize
  rows       quantize + pack with groups inside a token's channels, then unpack + dequantize
  codes      int8 codes to 32-bit words and back

K and V are normal values with a few channels fifteen times larger, as the tests have them.
"""
import math

import torch

from var_q_amd import VAR_Q, PackedKVCache, hooks, ops, pack_unpack, schedules
from var_q_amd.quant import fused_step

DTYPES = {'bf16': torch.bfloat16, 'fp16': torch.float16, 'fp32': torch.float32}
VAR_PATCHES = ','.join(str(p) for p in schedules.VAR_PATCH_NUMS)
INFINITY_PATCHES = ','.join(str(p) for p in schedules.INFINITY_PATCH_NUMS)
# dims of a [B,H,L,c] tensor that one scale spans
SPANS = {'head_dim': (0, 2), 'head': (0, 2, 3), 'token': (0, 1, 3), 'token_head': (0, 3), 'tensor': (0, 1, 2, 3)}


def listed():
    return [
        # the third scale of a schedule for one image (guided: batch 2): nothing to compute, all latency
        dict(name='early_step', kind='step', B=2, H=16, D=128, bits='4', group=128, start=5, n=16, layout='BHLc', dtype='bf16'),
        # its last scale: 4096 queries over 10 521 keys
        dict(name='last_step', kind='step', B=2, H=16, D=128, bits='4', group=128, start=6425, n=4096, layout='BHLc', dtype='bf16'),
        # four guided images over all 13 scales, a bit-width of its own for every head
        dict(name='mixed_schedule', kind='schedule', B=8, H=16, D=128, bits='2882888284244828', group=64, layout='BHLc', dtype='bf16',
             patches=INFINITY_PATCHES),
        # all 680 tokens of a sequence at once (scoring, or a training-style forward) in fp16, tokens first
        dict(name='masked_forward', kind='masked', B=8, H=16, D=64, bits='4', group=32, layout='BLHc', dtype='fp16', patches=VAR_PATCHES),
        # a middle scale behind the qkv projection: normalise, rotate, quantize, attend
        dict(name='producer_step', kind='producer', B=2, H=16, D=128, bits='4', group=128, start=1497, n=1024, l2norm=True, rope=True,
             dtype='bf16'),
        # a handful of queries over a long cache: reading the cache is the work
        dict(name='few_queries', kind='queries', B=2, H=16, D=128, bits='4', group=128, start=10521, n=16),
        # the shipped 8-bit rules, one layer over the whole schedule: batch 64 in fp16 and tokens first ...
        dict(name='rule_tokens_first', kind='rule', B=64, H=16, D=64, bits=8, method='G_SCALE_HEAD_DIM', layout='BLHc', dtype='fp16',
             symmetric=True, patches=VAR_PATCHES),
        # ... and one guided image, heads first
        dict(name='rule_heads_first', kind='rule', B=2, H=16, D=128, bits=8, method='G_SCALE_HEAD_DIM', layout='BHLc', dtype='bf16',
             symmetric=True, patches=INFINITY_PATCHES),
        # the reference's own call, with 30 heads
        dict(name='dropin_schedule', kind='dropin', B=8, H=30, D=64, bits=8, method='G_SCALE_HEAD_DIM', layout='BLHc', dtype='fp16',
             out='fp32', symmetric=True, patches=VAR_PATCHES),
        # a large cache tensor encoded with a scale per (head, channel) and decoded
        dict(name='shared_scales', kind='shared', B=32, H=30, L=680, D=64, bits=2, span='head_dim', dtype='bf16', out='bf16', symmetric=False),
        # an odd number of tokens, a row length that is no power of two
        dict(name='row_scales', kind='rows', B=3, H=7, L=1511, D=96, bits=4, group=32, dtype='fp32', out='fp32', symmetric=False),
        # codes whose rows do not fill their last word
        dict(name='ragged_codes', kind='codes', rows=40009, D=100, bits=4),
    ]


def _log(rng, lo, hi):
    """A whole number from lo to hi, spread over the logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def _patches(rng, most):
    """A schedule: growing patch numbers from 1 to at most `most`."""
    last, p = _log(rng, 4, most), [1]
    while p[-1] < last:
        p.append(min(last, max(p[-1] + 1, int(p[-1] * rng.uniform(1.1, 1.7)))))
    return ','.join(str(x) for x in p[-13:])


def _draw(rng):
    kind = rng.choice(('step', 'step', 'schedule', 'masked', 'producer', 'queries', 'rule', 'rule', 'dropin', 'shared', 'rows', 'codes'))
    D = rng.choice((64, 128))
    H = rng.choice((6, 8, 12, 16, 20, 24, 30))
    dtype = rng.choice(('bf16', 'fp16')) if D == 64 else 'bf16'
    layout = rng.choice(('BHLc', 'BLHc'))
    if kind in ('step', 'schedule', 'masked', 'producer', 'queries'):
        bits = rng.choice(('2', '4', '4', '8', 'mixed'))
        if bits == 'mixed':
            bits = ''.join(rng.choice('248') for _ in range(H))
        group = rng.choice((32, 64) if D == 64 else (64, 128, 128))
        case = dict(kind=kind, B=_log(rng, 1, 16), H=H, D=D, bits=bits, group=group)
        if kind == 'step':
            case.update(start=_log(rng, 1, 8192) - 1, n=_log(rng, 1, 4096), layout=layout, dtype=dtype)
        elif kind == 'producer':
            case.update(start=_log(rng, 1, 8192) - 1, n=_log(rng, 1, 4096), l2norm=rng.random() < 0.7, rope=rng.random() < 0.7, dtype='bf16')
        elif kind == 'queries':
            case.update(start=_log(rng, 1024, 42084), n=_log(rng, 1, 64))
        else:
            case.update(layout=layout, dtype=dtype, patches=_patches(rng, 40))
    elif kind in ('rule', 'dropin'):
        method = rng.choice(('G_SCALE_HEAD_DIM', 'G_SCALE_HEAD_DIM', 'G_TOKEN_HEAD', 'G_TOKEN', 'G_SCALE'))
        case = dict(kind=kind, B=_log(rng, 1, 64), H=H, D=D, bits=rng.choice((2, 4, 8, 8)), method=method, layout=layout, dtype=dtype,
                    symmetric=rng.random() < 0.7, patches=_patches(rng, 32))
        if kind == 'dropin':
            case['out'] = rng.choice(('fp32', 'fp32', dtype))
    elif kind == 'shared':
        case = dict(kind=kind, B=_log(rng, 1, 64), H=H, L=_log(rng, 1, 8192), D=rng.choice((40, 64, 64, 72, 96, 128, 128)),
                    bits=rng.choice((2, 4, 8)), span=rng.choice(tuple(SPANS)), dtype=rng.choice(tuple(DTYPES)), out=rng.choice(tuple(DTYPES)),
                    symmetric=rng.random() < 0.5)
    elif kind == 'rows':
        group = rng.choice((16, 32, 64, 128))
        case = dict(kind=kind, B=_log(rng, 1, 16), H=H, L=_log(rng, 1, 8192), D=group * rng.choice((1, 1, 2, 3)), bits=rng.choice((2, 4, 8)),
                    group=group, dtype=rng.choice(tuple(DTYPES)), out=rng.choice(tuple(DTYPES)), symmetric=rng.random() < 0.5)
    else:
        case = dict(kind=kind, rows=_log(rng, 1, 400000), D=_log(rng, 16, 256), bits=rng.choice((2, 4, 8)))
    return case


def draw(rng):
    while True:
        case = _draw(rng)
        w = work(case)
        # no more than the largest listed case, in time and in memory
        if w['bytes'] <= 6e8 and w['flops'] <= 1.5e12:
            return case


def _kv(shape, D, dtype, gen):
    x = torch.randn(*shape, device='cuda', generator=gen)
    few = torch.randperm(D, device='cuda', generator=gen)[:max(1, round(0.02 * D))]
    x[..., few] *= 15.0
    return x.to(dtype)


def _bits(case):
    return int(case['bits']) if len(case['bits']) == 1 else [int(b) for b in case['bits']]


def _counts(case):
    return [int(p) ** 2 for p in case['patches'].split(',')]


def _step_inputs(case, n, gen):
    """q (heads first, in the attention's type), k and v of a step of n tokens."""
    B, H, D = case['B'], case['H'], case['D']
    shape = (B, n, H, D) if case['layout'] == 'BLHc' else (B, H, n, D)
    q = torch.randn(B, H, n, D, device='cuda', generator=gen).to(DTYPES[case['dtype']])
    return q, _kv(shape, D, DTYPES[case['dtype']], gen), _kv(shape, D, DTYPES[case['dtype']], gen)


def prepare(case, seed):
    gen = torch.Generator(device='cuda').manual_seed(seed)
    kind, D = case['kind'], case['D']
    st = dict(case=case, scale=1.0 / math.sqrt(D))
    if kind in ('step', 'schedule', 'masked', 'producer', 'queries'):
        B, H = case['B'], case['H']
        total = sum(_counts(case)) if 'patches' in case else case['start'] + (0 if kind == 'queries' else case['n'])
        st['cache'] = PackedKVCache(B, H, total, D, _bits(case), case['group'], 'cuda')
        if kind == 'schedule':
            st['steps'] = [_step_inputs(case, n, gen) for n in _counts(case)]
        elif kind == 'masked':
            st['steps'] = [_step_inputs(case, total, gen)]
            st['limit'] = schedules.kv_limit([int(p) for p in case['patches'].split(',')], device='cuda')
        else:
            if case['start']:
                st['cache'].append(*(_kv((B, H, case['start'], D), D, torch.bfloat16, gen) for _ in range(2)))
            if kind == 'step':
                st['steps'] = [_step_inputs(case, case['n'], gen)]
            elif kind == 'producer':
                st['qkv'] = _kv((B, case['n'], 3, H, D), D, DTYPES[case['dtype']], gen)
                st['mul'] = torch.rand(H, device='cuda', generator=gen) * 4 + 2 if case['l2norm'] else None
                side = math.isqrt(total - 1) + 1
                cos, sin = hooks.rope2d_tables(D, [(side, side)], max_hw=max(128, side))
                st['rope'] = (cos.cuda(), sin.cuda()) if case['rope'] else None
            else:
                st['q'] = torch.randn(B, H, case['n'], D, device='cuda', generator=gen).bfloat16()
    elif kind in ('rule', 'dropin'):
        steps = [_step_inputs(case, n, gen) for n in _counts(case)]
        st['steps'] = [(q.transpose(1, 2).contiguous() if case['layout'] == 'BLHc' else q, k, v) for q, k, v in steps]
    elif kind in ('shared', 'rows'):
        st['x'] = _kv((case['B'], case['H'], case['L'], D), D, DTYPES[case['dtype']], gen)
    else:
        half = 1 << (case['bits'] - 1)
        st['codes'] = torch.randint(-half, half, (case['rows'], D), device='cuda', generator=gen, dtype=torch.int8)
    return st


def _quantizers(case):
    """What a module sets up when a generation begins."""
    pair = [VAR_Q(case['bits'], case['layout'], case['method'], symmetric=case['symmetric']) for _ in range(2)]
    for z in pair:
        z.reserve_tokens(sum(_counts(case)))
    return pair


def run(st):
    case, scale = st['case'], st['scale']
    kind = case['kind']
    if kind in ('step', 'schedule', 'masked'):
        cache = st['cache']
        cache.len = case.get('start', 0)       # (the same step again)
        outs = []
        for q, k, v in st['steps']:
            cache.append(k, v, layout=case['layout'])
            outs.append(cache.attend(q, scale, kv_limit=st.get('limit')))
        return {'out': outs, 'cache': cache.tensors()}
    if kind == 'producer':
        cache = st['cache']
        cache.len = case['start']
        q = cache.append_from_qkv(st['qkv'], st['mul'], case['l2norm'], rope=st['rope'])
        return {'q': q, 'out': cache.attend(q, 1.0 if case['l2norm'] else scale, out_layout='BLHc'), 'cache': cache.tensors()}
    if kind == 'queries':
        return st['cache'].attend(st['q'], scale)
    if kind == 'rule':
        kq, vq = _quantizers(case)
        return {'out': [fused_step(q, k, v, kq, vq, scale) for q, k, v in st['steps']], 'k': kq.cached_item, 'v': vq.cached_item}
    if kind == 'dropin':
        kq, vq = _quantizers(case)
        out = DTYPES[case['out']]
        return [(kq.use_var_q(k, out), vq.use_var_q(v, out)) for _, k, v in st['steps']]
    if kind == 'shared':
        words, s, z = ops.quant_pack(st['x'], SPANS[case['span']], case['bits'], asym=not case['symmetric'])
        return {'words': words, 'scale': s, 'zp': z, 'x': ops.dequant(words, s, z, case['D'], case['bits'], DTYPES[case['out']])}
    if kind == 'rows':
        words, s, z = ops.quant_pack_rows(st['x'], case['group'], case['bits'], asym=not case['symmetric'])
        return {'words': words, 'scale': s, 'zp': z, 'x': ops.dequant(words, s, z, case['D'], case['bits'], DTYPES[case['out']])}
    words, meta = pack_unpack.pack_last_dim_to_int32_hip(st['codes'], case['bits'])
    return {'words': words, 'codes': pack_unpack.unpack_last_dim_from_int32_hip(words, meta)}


def _size(name):
    return 4 if name == 'fp32' else 2


def work(case):
    kind, D = case['kind'], case['D']
    nbytes = flops = 0
    if kind in ('step', 'schedule', 'masked', 'producer', 'queries'):
        B, H, size = case['B'], case['H'], _size(case.get('dtype', 'bf16'))
        per_head = [int(b) for b in case['bits']] * (H if len(case['bits']) == 1 else 1)
        token = 2 * B * sum(D * b // 8 + D // case['group'] * 8 for b in per_head)     # K and V of one token, packed
        len_, counts = case.get('start', 0), [case.get('n', 0)]
        if kind == 'schedule':
            counts = _counts(case)
        if kind == 'masked':
            counts = [sum(_counts(case))]
        for n in counts:
            if kind == 'producer':
                nbytes += n * token + 3 * B * n * H * D * size + B * n * H * D * 2       # qkv in, packed k and v and q out
            elif kind != 'queries':
                nbytes += n * token + 2 * B * n * H * D * size
            len_ += 0 if kind == 'queries' else n
            nbytes += len_ * token + 2 * B * n * H * D * 2                               # the cache, q in, out
            flops += 4 * B * H * n * len_ * D
        if kind == 'masked':
            ns = _counts(case)
            flops = 4 * B * H * D * sum(n * sum(ns[:i + 1]) for i, n in enumerate(ns))
    elif kind in ('rule', 'dropin'):
        B, H, size, len_ = case['B'], case['H'], _size(case['dtype']), 0
        for n in _counts(case):
            len_ += n
            nbytes += 2 * B * n * H * D * size + 2 * B * n * H * D * case['bits'] // 8 + 2 * B * len_ * H * D * case['bits'] // 8
            if kind == 'rule':
                nbytes += 2 * B * n * H * D * 2
                flops += 4 * B * H * n * len_ * D
            else:
                nbytes += 2 * B * len_ * H * D * _size(case['out'])
    elif kind in ('shared', 'rows'):
        rows = case['B'] * case['H'] * case['L']
        nbytes = rows * D * (_size(case['dtype']) + _size(case['out'])) + 2 * rows * (D * case['bits'] // 8)
        if kind == 'rows':
            nbytes += 2 * rows * D // case['group'] * (4 if case['symmetric'] else 8)
    else:
        nbytes = 2 * case['rows'] * (D + D * case['bits'] // 8)
    return {'bytes': nbytes, 'flops': flops}


def tolerance(case):
    # codes, scales and dequantized values are fixed to the bit; attention rounds its weights and its result to 16 bits
    if case['kind'] in ('dropin', 'shared', 'rows', 'codes'):
        return 'exact'
    return {'rel': 1e-2, 'max': 0.2}
