"""What this framework is asked to do, as timed cases: the FP8 / FP4 GEMMs of dense
and MoE layers (decode, chunked prefill, prefill, backward), the activation cast
and whole MoE layers on one GPU, over the sizes of the repository's tests and
benchmark. `listed()` names the cases, `draw(rng)` gives more of the same ranges;
`prepare` builds a case's state on the GPU, `run` is one pass through the public
entry points, `exact` the same result in 64 bits from plain torch."""
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), 'deepgemm-amd_amd'))
import deep_gemm  # noqa: E402

DEV = 'cuda'
# (N, K) of the dense layers in the repository's tests, and of the grouped ones.
DENSE_NK = ((2112, 7168), (576, 7168), (24576, 1536), (32768, 512), (7168, 16384), (4096, 7168), (7168, 2048))
DGRAD_NK = ((7168, 2112), (7168, 576), (1536, 24576), (512, 32768), (16384, 7168), (7168, 4096), (2048, 7168))
GROUPED_NK = ((4096, 7168), (7168, 2048), (6144, 7168), (7168, 3072), (4096, 4096), (4096, 2048))


def listed():
    return [
        # A decode step's projection: 64 sequences, one token each (latency, launches).
        dict(name='dense_decode', kind='dense', m=64, n=2112, k=7168, sfa='k'),
        # A prefill chunk or a large decode batch of odd size.
        dict(name='dense_chunk', kind='dense', m=517, n=4096, k=7168, sfa='k'),
        # Prefill of 4096 tokens, the longest K of the dense layers.
        dict(name='dense_prefill', kind='dense', m=4096, n=7168, k=16384, sfa='mn'),
        # Backward, gradient of the input: K is the layer's N, not a multiple of 128.
        dict(name='dense_dgrad', kind='dense', m=4096, n=7168, k=2112, sfa='k'),
        # Backward, gradients of the expert weights, accumulated into FP32.
        dict(name='wgrad_grouped', kind='wgrad', groups=8, m=4096, n=7168, mean_k=4096),
        # MoE prefill: 8 experts, 32768 tokens split unevenly.
        dict(name='moe_contiguous', kind='contiguous', groups=8, tokens=32768, n=4096, k=7168, sfa='k'),
        # MoE decode: 16 experts with about 128 rows each.
        dict(name='moe_masked', kind='masked', groups=16, max_m=256, rows=128, n=4096, k=7168, sfa='k'),
        # Prefill with FP4 weights (MX scales packed once).
        dict(name='fp4_prefill', kind='fp4', m=4096, n=7168, k=7168),
        # MoE decode with FP4 weights.
        dict(name='fp4_masked', kind='fp4_masked', groups=16, max_m=256, rows=64, n=4096, k=7168),
        # Activation cast ahead of a GEMM.
        dict(name='cast', kind='cast', m=4096, k=7168, sfa='mn'),
        # A whole MoE layer in prefill: cast, dispatch, gate/up with SwiGLU, down, combine.
        dict(name='layer_prefill', kind='layer', tokens=4096, experts=32, topk=8, hidden=2048, inter=1024,
             layout='contiguous', fused=True),
        # The same in decode, in the masked layout, at the large hidden size.
        dict(name='layer_decode', kind='layer', tokens=128, experts=32, topk=8, hidden=7168, inter=2048,
             layout='masked', fused=True),
    ]


def _log(rng, lo, hi):
    """An integer spread evenly over the logarithm of [lo, hi]."""
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    kind = rng.choice(('dense', 'dense', 'dense', 'wgrad', 'contiguous', 'masked', 'fp4', 'fp4_masked', 'cast', 'layer'))
    major = rng.choice(('k', 'mn'))
    if kind == 'dense':
        how = rng.random()
        if how < 0.5:
            n, k = rng.choice(DENSE_NK)
        elif how < 0.7:
            n, k = rng.choice(DGRAD_NK)
        else:   # any layer: N a multiple of 8, K of 16
            n, k = 8 * _log(rng, 32, 1024), 16 * _log(rng, 16, 512)
        return dict(kind=kind, m=_log(rng, 1, 8192), n=n, k=k, sfa=major)
    if kind == 'wgrad':   # groups 0: one dense weight gradient
        return dict(kind=kind, groups=rng.choice((0, 1, 2, 4, 8)), m=rng.choice((576, 2112, 4096, 7168)),
                    n=rng.choice((2048, 4096)), mean_k=128 * _log(rng, 4, 32))
    if kind == 'contiguous':
        n, k = rng.choice(GROUPED_NK)
        return dict(kind=kind, groups=rng.choice((4, 8, 16, 32)), tokens=_log(rng, 1024, 32768), n=n, k=k, sfa=major)
    if kind in ('masked', 'fp4_masked'):
        n, k = rng.choice(GROUPED_NK)
        rows = _log(rng, 2, 256)
        case = dict(kind=kind, groups=rng.choice((4, 6, 8, 16, 32)), max_m=rng.choice((256, 512, 1024)), rows=rows,
                    n=n, k=k)
        return dict(case, sfa=major) if kind == 'masked' else case
    if kind == 'fp4':
        n, k = rng.choice(((2112, 7168), (24576, 1536), (4096, 7168), (7168, 2048), (7168, 7168)))
        return dict(kind=kind, m=_log(rng, 1, 4096), n=n, k=k)
    if kind == 'cast':
        return dict(kind=kind, m=_log(rng, 1, 32768), k=8 * _log(rng, 64, 2048), sfa=major)
    if rng.random() < 0.5:
        return dict(kind=kind, tokens=_log(rng, 256, 4096), experts=rng.choice((8, 16, 32, 64)), topk=rng.choice((2, 4, 8)),
                    hidden=rng.choice((1024, 2048, 4096)), inter=rng.choice((512, 768, 1024)), layout='contiguous',
                    fused=rng.random() < 0.5)
    return dict(kind=kind, tokens=_log(rng, 4, 256), experts=rng.choice((8, 16, 32)), topk=rng.choice((2, 4, 8)),
                hidden=rng.choice((2048, 4096, 7168)), inter=rng.choice((1024, 2048)), layout='masked',
                fused=rng.random() < 0.5)


# ---------------------------------------------------------------- inputs

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(shape, gen):
    return torch.randn(shape, generator=gen, device=DEV, dtype=torch.float32).bfloat16()


def _scale(amax, top, pow2):
    sf = amax.float().clamp(1e-4) * (1.0 / top)
    if pow2:   # up to the next power of two
        bits = sf.view(torch.int32)
        sf = (((bits >> 23) + ((bits & 0x7FFFFF) != 0).int()).clamp(1, 254) << 23).view(torch.float32)
    return sf


def _groups(x, gran):
    """[rows, k] -> [rows, groups, gran], zeros past k."""
    rows, k = x.shape
    return torch.nn.functional.pad(x, (0, -k % gran)).view(rows, -1, gran)


def _quant_rows(x, gran=128, pow2=False):
    """e4m3 codes with one scale per row and `gran` columns."""
    g = _groups(x, gran)
    sf = _scale(g.abs().amax(2), 448.0, pow2)
    q = (g * (1.0 / sf)[:, :, None]).to(torch.float8_e4m3fn).view(torch.uint8)
    return q.view(x.shape[0], -1)[:, :x.shape[1]].contiguous().view(torch.float8_e4m3fn), sf


def _quant_blocks(x):
    """e4m3 codes with one scale per 128 x 128 block."""
    n, k = x.shape
    p = torch.nn.functional.pad(x, (0, -k % 128, 0, -n % 128))
    b = p.view(p.shape[0] // 128, 128, -1, 128)
    sf = _scale(b.abs().amax(dim=(1, 3)), 448.0, False)
    q = (b * (1.0 / sf)[:, None, :, None]).to(torch.float8_e4m3fn).view(torch.uint8)
    return q.view(p.shape)[:n, :k].contiguous().view(torch.float8_e4m3fn), sf


def _quant_fp4(x):
    """Packed e2m1 codes (element 2i in the low nibble) with one power-of-two scale
    per row and 32 columns, round to nearest even."""
    g = _groups(x, 32)
    sf = _scale(g.abs().amax(2), 6.0, True)
    v = g * (1.0 / sf)[:, :, None]
    a = v.abs()
    code = torch.zeros_like(a, dtype=torch.uint8)
    for low, tie_up in ((0.25, False), (0.75, True), (1.25, False), (1.75, True), (2.5, False), (3.5, True), (5.0, False)):
        code += (a >= low) if tie_up else (a > low)
    code = (code | ((v < 0) & (code != 0)).to(torch.uint8) << 3).view(x.shape[0], -1)
    return (code[:, 0::2] | code[:, 1::2] << 4).view(torch.int8), sf


def _blocks(groups, n, k, gen):
    """Quantized weights of `groups` experts."""
    q = torch.empty((groups, n, k), dtype=torch.float8_e4m3fn, device=DEV)
    sf = torch.empty((groups, -(-n // 128), -(-k // 128)), device=DEV)
    for g in range(groups):
        q[g], sf[g] = _quant_blocks(_randn((n, k), gen))
    return q, sf


def _segments(case, seed):
    """Rows of each expert (a multinomial over uneven shares) and each row's expert,
    -1 where a segment is filled up to 128 rows and up to the buffer's capacity."""
    gen = torch.Generator().manual_seed(int(seed))
    share = -torch.log(torch.rand(case['groups'], generator=gen).clamp_min(1e-6))
    pick = torch.multinomial(share, case['tokens'], replacement=True, generator=gen)
    counts = torch.bincount(pick, minlength=case['groups']).tolist()
    index = [torch.full((-(-c // 128) * 128,), -1, dtype=torch.int32) for c in counts]
    for e, c in enumerate(counts):
        index[e][:c] = e
    used = sum(len(v) for v in index)
    capacity = -(-(case['tokens'] + 127 * case['groups']) // 128) * 128
    return counts, torch.cat(index + [torch.full((capacity - used,), -1, dtype=torch.int32)])


def _masked_rows(case, seed):
    """masked_m of each expert: rows x U(0.75, 1.25), at least 1."""
    gen = torch.Generator().manual_seed(int(seed))
    f = 0.75 + 0.5 * torch.rand(case['groups'], generator=gen)
    return [max(1, min(case['max_m'], int(case['rows'] * v))) for v in f.tolist()]


def _group_ks(case, seed):
    """K of each group: mean_k x U(0.7, 1.3) in blocks of 128."""
    if case['groups'] == 0:
        return [case['mean_k']]
    gen = torch.Generator().manual_seed(int(seed))
    f = 0.7 + 0.6 * torch.rand(case['groups'], generator=gen)
    return [-(-int(case['mean_k'] * v) // 128) * 128 for v in f.tolist()]


def _routing(case, gen):
    """Top-k experts of each token and their weights."""
    score = torch.rand((case['tokens'], case['experts']), generator=gen, device=DEV)
    w, idx = score.topk(min(case['topk'], case['experts']), dim=1)
    return idx, (w / w.sum(1, keepdim=True)).contiguous()


def _inputs(case, seed):
    """The case's operands, made from the seed alone: plain tensors, scales as quantized."""
    gen, kind = _gen(seed), case['kind']
    if kind == 'dense':
        return dict(a=_quant_rows(_randn((case['m'], case['k']), gen)), b=_quant_blocks(_randn((case['n'], case['k']), gen)))
    if kind == 'wgrad':
        ks = _group_ks(case, seed)
        a = [_quant_rows(_randn((case['m'], k), gen)) for k in ks]
        b = [_quant_rows(_randn((case['n'], k), gen)) for k in ks]
        c = torch.randn((len(ks), case['m'], case['n']), generator=gen, device=DEV) * 32
        return dict(ks=ks, a=a, b=b, c=c)
    if kind == 'contiguous':
        counts, index = _segments(case, seed)
        x = _randn((len(index), case['k']), gen)
        x[index.to(DEV) < 0] = 0
        return dict(a=_quant_rows(x), b=_blocks(case['groups'], case['n'], case['k'], gen), index=index.to(DEV))
    if kind == 'masked':
        rows = _masked_rows(case, seed)
        q, sf = _quant_rows(_randn((case['groups'] * case['max_m'], case['k']), gen))
        shape = (case['groups'], case['max_m'], -1)
        return dict(a=(q.view(shape), sf.view(shape)), b=_blocks(case['groups'], case['n'], case['k'], gen), rows=rows)
    if kind == 'fp4':
        return dict(a=_quant_rows(_randn((case['m'], case['k']), gen), pow2=True), b=_quant_fp4(_randn((case['n'], case['k']), gen)))
    if kind == 'fp4_masked':
        rows = _masked_rows(case, seed)
        q, sf = _quant_rows(_randn((case['groups'] * case['max_m'], case['k']), gen), pow2=True)
        shape = (case['groups'], case['max_m'], -1)
        b = [_quant_fp4(_randn((case['n'], case['k']), gen)) for _ in range(case['groups'])]
        return dict(a=(q.view(shape), sf.view(shape)), b=tuple(torch.stack(t) for t in zip(*b)), rows=rows)
    if kind == 'cast':
        return dict(x=_randn((case['m'], case['k']), gen))
    idx, w = _routing(case, gen)
    return dict(x=_randn((case['tokens'], case['hidden']), gen), idx=idx, w=w,
                l1=_blocks(case['experts'], 2 * case['inter'], case['hidden'], gen),
                l2=_blocks(case['experts'], case['hidden'], case['inter'], gen))


def _major(a, case):
    """The activation scales as the caller holds them: K-major, or MN-major."""
    return (a[0], deep_gemm.get_mn_major_tma_aligned_tensor(a[1])) if case['sfa'] == 'mn' else a


def _packed(a):
    return a[0], deep_gemm.get_mn_major_tma_aligned_packed_ue8m0_tensor(a[1])


def prepare(case, seed):
    kind, s = case['kind'], _inputs(case, seed)
    s['case'] = case
    if kind == 'dense':
        s['a'] = _major(s['a'], case)
        s['d'] = torch.empty((case['m'], case['n']), dtype=torch.bfloat16, device=DEV)
    elif kind == 'wgrad':
        if case['groups'] == 0:
            s['a'], s['b'], s['d'] = s['a'][0], s['b'][0], s['c'][0]
        else:
            s['a'], s['b'] = ((torch.cat([q.view(torch.uint8).view(-1) for q, _ in p]).view(torch.float8_e4m3fn),
                               torch.cat([sf for _, sf in p], dim=1)) for p in (s['a'], s['b']))
            s['d'], s['layout'] = s['c'], torch.tensor(s['ks'], dtype=torch.int32, device=DEV)
        del s['c']
    elif kind == 'contiguous':
        s['a'] = _major(s['a'], case)
        s['d'] = torch.zeros((len(s['index']), case['n']), dtype=torch.bfloat16, device=DEV)
    elif kind in ('masked', 'fp4_masked'):
        s['a'] = _major(s['a'], case) if kind == 'masked' else _packed(s['a'])
        s['b'] = s['b'] if kind == 'masked' else _packed(s['b'])
        s['masked_m'] = torch.tensor(s['rows'], dtype=torch.int32, device=DEV)
        s['d'] = torch.zeros((case['groups'], case['max_m'], case['n']), dtype=torch.bfloat16, device=DEV)
    elif kind == 'fp4':
        s['a'], s['b'] = _packed(s['a']), _packed(s['b'])
        s['d'] = torch.empty((case['m'], case['n']), dtype=torch.bfloat16, device=DEV)
    elif kind == 'layer' and case['fused']:
        s['l1'] = deep_gemm.transform_l1_weights_for_swiglu(s['l1'])
    return s


# ---------------------------------------------------------------- one pass

def _layer(s, case):
    inter, hidden = case['inter'], case['hidden']
    x = deep_gemm.per_token_cast_to_fp8(s['x'], use_ue8m0=False)
    masked = case['layout'] == 'masked'
    rows = case['tokens'] if masked else None
    expected = -(-case['tokens'] * s['idx'].shape[1] // case['experts'])
    a, sf, layout, pos, w = deep_gemm.moe_dispatch(x, s['idx'], case['experts'], case['layout'], max_m=rows,
                                                   topk_weights=s['w'])
    lead = a.shape[:-1]
    if case['fused']:
        h = (torch.empty(lead + (inter,), dtype=torch.float8_e4m3fn, device=DEV),
             torch.empty(lead + (inter // 128,), device=DEV))
        if masked:
            deep_gemm.m_grouped_fp8_gemm_nt_masked_swiglu((a, sf), s['l1'], h, layout, expected, row_weights=w)
        else:
            deep_gemm.m_grouped_fp8_gemm_nt_contiguous_swiglu((a, sf), s['l1'], h, layout, row_weights=w)
    else:
        g = torch.empty(lead + (2 * inter,), dtype=torch.bfloat16, device=DEV)
        if masked:
            deep_gemm.m_grouped_fp8_gemm_nt_masked((a, sf), s['l1'], g, layout, expected)
            h = deep_gemm.moe_swiglu_apply_weight_to_fp8(g.view(-1, 2 * inter), w.view(-1))
            h = h[0].view(lead + (inter,)), h[1].view(lead + (inter // 128,))
        else:
            deep_gemm.m_grouped_fp8_gemm_nt_contiguous((a, sf), s['l1'], g, layout)
            h = deep_gemm.moe_swiglu_apply_weight_to_fp8(g, w, layout)
    y = torch.empty(lead + (hidden,), dtype=torch.bfloat16, device=DEV)
    if masked:
        deep_gemm.m_grouped_fp8_gemm_nt_masked(h, s['l2'], y, layout, expected)
    else:
        deep_gemm.m_grouped_fp8_gemm_nt_contiguous(h, s['l2'], y, layout)
    return deep_gemm.moe_combine(y, pos)


def run(s):
    case = s['case']
    kind = case['kind']
    if kind == 'dense':
        deep_gemm.fp8_gemm_nt(s['a'], s['b'], s['d'])
    elif kind == 'wgrad':
        if case['groups'] == 0:
            deep_gemm.fp8_gemm_nt(s['a'], s['b'], s['d'], c=s['d'], recipe=(1, 1, 128))
        else:
            deep_gemm.k_grouped_fp8_gemm_nt_contiguous(s['a'], s['b'], s['d'], s['ks'], s['layout'], s['d'])
    elif kind == 'contiguous':
        deep_gemm.m_grouped_fp8_gemm_nt_contiguous(s['a'], s['b'], s['d'], s['index'])
    elif kind == 'masked':
        deep_gemm.m_grouped_fp8_gemm_nt_masked(s['a'], s['b'], s['d'], s['masked_m'], case['rows'])
    elif kind == 'fp4':
        deep_gemm.fp8_fp4_gemm_nt(s['a'], s['b'], s['d'], recipe_a=(1, 128), recipe_b=(1, 32))
    elif kind == 'fp4_masked':
        deep_gemm.m_grouped_fp8_fp4_gemm_nt_masked(s['a'], s['b'], s['d'], s['masked_m'], case['rows'],
                                                   recipe_a=(1, 128), recipe_b=(1, 32))
    elif kind == 'cast':
        if case['sfa'] == 'mn':
            q, sf = deep_gemm.per_token_cast_to_fp8_mn_major(s['x'], use_ue8m0=False)
        else:
            q, sf = deep_gemm.per_token_cast_to_fp8(s['x'], use_ue8m0=False)
        return q.view(torch.uint8), sf
    else:
        return _layer(s, case)
    return s['d']


def work(case):
    kind = case['kind']
    if kind == 'cast':
        m, k = case['m'], case['k']
        return dict(bytes=3 * m * k + 4 * m * -(-k // 128), flops=0)
    if kind == 'layer':
        t, h, i, e = case['tokens'], case['hidden'], case['inter'], case['experts']
        k = min(case['topk'], e)
        return dict(bytes=4 * t * h + 12 * t * k + min(e, t * k) * 3 * i * h, flops=2 * t * k * 3 * i * h)
    n, k = case['n'], case.get('k', case.get('mean_k'))
    if kind == 'wgrad':
        g, m = max(1, case['groups']), case['m']
        return dict(bytes=g * (k * (m + n) + (m + n) * k // 32 + 8 * m * n), flops=2 * g * m * n * k)
    groups = case.get('groups', 1)
    rows = case['m'] if kind in ('dense', 'fp4') else case['tokens'] if kind == 'contiguous' else \
        groups * min(case['rows'], case['max_m'])
    if kind in ('fp4', 'fp4_masked'):
        weights = groups * (n * k // 2 + n * k // 32)
        acts = rows * k + rows * k // 128
    else:
        weights = groups * (n * k + 4 * -(-n // 128) * -(-k // 128))
        acts = rows * k + 4 * rows * -(-k // 128)
    return dict(bytes=weights + acts + 2 * rows * n, flops=2 * rows * n * k)


def tolerance(case):
    kind = case['kind']
    if kind == 'cast':
        return 'exact'
    if kind == 'wgrad':   # four times what FP32 sums of the matrix cores' FP8 products are off
        return dict(rel=5e-5, max=2e-3)
    if kind == 'layer':   # sums in another order move BF16 and e4m3 roundings of the layer's middle
        return dict(rel=1e-2, max=0.2)
    return dict(rel=6.6e-3, max=2e-2)   # four times one BF16 rounding


# ---------------------------------------------------------------- 64 bits

_E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)


def _rows64(q, sf):
    """Codes times the scale of their row and column group, in 64 bits."""
    k = q.shape[1] * (2 if q.dtype == torch.int8 else 1)
    if q.dtype == torch.int8:
        u = q.view(torch.uint8)
        code = torch.stack((u & 15, u >> 4), dim=2).view(q.shape[0], k).long()
        v = torch.tensor(_E2M1, dtype=torch.float64, device=q.device)[code & 7]
        v = torch.where(code >= 8, -v, v)
    else:
        v = q.double()
    gran = 32 if q.dtype == torch.int8 else 128
    return v * sf.double().repeat_interleave(gran, 1)[:, :k]


def _blocks64(q, sf):
    n, k = q.shape
    return q.double() * sf.double().repeat_interleave(128, 0)[:n].repeat_interleave(128, 1)[:, :k]


def _layer64(s, case):
    """The layer's defined roundings (both casts to e4m3, BF16 between the steps) with every sum in 64 bits."""
    xq = _quant_rows(s['x'])
    x, out = _rows64(*xq), torch.zeros(s['x'].shape, dtype=torch.float64, device=DEV)
    i = case['inter']
    for e in range(case['experts']):
        t, slot = (s['idx'] == e).nonzero(as_tuple=True)
        if len(t) == 0:
            continue
        h = (x[t] @ _blocks64(s['l1'][0][e], s['l1'][1][e]).t()).bfloat16().double()
        gate, up = h[:, :i], h[:, i:]
        y = gate / (1 + torch.exp(-gate)) * up * s['w'][t, slot].double()[:, None]
        y = _rows64(*_quant_rows(y.float()))
        out.index_add_(0, t, (y @ _blocks64(s['l2'][0][e], s['l2'][1][e]).t()).bfloat16().double())
    return out


def exact(case, seed):
    s, kind = _inputs(case, seed), case['kind']
    if kind == 'dense':
        return _rows64(*s['a']) @ _blocks64(*s['b']).t()
    if kind == 'fp4':
        return _rows64(*s['a']) @ _rows64(*s['b']).t()
    if kind == 'wgrad':
        out = torch.stack([c.double() + _rows64(*a) @ _rows64(*b).t() for a, b, c in zip(s['a'], s['b'], s['c'])])
        return out[0] if case['groups'] == 0 else out
    if kind == 'contiguous':
        out = torch.zeros((len(s['index']), case['n']), dtype=torch.float64, device=DEV)
        for e in range(case['groups']):
            at = (s['index'] == e).nonzero()[:, 0]
            out[at] = _rows64(s['a'][0].view(torch.uint8)[at].view(torch.float8_e4m3fn), s['a'][1][at]) @ \
                _blocks64(s['b'][0][e], s['b'][1][e]).t()
        return out
    if kind in ('masked', 'fp4_masked'):
        deq = _blocks64 if kind == 'masked' else _rows64
        out = torch.zeros((case['groups'], case['max_m'], case['n']), dtype=torch.float64, device=DEV)
        for g, r in enumerate(s['rows']):
            out[g, :r] = _rows64(s['a'][0][g, :r], s['a'][1][g, :r]) @ deq(s['b'][0][g], s['b'][1][g]).t()
        return out
    if kind == 'cast':
        return None, _scale64(s['x'])
    return _layer64(s, case)


def _scale64(x):
    return _groups(x, 128).abs().double().amax(2).clamp(1e-4) / 448.0
