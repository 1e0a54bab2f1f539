"""GPU parity of the HIP kernels against the CPU oracle (run on an MI355X).

Bars (tolerances are the reference's, tests/generators.py:69-74):
  * calc_diff(D, oracle) < 1e-3 for FP8 x FP8 (measured ~1e-6: BF16 output rounding
    only), and the max relative error is printed; FP8 x FP4 < 1e-2.
  * 20 reruns bitwise identical (reference tests/test_fp8_fp4.py:72-82).
  * rows that must not be written (padding rows, rows >= masked_m, past M/N)
    keep a sentinel byte pattern bit-exactly.
  * a grouped call's segment equals the dense call on that segment bitwise.
"""
import numpy as np
import pytest
import torch

import deep_gemm
from oracle import gemm as ogemm
from oracle import quant as oquant
import generators as gen

pytestmark = pytest.mark.gpu

DEV = 'cuda'
SENTINEL = 0x7F7B   # bf16 bit pattern written before each call (a large finite value)


def e4m3(x):
    return gen.to_dev(x, torch.float8_e4m3fn)


def f32(x):
    return gen.to_dev(np.asarray(x, dtype=np.float32))


def sentinel_bf16(shape):
    return torch.full(shape, SENTINEL, dtype=torch.int16, device=DEV).view(torch.bfloat16)


def report(name, d, ref):
    diff = ogemm.calc_diff(d, ref)
    rel = ogemm.max_rel_err(d, ref)
    print(f'[{name}] calc_diff={diff:.3e} max_rel_err={rel:.3e}', flush=True)
    return diff, rel


# ----------------------------------------------------------------- dense

DENSE_CASES = [
    (64, 2112, 7168),    # config 1 shape
    (1, 256, 128),
    (128, 576, 7168),
    (129, 200, 384),     # ragged M and N, N not a multiple of 64
    (300, 4096, 512),
    (7, 16, 16),         # K shorter than one block
    (256, 512, 1040),    # K tail (K % 128 == 16)
    (512, 768, 36864),   # more K blocks than the 4-block SFA scale groups hold: per-stage SFA loads
]


@pytest.mark.parametrize('m,n,k', DENSE_CASES)
def test_dense_bf16_vs_oracle(m, n, k):
    print(f'dense m={m} n={n} k={k}', flush=True)
    x = gen.dense_inputs(m, n, k, seed=m + n + k)
    ref = ogemm.gemm_nt(oquant.dequant_per_token(x['qa'], x['sfa']), oquant.dequant_per_block(x['qb'], x['sfb']))
    d = torch.empty((m, n), dtype=torch.bfloat16, device=DEV)
    deep_gemm.fp8_gemm_nt((e4m3(x['qa']), f32(x['sfa'])), (e4m3(x['qb']), f32(x['sfb'])), d)
    torch.cuda.synchronize()
    out = d.float().cpu().numpy()
    diff, rel = report(f'dense {m}x{n}x{k}', out, ref)
    assert diff < 1e-3
    # Stronger than the reference bar: within one BF16 ulp of the FP64 oracle, plus an
    # accumulation term that dominates near zero (the MFMA's own summation error; the
    # bound stated against sum |a b| is in test_random_sweep_gpu.py).
    tol = np.abs(ref) * 2.0 ** -8 + 2.0 ** -20 * np.sqrt(k) * np.abs(ref).max()
    assert np.all(np.abs(out - ref) <= tol), 'further than one BF16 ulp from the FP64 oracle'
    # Against the unquantized product, the reference tests' own oracle (tests/generators.py:363)
    raw = x['a'].astype(np.float64) @ x['b'].astype(np.float64).T
    print(f'  calc_diff vs unquantized = {ogemm.calc_diff(out, raw):.3e}', flush=True)
    if k >= 128:
        assert ogemm.calc_diff(out, raw) < 1e-3


@pytest.mark.parametrize('m,n,k', [(200, 320, 1024), (512, 768, 2048), (300, 520, 1040)])
def test_all_tiles_bitwise_equal(m, n, k):
    """Every compiled tile shape gives the same bits (each output's K order is fixed).
    (512, 768, 2048) has interior tiles for every shape; the others are ragged."""
    x = gen.dense_inputs(m, n, k, seed=5)
    a, b = (e4m3(x['qa']), f32(x['sfa'])), (e4m3(x['qb']), f32(x['sfb']))
    outs = []
    try:
        for v, bm, bn in ((1, 64, 64), (1, 64, 128), (1, 128, 64), (1, 128, 128),
                          (2, 128, 128), (2, 128, 256), (2, 256, 128), (2, 256, 192), (2, 256, 256)):
            deep_gemm.set_tile_override(bm, bn, variant=v)
            d = torch.empty((m, n), dtype=torch.bfloat16, device=DEV)
            deep_gemm.fp8_gemm_nt(a, b, d)
            outs.append((v, d))
            print(deep_gemm.get_last_config(), flush=True)
    finally:
        deep_gemm.set_tile_override(0, 0)
    # both variants use the same MFMA shape and per-K-block order, so every tile
    # shape of either kernel gives the same bits
    for _, o in outs[1:]:
        assert torch.equal(o.view(torch.int16), outs[0][1].view(torch.int16))


@pytest.mark.parametrize('m,n,k,pad', [(512, 4096, 1040, 112), (300, 520, 144, 0), (257, 264, 16, 16), (200, 320, 2032, 144),
                                       (2100, 4104, 240, 16), (4000, 7176, 272, 0)])
def test_k_tail_ignores_what_follows_k(m, n, k, pad):
    """K % 128 != 0 (one to seven 16-byte chunks in the last block, with and without
    whole blocks before it): every tile, and the heuristic's own choice (the 256 x 256
    tile at the larger sizes), gives the bits of the register-staged kernel, whatever
    follows K in the rows' padding (NaN codes in A and B here)."""
    x = gen.dense_inputs(m, n, k, seed=m + k)
    a_buf = torch.full((m, k + pad), 0x7F, dtype=torch.uint8, device=DEV)
    b_buf = torch.full((n, k + pad), 0xFF, dtype=torch.uint8, device=DEV)
    a_buf[:, :k] = gen.to_dev(x['qa'])
    b_buf[:, :k] = gen.to_dev(x['qb'])
    a = (a_buf[:, :k].view(torch.float8_e4m3fn), f32(x['sfa']))
    b = (b_buf[:, :k].view(torch.float8_e4m3fn), f32(x['sfb']))
    outs, cfgs = [], []
    for v, bm, bn in ((1, 64, 64), (0, 0, 0), (2, 128, 128), (2, 128, 256), (2, 256, 128), (2, 256, 192),
                      (2, 256, 256)):
        deep_gemm.set_tile_override(bm, bn, variant=v)
        try:
            d = sentinel_bf16((m, n))
            deep_gemm.fp8_gemm_nt(a, b, d)
            cfgs.append(deep_gemm.get_last_config())
        finally:
            deep_gemm.set_tile_override(0, 0)
        outs.append(d.view(torch.int16))
    torch.cuda.synchronize()
    print(f'k-tail m={m} n={n} k={k}: {cfgs[1]}', flush=True)
    if m == 4000:
        assert 'block_m=256 block_n=256' in cfgs[1], cfgs[1]
    for o, c in zip(outs[1:], cfgs[1:]):
        assert torch.equal(o, outs[0]), c
    ref = ogemm.gemm_nt(oquant.dequant_per_token(x['qa'], x['sfa'])[:64], oquant.dequant_per_block(x['qb'], x['sfb']))
    assert ogemm.calc_diff(outs[1].view(torch.bfloat16)[:64].float().cpu().numpy(), ref) < 1e-3


@pytest.mark.parametrize('m,n,k,acc', [(4096, 7168, 4096, False), (4096, 7168, 4096, True), (8192, 7168, 4096, False),
                                        (4096, 7040, 4096, False)])   # the 256 x 192 launch ends in a 64-column tile
def test_dense_column_split_equals_one_launch(m, n, k, acc):
    """Dense calls (K >= 4096) whose 256 x 256 tiles would leave the last round part
    empty run as two launches (256 x 256 tiles over the first columns, 256 x 192 over the rest):
    bitwise the single 256 x 256 launch, BF16 out and FP32 C in place, and the
    split rows and columns hold the oracle's values."""
    print(f'dense column split m={m} n={n} k={k} acc={acc}', flush=True)
    x = gen.dense_inputs(m, n, k, seed=21)
    a, b = (e4m3(x['qa']), f32(x['sfa'])), (e4m3(x['qb']), f32(x['sfb']))
    c_np = gen.randn_bf16((m, n), 23) * 32.0 if acc else None

    def run():
        if acc:
            d = f32(c_np)
            deep_gemm.fp8_gemm_nt(a, b, d, c=d)
        else:
            d = torch.empty((m, n), dtype=torch.bfloat16, device=DEV)
            deep_gemm.fp8_gemm_nt(a, b, d)
        return d, deep_gemm.get_last_config()

    split, cfg = run()
    print(cfg, flush=True)
    assert 'split_n=' in cfg, cfg
    try:
        deep_gemm.set_tile_override(256, 256, variant=2)
        whole, cfg1 = run()
        assert 'split_n=' not in cfg1, cfg1
    finally:
        deep_gemm.set_tile_override(0, 0)
    torch.cuda.synchronize()
    assert torch.equal(split.view(torch.int32 if acc else torch.int16), whole.view(torch.int32 if acc else torch.int16))
    # rows on both sides of the split column, against the oracle
    n1 = int(cfg.split('split_n=')[1].split(':')[0])
    rows = np.array([0, 1, 255, 256, 2047, m - 1])
    cols = np.r_[0:8, n1 - 8:n1 + 8, n - 8:n]
    ref = ogemm.gemm_nt(oquant.dequant_per_token(x['qa'][rows], x['sfa'][rows]),
                        oquant.dequant_per_block(x['qb'], x['sfb']), None if c_np is None else c_np[rows])
    out = split.float().cpu().numpy()[rows]
    diff, _ = report('column split', out[:, cols], ref[:, cols])
    assert diff < 1e-5


@pytest.mark.parametrize('inplace', [True, False])
def test_dense_c_accumulate_f32(inplace):
    m, n, k = 256, 384, 896
    print(f'dense f32 C accumulate inplace={inplace}', flush=True)
    x = gen.dense_inputs(m, n, k, seed=11)
    c_np = gen.randn_bf16((m, n), 99) * 32.0
    ref = ogemm.gemm_nt(oquant.dequant_per_token(x['qa'], x['sfa']), oquant.dequant_per_block(x['qb'], x['sfb']),
                        c_np)
    c = f32(c_np)
    d = c if inplace else torch.empty((m, n), dtype=torch.float32, device=DEV)
    deep_gemm.fp8_gemm_nt((e4m3(x['qa']), f32(x['sfa'])), (e4m3(x['qb']), f32(x['sfb'])), d, c=c)
    torch.cuda.synchronize()
    out = d.cpu().numpy()
    diff, rel = report('c-accumulate', out, ref)
    assert diff < 1e-6
    # D = C + (A.B^T) with one FP32 add: matches C + FP32(acc) up to the accumulation error.
    assert np.max(np.abs(out - ref)) < 1e-3 * np.max(np.abs(ref))


def test_dense_bf16_c_accumulate():
    m, n, k = 128, 256, 512
    x = gen.dense_inputs(m, n, k, seed=12)
    c_np = oquant.bf16_round(gen.randn_bf16((m, n), 98))
    ref = ogemm.gemm_nt(oquant.dequant_per_token(x['qa'], x['sfa']), oquant.dequant_per_block(x['qb'], x['sfb']),
                        c_np)
    d = gen.to_dev(c_np).bfloat16()
    deep_gemm.fp8_gemm_nt((e4m3(x['qa']), f32(x['sfa'])), (e4m3(x['qb']), f32(x['sfb'])), d, c=d)
    diff, _ = report('bf16 c-accumulate', d.float().cpu().numpy(), ref)
    assert diff < 1e-3


def test_dense_determinism_and_bounds():
    """20 reruns are bitwise equal; a view into a sentinel-filled buffer is written only inside the view."""
    m, n, k = 200, 264, 2048
    x = gen.dense_inputs(m, n, k, seed=3)
    a, b = (e4m3(x['qa']), f32(x['sfa'])), (e4m3(x['qb']), f32(x['sfb']))
    big = sentinel_bf16((m + 8, n + 64))
    d = big[4:4 + m, 8:8 + n]
    deep_gemm.fp8_gemm_nt(a, b, d)
    first = d.clone()
    for _ in range(20):
        d.fill_(0)
        deep_gemm.fp8_gemm_nt(a, b, d)
        assert torch.equal(d.view(torch.int16), first.view(torch.int16))
    mask = torch.ones_like(big, dtype=torch.bool)
    mask[4:4 + m, 8:8 + n] = False
    assert bool((big.view(torch.int16)[mask] == SENTINEL).all())


@pytest.mark.parametrize('tile', [None, (2, 256, 256), (2, 256, 192), (2, 128, 256)])
@pytest.mark.parametrize('m,n,k', [(130, 256, 1024), (300, 520, 2048), (257, 384, 1408), (64, 256, 512),
                                   (200, 256, 1536), (260, 256, 7168), (200, 384, 4608)])
def test_mn_major_sfa_equals_k_major(tile, m, n, k):
    """SFA in the reference's MN-major TMA-aligned layout gives the same bits as K-major SFA.
    With two-stage tiles, K-major SFA is read through the kernel's scale groups of
    4 K blocks (K % 512 == 0; K = 1408 keeps the per-stage loads), and each case
    is checked against the oracle as well."""
    x = gen.dense_inputs(m, n, k, seed=4)
    a_t, b = e4m3(x['qa']), (e4m3(x['qb']), f32(x['sfb']))
    sfa = f32(x['sfa'])
    sfa_mn = deep_gemm.get_mn_major_tma_aligned_tensor(sfa)
    assert sfa_mn.stride() == (1, deep_gemm.get_tma_aligned_size(m, 4))
    d1 = torch.empty((m, n), dtype=torch.bfloat16, device=DEV)
    d2 = torch.empty_like(d1)
    if tile is not None:
        deep_gemm.set_tile_override(tile[1], tile[2], variant=tile[0])
    try:
        deep_gemm.fp8_gemm_nt((a_t, sfa), b, d1)
        print(deep_gemm.get_last_config(), flush=True)
        deep_gemm.fp8_gemm_nt((a_t, sfa_mn), b, d2)
    finally:
        deep_gemm.set_tile_override(0, 0)
    assert torch.equal(d1.view(torch.int16), d2.view(torch.int16))
    ref = ogemm.gemm_nt(oquant.dequant_per_token(x['qa'], x['sfa']), oquant.dequant_per_block(x['qb'], x['sfb']))
    diff, _ = report(f'sfa layouts {m}x{n}x{k} {tile}', d1.float().cpu().numpy(), ref)
    assert diff < 1e-3


@pytest.mark.parametrize('tile', [None, (2, 256, 256), (2, 256, 192)])
@pytest.mark.parametrize('k', [1024, 1408, 2048])
def test_contiguous_mn_major_sfa_equals_k_major(tile, k):
    """m-grouped contiguous with MN-major SFA (per-stage scale loads and the split
    stage hand-off) gives the bits of K-major SFA (4-block scale groups when
    K % 512 == 0), with an empty expert and 256-row tiles that straddle two
    experts (two passes), padding rows untouched."""
    ms, n = [300, 0, 150, 420], 512
    aligned = [(x + 127) // 128 * 128 for x in ms]
    m_pad = sum(aligned)
    layout_np = np.full(m_pad, -1, dtype=np.int32)
    start = 0
    for e, (mi, ai) in enumerate(zip(ms, aligned)):
        layout_np[start:start + mi] = e
        start += ai
    dg = torch.Generator(device=DEV).manual_seed(43 + k)
    a_bf = torch.randn((m_pad, k), generator=dg, device=DEV).bfloat16()
    a_bf[torch.from_numpy(layout_np < 0).to(DEV)] = 0
    aq, asf = deep_gemm.per_token_cast_to_fp8(a_bf, use_ue8m0=False)
    asf_mn = deep_gemm.get_mn_major_tma_aligned_tensor(asf)
    bq = torch.empty((len(ms), n, k), dtype=torch.float8_e4m3fn, device=DEV)
    bs = torch.empty((len(ms), n // 128, (k + 127) // 128), device=DEV)
    for e in range(len(ms)):
        bq[e], bs[e] = deep_gemm.per_block_cast_to_fp8(torch.randn((n, k), generator=dg, device=DEV).bfloat16(),
                                                       use_ue8m0=False)
    layout = gen.to_dev(layout_np)
    outs = []
    if tile is not None:
        deep_gemm.set_tile_override(tile[1], tile[2], variant=tile[0])
    try:
        for sf in (asf, asf_mn):
            d = sentinel_bf16((m_pad, n))
            deep_gemm.m_grouped_fp8_gemm_nt_contiguous((aq, sf), (bq, bs), d, layout)
            print(f'contiguous sfa layouts k={k} tile={tile}: {deep_gemm.get_last_config()}', flush=True)
            outs.append(d)
    finally:
        deep_gemm.set_tile_override(0, 0)
    torch.cuda.synchronize()
    assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))
    pad = torch.from_numpy(layout_np < 0).to(DEV)
    assert bool((outs[1].view(torch.int16)[pad] == SENTINEL).all())


def test_k_zero_and_empty():
    m, n = 64, 128
    a = torch.empty((m, 0), dtype=torch.float8_e4m3fn, device=DEV)
    b = torch.empty((n, 0), dtype=torch.float8_e4m3fn, device=DEV)
    sfa = torch.empty((m, 0), dtype=torch.float32, device=DEV)
    sfb = torch.empty((1, 0), dtype=torch.float32, device=DEV)
    d = torch.full((m, n), 3.0, dtype=torch.float32, device=DEV)
    deep_gemm.fp8_gemm_nt((a, sfa), (b, sfb), d)          # K == 0, no C -> zeros
    assert bool((d == 0).all())
    c = torch.randn((m, n), device=DEV)
    deep_gemm.fp8_gemm_nt((a, sfa), (b, sfb), d, c=c)     # K == 0 with C -> D = C
    assert torch.equal(d, c)
    a0 = torch.empty((0, 256), dtype=torch.float8_e4m3fn, device=DEV)
    deep_gemm.fp8_gemm_nt((a0, torch.empty((0, 2), device=DEV)),
                          (torch.empty((n, 256), dtype=torch.float8_e4m3fn, device=DEV),
                           torch.ones((1, 2), device=DEV)), torch.empty((0, n), dtype=torch.bfloat16, device=DEV))


# ----------------------------------------------------------------- grouped

CONTIG_TILES = [None, (2, 256, 256), (2, 256, 192), (2, 128, 256), (1, 128, 128)]


@pytest.mark.parametrize('tile', CONTIG_TILES)
@pytest.mark.parametrize('ms', [None, [130, 100, 300, 0, 250, 1]])
def test_contiguous_vs_oracle_and_dense(tile, ms):
    """Random segments, and segments whose 128-aligned boundaries fall inside
    256-row tiles (a tile then holds two experts)."""
    if ms is None:
        ms, aligned = gen.contiguous_sizes(4, 900, seed=7)
    else:
        aligned = [(mi + 127) // 128 * 128 for mi in ms]
    n, k = 384, 1024
    print(f'contiguous ms={ms} aligned={aligned} tile={tile}', flush=True)
    if tile is not None:
        deep_gemm.set_tile_override(tile[1], tile[2], variant=tile[0])
    try:
        _contiguous_case(ms, aligned, n, k)
    finally:
        deep_gemm.set_tile_override(0, 0)


def _contiguous_case(ms, aligned, n, k):
    x = gen.contiguous_inputs(ms, aligned, n, k, seed=7)
    a_deq = oquant.dequant_per_token(x['qa'], x['sfa'])
    b_deq = np.stack([oquant.dequant_per_block(x['qb'][i], x['sfb'][i]) for i in range(len(ms))])
    ref, valid = ogemm.gemm_contiguous(a_deq, b_deq, x['m_indices'])
    m_pad = sum(aligned)
    a, b = (e4m3(x['qa']), f32(x['sfa'])), (e4m3(x['qb']), f32(x['sfb']))
    mi = gen.to_dev(x['m_indices'])
    d = sentinel_bf16((m_pad, n))
    deep_gemm.m_grouped_fp8_gemm_nt_contiguous(a, b, d, mi)
    torch.cuda.synchronize()
    out = d.float().cpu().numpy()
    report('contiguous', out[valid], ref[valid])
    assert ogemm.calc_diff(out[valid], ref[valid]) < 1e-3
    # padding rows untouched, bit-exact
    assert bool((d.view(torch.int16)[torch.from_numpy(~valid).to(DEV)] == SENTINEL).all())
    # each segment equals the dense call on that segment's rows (same tile shape)
    start = 0
    for i, (mi_, ai) in enumerate(zip(ms, aligned)):
        if mi_ > 0:
            dd = torch.empty((mi_, n), dtype=torch.bfloat16, device=DEV)
            gen.dense_call_same_order(deep_gemm, (a[0][start:start + mi_], a[1][start:start + mi_]), (b[0][i], b[1][i]), dd)
            assert torch.equal(dd.view(torch.int16), d[start:start + mi_].view(torch.int16)), f'segment {i}'
        start += ai
    # determinism
    first = d.clone()
    for _ in range(20):
        deep_gemm.m_grouped_fp8_gemm_nt_contiguous(a, b, d, mi)
    assert torch.equal(d.view(torch.int16), first.view(torch.int16))


@pytest.mark.parametrize('ms,mn_major,two_launches', [(None, False, False), ([2000, 0, 4500, 2200], True, False),
                                                      ([9000], True, True), ([9000], False, True)])
def test_contiguous_row_split_equals_one_launch(ms, mn_major, two_launches):
    """m-grouped contiguous calls (K >= 4096) whose 256 x 256 tiles would leave the last
    round mostly empty: one group runs as two launches (the first rows on 256 x 256
    tiles, the last M blocks on smaller ones), several groups as one. Bitwise the
    single per-tile 256 x 256 launch, padding rows untouched, and rows around where
    one group is split against the oracle. Cases: 8 experts with Dirichlet sizes over
    8192 tokens (35 M blocks, 2.2 rounds), an empty expert and long segments, and one
    expert of 9000 rows, with K- and MN-major SFA."""
    n, k = 4096, 4096
    if ms is None:
        ms, aligned = gen.contiguous_sizes(8, 8192, seed=7)
    else:
        aligned = [(x + 127) // 128 * 128 for x in ms]
    g, m_pad = len(ms), sum(aligned)
    print(f'contiguous row split ms={ms} m_pad={m_pad} mn_major={mn_major}', flush=True)
    dg = torch.Generator(device=DEV).manual_seed(41)
    a_bf = torch.randn((m_pad, k), generator=dg, device=DEV).bfloat16()
    layout_np = np.full(m_pad, -1, dtype=np.int32)
    start = 0
    for e, (mi, ai) in enumerate(zip(ms, aligned)):
        layout_np[start:start + mi] = e
        a_bf[start + mi:start + ai] = 0   # padding rows of A are zero, as the reference's generator writes them
        start += ai
    layout = gen.to_dev(layout_np)
    aq, asf = deep_gemm.per_token_cast_to_fp8(a_bf, use_ue8m0=False)
    if mn_major:
        asf = deep_gemm.get_mn_major_tma_aligned_tensor(asf)
    bq = torch.empty((g, n, k), dtype=torch.float8_e4m3fn, device=DEV)
    bs = torch.empty((g, n // 128, k // 128), device=DEV)
    for e in range(g):
        bq[e], bs[e] = deep_gemm.per_block_cast_to_fp8(torch.randn((n, k), generator=dg, device=DEV).bfloat16(),
                                                       use_ue8m0=False)

    def run():
        d = sentinel_bf16((m_pad, n))
        deep_gemm.m_grouped_fp8_gemm_nt_contiguous((aq, asf), (bq, bs), d, layout)
        return d, deep_gemm.get_last_config()

    split, cfg = run()
    print(cfg, flush=True)
    if deep_gemm.get_num_sms() >= 256:
        assert ('split_m=' in cfg) == two_launches and ' v4 ' in cfg, cfg
    try:
        deep_gemm.set_tile_override(256, 256, variant=2)
        whole, cfg1 = run()
        assert 'split_m=' not in cfg1, cfg1
    finally:
        deep_gemm.set_tile_override(0, 0)
    torch.cuda.synchronize()
    assert torch.equal(split.view(torch.int16), whole.view(torch.int16))
    valid = torch.from_numpy(layout_np >= 0).to(DEV)
    assert bool((split.view(torch.int16)[~valid] == SENTINEL).all()), 'padding rows touched'
    # rows on both sides of the split row, and the first and last valid rows, against the oracle
    r1 = int(cfg.split('split_m=')[1].split(':')[0]) if 'split_m=' in cfg else 8192
    cand = [0, r1 - 2, r1 - 1, r1, r1 + 1, int(np.nonzero(layout_np >= 0)[0][-1])]
    rows = np.array(sorted({r for r in cand if 0 <= r < m_pad and layout_np[r] >= 0}))
    a_deq = oquant.dequant_per_token(aq[rows].view(torch.uint8).cpu().numpy(), asf[rows].cpu().numpy())
    out = split[torch.from_numpy(rows).to(DEV)].float().cpu().numpy()
    ref = np.empty_like(out, dtype=np.float64)
    for e in np.unique(layout_np[rows]):
        sel = layout_np[rows] == e
        b_deq = oquant.dequant_per_block(bq[e].view(torch.uint8).cpu().numpy(), bs[e].cpu().numpy())
        ref[sel] = ogemm.gemm_nt(a_deq[sel], b_deq)
    diff, _ = report('contiguous row split', out, ref)
    assert diff < 1e-5


def test_psum_layout():
    """psum layout against the oracle's restatement of the reference's psum walk
    (oracle/gemm.py psum_blocks / gemm_psum): computed rows match the FP64
    oracle, rows the call must not write keep the sentinel, the padding rows are
    zero with ensure_zero_padding (the reference's assert_psum_zero_padding,
    tests/utils.py:9-18, on both A and D), and each group equals a dense call."""
    g, n, k = 4, 256, 512
    ms = [100, 0, 257, 64]
    align = deep_gemm.get_mk_alignment_for_contiguous_layout()
    ends, starts, prev = [], [], 0
    for mi in ms:
        s = (prev + align - 1) // align * align
        starts.append(s)
        ends.append(s + mi)
        prev = s + mi
    m_pad = (ends[-1] + align - 1) // align * align
    x = gen.contiguous_inputs(ms, [((mi + align - 1) // align) * align for mi in ms], n, k, seed=21)
    # x rows are laid out with per-group aligned starts, identical to the psum starts above
    a, b = (e4m3(x['qa']), f32(x['sfa'])), (e4m3(x['qb']), f32(x['sfb']))
    a_deq = oquant.dequant_per_token(x['qa'], x['sfa'])
    b_deq = np.stack([oquant.dequant_per_block(x['qb'][i], x['sfb'][i]) for i in range(g)])
    psum = torch.tensor(ends, dtype=torch.int32, device=DEV)
    for zero_pad in (False, True):
        ref, written = ogemm.gemm_psum(a_deq, b_deq, ends, align, align, zero_pad)
        d = sentinel_bf16((m_pad, n))
        deep_gemm.m_grouped_fp8_gemm_nt_contiguous(a, b, d, psum, use_psum_layout=True,
                                                   ensure_zero_padding=zero_pad)
        torch.cuda.synchronize()
        out = d.float().cpu().numpy()
        computed = written & ~np.isnan(ref).any(axis=1) & np.any(ref != 0.0, axis=1)
        diff, _ = report(f'psum zero_pad={zero_pad}', out[computed], ref[computed])
        assert diff < 1e-3
        tol = np.abs(ref[computed]) * 2.0 ** -8 + 2.0 ** -20 * np.sqrt(k) * np.abs(ref[computed]).max()
        assert np.all(np.abs(out[computed] - ref[computed]) <= tol)
        assert np.all(out[written & ~computed] == 0.0)
        assert bool((d.view(torch.int16)[torch.from_numpy(~written).to(DEV)] == SENTINEL).all()), 'rows touched'
        for i in range(g):
            s, e = starts[i], ends[i]
            if e > s:
                dd = torch.empty((e - s, n), dtype=torch.bfloat16, device=DEV)
                gen.dense_call_same_order(deep_gemm, (a[0][s:e], a[1][s:e]), (b[0][i], b[1][i]), dd)
                assert torch.equal(dd.view(torch.int16), d[s:e].view(torch.int16)), f'group {i}'
            pe = (e + align - 1) // align * align
            if zero_pad and pe > e:
                # the reference's assert_psum_zero_padding: A and D padding rows are zero
                assert np.all(x['qa'][e:pe] == 0), f'group {i} A padding not zero'
                assert bool((d[e:pe].view(torch.int16) == 0).all()), f'group {i} padding not zeroed'


@pytest.mark.parametrize('n,k', [(512, 1024), (256, 2048)])
def test_masked_vs_oracle(n, k):
    g, max_m = 6, 256
    x = gen.masked_inputs(g, max_m, n, k, seed=n + k)
    print(f'masked masked_m={x["masked_m"].tolist()}', flush=True)
    a_deq = np.stack([oquant.dequant_per_token(x['qa'][i], x['sfa'][i]) for i in range(g)])
    b_deq = np.stack([oquant.dequant_per_block(x['qb'][i], x['sfb'][i]) for i in range(g)])
    ref, valid = ogemm.gemm_masked(a_deq, b_deq, x['masked_m'])
    a, b = (e4m3(x['qa']), f32(x['sfa'])), (e4m3(x['qb']), f32(x['sfb']))
    mm = gen.to_dev(x['masked_m'])
    d = sentinel_bf16((g, max_m, n))
    deep_gemm.m_grouped_fp8_gemm_nt_masked(a, b, d, mm, expected_m=128)
    torch.cuda.synchronize()
    out = d.float().cpu().numpy()
    report('masked', out[valid], ref[valid])
    assert ogemm.calc_diff(out[valid], ref[valid]) < 1e-3
    assert bool((d.view(torch.int16)[torch.from_numpy(~valid).to(DEV)] == SENTINEL).all())
    # each group equals a dense call on its valid rows
    for i in range(g):
        r = int(x['masked_m'][i])
        dd = torch.empty((r, n), dtype=torch.bfloat16, device=DEV)
        gen.dense_call_same_order(deep_gemm, (a[0][i, :r], a[1][i, :r]), (b[0][i], b[1][i]), dd)
        assert torch.equal(dd.view(torch.int16), d[i, :r].view(torch.int16))


def test_masked_edge_counts():
    """masked_m of 0, 1, exactly max_m and a block boundary."""
    g, max_m, n, k = 4, 256, 128, 256
    x = gen.masked_inputs(g, max_m, n, k, seed=1)
    x['masked_m'][:] = [0, 1, 256, 128]
    a, b = (e4m3(x['qa']), f32(x['sfa'])), (e4m3(x['qb']), f32(x['sfb']))
    d = sentinel_bf16((g, max_m, n))
    deep_gemm.m_grouped_fp8_gemm_nt_masked(a, b, d, gen.to_dev(x['masked_m']), expected_m=64)
    for i, r in enumerate(x['masked_m']):
        assert bool((d[i, r:].view(torch.int16) == SENTINEL).all())
        if r:
            assert not bool((d[i, :r].view(torch.int16) == SENTINEL).any())


@pytest.mark.parametrize('bn,mn_major', [(128, False), (160, True), (192, False), (224, True), (256, False),
                                         (256, True)])
def test_masked_stream_equals_pipelined(bn, mn_major):
    """The weight-streaming masked kernel (variant 5) is bitwise equal to the
    pipelined 256 x 256 kernel: masked_m of 0, 1, one pass (97, 160), two passes
    (161, 300), N not a multiple of block_n, K-major and MN-major SFA."""
    g, max_m, n, k = 6, 320, 480, 1024
    x = gen.masked_inputs(g, max_m, n, k, seed=bn + int(mn_major))
    x['masked_m'][:] = [0, 1, 160, 161, 300, 97]
    print(f'masked stream block_n={bn} mn_major={mn_major} masked_m={x["masked_m"].tolist()}', flush=True)
    sfa = f32(x['sfa'])
    if mn_major:
        sfa = deep_gemm.get_mn_major_tma_aligned_tensor(sfa)
    a, b = (e4m3(x['qa']), sfa), (e4m3(x['qb']), f32(x['sfb']))
    mm = gen.to_dev(x['masked_m'])
    outs = {}
    for v, (bm_, bn_) in [(2, (256, 256)), (5, (160, bn))]:
        d = sentinel_bf16((g, max_m, n))
        deep_gemm.set_tile_override(bm_, bn_, variant=v)
        try:
            deep_gemm.m_grouped_fp8_gemm_nt_masked(a, b, d, mm, expected_m=128)
            cfg = deep_gemm.get_last_config()
        finally:
            deep_gemm.set_tile_override(0, 0)
        torch.cuda.synchronize()
        assert f' v{v} ' in cfg and f'block_n={bn_}' in cfg, cfg
        outs[v] = d
    assert torch.equal(outs[2].view(torch.int16), outs[5].view(torch.int16))


def _masked_call(a, b, d, mm, override=None, expected_m=16):
    if override:
        deep_gemm.set_tile_override(override[1], override[2], variant=override[0])
    try:
        deep_gemm.m_grouped_fp8_gemm_nt_masked(a, b, d, mm, expected_m=expected_m)
        return deep_gemm.get_last_config()
    finally:
        if override:
            deep_gemm.set_tile_override(0, 0)


@pytest.mark.parametrize('bn', [128, 256])
def test_masked_mfma16_vs_oracle(bn):
    """Passes of at most 16 rows on 16 x 16 x 128 MFMAs (block_m 16): the oracle to
    one BF16 ulp, rows >= masked_m untouched, and within rounding of the
    32 x 32 x 64 configuration (block_m 160) on the same inputs. masked_m covers
    0, 1, a partial and a full 16-row pass, 17 (a 32-row pass) and a second pass
    of 16 rows (176)."""
    g, max_m, n, k = 6, 192, 320, 1024
    x = gen.masked_inputs(g, max_m, n, k, seed=60 + bn)
    x['masked_m'][:] = [0, 1, 7, 16, 17, 176]
    a_deq = np.stack([oquant.dequant_per_token(x['qa'][i], x['sfa'][i]) for i in range(g)])
    b_deq = np.stack([oquant.dequant_per_block(x['qb'][i], x['sfb'][i]) for i in range(g)])
    ref, valid = ogemm.gemm_masked(a_deq, b_deq, x['masked_m'])
    a, b = (e4m3(x['qa']), f32(x['sfa'])), (e4m3(x['qb']), f32(x['sfb']))
    mm = gen.to_dev(x['masked_m'])
    outs = {}
    for bm in (16, 160):
        d = sentinel_bf16((g, max_m, n))
        cfg = _masked_call(a, b, d, mm, (5, bm, bn))
        torch.cuda.synchronize()
        assert f'block_m={bm} ' in cfg, cfg
        out = d.float().cpu().numpy()
        diff, _ = report(f'masked stream block_m={bm} block_n={bn}', out[valid], ref[valid])
        assert diff < 1e-3
        tol = np.abs(ref[valid]) * 2.0 ** -8 + 2.0 ** -20 * np.sqrt(k) * np.abs(ref[valid]).max()
        assert np.all(np.abs(out[valid] - ref[valid]) <= tol)
        assert bool((d.view(torch.int16)[torch.from_numpy(~valid).to(DEV)] == SENTINEL).all())
        outs[bm] = out[valid]
    # the two MFMA shapes agree to FP32 rounding of the sums
    assert ogemm.calc_diff(outs[16], outs[160]) < 1e-9
    # the default configuration for decode-sized groups is block_m 16
    d = sentinel_bf16((g, max_m, n))
    cfg = _masked_call(a, b, d, mm, None, expected_m=16)
    assert ' v5 ' in cfg and 'block_m=16 ' in cfg, cfg


@pytest.mark.parametrize('m', [1, 5, 16])
def test_dense_tiny_m_on_stream_kernel(m):
    """Dense calls of at most 16 rows forced onto the weight-streaming kernel's
    16 x 16 x 128 pass run as one group: the oracle, and bitwise equal to a
    masked call whose group has the same rows."""
    n, k = 2112, 7168
    x = gen.dense_inputs(m, n, k, seed=70 + m)
    ref = ogemm.gemm_nt(oquant.dequant_per_token(x['qa'], x['sfa']), oquant.dequant_per_block(x['qb'], x['sfb']))
    a, b = (e4m3(x['qa']), f32(x['sfa'])), (e4m3(x['qb']), f32(x['sfb']))
    d = torch.empty((m, n), dtype=torch.bfloat16, device=DEV)
    deep_gemm.set_tile_override(16, 128, variant=5)
    try:
        deep_gemm.fp8_gemm_nt(a, b, d)
        cfg = deep_gemm.get_last_config()
    finally:
        deep_gemm.set_tile_override(0, 0, variant=0)
    torch.cuda.synchronize()
    assert ' v5 ' in cfg and 'block_m=16 ' in cfg, cfg
    out = d.float().cpu().numpy()
    diff, _ = report(f'dense tiny M={m}', out, ref)
    assert diff < 1e-3
    tol = np.abs(ref) * 2.0 ** -8 + 2.0 ** -20 * np.sqrt(k) * np.abs(ref).max()
    assert np.all(np.abs(out - ref) <= tol)
    # a masked group of the same rows (max_m 32, one group) gives the same bits
    qa = np.zeros((1, 32, k), np.uint8)
    qa[0, :m] = x['qa']
    sfa = np.zeros((1, 32, k // 128), np.float32)
    sfa[0, :m] = x['sfa']
    qb = np.empty((1,) + x['qb'].shape, np.uint8)      # (a fresh array: a [None] view has a 0 group stride)
    qb[0] = x['qb']
    sfb = np.empty((1,) + x['sfb'].shape, np.float32)
    sfb[0] = x['sfb']
    dm = sentinel_bf16((1, 32, n))
    cfg_m = _masked_call((e4m3(qa), f32(sfa)), (e4m3(qb), f32(sfb)), dm,
                         gen.to_dev(np.array([m], np.int32)), None, expected_m=m)
    assert 'block_m=16 ' in cfg_m, cfg_m
    assert torch.equal(dm[0, :m].view(torch.int16), d.view(torch.int16))


@pytest.mark.parametrize('m,n,k', [(1, 2112, 7168), (5, 2112, 7168), (16, 7168, 2048), (3, 104, 384),
                                   (16, 24576, 1536), (7, 4096, 16384), (1, 576, 128), (33, 2112, 7168),
                                   (64, 2112, 7168), (50, 104, 1024), (17, 4096, 4096), (3, 104, 32768),
                                   (96, 2112, 7168), (128, 576, 4096), (100, 104, 1024),   # two to eight row groups
                                   (160, 576, 4096), (256, 104, 1024)])                     # up to sixteen
def test_dense_tiny_m_split_k_kernel(m, n, k):
    """The tiny-M kernel (K split over the waves of a workgroup, partial sums
    added in wave order; up to four 16-row tiles per workgroup), in each of its
    configurations (8 or 4 waves; 16, 32 or 64 columns and 16, 32 or 64 rows per
    workgroup, 64 columns up to 32 rows; M up to 256): the oracle within one BF16 ulp plus
    2^-15 x sum |a b|, ragged M and N (104, not a multiple of 16 or 32), fewer K
    blocks than waves (K = 128, 384), the largest K (256 blocks: 64 per wave at 4
    waves), MN-major SFA equal to K-major, bitwise-identical reruns, and the same
    bits for every split of the rows over workgroups. The default routing takes
    it for N up to 7168; config 1 of the benchmark (64 x 2112 x 7168) is one of these."""
    x = gen.dense_inputs(m, n, k, seed=90 + m + n)
    a_deq, b_deq = oquant.dequant_per_token(x['qa'], x['sfa']), oquant.dequant_per_block(x['qb'], x['sfb'])
    ref = ogemm.gemm_nt(a_deq, b_deq)
    s_abs = ogemm.gemm_nt(np.abs(a_deq), np.abs(b_deq))
    a, b = (e4m3(x['qa']), f32(x['sfa'])), (e4m3(x['qb']), f32(x['sfb']))
    sfa_mn = deep_gemm.get_mn_major_tma_aligned_tensor(a[1])
    tol = np.abs(ref) * 2.0 ** -8 + 2.0 ** -15 * s_abs
    by_cfg = {}
    for v, bn, rows in [(v, bn, rows) for v in (8, 9) for bn in (16, 32, 64) for rows in (64, 32, 16)] + [(0, 0, 0)]:
        if bn == 64 and rows > 32 and m > 32:
            continue
        deep_gemm.set_tile_override(rows, bn, variant=v)
        try:
            d = sentinel_bf16((m, n))
            deep_gemm.fp8_gemm_nt(a, b, d)
            cfg = deep_gemm.get_last_config()
            d2 = torch.empty_like(d)
            deep_gemm.fp8_gemm_nt((a[0], sfa_mn), b, d2)
            for _ in range(5):
                deep_gemm.fp8_gemm_nt(a, b, d)
        finally:
            deep_gemm.set_tile_override(0, 0)
        torch.cuda.synchronize()
        print(f'  {cfg}', flush=True)
        if v:
            assert f' v{v} ' in cfg and f'block_m={rows} block_n={bn} ' in cfg, cfg
        elif 8 < m <= 64 and k >= 6144 and (n + 63) // 64 <= 256:
            assert ' v10 ' in cfg, cfg   # the split-K kernel (below) takes these by default
        elif n <= 7168:
            assert ' v8 ' in cfg or ' v9 ' in cfg, cfg
        out = d.float().cpu().numpy()
        diff, _ = report(f'dense tiny M={m} N={n} K={k} [{cfg.split(" kind")[0]} {rows}x{bn}]', out, ref)
        assert diff < 1e-3
        assert np.all(np.abs(out - ref) <= tol)
        assert torch.equal(d2.view(torch.int16), d.view(torch.int16))
        if v:   # a row tile's arithmetic does not depend on how the rows are split
            first = by_cfg.setdefault((v, bn), d)
            assert torch.equal(first.view(torch.int16), d.view(torch.int16)), f'rows {rows} differ'


@pytest.mark.parametrize('m,n,k', [(64, 2112, 7168), (1, 2112, 7168), (16, 7168, 2048), (33, 4096, 7168),
                                   (7, 576, 7168), (3, 104, 384), (50, 138, 1024), (64, 7168, 16384),
                                   (17, 4096, 4096), (1, 24576, 1536), (64, 64, 32768)])
def test_dense_split_k_kernel(m, n, k):
    """The split-K kernel (64 columns x a chunk of K blocks per workgroup, FP32
    partials in a workspace, added in chunk order by a second kernel): the oracle
    within one BF16 ulp plus 2^-15 x sum |a b| for the heuristic's chunk count and
    forced counts (1, 3, 8, one chunk per K block), ragged M and N (104; 138 in a
    D whose rows are padded to 144, so the last 4-column group is partial),
    MN-major SFA equal to K-major, bitwise-identical reruns. The default routing
    (a workspace from torch) takes it for M <= 64 when it gives at least two
    chunks, more than 8 rows and K >= 6144; config 1 (64 x 2112 x 7168) is one of these."""
    x = gen.dense_inputs(m, n, k, seed=190 + m + n)
    a_deq, b_deq = oquant.dequant_per_token(x['qa'], x['sfa']), oquant.dequant_per_block(x['qb'], x['sfb'])
    ref = ogemm.gemm_nt(a_deq, b_deq)
    s_abs = ogemm.gemm_nt(np.abs(a_deq), np.abs(b_deq))
    a, b = (e4m3(x['qa']), f32(x['sfa'])), (e4m3(x['qb']), f32(x['sfb']))
    sfa_mn = deep_gemm.get_mn_major_tma_aligned_tensor(a[1])
    tol = np.abs(ref) * 2.0 ** -8 + 2.0 ** -15 * s_abs
    nkb = k // 128
    pitch = (n + 7) // 8 * 8   # 16-byte rows

    full = {}

    def out_d():
        full['d'] = sentinel_bf16((m, pitch))
        return full['d'][:, :n]
    for splits in (0, 1, 3, 8, nkb):
        if splits > nkb:
            continue
        deep_gemm.set_tile_override(0, splits, variant=10)
        try:
            d2, d3 = out_d(), out_d()
            d = out_d()
            deep_gemm.fp8_gemm_nt(a, b, d)
            cfg = deep_gemm.get_last_config()
            deep_gemm.fp8_gemm_nt((a[0], sfa_mn), b, d2)
            for _ in range(3):
                deep_gemm.fp8_gemm_nt(a, b, d3)
        finally:
            deep_gemm.set_tile_override(0, 0)
        torch.cuda.synchronize()
        print(f'  {cfg}', flush=True)
        assert ' v10 ' in cfg, cfg
        out = d.float().cpu().numpy()
        diff, _ = report(f'dense split-K M={m} N={n} K={k} [{cfg.split("groups=1 ")[-1]}]', out, ref)
        assert diff < 1e-3
        assert np.all(np.abs(out - ref) <= tol)
        assert torch.equal(d2.view(torch.int16), d.view(torch.int16))
        assert torch.equal(d3.view(torch.int16), d.view(torch.int16))
        if pitch > n:   # the padding columns of D stay untouched
            assert bool((full['d'][:, n:].view(torch.int16) == SENTINEL).all())
    d = out_d()
    deep_gemm.fp8_gemm_nt(a, b, d)
    cfg = deep_gemm.get_last_config()
    torch.cuda.synchronize()
    if m > 8 and k >= 6144 and (n + 63) // 64 <= 256:
        assert ' v10 ' in cfg, cfg
    else:
        assert ' v10 ' not in cfg, cfg
    assert np.all(np.abs(d.float().cpu().numpy() - ref) <= tol)


def test_dense_split_k_workspace_rules():
    """The workspace entry point: the size query matches what a call needs, a
    workspace one byte short runs the workspace-free kernels instead (same
    oracle bound), and the plain entry point never takes the split-K path."""
    m, n, k = 64, 2112, 7168
    lib = deep_gemm._ffi.lib
    need = lib.dg_fp8_gemm_nt_workspace_size(m, n, k)
    assert need == 33 * 7 * 64 * 64 * 4, need   # FP32 partials: column slices x chunks x rows x 64
    assert lib.dg_fp8_gemm_nt_workspace_size(65, n, k) == 0       # more than 64 rows
    assert lib.dg_fp8_gemm_nt_workspace_size(8, n, k) == 0        # 8 rows: the single-launch kernels win
    assert lib.dg_fp8_gemm_nt_workspace_size(m, n, 4096) == 0     # K < 6144 likewise
    assert lib.dg_fp8_gemm_nt_workspace_size(m, n, 7168 + 64) == 0  # K tail
    assert lib.dg_fp8_gemm_nt_workspace_size(m, 24576, 1536) == 0   # one chunk per CU already
    x = gen.dense_inputs(m, n, k, seed=201)
    ref = ogemm.gemm_nt(oquant.dequant_per_token(x['qa'], x['sfa']), oquant.dequant_per_block(x['qb'], x['sfb']))
    a, b = (e4m3(x['qa']), f32(x['sfa'])), (e4m3(x['qb']), f32(x['sfb']))
    from deep_gemm._ffi import describe, ref as cref
    outs = []
    for nbytes, entry in ((need, 'ws'), (need - 16, 'ws'), (0, 'plain')):
        d = sentinel_bf16((m, n))
        dd = describe(d)
        args = [cref(describe(t)) for t in (a[0], a[1], b[0], b[1])] + [cref(dd), None, None, 0, None]
        if entry == 'ws':
            ws = torch.empty((max(nbytes, 16),), dtype=torch.uint8, device=DEV)
            st = lib.dg_fp8_fp4_gemm_nt_ws(*args, cref(describe(ws)), deep_gemm._ffi.stream_of(d))
        else:
            st = lib.dg_fp8_fp4_gemm_nt(*args, deep_gemm._ffi.stream_of(d))
        assert st == 0, lib.dg_last_error()
        outs.append((deep_gemm.get_last_config(), d))
    torch.cuda.synchronize()
    assert ' v10 ' in outs[0][0] and ' v10 ' not in outs[1][0] and ' v10 ' not in outs[2][0], [o[0] for o in outs]
    assert torch.equal(outs[1][1].view(torch.int16), outs[2][1].view(torch.int16))
    for _, d in outs:
        assert ogemm.calc_diff(d.float().cpu().numpy(), ref) < 1e-3


def test_dense_tiny_m_k_bound():
    """The tiny-M kernel keeps a wave's B scales in one register (at most 64 K
    blocks per wave, 256 in all): with 257 K blocks a forced call is refused
    before any launch, and the default routing takes a tiled kernel, which
    agrees with the oracle."""
    m, n, k = 3, 104, 257 * 128
    x = gen.dense_inputs(m, n, k, seed=97)
    ref = ogemm.gemm_nt(oquant.dequant_per_token(x['qa'], x['sfa']), oquant.dequant_per_block(x['qb'], x['sfb']))
    a, b = (e4m3(x['qa']), f32(x['sfa'])), (e4m3(x['qb']), f32(x['sfb']))
    d = sentinel_bf16((m, n))
    deep_gemm.set_tile_override(64, 16, variant=9)
    try:
        with pytest.raises(RuntimeError, match='tiny-M'):
            deep_gemm.fp8_gemm_nt(a, b, d)
    finally:
        deep_gemm.set_tile_override(0, 0)
    torch.cuda.synchronize()
    assert bool((d.view(torch.int16) == SENTINEL).all())
    deep_gemm.fp8_gemm_nt(a, b, d)
    cfg = deep_gemm.get_last_config()
    assert ' v8 ' not in cfg and ' v9 ' not in cfg, cfg
    out = d.float().cpu().numpy()
    diff, _ = report(f'dense M={m} K={k} [{cfg.split(" kind")[0]}]', out, ref)
    assert diff < 1e-3


@pytest.mark.parametrize('m', [17, 33, 64])
def test_dense_small_m_stream_equals_tiled(m):
    """Dense calls of 17 to 64 rows forced onto the weight-streaming kernel's
    32 x 32 x 64 passes (block_m 160) are bitwise equal to the pipelined tiles
    (same MFMA pair, same per-K-block promotion order) and to the oracle within
    one BF16 ulp."""
    n, k = 7168, 2048
    x = gen.dense_inputs(m, n, k, seed=80 + m)
    a, b = (e4m3(x['qa']), f32(x['sfa'])), (e4m3(x['qb']), f32(x['sfb']))
    d = torch.empty((m, n), dtype=torch.bfloat16, device=DEV)
    deep_gemm.set_tile_override(160, 224, variant=5)
    try:
        deep_gemm.fp8_gemm_nt(a, b, d)
        cfg = deep_gemm.get_last_config()
    finally:
        deep_gemm.set_tile_override(0, 0)
    assert ' v5 ' in cfg and 'block_m=160 ' in cfg, cfg
    d2 = torch.empty_like(d)
    deep_gemm.set_tile_override(128, 128, variant=2)
    try:
        deep_gemm.fp8_gemm_nt(a, b, d2)
    finally:
        deep_gemm.set_tile_override(0, 0)
    torch.cuda.synchronize()
    assert torch.equal(d.view(torch.int16), d2.view(torch.int16))
    ref = ogemm.gemm_nt(oquant.dequant_per_token(x['qa'], x['sfa']), oquant.dequant_per_block(x['qb'], x['sfb']))
    out = d.float().cpu().numpy()
    diff, _ = report(f'dense small M={m} (stream)', out, ref)
    tol = np.abs(ref) * 2.0 ** -8 + 2.0 ** -20 * np.sqrt(k) * np.abs(ref).max()
    assert diff < 1e-3 and np.all(np.abs(out - ref) <= tol)


# ------------------------------------------------- persistent workgroups (variant 4)

def _with_variant(v, fn):
    try:
        deep_gemm.set_tile_override(256, 256, variant=v)
        out = fn()
        torch.cuda.synchronize()
        return out, deep_gemm.get_last_config()
    finally:
        deep_gemm.set_tile_override(0, 0)


@pytest.mark.parametrize('num_sms', [0, 7])
@pytest.mark.parametrize('case', ['dense', 'dense_ragged', 'contiguous', 'masked', 'psum'])
def test_persistent_equals_per_tile_launch(case, num_sms):
    """The persistent scheduler (grid = CU count, tile stride = grid, masked and
    psum group walks) gives the same bits as one workgroup per tile: same tile
    shape, same per-output K order; rows it must not touch stay untouched. With
    num_sms = 7 every workgroup walks several tiles, so the dense and masked
    walks also issue each next tile's first stage during the epilogue (ragged
    M and N edges and one-row groups included)."""
    print(f'persistent {case} num_sms={num_sms or "all"}', flush=True)
    if case in ('dense', 'dense_ragged'):
        m, n, k = (1024, 2048, 1024) if case == "dense" else (1300, 712, 896)
        x = gen.dense_inputs(m, n, k, seed=91)
        a, b = (e4m3(x['qa']), f32(x['sfa'])), (e4m3(x['qb']), f32(x['sfb']))

        def run():
            d = sentinel_bf16((m, n))
            deep_gemm.fp8_gemm_nt(a, b, d)
            return d
    elif case == 'contiguous':
        ms = [130, 100, 300, 0, 250, 1, 700]
        aligned = [(mi + 127) // 128 * 128 for mi in ms]
        x = gen.contiguous_inputs(ms, aligned, 384, 1024, seed=92)
        a, b = (e4m3(x['qa']), f32(x['sfa'])), (e4m3(x['qb']), f32(x['sfb']))
        mi_dev = gen.to_dev(x['m_indices'])

        def run():
            d = sentinel_bf16((sum(aligned), 384))
            deep_gemm.m_grouped_fp8_gemm_nt_contiguous(a, b, d, mi_dev)
            return d
    elif case == 'masked':
        x = gen.masked_inputs(6, 512, 512, 1024, seed=93)
        x['masked_m'][:] = [0, 1, 256, 300, 512, 129]
        a, b = (e4m3(x['qa']), f32(x['sfa'])), (e4m3(x['qb']), f32(x['sfb']))
        mm = gen.to_dev(x['masked_m'])

        def run():
            d = sentinel_bf16((6, 512, 512))
            deep_gemm.m_grouped_fp8_gemm_nt_masked(a, b, d, mm, expected_m=256)
            return d
    else:
        # 256-row tiles need a 256-row psum alignment
        ms = [100, 0, 257, 64, 513]
        align = 256
        aligned = [(mi + align - 1) // align * align for mi in ms]
        x = gen.contiguous_inputs(ms, aligned, 256, 512, seed=94)
        a, b = (e4m3(x['qa']), f32(x['sfa'])), (e4m3(x['qb']), f32(x['sfb']))
        ends, prev = [], 0
        for mi in ms:
            st = (prev + align - 1) // align * align
            ends.append(st + mi)
            prev = st + mi
        psum = torch.tensor(ends, dtype=torch.int32, device=DEV)
        m_pad = (ends[-1] + align - 1) // align * align

        def run():
            d = sentinel_bf16((m_pad, 256))
            deep_gemm.m_grouped_fp8_gemm_nt_contiguous(a, b, d, psum, use_psum_layout=True,
                                                       ensure_zero_padding=True)
            return d
    old_align = deep_gemm.get_mk_alignment_for_contiguous_layout()
    old_sms = deep_gemm.get_num_sms()
    if case == 'psum':
        deep_gemm.set_mk_alignment_for_contiguous_layout(256)
    try:
        if num_sms:
            deep_gemm.set_num_sms(num_sms)
        ref, cfg_ref = _with_variant(2, run)
        got, cfg = _with_variant(4, run)
    finally:
        deep_gemm.set_mk_alignment_for_contiguous_layout(old_align)
        deep_gemm.set_num_sms(old_sms)
    print(cfg_ref, '|', cfg, flush=True)
    assert 'v4' in cfg
    assert torch.equal(ref.view(torch.int16), got.view(torch.int16))
    # and against the oracle: the rows the call writes, within one BF16 ulp plus the
    # accumulation term; the rest keep the sentinel
    if case in ('dense', 'dense_ragged'):
        oref = ogemm.gemm_nt(oquant.dequant_per_token(x['qa'], x['sfa']), oquant.dequant_per_block(x['qb'], x['sfb']))
        written = np.ones(oref.shape[0], dtype=bool)
    else:
        groups = x['qb'].shape[0]
        b_deq = np.stack([oquant.dequant_per_block(x['qb'][i], x['sfb'][i]) for i in range(groups)])
        if case == 'masked':
            a_deq = np.stack([oquant.dequant_per_token(x['qa'][i], x['sfa'][i]) for i in range(groups)])
            oref, written = ogemm.gemm_masked(a_deq, b_deq, x['masked_m'])
        else:
            a_deq = oquant.dequant_per_token(x['qa'], x['sfa'])
            if case == 'contiguous':
                oref, written = ogemm.gemm_contiguous(a_deq, b_deq, x['m_indices'])
            else:
                oref, written = ogemm.gemm_psum(a_deq, b_deq, ends, 256, 256, True)
    out = got.float().cpu().numpy()
    diff, _ = report(f'persistent {case} vs oracle', out[written], oref[written])
    assert diff < 1e-3
    k = x['qa'].shape[-1]
    tol = np.abs(oref[written]) * 2.0 ** -8 + 2.0 ** -20 * np.sqrt(k) * np.abs(oref[written]).max()
    assert np.all(np.abs(out[written] - oref[written]) <= tol)
    assert bool((got.view(torch.int16)[torch.from_numpy(~written).to(DEV)] == SENTINEL).all())


@pytest.mark.parametrize('expected_m,persistent', [(200, True), (1000, True), (1100, False)])
def test_masked_routing_persistent_when_sparse(expected_m, persistent):
    """Masked calls whose expected_m leaves at least half of max_m's 256-row blocks
    empty run the persistent walk (variant 4) by default, otherwise one workgroup
    per tile; either way the bits are those of the forced per-tile launch, and rows
    past masked_m keep the sentinel. masked_m values far from expected_m (0, 1,
    a whole group) only change the speed."""
    print(f'masked routing expected_m={expected_m}', flush=True)
    g, max_m, n, k = 5, 2048, 4096, 1024
    x = gen.masked_inputs(g, max_m, n, k, seed=95)
    x['masked_m'][:] = [0, 1, 300, 2048, 700]
    a, b = (e4m3(x['qa']), f32(x['sfa'])), (e4m3(x['qb']), f32(x['sfb']))
    mm = gen.to_dev(x['masked_m'])

    def run():
        d = sentinel_bf16((g, max_m, n))
        deep_gemm.m_grouped_fp8_gemm_nt_masked(a, b, d, mm, expected_m=expected_m)
        return d

    deep_gemm.set_tile_override(0, 0)
    got = run()
    torch.cuda.synchronize()
    cfg = deep_gemm.get_last_config()
    ref, cfg_ref = _with_variant(2, run)
    print(cfg, '|', cfg_ref, flush=True)
    assert ('v4' in cfg) == persistent and 'block_m=256 block_n=256' in cfg
    assert torch.equal(ref.view(torch.int16), got.view(torch.int16))
    rows = torch.arange(max_m, device=DEV)[None, :] >= mm[:, None]
    assert bool((got.view(torch.int16)[rows] == SENTINEL).all())


@pytest.mark.parametrize('case,k,persistent', [('dense', 1536, True), ('dense', 2176, False),
                                               ('contiguous', 2048, True), ('contiguous', 4096, True)])
def test_many_rounds_routes_persistent(case, k, persistent):
    """Contiguous calls, and dense calls with K <= 2048, with at least four rounds
    of 256 x 256 tiles on the CUs (BF16 D, no C) run the persistent walk by
    default, in one launch; the bits are those of the forced per-tile launch."""
    print(f'many-rounds routing {case} k={k}', flush=True)
    if case == 'dense':
        m, n = 4096, 16384   # 16 x 64 = 1024 tiles: four rounds on 256 CUs
        x = gen.dense_inputs(m, n, k, seed=96)
        a, b = (e4m3(x['qa']), f32(x['sfa'])), (e4m3(x['qb']), f32(x['sfb']))

        def run():
            d = sentinel_bf16((m, n))
            deep_gemm.fp8_gemm_nt(a, b, d)
            return d
    else:
        ms = [3000, 0, 5000, 129, 7000, 1200]
        aligned = [(mi + 127) // 128 * 128 for mi in ms]
        x = gen.contiguous_inputs(ms, aligned, 4096, k, seed=97)
        a, b = (e4m3(x['qa']), f32(x['sfa'])), (e4m3(x['qb']), f32(x['sfb']))
        mi_dev = gen.to_dev(x['m_indices'])

        def run():
            d = sentinel_bf16((sum(aligned), 4096))
            deep_gemm.m_grouped_fp8_gemm_nt_contiguous(a, b, d, mi_dev)
            return d
    deep_gemm.set_tile_override(0, 0)
    got = run()
    torch.cuda.synchronize()
    cfg = deep_gemm.get_last_config()
    ref, cfg_ref = _with_variant(2, run)
    print(cfg, '|', cfg_ref, flush=True)
    if deep_gemm.get_num_sms() >= 256:
        assert ('v4' in cfg) == persistent
        assert 'split_m=' not in cfg, cfg
    assert torch.equal(ref.view(torch.int16), got.view(torch.int16))


@pytest.mark.parametrize('num_sms', [48, 7])
def test_persistent_routes_with_fewer_cus(num_sms):
    """With set_num_sms below the chip's CU count the persistent launches run that
    many workgroups (each walks more tiles), and the four-round rule counts
    rounds on that many CUs: contiguous and sparse masked calls give the bits of
    the per-tile launch."""
    old = deep_gemm.get_num_sms()
    print(f'persistent with num_sms={num_sms}', flush=True)
    ms = [1500, 0, 1800, 129, 900]   # 19 M blocks x 16 N blocks: >= 4 rounds on 48 CUs
    aligned = [(mi + 127) // 128 * 128 for mi in ms]
    x = gen.contiguous_inputs(ms, aligned, 4096, 1024, seed=98)
    a, b = (e4m3(x['qa']), f32(x['sfa'])), (e4m3(x['qb']), f32(x['sfb']))
    mi_dev = gen.to_dev(x['m_indices'])
    xm = gen.masked_inputs(4, 1024, 2048, 1024, seed=99)
    xm['masked_m'][:] = [0, 1, 256, 300]
    am, bm = (e4m3(xm['qa']), f32(xm['sfa'])), (e4m3(xm['qb']), f32(xm['sfb']))
    mm = gen.to_dev(xm['masked_m'])

    def run_c():
        d = sentinel_bf16((sum(aligned), 4096))
        deep_gemm.m_grouped_fp8_gemm_nt_contiguous(a, b, d, mi_dev)
        return d

    def run_m():
        d = sentinel_bf16((4, 1024, 2048))
        deep_gemm.m_grouped_fp8_gemm_nt_masked(am, bm, d, mm, expected_m=200)
        return d

    try:
        deep_gemm.set_num_sms(num_sms)
        for run in (run_c, run_m):
            deep_gemm.set_tile_override(0, 0)
            got = run()
            torch.cuda.synchronize()
            cfg = deep_gemm.get_last_config()
            ref, cfg_ref = _with_variant(2, run)
            print(cfg, '|', cfg_ref, flush=True)
            assert ' v4 ' in cfg
            assert torch.equal(ref.view(torch.int16), got.view(torch.int16))
    finally:
        deep_gemm.set_num_sms(old)


# ----------------------------------------------------------------- SF layouts

# the reference's grid (tests/generators.py:276-285, tests/test_layout.py:45-80), plus a ragged mn
SF_LAYOUT_CASES = [(mn, k, g) for mn in (4096, 4097, 8192) for k in (128, 7168, 7296) for g in (1, 2, 4)] + \
                  [(300, 7296, 4)]


@pytest.mark.parametrize('mn,k,g', SF_LAYOUT_CASES)
def test_sf_transpose_and_pack(mn, k, g):
    sfk = (k + 127) // 128
    rng = np.random.default_rng(mn + k)
    sf_np = rng.standard_normal((g, mn, sfk)).astype(np.float32)
    sf = gen.to_dev(sf_np)
    out = deep_gemm.get_mn_major_tma_aligned_tensor(sf)
    amn = deep_gemm.get_tma_aligned_size(mn, 4)
    assert out.stride() == (amn * sfk, 1, amn)
    assert torch.equal(out, sf)
    # transposed (non-contiguous) input takes the strided path
    sf_t = sf.transpose(-1, -2).contiguous().transpose(-1, -2)
    assert torch.equal(deep_gemm.get_mn_major_tma_aligned_tensor(sf_t), sf)
    # UE8M0 packing, bitwise against the oracle's restatement of tests/test_layout.py:20-42
    pow2 = np.ldexp(np.float32(1.0), rng.integers(-20, 20, size=(g, mn, sfk))).astype(np.float32)
    packed = deep_gemm.get_mn_major_tma_aligned_packed_ue8m0_tensor(gen.to_dev(pow2))
    ref_storage = ogemm.pack_ue8m0_mn_major(pow2)       # [g, ceil(k/4), amn]
    pk = (sfk + 3) // 4
    assert packed.shape == (g, mn, pk) and packed.stride() == (amn * pk, 1, amn)
    got = packed.cpu().numpy()
    assert np.array_equal(got, np.swapaxes(ref_storage, 1, 2)[:, :mn, :])


# ----------------------------------------------------------------- FP8 x FP4

@pytest.mark.parametrize('m,n,k,a_fp4,gka', [(256, 384, 1024, False, 128), (100, 200, 512, False, 128),
                                              (128, 256, 512, True, 32)])
def test_fp8_fp4_vs_oracle(m, n, k, a_fp4, gka):
    print(f'fp8xfp4 m={m} n={n} k={k} a_fp4={a_fp4}', flush=True)
    x = gen.fp8_fp4_inputs(m, n, k, seed=m + k, gran_k_a=gka, gran_k_b=32, a_fp4=a_fp4)
    a_deq = oquant.dequant_fp4(x['qa'], x['sfa'], gka) if a_fp4 else oquant.dequant_per_token(x['qa'], x['sfa'], gka)
    ref = ogemm.gemm_nt(a_deq, oquant.dequant_fp4(x['qb'], x['sfb'], 32))
    a_t = gen.to_dev(x['qa'], torch.int8) if a_fp4 else e4m3(x['qa'])
    a = (a_t, f32(x['sfa']))
    b = (gen.to_dev(x['qb'], torch.int8), f32(x['sfb']))
    d = torch.empty((m, n), dtype=torch.bfloat16, device=DEV)
    deep_gemm.fp8_fp4_gemm_nt(a, b, d, recipe_a=(1, gka), recipe_b=(1, 32))
    torch.cuda.synchronize()
    out = d.float().cpu().numpy()
    diff, rel = report('fp8xfp4', out, ref)
    assert diff < 1e-5   # power-of-two scales: only BF16 output rounding remains
    # packed-UE8M0 SFs give the same bits
    pa = deep_gemm.transform_sf_into_required_layout(a[1], m, k, (1, gka))
    pb = deep_gemm.transform_sf_into_required_layout(b[1], n, k, (1, 32))
    assert pa.dtype == torch.int32 or gka == 128
    d2 = torch.empty_like(d)
    pa_i = deep_gemm.get_mn_major_tma_aligned_packed_ue8m0_tensor(a[1])
    deep_gemm.fp8_fp4_gemm_nt((a[0], pa_i), (b[0], pb), d2, recipe_a=(1, gka), recipe_b=(1, 32))
    assert torch.equal(d.view(torch.int16), d2.view(torch.int16))


# ------------------------------------------------- UE8M0: 256 x 256 pipelined kernel

def _ue8m0_quant(x, fp4, gran):
    """Codes and FP32 power-of-two SFs of one operand (rows x K), and its dequant."""
    if fp4:
        q, sf = oquant.per_token_cast_to_fp4(x, use_ue8m0=True, gran_k=gran)
        return q, sf, oquant.dequant_fp4(q, sf, gran)
    q, sf = oquant.per_token_cast_to_fp8(x, use_ue8m0=True, gran_k=gran)
    return q, sf, oquant.dequant_per_token(q, sf, gran)


def _ue8m0_grouped(x, fp4, gran):
    """_ue8m0_quant over the leading group axis."""
    parts = [_ue8m0_quant(x[i], fp4, gran) for i in range(x.shape[0])]
    return tuple(np.stack([p[j] for p in parts]) for j in range(3))


def _codes_dev(q, fp4):
    return gen.to_dev(q, torch.int8) if fp4 else e4m3(q)


def _packed(sf):
    """FP32 power-of-two SFs -> packed MN-major UE8M0 words on the device."""
    return deep_gemm.get_mn_major_tma_aligned_packed_ue8m0_tensor(f32(sf))


def _run_both_kernels(fn):
    """Runs fn() on the 128 x 128 UE8M0 kernel and on the pipelined one; returns
    (outputs, configs) of both."""
    outs, cfgs = [], []
    try:
        for v, bm, bn in ((1, 128, 128), (2, 256, 256)):
            deep_gemm.set_tile_override(bm, bn, variant=v)
            outs.append(fn())
            cfgs.append(deep_gemm.get_last_config())
            print(cfgs[-1], flush=True)
    finally:
        deep_gemm.set_tile_override(0, 0)
    assert 'pipe' in cfgs[1] and 'pipe' not in cfgs[0]
    return outs, cfgs


UE8M0_DENSE = [
    # m, n, k, a_fp4, b_fp4, gran_k_a, gran_k_b
    (512, 768, 1024, False, True, 128, 32),    # config 5 recipe, interior tiles
    (300, 520, 640, False, True, 128, 32),     # ragged M and N, 5 K blocks (gran-128 word tail)
    (1, 64, 128, False, True, 128, 32),        # one row, one K block
    (257, 384, 768, False, False, 32, 32),     # e4m3 x e4m3, 1x32 scales
    (200, 256, 512, False, False, 128, 128),   # e4m3 x e4m3, 1x128 scales
    (320, 448, 1024, True, True, 32, 32),      # e2m1 x e2m1
    (130, 300, 384, True, False, 32, 128),     # e2m1 x e4m3
]


@pytest.mark.parametrize('m,n,k,a_fp4,b_fp4,gka,gkb', UE8M0_DENSE)
def test_ue8m0_pipe_dense(m, n, k, a_fp4, b_fp4, gka, gkb):
    """Pipelined UE8M0 kernel: oracle parity, the same bits as the 128 x 128 kernel
    (same MFMA, same per-output K order), bounds and 20-rerun determinism."""
    print(f'ue8m0 pipe dense m={m} n={n} k={k} a_fp4={a_fp4} b_fp4={b_fp4} gk=({gka},{gkb})', flush=True)
    qa, sfa, a_deq = _ue8m0_quant(gen.randn_bf16((m, k), m + 3), a_fp4, gka)
    qb, sfb, b_deq = _ue8m0_quant(gen.randn_bf16((n, k), n + 5), b_fp4, gkb)
    ref = ogemm.gemm_nt(a_deq, b_deq)
    a = (_codes_dev(qa, a_fp4), _packed(sfa))
    b = (_codes_dev(qb, b_fp4), _packed(sfb))
    # d is a strided view (row pitch a multiple of 16 bytes); the rest must stay untouched
    big = sentinel_bf16((m + 8, (n + 72 + 7) // 8 * 8))

    def call():
        big.view(torch.int16).fill_(SENTINEL)
        d = big[:m, :n]
        deep_gemm.fp8_fp4_gemm_nt(a, b, d, recipe_a=(1, gka), recipe_b=(1, gkb))
        torch.cuda.synchronize()
        return big.clone()

    (old, new), _ = _run_both_kernels(call)
    out = new[:m, :n].float().cpu().numpy()
    diff, _ = report('ue8m0 pipe', out, ref)
    assert diff < 1e-5   # power-of-two scales: only FP32 accumulation and BF16 rounding remain
    assert torch.equal(old.view(torch.int16), new.view(torch.int16))
    outside = torch.ones_like(new, dtype=torch.bool)
    outside[:m, :n] = False
    assert bool((new.view(torch.int16)[outside] == SENTINEL).all())
    # determinism (few rows are the tiny-M kernel's by default, test_ue8m0_tiny_m)
    d = big[:m, :n]
    deep_gemm.set_tile_override(256, 256, variant=2)
    try:
        for _ in range(20):
            deep_gemm.fp8_fp4_gemm_nt(a, b, d, recipe_a=(1, gka), recipe_b=(1, gkb))
    finally:
        deep_gemm.set_tile_override(0, 0)
    assert 'pipe' in deep_gemm.get_last_config()
    assert torch.equal(big.view(torch.int16), new.view(torch.int16))


@pytest.mark.parametrize('m,n,k,b_fp4,kernel', [
    (1, 64, 128, True, 'tinym'), (64, 4096, 512, True, 'tinym'), (100, 4096, 1024, False, 'tinym'),
    (64, 520, 1152, True, 'tinym'), (400, 7168, 512, True, 'pipe'), (4096, 4096, 1024, False, 'pipe')])
def test_ue8m0_few_rows_route(m, n, k, b_fp4, kernel):
    """The kernel of a dense call follows from its size at every K; what it gives is the
    pipelined kernel's result but for the order of the sums."""
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    x, w = torch.randn((m, k), generator=g, device=DEV).bfloat16(), torch.randn((n, k), generator=g, device=DEV).bfloat16()
    pack = deep_gemm.get_mn_major_tma_aligned_packed_ue8m0_tensor
    qa, sfa = deep_gemm.per_token_cast_to_fp8(x, use_ue8m0=True)
    qb, sfb = (deep_gemm.per_token_cast_to_fp4(w, use_ue8m0=True, gran_k=32) if b_fp4 else
               deep_gemm.per_token_cast_to_fp8(w, use_ue8m0=True))
    a, b, outs = (qa, pack(sfa)), (qb, pack(sfb)), []
    for v in (0, 2):
        d = torch.empty((m, n), dtype=torch.bfloat16, device=DEV)
        deep_gemm.set_tile_override(256 if v else 0, 256 if v else 0, variant=v)
        try:
            deep_gemm.fp8_fp4_gemm_nt(a, b, d, recipe_a=(1, 128), recipe_b=(1, 32 if b_fp4 else 128))
            if v == 0 and deep_gemm.get_num_sms() >= 256:
                assert f'ue8m0_{kernel} ' in deep_gemm.get_last_config()
        finally:
            deep_gemm.set_tile_override(0, 0)
        outs.append(d.float())
    torch.cuda.synchronize()
    # (one BF16 rounding apart where FP32 sums of another order straddle one)
    assert bool(((outs[0] - outs[1]).abs() <= outs[1].abs() * 2.0 ** -7 + 2.0 ** -15 * k ** 0.5 * 8).all())


@pytest.mark.parametrize('out_f32,with_c', [(True, True), (True, False), (False, True)])
def test_ue8m0_pipe_dense_c_and_f32(out_f32, with_c):
    m, n, k = 384, 512, 512
    qa, sfa, a_deq = _ue8m0_quant(gen.randn_bf16((m, k), 61), False, 128)
    qb, sfb, b_deq = _ue8m0_quant(gen.randn_bf16((n, k), 62), True, 32)
    c_np = gen.randn_bf16((m, n), 63).astype(np.float32)
    ref = ogemm.gemm_nt(a_deq, b_deq, c_np if with_c else None)
    a = (e4m3(qa), _packed(sfa))
    b = (gen.to_dev(qb, torch.int8), _packed(sfb))
    dt = torch.float32 if out_f32 else torch.bfloat16
    c = torch.from_numpy(c_np).to(dt).to(DEV) if with_c else None

    def call():
        d = torch.empty((m, n), dtype=dt, device=DEV)
        deep_gemm.fp8_fp4_gemm_nt(a, b, d, c=c, recipe_a=(1, 128), recipe_b=(1, 32))
        torch.cuda.synchronize()
        return d

    (old, new), _ = _run_both_kernels(call)
    diff, _ = report(f'ue8m0 pipe f32={out_f32} c={with_c}', new.float().cpu().numpy(), ref)
    assert diff < 1e-5
    assert torch.equal(old, new)


def test_ue8m0_pipe_masked():
    g, max_m, n, k = 5, 320, 384, 768
    masked = np.array([0, 1, 128, 320, 200], np.int32)
    qa, sfa, a_deq = _ue8m0_grouped(gen.randn_bf16((g, max_m, k), 71), False, 128)
    qb, sfb, b_deq = _ue8m0_grouped(gen.randn_bf16((g, n, k), 72), True, 32)
    ref, valid = ogemm.gemm_masked(a_deq, b_deq, masked)
    a = (e4m3(qa), _packed(sfa))
    b = (gen.to_dev(qb, torch.int8), _packed(sfb))
    mm = gen.to_dev(masked)

    def call():
        d = sentinel_bf16((g, max_m, n))
        deep_gemm.m_grouped_fp8_fp4_gemm_nt_masked(a, b, d, mm, 128, recipe_a=(1, 128), recipe_b=(1, 32))
        torch.cuda.synchronize()
        return d

    (old, new), _ = _run_both_kernels(call)
    out = new.float().cpu().numpy()
    diff, _ = report('ue8m0 pipe masked', out[valid], ref[valid])
    assert diff < 1e-5
    assert bool((new.view(torch.int16)[torch.from_numpy(~valid).to(DEV)] == SENTINEL).all())
    assert torch.equal(old.view(torch.int16), new.view(torch.int16))
    # each group equals the dense call on its valid rows
    for i in range(g):
        r = int(masked[i])
        if r:
            dd = torch.empty((r, n), dtype=torch.bfloat16, device=DEV)
            deep_gemm.fp8_fp4_gemm_nt((a[0][i, :r], _packed(sfa[i, :r])), (b[0][i], b[1][i]), dd,
                                      recipe_a=(1, 128), recipe_b=(1, 32))
            assert torch.equal(dd.view(torch.int16), new[i, :r].view(torch.int16)), f'group {i}'


@pytest.mark.parametrize('ms', [[130, 100, 300, 0, 250, 1], [256, 512, 128]])
def test_ue8m0_pipe_contiguous(ms):
    """Segments 128-aligned, so 256-row tiles straddle two experts (two-pass tiles)."""
    aligned = [(mi + 127) // 128 * 128 for mi in ms]
    g, n, k = len(ms), 384, 512
    m_pad = sum(aligned)
    m_indices = np.full(m_pad, -1, np.int32)
    start = 0
    for i, (mi, ai) in enumerate(zip(ms, aligned)):
        m_indices[start:start + mi] = i
        start += ai
    qa, sfa, a_deq = _ue8m0_quant(gen.randn_bf16((m_pad, k), 81), False, 128)
    qb, sfb, b_deq = _ue8m0_grouped(gen.randn_bf16((g, n, k), 82), True, 32)
    ref, valid = ogemm.gemm_contiguous(a_deq, b_deq, m_indices)
    a = (e4m3(qa), _packed(sfa))
    b = (gen.to_dev(qb, torch.int8), _packed(sfb))
    mi_dev = gen.to_dev(m_indices)

    def call():
        d = sentinel_bf16((m_pad, n))
        deep_gemm.m_grouped_fp8_fp4_gemm_nt_contiguous(a, b, d, mi_dev, recipe_a=(1, 128), recipe_b=(1, 32))
        torch.cuda.synchronize()
        return d

    (old, new), _ = _run_both_kernels(call)
    out = new.float().cpu().numpy()
    diff, _ = report('ue8m0 pipe contiguous', out[valid], ref[valid])
    assert diff < 1e-5
    assert bool((new.view(torch.int16)[torch.from_numpy(~valid).to(DEV)] == SENTINEL).all())
    assert torch.equal(old.view(torch.int16), new.view(torch.int16))
    start = 0
    for i, (mi, ai) in enumerate(zip(ms, aligned)):
        if mi:
            dd = torch.empty((mi, n), dtype=torch.bfloat16, device=DEV)
            deep_gemm.fp8_fp4_gemm_nt((a[0][start:start + mi], _packed(sfa[start:start + mi])), (b[0][i], b[1][i]),
                                      dd, recipe_a=(1, 128), recipe_b=(1, 32))
            assert torch.equal(dd.view(torch.int16), new[start:start + mi].view(torch.int16)), f'segment {i}'
        start += ai


# ----------------------------------------------------------------- quantizers

def test_product_quantizers_match_oracle_on_gpu():
    a = gen.randn_bf16((96, 1000), 31)
    ta = torch.from_numpy(a).bfloat16().to(DEV)
    q, s = deep_gemm.per_token_cast_to_fp8(ta, use_ue8m0=False)
    oq, os_ = oquant.per_token_cast_to_fp8(a, use_ue8m0=False)
    assert np.array_equal(q.view(torch.uint8).cpu().numpy(), oq) and np.array_equal(s.cpu().numpy(), os_)
    q, s = deep_gemm.per_block_cast_to_fp8(ta, use_ue8m0=True)
    oq, os_ = oquant.per_block_cast_to_fp8(a, use_ue8m0=True)
    assert np.array_equal(q.view(torch.uint8).cpu().numpy(), oq) and np.array_equal(s.cpu().numpy(), os_)
    q, s = deep_gemm.per_token_cast_to_fp4(ta, use_ue8m0=True, gran_k=32)
    oq, os_ = oquant.per_token_cast_to_fp4(a, use_ue8m0=True, gran_k=32)
    assert np.array_equal(q.view(torch.uint8).cpu().numpy(), oq) and np.array_equal(s.cpu().numpy(), os_)


def test_fp8_ue8m0_gran32_vs_oracle():
    """e4m3 x e4m3 with 1x32 power-of-two scales on both sides (scaled-MFMA path)."""
    m, n, k = 192, 320, 768
    a = gen.randn_bf16((m, k), 41)
    b = gen.randn_bf16((n, k), 42)
    qa, sfa = oquant.per_token_cast_to_fp8(a, use_ue8m0=True, gran_k=32)
    qb, sfb = oquant.per_token_cast_to_fp8(b, use_ue8m0=True, gran_k=32)
    ref = ogemm.gemm_nt(oquant.dequant_per_token(qa, sfa, 32), oquant.dequant_per_token(qb, sfb, 32))
    d = torch.empty((m, n), dtype=torch.bfloat16, device=DEV)
    deep_gemm.fp8_fp4_gemm_nt((e4m3(qa), f32(sfa)), (e4m3(qb), f32(sfb)), d, recipe_a=(1, 32), recipe_b=(1, 32))
    diff, _ = report('fp8 ue8m0 gran32', d.float().cpu().numpy(), ref)
    assert diff < 1e-5


def test_fp8_fp4_masked_vs_oracle():
    g, max_m, n, k = 4, 256, 256, 512
    rng = np.random.default_rng(3)
    masked = rng.integers(96, 161, size=g).astype(np.int32)
    a = gen.randn_bf16((g, max_m, k), 51)
    b = gen.randn_bf16((g, n, k), 52)
    qa = np.empty((g, max_m, k), np.uint8)
    sfa = np.empty((g, max_m, k // 128), np.float32)
    qb = np.empty((g, n, k // 2), np.uint8)
    sfb = np.empty((g, n, k // 32), np.float32)
    for i in range(g):
        qa[i], sfa[i] = oquant.per_token_cast_to_fp8(a[i], use_ue8m0=True)
        qb[i], sfb[i] = oquant.per_token_cast_to_fp4(b[i], use_ue8m0=True, gran_k=32)
    a_deq = np.stack([oquant.dequant_per_token(qa[i], sfa[i]) for i in range(g)])
    b_deq = np.stack([oquant.dequant_fp4(qb[i], sfb[i], 32) for i in range(g)])
    ref, valid = ogemm.gemm_masked(a_deq, b_deq, masked)
    d = sentinel_bf16((g, max_m, n))
    deep_gemm.m_grouped_fp8_fp4_gemm_nt_masked((e4m3(qa), f32(sfa)), (gen.to_dev(qb, torch.int8), f32(sfb)), d,
                                               gen.to_dev(masked), 128, recipe_a=(1, 128), recipe_b=(1, 32))
    out = d.float().cpu().numpy()
    diff, _ = report('fp8xfp4 masked', out[valid], ref[valid])
    assert diff < 1e-5
    assert bool((d.view(torch.int16)[torch.from_numpy(~valid).to(DEV)] == SENTINEL).all())


def _pad_packed_k(sf, padding=4):
    """Packed MN-major SF words with a K pitch padding words longer than the aligned
    MN, the padding poisoned with -1 (UE8M0 NaN bytes): the reference's
    add_sf_k_padding (tests/utils.py:41-50), which exposes reads that assume a
    compact pitch."""
    mn = sf.size(-2)
    pitch = (mn + 3) // 4 * 4 + padding
    storage = sf.new_full((sf.numel() // mn, pitch), -1)
    return storage.as_strided(sf.shape, (1, pitch)).copy_(sf)


@pytest.mark.parametrize('m,n,k', [(256, 384, 1024), (300, 520, 640)])
def test_ue8m0_packed_sf_k_pitch(m, n, k):
    """Packed SFs with a padded K pitch give the same bits on both UE8M0 kernels
    (the reference's 'packed SF K-stride' check, tests/test_fp8_fp4.py:86-97)."""
    qa, sfa, _ = _ue8m0_quant(gen.randn_bf16((m, k), 71), False, 128)
    qb, sfb, _ = _ue8m0_quant(gen.randn_bf16((n, k), 72), True, 32)
    a = (e4m3(qa), _packed(sfa))
    b = (gen.to_dev(qb, torch.int8), _packed(sfb))
    a_p = (a[0], _pad_packed_k(a[1]))
    b_p = (b[0], _pad_packed_k(b[1]))
    assert a_p[1].stride(-1) > a[1].stride(-1)

    def call(x, y):
        d = torch.empty((m, n), dtype=torch.bfloat16, device=DEV)
        deep_gemm.fp8_fp4_gemm_nt(x, y, d, recipe_a=(1, 128), recipe_b=(1, 32))
        torch.cuda.synchronize()
        return d

    (c0, c1), _ = _run_both_kernels(lambda: call(a, b))
    (p0, p1), _ = _run_both_kernels(lambda: call(a_p, b_p))
    assert torch.equal(c0.view(torch.int16), p0.view(torch.int16))
    assert torch.equal(c1.view(torch.int16), p1.view(torch.int16))


def test_fp4_equals_converted_fp8():
    """E2M1 operands and their exact E4M3 conversion (same scales) give the same GEMM
    up to rounding (reference tests/test_fp8_fp4.py:98-103, whose bar is 1e-14 for
    NVIDIA's UMMA). The gfx950 matrix core sums E2M1 and E4M3 operands in different
    internal orders, so some FP32 results differ in their last bits and a few BF16
    outputs round the other way: measured calc_diff 1.1e-11 at this shape (13 of
    131072 outputs). The bar here is 1e-9, at most 1% of the outputs may differ,
    and no difference may exceed half a BF16 step at the output's scale."""
    from oracle import fp8 as ofp8
    m, n, k = 256, 512, 1024
    qa, sfa, _ = _ue8m0_quant(gen.randn_bf16((m, k), 81), False, 128)
    qb, sfb, _ = _ue8m0_quant(gen.randn_bf16((n, k), 82), True, 32)
    qb8 = ofp8.e4m3_encode(ofp8.e2m1_decode(ofp8.e2m1_unpack(qb)))
    assert np.array_equal(ofp8.e4m3_decode(qb8), ofp8.e2m1_decode(ofp8.e2m1_unpack(qb)))   # exact
    a = (e4m3(qa), _packed(sfa))
    outs = []
    for bq in (gen.to_dev(qb, torch.int8), e4m3(qb8)):
        d = torch.empty((m, n), dtype=torch.bfloat16, device=DEV)
        deep_gemm.fp8_fp4_gemm_nt(a, (bq, _packed(sfb)), d, recipe_a=(1, 128), recipe_b=(1, 32))
        torch.cuda.synchronize()
        outs.append(d.float().cpu().numpy())
    diff = ogemm.calc_diff(outs[0], outs[1])
    neq = outs[0] != outs[1]
    worst = np.abs(outs[0] - outs[1]).max()
    scale = np.abs(outs[0]).max()
    print(f'fp4 vs converted fp8 calc_diff={diff:.3e}, {neq.sum()} of {neq.size} outputs differ, '
          f'max difference {worst:.3e} (output scale {scale:.3e})', flush=True)
    assert diff < 1e-9
    assert neq.mean() < 0.01
    assert worst <= 2 ** -9 * scale


def _table_layout(case):
    """(m_indices, groups) of a contiguous layout that exercises the block table."""
    def seg(*parts):   # (expert, rows, blocks)
        out = []
        for e, r, b in parts:
            out += [e] * r + [-1] * (b * 128 - r)
        return np.array(out, np.int32)
    if case == 'odd_even_runs':   # runs of 1, 2, 3, 4 and 5 blocks, an expert without rows, one in two runs
        return seg((0, 100, 1), (2, 256, 2), (3, 300, 3), (0, 512, 4), (4, 600, 5), (5, 1, 1)), 6
    if case == 'padding_blocks':   # blocks without a row inside and after the segments
        return seg((0, 130, 2), (1, 0, 1), (1, 128, 1), (1, 0, 3), (2, 200, 4)), 3
    if case == 'first_row_padding':   # a block's expert is max(0, its first row's id)
        x = seg((0, 128, 1), (1, 256, 2), (2, 128, 1))
        x[128:140] = -1
        return x, 3
    if case == 'ids_past_last':
        return seg((0, 128, 1), (7, 256, 2), (1, 90, 1)), 2
    if case == 'all_padding':
        return seg((0, 0, 5)), 2
    if case == 'ragged_end':   # the last block is cut
        return seg((0, 256, 2), (1, 256, 2), (1, 128, 1))[:-55], 2
    assert case == 'two_launches'   # more 128-row blocks than one table holds
    return np.concatenate([np.full(128 * 4095, 0, np.int32), np.full(128 * 3, 1, np.int32)]), 2


@pytest.mark.parametrize('case', ['odd_even_runs', 'padding_blocks', 'first_row_padding', 'ids_past_last', 'all_padding',
                                  'ragged_end', 'two_launches'])
@pytest.mark.parametrize('shift', [0, 1])
def test_contiguous_block_table(case, shift):
    """The persistent contiguous walk over its block table (variant 4) equals one
    workgroup per 128-row tile bit for bit and leaves the same rows alone, also with
    m_indices 4 bytes off a 16-byte boundary, and with fewer CUs than tiles."""
    idx, g = _table_layout(case)
    m, n, k = len(idx), 256 if case == 'two_launches' else 520, 128 if case == 'two_launches' else 256
    print(f'block table {case} shift={shift} m={m}', flush=True)
    dg = torch.Generator(device=DEV).manual_seed(5)
    a = deep_gemm.per_token_cast_to_fp8(torch.randn((m, k), generator=dg, device=DEV).bfloat16(), use_ue8m0=False)
    w = [deep_gemm.per_block_cast_to_fp8(torch.randn((n, k), generator=dg, device=DEV).bfloat16(), use_ue8m0=False)
         for _ in range(g)]
    b = (torch.stack([q.view(torch.uint8) for q, _ in w]).view(torch.float8_e4m3fn), torch.stack([s for _, s in w]))
    gl = torch.zeros(m + shift, dtype=torch.int32, device=DEV)[shift:]
    gl.copy_(torch.from_numpy(idx))
    outs = []
    for v, bm, bn, cus in ((2, 128, 128, 0), (4, 256, 256, 0), (4, 256, 256, 3)):
        before = deep_gemm.get_num_sms()
        deep_gemm.set_tile_override(bm, bn, variant=v)
        if cus:
            deep_gemm.set_num_sms(cus)
        try:
            d = sentinel_bf16((m, n))
            deep_gemm.m_grouped_fp8_gemm_nt_contiguous(a, b, d, gl)
        finally:
            deep_gemm.set_tile_override(0, 0)
            deep_gemm.set_num_sms(before)
        outs.append(d.view(torch.int16))
    torch.cuda.synchronize()
    assert torch.equal(outs[1], outs[0]) and torch.equal(outs[2], outs[0])
    assert bool((outs[1][gl < 0] == SENTINEL).all())
    if case != 'all_padding':
        rows = np.nonzero(idx >= 0)[0][[0, -1]]
        e = np.minimum(np.maximum(idx[rows // 128 * 128], 0), g - 1)
        for r, ei in zip(rows, e):
            ref = ogemm.gemm_nt(oquant.dequant_per_token(a[0][r:r + 1].view(torch.uint8).cpu().numpy(),
                                                         a[1][r:r + 1].cpu().numpy()),
                                oquant.dequant_per_block(b[0][ei].view(torch.uint8).cpu().numpy(), b[1][ei].cpu().numpy()))
            assert ogemm.calc_diff(outs[1][r:r + 1].view(torch.bfloat16).float().cpu().numpy(), ref) < 1e-3


@pytest.mark.parametrize('m,n,k', [(1, 32, 128), (33, 72, 896), (64, 2112, 1152), (100, 264, 7168), (130, 520, 128 * 9)])
@pytest.mark.parametrize('b_fp4,gka,gkb', [(True, 128, 32), (True, 32, 32), (False, 128, 128), (False, 32, 128)])
def test_ue8m0_tiny_m(m, n, k, b_fp4, gka, gkb):
    """Every workgroup shape of the UE8M0 tiny-M kernel (ragged rows and columns, fewer K
    blocks than waves, uneven shares of them) against the FP64 oracle: one BF16 ulp plus
    2^-15 sum |a b|; shapes agree bit for bit (an output's K split does not depend on
    them), reruns too, and alpha scales the sum before the rounding."""
    a_np, b_np = gen.randn_bf16((m, k), m + k), gen.randn_bf16((n, k), n)
    qa, sfa = oquant.per_token_cast_to_fp8(a_np, use_ue8m0=True, gran_k=gka)
    if b_fp4:
        qb, sfb = oquant.per_token_cast_to_fp4(b_np, use_ue8m0=True, gran_k=gkb)
        b_deq = oquant.dequant_fp4(qb, sfb, gkb)
    else:
        qb, sfb = oquant.per_token_cast_to_fp8(b_np, use_ue8m0=True, gran_k=gkb)
        b_deq = oquant.dequant_per_token(qb, sfb, gran_k=gkb)
    a_deq = oquant.dequant_per_token(qa, sfa, gran_k=gka)
    ref = ogemm.gemm_nt(a_deq, b_deq)
    tol = np.abs(ref) * 2.0 ** -8 + 2.0 ** -15 * ogemm.gemm_nt(np.abs(a_deq), np.abs(b_deq))
    a = (e4m3(qa), deep_gemm.get_mn_major_tma_aligned_packed_ue8m0_tensor(f32(sfa)))
    b = (gen.to_dev(qb, torch.int8 if b_fp4 else torch.float8_e4m3fn),
         deep_gemm.get_mn_major_tma_aligned_packed_ue8m0_tensor(f32(sfb)))
    outs = []
    for rows in (32, 64):
        for cols in (32, 64):
            for _ in range(2):
                d = sentinel_bf16((m, n))
                deep_gemm.set_tile_override(rows, cols, variant=11)
                try:
                    deep_gemm.fp8_fp4_gemm_nt(a, b, d, recipe_a=(1, gka), recipe_b=(1, gkb))
                finally:
                    deep_gemm.set_tile_override(0, 0)
                assert f'tinym v11 kind=normal block_m={rows} block_n={cols}' in deep_gemm.get_last_config()
                outs.append(d)
    torch.cuda.synchronize()
    assert np.all(np.abs(outs[0].float().cpu().numpy() - ref) <= tol)
    for o in outs[1:]:
        assert torch.equal(o.view(torch.int16), outs[0].view(torch.int16))
    d = sentinel_bf16((m, n))
    deep_gemm.set_tile_override(32, 32, variant=11)
    try:
        deep_gemm.fp8_fp4_gemm_nt(a, b, d, recipe_a=(1, gka), recipe_b=(1, gkb), alpha=0.5)
    finally:
        deep_gemm.set_tile_override(0, 0)
    assert torch.equal(d.float(), (outs[0].float() * 0.5).bfloat16().float())   # (a power of two: exact)


@pytest.mark.parametrize('m,n,k', [
    (1, 8, 128),           # one row, a short tile and one block: the odd group has none
    (128, 128, 128),
    (129, 136, 256),       # a row and eight columns past a tile, a block per group
    (100, 200, 384),       # the odd group's last block is missing
    (257, 264, 1024),      # scales four blocks at a time where K-major
    (1100, 104, 1152),     # more m-blocks than a raster group; an odd number of blocks
    (517, 384, 7168),
])
@pytest.mark.parametrize('row_major_sfa', [False, True])
def test_dense_k_split_groups(m, n, k, row_major_sfa):
    """Even and odd K blocks on two wave groups, against the FP64 oracle: one BF16 ulp plus
    2^-15 sum |a b|; what lies past K in memory, NaN included, stays out of the sums."""
    a_np, b_np = gen.randn_bf16((m, k), m + k), gen.randn_bf16((n, k), n)
    qa, sfa = oquant.per_token_cast_to_fp8(a_np, use_ue8m0=False, gran_k=128)
    qb, sfb = oquant.per_block_cast_to_fp8(b_np, use_ue8m0=False)
    a_deq, b_deq = oquant.dequant_per_token(qa, sfa, gran_k=128), oquant.dequant_per_block(qb, sfb)
    ref = ogemm.gemm_nt(a_deq, b_deq)
    tol = np.abs(ref) * 2.0 ** -8 + 2.0 ** -15 * ogemm.gemm_nt(np.abs(a_deq), np.abs(b_deq))
    sf = f32(sfa) if row_major_sfa else deep_gemm.get_mn_major_tma_aligned_tensor(f32(sfa))
    outs = []
    for pad in (0, 128):   # rows of K bytes, and rows followed by NaN
        a, b = [torch.full((r, k + pad), 0x7F, dtype=torch.uint8, device='cuda').view(torch.float8_e4m3fn) for r in (m, n)]
        a.view(torch.uint8)[:, :k] = e4m3(qa).view(torch.uint8)
        b.view(torch.uint8)[:, :k] = e4m3(qb).view(torch.uint8)
        d = sentinel_bf16((m, n))
        deep_gemm.set_tile_override(128, 128, variant=12)
        try:
            deep_gemm.fp8_gemm_nt((a[:, :k], sf), (b[:, :k], f32(sfb)), d)
        finally:
            deep_gemm.set_tile_override(0, 0)
        assert 'v12 kind=normal block_m=128 block_n=128' in deep_gemm.get_last_config()
        outs.append(d)
    torch.cuda.synchronize()
    assert np.all(np.abs(outs[0].float().cpu().numpy() - ref) <= tol)
    assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))
