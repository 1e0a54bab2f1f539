"""Operands and scales that are column slices of very wide buffers: the bits of the same
call on compact operands, where a tile's rows span more than 4 GB (the kernels load
through 32-bit lane offsets)."""
import pytest
import torch

import deep_gemm

pytestmark = pytest.mark.gpu
DEV = 'cuda:0'


def _wide(t, pitch):
    """t as a column slice of a buffer whose rows are `pitch` elements (not filled)."""
    if pitch <= t.shape[1]:
        return t
    raw = t.view(torch.uint8) if t.dtype == torch.float8_e4m3fn else t
    out = torch.empty((t.shape[0] - 1) * pitch + t.shape[1], dtype=raw.dtype, device=DEV).as_strided(t.shape, (pitch, 1))
    out.copy_(raw)
    return out.view(torch.float8_e4m3fn) if raw is not t else out


def _quant(m, n, k, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    a = deep_gemm.per_token_cast_to_fp8(torch.randn((m, k), generator=g, device=DEV).bfloat16(), use_ue8m0=False)
    b = deep_gemm.per_block_cast_to_fp8(torch.randn((n, k), generator=g, device=DEV).bfloat16(), use_ue8m0=False)
    return a, b


# 255 rows pass 2^32 bytes from a pitch of 16.85 MB, 127 rows from 33.8 MB and 7 rows from 614 MB.
@pytest.mark.parametrize('m,n,k,a_pitch,sf_pitch,b_pitch', [
    (256, 264, 1040, 17_000_000, 0, 0),        # K tail, A
    (256, 264, 1040, 0, 4_300_000, 0),         # its scales
    (72, 264, 1040, 0, 0, 17_000_000),         # B
    (256, 520, 2048, 17_000_000, 0, 0),        # whole K blocks
    (256, 520, 2048, 0, 4_300_000, 0),         # scale groups
    (130, 264, 2048, 34_000_000, 0, 0),
    (64, 264, 7168, 0, 17_100_000, 0),         # split K
    (9, 264, 1040, 614_000_000, 0, 0),         # wider than the pipelined kernel's offsets
    (9, 264, 1024, 614_000_000, 0, 0),
])
def test_dense(m, n, k, a_pitch, sf_pitch, b_pitch):
    (qa, sfa), (qb, sfb) = _quant(m, n, k, m + k)
    ref = torch.empty((m, n), dtype=torch.bfloat16, device=DEV)
    got = torch.empty_like(ref)
    print(f'wide pitch dense m={m} n={n} k={k} a={a_pitch} sf={sf_pitch} b={b_pitch}', flush=True)
    deep_gemm.set_tile_override(64, 64, variant=1)   # (64-bit addresses)
    try:
        deep_gemm.fp8_gemm_nt((qa, sfa), (qb, sfb), ref)
    finally:
        deep_gemm.set_tile_override(0, 0)
    a, sf, b = _wide(qa, a_pitch), _wide(sfa, sf_pitch), _wide(qb, b_pitch)
    for tile in (None, (256, 192), (256, 128), (128, 256), (128, 128)):
        wide = a_pitch > 600_000_000 or sf_pitch > 17_000_000
        deep_gemm.set_tile_override(*(tile or (0, 0)), variant=2 if tile else 0)
        try:
            got.zero_()
            if tile and wide:   # refused, not computed from other rows
                with pytest.raises(RuntimeError, match='Unsupported'):
                    deep_gemm.fp8_gemm_nt((a, sf), (b, sfb), got)
                continue
            deep_gemm.fp8_gemm_nt((a, sf), (b, sfb), got)
            cfg = deep_gemm.get_last_config()
        finally:
            deep_gemm.set_tile_override(0, 0)
        torch.cuda.synchronize()
        if tile is None and any(v in cfg for v in (' v8 ', ' v9 ', ' v10 ', ' v12 ')):   # sums in another order
            err = (got.float() - ref.float()).norm() / ref.float().norm()
            assert err < 2.0 ** -8, (cfg, err)
        else:
            assert torch.equal(got.view(torch.int16), ref.view(torch.int16)), cfg


@pytest.mark.parametrize('tile', [128, 256])
@pytest.mark.parametrize('a_pitch,sf_pitch', [(17_000_000, 0), (0, 4_300_000)])
def test_1d1d(tile, a_pitch, sf_pitch):
    m, n, k = 256, 264, 256
    g = torch.Generator(device=DEV).manual_seed(3)
    a, b = [deep_gemm.per_token_cast_to_fp8(torch.randn((r, k), generator=g, device=DEV).bfloat16(), use_ue8m0=False)
            for r in (m, n)]
    c = torch.randn((m, n), generator=g, device=DEV)
    outs = []
    print(f'wide pitch 1D1D tile={tile} a={a_pitch} sf={sf_pitch}', flush=True)
    for wide in (False, True):
        pair = [(_wide(q, a_pitch), _wide(sf, sf_pitch)) if wide else (q, sf) for q, sf in (a, b)]
        d = torch.empty_like(c)
        deep_gemm.set_tile_override(tile, tile, variant=7)
        try:
            deep_gemm.fp8_gemm_nt(*pair, d, c=c, recipe=(1, 1, 128))
        finally:
            deep_gemm.set_tile_override(0, 0)
        outs.append(d)
        torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1])


@pytest.mark.parametrize('k', [208, 256])
def test_contiguous_and_fused(k):
    """Grouped calls, and the fused SwiGLU launch, on a wide A (two segments, 256 rows)."""
    m, inter, e = 256, 128, 2
    g = torch.Generator(device=DEV).manual_seed(k)
    qa, sfa = deep_gemm.per_token_cast_to_fp8(torch.randn((m, k), generator=g, device=DEV).bfloat16(), use_ue8m0=False)
    w = [deep_gemm.per_block_cast_to_fp8(torch.randn((2 * inter, k), generator=g, device=DEV).bfloat16(), use_ue8m0=False)
         for _ in range(e)]
    b = (torch.stack([q.view(torch.uint8) for q, _ in w]).view(torch.float8_e4m3fn), torch.stack([s for _, s in w]))
    idx = (torch.arange(m, device=DEV) // 128).int()
    a = _wide(qa, 34_000_000)
    print(f'wide pitch contiguous k={k}', flush=True)
    plain, fused = [], []
    for op in (qa, a):
        d = torch.empty((m, 2 * inter), dtype=torch.bfloat16, device=DEV)
        deep_gemm.m_grouped_fp8_gemm_nt_contiguous((op, sfa), b, d, idx)
        plain.append(d.view(torch.int16))
        q = torch.empty((m, inter), dtype=torch.float8_e4m3fn, device=DEV)
        sf = torch.empty((m, inter // 128), device=DEV)
        deep_gemm.m_grouped_fp8_gemm_nt_contiguous_swiglu((op, sfa), b, (q, sf), idx)
        fused.append((q.view(torch.uint8), sf))
        torch.cuda.synchronize()
    assert torch.equal(plain[0], plain[1])
    assert torch.equal(fused[0][0], fused[1][0]) and torch.equal(fused[0][1], fused[1][1])


def test_ue8m0():
    """FP8 x FP8 with packed scales: the pipelined kernel's rows are 256 to a tile."""
    m, n, k = 256, 264, 1280
    g = torch.Generator(device=DEV).manual_seed(7)
    a, b = [deep_gemm.per_token_cast_to_fp8(torch.randn((r, k), generator=g, device=DEV).bfloat16(), use_ue8m0=True)
            for r in (m, n)]
    pack = deep_gemm.get_mn_major_tma_aligned_packed_ue8m0_tensor
    print('wide pitch ue8m0', flush=True)
    outs = []
    for q in (a[0], _wide(a[0], 17_000_000)):
        d = torch.empty((m, n), dtype=torch.float32, device=DEV)
        deep_gemm.fp8_fp4_gemm_nt((q, pack(a[1])), (b[0], pack(b[1])), d, recipe_a=(1, 128), recipe_b=(1, 128))
        outs.append(d)
        torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1])
