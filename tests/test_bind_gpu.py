"""The native half of the Python binding (deep_gemm._dgbind): the same errors as the
described tensors of the ctypes half give, tensors of every rank and stride, and
allocation of the split-K workspace on the caller's stream."""
import pytest
import torch

import deep_gemm
from deep_gemm import _ffi

pytestmark = pytest.mark.gpu
DEV = 'cuda:0'


def _dense(m, n, k):
    a = deep_gemm.per_token_cast_to_fp8(torch.randn((m, k), device=DEV).bfloat16(), use_ue8m0=False)
    b = deep_gemm.per_block_cast_to_fp8(torch.randn((n, k), device=DEV).bfloat16(), use_ue8m0=False)
    return a, b, torch.empty((m, n), dtype=torch.bfloat16, device=DEV)


def test_errors():
    a, b, d = _dense(16, 256, 512)
    with pytest.raises(TypeError, match='torch.Tensor'):
        deep_gemm.fp8_gemm_nt((a[0], None), b, d)
    with pytest.raises(TypeError, match='torch.Tensor'):
        deep_gemm.m_grouped_fp8_gemm_nt_contiguous(a, (b[0][None], b[1][None]), d, None)
    with pytest.raises(RuntimeError, match='unsupported dtype'):
        deep_gemm.fp8_gemm_nt((a[0], a[1].double()), b, d)
    with pytest.raises(RuntimeError, match='rank > 4'):
        deep_gemm.fp8_gemm_nt(a, b, d[None, None, None])
    with pytest.raises(RuntimeError, match='Assertion'):
        deep_gemm.fp8_gemm_nt((a[0].cpu(), a[1]), b, d)
    with pytest.raises(TypeError):
        _ffi.bind.gemm_nt(a[0])
    deep_gemm.fp8_gemm_nt(a, b, d)   # and the binding goes on working


@pytest.mark.parametrize('m,n,k', [(1, 256, 512), (64, 2112, 7168)])
def test_matches_ctypes_on_a_side_stream(m, n, k):
    """The bits of the ctypes call, launched on the current (side) stream, for a call
    without and one with a workspace."""
    a, b, d = _dense(m, n, k)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        outs = []
        for _ in range(20):   # (workspaces go back to the side stream's pool between the calls)
            out = torch.empty_like(d)
            deep_gemm.fp8_gemm_nt(a, b, out)
            outs.append(out)
    side.synchronize()
    desc = [_ffi.describe(t) for t in (a[0], a[1], b[0], b[1], d)]
    ws_bytes = _ffi.lib.dg_fp8_gemm_nt_workspace_size(m, n, k)
    args = [_ffi.ref(x) for x in desc] + [None, None, 0, None]
    if ws_bytes > 0:
        ws = torch.empty(ws_bytes, dtype=torch.uint8, device=DEV)
        _ffi.check(_ffi.lib.dg_fp8_fp4_gemm_nt_ws(*args, _ffi.ref(_ffi.describe(ws)), _ffi.stream_of(d)))
    else:
        _ffi.check(_ffi.lib.dg_fp8_fp4_gemm_nt(*args, _ffi.stream_of(d)))
    torch.cuda.synchronize()
    for out in outs:
        assert torch.equal(out.view(torch.int16), d.view(torch.int16))
