"""The GEMM + quant entries around the width up to which the quant reduces the row maxima itself (16 384 columns; wider rows
take them from the GEMM's epilogue): codes and scales equal kernel 1's on the entry's own bf16 rows, and the workspace
receives the maxima, on either side; a NaN row keeps its NaN scale."""
import pytest
import torch

from _util import serving_like

pytestmark = pytest.mark.gpu
E4M3 = torch.float8_e4m3fn


@pytest.mark.parametrize("M,N,K", [(5, 16384, 256), (5, 16400, 256), (300, 1040, 384)])
@pytest.mark.parametrize("swiglu", [False, True])
def test_quant_behind_gemm(cuda, M, N, K, swiglu):
    from h3_tp2_amd import _lib, ops
    a, w, sa, sb = serving_like(M, 2 * N if swiglu else N, K, seed=N, device=cuda)
    sa = sa.clone()
    sa[1] = float("nan")
    y = torch.empty((M, N), device=cuda, dtype=torch.bfloat16)
    q, s = torch.empty((M, N), device=cuda, dtype=E4M3), torch.empty((M, 1), device=cuda)
    am = torch.full((M,), -1.0, device=cuda)
    st = torch.cuda.current_stream().cuda_stream
    head = [a.data_ptr(), K, w.data_ptr(), K, sa.data_ptr(), 1, sb.data_ptr(), 1, None]
    if swiglu:
        _lib.call("h3fp8_gemm_swiglu_quant", *head, M, N, K, y.data_ptr(), am.data_ptr(), q.data_ptr(), N, s.data_ptr(), st)
    else:
        _lib.call("h3fp8_gemm_quant", *head, y.data_ptr(), N, M, N, K, am.data_ptr(), q.data_ptr(), N, s.data_ptr(), st)
    q_ref, s_ref = ops.quant_rows(y)
    torch.cuda.synchronize()
    rows = torch.arange(M, device=cuda) != 1
    assert torch.equal(q.view(torch.uint8)[rows], q_ref.view(torch.uint8)[rows])
    assert torch.equal(s.view(-1)[rows], s_ref.view(-1)[rows]) and bool(s[1].isnan().all()) and bool(am[1].isnan())
    assert torch.equal(am[rows], y.float().abs().amax(dim=1)[rows])


@pytest.mark.parametrize("swiglu", [False, True])
def test_workspace_that_is_the_scale_array(cuda, swiglu):
    """One [M] array as workspace and scale: the scales remain (the maxima are only passed through)."""
    from h3_tp2_amd import _lib, ops
    M, N, K = 300, 1040, 256
    a, w, sa, sb = serving_like(M, 2 * N if swiglu else N, K, seed=7, device=cuda)
    y = torch.empty((M, N), device=cuda, dtype=torch.bfloat16)
    q, s = torch.empty((M, N), device=cuda, dtype=E4M3), torch.empty((M, 1), device=cuda)
    st = torch.cuda.current_stream().cuda_stream
    head = [a.data_ptr(), K, w.data_ptr(), K, sa.data_ptr(), 1, sb.data_ptr(), 1, None]
    if swiglu:
        _lib.call("h3fp8_gemm_swiglu_quant", *head, M, N, K, y.data_ptr(), s.data_ptr(), q.data_ptr(), N, s.data_ptr(), st)
    else:
        _lib.call("h3fp8_gemm_quant", *head, y.data_ptr(), N, M, N, K, s.data_ptr(), q.data_ptr(), N, s.data_ptr(), st)
    q_ref, s_ref = ops.quant_rows(y)
    torch.cuda.synchronize()
    assert torch.equal(s, s_ref) and torch.equal(q.view(torch.uint8), q_ref.view(torch.uint8))
