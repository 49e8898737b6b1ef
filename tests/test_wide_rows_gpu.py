"""The producers and the out consumer on rows wider than 4096 (four waves per row; the qkv producer up to 8 rows per CU):
the oracle's bits at the edges of the forms -- the narrowest row, whole and partial last waves, the row counts on both
sides of the qkv producer's limit -- and on rows whose fp32 variance depends on the order of the summation, which the four
waves continue from one to the next."""
import shutil

import pytest
import torch

from _util import assert_quant_equal, bits16
from h3_tp2_amd import _lib, ops
from oracle import oracle as O
from test_producers_gpu import EPS, _nan_aware_equal, _order_rows, _tables, mod_inputs

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def _run(cuda, form, x, idx, H, ph=False):
    M = x.shape[0]
    res, w, sh, sc, gt, _ = mod_inputs(M, H, seed=H + 7)
    gd, shd, scd = _tables(cuda, gt, sh, sc)
    i = idx.to(cuda)
    if form == "rms":
        h = torch.full((M, H), float("nan"), dtype=BF16, device=cuda)
        q, s = ops.rms_quant(x.to(cuda), w.to(cuda), shd, scd, i, EPS, h)
        torch.cuda.synchronize()
        h_ref, q_ref, s_ref = O.rms_quant(bits16(x), bits16(w), bits16(sh), bits16(sc), idx.numpy(), EPS)
        _nan_aware_equal(bits16(h), h_ref, "h")
    else:
        br = torch.zeros(M, H, dtype=BF16)                # the branch is zero: u is the residual, the order rows as given
        if form == "gate":
            u, q, s = ops.gate_rms_quant(x.to(cuda), gd, br.to(cuda), w.to(cuda), shd, scd, i, EPS)
        else:
            sa, sb = torch.full((M,), 0.5, device=cuda), torch.full((H,), 0.25, device=cuda)
            u, q, s = ops.scale_gate_rms_quant(torch.zeros(M, H, device=cuda), sa, sb, None, x.to(cuda), gd, w.to(cuda),
                                               shd, scd, i, EPS, quant=True, modulated=False)
        torch.cuda.synchronize()
        u_ref, _, q_ref, s_ref = O.gate_rms_quant(bits16(x), bits16(gt), bits16(br), bits16(w), bits16(sh), bits16(sc),
                                                  idx.numpy(), EPS)
        _nan_aware_equal(bits16(u), u_ref, "residual_out")
    assert_quant_equal(q, s, q_ref, s_ref)


@pytest.mark.parametrize("form", ["rms", "gate", "out"])
@pytest.mark.parametrize("H", [4608, 5632, 6144, 8192])
def test_order_sensitive_sums(cuda, form, H):
    x, idx = _order_rows(H)
    _run(cuda, form, x, idx, H)


def test_form_rule_before_set_up(cuda, tmp_path):
    """The producers need no h3fp8_init: a library that has run none (a copy has state of its own) counts the device's
    compute units all the same, so it takes the same form, and gives the same bits."""
    lib = _lib.load(shutil.copy(_lib.LIB_PATH, tmp_path / "libh3fp8.so"))
    assert lib["_ZN6h3host8cu_countEv"]() == torch.cuda.get_device_properties(cuda).multi_processor_count
    M, H = 100, 5376
    x, w, sh, sc, gt, _ = mod_inputs(M, H, seed=5)
    _, shd, scd = _tables(cuda, gt, sh, sc)
    x, w, idx = x.to(cuda), w.to(cuda), torch.arange(M, device=cuda) % 3
    q, s = torch.empty((M, H), device=cuda, dtype=torch.float8_e4m3fn), torch.empty((M, 1), device=cuda)
    rc = lib.h3fp8_rms_quant(x.data_ptr(), H, w.data_ptr(), shd.data_ptr(), shd.stride(0), scd.data_ptr(), scd.stride(0), 3,
                             idx.data_ptr(), 1, 8, M, H, EPS, q.data_ptr(), H, s.data_ptr(), None, 0,
                             torch.cuda.current_stream().cuda_stream)
    assert rc == 0, lib.h3fp8_last_error()
    q_ref, s_ref = ops.rms_quant(x, w, shd, scd, idx, EPS)
    torch.cuda.synchronize()
    assert torch.equal(q.view(torch.uint8), q_ref.view(torch.uint8)) and torch.equal(s, s_ref)


@pytest.mark.parametrize("form,M,H", [(f, M, H) for f in ("rms", "gate", "out")
                                      for M, H in ((5, 4104), (3, 6136), (2, 6152), (33, 8184), (1, 8192))]
                         + [("rms", 2048, 4104), ("rms", 2049, 4104)])
def test_edges(cuda, form, M, H):
    g = torch.Generator().manual_seed(M + H)
    x = (torch.randn(M, H, generator=g) * torch.exp(torch.randn(M, 1, generator=g) * 2)).to(BF16)
    x[M // 2] = 0
    if M > 2:
        x[0, H - 1] = float("inf")
        x[1, H // 2] = float("nan")
    _run(cuda, form, x, torch.randint(0, 3, (M,), generator=g), H)


def test_more_rows_than_a_grid_dimension_takes(cuda):
    """2^20 + 5 rows: the launch's second dimension (one dimension of one workgroup per row ends below 2^24).  The rows
    repeat with a period, in place, with the branch read from the residual's own rows."""
    period, M, H = 4099, (1 << 20) + 5, 4104
    tile, w, sh, sc, gt, _ = mod_inputs(period, H, seed=11)
    gd, shd, scd = _tables(cuda, gt, sh, sc)
    tile, w = tile.to(cuda), w.to(cuda)
    rows = torch.arange(M, device=cuda) % period
    idx = rows % 3
    u_ref, q_ref, s_ref = ops.gate_rms_quant(tile, gd, tile, w, shd, scd, idx[:period], EPS)
    x = tile[rows]
    q, s = torch.empty((M, H), device=cuda, dtype=torch.float8_e4m3fn), torch.empty((M, 1), device=cuda)
    _lib.call("h3fp8_gate_rms_quant", x.data_ptr(), H, gd.data_ptr(), gd.stride(0), x.data_ptr(), H, w.data_ptr(),
              shd.data_ptr(), shd.stride(0), scd.data_ptr(), scd.stride(0), 3, idx.data_ptr(), 1, 8, M, H, EPS,
              x.data_ptr(), H, q.data_ptr(), H, s.data_ptr(), None, 0, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    for r0 in range(0, M, 65536):
        r = rows[r0:r0 + 65536]
        assert torch.equal(x[r0:r0 + 65536].view(torch.int16), u_ref[r].view(torch.int16))
        assert torch.equal(q[r0:r0 + 65536].view(torch.uint8), q_ref.view(torch.uint8)[r])
        assert torch.equal(s[r0:r0 + 65536].view(torch.int32), s_ref[r].view(torch.int32))
    del x, q, s
    torch.cuda.empty_cache()
