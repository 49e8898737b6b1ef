"""The producers and the out consumer on rows wider than 4096 (four waves per row; the qkv producer up to 8 rows per CU):
the oracle's bits at the edges of the forms -- the narrowest row, whole and partial last waves, the row counts on both
sides of the qkv producer's limit -- and on rows whose fp32 variance depends on the order of the summation, which the four
waves continue from one to the next."""
import pytest
import torch

from _util import assert_quant_equal, bits16
from oracle import oracle as O
from test_producers_gpu import EPS, _nan_aware_equal, _order_rows, _tables, mod_inputs

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def _run(cuda, form, x, idx, H, ph=False):
    from h3_tp2_amd import ops
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
