"""The smaller tiles of kernel 2 (one tile per workgroup; 32 x 64 ... 256 x 128 weight rows x token rows) and the last
rounds cut into them.

Each case's sizes take one form on 256 CUs (asserted from the library's own plan), with ragged edges in M and N, K tails
and one to five k-steps (the ring is deeper than the problem, or its parity differs).  Bits: equal to the grouped launch, which
always runs 256 x 256 tiles, on random operands, where the MFMA's inexact accumulation would expose any change of order;
integer operands are exact against the oracle, with sentinels around the output.
"""
import numpy as np
import pytest
import torch

from _util import bits16, f32, gemm_plan, int_operands, ref_gemm, serving_like
from oracle import oracle as O

pytestmark = pytest.mark.gpu

# the form (index of _util.FORMS), then M, N, K
WHOLE = [(0, 33, 16, 16), (0, 65, 528, 1040), (1, 260, 1840, 272), (2, 500, 2320, 400), (3, 700, 2320, 144),
         (4, 1000, 3008, 96), (5, 2040, 2992, 640), (6, 2300, 3312, 192), (6, 320, 21504, 256)]
# last rounds: the form of the tail, then M, N, K, and whether the full tiles leave the ragged rows to it: 264, 266, 286,
# 316 and 356 full tiles in all panels; 368 in the whole panels (391 in all) and 256 (272) with 4 rows past them
TAILS = [(0, 8300, 2032, 160, False), (1, 3400, 4800, 64, False), (3, 5600, 3200, 272, False),
         (4, 20200, 912, 128, False), (6, 22600, 1008, 400, False), (6, 4100, 5888, 272, True),
         (0, 4100, 4096, 400, "only")]


def _takes(form, M, N, K, tail, edge=False, swiglu=False):
    """The library runs these sizes as the case says (edge: the ragged rows go to the tail; "only": nothing else does)."""
    p = gemm_plan(M, N, K, swiglu, torch.cuda.get_device_properties(0).multi_processor_count)
    if not tail:
        return p["form"] == form
    return (p["form"] is None and p["full"] > 0 and p["tail"] == form and (p["panels"] * 256 < M) == bool(edge)
            and (p["rest"] == 0) == (edge == "only"))


CASES = [(*c, False, False) for c in WHOLE] + [(*c[:4], True, c[4]) for c in TAILS]


@pytest.mark.parametrize("form,M,N,K,tail,edge", CASES)
def test_form_equals_full_tiles(cuda, form, M, N, K, tail, edge):
    from h3_tp2_amd import ops
    assert _takes(form, M, N, K, tail, edge)
    a, w, sa, sb = serving_like(M, N, K, seed=M + K, device=cuda)
    y = ops.gemm(a, w, sa, sb)
    (ref,) = ops.grouped_gemm([(a, w, sa, sb)])
    torch.cuda.synchronize()
    assert torch.equal(y.view(torch.int16), ref.view(torch.int16))


@pytest.mark.parametrize("form,M,N,K,tail,edge", CASES)
def test_form_integer_exact_with_guards(cuda, form, M, N, K, tail, edge):
    from h3_tp2_amd import ops
    a, w, sa, sb = int_operands(M, N, K, seed=M + N, device=cuda)
    guard = 4096
    buf = torch.full((M * N + 2 * guard,), float("nan"), device=cuda, dtype=torch.bfloat16)
    buf[:guard] = 7.0
    buf[-guard:] = 7.0
    y = ops.gemm(a, w, sa, sb, out=buf[guard:guard + M * N].view(M, N))
    torch.cuda.synchronize()
    assert np.array_equal(bits16(y), ref_gemm(a, w, sa, sb))
    assert bool((buf[:guard] == 7.0).all()) and bool((buf[-guard:] == 7.0).all())


# one case of each form: fp16, bias, row maxima, scalar scales, strided output rows, the raw accumulator
@pytest.mark.parametrize("form,M,N,K,tail,edge", [c for c in CASES if c[1:3] not in ((33, 16), (320, 21504))])
def test_form_epilogues(cuda, form, M, N, K, tail, edge):
    from h3_tp2_amd import ops
    a, w, sa, sb = int_operands(M, N, K, seed=N + K, device=cuda)
    g = torch.Generator().manual_seed(N)
    for dt, with_bias in ((torch.bfloat16, True), (torch.float16, False), (torch.float16, True)):
        bias = (torch.randn(N, generator=g) * 0.3).to(dt).to(cuda) if with_bias else None
        am = torch.full((M,), -1.0, device=cuda)
        full = torch.full((M, N + 24), 3.0, device=cuda, dtype=dt)
        y = ops.gemm(a, w, sa[:1].reshape(()), sb, dt, bias, out=full[:, :N], row_amax=am)
        torch.cuda.synchronize()
        assert np.array_equal(bits16(y), ref_gemm(a, w, sa[:1].expand(M), sb, bias, dt == torch.float16))
        assert bool((full[:, N:] == 3.0).all())
        assert np.array_equal(f32(am), np.abs(f32(y)).max(axis=1))
    acc = ops.gemm(a, w, sa, sb, torch.float32)
    one = torch.ones(1, device=cuda)
    torch.cuda.synchronize()
    # |acc| <= 8 K, an integer: its bf16 rounding is the scaled output at unit scales
    assert np.array_equal(bits16(acc.to(torch.bfloat16)), ref_gemm(a, w, one.expand(M), one.expand(N)))


# operand rows with a stride past K, strided scales: the same bits as from contiguous ones
def _strided(a, w, sa, sb):
    wide = []
    for t in (a, w):
        v = torch.full((t.shape[0], t.shape[1] + 48), 3.0, device=t.device).to(t.dtype)
        v[:, :t.shape[1]] = t
        wide.append(v[:, :t.shape[1]])
    return (*wide, torch.stack((sa, sa * 3), 1)[:, 0], torch.stack((sb * 5, sb, sb * 7), 1)[:, 1])


@pytest.mark.parametrize("form,M,N,K,tail,edge", [c for c in CASES if c[1:3] not in ((33, 16), (320, 21504))])
def test_form_strides(cuda, form, M, N, K, tail, edge):
    from h3_tp2_amd import ops
    ops4 = int_operands(M, N, K, seed=M + N + K, device=cuda)
    a, w, sa, sb = _strided(*ops4)
    assert a.stride(0) > K and w.stride(0) > K and sa.stride(0) == 2 and sb.stride(0) == 3
    y = ops.gemm(a, w, sa, sb)
    torch.cuda.synchronize()
    assert np.array_equal(bits16(y), ref_gemm(*ops4))


# kernel 3's forms: the same tiles with gate and up rows in pairs (N = 2F)
SWIGLU = [(1, 1, 64, 16, False, False), (1, 40, 1008, 272, False, False), (3, 300, 2000, 400, False, False),
          (4, 600, 2000, 144, False, False), (5, 1000, 2320, 640, False, False), (6, 1250, 2992, 192, False, False),
          (1, 2000, 4208, 128, True, False), (3, 5600, 1648, 272, True, False), (4, 20200, 496, 96, True, False),
          (6, 22600, 496, 400, True, False), (6, 4100, 2944, 272, True, True), (1, 4100, 2048, 144, True, False),
          (1, 4100, 4096, 144, True, "only")]


@pytest.mark.parametrize("form,M,F,K,tail,edge", SWIGLU)
def test_swiglu_form_strides(cuda, form, M, F, K, tail, edge):
    from h3_tp2_amd import ops
    ops4 = serving_like(M, 2 * F, K, seed=M + F + K, device=cuda)
    h, ref = ops.gemm_swiglu(*_strided(*ops4)), ops.gemm_swiglu(*ops4)
    torch.cuda.synchronize()
    assert torch.equal(h.view(torch.int16), ref.view(torch.int16))


@pytest.mark.parametrize("form,M,F,K,tail,edge", SWIGLU)
@pytest.mark.parametrize("bias", [False, True])
def test_swiglu_form_equals_oracle_of_the_accumulator(cuda, form, M, F, K, tail, edge, bias):
    """h and the row maxima against the oracle's SwiGLU of the kernel's own fp32 accumulator, bit for bit; some rows'
    gates are zero or far outside the compact SiLU table (those blocks take the full table), the output has guards."""
    from h3_tp2_amd import ops
    assert _takes(form, M, F, K, tail, edge, True)
    a, w, sa, sb = serving_like(M, 2 * F, K, seed=M + F, device=cuda)
    sa = sa.clone()
    sa[5::37] = 0.0
    sa[11::41] *= 1e7
    b = (torch.randn(2 * F, generator=torch.Generator().manual_seed(F)) * 0.5).to(torch.bfloat16).to(cuda) if bias else None
    acc = ops.gemm(a, w, sa, sb, torch.float32)
    guard = 4096
    buf = torch.full((M * F + 2 * guard,), 7.0, device=cuda, dtype=torch.bfloat16)
    am = torch.full((M,), -1.0, device=cuda)
    h = ops.gemm_swiglu(a, w, sa, sb, b, row_amax=am, out=buf[guard:guard + M * F].view(M, F))
    torch.cuda.synchronize()
    ref = O.scale_swiglu(f32(acc), f32(sa), f32(sb), bits16(b) if bias else None)
    got = bits16(h)
    nan = (ref & 0x7FFF) > 0x7F80
    assert np.array_equal((got & 0x7FFF) > 0x7F80, nan) and np.array_equal(got[~nan], ref[~nan])
    assert bool((buf[:guard] == 7.0).all()) and bool((buf[-guard:] == 7.0).all())
    if not nan.any():
        assert torch.equal(am, h.float().abs().amax(dim=1))


# the small-M form's rings: 8 / 6 stages with at most 4 waves per CU (16 384 weight rows), 4 / 3 beyond; fewer k-steps
# than stages, as many, one more, odd counts and a K tail
@pytest.mark.parametrize("N", [528, 16384, 16400])
@pytest.mark.parametrize("M,K", [(1, 16), (8, 1024), (8, 1040), (9, 768), (32, 400), (17, 896), (5, 2192)])
def test_small_m_rings_equal_full_tiles(cuda, M, N, K):
    from h3_tp2_amd import ops
    a, w, sa, sb = serving_like(M, N, K, seed=M + N + K, device=cuda)
    y = ops.gemm(a, w, sa, sb)
    (ref,) = ops.grouped_gemm([(a, w, sa, sb)])
    torch.cuda.synchronize()
    assert torch.equal(y.view(torch.int16), ref.view(torch.int16))
