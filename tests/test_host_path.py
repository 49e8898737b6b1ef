"""The native host path of the common calls (csrc/host.cpp) against the Python path of the same functions: the same
outputs for every form it takes, and every other form left to the Python path -- taken or refused with the same error."""
import os
import shutil
import subprocess
import sys

import pytest
import torch

from _util import int_operands
from h3_tp2_amd import _lib, fp8_gemm, ops

E4M3 = torch.float8_e4m3fn
BF16 = torch.bfloat16


class Sub(torch.Tensor):
    pass


def test_leaves_cpu_tensors_subclasses_and_other_arguments_to_python():
    h = _lib.host()
    assert h is not None, "the native host path is not built"
    x = torch.zeros(4, 64, dtype=BF16)
    a, s = torch.zeros(4, 64).to(E4M3), torch.ones(4)
    for bad in (x, None, 3, x.as_subclass(Sub)):
        assert h.quant_rows(bad) is None and h.silu_mul_quant(bad) is None
        assert h.gemm(bad, a, s, s, BF16, None) is None and h.scaled_mm(bad, a, s, s, BF16, None) is None
        assert h.gemm_quant(bad, a, s, s, None) is None and h.gemm_swiglu_quant(bad, a, s, s, None) is None
        assert h.rms_quant(bad, x, x, x, s, 1e-6) is None and h.gate_rms_quant(bad, x, x, x, x, x, s, 1e-6) is None
    for f in (h.quant_rows, h.gemm, h.scaled_mm, h.gemm_quant, h.gemm_swiglu_quant, h.rms_quant, h.gate_rms_quant):
        assert f() is None


# A package whose native part cannot be loaded, or belongs to another torch, imports and keeps the Python path.
@pytest.mark.parametrize("how", ["not a library", "another torch"])
def test_an_unloadable_native_part_leaves_the_python_path(tmp_path, how):
    src = os.path.dirname(_lib.__file__)
    pkg = tmp_path / "h3_tp2_amd"
    shutil.copytree(src, pkg, ignore=shutil.ignore_patterns("__pycache__", "*.so"))
    for f in os.listdir(src):
        if f.endswith(".so"):
            shutil.copy(os.path.join(src, f), pkg / f)
            if how == "not a library" and f.startswith("_host"):
                (pkg / f).write_bytes(b"no library")
    head = "import torch; torch.__version__ = '0.0'; " if how == "another torch" else ""
    code = head + ("import h3_tp2_amd.ops as o, h3_tp2_amd._lib as l; assert o.__file__.startswith(%r); "
                   "assert o._host is None; l.load(); print('imported')" % str(pkg))
    r = subprocess.run([sys.executable, "-c", code], env=dict(os.environ, PYTHONPATH=str(tmp_path)), capture_output=True,
                       text=True, timeout=300)
    assert r.returncode == 0 and "imported" in r.stdout, r.stderr
    assert "native host path does not load" in r.stderr


def _bits(out):
    out = out if isinstance(out, tuple) else (out,)
    return [(t.dtype, tuple(t.shape), t.stride(), t.contiguous().view(torch.uint8).cpu()) for t in out]


def _result(f):
    try:
        return "out", _bits(f())
    except Exception as e:  # noqa: BLE001
        return type(e), str(e)


def _both(monkeypatch, f):
    """f through the native path and through the Python path alone: the same outputs, or the same refusal."""
    got = _result(f)
    with monkeypatch.context() as m:
        m.setattr(ops, "_host", None)
        ref = _result(f)
    assert got[0] == ref[0], (got, ref)
    if got[0] == "out":
        assert [g[:3] for g in got[1]] == [r[:3] for r in ref[1]]
        assert all(torch.equal(g[3], r[3]) for g, r in zip(got[1], ref[1]))
    else:
        assert got[1] == ref[1]
    return got


@pytest.mark.gpu
def test_products_match_the_python_path(cuda, monkeypatch):
    stock = []
    mm = fp8_gemm.make_scaled_mm(lambda *args: stock.append(args) or args[0])
    monkeypatch.setattr(fp8_gemm, "_state", dict(fp8_gemm._state, fused=True, level="hip"))
    monkeypatch.setattr(fp8_gemm, "_routers", [])
    monkeypatch.setattr(fp8_gemm, "_stash_hooks", [])
    for M, N, K in ((1, 64, 128), (5, 96, 272), (130, 528, 1040)):
        a, w, sa, sb = int_operands(M, N, K, seed=M, device=cuda)
        bias = torch.randn(N, device=cuda).to(BF16)
        wide = torch.zeros(M, K + 64, device=cuda).to(E4M3)
        wide[:, :K] = a
        scales = [(sa, sb), (sa.view(M, 1), sb.view(1, N)), (sa[:1], sb), (sa, sb[:1].reshape(())), (sa[:1], sb[:1]),
                  (torch.stack((sa, sa), 1)[:, 0], torch.stack((sb, sb), 1)[:, :1]), (sa.double(), sb), (sa[:0], sb)]
        for s_a, s_b in scales:
            for b in (None, bias, bias.half(), bias[:-1], torch.stack((bias, bias), 1)[:, 0]):
                for dt in (BF16, torch.float16, torch.float32):
                    n = len(stock)
                    _both(monkeypatch, lambda: mm(a, w.t(), s_a, s_b, dt, b))
                    assert (len(stock) - n) % 2 == 0                  # both paths kept the stock op, or neither
                    _both(monkeypatch, lambda: ops.gemm(a, w, s_a, s_b, dt, b))
                _both(monkeypatch, lambda: ops.gemm_quant(a, w, s_a, s_b, b))
                _both(monkeypatch, lambda: ops.gemm_swiglu_quant(a, w, s_a, s_b, b))
        for x in (wide[:, :K], a[:0], a.t().contiguous().t(), a.cpu(), a.float(), a[0], a[:, :K - 8]):
            _both(monkeypatch, lambda: ops.gemm(x, w, sa, sb))
            _both(monkeypatch, lambda: ops.gemm_swiglu_quant(x, w, sa, sb))
            n = len(stock)
            if x.is_cuda:
                _both(monkeypatch, lambda: mm(x, w.t(), sa, sb, BF16))
                _both(monkeypatch, lambda: mm(x, w.t().contiguous(), sa, sb, BF16))
                assert (len(stock) - n) % 2 == 0
        assert _both(monkeypatch, lambda: ops.gemm(a, w, sa, sb))[0] == "out"
    # a size the C side refuses: the library's error through either path
    assert _both(monkeypatch, lambda: ops.gemm(*int_operands(4, 24, 40, 1, cuda)))[0] is _lib.H3Fp8Error


@pytest.mark.gpu
def test_quants_and_producers_match_the_python_path(cuda, monkeypatch):
    g = torch.Generator(device=cuda).manual_seed(3)
    for M, H in ((1, 64), (7, 1000), (300, 3072)):
        wide = torch.randn(M, 2 * H, generator=g, device=cuda).to(BF16)
        x = wide[:, :H].contiguous()
        for t in (x, wide, wide[:, :H], wide[:, ::2], x[:0], x.float(), x[0], x.t()):
            _both(monkeypatch, lambda: ops.quant_rows(t))
            _both(monkeypatch, lambda: ops.silu_mul_quant(t))
        ada = torch.randn(3, 6 * H, generator=g, device=cuda).to(BF16)
        w = torch.randn(H, generator=g, device=cuda).to(BF16)
        idx = torch.randint(0, 3, (M,), generator=g, device=cuda)
        sh, sc, ga = ada[:, :H], ada[:, H:2 * H], ada[:, 2 * H:3 * H]
        for i in (idx, idx.int(), idx.float(), torch.stack((idx, idx), 1)[:, 0], idx[:-1]):
            for weight, eps in ((w, 1e-6), (w.view(1, H), 1e-6), (w[:-1], 1e-6), (w, 1)):
                _both(monkeypatch, lambda: ops.rms_quant(x, weight, sh, sc, i, eps))
                _both(monkeypatch, lambda: ops.gate_rms_quant(x, ga, wide[:, H:], weight, sh, sc, i, eps))
        _both(monkeypatch, lambda: ops.rms_quant(x, w, sh[:, :-8], sc, idx, 1e-6))
        _both(monkeypatch, lambda: ops.gate_rms_quant(x, ga, x[:, :-8], w, sh, sc, idx, 1e-6))
        _both(monkeypatch, lambda: ops.gate_rms_quant(x, ga[:1], x, w, sh, sc, idx * 0, 1e-6))


def _operands(cuda, M=130, N=96, K=272):
    a, w, sa, sb = int_operands(M, N, K, seed=M, device=cuda)
    g = torch.Generator(device=cuda).manual_seed(9)
    x = torch.randn(M, K, generator=g, device=cuda).to(BF16)
    ada = torch.randn(3, 6 * K, generator=g, device=cuda).to(BF16)
    norm = torch.randn(K, generator=g, device=cuda).to(BF16)
    idx = torch.randint(0, 3, (M,), generator=g, device=cuda)
    bias = torch.randn(N, generator=g, device=cuda).to(BF16)
    return dict(a=a, w=w, sa=sa, sb=sb, x=x, gate=ada[:, 2 * K:3 * K], sh=ada[:, :K], sc=ada[:, K:2 * K], norm=norm, idx=idx,
                bias=bias, M=M, N=N, K=K)


@pytest.mark.gpu
def test_takes_the_plain_forms_itself(cuda, monkeypatch):
    """Called directly, each of the eight functions computes its plain forms (it does not decline them), with the bits of
    the Python path."""
    h = _lib.host()
    o = _operands(cuda)
    a, w, sa, sb, x, bias = (o[k] for k in ("a", "w", "sa", "sb", "x", "bias"))
    gate, sh, sc, norm, idx = (o[k] for k in ("gate", "sh", "sc", "norm", "idx"))
    M, K = o["M"], o["K"]
    wide = torch.cat((x, x), 1)
    a_wide = torch.zeros(M, K + 48, device=cuda).to(E4M3)
    a_wide[:, :K] = a
    mm = ops.scaled_mm_eligible
    cases = [("quant_rows", ops.quant_rows, [(x,), (wide[:, :K],), (x[:1],)]),
             ("gemm", ops.gemm, [(a, w, sa, sb, BF16, None), (a_wide[:, :K], w, sa.view(M, 1), sb.view(1, -1), BF16, bias),
                                 (a, w, sa[:1], sb[:1].reshape(()), torch.float16, bias.half()),
                                 (a, w, sa, sb, torch.float32, None), (a[:1], w, sa[:1], sb, BF16, None)]),
             ("scaled_mm", mm, [(a, w.t(), sa, sb, BF16, None), (a, w.t(), sa.view(M, 1), sb.view(1, -1), BF16, bias),
                                (a, w.t(), sa[:1], sb, torch.float16, bias.half())]),
             ("gemm_quant", ops.gemm_quant, [(a, w, sa, sb, None), (a_wide[:, :K], w, sa, sb[:1], bias)]),
             ("gemm_swiglu_quant", ops.gemm_swiglu_quant, [(a, w, sa, sb, None), (a, w, sa[:1], sb, bias)]),
             ("silu_mul_quant", ops.silu_mul_quant, [(x,), (wide[:, :K],)]),
             ("rms_quant", ops.rms_quant, [(x, norm, sh, sc, idx, 1e-6), (wide[:, :K], norm, sh, sc, idx.int(), 1e-6)]),
             ("gate_rms_quant", ops.gate_rms_quant, [(x, gate, wide[:, K:], norm, sh, sc, idx, 1e-6)])]
    monkeypatch.setattr(ops, "_host", None)                    # the functions of ops below: the Python path
    assert len(cases) == 8
    for name, python, forms in cases:
        for args in forms:
            got = getattr(h, name)(*args)
            assert got is not None, (name, [getattr(t, "shape", t) for t in args])
            ref = python(*args)
            got, ref = _bits(got), _bits(ref)
            assert [g[:3] for g in got] == [r[:3] for r in ref], name
            assert all(torch.equal(g[3], r[3]) for g, r in zip(got, ref)), name


@pytest.mark.gpu
def test_declines_what_python_checks(cuda):
    h = _lib.host()
    o = _operands(cuda)
    a, w, sa, sb, x, bias = (o[k] for k in ("a", "w", "sa", "sb", "x", "bias"))
    gate, sh, sc, norm, idx = (o[k] for k in ("gate", "sh", "sc", "norm", "idx"))
    strided = torch.stack((bias, bias), 1)[:, 0]
    for ops4 in ((a, w, sa.double(), sb), (a, w, sa, sb[:-1]), (a.float(), w, sa, sb), (a, w[:, :-16], sa, sb),
                 (a.t().contiguous().t(), w, sa, sb), (a.cpu(), w, sa, sb), (a, w.cpu(), sa, sb), (a[:0], w, sa[:0], sb)):
        assert h.gemm(*ops4, BF16, None) is None and h.gemm_quant(*ops4, None) is None
        assert h.gemm_swiglu_quant(*ops4, None) is None
        assert h.scaled_mm(ops4[0], ops4[1].t(), *ops4[2:], BF16, None) is None
    for b in (strided, bias.half(), bias[:-1], bias.view(1, -1), bias.cpu()):
        assert h.gemm(a, w, sa, sb, BF16, b) is None and h.scaled_mm(a, w.t(), sa, sb, BF16, b) is None
        assert h.gemm_quant(a, w, sa, sb, b) is None and h.gemm_swiglu_quant(a, w, sa, sb, b) is None
    assert h.gemm(a, w, sa, sb, torch.float32, bias) is None and h.gemm(a, w, sa, sb, torch.float64, None) is None
    assert h.scaled_mm(a, w.t(), sa[:1], sb[:1], BF16, None) is None         # per-tensor scales on both sides
    assert h.scaled_mm(a, w.t(), sa, sb, torch.float32, None) is None
    assert h.scaled_mm(a, w.t().contiguous(), sa, sb, BF16, None) is None
    assert h.gemm_swiglu_quant(a, w[:-1], sa, sb[:-1], None) is None         # an odd number of gate | up rows
    for t in (x.float(), x[0], x.t(), x[:, ::2], x[:0], x.cpu()):
        assert h.quant_rows(t) is None and h.silu_mul_quant(t) is None
    assert h.silu_mul_quant(x[:, :-4]) is None
    for args in ((x, norm.view(1, -1), sh, sc, idx, 1e-6), (x, norm, sh[:, :-8], sc, idx, 1e-6),
                 (x, norm, sh, sc.float(), idx, 1e-6), (x, norm, sh, sc, idx.float(), 1e-6), (x, norm, sh, sc, idx[:-1], 1e-6),
                 (x, norm, sh, sc, idx, 1)):
        assert h.rms_quant(*args) is None
        assert h.gate_rms_quant(args[0], gate, x, *args[1:]) is None
    assert h.gate_rms_quant(x, gate, x[:-1], norm, sh, sc, idx, 1e-6) is None


@pytest.mark.gpu
def test_runs_on_the_current_stream_and_under_capture(cuda):
    a, w, sa, sb = int_operands(40, 96, 256, seed=1, device=cuda)
    ref = ops.gemm(a, w, sa, sb)
    x = torch.randn(40, 256, device=cuda).to(BF16)
    q_ref, s_ref = ops.quant_rows(x)
    graph = torch.cuda.CUDAGraph()
    h = _lib.host()
    with torch.cuda.graph(graph):                              # the native functions themselves: None would not unpack
        y = h.gemm(a, w, sa, sb, BF16, None)
        q, s = h.quant_rows(x)
    for _ in range(3):
        y.zero_()
        s.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, ref) and torch.equal(s, s_ref) and torch.equal(q.view(torch.uint8), q_ref.view(torch.uint8))


@pytest.mark.gpu
def test_function_transforms_stay_on_the_python_path(cuda, monkeypatch):
    x = torch.randn(2, 4, 64, device=cuda).to(BF16)
    _both(monkeypatch, lambda: torch.func.vmap(ops.quant_rows)(x))
    _both(monkeypatch, lambda: torch.func.functionalize(ops.silu_mul_quant)(x[0]))
    _both(monkeypatch, lambda: ops.quant_rows(x[0].clone().requires_grad_()))
    with torch.inference_mode():
        _both(monkeypatch, lambda: ops.quant_rows(x[0]))
