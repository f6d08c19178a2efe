"""The decode kernels for any cols (csrc/q8_gemv_any.hip): K from one block to 16384 that is no multiple
of 1024, at the edges of the wave classes (4, 8, 12, 16 waves), with the last wave from one unit to
full, against F64; a token's bits whatever the token count, a round's products as their own launches',
the epilogues, and an infinite scale in the block that dead lanes load."""
import ctypes as c

import numpy as np
import pytest

import synth
from parity import assert_parity
from test_gpu_tile import Case, kernels

pytestmark = pytest.mark.gpu
P = c.c_void_p

SHAPES = [(16, 32), (64, 96), (2048, 1056), (5136, 2784), (4096, 4064), (1888, 4128), (2048, 8160), (528, 8224), (1024, 12320), (512, 16352), (512, 12256),
          (2048, 5120), (256, 15360), (1024, 1088), (2048, 4352), (64, 16384 - 32), (32, 14336 + 896)]


def rms(x, nw, eps=1e-6):
    x = x.astype(np.float64)
    return (nw * x / np.sqrt(eps + (x * x).mean(axis=1, keepdims=True))).astype(np.float64)


@pytest.mark.parametrize("rows,cols", SHAPES)
def test_any_cols(rt, oracle, rows, cols):
    case = Case(rt, rows, cols, 4, rows + cols)
    try:
        got = {}
        for kind in ("product", "residual", "norm", "pair", "pair_norm", "round", "round_norm"):
            for t in (4, 3, 2, 1):
                case.nan()
                name = kernels(rt, lambda: case.run(kind, 0, t))[0]
                y, z = case.out()
                if t == 4:
                    got[kind] = y
                    print("any cols", rows, cols, kind, name, flush=True)
                assert np.array_equal(y[:t].view(np.uint32), got[kind][:t].view(np.uint32)), (kind, t)
                if kind.startswith("round"):
                    case.rt.lib.rt_gemm_dev(rt.R, P(case.w[1]), 16, cols, P(case.p["x"]), cols, t, P(case.z))
                    if kind == "round":
                        assert np.array_equal(case.out()[1][:t].view(np.uint32), z[:t].view(np.uint32)), t
        assert np.array_equal(got["round"].view(np.uint32), got["product"].view(np.uint32))
        assert np.array_equal(got["residual"].view(np.uint32), (case.res + got["product"]).view(np.uint32))
        xn = rms(case.x, case.nw)
        g, u = (oracle.gemm_f64(q, rows, cols, case.x) for q in case.q8)
        gn, un = (oracle.gemm_f64(q, rows, cols, xn.astype(np.float32)) for q in case.q8)
        for kind, want in (("product", g), ("pair", oracle.swiglu_f64(g, u)), ("norm", gn), ("round_norm", gn), ("pair_norm", oracle.swiglu_f64(gn, un))):
            assert_parity(got[kind], want, f"{kind} {rows}x{cols}")
    finally:
        case.close()


def test_any_cols_infinite_scale(rt):
    """Dead lanes load unit 0: an infinite scale there reaches its own row as the looping sum of the
    same blocks gives it (infinite, or NaN), and no other row."""
    rows, cols = 64, 1056
    rng = np.random.default_rng(3)
    q, d = synth.split(synth.q8_rows(rng, rows, cols), rows, cols)
    d = d.copy()
    d[5, 0] = np.inf
    case = Case(rt, rows, cols, 4, 11, q8=[synth.join(q, d)] * 2)
    try:
        case.run("product", 0, 4)
        y = case.out()[0]
        assert np.all(np.isinf(y[:, 5])) and np.all(np.isfinite(np.delete(y, 5, axis=1)))
    finally:
        case.close()


@pytest.mark.parametrize("cols", [32, 1056, 1536, 4128, 5632])
def test_any_cols_infinite_norm_weight(rt, cols):
    """Lanes past the row's last unit, and the threads that take none of the tail's, load unit 0: an
    infinite norm weight there makes a row infinite (NaN where its quant is 0), as with the norm
    apart, not NaN from those lanes' 0 * inf. A NaN x there stays its own token's."""
    case = Case(rt, 64, cols, 4, cols)
    nw, x = case.nw.copy(), case.x.copy()
    nw[3], x[2, 5] = np.inf, np.nan
    rt.to_dev(case.p["nw"], nw)
    rt.to_dev(case.p["x"], x)
    try:
        for kind in ("norm", "pair_norm", "round_norm"):
            for t in (1, 2, 4):
                out = []
                for apart in (False, True):
                    rt.set_epi_apart(apart)
                    case.nan()
                    case.run(kind, 0, t)
                    out.append([a[:t] for a in case.out()])
                rt.set_epi_apart(False)
                for a, b in zip(*out):
                    assert np.array_equal(np.isnan(a), np.isnan(b)), (kind, t)
                    assert np.array_equal(a[np.isinf(a)], b[np.isinf(a)]), (kind, t)
                assert np.isinf(out[1][0][0]).any(), (kind, t)
    finally:
        rt.set_epi_apart(False)
        case.close()


@pytest.mark.parametrize("rows,cols,kind,t,name", [
    (1008, 8192, "residual", 4, "gemv_ke<4, 4, 1, 8, 0, 2>"), (1008, 8192, "norm", 3, "gemv_ke<3, 4, 1, 8, 0, 1>"),
    (4112, 8192, "norm", 4, "gemv_k<4, 8, 1, 8, 0>"), (4096, 8192, "round_norm", 4, "gemv_round<4, 8, 1, 8>"),
    (4080, 8192, "round_norm", 4, "gemv_round_norm<4, 8, 1, 8>"), (4112, 5152, "norm", 4, "gemv_any<4, 8, 8, 0, 0>"),
    (4096, 5152, "norm", 4, "gemv_any<4, 8, 8, 0, 1>"), (4112, 5152, "residual", 4, "gemv_any<4, 8, 8, 0, 0>"),
    (4112, 5152, "residual", 3, "gemv_any<3, 8, 8, 0, 2>"), (4112, 5152, "round_norm", 4, "gemv_round_any<4, 8, 8, 0>"),
    (6144, 5152, "pair", 3, "gemv_any<3, 4, 8, 1, 0>"), (6144, 5152, "pair_norm", 3, "gemv_any<3, 4, 8, 1, 1>"),
    (6144, 5152, "pair_norm", 2, "gemv_any<2, 8, 8, 1, 1>"), (2048, 5152, "pair_norm", 4, "gemv_any<4, 2, 8, 1, 1>")])
def test_five_to_eight_waves(rt, rows, cols, kind, t, name):
    """The instances that 5 to 8 waves choose at the rows where the rules change: fused up to a few thousand
    rows, apart above, four rows of the pair; each against the epilogue apart (the residual and the pair
    the same bits, the norm within its order of summation)."""
    case = Case(rt, rows, cols, t, rows + cols + t)
    try:
        out = []
        for apart in (False, True):
            rt.set_epi_apart(apart)
            case.nan()
            names = kernels(rt, lambda: case.run(kind, 0, t))
            if not apart:
                assert names[0] == name
            out.append(case.out())
        for a, b in zip(*out):
            if "norm" not in kind:
                assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
            elif not np.isnan(a).all():
                assert_parity(a, b.astype(np.float64), f"{kind} {rows}x{cols} t={t}")
    finally:
        rt.set_epi_apart(False)
        case.close()


@pytest.mark.parametrize("rows,cols,kind", [(4112, 8192, "norm"), (4112, 5152, "residual"), (4112, 5152, "norm"), (4112, 8192, "round_norm"), (4112, 5152, "round_norm")])
def test_recorded_without_a_workspace(q8rt, rt, rows, cols, kind):
    """Rows on which the epilogue runs apart, recorded by a runtime that has run nothing: fused, as it needs no
    workspace then."""
    case = Case(rt, rows, cols, 4, 5)
    try:
        case.nan()
        case.run(kind, 0, 4)
        want = case.out()
    finally:
        case.close()
    with q8rt.Runtime() as r2:
        c2 = Case(r2, rows, cols, 4, 5)
        r2.lib.rt_graph_begin(r2.R)
        c2.run(kind, 0, 4)
        g = P(r2.lib.rt_graph_end(r2.R))
        for _ in range(2):
            c2.nan()
            r2.lib.rt_graph_launch(r2.R, g)
            for a, b in zip(c2.out(), want):
                if not np.isnan(b).all():
                    assert_parity(a, b.astype(np.float64), f"{kind} {rows}x{cols}")
        r2.lib.rt_graph_free(r2.R, g)
        c2.close()
