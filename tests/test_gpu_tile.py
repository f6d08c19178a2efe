"""Products of more than 64 tokens as one launch (csrc/q8_tile.hip) against the 64-token launches,
bit for bit: the same sums in the same order, at every tile configuration (by name), partial tiles of rows and
tokens, x rows apart, odd block counts (half a last pair, 2-byte aligned scales), forced K splits (one, and a
shorter last one), the residual (in place too), the norm, the fused pair, rounds, non-finite x and scales, chunks of
the limb image, and under graph capture."""
import ctypes as c

import numpy as np
import pytest

import synth
from parity import assert_parity

pytestmark = pytest.mark.gpu

P = c.c_void_p


def kernels(rt, fn):
    """The names of the first kernels of the products fn launches (the runtime's records)."""
    n = 256
    rt.lib.rt_ktime(rt.R, 1)
    fn()
    arrs = [np.zeros(n, np.int32), np.zeros(n, np.int64), np.zeros(n, np.int64), np.zeros(n, np.int64), np.zeros(n, np.float32)]
    names, grid = c.create_string_buffer(64 * n), np.zeros(n, np.int64)
    got = rt.lib.rt_ktime_read(rt.R, *(a.ctypes.data_as(P) for a in arrs), names, grid.ctypes.data_as(P), n)
    rt.lib.rt_ktime(rt.R, 0)
    return [names.raw[64 * i:64 * i + 64].split(b"\0")[0].decode() for i in range(got)]


class Case:
    """Two matrices and x on the device (its rows cols + pad floats apart); run(kind, k, n) is one call on
    tokens [k, k + n)."""

    def __init__(self, rt, rows, cols, t, seed, x=None, q8=None, pad=0):
        rng = np.random.default_rng(seed)
        self.rt, self.rows, self.cols, self.t = rt, rows, cols, t
        self.q8 = q8 or [synth.q8_rows(rng, rows, cols) for _ in range(2)]
        self.x = synth.x_f32(rng, t, cols) if x is None else x
        self.nw = (1.0 + 0.1 * rng.standard_normal(cols)).astype(np.float32)
        self.res = rng.standard_normal((t, rows)).astype(np.float32)
        self.w = [rt.upload(q, rows, cols) for q in self.q8]
        self.xs = cols + pad
        self.p = {k: self.put(v) for k, v in (("x", np.pad(self.x, ((0, 0), (0, pad)), constant_values=np.nan)), ("nw", self.nw), ("res", self.res))}
        self.y, self.z = rt.alloc(4 * t * rows), rt.alloc(4 * t * 16)

    def put(self, a):
        p = self.rt.alloc(a.nbytes)
        self.rt.to_dev(p, a)
        return p

    def close(self):
        for w in self.w:
            self.rt.lib.rt_q8_free(self.rt.R, P(w))
        for p in (*self.p.values(), self.y, self.z):
            self.rt.free(p)

    def run(self, kind, k, n):
        lib, R, rows, cols, eps = self.rt.lib, self.rt.R, self.rows, self.cols, c.c_float(1e-6)
        xs = self.xs
        x, y, nw, res = P(self.p["x"] + 4 * k * xs), P(self.y + 4 * k * rows), P(self.p["nw"]), P(self.p["res"] + 4 * k * rows)
        w = [P(v) for v in self.w]
        if kind == "product":
            lib.rt_gemm_dev(R, w[0], rows, cols, x, xs, n, y)
        elif kind == "noalloc":
            lib.rt_gemm_dev_noalloc(R, w[0], rows, cols, x, xs, n, y)
        elif kind == "residual":
            lib.rt_gemm_residual_dev(R, w[0], rows, cols, x, xs, n, res, y)
        elif kind == "inplace":  # the residual in y itself
            lib.rt_gemm_residual_dev(R, w[0], rows, cols, x, xs, n, y, y)
        elif kind == "norm":
            lib.rt_gemm_norm_dev(R, w[0], rows, cols, x, xs, n, nw, eps, y)
        elif kind == "pair":
            lib.rt_gemv_swiglu_dev(R, w[0], w[1], rows, cols, x, xs, n, y)
        elif kind == "pair_norm":
            lib.rt_gemv_swiglu_norm_dev(R, w[0], w[1], rows, cols, x, xs, n, nw, eps, y)
        else:  # rounds: the matrix and a 16-row prefix of the other
            ws, rr = (P * 2)(self.w[0], self.w[1]), (c.c_long * 2)(rows, 16)
            ys = (P * 2)(self.y + 4 * k * rows, self.z + 4 * k * 16)
            if kind == "round":
                lib.rt_gemv_round_dev(R, 2, ws, rr, cols, x, xs, n, ys)
            else:
                lib.rt_gemv_round_norm_dev(R, 2, ws, rr, cols, x, xs, n, nw, eps, ys)

    def out(self):
        y, z = np.empty((self.t, self.rows), np.float32), np.empty((self.t, 16), np.float32)
        self.rt.from_dev(y, self.y)
        self.rt.from_dev(z, self.z)
        return y, z

    def nan(self):
        self.rt.to_dev(self.y, np.full((self.t, self.rows), np.nan, np.float32))
        self.rt.to_dev(self.z, np.full((self.t, 16), np.nan, np.float32))

    def whole_and_parts(self, kind):
        """(kernel name, outputs of one call, outputs of calls of up to 64 tokens and 5 or more)"""
        self.nan()
        if kind == "inplace":
            self.rt.to_dev(self.y, self.res)
        names = kernels(self.rt, lambda: self.run(kind, 0, self.t))
        one = self.out()
        self.nan()
        if kind == "inplace":
            self.rt.to_dev(self.y, self.res)
        step = 64 if self.t % 64 == 0 or self.t % 64 >= 5 else 59  # every call on the matrix cores, no token twice
        for k in range(0, self.t, step):
            self.run(kind, k, min(step, self.t - k))
        return names[0], one, self.out()


KINDS = ("product", "noalloc", "residual", "inplace", "norm", "pair", "pair_norm", "round", "round_norm")
# (rows, cols, tokens, forced K splits): the tiles' edges. 512 x 4096 rows fill the device with the
# small tiles and 12288 with the large ones
SHAPES = [(256, 64, 300, 0), (512, 96, 2000, 0), (1888, 1056, 131, 0), (1888, 1056, 500, 3), (1888, 1056, 200, 1), (2048, 6144, 203, 0), (2048, 2048, 203, 5), (4096, 1024, 513, 1), (5136, 2784, 300, 0),
          (12288, 1024, 512, 0), (12288, 1024, 257, 3), (12272, 1056, 250, 0), (16400, 512, 1030, 0)]


@pytest.mark.parametrize("rows,cols,t,ks", SHAPES)
def test_long_prompt_bits(rt, rows, cols, t, ks):
    case = Case(rt, rows, cols, t, rows + cols + t, pad=4 * (rows % 7))
    rt.gemm_force(False, ks)
    try:
        for kind in KINDS:
            name, one, parts = case.whole_and_parts(kind)
            print("long prompt", rows, cols, t, ks, kind, name, flush=True)
            assert name.startswith("gemm_tile<"), kind
            for a, b in zip(one, parts):
                assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), kind
    finally:
        rt.gemm_force()
        case.close()


# each configuration, at several K splits of odd block counts, with partial tiles of rows and tokens
TILES = [("8, 2, 8, 1, 3, 1", 12304, 736, 260), ("4, 2, 8, 1, 4, 1", 10256, 736, 130), ("4, 2, 4, 1, 2, 2", 11280, 736, 66), ("4, 2, 2, 1, 2, 2", 1040, 736, 513),
         ("3, 2, 2, 1, 2, 2", 528, 736, 560), ("2, 2, 2, 1, 2, 2", 240, 736, 66), ("8, 1, 8, 2, 3, 1", 11280, 736, 130), ("4, 1, 8, 2, 4, 1", 11280, 736, 66),
         ("4, 1, 4, 2, 2, 2", 528, 736, 513), ("2, 1, 4, 2, 2, 2", 240, 736, 66)]


@pytest.mark.parametrize("tile,rows,cols,t", TILES)
def test_every_tile_bits(rt, tile, rows, cols, t):
    """Every configuration by name, where the rule chooses it, bit for bit the 64-token launches."""
    case = Case(rt, rows, cols, t, rows + t)
    try:
        name, one, parts = case.whole_and_parts("pair" if tile.split(", ")[3] == "2" else "product")
        assert name == f"gemm_tile<{tile}>"
        assert np.array_equal(one[0].view(np.uint32), parts[0].view(np.uint32))
    finally:
        case.close()


@pytest.mark.parametrize("kind,rows,cols,t,name", [
    ("product", 5232, 4352, 148, "gemm_tile<2, 2, 2, 1, 2, 2>"), ("product", 1024, 3072, 91, "gemm_mfma<"), ("product", 16, 8192, 200, "gemm_mfma<"),
    ("norm", 5376, 3040, 116, "gemm_tile<"), ("round_norm", 256, 1984, 60, "gemm_mfma_round<"), ("round_norm", 2480, 3072, 53, "gemm_mfma_round<"),
    ("round", 256, 4096, 65, "gemm_mfma_round<")])
def test_the_rule(rt, kind, rows, cols, t, name):
    """Sizes at which another route was up to 1.9 times slower: tiles whose row tiles and token groups fill one
    XCD past its compute units, few rows (the 64-token launches split K over the device), and rounds of 65
    tokens."""
    case = Case(rt, rows, cols, t, 3)
    try:
        assert kernels(rt, lambda: case.run(kind, 0, t))[0].startswith(name)
    finally:
        case.close()


def test_long_prompt_parity_and_image_chunks(rt, oracle):
    """Against F64, with heavy-tailed scales; and a prompt whose limb image takes two chunks of
    rt_gemm_dev_noalloc's 32 MiB (12288 columns: 384 tokens a chunk), bit for bit the one of 64 MiB."""
    rng = np.random.default_rng(5)
    q8 = synth.q8_rows(rng, 512, 12288, "lognormal")
    case = Case(rt, 512, 12288, 450, 6, q8=[q8, q8])
    try:
        case.run("product", 0, 450)
        whole = case.out()[0]
        assert_parity(whole[:96], oracle.gemm_f64(q8, 512, 12288, case.x[:96]), "512x12288 t=450")
        case.nan()
        case.run("noalloc", 0, 450)
        assert np.array_equal(case.out()[0].view(np.uint32), whole.view(np.uint32))
    finally:
        case.close()


def test_long_prompt_non_finite(rt):
    """Infinite and NaN x, and an infinite scale in a row's last block of an odd count: the same
    values, NaN for NaN, as the 64-token launches."""
    rows, cols, t = 256, 1056, 200
    rng = np.random.default_rng(7)
    q, d = synth.split(synth.q8_rows(rng, rows, cols), rows, cols)
    d = d.copy()
    d[3, -1], d[17, 5] = np.inf, np.inf
    q8 = synth.join(q, d)
    x = synth.x_f32(rng, t, cols)
    x[0, 5], x[70, 40], x[150, cols - 1], x[199, 0] = np.inf, -np.inf, np.nan, 3e38
    case = Case(rt, rows, cols, t, 8, x=x, q8=[q8, q8])
    try:
        for kind in ("product", "pair", "norm"):
            name, one, parts = case.whole_and_parts(kind)
            assert name.startswith("gemm_tile<"), name
            assert np.array_equal(one[0], parts[0], equal_nan=True), kind
    finally:
        case.close()


def test_long_prompt_recorded(q8rt, rt):
    """Recorded and replayed three times with eager work between, bit for bit; and a runtime whose
    limb image does not exist yet records the 64-token launches instead of refusing."""
    case = Case(rt, 1024, 1024, 200, 9)
    try:
        case.run("pair", 0, 200)
        case.run("product", 0, 200)
        eager = case.out()[0]
        rt.lib.rt_graph_begin(rt.R)
        case.run("product", 0, 200)
        g = rt.lib.rt_graph_end(rt.R)
        for _ in range(3):
            case.run("pair", 0, 200)
            case.nan()
            rt.lib.rt_graph_launch(rt.R, P(g))
            assert np.array_equal(case.out()[0].view(np.uint32), eager.view(np.uint32))
        rt.lib.rt_graph_free(rt.R, P(g))
    finally:
        case.close()
    with q8rt.Runtime() as r2:
        c2 = Case(r2, 1024, 1024, 200, 9)
        c2.run("product", 0, 40)  # the 64-token launches' workspace, but no limb image
        r2.lib.rt_graph_begin(r2.R)
        c2.run("product", 0, 200)
        g = r2.lib.rt_graph_end(r2.R)
        c2.nan()
        r2.lib.rt_graph_launch(r2.R, P(g))
        assert np.array_equal(c2.out()[0].view(np.uint32), eager.view(np.uint32))
        r2.lib.rt_graph_free(r2.R, P(g))
        c2.close()


@pytest.mark.parametrize("rows,cols", [(1040, 1056), (64, 2048)])
@pytest.mark.parametrize("t", [65, 130, 300])
def test_long_prompt_host_calls(rt, t, rows, cols):
    """rt_gemm, and two products queued with another of one token, on host arrays: y goes through HBM
    where the tiles run and over the link from the sums where they do not (64 rows); bit for bit the device products, with x and y sizes that grow and shrink."""
    case = Case(rt, rows, cols, t, 21 + t)
    try:
        case.run("product", 0, t)
        want = case.out()[0]
        y = [np.full((t, rows), np.nan, np.float32) for _ in range(3)]
        x1, y1 = np.ascontiguousarray(case.x[:1]), np.full((1, rows), np.nan, np.float32)
        rt.gemm(case.w[0], rows, cols, case.x, t, y[0])
        rt.gemm_q(case.w[0], rows, cols, case.x, t, y[1])
        rt.gemv_q(case.w[1], rows, cols, x1, y1)
        rt.gemm_q(case.w[0], rows, cols, case.x, t, y[2])
        rt.gemv_go()
        for a in y:
            assert np.array_equal(a.view(np.uint32), want.view(np.uint32))
        rt.lib.rt_gemv_dev(rt.R, P(case.w[1]), rows, cols, P(case.p["x"]), P(case.y))
        assert np.array_equal(case.out()[0][0].view(np.uint32), y1[0].view(np.uint32))
    finally:
        case.close()


@pytest.mark.parametrize("shapes,cols,t,tile", [([8192, 4096, 32, 32], 4096, 64, True), ([8192, 4096, 32, 32], 4096, 33, False), ([4096, 4096, 4096, 48], 1056, 63, True),
                                                ([12288, 16], 4096, 64, False), ([6144, 16], 1056, 33, False)])
def test_round_on_a_norm_up_to_64_tokens(rt, shapes, cols, t, tile):
    """Rounds on a norm from 33 tokens: the norm in the limb image and the tiles where that is the faster,
    against the norm, the 64-token round and its sums apart, bit for bit. x rows apart."""
    rng, n, xs = np.random.default_rng(t), len(shapes), cols + 12
    q8 = [synth.q8_rows(rng, r, cols) for r in shapes]
    x, nw = rng.standard_normal((t, xs)).astype(np.float32), (1.0 + 0.1 * rng.standard_normal(cols)).astype(np.float32)
    w = [rt.upload(q, r, cols) for q, r in zip(q8, shapes)]
    px, pn, py = rt.alloc(x.nbytes), rt.alloc(nw.nbytes), [rt.alloc(4 * t * r) for r in shapes]
    rt.to_dev(px, x)
    rt.to_dev(pn, nw)

    def run():
        rt.lib.rt_gemv_round_norm_dev(rt.R, n, (P * n)(*w), (c.c_long * n)(*shapes), cols, P(px), xs, t, P(pn), c.c_float(1e-6), (P * n)(*py))

    def out():
        got = [np.empty((t, r), np.float32) for r in shapes]
        for a, p in zip(got, py):
            rt.from_dev(a, p)
        return got

    try:
        name = kernels(rt, run)[0]
        got = out()
        rt.set_epi_apart(True)
        run()
        print("round on a norm", shapes, cols, t, name, flush=True)
        assert name.startswith("gemm_tile<" if tile else "gemm_mfma_"), name
        for a, b in zip(got, out()):
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    finally:
        rt.set_epi_apart(False)
        for p in (px, pn, *py):
            rt.free(p)
        for v in w:
            rt.lib.rt_q8_free(rt.R, P(v))


@pytest.mark.parametrize("t", [65, 68, 70])
@pytest.mark.parametrize("shapes", [[8192, 1024, 1024], [2048, 2048]], ids=["qkv", "pair"])
def test_rounds_of_64_tokens_and_a_rest(q8rt, rt, t, shapes):
    """The 64-token round and one of the last 1, 4 and 6 tokens, as a runtime without a limb image records
    them: the bits of the tiles' round."""
    rng = np.random.default_rng(t)
    q8, x, n = [synth.q8_rows(rng, r, 4096) for r in shapes], synth.x_f32(rng, t, 4096), len(shapes)

    def run(r, record):
        w = [r.upload(q, k, 4096) for q, k in zip(q8, shapes)]
        px, py = r.alloc(x.nbytes), [r.alloc(4 * t * k) for k in shapes]
        r.to_dev(px, x)
        args = (r.R, n, (P * n)(*w), (c.c_long * n)(*shapes), 4096, P(px), 4096)
        if record:
            r.lib.rt_gemv_round_dev(*args, 64, (P * n)(*py))  # the rounds' workspace
            r.lib.rt_graph_begin(r.R)
        r.lib.rt_gemv_round_dev(*args, t, (P * n)(*py))
        if record:
            g = P(r.lib.rt_graph_end(r.R))
            r.lib.rt_graph_launch(r.R, g)
            r.lib.rt_graph_launch(r.R, g)
        out = [np.empty((t, k), np.float32) for k in shapes]
        for a, p in zip(out, py):
            r.from_dev(a, p)
        if record:
            r.lib.rt_graph_free(r.R, g)
        for p in (px, *py):
            r.free(p)
        for v in w:
            r.lib.rt_q8_free(r.R, P(v))
        return out

    assert kernels(rt, lambda: run(rt, False))[0].startswith("gemm_tile<")
    with q8rt.Runtime() as r2:
        for a, b in zip(run(rt, False), run(r2, True)):
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


@pytest.mark.parametrize("cols", [1024, 3104])
def test_round_sums_of_many_outputs(rt, cols):
    """A round of 788480 outputs at 64 tokens sums four outputs a thread where its products have at most 32
    splits (1024 columns), and one where its 32 rows have 49 (3104): each product's bits are its own
    launch's."""
    t, shapes = 64, [12288, 32]
    rng = np.random.default_rng(cols)
    q8, x = [synth.q8_rows(rng, r, cols) for r in shapes], synth.x_f32(rng, t, cols)
    w = [rt.upload(q, r, cols) for q, r in zip(q8, shapes)]
    px, py, pz = rt.alloc(x.nbytes), [rt.alloc(4 * t * r) for r in shapes], [rt.alloc(4 * t * r) for r in shapes]
    try:
        rt.to_dev(px, x)
        rt.lib.rt_gemv_round_dev(rt.R, 2, (P * 2)(*w), (c.c_long * 2)(*shapes), cols, P(px), cols, t, (P * 2)(*py))
        for v, r, a, b in zip(w, shapes, py, pz):
            rt.lib.rt_gemm_dev(rt.R, P(v), r, cols, P(px), cols, t, P(b))
            one, two = np.empty((t, r), np.float32), np.empty((t, r), np.float32)
            rt.from_dev(one, a)
            rt.from_dev(two, b)
            assert np.array_equal(one.view(np.uint32), two.view(np.uint32)), r
    finally:
        for p in (px, *py, *pz):
            rt.free(p)
        for v in w:
            rt.lib.rt_q8_free(rt.R, P(v))


@pytest.mark.parametrize("rows,cols,first,t", [(1024, 1024, 66, 500), (64, 2048, 64, 210), (64, 2048, 70, 130), (2048, 1056, 130, 131)])
@pytest.mark.parametrize("exact", [False, True])
def test_recorded_at_more_tokens_than_ran(q8rt, rt, rows, cols, first, t, exact):
    """A runtime that ran each product once, at 64 tokens or a few more, records them at more: on the tiles,
    which need no workspace but the image, or 64 tokens at a time where the rule refuses them (64 rows).
    Replayed twice with eager work between, bit for bit the eager products."""
    kinds = ("product", "residual", "norm", "pair", "pair_norm", "round", "round_norm")
    want, case = {}, Case(rt, rows, cols, t, 31)
    rt.set_exact(exact)
    try:
        for kind in kinds:
            case.nan()
            case.run(kind, 0, t)
            want[kind] = case.out()
    finally:
        rt.set_exact(False)
        case.close()
    with q8rt.Runtime() as r2:
        r2.set_exact(exact)
        c2 = Case(r2, rows, cols, t, 31)
        for kind in kinds:
            c2.run(kind, 0, first)
        for kind in kinds:
            r2.lib.rt_graph_begin(r2.R)
            c2.run(kind, 0, t)
            g = P(r2.lib.rt_graph_end(r2.R))
            for _ in range(2):
                c2.run("pair", 0, 5)
                c2.nan()
                r2.lib.rt_graph_launch(r2.R, g)
                for a, b in zip(c2.out(), want[kind]):
                    assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), kind
            r2.lib.rt_graph_free(r2.R, g)
        c2.close()
