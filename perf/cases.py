"""The workloads this library is measured on, through its public entry points (include/q8_rt.h, as
the package binds them), and their answers in 64 bits.

Three kinds of case, all on Q8_0 weights quantised as GGUF files hold them (per 32 columns the
largest magnitude over 127 as a binary16 scale, and rounded int8):

  layer    the products of transformer layers with their epilogues, activations in HBM: the RMS norm
           and the mixer's products that share it (one launch round), the output product with its
           residual, the fused gate and up on the second norm, down with its residual. With a
           vocabulary, the tokens' embedding rows are gathered first and the head (the tied matrix,
           behind a norm of its own) gives logits and the greedy next token: of every token up to
           4, as verifying drafts needs them, and of the last one of a prompt. graph: recorded once
           into the library's graph and replayed, as a decode loop does.
  product  one product (or the fused gate and up) of activations in HBM, for sizes that no tuned
           configuration names: columns that are no multiple of 1024, odd block counts.
  host     the drop-in entry points on host arrays: rt_gemv, or products queued with rt_gemm_q and
           run by rt_gemv_go.
"""
import ctypes as c
import importlib.util
import os
import sys

import numpy as np
import torch

EPS = 1e-6
_SHARED = {}


def listed():
    nine = {"kind": "layer", "hidden": 4096, "ffn": 12288, "layers": 1, "vocab": 0, "graph": False}
    quartet, attention = "8192,4096,32,32", "8192,1024,1024"
    return [
        # the smallest calls: a 2B-class decode step's 96 short dependent products, recorded once
        {"name": "decode_2b_t1", "kind": "layer", "hidden": 2048, "ffn": 6144, "mix": "3072", "layers": 24, "vocab": 0, "tokens": 1, "graph": True},
        # a 9B-class decode step cut to 4 of its layers, with the embedding read, the 151936-row head and the next token
        {"name": "decode_9b_t1", **nine, "mix": quartet, "layers": 4, "vocab": 151936, "tokens": 1, "graph": True},
        # speculative verify: an attention layer on a token and its three drafts
        {"name": "verify_9b_t4", **nine, "mix": attention, "tokens": 4},
        # prompt chunks of the sizes that the engine sends (16 and 40) and the largest one the matrix cores take in a launch
        {"name": "prompt_9b_t16", **nine, "mix": quartet, "tokens": 16},
        {"name": "prompt_9b_t40", **nine, "mix": attention, "tokens": 40},
        {"name": "prompt_9b_t64", **nine, "mix": quartet, "tokens": 64},
        # a whole prompt in one call, with the embedding read and the draft head (32768 rows) on its last token
        {"name": "prompt_9b_t512", **nine, "mix": attention, "vocab": 32768, "tokens": 512},
        # a prompt of an odd length on the small model's layer
        {"name": "prompt_2b_t203", "kind": "layer", "hidden": 2048, "ffn": 6144, "mix": "3072", "layers": 1, "vocab": 0, "tokens": 203, "graph": False},
        # decode and prompt on matrices of other sizes: 129 and 87 blocks a row, 321 groups of rows
        {"name": "pair_odd_t3", "kind": "product", "rows": 11008, "cols": 4128, "tokens": 3, "pair": True},
        {"name": "gemm_odd_t37", "kind": "product", "rows": 5136, "cols": 2784, "tokens": 37, "pair": False},
        # the drop-in path: one product a call, and the FFN's gate and up queued at 16 tokens
        {"name": "host_gemv", "kind": "host", "rows": 4096, "cols": 4096, "tokens": 1, "products": 1},
        {"name": "host_round_t16", "kind": "host", "rows": 12288, "cols": 4096, "tokens": 16, "products": 2},
    ]


def _log(rng, low, high, step):
    """A multiple of step in [low, high], spread over the logarithm."""
    v = int(round(low * (high / low) ** rng.random() / step)) * step
    return min(high, max(low, v))


def draw(rng):
    kind = rng.choice(["layer", "layer", "layer", "product", "product", "host"])
    if kind == "layer":
        tokens = rng.choice([1, rng.randint(2, 4), _log(rng, 5, 64, 1), _log(rng, 65, 512, 1)])
        hidden = _log(rng, 1024, 4096, rng.choice([32, 256, 1024]))
        ffn = min(12288, int(hidden * rng.uniform(2.0, 3.5)) // 256 * 256)
        kv = max(1, hidden // 512) * 128
        mix = rng.choice(["%d" % (hidden + 2 * kv), "%d,%d,32,32" % (2 * hidden, hidden), "%d,%d,%d" % (2 * hidden, kv, kv)])
        vocab = rng.choice([0, _log(rng, 8192, 65536, 16)])
        return {"kind": "layer", "hidden": hidden, "ffn": ffn, "mix": mix, "layers": rng.randint(2, 8) if tokens == 1 else 1, "vocab": vocab,
                "tokens": tokens, "graph": tokens == 1}
    rows, cols = _log(rng, 2048, 12288, 16), _log(rng, 1024, 12288, 32)
    if kind == "product":
        return {"kind": "product", "rows": rows, "cols": cols, "tokens": _log(rng, 1, 300, 1), "pair": rng.random() < 0.4}
    return {"kind": "host", "rows": rows, "cols": min(cols, 4096), "tokens": _log(rng, 1, 64, 1), "products": rng.randint(1, 3)}


# ---- the inputs, in one order for prepare() and exact()


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _blocks(gen, rows, cols, sigma):
    """(q int8 [rows, blocks, 32], d binary16 [rows, blocks, 1]) of N(0, sigma) weights as GGUF quantises them."""
    w = torch.randn(rows, cols // 32, 32, generator=gen, device="cuda", dtype=torch.float32).mul_(sigma)
    d = (w.abs().amax(dim=2, keepdim=True) / 127.0).half()
    q = torch.clamp(torch.round(w / d.float().clamp_min(1e-12)), -127, 127).to(torch.int8)
    return q, d


def _gguf(gen, rows, cols, sigma):
    """The same as GGUF Q8_0 rows: 34-byte blocks."""
    out = torch.empty(rows, cols // 32, 34, dtype=torch.uint8, device="cuda")
    for r in range(0, rows, 16384):
        q, d = _blocks(gen, min(16384, rows - r), cols, sigma)
        out[r:r + 16384, :, :2] = d.view(torch.uint8)
        out[r:r + 16384, :, 2:] = q.view(torch.uint8)
    return out


def _dense(gen, rows, cols, sigma):
    """The same as float64 [rows, cols]."""
    out = torch.empty(rows, cols, dtype=torch.float64, device="cuda")
    for r in range(0, rows, 16384):
        q, d = _blocks(gen, min(16384, rows - r), cols, sigma)
        out[r:r + 16384] = (q.double() * d.double()).reshape(-1, cols)
    return out


def _mix(case):
    return [int(v) for v in case["mix"].split(",")]


def _layer_inputs(case, seed, matrix):
    """Every input of a layer case, its matrices made by matrix(gen, rows, cols, sigma)."""
    gen, h, f, t = _gen(seed), case["hidden"], case["ffn"], case["tokens"]
    made = {"layers": []}
    for _ in range(case["layers"]):
        made["layers"].append({
            "mix": [matrix(gen, r, h, h ** -0.5) for r in _mix(case)], "out": matrix(gen, h, h, h ** -0.5),
            "gate": matrix(gen, f, h, h ** -0.5), "up": matrix(gen, f, h, h ** -0.5), "down": matrix(gen, h, f, f ** -0.5),
            "anorm": 1.0 + 0.1 * torch.randn(h, generator=gen, device="cuda"), "pnorm": 1.0 + 0.1 * torch.randn(h, generator=gen, device="cuda")})
    if case["vocab"]:
        made["head"] = matrix(gen, case["vocab"], h, h ** -0.5)
        made["fnorm"] = 1.0 + 0.1 * torch.randn(h, generator=gen, device="cuda")
        made["ids"] = torch.randint(0, case["vocab"], (t,), generator=gen, device="cuda", dtype=torch.int64)
    else:
        made["x"] = torch.randn(t, h, generator=gen, device="cuda")
    return made


def _product_inputs(case, seed, matrix):
    gen, n = _gen(seed), case.get("products", 2 if case.get("pair") else 1)
    w = [matrix(gen, case["rows"], case["cols"], case["cols"] ** -0.5) for _ in range(n)]
    return w, torch.randn(case["tokens"], case["cols"], generator=gen, device="cuda")


# ---- the library


def _runtime():
    if "rt" not in _SHARED:
        if "q8rt" in sys.modules:
            mod = sys.modules["q8rt"]
        else:
            root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
            spec = importlib.util.spec_from_file_location("q8rt", os.path.join(root, "intel-phi-apl_amd", "__init__.py"))
            mod = importlib.util.module_from_spec(spec)
            sys.modules["q8rt"] = mod
            spec.loader.exec_module(mod)
        _SHARED["rt"] = mod.Runtime()
    return _SHARED["rt"]


class _Graph:
    """A recorded sequence, freed with its state."""

    def __init__(self, rt, record):
        self.rt = rt
        record()
        rt.sync()
        rt.lib.rt_graph_begin(rt.R)
        record()
        self.handle = c.c_void_p(rt.lib.rt_graph_end(rt.R))

    def launch(self):
        self.rt.lib.rt_graph_launch(self.rt.R, self.handle)

    def __del__(self):
        self.rt.sync()
        self.rt.lib.rt_graph_free(self.rt.R, self.handle)


def _handles(rt):
    """matrix() for the inputs: the weights in the library's device form, registered as handles."""

    def matrix(gen, rows, cols, sigma):
        raw = _gguf(gen, rows, cols, sigma)
        w = torch.empty(raw.numel(), dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()
        rt.lib.rt_q8_repack_dev(rt.R, _p(raw), rows, cols, _p(w))
        rt.sync()
        return w

    return matrix


def _p(tensor):
    return c.c_void_p(tensor.data_ptr())


def _f32(*shape):
    return torch.empty(*shape, dtype=torch.float32, device="cuda")


def _layer_state(case, seed, rt):
    h, f, t, mix = case["hidden"], case["ffn"], case["tokens"], _mix(case)
    made = _layer_inputs(case, seed, _handles(rt))
    out = {"mix": [_f32(t, r) for r in mix], "mid": _f32(t, h), "x": _f32(t, h)}
    act, other, lib, R, calls = _f32(t, f), _f32(t, h), rt.lib, rt.R, []
    x = made.get("x")
    if case["vocab"]:
        x = _f32(t, h)
        calls.append((lib.rt_q8_rows_dev, (R, _p(made["head"]), h, _p(made["ids"]), t, _p(x))))
    rows, n, eps = (c.c_long * len(mix))(*mix), len(mix), c.c_float(EPS)
    ys = (c.c_void_p * n)(*[y.data_ptr() for y in out["mix"]])
    for k, lay in enumerate(made["layers"]):
        new = out["x"] if (case["layers"] - k) % 2 else other
        if n == 1:
            calls.append((lib.rt_gemm_norm_dev, (R, _p(lay["mix"][0]), mix[0], h, _p(x), h, t, _p(lay["anorm"]), eps, _p(out["mix"][0]))))
        else:
            ws = (c.c_void_p * n)(*[w.data_ptr() for w in lay["mix"]])
            calls.append((lib.rt_gemv_round_norm_dev, (R, n, ws, rows, h, _p(x), h, t, _p(lay["anorm"]), eps, ys)))
        calls.append((lib.rt_gemm_residual_dev, (R, _p(lay["out"]), h, h, _p(out["mix"][0]), mix[0], t, _p(x), _p(out["mid"]))))
        calls.append((lib.rt_gemv_swiglu_norm_dev, (R, _p(lay["gate"]), _p(lay["up"]), f, h, _p(out["mid"]), h, t, _p(lay["pnorm"]), eps, _p(act))))
        calls.append((lib.rt_gemm_residual_dev, (R, _p(lay["down"]), h, f, _p(act), f, t, _p(out["mid"]), _p(new))))
        x = new
    if case["vocab"]:
        last = t if t <= 4 else 1
        out["logits"], out["next"] = _f32(last, case["vocab"]), torch.empty(last, dtype=torch.int64, device="cuda")
        calls.append((lib.rt_gemm_norm_dev, (R, _p(made["head"]), case["vocab"], h, _p(x[t - last:]), h, last, _p(made["fnorm"]), eps, _p(out["logits"]))))
        for k in range(last):
            calls.append((lib.rt_argmax_dev, (R, _p(out["logits"][k]), case["vocab"], _p(out["next"][k:]))))
    return {"calls": calls, "out": out, "keep": (made, act, other, x, rows, ys)}


def prepare(case, seed):
    rt = _runtime()
    if case["kind"] == "layer":
        state = _layer_state(case, seed, rt)
    else:
        w, x = _product_inputs(case, seed, _handles(rt))
        rows, cols, t = case["rows"], case["cols"], case["tokens"]
        if case["kind"] == "product":
            y = _f32(t, rows)
            call = (rt.lib.rt_gemv_swiglu_dev, (rt.R, _p(w[0]), _p(w[1]), rows, cols, _p(x), cols, t, _p(y))) if case["pair"] else \
                (rt.lib.rt_gemm_dev, (rt.R, _p(w[0]), rows, cols, _p(x), cols, t, _p(y)))
            state = {"calls": [call], "out": {"y": y}, "keep": (w, x)}
        else:
            x = x.cpu().numpy()
            y = [np.zeros((t, rows), np.float32) for _ in w]
            handles = [c.c_void_p(a.data_ptr()) for a in w]
            px, py = x.ctypes.data_as(c.c_void_p), [a.ctypes.data_as(c.c_void_p) for a in y]
            if len(w) == 1:
                calls = [(rt.lib.rt_gemv, (rt.R, handles[0], rows, cols, px, py[0])) if t == 1 else
                         (rt.lib.rt_gemm, (rt.R, handles[0], rows, cols, px, t, py[0]))]
            else:
                calls = [(rt.lib.rt_gemm_q, (rt.R, a, rows, cols, px, t, b)) for a, b in zip(handles, py)] + [(rt.lib.rt_gemv_go, (rt.R,))]
            state = {"calls": calls, "out": {"y": y}, "keep": (w, x)}
    torch.cuda.synchronize()
    if case.get("graph"):
        calls = list(state["calls"])

        def record():
            for fn, args in calls:
                fn(*args)

        state["graph"] = _Graph(rt, record)
        state["calls"] = []
    return state


def run(state):
    if "graph" in state:
        state["graph"].launch()
    for fn, args in state["calls"]:
        fn(*args)
    return state["out"]


# ---- what a pass cannot do without


def work(case):
    def weights(rows, cols):
        return rows * cols // 32 * 34

    t = case["tokens"]
    if case["kind"] != "layer":
        n = case.get("products", 2 if case.get("pair") else 1)
        outs = 1 if case.get("pair") else n
        return {"bytes": n * weights(case["rows"], case["cols"]) + 4 * t * case["cols"] + outs * 4 * t * case["rows"],
                "flops": 2.0 * n * t * case["rows"] * case["cols"]}
    h, f, mix = case["hidden"], case["ffn"], _mix(case)
    cells = (sum(mix) + h) * h + 3 * f * h
    nbytes = case["layers"] * (weights(1, h) * (sum(mix) + h + 3 * f) + 8 * h) + 4 * t * (2 * h + sum(mix))
    flops = 2.0 * t * cells * case["layers"]
    if case["vocab"]:
        last = t if t <= 4 else 1
        nbytes += weights(case["vocab"], h) + 4 * last * case["vocab"] + t * weights(1, h)
        flops += 2.0 * last * case["vocab"] * h
    else:
        nbytes += 4 * t * h
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # F32 sums: products are measured 1.0e-7 to 1.7e-7 off the F64 answer (the fused pair's SiLU
    # included); one layer's outputs 1.2e-7 to 2.7e-7, and 24 layers' 4.7e-7, each layer's rounding
    # travelling on through the next. About four times that
    if case["kind"] != "layer":
        return {"rel": 7e-7, "max": 3e-5}
    return {"rel": 2e-6, "max": 8e-5, "differ": 0.0}


# ---- the answers in 64 bits


def _rms(x, nw):
    return nw.double() * (x * (EPS + x.square().mean(dim=1, keepdim=True)).rsqrt())


def _swiglu(g, u):
    return g / (1.0 + torch.exp(-g)) * u


def exact(case, seed):
    if case["kind"] != "layer":
        w, x = _product_inputs(case, seed, _dense)
        y = [x.double() @ a.T for a in w]
        if case.get("pair"):
            return {"y": _swiglu(*y)}
        return {"y": y if case["kind"] == "host" else y[0]}
    made = _layer_inputs(case, seed, _dense)
    h, t = case["hidden"], case["tokens"]
    x = made["head"][made["ids"]] if case["vocab"] else made["x"].double()
    for lay in made["layers"]:
        xn = _rms(x, lay["anorm"])
        mix = [xn @ w.T for w in lay["mix"]]
        mid = x + mix[0][:, :h] @ lay["out"].T
        xn = _rms(mid, lay["pnorm"])
        x = mid + _swiglu(xn @ lay["gate"].T, xn @ lay["up"].T) @ lay["down"].T
    out = {"mix": mix, "mid": mid, "x": x}
    if case["vocab"]:
        last = t if t <= 4 else 1
        out["logits"], out["next"] = _rms(x[t - last:], made["fnorm"]) @ made["head"].T, None
    return out
