"""The calls this library is timed on.

A user of the library runs the linear layers of a model with low-precision
weights: the weights are quantised and laid out once, every call quantises its
bf16 activations on the GPU and multiplies. The cases are such layers in each
scale mode (MXFP8, MXFP4, DeepSeek block scale, per-tensor), the product on
resident operands (the library's headline figure), the backward product with
E5M2 gradients, and the bf16 split-K product, from a few rows (decode) over a
prefill chunk of any length to whole training batches. Sizes are those of the
benchmark's configurations; draw() spreads the rows over 1 to 8192 and adds
widths that are no multiple of a tile.

prepare() holds what a program keeps between calls (activations, prepared
weights, kernel handles, a workspace slot), run() is one call, exact() the same
product in 64 bits from plain torch.
"""
import math

import torch

from gcnasm_amd import f4gemm, flatmm_splitk, ops, opus_gemm

# The largest drawn product costs no more than the largest listed one.
MAX_FLOPS = 2.0 * 8192 ** 3

# (N, K) of weights: the benchmark's MX, DeepSeek and square configurations,
# and widths that leave remainders in every tile.
MX_WEIGHTS = [(28672, 8192), (8192, 28672), (8192, 8192), (4096, 4096), (2048, 2048),
              (10240, 8192), (5120, 5120), (3072, 1024), (13824, 5120), (1040, 4096)]
DEEPSEEK_WEIGHTS = [(7168, 2048), (2112, 7168), (24576, 1536), (8192, 8192), (4096, 4096),
                    (2048, 2048), (7168, 4608), (1000, 1024), (3080, 1536)]
SPLITK_WEIGHTS = [(512, 7168), (7168, 2048), (256, 7168), (1024, 4096), (576, 7168), (2048, 2048),
                  (1000, 1000)]


def listed():
    return [
        # The headline: a square MXFP8 product on operands already in memory.
        {"name": "mx8_gemm_8192", "kind": "mx_gemm", "fmt": "e4m3", "m": 8192, "n": 8192,
         "k": 8192, "split": 0},
        # The smallest configuration: a call whose launches and latency are all of it.
        {"name": "mx8_layer_256x256x512", "kind": "mx_layer", "fmt": "e4m3", "m": 256, "n": 256,
         "k": 512, "split": 0},
        # Decode of a 16-sequence batch: the up projection, bound by reading the weights.
        {"name": "mx8_layer_16x28672x8192", "kind": "mx_layer", "fmt": "e4m3", "m": 16,
         "n": 28672, "k": 8192, "split": 0},
        # Decode of a 64-sequence batch: the down projection, with the split the library picks.
        {"name": "mx8_layer_64x8192x28672", "kind": "mx_layer", "fmt": "e4m3", "m": 64,
         "n": 8192, "k": 28672, "split": -1},
        # Prefill of a prompt whose length is no multiple of anything.
        {"name": "mx8_layer_1000x8192x8192", "kind": "mx_layer", "fmt": "e4m3", "m": 1000,
         "n": 8192, "k": 8192, "split": 0},
        # Prefill with MXFP4 weights and activations.
        {"name": "mx4_layer_2048x8192x8192", "kind": "mx_layer", "fmt": "e2m1", "m": 2048,
         "n": 8192, "k": 8192, "split": 0},
        # Backward: E5M2 gradients times E4M3 weights (the input's gradient).
        {"name": "mx8_dgrad_4096", "kind": "mx_dgrad", "fmt": "e5m2", "m": 4096, "n": 4096,
         "k": 4096, "split": 0},
        # DeepSeek prefill, 4096 tokens.
        {"name": "bs_layer_4096x7168x2048", "kind": "bs_layer", "out": "bf16", "m": 4096,
         "n": 7168, "k": 2048, "group_n": 128},
        # DeepSeek prefill of a short prompt, few columns and a long K.
        {"name": "bs_layer_300x2112x7168", "kind": "bs_layer", "out": "bf16", "m": 300,
         "n": 2112, "k": 7168, "group_n": 128},
        # DeepSeek decode of a 32-sequence batch.
        {"name": "bs_layer_32x7168x2048", "kind": "bs_layer", "out": "bf16", "m": 32, "n": 7168,
         "k": 2048, "group_n": 128},
        # Per-tensor FP8: one scale for the activations, one for the weights.
        {"name": "pt_layer_4096", "kind": "pt_layer", "out": "bf16", "m": 4096, "n": 4096,
         "k": 4096},
        # bf16 split-K at its driver's default problem.
        {"name": "bf16_splitk_1024x512x7168", "kind": "bf16_splitk", "m": 1024, "n": 512,
         "k": 7168, "split_k": 2, "bias": False},
    ]


def _rows(rng, cap):
    """Rows over 1 .. 8192 by their logarithm, at most cap, odd ones among them."""
    m = int(round(2.0 ** rng.uniform(0.0, 13.0)))
    return max(1, min(m, int(cap), 8192))


def draw(rng):
    kind = rng.choice(["mx_gemm", "mx_layer", "mx_layer", "mx_layer", "mx_dgrad", "bs_layer",
                       "bs_layer", "bs_layer", "pt_layer", "bf16_splitk"])
    if kind in ("mx_gemm", "mx_layer", "mx_dgrad"):
        n, k = rng.choice(MX_WEIGHTS)
        if rng.random() < 0.3:
            n = 16 * int(round(2.0 ** rng.uniform(2.0, 10.0)))
        m = _rows(rng, MAX_FLOPS / (2.0 * n * k))
        fmt = "e5m2" if kind == "mx_dgrad" else rng.choice(["e4m3", "e4m3", "e2m1"])
        split = -1 if kind == "mx_layer" and m <= 64 and rng.random() < 0.5 else 0
        return {"kind": kind, "fmt": fmt, "m": m, "n": n, "k": k, "split": split}
    if kind in ("bs_layer", "pt_layer"):
        n, k = rng.choice(DEEPSEEK_WEIGHTS)
        if rng.random() < 0.3:
            n = 8 * int(round(2.0 ** rng.uniform(4.0, 10.0)))
        m = _rows(rng, MAX_FLOPS / (2.0 * n * k))
        c = {"kind": kind, "out": rng.choice(["bf16", "bf16", "f32"]), "m": m, "n": n, "k": k}
        if kind == "bs_layer":
            c["group_n"] = rng.choice([128, 128, 128, 1])
        return c
    n, k = rng.choice(SPLITK_WEIGHTS)
    return {"kind": kind, "m": _rows(rng, 8192), "n": n, "k": k,
            "split_k": rng.choice([1, 2, 2, 3, 4, 8]), "bias": rng.random() < 0.5}


# ---- inputs --------------------------------------------------------------------

def _randn(shape, seed, which, std=1.0):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 16 + which)
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32) * std


def _inputs(case, seed):
    """Activations (or gradients) [M, K] and weights [N, K], bf16: N(0, 1) and
    N(0, 0.02), activations with a few channels eight times as large, as a
    model's are; the headline product keeps the benchmark's per-block spread."""
    m, n, k = case["m"], case["n"], case["k"]
    x, w = _randn((m, k), seed, 0), _randn((n, k), seed, 1)
    if case["kind"] == "mx_gemm":
        for t, which in ((x, 2), (w, 3)):
            g = torch.Generator(device="cuda")
            g.manual_seed(seed * 16 + which)
            u = torch.randint(-4, 5, (t.shape[0], k // 32, 1), generator=g, device="cuda")
            t.view(t.shape[0], k // 32, 32).mul_(torch.pow(2.0, u.float()))
    elif case["kind"] == "bf16_splitk":
        w.mul_(0.02)
    else:
        w.mul_(0.02)
        x.view(m, k)[:, ::64].mul_(8.0)
    return x.to(torch.bfloat16), w.to(torch.bfloat16)


def prepare(case, seed):
    x, w = _inputs(case, seed)
    kind, m, n, k = case["kind"], case["m"], case["n"], case["k"]
    s = {"case": case, "x": x}
    if kind in ("mx_gemm", "mx_layer"):
        mx4 = case["fmt"] == "e2m1"
        s["w"] = (ops.prepare_mx4_b if mx4 else ops.prepare_mx_b)(w)
        if kind == "mx_gemm":
            s["a"] = (ops.prepare_mx4_a if mx4 else ops.prepare_mx_a)(x)
            del s["x"]
    elif kind == "mx_dgrad":
        s["w"] = ops.prepare_mx_b(w)
        sh = f4gemm.Shape(m, n, k)
        cfgs = f4gemm.manifest()
        idx, l2 = f4gemm.select_kernel(m, n, k, 256, 0, 1)
        s["shape"] = sh
        s["kernel"] = f4gemm.Kernel().load(None, cfgs[idx])
        s["launch"] = f4gemm.make_launch(cfgs[idx], m, n, k, l2)
    elif kind == "bs_layer":
        if case["group_n"] == 128:
            s["w"], s["sw"] = ops.quant_fp8_128x128(w)
        else:
            s["w"], s["sw"] = ops.quant_fp8_1x128(w)
    elif kind == "pt_layer":
        s["w"], s["sw"] = ops.quant_fp8_per_tensor(w)
    else:
        s["w"] = w
        s["bias"] = _randn((n,), seed, 4).to(torch.bfloat16) if case["bias"] else None
        pad = flatmm_splitk.WS_PAD
        rows, cols = -(-m // pad) * pad, -(-n // pad) * pad
        s["handle"] = _Slot(case["split_k"] * rows * cols * 4)
    return s


class _Slot(flatmm_splitk.WorkspaceHandle):
    """A workspace slot given back with the state that holds it."""

    def __del__(self):
        self.close()


def _dtype(case):
    return torch.float32 if case["out"] == "f32" else torch.bfloat16


# ---- one call --------------------------------------------------------------------

def run(state):
    case = state["case"]
    kind, m, n, k = case["kind"], case["m"], case["n"], case["k"]
    if kind == "mx_gemm":
        gemm = ops.mxfp4_gemm if case["fmt"] == "e2m1" else ops.mxfp8_gemm
        return gemm(state["a"], state["w"], log2_k_split=case["split"])[0][:m]
    if kind == "mx_layer":
        if case["fmt"] == "e2m1":
            a = ops.prepare_mx4_a(state["x"])
            return ops.mxfp4_gemm(a, state["w"], log2_k_split=case["split"])[0][:m]
        a = ops.prepare_mx_a(state["x"])
        return ops.mxfp8_gemm(a, state["w"], log2_k_split=case["split"])[0][:m]
    if kind == "mx_dgrad":
        sh, ld, w = state["shape"], state["launch"], state["w"]
        q, s = ops.quant_mx8(state["x"], 1)
        ss = ops.shuffle_scale(s, sh.scale_a_rows(), sh.scale_cols())
        out = torch.empty((m, n), dtype=torch.bfloat16, device=q.device)
        args = f4gemm.fill_args(out, None, q, w.codes, ss, w.scales, m, n, k, n, sh.scale_cols(),
                                sh.scale_cols(), 1.0, 0.0, ld.log2_k_split)
        state["kernel"].launch(args, ld.gdx, ld.gdy, ld.gdz, fmt_a=1)
        return out
    if kind == "bs_layer":
        q, s = ops.quant_fp8_1x128(state["x"])
        out = torch.empty((m, n), dtype=_dtype(case), device=q.device)
        return opus_gemm.blockscale_gemm(q, state["w"], s, state["sw"], out,
                                         group_n=case["group_n"])
    if kind == "pt_layer":
        q, s = ops.quant_fp8_per_tensor(state["x"])
        out = torch.empty((m, n), dtype=_dtype(case), device=q.device)
        return opus_gemm.per_tensor_gemm(q, state["w"], s, state["sw"], out)
    out = torch.empty((m, n), dtype=torch.bfloat16, device=state["x"].device)
    return flatmm_splitk.splitk_gemm(state["x"], state["w"], out, case["split_k"],
                                     state["handle"], bias=state["bias"])


def work(case):
    kind, m, n, k = case["kind"], case["m"], case["n"], case["k"]
    flops = 2.0 * m * n * k
    if kind == "bf16_splitk":
        return {"bytes": 2.0 * (m * k + n * k + m * n), "flops": flops}
    out = 4 if case.get("out") == "f32" else 2
    el = 0.5 if case.get("fmt") == "e2m1" else 1.0
    scales = {"mx_gemm": n * k / 32, "mx_layer": n * k / 32, "mx_dgrad": n * k / 32,
              "pt_layer": 4}.get(kind)
    if scales is None:  # fp32 block scales of the weights
        scales = 4.0 * (math.ceil(n / 128) if case["group_n"] == 128 else n) * (k // 128)
    x = m * k * el + m * k / 32 if kind == "mx_gemm" else 2.0 * m * k
    return {"bytes": x + n * k * el + scales + out * m * n, "flops": flops}


def tolerance(case):
    # Four times what exact() shows. bf16 outputs: one rounding to 8 significant
    # bits, 1.7e-3 in the 2-norm, and one unit in the last place at most, 2^-7.
    # fp32 outputs keep what the FP8 matrix instruction leaves (products cut 13
    # bits below the largest of their eight): 2.2e-5 in the 2-norm.
    if case.get("out") == "f32":
        return {"rel": 9e-5, "max": 1e-3}
    return {"rel": 7e-3, "max": 3e-2}


# ---- the same in 64 bits -----------------------------------------------------------

def _pow2(e):
    return torch.pow(2.0, e.double())


_E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)


def _mx_values(x, fmt):
    """What x stands for after MX quantisation along K: per 1x32 block the scale
    2^floor(log2(amax / max)), elements rounded to nearest even, saturated."""
    top, frac, emax = {"e4m3": (448.0, 1.75, 8), "e5m2": (57344.0, 1.75, 15),
                       "e2m1": (6.0, 1.5, 2)}[fmt]
    v = x.float().view(x.shape[0], -1, 32)
    mant, e = torch.frexp(v.abs().amax(dim=2, keepdim=True).double())  # mant in [0.5, 1)
    e = torch.where(2.0 * mant >= frac, e - 1 - emax, e - 2 - emax)
    e = torch.where(mant == 0, torch.full_like(e, -127), e).clamp(-127, 127)
    t = (v.double() * _pow2(-e)).clamp(-top, top).float()
    if fmt == "e2m1":
        codes = torch.tensor(_E2M1, device=x.device)
        mid = (codes[:-1] + codes[1:]) / 2
        a = t.abs()
        lo = torch.bucketize(a, mid, right=False)  # a midpoint goes down ...
        hi = torch.bucketize(a, mid, right=True)   # ... or up, to the even code
        q = torch.copysign(codes[torch.where(lo % 2 == 0, lo, hi)], t)
    else:
        q = t.to(torch.float8_e4m3fn if fmt == "e4m3" else torch.float8_e5m2).float()
    return (q.double() * _pow2(e)).view(x.shape)


def _fp8_values(x, s):
    """x quantised to E4M3 with the fp32 scale s (broadcast against x), in 64 bits."""
    t = (x.double() / s.double()).float().clamp(-448.0, 448.0)
    return t.to(torch.float8_e4m3fn).float().double() * s.double()


def _scale(amax):
    s = (amax.double() / 448.0).float()
    return torch.where(amax > 0, s, torch.ones_like(s))


def _row_block_values(x):
    v = x.float().view(x.shape[0], -1, 128)
    return _fp8_values(v, _scale(v.abs().amax(dim=2, keepdim=True))).view(x.shape)


def _tile_values(w):
    n, k = w.shape
    pad = -n % 128
    v = torch.nn.functional.pad(w.float(), (0, 0, 0, pad)).view((n + pad) // 128, 128, k // 128,
                                                                128)
    q = _fp8_values(v, _scale(v.abs().amax(dim=(1, 3), keepdim=True)))
    return q.reshape(n + pad, k)[:n]


def exact(case, seed):
    x, w = _inputs(case, seed)
    kind = case["kind"]
    if kind == "mx_dgrad":
        return _mx_values(x, "e5m2") @ _mx_values(w, "e4m3").t()
    if kind in ("mx_gemm", "mx_layer"):
        return _mx_values(x, case["fmt"]) @ _mx_values(w, case["fmt"]).t()
    if kind == "bs_layer":
        wv = _tile_values(w) if case["group_n"] == 128 else _row_block_values(w)
        return _row_block_values(x) @ wv.t()
    if kind == "pt_layer":
        xf, wf = x.float(), w.float()
        return _fp8_values(xf, _scale(xf.abs().amax())) @ _fp8_values(wf, _scale(wf.abs().amax())).t()
    y = x.double() @ w.double().t()
    return y + _randn((case["n"],), seed, 4).to(torch.bfloat16).double() if case["bias"] else y
