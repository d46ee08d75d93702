"""What a program that uses the mHC operators has them do: the cases whose
time, outputs and accuracy this repository is measured by.

A case is one pass of a serving or a training program through the package's
public entry points (``FlagOS_mhc`` and ``torch.ops.flagos_mhc``), with its
inputs resident on the GPU.  Sizes are those of the repository's benchmark
configurations and tests, or generic ones around them: N = 4 or 8 streams (2
and 6 too for mhc_post), D from 256 to 8192, one token to 65536 tokens.

Keys of a case:
  op       what the program calls (see ``run``)
  B, S     tokens as a (B, S, N, D) batch; B = 0: S tokens as (S, N, D)
  N, D     streams and width
  dtype    of the activations; phi: of the projection (fp32 where a program
           keeps its master weight, else the activations' own type)
  clamp    logits clamped to [-clamp, clamp], 0: not clamped
  iters    Sinkhorn iterations
  layers   (op "decode") layers in the captured graph
  comp     (op "pre_train") compensated reductions over the tokens
"""

from __future__ import annotations

import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "flagos-mhc_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

_DT = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
_SIZE = {"bf16": 2, "f16": 2, "f32": 4}
_NORM_EPS = _HC_EPS = 1e-6


def _case(name, op, B, S, N, D, dtype="bf16", phi="bf16", clamp=10.0, iters=20, layers=1, comp=False):
    c = dict(op=op, B=B, S=S, N=N, D=D, dtype=dtype, phi=phi, clamp=clamp, iters=iters, layers=layers, comp=comp)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # one token of a decoding loop: the mHC operators of four layers, replayed from a HIP graph as a
        # server does where launches would dominate; phi kept in fp32
        _case("decode_t1", "decode", 0, 1, 4, 7168, phi="f32", layers=4),
        # a decoding batch of 64 sequences, called eagerly
        _case("decode_t64", "infer", 64, 1, 4, 7168),
        # a short prompt of odd length, phi in fp32
        _case("prefill_short", "infer", 0, 777, 4, 4096, phi="f32", clamp=3.0),
        # a packed batch of prompts between two sublayers: mhc_post of one layer and the pre operator of
        # the next in one call
        _case("prefill_fused", "fused_infer", 0, 5999, 4, 5120),
        # the reference's training forward, which keeps every tensor that its backward takes, x_scaled too
        _case("pre_fwd_saved", "pre_full", 4, 4096, 4, 4096),
        # training through autograd: the pre operator with eight streams
        _case("pre_train_n8", "pre_train", 4, 8192, 8, 2048),
        # the pre operator with an fp32 master phi, a width between the powers of two, ragged tokens
        _case("pre_train_phi32", "pre_train", 3, 2731, 4, 3584, phi="f32", clamp=3.0),
        # training through autograd: the post operator
        _case("post_train", "post_train", 4, 4096, 4, 4096),
        # a small fp32 model: one mHC layer, forward and backward
        _case("layer_train_f32", "layer_train", 1, 1024, 4, 256, dtype="f32", phi="f32"),
        # one mHC layer in fp16, odd sizes: rows that are no multiple of 16 bytes wide
        _case("layer_train_f16", "layer_train", 0, 2049, 4, 1003, dtype="f16", phi="f16", clamp=0.0),
        # a layer of a stack, forward and backward, post and pre fused
        _case("fused_train", "fused_train", 2, 8192, 4, 7168),
        # the benchmark's chain: all four operators over a large batch
        _case("chain_large", "chain", 8, 8192, 4, 7168),
    ]


#: tokens that each op sees
_TOKENS = {"decode": (1, 256), "infer": (1, 16384), "fused_infer": (1, 16384), "pre_full": (64, 32768),
           "pre_train": (256, 65536), "post_train": (256, 65536), "layer_train": (256, 32768),
           "fused_train": (256, 32768), "chain": (1024, 65536)}


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(sorted(_TOKENS))
    N = rng.choice((4, 4, 4, 8) if op != "post_train" else (2, 4, 4, 6, 8))
    width = rng.random()
    D = _log_uniform(rng, 256, 8192)
    if width < 0.65:
        D = max(256, D // 128 * 128)   # what models have
    elif width < 0.85:
        D = D // 8 * 8
    dtype = rng.choice(("bf16", "bf16", "bf16", "bf16", "f16", "f32"))
    phi = "f32" if rng.random() < 0.3 else dtype
    lo, hi = _TOKENS[op]
    # large batches are in bf16; the other types stand for smaller runs
    most = (1 << 30 if dtype == phi == "bf16" else 1 << 28 if dtype == "bf16" else 1 << 26) // (N * D)
    T = max(1, _log_uniform(rng, min(lo, max(1, most)), max(1, min(hi, most))))
    B = 0 if rng.random() < 0.5 else rng.choice((1, 2, 3, 4, 8))
    S = T if B == 0 else max(1, T // B)
    clamp = rng.choice((0.0, 3.0, 10.0))
    iters = rng.choice((20, 20, 20, 10, 5, 33))
    layers = rng.choice((2, 4, 8)) if op == "decode" else 1
    comp = op == "pre_train" and rng.random() < 0.2
    return _case(None, op, B, S, N, D, dtype, phi, clamp, iters, layers, comp)


def _tokens(c):
    return c["S"] * max(1, c["B"])


def _kw(c):
    return dict(norm_eps=_NORM_EPS, hc_eps=_HC_EPS, clamp_min=-c["clamp"], clamp_max=c["clamp"],
                iter_times=c["iters"])


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
_PRE = ("decode", "infer", "pre_full", "pre_train", "layer_train", "chain", "fused_infer", "fused_train")


def _inputs(c, seed):
    """The tensors of a case, from the seed alone: normal activations and
    upstream gradients, phi of unit-variance mixes, gates as the pre operator
    makes them (a doubly stochastic h_res, h_post in (0, 2))."""
    T, N, D, op = _tokens(c), c["N"], c["D"], c["op"]
    M = 2 * N + N * N
    dt, dev = _DT[c["dtype"]], torch.device("cuda")
    lead = (T,) if c["B"] == 0 else (c["B"], c["S"])
    g = torch.Generator(device=dev)
    g.manual_seed(int(seed))

    def normal(*shape, dtype=torch.float32, scale=1.0):
        t = torch.randn(*shape, device=dev, generator=g)
        return (t.mul_(scale) if scale != 1.0 else t).to(dtype)

    s = {"x": normal(*lead, N, D, dtype=dt)}
    if op in _PRE:
        s["phi"] = [normal(M, N * D, dtype=_DT[c["phi"]], scale=(N * D) ** -0.5) for _ in range(c["layers"])]
        s["alpha"] = [torch.tensor([0.5, 0.5, 1.0], device=dev) for _ in range(c["layers"])]
        s["base"] = [normal(M, scale=0.1) for _ in range(c["layers"])]
    if op in ("post_train", "fused_infer", "fused_train"):
        h = torch.softmax(normal(*lead, N, N), dim=-1)
        for _ in range(5):
            h = h / h.sum(dim=-2, keepdim=True)
            h = h / h.sum(dim=-1, keepdim=True)
        s["h_res"] = h
        s["h_post"] = 2 * torch.sigmoid(normal(*lead, N))
    if op in ("post_train", "fused_infer", "fused_train", "infer", "chain"):
        s["h_out"] = normal(*lead, D, dtype=dt)
    if op in ("post_train", "layer_train", "chain", "fused_train"):
        s["g_next"] = normal(*lead, N, D, dtype=dt)
    if op in ("pre_train", "fused_train"):
        s["g_y"] = normal(*lead, D, dtype=dt)
        s["g_post"] = normal(T, N)
        s["g_comb"] = normal(T, N, N)
    return s


_LEAVES = {"pre_train": ("x",), "post_train": ("x", "h_res", "h_out", "h_post"), "layer_train": ("x",),
           "fused_train": ("x", "h_res", "h_out", "h_post")}


def _layers(m, s, kw):
    """The mHC operators of a stack of layers whose sublayers pass y on."""
    x, outs = s["x"], []
    for phi, alpha, base in zip(s["phi"], s["alpha"], s["base"]):
        out = m.mhc_pre_clamp_sinkhorn(x, phi, alpha, base, **kw)
        x = m.mhc_post(x, out["comb_frag"], out["y"], out["post_out"])
        outs += [out["y"], out["comb_frag"]]
    return [x] + outs


def prepare(case, seed):
    import FlagOS_mhc as m

    s = _inputs(case, seed)
    s["case"], s["m"] = case, m
    op = case["op"]
    if op in _LEAVES:
        s["leaves"] = [s[k].requires_grad_(True) for k in _LEAVES[op]]
        if op in _PRE:
            s["leaves"] += [s[k][0].requires_grad_(True) for k in ("phi", "alpha", "base")]
    if op == "decode":
        kw = _kw(case)
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _layers(m, s, kw)
        torch.cuda.current_stream().wait_stream(side)
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            s["outs"] = _layers(m, s, kw)
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(s):
    c, m = s["case"], s["m"]
    kw, op = _kw(c), c["op"]
    x = s["x"]
    if op == "decode":
        s["graph"].replay()
        return s["outs"]
    if op == "post_train":
        out = m.mhc_post_fn(x, s["h_res"], s["h_out"], s["h_post"])
        return [out.detach(), *torch.autograd.grad(out, s["leaves"], s["g_next"])]
    if op in _PRE:
        phi, alpha, base = s["phi"][0], s["alpha"][0], s["base"][0]
    if op == "infer":
        out = m.mhc_pre_clamp_sinkhorn(x, phi, alpha, base, **kw)
        return [out["y"], out["post_out"], out["comb_frag"],
                m.mhc_post(x, out["comb_frag"], s["h_out"], out["post_out"])]
    if op == "fused_infer":
        x_next, out = m.mhc_post_pre_clamp_sinkhorn(x, s["h_res"], s["h_out"], s["h_post"], phi, alpha, base, **kw)
        return [x_next, out["y"], out["post_out"], out["comb_frag"]]
    if op == "pre_full":
        out = m.mhc_pre_clamp_sinkhorn(x, phi, alpha, base, need_backward=True, **kw)
        return [out[k] for k in ("y", "post_out", "comb_frag", "inv_rms", "x_scaled", "mixes", "h_res_logits", "pre")]
    if op == "pre_train":
        out = m.mhc_pre_clamp_sinkhorn_fn(x, phi, alpha, base, **kw, compensated=c["comp"])
        return [t.detach() for t in out] + list(
            torch.autograd.grad(out, s["leaves"], (s["g_y"], s["g_post"], s["g_comb"])))
    if op == "layer_train":
        y, post_out, comb = m.mhc_pre_clamp_sinkhorn_fn(x, phi, alpha, base, **kw)
        out = m.mhc_post_fn(x, comb, y, post_out)
        return [out.detach(), *torch.autograd.grad(out, s["leaves"], s["g_next"])]
    if op == "fused_train":
        out = m.mhc_post_pre_clamp_sinkhorn_fn(x, s["h_res"], s["h_out"], s["h_post"], phi, alpha, base, **kw)
        return [t.detach() for t in out] + list(
            torch.autograd.grad(out, s["leaves"], (s["g_next"], s["g_y"], s["g_post"], s["g_comb"])))
    ops = torch.ops.flagos_mhc
    scal = (_NORM_EPS, _HC_EPS, -c["clamp"], c["clamp"], c["iters"])
    y, post_out, comb, inv, mixes, pre = ops.mhc_pre_clamp_sinkhorn(x, phi, alpha, base, *scal)
    x_next = ops.mhc_post(x, comb, s["h_out"], post_out)
    gx, g_res, g_out, g_post = ops.mhc_post_backward(s["g_next"], x, comb, s["h_out"], post_out)
    grads = ops.mhc_pre_clamp_sinkhorn_backward(x, phi, alpha, base, inv, mixes, pre, g_out, g_post, g_res, *scal)
    return [y, post_out, comb, x_next, gx, g_res, g_out, g_post, *grads]


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def work(c):
    """Every call's inputs read once and its outputs written once (a forward
    and a backward are two calls), and its multiply-adds."""
    T, N, D, op = _tokens(c), c["N"], c["D"], c["op"]
    b, M, ND = _SIZE[c["dtype"]], 2 * N + N * N, N * D
    phi = M * ND * _SIZE[c["phi"]]
    gates, saved = 4 * (N * N + N), 4 * (1 + M + N)
    f = {
        "pre_infer": T * ((ND + D) * b + gates) + phi,
        "pre_fwd": T * ((ND + D) * b + gates + saved) + phi,
        "pre_full": T * ((ND + D) * b + gates + saved + 4 * N * N + 4 * ND) + phi,
        "pre_bwd": T * ((2 * ND + D) * b + gates + saved) + phi + M * ND * 4,
        "post_fwd": T * ((2 * ND + D) * b + gates),
        "post_bwd": T * ((3 * ND + 2 * D) * b + 2 * gates),
        # x and h_out in, x_next and y out
        "fused_infer": T * ((2 * ND + 2 * D) * b + 2 * gates) + phi,
        "fused_fwd": T * ((2 * ND + 2 * D) * b + 2 * gates + saved) + phi,
        # x_next's gradient, x, x_next, h_out and grad_y in, grad_x and grad_h_out out
        "fused_bwd": T * ((4 * ND + 3 * D) * b + 3 * gates + saved) + phi + M * ND * 4,
    }
    m = {"pre": 2 * T * ND * (M + 2), "pre_bwd": 4 * T * ND * (M + 2), "post": 2 * T * ND * (N + 1),
         "post_bwd": 4 * T * ND * (N + 1)}
    calls = {
        "decode": ("pre_infer", "post_fwd"), "infer": ("pre_infer", "post_fwd"), "fused_infer": ("fused_infer",),
        "pre_full": ("pre_full",), "pre_train": ("pre_fwd", "pre_bwd"), "post_train": ("post_fwd", "post_bwd"),
        "layer_train": ("pre_fwd", "post_fwd", "post_bwd", "pre_bwd"), "fused_train": ("fused_fwd", "fused_bwd"),
        "chain": ("pre_fwd", "post_fwd", "post_bwd", "pre_bwd"),
    }[op]
    flops = 0
    if op != "post_train":
        flops += m["pre"] + (m["pre_bwd"] if op in ("pre_train", "layer_train", "fused_train", "chain") else 0)
    if op not in ("pre_full", "pre_train"):
        flops += m["post"] + (m["post_bwd"] if op in ("post_train", "layer_train", "fused_train", "chain") else 0)
    return {"bytes": c["layers"] * sum(f[k] for k in calls), "flops": c["layers"] * flops}


def tolerance(c):
    """About four times the error against 64 bits: one rounding of an output
    costs 1.7e-3 in bf16 and 2.5e-4 in fp16 (2-norm), the gradients that take
    a rounded intermediate up to 3.3e-3, a stack of layers up to 3.3e-3 after
    four; fp32 sums and bf16 planes of fp32 operands up to 4.4e-6."""
    rel = {"bf16": 1e-2, "f16": 1.5e-3, "f32": 2e-5}[c["dtype"]]
    return {"rel": 1.5 * rel if c["op"] == "decode" else rel}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def _pre64(x, phi, alpha, base, c):
    T, N, D = x.shape
    x2 = x.reshape(T, N * D)
    inv = torch.rsqrt(x2.square().mean(dim=-1, keepdim=True) + _NORM_EPS)
    mixes = (x2 @ phi.t()) * inv
    pre = torch.sigmoid(mixes[:, :N] * alpha[0] + base[:N]) + _HC_EPS
    post = 2 * torch.sigmoid(mixes[:, N:2 * N] * alpha[1] + base[N:2 * N])
    logits = (mixes[:, 2 * N:] * alpha[2] + base[2 * N:]).reshape(T, N, N)
    h = logits.clamp(-c["clamp"], c["clamp"]) if c["clamp"] else logits
    h = torch.softmax(h, dim=-1) + _HC_EPS
    h = h / (h.sum(dim=-2, keepdim=True) + _HC_EPS)
    for _ in range(c["iters"] - 1):
        h = h / (h.sum(dim=-1, keepdim=True) + _HC_EPS)
        h = h / (h.sum(dim=-2, keepdim=True) + _HC_EPS)
    y = sum(pre[:, n:n + 1] * x[:, n] for n in range(N))
    return {"y": y, "post_out": post, "comb_frag": h, "inv_rms": inv[:, 0], "x_scaled": x2 * inv, "mixes": mixes,
            "h_res_logits": logits, "pre": pre}


def _post64(x, h_res, h_out, h_post):
    N = x.shape[1]
    return torch.stack([sum(h_res[:, j, i, None] * x[:, j] for j in range(N)) + h_post[:, i, None] * h_out
                        for i in range(N)], dim=1)


def exact(case, seed):
    c, op = case, case["op"]
    s = _inputs(case, seed)
    T, N, D = _tokens(c), c["N"], c["D"]
    flat = {"x": (T, N, D), "h_res": (T, N, N), "h_post": (T, N), "h_out": (T, D), "g_next": (T, N, D),
            "g_y": (T, D), "g_post": (T, N), "g_comb": (T, N, N)}
    weights = [[t.double() for t in w] for w in zip(s["phi"], s["alpha"], s["base"])] if op in _PRE else []
    train = op in _LEAVES
    rows, sums = [], None
    step = max(1, (1 << 26) // (N * D))
    for a in range(0, T, step):
        t = {k: s[k].reshape(flat[k])[a:a + step].double() for k in flat if k in s}
        leaves = [t[k].requires_grad_(True) for k in _LEAVES.get(op, ())]
        w = [v.detach().requires_grad_(train or op == "chain") for v in weights[0]] if weights else []
        x, red = t["x"], []
        if op == "decode":
            outs = []
            for phi, alpha, base in weights:
                o = _pre64(x, phi, alpha, base, c)
                x = _post64(x, o["comb_frag"], o["y"], o["post_out"])
                outs += [o["y"], o["comb_frag"]]
            row = [x] + outs
        elif op == "infer":
            o = _pre64(x, *w, c)
            row = [o["y"], o["post_out"], o["comb_frag"], _post64(x, o["comb_frag"], t["h_out"], o["post_out"])]
        elif op == "pre_full":
            o = _pre64(x, *w, c)
            row = [o[k] for k in ("y", "post_out", "comb_frag", "inv_rms", "x_scaled", "mixes", "h_res_logits", "pre")]
        elif op == "post_train":
            out = _post64(x, t["h_res"], t["h_out"], t["h_post"])
            row = [out, *torch.autograd.grad(out, leaves, t["g_next"])]
        elif op in ("fused_infer", "fused_train"):
            x_next = _post64(x, t["h_res"], t["h_out"], t["h_post"])
            o = _pre64(x_next, *w, c)
            row = [x_next, o["y"], o["post_out"], o["comb_frag"]]
            if train:
                grads = torch.autograd.grad(row, leaves + w, (t["g_next"], t["g_y"], t["g_post"], t["g_comb"]))
                row, red = row + list(grads[:4]), grads[4:]
        elif op == "pre_train":
            o = _pre64(x, *w, c)
            row = [o["y"], o["post_out"], o["comb_frag"]]
            grads = torch.autograd.grad(row, leaves + w, (t["g_y"], t["g_post"], t["g_comb"]))
            row, red = row + [grads[0]], grads[1:]
        elif op == "layer_train":
            o = _pre64(x, *w, c)
            out = _post64(x, o["comb_frag"], o["y"], o["post_out"])
            grads = torch.autograd.grad(out, leaves + w, t["g_next"])
            row, red = [out, grads[0]], grads[1:]
        else:
            o = _pre64(x.requires_grad_(True), *w, c)
            v = {k: o[k].detach().requires_grad_(True) for k in ("comb_frag", "post_out")}
            xp, ho = x.detach().requires_grad_(True), t["h_out"].requires_grad_(True)
            x_next = _post64(xp, v["comb_frag"], ho, v["post_out"])
            gx, g_res, g_out, g_post = torch.autograd.grad(x_next, (xp, v["comb_frag"], ho, v["post_out"]),
                                                           t["g_next"])
            grads = torch.autograd.grad([o["y"], o["post_out"], o["comb_frag"]], [x] + w, (g_out, g_post, g_res))
            row = [o["y"], o["post_out"], o["comb_frag"], x_next, gx, g_res, g_out, g_post, grads[0]]
            red = grads[1:]
        rows.append([v.detach() for v in row])
        sums = [p + q for p, q in zip(sums, red)] if sums else list(red)
    outs = [torch.cat(parts) if len(parts) > 1 else parts[0] for parts in map(list, zip(*rows))]
    return outs + (sums or [])
