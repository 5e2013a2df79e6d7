"""The work users of this package have it do, as cases that can be timed and checked.

A case is one call (or one training step) through the package's public entry
points: ``MHCLiteBlock`` and the ``torch.ops.flash_mhc`` operators.  Kinds:

  eval          MHCLiteBlock forward without autograd (decoding, prefill)
  train         MHCLiteBlock forward + backward: output and every gradient
  project       fused_rmsnorm_project (K1) forward + backward with grad_W
  pre_map       mhc_pre_map forward (K1, K2, K3 as one op)
  pre_map_bwd   mhc_pre_map_backward, with post-res's gradient of x coming in
  mix           fused_pre_map (K3) forward + backward
  post_res      fused_post_res (K4) forward
  post_res_bwd  fused_post_res_backward

``graph`` replays the call from a HIP graph, as a serving loop or a captured
training step does; otherwise the call is made eagerly.  ``rms`` gives the
block its learnable RMSNorm weight.  Everything is bf16 with n = 4 streams,
the only inputs the fused path takes.
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import torch
import torch.nn as nn

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "flash-mhc_amd"))

import flash_mhc  # noqa: E402

BF16 = torch.bfloat16
F64 = torch.float64
N = 4
D = 32  # 2 n + n!
EPS = 1e-6  # K1's RMSNorm epsilon
DEV = "cuda"

KINDS = ("eval", "train", "project", "pre_map", "pre_map_bwd", "mix", "post_res", "post_res_bwd")


def listed():
    return [
        # Decoding one token at the training width, called eagerly: host and launch latency.
        {"name": "eval_T1_C4096", "kind": "eval", "T": 1, "C": 4096, "graph": False, "rms": False},
        # A decoding batch in a serving loop, replayed from a graph: kernel latency.
        {"name": "eval_T64_C4096_graph", "kind": "eval", "T": 64, "C": 4096, "graph": True, "rms": False},
        # A prompt of ragged length at the reference benchmark's default width, replayed from a graph.
        {"name": "eval_T1003_C2560_graph", "kind": "eval", "T": 1003, "C": 2560, "graph": True, "rms": False},
        # A small captured training step.
        {"name": "train_T4096_C1024_graph", "kind": "train", "T": 4096, "C": 1024, "graph": True, "rms": False},
        # The full training step of the block configuration, RMSNorm weight included.
        {"name": "train_T65536_C2048", "kind": "train", "T": 65536, "C": 2048, "graph": False, "rms": True},
        # A training step of a small model whose width is not a multiple of eight, ragged batch.
        {"name": "train_T20011_C300", "kind": "train", "T": 20011, "C": 300, "graph": False, "rms": False},
        # K1 alone, both directions, at the training width.
        {"name": "project_T16384_C4096", "kind": "project", "T": 16384, "C": 4096},
        # The pre-map region at the microbenchmark's size, each direction.
        {"name": "pre_map_T65536_C1024", "kind": "pre_map", "T": 65536, "C": 1024},
        {"name": "pre_map_bwd_T65536_C1024", "kind": "pre_map_bwd", "T": 65536, "C": 1024},
        # K3 alone, both directions, at an odd width and token count.
        {"name": "mix_T30011_C1001", "kind": "mix", "T": 30011, "C": 1001},
        # K4 forward at the training width and many tokens (the most bytes of a single kernel here).
        {"name": "post_res_T65536_C4096", "kind": "post_res", "T": 65536, "C": 4096},
        # K4 backward at the reference benchmark's default width, one token over a round count.
        {"name": "post_res_bwd_T65537_C2560", "kind": "post_res_bwd", "T": 65537, "C": 2560},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(KINDS)
    # A third each: the configurations' widths, any multiple of eight, any width of a small model.
    pick = rng.randrange(3)
    if pick == 0:
        C = rng.choice([256, 512, 1024, 2048, 2560, 4096])
    elif pick == 1:
        C = rng.randrange(64, 4097, 8)
    else:
        C = rng.randrange(17, 1025)
    case = {"kind": kind, "T": 0, "C": C}
    if kind == "eval":
        T = _log_uniform(rng, 1, 4096)
        case["graph"] = rng.random() < 0.5
        case["rms"] = rng.random() < 0.25
    elif kind == "train":
        T = _log_uniform(rng, 64, 65536)
        case["graph"] = rng.random() < 0.5
        case["rms"] = not case["graph"] and rng.random() < 0.5
    else:
        T = _log_uniform(rng, 512, 131072)
    most = (1 << 25) if C % 8 else (1 << 27) if kind == "train" else (1 << 28)
    case["T"] = max(1, min(T, most // C))
    return case


# ---------------------------------------------------------------------------
# Inputs


class _Draws:
    """Seeded normal tensors on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV).manual_seed(int(seed))

    def __call__(self, *shape, scale=1.0, mean=0.0, dtype=BF16):
        t = torch.randn(shape, device=DEV, dtype=dtype if dtype is BF16 else torch.float32, generator=self.g)
        if scale != 1.0:
            t *= scale
        if mean != 0.0:
            t += mean
        return t.to(dtype)


def _streams(rn, T, C):
    """x ~ N(m, 1), every feature with a mean m of its own (so that the gates'
    gradients, sums over all tokens, do not vanish); every 100th token scaled
    by 100, the outliers that an RMSNorm meets."""
    x = rn(T, N, C)
    x += rn(1, N, C, scale=0.5)
    x[::100] *= 100
    return x


def _params(rn, C):
    """Projection weight, gates a little way into training, and the permutations."""
    W = rn(D, N * C, scale=0.02)
    alphas = [torch.full((1,), a, device=DEV, dtype=BF16) for a in (0.25, 0.375, 0.5)]
    bias = rn(D, scale=0.1)
    perm = flash_mhc.build_permutation_matrices(N)[0].to(DEV, BF16)
    return W, alphas, bias, perm


def _chain(proj, alphas, bias, perm):
    """The coefficients in proj's dtype (plain torch)."""
    pre, post, res = proj.split([N, N, D - 2 * N], dim=-1)
    h_pre = torch.sigmoid(alphas[0] * pre + bias[:N])
    h_post = 2.0 * torch.sigmoid(alphas[1] * post + bias[N:2 * N])
    a = torch.softmax(alphas[2] * res + bias[2 * N:], dim=-1)
    H = (a @ perm).unflatten(-1, (N, N)) - h_post.unsqueeze(-1) * h_pre.unsqueeze(-2)
    return h_pre, h_post, H


def _coefficients(rn, T):
    """(h_pre, h_post, H) fp32 as K2 makes them from a projection of spread one."""
    _W, alphas, bias, perm = _params(rn, 1)
    h_pre, h_post, H = _chain(rn(T, D), alphas, bias, perm)
    return h_pre.float(), h_post.float(), H.float().contiguous()


def _inputs(case, seed):
    rn = _Draws(seed)
    kind, T, C = case["kind"], case["T"], case["C"]
    s = {"x": _streams(rn, T, C)}
    if kind in ("eval", "train"):
        W, alphas, bias, _perm = _params(rn, C)
        s.update(W=W, alphas=alphas, bias=bias, layer=rn(C, C, scale=C ** -0.5))
        if case["rms"]:
            s["rms"] = rn(N * C, scale=0.02, mean=1.0)
        if kind == "train":
            s["g"] = rn(T, N, C)
            s["g"] += rn(1, N, C, scale=0.5)
    elif kind == "project":
        s.update(x=s["x"].view(T, N * C), W=rn(D, N * C, scale=0.02), g=rn(T, D))
    elif kind in ("pre_map", "pre_map_bwd"):
        W, alphas, bias, perm = _params(rn, C)
        s.update(W=W, alphas=alphas, bias=bias, perm=perm)
        if kind == "pre_map_bwd":
            xf = s["x"].view(T, N * C)
            # What the forward has left: in plain torch, from the same inputs, in pieces of tokens.
            inv = torch.cat([torch.rsqrt(p.float().square().mean(-1) + EPS) for p in xf.split(16384)])
            proj = (inv.unsqueeze(-1) * (xf @ W.t()).float()).to(BF16)
            h_pre = _chain(proj, alphas, bias, perm)[0].float().contiguous()
            s.update(inv=inv, proj=proj, h_pre=h_pre, g_li=rn(T, C), g_x=rn(T, N, C),
                     g_hp=rn(T, N, dtype=torch.float32) + rn(1, N, dtype=torch.float32),
                     g_H=rn(T, N, N, dtype=torch.float32) + rn(1, N, N, dtype=torch.float32))
    elif kind == "mix":
        s.update(h_pre=_coefficients(rn, T)[0], g=rn(T, C))
    else:
        _h_pre, h_post, H = _coefficients(rn, T)
        s.update(lo=rn(T, C), h_post=h_post, H=H)
        if kind == "post_res_bwd":
            s["g"] = rn(T, N, C)
    return s


# ---------------------------------------------------------------------------
# The calls


def _block(case, s):
    C = case["C"]
    layer = nn.Linear(C, C, bias=False, device=DEV, dtype=BF16)
    with torch.device(DEV):
        block = flash_mhc.MHCLiteBlock(N, C, layer, rmsnorm_weight=case["rms"]).to(BF16)
    with torch.no_grad():
        block.W_all.weight.copy_(s["W"])
        block.W_all.bias.copy_(s["bias"])
        for p, a in zip((block.alpha_pre, block.alpha_post, block.alpha_res), s["alphas"]):
            p.copy_(a)
        layer.weight.copy_(s["layer"])
        if case["rms"]:
            block.rms_weight.copy_(s["rms"])
    return block


def _eval_step(s):
    with torch.no_grad():
        return s["block"](s["x"])


def _train_step(s):
    out = s["block"](s["x"])
    return (out.detach(), *torch.autograd.grad(out, [s["x"], *s["params"]], s["g"]))


def _captured(step, s):
    """step(s) captured in a HIP graph: (graph, its outputs)."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            step(s)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step(s)
    return graph, out


def prepare(case, seed):
    s = _inputs(case, seed)
    kind = s["kind"] = case["kind"]
    if kind in ("eval", "train"):
        block = s["block"] = _block(case, s)
        if kind == "eval":
            block.eval()
        else:
            s["x"].requires_grad_(True)
            s["params"] = [block.W_all.weight, block.W_all.bias, block.alpha_pre, block.alpha_post, block.alpha_res,
                           block.layer.weight, *([block.rms_weight] if case["rms"] else [])]
        s["step"] = _eval_step if kind == "eval" else _train_step
        if case["graph"]:
            s["graph"], s["out"] = _captured(s["step"], s)
    elif kind == "project":
        s["x"].requires_grad_(True)
        s["W"].requires_grad_(True)
    elif kind == "mix":
        s["x"].requires_grad_(True)
        s["h_pre"].requires_grad_(True)
    return s


def run(s):
    ops = torch.ops.flash_mhc
    kind = s["kind"]
    if kind in ("eval", "train"):
        if "graph" in s:
            s["graph"].replay()
            return s["out"]
        return s["step"](s)
    if kind == "project":
        proj, inv = ops.fused_rmsnorm_project(s["x"], s["W"])
        return (proj.detach(), inv.detach(), *torch.autograd.grad(proj, [s["x"], s["W"]], s["g"]))
    if kind == "pre_map":
        return ops.mhc_pre_map(s["x"], s["W"], *s["alphas"], s["bias"], s["perm"])[:6]
    if kind == "pre_map_bwd":
        return ops.mhc_pre_map_backward(s["g_li"], s["g_H"], s["g_hp"], None, None, s["g_x"], s["x"], s["W"],
                                        *s["alphas"], s["bias"], s["perm"], s["h_pre"], s["proj"], s["inv"])
    if kind == "mix":
        out = ops.fused_pre_map(s["x"], s["h_pre"])
        return (out.detach(), *torch.autograd.grad(out, [s["x"], s["h_pre"]], s["g"]))
    if kind == "post_res":
        return ops.fused_post_res(s["x"], s["lo"], s["H"], s["h_post"])
    return ops.fused_post_res_backward(s["g"], s["x"], s["lo"], s["H"], s["h_post"])


# ---------------------------------------------------------------------------
# What a pass cannot do without (a forward and a backward counted as the two calls they are)


def work(case):
    kind, T, C = case["kind"], case["T"], case["C"]
    x = 2 * T * N * C        # the streams, or a gradient of them
    row = 2 * T * C          # layer input or output, or a gradient of it
    w = 2 * D * N * C        # the projection's weight, or its gradient
    coef = 4 * T * (N + N * N)  # h_post and H_merged, or their gradients
    small = T * (2 * D + 4 + 4 * N)  # proj, inv_rms, h_pre
    k1 = 2 * T * D * N * C
    pre_map = (x + w + row + coef + small, k1 + 2 * T * N * C)
    pre_map_bwd = (x + w + row + coef + small + x + x + w, 2 * k1 + 6 * T * N * C)
    post_res = (x + row + coef + x, 2 * T * N * (N + 1) * C)
    post_res_bwd = (2 * x + row + coef + x + row + coef, 4 * T * N * (N + 1) * C)
    layer = (2 * row + 2 * C * C, 2 * T * C * C)
    layer_bwd = (3 * row + 4 * C * C, 4 * T * C * C)
    parts = {
        "eval": (pre_map, layer, post_res),
        "train": (pre_map, layer, post_res, post_res_bwd, layer_bwd, pre_map_bwd),
        "project": ((x + w + T * (2 * D + 4), k1), (x + w + T * (4 * D + 4) + x + w, 2 * k1)),
        "pre_map": (pre_map,),
        "pre_map_bwd": (pre_map_bwd,),
        "mix": ((x + 4 * T * N + row, 2 * T * N * C), (x + 4 * T * N + row + x + 4 * T * N, 3 * T * N * C)),
        "post_res": (post_res,),
        "post_res_bwd": (post_res_bwd,),
    }[kind]
    return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}


# Relative errors (2-norm) that another correct implementation at these
# precisions shows: an output rounded once to bf16 is 1.7e-3 from its value, the
# coefficients' chain of bf16 roundings and whatever is computed from them 2e-3
# to 6e-3 (the largest at the gate gradients, sums of rounded terms).
def tolerance(case):
    return {"rel": {"eval": 1.2e-2, "train": 2.4e-2, "project": 7e-3, "pre_map": 1e-2, "pre_map_bwd": 2.4e-2,
                    "mix": 7e-3, "post_res": 7e-3, "post_res_bwd": 7e-3}[case["kind"]]}


# ---------------------------------------------------------------------------
# The same in 64 bits, plain torch.  Not for the gates' gradients: each is one
# value, a sum of rounded terms rounded to bf16, and how far it lands from the
# 64-bit sum is chance.


def _exact_project(xf, W):
    inv = torch.rsqrt(xf.square().mean(-1) + EPS)
    return inv.unsqueeze(-1) * (xf @ W.t()), inv


def _exact_pre_map(x, W, alphas, bias, perm):
    proj, inv = _exact_project(x.flatten(1), W)
    h_pre, h_post, H = _chain(proj, alphas, bias, perm)
    return (h_pre.unsqueeze(-1) * x).sum(1), H, h_post, h_pre, proj, inv


def _exact_post_res(x, lo, H, h_post):
    out = h_post.unsqueeze(-1) * lo.unsqueeze(1)
    for j in range(N):
        out = out + H[:, :, j:j + 1] * x[:, j:j + 1]
    return out


def exact(case, seed):
    kind, T, C = case["kind"], case["T"], case["C"]
    if T * C > (1 << 28):
        return None
    s = _inputs(case, seed)
    d = {k: [a.to(F64) for a in v] if isinstance(v, list) else v.to(F64) for k, v in s.items()}
    del s
    if kind in ("eval", "train"):
        perm = flash_mhc.build_permutation_matrices(N)[0].to(DEV, F64)
        leaves = [d["x"], d["W"], d["bias"], *d["alphas"], d["layer"], *([d["rms"]] if case["rms"] else [])]
        if kind == "train":
            for t in leaves:
                t.requires_grad_(True)
        W = d["W"] * d["rms"] if case["rms"] else d["W"]
        with torch.set_grad_enabled(kind == "train"):
            li, H, h_post, _h_pre, _proj, _inv = _exact_pre_map(d["x"], W, d["alphas"], d["bias"], perm)
            out = _exact_post_res(d["x"], li @ d["layer"].t(), H, h_post)
        if kind == "eval":
            return out
        gx, gW, gb, _ga, _gq, _gr, *rest = torch.autograd.grad(out, leaves, d["g"])
        return (out.detach(), gx, gW, gb, None, None, None, *rest)
    if kind == "project":
        d["x"].requires_grad_(True)
        d["W"].requires_grad_(True)
        proj, inv = _exact_project(d["x"], d["W"])
        return (proj.detach(), inv.detach(), *torch.autograd.grad(proj, [d["x"], d["W"]], d["g"]))
    if kind == "pre_map":
        return _exact_pre_map(d["x"], d["W"], d["alphas"], d["bias"], d["perm"])
    if kind == "pre_map_bwd":
        leaves = [d["x"], d["W"], *d["alphas"], d["bias"]]
        for t in leaves:
            t.requires_grad_(True)
        li, H, h_post, _h_pre, _proj, _inv = _exact_pre_map(d["x"], d["W"], d["alphas"], d["bias"], d["perm"])
        gx, gW, _ga, _gq, _gr, gb = torch.autograd.grad((li, H, h_post), leaves, (d["g_li"], d["g_H"], d["g_hp"]))
        return (gx + d["g_x"], gW, None, None, None, gb)
    if kind == "mix":
        g = d["g"].unsqueeze(1)
        h = d["h_pre"].unsqueeze(-1)
        return (h * d["x"]).sum(1), h * g, (d["x"] * g).sum(-1)
    if kind == "post_res":
        return _exact_post_res(d["x"], d["lo"], d["H"], d["h_post"])
    gx = torch.zeros_like(d["x"])
    gH = torch.empty_like(d["H"])
    for i in range(N):
        gx += d["H"][:, i].unsqueeze(-1) * d["g"][:, i:i + 1]
        gH[:, i] = (d["g"][:, i:i + 1] * d["x"]).sum(-1)
    g_lo = (d["h_post"].unsqueeze(-1) * d["g"]).sum(1)
    return gx, g_lo, gH, (d["g"] * d["lo"].unsqueeze(1)).sum(-1)
