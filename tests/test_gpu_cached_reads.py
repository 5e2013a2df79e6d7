"""A token's outputs do not depend on how many tokens a launch has: K1, K3 and
K4 and the pre-map backward at two token counts, one block of 16 tokens and a
ragged one apart, at sizes where a launch reads about as much as stays in the
memory-side cache (80 MiB of the 256).  For the tokens the two share, the larger
launch must give the bits of the smaller one.  K1's grad_W, a sum over the
tokens, is checked against the oracle at both.
"""

from __future__ import annotations

import pytest
import torch

from flash_mhc import build_permutation_matrices
from flash_mhc import kernels as K
from oracle import mhc_oracle as O
from parity import check_bf16

pytestmark = pytest.mark.gpu

DEV = "cuda"
BF16 = torch.bfloat16
LINE = 80 << 20


# 1000 and 1008: rows off and on 128-byte lines (4 C a multiple of 64), neither a power of two.
@pytest.mark.parametrize("C", [256, 512, 1000, 1008])
@pytest.mark.parametrize("kernel", ["k1_fwd", "k1_bwd_dx", "k1_bwd", "k3_fwd", "k3_bwd", "k4_fwd", "k4_bwd"])
def test_same_bits_on_both_sides(kernel, C):
    read = {"k1_fwd": 8, "k1_bwd_dx": 8, "k1_bwd": 8, "k3_fwd": 8, "k3_bwd": 10, "k4_fwd": 10, "k4_bwd": 36}[kernel] * C
    T0 = LINE // read // 16 * 16  # whole token blocks, at or below the line
    T1 = T0 + 16 + 1
    assert T0 * read <= LINE < T1 * read
    g = torch.Generator(device=DEV).manual_seed(C)

    def rn(*s):
        return torch.randn(s, device=DEV, generator=g).to(BF16)

    x, W, lo, go = rn(T1, 4, C), rn(32, 4 * C), rn(T1, C), rn(T1, 4, C)
    h, H = torch.rand(T1, 4, device=DEV, generator=g), torch.randn(T1, 4, 4, device=DEV, generator=g)
    gp, proj, inv = rn(T1, 32), rn(T1, 32), torch.rand(T1, device=DEV, generator=g)

    def run(T):
        xf = x[:T].view(T, 4 * C)
        if kernel == "k1_fwd":
            return K.k1_fwd(xf, W)
        if kernel == "k1_bwd_dx":
            return (K.k1_bwd_dx(gp[:T], xf, W, proj[:T], inv[:T]),)
        if kernel == "k1_bwd":
            gx, gW = K.k1_bwd(gp[:T], xf, W, proj[:T], inv[:T])  # grad_W is a sum over the tokens
            R, S = O.k1_grad_W(gp[:T].cpu(), xf.cpu(), inv[:T].cpu())
            check_bf16("grad_W", gW, R, S, T)
            return (gx,)
        if kernel == "k3_fwd":
            return (K.k3_fwd(x[:T], h[:T]),)
        if kernel == "k3_bwd":
            return K.k3_bwd(lo[:T], x[:T], h[:T])
        if kernel == "k4_fwd":
            return (K.k4_fwd(x[:T], lo[:T], H[:T], h[:T]),)
        return K.k4_bwd(go[:T], x[:T], lo[:T], H[:T], h[:T])

    for a, b in zip(run(T0), run(T1)):
        assert torch.equal(a, b.reshape(T1, -1)[:T0].reshape(a.shape))


@pytest.mark.parametrize("C", [256, 1000])
def test_pre_map_backward_same_bits(C):
    T0 = LINE // (18 * C) // 16 * 16
    T1 = T0 + 16 + 1
    g = torch.Generator(device=DEV).manual_seed(C)

    def rn(*s):
        return torch.randn(s, device=DEV, generator=g).to(BF16)

    x, W, g3, gi = rn(T1, 4, C), rn(32, 4 * C), rn(T1, C), rn(T1, 4, C)
    proj, inv = K.k1_fwd(x.view(T1, 4 * C), W)
    hq, H = torch.rand(T1, 4, device=DEV, generator=g), torch.randn(T1, 4, 4, device=DEV, generator=g)
    p = [torch.tensor([a], device=DEV) for a in (0.8, 1.2, 1.7)]
    p += [torch.randn(32, device=DEV, generator=g), build_permutation_matrices(4)[0].to(DEV)]
    hp = K.k2_fwd(proj, *p)[0]

    def run(T):
        return K.premap_bwd(x[:T], W, *p, hp[:T], proj[:T], inv[:T], g3[:T], hq[:T], H[:T], gi[:T])[0]

    assert torch.equal(run(T0), run(T1)[:T0])
