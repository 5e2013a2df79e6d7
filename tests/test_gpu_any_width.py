"""Widths that are not a multiple of eight, and operands off 16-byte alignment,
on the matrix-core and 16-byte kernels: the last columns of a row (fewer than
eight), rows shorter than a wave's slice, the first and last rows of a 16-token
block, and base addresses 2 and 6 bytes off a 16-byte boundary.  Against the
oracle (tests/parity.py's bounds), and bit for bit against the separate
kernels where both do the same arithmetic."""

from __future__ import annotations

import pytest
import torch

from flash_mhc import build_permutation_matrices
from flash_mhc import _abi
from flash_mhc import kernels as K
from oracle import mhc_oracle as O
from parity import bf16_ulp, check_bf16, check_fp32, check_rel

pytestmark = pytest.mark.gpu

DEV = "cuda"
BF16 = torch.bfloat16

# C = 8 ... 17: rows of one or two groups; 127 / 129 / 131: either side of a
# 128-column slice; 257, 1001: several slices, odd.  T around the 16-token
# block and beyond the few-token forms (1037, 6150).
SHAPES = [(1, 9), (15, 15), (16, 8), (17, 17), (33, 127), (300, 129), (1037, 131), (6150, 257), (2100, 1001)]


def _at(t: torch.Tensor, off: int) -> torch.Tensor:
    """t on the GPU, its base `off` elements past a 16-byte boundary."""
    buf = torch.empty(t.numel() + 8, device=DEV, dtype=t.dtype)
    view = buf[off:off + t.numel()].view(t.shape)
    view.copy_(t)
    return view


def _inputs(T, C, off, seed):
    g = torch.Generator().manual_seed(seed)
    rn = lambda *s, scale=1.0: (torch.randn(s, generator=g) * scale).to(BF16)
    x = rn(T, 4, C)
    x[::5] *= 50
    return rn, _at(x, off), _at(rn(32, 4 * C, scale=0.02), off)


def _params(C):
    g = torch.Generator().manual_seed(C)
    return [t.to(DEV) for t in (torch.tensor([0.8]), torch.tensor([1.2]), torch.tensor([1.7]),
                                torch.randn(32, generator=g) * 0.5, build_permutation_matrices(4)[0])]


# The forward's tiles of 16, 32, 48 and 64 tokens (from T = 4097, 8193, 12289),
# its column split (up to 2720 tokens, nC of two chunks and more) and its last
# chunk of 1 to 63 columns: C = 2 and 3 (one group, rows of 8 and 12 columns),
# 15 ... 17 around one 64-column chunk.
FWD = [*SHAPES, (5, 2), (40, 3), (4096, 16), (2721, 129), (5000, 131), (9000, 33), (12300, 25), (20011, 300),
       (2720, 4099), (3, 4103),
       # The split's blocks of 16 (up to 896 tokens) and of 32, and its last token counts.
       (896, 1100), (897, 1101), (912, 1100), (913, 1101), (929, 1100), (1168, 1024), (1169, 1024), (1600, 1423), (1601, 1420), (2719, 1424),
       # The split's finish: x ahead of the sums from 257 groups of 8 columns on, up to 1024 tokens.
       (30, 2054), (30, 2060), (1024, 2060), (1025, 2060)]


@pytest.mark.parametrize("off", [0, 1, 3])
@pytest.mark.parametrize("T,C", FWD)
def test_k1_fwd(T, C, off):
    nC = 4 * C
    rn, x, W = _inputs(T, C, off, 7 * T + C + off)
    proj, inv = K.k1_fwd(x.view(T, nC), W, out=_at(torch.zeros(T, 32, dtype=BF16), off))
    R, S, invR = O.k1_fwd(x.view(T, nC).cpu(), W.cpu())
    check_bf16("proj", proj, R, S, nC)
    check_rel("inv_rms", inv, invR, rtol=4 * nC ** 0.5 * 2.0**-24 + 4 * 2.0**-24)


@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("T,C", FWD)
def test_premap_fwd(T, C, off):
    nC = 4 * C
    rn, x, W = _inputs(T, C, off, 5 * T + C + off)
    p = _params(C)
    li, H, hq, hp, proj, inv = K.premap_fwd(x, W, *p)
    proj1, inv1 = K.k1_fwd(x.view(T, nC), W)
    hp1, hq1, H1 = K.k2_fwd(proj1, *p)
    want = (K.k3_fwd(x, hp1), H1, hq1, hp1, proj1, inv1)
    for name, u, v in zip(("layer_input", "H", "h_post", "h_pre", "proj", "inv_rms"), (li, H, hq, hp, proj, inv), want):
        assert torch.equal(u, v), name


@pytest.mark.parametrize("off", [0, 1, 3])
@pytest.mark.parametrize("T,C", SHAPES)
def test_k1_bwd(T, C, off):
    nC = 4 * C
    rn, x, W = _inputs(T, C, off, 11 * T + C + off)
    x = x.view(T, nC)
    proj, inv = K.k1_fwd(x, W)
    go = _at(rn(T, 32), off)
    inv = _at(inv.cpu(), off)  # 4-byte alignment only
    gx, gW = K.k1_bwd(go, x, W, proj, inv)
    R, S = O.k1_bwd_dx(go.cpu(), x.cpu(), W.cpu(), proj.cpu(), inv.cpu())
    check_bf16("grad_x", gx, R, S, 64)
    assert torch.equal(K.k1_bwd_dx(go, x, W, proj, inv), gx)
    R, S = O.k1_grad_W(go.cpu(), x.cpu(), inv.cpu())
    check_bf16("grad_W", gW, R, S, T)


# K3's reduce and K2's backward in one kernel: half a wave per token, one and two
# groups of 8 per lane (17 to 64), the second partly filled, then a wave.
FUSED_BWD = [(9, 136), (41, 256), (40, 263), (300, 264), (700, 384), (33, 448), (16, 512), (20, 519), (9, 520), (9, 768)]


@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("T,C", [*SHAPES, *FUSED_BWD])
def test_premap_bwd(T, C, off):
    nC = 4 * C
    rn, x, W = _inputs(T, C, off, 13 * T + C + off)
    p = _params(C)
    li, H, hq, hp, proj, inv = K.premap_fwd(x, W, *p)
    g_li, g_in = _at(rn(T, C), off), _at(rn(T, 4, C), off)
    gx, gW, *pg = K.premap_bwd(x, W, *p, hp, proj, inv, g_li, hq, H, g_in)
    gx3, gh = K.k3_bwd(g_li, x, hp)
    gp, *rpg = K.k2_bwd(proj, *p, gh, hq, H)
    dx, _ = K.k1_bwd(gp, x.view(T, nC), W, proj, inv)
    # Three gradients of x, each rounded to bf16, added in autograd's order.
    assert torch.equal(gx, g_in + (gx3 + dx.view(T, 4, C)))
    for u, v in zip(pg, rpg):
        assert torch.equal(u, v)
    R, S = O.k1_grad_W(gp.cpu(), x.view(T, nC).cpu(), inv.cpu())
    check_bf16("grad_W", gW, R, S, T)


# K3 / K4: one 16-byte group per lane over 8, 16, 32, 64, 128, 192, ... 448
# lanes per token and several groups per lane beyond; rows that end inside a
# group, at a wave's edge, or one group into the next wave.  From (16500, 519)
# on enough workgroups (4096) for the residency caps, at one wave per token, two
# and more; (20001, 200) has them too, at 32 lanes per token, which take no cap.
K34 = [(1, 1), (33, 7), (9, 8), (130, 65), (65, 136), (31, 264), (77, 512), (45, 519), (5, 520), (19, 1032),
       (7, 1535), (3, 1536), (6, 2056), (4, 3079), (2, 3592), (3, 4100), (20001, 200), (16500, 519), (9001, 1000), (4200, 1535), (4100, 2049),
       (4100, 2560), (4100, 3003), (4100, 3583)]


@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("T,C", K34)
def test_k3_k4(T, C, off):
    rn, x, _W = _inputs(T, C, off, 17 * T + C + off)
    g = torch.Generator().manual_seed(T + C)
    h = torch.rand(T, 4, generator=g).to(DEV)
    H = torch.randn(T, 4, 4, generator=g).to(DEV)
    lo, go3, go4 = _at(rn(T, C), off), _at(rn(T, C), off), _at(rn(T, 4, C), off)
    c = lambda t: t.cpu()
    check_bf16("k3 out", K.k3_fwd(x, h), *O.k3_fwd(c(x), c(h)), 4)
    gx, gh = K.k3_bwd(go3, x, h)
    gxR, gxS, ghR, ghS = O.k3_bwd(c(go3), c(x), c(h))
    check_bf16("k3 grad_x", gx, gxR, gxS, 1)
    check_fp32("k3 grad_h_pre", gh, ghR, ghS, C)
    check_bf16("k4 out", K.k4_fwd(x, lo, H, h), *O.k4_fwd(c(x), c(lo), c(H), c(h)), 5)
    gx, glo, gH, ghp = K.k4_bwd(go4, x, lo, H, h)
    ref = O.k4_bwd(c(go4), c(x), c(lo), c(H), c(h))
    check_bf16("k4 grad_x", gx, *ref["grad_x"], 4)
    check_bf16("k4 grad_lo", glo, *ref["grad_lo"], 4)
    check_fp32("k4 grad_H", gH, *ref["grad_H"], C)
    check_fp32("k4 grad_hp", ghp, *ref["grad_hp"], C)


# grad_W's reduce: 16 shares of five runs and more up to 8 slices of 128 columns
# (C = 256), four up to 16, one above and for fewer runs; one run to several
# hundred, fewer runs than shares (T = 304: four runs, 305: five).
@pytest.mark.parametrize("T,C", [(1, 64), (40, 24), (9000, 24), (16001, 33), (3000, 256), (3000, 264), (2000, 512),
                                 (2000, 520), (304, 64), (305, 64), (304, 256), (305, 256), (130, 300)])
def test_grad_W_reduce(T, C):
    nC = 4 * C
    rn, x, W = _inputs(T, C, 0, 17 * T + C)
    x = x.view(T, nC)
    proj, inv = K.k1_fwd(x, W)
    go = _at(rn(T, 32), 0)
    _, gW = K.k1_bwd(go, x, W, proj, inv)
    R, S = O.k1_grad_W(go.cpu(), x.cpu(), inv.cpu())
    check_bf16("grad_W", gW, R, S, T)


# Workspaces of the sizes that rows off 8 columns have had (none, and no room
# for grad_W's partial sums): the calls still run, on other kernels.
@pytest.mark.parametrize("T,C", [(300, 129), (1037, 131)])
def test_without_partials(T, C, monkeypatch):
    nC = 4 * C
    rn, x, W = _inputs(T, C, 0, 19 * T + C)
    p = _params(C)
    go, g_li, g_in = _at(rn(T, 32), 0), _at(rn(T, C), 0), _at(rn(T, 4, C), 0)

    def run():
        proj, inv = K.k1_fwd(x.view(T, nC), W)
        li, H, hq, hp, pj, iv = K.premap_fwd(x, W, *p)
        return (proj, inv, li, H, hq, hp, *K.k1_bwd(go, x.view(T, nC), W, proj, inv),
                *K.premap_bwd(x, W, *p, hp, pj, iv, g_li, hq, H, g_in))

    want = run()
    lib = _abi.load()
    up = lambda n: (n + 255) // 256 * 256
    small = up(16 * T) + up(64 * T) + up(int(lib.fmhc_k2_bwd_workspace_bytes(T)))
    assert small < int(lib.fmhc_premap_bwd_workspace_bytes(T, C))
    for name in ("fmhc_k1_fwd_workspace_bytes", "fmhc_premap_fwd_workspace_bytes", "fmhc_k1_bwd_workspace_bytes"):
        monkeypatch.setattr(lib, name, lambda *a: 0)
    monkeypatch.setattr(lib, "fmhc_premap_bwd_workspace_bytes", lambda *a: small)
    got = run()
    proj, inv, li, H, hq, hp, gx1, gW1, gx, gW, *_ = [t.cpu() for t in got]
    c = lambda t: t.cpu()
    xc = x.view(T, nC).cpu()
    check_bf16("proj", proj, *O.k1_fwd(xc, c(W))[:2], nC)
    check_bf16("layer_input", li, *O.k3_fwd(c(x), hp), 4)
    dx, dxS = O.k1_bwd_dx(c(go), xc, c(W), proj, inv)
    check_bf16("k1 grad_x", gx1, dx, dxS, 64)
    check_bf16("k1 grad_W", gW1, *O.k1_grad_W(c(go), xc, inv), T)
    # The pre-map's gradients from K2's gradient of proj, which the separate kernels give.
    gh = K.k3_bwd(g_li, x, hp.to(DEV))[1]
    gp = c(K.k2_bwd(proj.to(DEV), *p, gh, hq.to(DEV), H.to(DEV))[0])
    check_bf16("grad_W", gW, *O.k1_grad_W(gp, xc, inv), T)
    dx, dxS = (t.view(T, 4, C) for t in O.k1_bwd_dx(gp, xc, c(W), proj, inv))
    gx3 = hp.double().unsqueeze(-1) * c(g_li).double().unsqueeze(1)
    # Three values and two sums of them, each rounded once: half an ulp of at most M each, 2.5 in all.
    M = c(g_in).double().abs() + gx3.abs() + dx.abs()
    err = (gx.double() - (c(g_in).double() + gx3 + dx)).abs()
    assert bool((err <= 2.5 * bf16_ulp(M) + 4 * 64 ** 0.5 * 2.0**-24 * dxS).all())
    for a, b in zip(got, want):
        a, b = a.double(), b.double()
        # One more bf16 rounding here or there (K1's projection feeds the rest): 2^-8 of each value, 2^-6 of the whole.
        assert float((a - b).norm()) <= 2.0 ** -6 * float(b.norm())


# K1's few-token forward with no workspace: one pass where any of x, W and out
# is off 16 bytes, as ever; refused, as ever, where all three are aligned.
@pytest.mark.parametrize("x_off,w_off,out_off", [(1, 0, 0), (0, 1, 0), (0, 0, 1), (0, 0, 0)])
def test_k1_fwd_without_workspace(x_off, w_off, out_off):
    T, nC = 64, 1024
    g = torch.Generator().manual_seed(41)
    x = _at(torch.randn(T, nC, generator=g).to(BF16), x_off)
    W = _at((torch.randn(32, nC, generator=g) * 0.02).to(BF16), w_off)
    out = _at(torch.zeros(T, 32, dtype=BF16), out_off)
    inv = torch.zeros(T, device=DEV)
    lib = _abi.load()
    assert lib.fmhc_k1_fwd_workspace_bytes(T, nC) > 0
    st = lib.fmhc_k1_fwd_ws(x.data_ptr(), W.data_ptr(), out.data_ptr(), inv.data_ptr(), None, 0, T, nC, 32,
                            _abi.stream_of(x))
    if not (x_off or w_off or out_off):
        assert st == 1
        return
    assert st == 0
    R, S, invR = O.k1_fwd(x.cpu(), W.cpu())
    check_bf16("proj", out, R, S, nC)
    check_rel("inv_rms", inv, invR, rtol=4 * nC ** 0.5 * 2.0**-24 + 4 * 2.0**-24)


# grad_x written over x: 1, 4 and 7 columns past a 128-column slice, whose last
# lane shares columns with the slice before; whole groups beside them.
@pytest.mark.parametrize("T,nC", [(3000, 129), (3000, 132), (700, 1031), (700, 1024), (300, 136), (40, 9)])
def test_k1_bwd_dx_in_place(T, nC):
    g = torch.Generator().manual_seed(T + nC)
    x = torch.randn(T, nC, generator=g).to(BF16).to(DEV)
    W = (torch.randn(32, nC, generator=g) * 0.02).to(BF16).to(DEV)
    go = torch.randn(T, 32, generator=g).to(BF16).to(DEV)
    proj, inv = K.k1_fwd(x, W)
    R, S = O.k1_bwd_dx(go.cpu(), x.cpu(), W.cpu(), proj.cpu(), inv.cpu())
    got = K.k1_bwd_dx(go, x, W, proj, inv, grad_x=x)
    assert got.data_ptr() == x.data_ptr()
    check_bf16("grad_x", got, R, S, 64)


# One infinity or NaN in x, in columns that the last, shifted group of a row
# loads together with the group before it (nC - 8 ...), at either side of a
# 128-column slice, and first: it reaches what the formulas say (its token's
# projection and grad_x, its column of grad_W) and nothing else.
@pytest.mark.parametrize("value", [float("inf"), float("nan")])
@pytest.mark.parametrize("T,nC", [(40, 9), (40, 12), (33, 129), (300, 132), (2100, 1031), (20, 4404), (700, 1200)])
def test_k1_one_odd_value(T, nC, value):
    g = torch.Generator().manual_seed(T + nC)
    x = torch.randn(T, nC, generator=g).to(BF16).to(DEV)
    W = (torch.randn(32, nC, generator=g) * 0.02 + 0.5).to(BF16).to(DEV)
    go = torch.randn(T, 32, generator=g).to(BF16).to(DEV)
    proj, inv = K.k1_fwd(x, W)
    gx, gW = K.k1_bwd(go, x, W, proj, inv)
    for c in sorted({0, 127, 128, nC - 9, nC - 8, nC - 7, nC - 2, nC - 1} & set(range(nC))):
        t = (7 * c + 3) % T
        y = x.clone()
        y[t, c] = value
        proj1, inv1 = K.k1_fwd(y, W)
        # The sum of squares is inf or NaN: 1 / rms is 0 or NaN, and the projection NaN either way.
        assert bool(proj1[t].isnan().all()) and not float(inv1[t]) > 0
        keep = torch.arange(T, device=DEV) != t
        assert torch.equal(proj1[keep], proj[keep]) and torch.equal(inv1[keep], inv[keep])
        # The backward with the finite token's proj and inv_rms: only x itself is odd.
        gx1, gW1 = K.k1_bwd(go, y, W, proj, inv)
        odd = torch.zeros(T, nC, dtype=torch.bool, device=DEV)
        odd[t, c] = True
        assert torch.equal(~gx1.isfinite(), odd) and torch.equal(gx1[~odd], gx[~odd])
        assert torch.equal(~gW1.isfinite(), odd[t].expand(32, nC))
        assert torch.equal(gW1[:, ~odd[t]], gW[:, ~odd[t]])
        assert torch.equal(K.k1_bwd_dx(go, y, W, proj, inv)[~odd], gx[~odd])
