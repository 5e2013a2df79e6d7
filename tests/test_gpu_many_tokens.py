"""K3, K4 and element-wise K1 for more tokens than one launch can hold: a HIP
launch stays below 2^32 threads, which K3's and K4's eight lanes per token at
C = 1 reach at T = 2^29 and element-wise K1's 64 (rows of fewer than eight
columns) at T = 2^26, and the entry points then launch pieces of the tokens.  Every output element must be
written, and tokens at the ends and around the seam must have the bits of a
call on those tokens alone."""

from __future__ import annotations

import pytest
import torch

from flash_mhc import kernels as K

pytestmark = pytest.mark.gpu

DEV = "cuda"
BF16 = torch.bfloat16
T = (1 << 29) + 24
SEAM = ((1 << 32) - 1) // 256 * 32  # tokens of the first launch: 32 per 256 threads
WINDOWS = [slice(0, 100), slice(SEAM - 70, SEAM + 56), slice(T - 90, T)]


def _rand(*shape, dtype=BF16):
    g = torch.Generator(device=DEV).manual_seed(len(shape) + shape[-1])
    return torch.rand(shape, device=DEV, dtype=dtype, generator=g)


def _nan(*shape, dtype=BF16):
    return torch.full(shape, float("nan"), device=DEV, dtype=dtype)


def _check(outs, alone, windows=WINDOWS):
    for o in outs:
        for piece in o.view(-1).split(1 << 28):
            assert not bool(torch.isnan(piece).any())
    for w in windows:
        for o, want in zip(outs, alone(w)):
            assert torch.equal(o[w], want), w


@pytest.mark.parametrize("kernel", ["k3_fwd", "k3_bwd", "k4_fwd", "k4_bwd"])
def test_pieces(kernel):
    assert 0 < T - SEAM < 128
    x, h = _rand(T, 4, 1), _rand(T, 4, dtype=torch.float32)
    if kernel == "k3_fwd":
        out = K.k3_fwd(x, h, out=_nan(T, 1))
        _check([out], lambda w: [K.k3_fwd(x[w], h[w])])
    elif kernel == "k3_bwd":
        go = _rand(T, 1)
        outs = K.k3_bwd(go, x, h, grad_x=_nan(T, 4, 1), grad_h_pre=_nan(T, 4, dtype=torch.float32))
        _check(outs, lambda w: K.k3_bwd(go[w], x[w], h[w]))
    else:
        H, lo = _rand(T, 4, 4, dtype=torch.float32), _rand(T, 1)
        if kernel == "k4_fwd":
            out = K.k4_fwd(x, lo, H, h, out=_nan(T, 4, 1))
            _check([out], lambda w: [K.k4_fwd(x[w], lo[w], H[w], h[w])])
        else:
            go = _rand(T, 4, 1)
            outs = K.k4_bwd(go, x, lo, H, h, grad_x=_nan(T, 4, 1), grad_layer_output=_nan(T, 1),
                            grad_H=_nan(T, 4, 4, dtype=torch.float32), grad_h_post=_nan(T, 4, dtype=torch.float32))
            _check(outs, lambda w: K.k4_bwd(go[w], x[w], lo[w], H[w], h[w]))
    del x, h
    torch.cuda.empty_cache()


def test_element_wise_k1():
    tokens, nC = (1 << 26) + 40, 7
    seam = ((1 << 32) - 1) // 256 * 4 & ~7
    assert 0 < tokens - seam < 128
    windows = [slice(0, 90), slice(seam - 64, seam + 32), slice(tokens - 90, tokens)]
    x, W, go = _rand(tokens, nC), _rand(32, nC), _rand(tokens, 32)
    outs = K.k1_fwd(x, W, out=_nan(tokens, 32), inv_rms=_nan(tokens, dtype=torch.float32))
    _check(outs, lambda w: K.k1_fwd(x[w], W), windows)
    proj, inv = outs
    gx = K.k1_bwd_dx(go, x, W, proj, inv, grad_x=_nan(tokens, nC))
    _check([gx], lambda w: [K.k1_bwd_dx(go[w], x[w], W, proj[w], inv[w])], windows)
