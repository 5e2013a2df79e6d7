"""K3 and K4 for more tokens than one launch can hold: a HIP launch stays below
2^32 threads, eight lanes per token at C = 1 reach that at T = 2^29, and the
entry points then launch pieces of the tokens.  Every output element must be
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


def _check(outs, alone):
    for o in outs:
        for piece in o.view(-1).split(1 << 28):
            assert not bool(torch.isnan(piece).any())
    for w in WINDOWS:
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
