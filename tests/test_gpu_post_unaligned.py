"""mhc_post and its backward on rows that are no multiple of 16 bytes or start
off a 16-byte boundary: the last lane of a row takes elements its neighbour
also has, which every output must hold once and every dot product count once.

Forward and grad_x / grad_h_out of the unaligned rows are bit-identical to the
same rows padded to an aligned width (same fp32 order, zero columns)."""

from __future__ import annotations

import pytest
import torch

import FlagOS_mhc as m
from test_gpu_post import DEV, post_inputs

pytestmark = pytest.mark.gpu

BF, HF, F32 = torch.bfloat16, torch.float16, torch.float32


def _pad(t, D, P):
    out = torch.zeros(*t.shape[:-1], P, device=DEV, dtype=t.dtype)
    out[..., :D] = t
    return out


def _shifted(t):
    buf = torch.empty(t.numel() + 1, device=DEV, dtype=t.dtype)
    buf[1:] = t.reshape(-1)
    return buf[1:].view(t.shape)


@pytest.mark.parametrize("dtype", [BF, HF, F32])
@pytest.mark.parametrize("N", [2, 4, 6, 8])
@pytest.mark.parametrize("T,D,shift", [(3, 1, False), (5, 3, False), (7, 9, False), (1, 511, False), (2, 513, False),
                                       (1030, 67, False), (70, 520, True), (1040, 1003, False), (4, 4099, False)])
def test_unaligned_rows(T, N, D, dtype, shift):
    print(f"[post unaligned] T={T} N={N} D={D} {dtype}", flush=True)
    x, h_res, h_out, h_post, gy = post_inputs(T, N, D, dtype, seed=D)
    P = (D + 15) // 8 * 8
    px, ph, pg = _pad(x, D, P), _pad(h_out, D, P), _pad(gy, D, P)
    if shift:
        x, h_out, gy = _shifted(x), _shifted(h_out), _shifted(gy)
    y = m.mhc_post(x, h_res, h_out, h_post)
    assert torch.equal(y, m.mhc_post(px, h_res, ph, h_post)[..., :D])
    gx, ghr, gho, ghp = m.mhc_post_backward(gy, x, h_res, h_out, h_post)
    wx, whr, who, whp = m.mhc_post_backward(pg, px, h_res, ph, h_post)
    torch.cuda.synchronize()
    assert torch.equal(gx, wx[..., :D]) and torch.equal(gho, who[..., :D])
    for got, want in ((ghr, whr), (ghp, whp)):  # the same products in another order
        assert bool(((got - want).abs() <= 1e-5 * want.abs().max() + 1e-5 * want.abs()).all())
    sx, shr, sho, shp = m.mhc_post_backward_sum(gy, gy, x, h_res, h_out, h_post)
    vx, vhr, vho, vhp = m.mhc_post_backward_sum(pg, pg, px, h_res, ph, h_post)
    assert torch.equal(sx, vx[..., :D]) and torch.equal(sho, vho[..., :D])
    for got, want in ((shr, vhr), (shp, vhp)):
        assert bool(((got - want).abs() <= 1e-5 * want.abs().max() + 1e-5 * want.abs()).all())
