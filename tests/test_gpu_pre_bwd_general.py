"""The pre backward's general kernel (csrc/pre_bwd_gen.hpp) where its pieces
end: widths that are no multiple of a lane's four columns (a lane's columns
run on into the next stream), fewer columns than a lane holds, tokens around
a tile, unaligned bases, grad_x_in.

grad_x: bf16 / fp16 at rtol / atol 2e-2; fp32 within 1e-4 of max|grad_x| (two
bf16 planes of grad_mixes and phi leave 2^-16 of the product's terms).  The
token reductions as everywhere, rtol 1e-4 with atol 1e-5 max|ref|."""

from __future__ import annotations

import pytest
import torch

import FlagOS_mhc as m
from FlagOS_mhc.mhc_pre_clamp_sinkhorn import _pre_forward
from FlagOS_mhc.mhc_pre_clamp_sinkhorn_backward import _pre_backward
from gpu_ref import check_reductions, pre_bwd_fp64
from oracle import mhc_oracle as orc
from test_gpu_post import DEV, _np, _subset, assert_close
from test_gpu_pre import pre_inputs

pytestmark = pytest.mark.gpu

BF, HF, F32 = torch.bfloat16, torch.float16, torch.float32
KW = dict(norm_eps=1e-6, hc_eps=1e-6, clamp_min=-10.0, clamp_max=10.0, iter_times=20)

CASES = [
    (1, 4, 1, F32, F32), (17, 4, 2, HF, HF), (40, 8, 3, BF, BF), (5, 4, 4, BF, F32), (16, 4, 5, F32, F32),
    (15, 8, 5, HF, HF), (33, 4, 63, BF, BF), (64, 4, 65, HF, F32), (31, 4, 66, F32, F32), (100, 8, 67, BF, F32),
    (129, 4, 1003, HF, HF), (2049, 4, 1003, BF, BF), (300, 8, 517, F32, F32), (1030, 8, 1029, HF, F32),
    (70, 4, 1028, BF, BF), (257, 4, 2048, F32, F32), (700, 8, 1024, HF, HF), (1000, 4, 1000, HF, F32),
]


def _shifted(t):
    buf = torch.empty(t.numel() + 1, device=DEV, dtype=t.dtype)
    buf[1:] = t.reshape(-1)
    return buf[1:].view(t.shape)


def _check(T, N, D, dtype, phi_dtype, what, shift=False, gin=False):
    x, phi, alpha, base, gy, gpost, gcomb = pre_inputs(T, N, D, dtype, phi_dtype, seed=T + 3 * D)
    if shift:
        x, gy = _shifted(x), _shifted(gy)
    out = m.mhc_pre_clamp_sinkhorn(x, phi, alpha, base, need_backward=True, **KW)
    add = torch.randn(x.shape, device=DEV).to(dtype) if gin else None
    if gin and shift:
        add = _shifted(add)
    gx, gphi, ga, gb = _pre_backward(x, phi, alpha, base, out["inv_rms"], out["mixes"], out["pre"], gy, gpost, gcomb,
                                     1e-6, 1e-6, -10.0, 10.0, 20, grad_x_in=add)
    torch.cuda.synchronize()
    idx = _subset(T, k=40, seed=T)
    want = orc.pre_bwd(_np(x[idx]), _np(phi), _np(alpha), _np(base), _np(gy[idx]), _np(gpost[idx]), _np(gcomb[idx]),
                       **KW)[0]
    if gin:
        want = want + _np(add[idx])
    scale = abs(want).max()
    tol = (0.0, 1e-4 * scale) if dtype == F32 else (2e-2, 2e-2)
    assert_close(gx[idx], want, *tol, what + " grad_x")
    ref = pre_bwd_fp64(x, phi, alpha, base, gy, gpost, gcomb, KW)
    check_reductions(gphi, ga, gb, ref, what)
    return gx, gphi


@pytest.mark.parametrize("T,N,D,dtype,phi_dtype", CASES)
def test_general_backward(T, N, D, dtype, phi_dtype):
    print(f"[pre_bwd general] T={T} N={N} D={D} {dtype} phi={phi_dtype}", flush=True)
    _check(T, N, D, dtype, phi_dtype, f"T={T} N={N} D={D}")


@pytest.mark.parametrize("T,N,D,dtype,phi_dtype", [(50, 4, 520, BF, BF), (50, 8, 264, HF, F32), (20, 4, 131, F32, F32)])
def test_unaligned_bases_and_grad_x_in(T, N, D, dtype, phi_dtype):
    print(f"[pre_bwd general] unaligned T={T} N={N} D={D} {dtype}", flush=True)
    _check(T, N, D, dtype, phi_dtype, "unaligned", shift=True)
    _check(T, N, D, dtype, phi_dtype, "unaligned, grad_x_in", shift=True, gin=True)
    _check(T, N, D, dtype, phi_dtype, "grad_x_in", gin=True)


@pytest.mark.parametrize("T,N,D,dtype", [(32768, 8, 4100, BF), (32768, 4, 8190, BF)])
def test_grad_phi_of_long_chains(T, N, D, dtype):
    """Wide rows and many tokens: few token splits, a block walks 680 or 2048
    tiles.  bf16 x is exact; the two bf16 planes of g leave at most 2^-18 of
    each term, at random, 2^-18 / sqrt(3) = 2.2e-6 of the sum in 2-norm; fp32
    sums and the forward's mixes add some 1e-7 (one MFMA chain over a block's
    tiles: 3.2e-6 and 3.4e-6)."""
    print(f"[pre_bwd general] grad_phi chains T={T} N={N} D={D} {dtype}", flush=True)
    x, phi, alpha, base, gy, gpost, gcomb = pre_inputs(T, N, D, dtype, dtype, seed=1)
    out = _pre_forward(x, phi, alpha, base, 1e-6, 1e-6, -10.0, 10.0, 20, True, False)
    gphi = _pre_backward(x, phi, alpha, base, out["inv_rms"], out["mixes"], out["pre"], gy, gpost, gcomb,
                         1e-6, 1e-6, -10.0, 10.0, 20)[1]
    want = pre_bwd_fp64(x, phi, alpha, base, gy, gpost, gcomb, KW)["grad_phi"]
    assert float((gphi.double().reshape(want.shape) - want).norm() / want.norm()) < 2.7e-6
