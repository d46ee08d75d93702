"""The pre forward's general contraction and finish kernels (csrc/pre_fwd_gen.hpp)
at the edges of their tiles, runs and pieces, against the float64 oracle.

Tolerances as in test_gpu_pre.py; with fp32 x and phi the three-plane products
keep the mixes within 1e-4 and y is fp32, rtol / atol 1e-5."""

from __future__ import annotations

import pytest
import torch

import FlagOS_mhc as m
from FlagOS_mhc import _lib
from FlagOS_mhc.mhc_pre_clamp_sinkhorn import _pre_forward
from test_gpu_post import DEV, _subset, assert_close
from test_gpu_pre import FWD_KEYS, _oracle_fwd, check_fwd, pre_inputs

pytestmark = pytest.mark.gpu

BF, HF, F32 = torch.bfloat16, torch.float16, torch.float32

CASES = [
    # T, N, D, x, phi: 16-token tiles (T <= 64), one stage a tile or several
    # tiles a block; K and D that end inside a stage, a 32-column step, an
    # 8-element group and a 4-element piece
    (1, 4, 7168, BF, F32), (1, 4, 64, F32, F32), (2, 8, 9, HF, F32), (16, 4, 1003, HF, HF), (17, 8, 200, BF, F32),
    (64, 4, 4096, BF, F32), (64, 8, 1031, F32, F32), (33, 4, 3, BF, BF), (5, 8, 2048, BF, F32),
    # 128-token tiles: one token past a tile, runs that end inside a tile
    # (65 tiles), the finish kernel's largest T and one more
    (65, 4, 256, F32, F32), (128, 4, 1003, HF, HF), (129, 4, 515, BF, F32), (777, 4, 4096, BF, F32),
    (2048, 4, 130, HF, F32), (2049, 4, 1003, HF, HF), (8193, 4, 3584, BF, F32), (2049, 8, 517, BF, F32),
    (3000, 8, 1024, F32, F32), (1025, 8, 640, HF, HF), (1030, 8, 333, HF, BF), (1030, 4, 1030, F32, BF),
    (2500, 4, 6001, F32, F32), (66000, 4, 24, BF, F32),
    # finish blocks of more waves than rows of 512 columns (N = 8, at most 1024 tokens)
    (1, 8, 1024, BF, F32), (257, 8, 513, F32, F32), (1024, 8, 640, HF, HF),
]


def _kw(clamp=10.0, iters=20):
    return dict(norm_eps=1e-6, hc_eps=1e-6, clamp_min=-clamp, clamp_max=clamp, iter_times=iters)


def _check(x, phi, alpha, base, kw, what):
    T, dtype = x.shape[0], x.dtype
    out = m.mhc_pre_clamp_sinkhorn(x, phi, alpha, base, need_backward=True, **kw)
    torch.cuda.synchronize()
    idx = _subset(T, k=48, seed=T)
    want = _oracle_fwd(idx, x, phi, alpha, base, kw)
    check_fwd(out, want, dtype, idx, what)
    if dtype == F32:
        assert_close(out["y"][idx], want["y"], 1e-5, 1e-5, what + " y")
    assert_close(out["x_scaled"][idx], want["x_scaled"], 1e-5, 1e-6, what + " x_scaled")
    small = m.mhc_pre_clamp_sinkhorn(x, phi, alpha, base, **kw)
    for k in small:
        assert torch.equal(small[k], out[k]), what + " " + k
    return out


@pytest.mark.parametrize("T,N,D,dtype,phi_dtype", CASES)
def test_general_contraction(T, N, D, dtype, phi_dtype):
    print(f"[pre_fwd general] T={T} N={N} D={D} {dtype} phi={phi_dtype}", flush=True)
    x, phi, alpha, base, *_ = pre_inputs(T, N, D, dtype, phi_dtype, seed=T + D)
    _check(x, phi, alpha, base, _kw(iters=7 if D % 2 else 20), f"T={T} N={N} D={D}")


@pytest.mark.parametrize("dtype,phi_dtype,T", [(BF, F32, 70), (HF, HF, 3), (F32, F32, 200), (BF, BF, 300)])
def test_unaligned_bases(dtype, phi_dtype, T):
    """x, phi and the gates as views one element into their storage."""
    N, D = 4, 520
    x, phi, alpha, base, *_ = pre_inputs(T, N, D, dtype, phi_dtype, seed=5)

    def shifted(t):
        buf = torch.empty(t.numel() + 1, device=DEV, dtype=t.dtype)
        buf[1:] = t.reshape(-1)
        return buf[1:].view(t.shape)

    print(f"[pre_fwd general] unaligned {dtype} {phi_dtype} T={T}", flush=True)
    got = _check(shifted(x), shifted(phi), alpha, base, _kw(), "unaligned")
    if (dtype, phi_dtype) != (BF, BF):  # the aligned bf16 pair has a kernel of its own
        want = m.mhc_pre_clamp_sinkhorn(x, phi, alpha, base, need_backward=True, **_kw())
        for k in want:
            assert torch.equal(got[k], want[k]), k


def test_inf_and_nan_rows_stay_in_their_rows():
    """An infinite or NaN activation spoils its own token only (D ends inside
    a stage: the columns past it must not meet the value)."""
    x, phi, alpha, base, *_ = pre_inputs(140, 4, 133, BF, F32, seed=3)
    clean = m.mhc_pre_clamp_sinkhorn(x, phi, alpha, base, **_kw())
    x = x.clone()
    x[3, 3, 132], x[137, 0, 0] = float("inf"), float("nan")
    out = m.mhc_pre_clamp_sinkhorn(x, phi, alpha, base, **_kw())
    torch.cuda.synchronize()
    keep = torch.ones(140, dtype=torch.bool, device=DEV)
    keep[[3, 137]] = False
    for k in clean:
        assert torch.equal(out[k][keep], clean[k][keep]), k
    assert not torch.isfinite(out["y"][137].float()).any()


@pytest.mark.parametrize("share,T", [(1.0, 9000), (0.6, 9000), (0.0, 300)])
def test_workspace_smaller_than_asked(share, T):
    """mhc_pre_fwd with less workspace than mhc_pre_fwd_workspace_size: the
    tokens in chunks that fit, or the form that keeps no sums in memory; the
    same results to rounding."""
    N, D = 4, 260
    x, phi, alpha, base, *_ = pre_inputs(T, N, D, BF, F32, seed=9)
    lib, M = _lib.load(), 24
    full = lib.mhc_pre_fwd_workspace_size(T, N, D, 0)
    planes = 3 * M * N * D * 2
    want = m.mhc_pre_clamp_sinkhorn(x, phi, alpha, base, need_backward=True, **_kw())
    f32 = dict(device=DEV, dtype=F32)
    o = {"y": torch.empty(T, D, device=DEV, dtype=BF), "post_out": torch.empty(T, N, **f32),
         "comb_frag": torch.empty(T, N, N, **f32), "inv_rms": torch.empty(T, **f32),
         "mixes": torch.empty(T, M, **f32), "h_res_logits": torch.empty(T, N, N, **f32),
         "pre": torch.empty(T, N, **f32), "x_scaled": torch.empty(T, N * D, **f32)}
    size = max(int(full * share), planes)
    ws = torch.empty(size, dtype=torch.uint8, device=DEV)
    print(f"[pre_fwd general] workspace {size} of {full}", flush=True)
    rc = lib.mhc_pre_fwd(x.data_ptr(), 1, phi.data_ptr(), 0, alpha.data_ptr(), base.data_ptr(), 1e-6, 1e-6, -10.0,
                         10.0, 20, *(t.data_ptr() for t in o.values()), ws.data_ptr(), size, T, N, D,
                         torch.cuda.current_stream().cuda_stream)
    _lib.check(rc, "mhc_pre_fwd")
    torch.cuda.synchronize()
    assert_close(o["y"], want["y"].double().cpu().numpy(), 2e-2, 2e-2, "y")
    for k in FWD_KEYS:
        assert_close(o[k], want[k].double().cpu().numpy(), 1e-4, 1e-5, k)
    assert_close(o["x_scaled"], want["x_scaled"].double().cpu().numpy().reshape(T, N * D), 1e-5, 1e-6, "x_scaled")


@pytest.mark.parametrize("T,N,D,size", [(16512, 4, 256, 4326656), (8297, 4, 512, 3900000), (11826, 8, 82, 13861120)])
def test_chunks_write_inside_the_workspace(T, N, D, size):
    """Chunks whose last, shorter piece would by a plan of its own take more
    slots than a whole one: the bytes behind the workspace stay as they are,
    and every output is that of the call with the full workspace, to rounding."""
    print(f"[pre_fwd general] guarded workspace T={T} N={N} D={D} {size}", flush=True)
    x, phi, alpha, base, *_ = pre_inputs(T, N, D, BF, F32, seed=D)
    lib = _lib.load()
    full, guard = lib.mhc_pre_fwd_workspace_size(T, N, D, 0), 16 << 20
    assert size < full < size + guard
    want = m.mhc_pre_clamp_sinkhorn(x, phi, alpha, base, **_kw())
    ws = torch.full((size + guard,), 0x5a, dtype=torch.uint8, device=DEV)
    y, post = torch.empty(T, D, device=DEV, dtype=BF), torch.empty(T, N, device=DEV, dtype=F32)
    comb = torch.empty(T, N, N, device=DEV, dtype=F32)
    rc = lib.mhc_pre_fwd(x.data_ptr(), 1, phi.data_ptr(), 0, alpha.data_ptr(), base.data_ptr(), 1e-6, 1e-6, -10.0,
                         10.0, 20, y.data_ptr(), post.data_ptr(), comb.data_ptr(), None, None, None, None, None,
                         ws.data_ptr(), size, T, N, D, torch.cuda.current_stream().cuda_stream)
    _lib.check(rc, "mhc_pre_fwd")
    torch.cuda.synchronize()
    assert bool((ws[size:] == 0x5a).all())
    assert_close(y, want["y"].double().cpu().numpy(), 2e-2, 2e-2, "y")
    assert_close(post, want["post_out"].double().cpu().numpy(), 1e-4, 1e-5, "post_out")
    assert_close(comb, want["comb_frag"].double().cpu().numpy(), 1e-4, 1e-5, "comb_frag")


@pytest.mark.parametrize("which", ["x", "phi", "both"])
@pytest.mark.parametrize("T,D", [(1, 7168), (40, 1024), (8200, 520), (16157, 1040)])
def test_unaligned_bf16_calls_get_the_general_workspace(T, D, which):
    """bf16 x and phi one element into their storage, few tokens and many:
    such a call runs the general form and needs its workspace (a phi that is
    not aligned was refused at few tokens, its planes not fitting)."""
    N = 4
    print(f"[pre_fwd general] unaligned bf16 {which} T={T} D={D}", flush=True)
    x, phi, alpha, base, *_ = pre_inputs(T, N, D, BF, BF, seed=T)
    want = m.mhc_pre_clamp_sinkhorn(x, phi, alpha, base, **_kw())

    def shifted(t):
        buf = torch.empty(t.numel() + 1, device=DEV, dtype=t.dtype)
        buf[1:] = t.reshape(-1)
        return buf[1:].view(t.shape)

    xs, ps = (shifted(x) if which != "phi" else x), (shifted(phi) if which != "x" else phi)
    assert _lib.pre_fwd_size_code(1, 1, xs.data_ptr() | ps.data_ptr()) == 0
    assert _lib.pre_fwd_size_code(1, 1, x.data_ptr() | phi.data_ptr()) == 1
    out = m.mhc_pre_clamp_sinkhorn(xs, ps, alpha, base, **_kw())
    h_res, h_post = want["comb_frag"], want["post_out"]
    h_out = x[:, 0].contiguous()
    x_next, fused = m.mhc_post_pre_clamp_sinkhorn(xs, h_res, h_out, h_post, ps, alpha, base, **_kw())
    x_want, fused_want = m.mhc_post_pre_clamp_sinkhorn(x, h_res, h_out, h_post, phi, alpha, base, **_kw())
    torch.cuda.synchronize()
    assert torch.equal(x_next, x_want)
    for got, ref in ((out, want), (fused, fused_want)):
        assert_close(got["y"], ref["y"].double().cpu().numpy(), 2e-2, 2e-2, "y")
        for k in ("post_out", "comb_frag"):
            assert_close(got[k], ref[k].double().cpu().numpy(), 1e-4, 1e-5, k)


@pytest.mark.parametrize("T,N,D,dtype", [(65536, 4, 4096, BF), (65536, 8, 1031, BF), (32768, 4, 4096, HF)])
def test_inv_rms_of_long_runs(T, N, D, dtype):
    """Many tokens, so that a block sums most of a row by itself: inv_rms keeps
    fp32 accuracy.  A lane adds at most 260 stages' squares (32 or 16 each, in
    chains of their own) to its quarter of the row; 260 roundings of at most
    2^-24 of the running sum, at random, are below sqrt(260 / 3) 2^-24 = 5.6e-7
    of it, four quarters and the square root take that to 1.4e-7, and inv_rms
    itself is rounded (2^-24): 3e-7 in 2-norm (one chain over the run:
    1e-6 to 3e-6)."""
    print(f"[pre_fwd general] inv_rms T={T} N={N} D={D} {dtype}", flush=True)
    x, phi, alpha, base, *_ = pre_inputs(T, N, D, dtype, F32, seed=7)
    got = _pre_forward(x, phi, alpha, base, 1e-6, 1e-6, -10.0, 10.0, 20, True, False)["inv_rms"]
    want = torch.cat([torch.rsqrt(c.double().reshape(len(c), -1).square().mean(1) + 1e-6) for c in x.split(4096)])
    assert float((got.double() - want).norm() / want.norm()) < 3e-7


def test_more_tokens_than_a_launch_takes():
    """A chunk and 777 tokens of a second one, in the workspace that is asked for."""
    T, N, D = (1 << 22) - 128 + 777, 4, 3
    print(f"[pre_fwd general] T={T} N={N} D={D}", flush=True)
    x, phi, alpha, base, *_ = pre_inputs(T, N, D, F32, F32, seed=2)
    out = _pre_forward(x, phi, alpha, base, 1e-6, 1e-6, -10.0, 10.0, 20, True, True)
    torch.cuda.synchronize()
    idx = torch.cat([_subset(T, k=48, seed=T), torch.arange((1 << 22) - 140, (1 << 22) - 110, device=DEV)])
    want = _oracle_fwd(idx, x, phi, alpha, base, _kw())
    check_fwd(out, want, F32, idx, "two chunks")
    assert_close(out["x_scaled"][idx], want["x_scaled"], 1e-5, 1e-6, "x_scaled")
