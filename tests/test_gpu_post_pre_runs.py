"""The fused post + pre forward's tiles and runs (csrc/post_pre.hip): fewer
tiles than CUs, one token more than whole rounds of tiles, runs that start and
end inside a tile, whole rounds (heads in the kernel), against the two
operators in turn.  x_next is bit-identical; the others to the rounding of
differently ordered fp32 sums (rtol 1e-4, atol 1e-5 + 1e-4 max)."""

from __future__ import annotations

import pytest
import torch

import FlagOS_mhc as m
from FlagOS_mhc import _lib
from test_gpu_post import DEV, post_inputs
from test_gpu_pre import FWD_KEYS, pre_inputs

pytestmark = pytest.mark.gpu

BF = torch.bfloat16
KW = dict(norm_eps=1e-6, hc_eps=1e-6, clamp_min=-10.0, clamp_max=10.0, iter_times=20)
CASES = [(1, 256), (33, 320), (100, 7168), (1024, 256), (3000, 1024), (8191, 256), (8192, 320), (8193, 256),
         (8225, 448), (16384, 256), (16500, 512)]


def _close(got, want, what):
    got, want = got.float(), want.float()
    tol = 1e-5 + 1e-4 * want.abs().max() + 1e-4 * want.abs()
    assert bool(((got - want).abs() <= tol).all()), what


@pytest.mark.parametrize("T,D", CASES)
def test_runs_match_the_two_operators(T, D):
    print(f"[post_pre runs] T={T} D={D}", flush=True)
    x, h_res, h_out, h_post, _ = post_inputs(T, 4, D, BF, seed=T)
    _, phi, alpha, base, *_ = pre_inputs(1, 4, D, BF, BF, seed=D)
    x_next, out = m.mhc_post_pre_clamp_sinkhorn(x, h_res, h_out, h_post, phi, alpha, base, need_backward=True, **KW)
    y = m.mhc_post(x, h_res, h_out, h_post)
    want = m.mhc_pre_clamp_sinkhorn(y, phi, alpha, base, need_backward=True, **KW)
    torch.cuda.synchronize()
    assert torch.equal(x_next, y)
    for k in FWD_KEYS:
        _close(out[k], want[k], f"T={T} D={D} {k}")
    assert bool(((out["y"].float() - want["y"].float()).abs() <= 2e-2 + 2e-2 * want["y"].float().abs()).all())


def test_less_workspace_gives_the_same_results():
    T, N, D, M = 500, 4, 512, 24
    x, h_res, h_out, h_post, _ = post_inputs(T, N, D, BF, seed=1)
    _, phi, alpha, base, *_ = pre_inputs(1, N, D, BF, BF, seed=2)
    lib = _lib.load()
    f32 = dict(device=DEV, dtype=torch.float32)
    x_next, y = torch.empty_like(x), torch.empty(T, D, device=DEV, dtype=BF)
    post, comb = torch.empty(T, N, **f32), torch.empty(T, N, N, **f32)
    size = 256 + T * 20 + 512  # pre and inv_rms, no room for sums
    assert size < lib.mhc_post_pre_fwd_workspace_size(T, N, D, 1)
    ws = torch.empty(size, dtype=torch.uint8, device=DEV)
    rc = lib.mhc_post_pre_fwd(x.data_ptr(), h_res.data_ptr(), h_out.data_ptr(), h_post.data_ptr(), 1, phi.data_ptr(), 1,
                              alpha.data_ptr(), base.data_ptr(), 1e-6, 1e-6, -10.0, 10.0, 20, x_next.data_ptr(),
                              y.data_ptr(), post.data_ptr(), comb.data_ptr(), None, None, None, None, ws.data_ptr(),
                              size, T, N, D, torch.cuda.current_stream().cuda_stream)
    _lib.check(rc, "mhc_post_pre_fwd")
    xw, want = m.mhc_post_pre_clamp_sinkhorn(x, h_res, h_out, h_post, phi, alpha, base, **KW)
    torch.cuda.synchronize()
    assert torch.equal(x_next, xw)
    _close(post, want["post_out"], "post_out")
    _close(comb, want["comb_frag"], "comb_frag")


def _c_call(x, h_res, h_out, h_post, phi, alpha, base, ws, size):
    """mhc_post_pre_fwd in the first `size` bytes of ws: (x_next, dict)."""
    T, N, D = x.shape
    f32 = dict(device=DEV, dtype=torch.float32)
    x_next, y = torch.empty_like(x), torch.empty(T, D, device=DEV, dtype=BF)
    o = {"post_out": torch.empty(T, N, **f32), "comb_frag": torch.empty(T, N, N, **f32), "inv_rms": torch.empty(T, **f32),
         "mixes": torch.empty(T, 24, **f32), "h_res_logits": torch.empty(T, N, N, **f32), "pre": torch.empty(T, N, **f32)}
    rc = _lib.load().mhc_post_pre_fwd(
        x.data_ptr(), h_res.data_ptr(), h_out.data_ptr(), h_post.data_ptr(), 1, phi.data_ptr(), 1, alpha.data_ptr(),
        base.data_ptr(), 1e-6, 1e-6, -10.0, 10.0, 20, x_next.data_ptr(), y.data_ptr(), *(t.data_ptr() for t in o.values()),
        ws.data_ptr(), size, T, N, D, torch.cuda.current_stream().cuda_stream)
    _lib.check(rc, "mhc_post_pre_fwd")
    return x_next, dict(o, y=y)


@pytest.mark.parametrize("T,D", [(1, 256), (100, 7168), (3000, 1024), (8193, 256), (8225, 448), (16500, 512), (24700, 5120)])
def test_sums_stay_in_the_workspace(T, D):
    """The workspace that is asked for, with a guard region behind it."""
    print(f"[post_pre runs] guarded workspace T={T} D={D}", flush=True)
    x, h_res, h_out, h_post, _ = post_inputs(T, 4, D, BF, seed=T)
    _, phi, alpha, base, *_ = pre_inputs(1, 4, D, BF, BF, seed=D)
    size, guard = _lib.load().mhc_post_pre_fwd_workspace_size(T, 4, D, 1), 4 << 20
    ws = torch.full((size + guard,), 0x5a, dtype=torch.uint8, device=DEV)
    x_next, out = _c_call(x, h_res, h_out, h_post, phi, alpha, base, ws, size)
    y = m.mhc_post(x, h_res, h_out, h_post)
    want = m.mhc_pre_clamp_sinkhorn(y, phi, alpha, base, need_backward=True, **KW)
    torch.cuda.synchronize()
    assert bool((ws[size:] == 0x5a).all())
    assert torch.equal(x_next, y)
    for k in FWD_KEYS:
        _close(out[k], want[k], f"T={T} D={D} {k}")


@pytest.mark.parametrize("T,D", [(1, 256), (33, 7168), (500, 512), (8193, 256), (9000, 1024), (16500, 320)])
def test_whole_tiles_without_room_for_sums(T, D):
    """A workspace that holds pre and inv_rms only: the fused kernel in whole
    tiles, one a block in the last round (it leaves pre at the workspace's
    start; the two operators in turn do not)."""
    print(f"[post_pre runs] whole tiles T={T} D={D}", flush=True)
    x, h_res, h_out, h_post, _ = post_inputs(T, 4, D, BF, seed=T)
    _, phi, alpha, base, *_ = pre_inputs(1, 4, D, BF, BF, seed=D)
    size, guard = (16 * T + 255) // 256 * 256 + (4 * T + 255) // 256 * 256, 1 << 20
    ws = torch.full((size + guard,), 0x5a, dtype=torch.uint8, device=DEV)
    x_next, out = _c_call(x, h_res, h_out, h_post, phi, alpha, base, ws, size)
    y = m.mhc_post(x, h_res, h_out, h_post)
    want = m.mhc_pre_clamp_sinkhorn(y, phi, alpha, base, need_backward=True, **KW)
    torch.cuda.synchronize()
    assert bool((ws[size:] == 0x5a).all())
    assert torch.equal(ws[:16 * T].view(torch.float32), out["pre"].reshape(-1))
    assert torch.equal(x_next, y)
    for k in FWD_KEYS:
        _close(out[k], want[k], f"T={T} D={D} {k}")
    assert bool(((out["y"].float() - want["y"].float()).abs() <= 2e-2 + 2e-2 * want["y"].float().abs()).all())
