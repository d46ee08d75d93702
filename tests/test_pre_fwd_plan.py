"""The plans of the general pre forward and of the fused post + pre forward
(csrc/pre_fwd_plan.hpp), on the CPU: whatever workspace a caller gives, every
sum that a block of any chunk writes, and the chunk's pre and inv_rms, lie
inside it, in regions of their own.  The walks repeat the kernels' indexing:
block b takes stages b * w .. of the tiles (fused: of those left after whole
rounds), and its sums of a tile go to slot b - tile * nst / w."""

from __future__ import annotations

import os
import shutil
import subprocess

import pytest

from conftest import PKG_DIR
from FlagOS_mhc import _lib

WALK = r"""
#include <stdio.h>
#include <stdlib.h>
#include <random>
#include "pre_fwd_plan.hpp"
using namespace mhc;

static long bad = 0, chunked = 0;

static void fail(const char* what, int64_t T, int N, int D, size_t bytes, int64_t n) {
  if (bad++ < 20)
    printf("%s: T=%lld N=%d D=%d workspace=%zu, chunk of %lld\n", what, (long long)T, N, D, bytes, (long long)n);
}

// one call in `bytes` of workspace
static void walk(int64_t T, int N, int D, int cus, size_t bytes) {
  const int64_t chunk = gen_chunk(T, N, D, cus, bytes);
  if (chunk <= 0) return;
  if (chunk < T) ++chunked;
  if (chunk * 1024 >= (int64_t)1 << 32) fail("too many threads", T, N, D, bytes, chunk);
  const GenPlan p = gen_plan(chunk, N, D, cus);
  const size_t room = bytes - kPreFwdWsBase, M = 2 * N + N * N;
  for (int64_t t0 = 0; t0 < T; t0 += chunk) {
    const int64_t n = T - t0 < chunk ? T - t0 : chunk;
    const int64_t ntiles = (n + p.tt - 1) / p.tt, total = ntiles * p.nst;
    int64_t rows = 0;  // of the sums: [slot][n]
    for (int64_t b = 0; b < p.blocks(n); ++b) {
      const int64_t u0 = b * p.w, u1 = u0 + p.w < total ? u0 + p.w : total;
      if (u0 >= u1) fail("a block without a run", T, N, D, bytes, n);
      for (int64_t tile = u0 / p.nst; tile <= (u1 - 1) / p.nst; ++tile) {
        const int64_t slot = b - tile * p.nst / p.w, last = (tile + 1) * p.tt < n ? (tile + 1) * p.tt : n;
        if (slot < 0) fail("a negative slot", T, N, D, bytes, n);
        if (slot * n + last > rows) rows = slot * n + last;
        if (slot >= ((tile + 1) * p.nst - 1) / p.w - tile * p.nst / p.w + 1) fail("a slot that is not added", T, N, D, bytes, n);
      }
    }
    if (p.blocks(n) * p.w < total) fail("stages without a block", T, N, D, bytes, n);
    if (rows * M * 4 > p.ssq_off) fail("sums past their region", T, N, D, bytes, n);
    if (p.ssq_off + rows * 4 > p.pre_off) fail("squares past their region", T, N, D, bytes, n);
    if (p.pre_off + (size_t)n * N * 4 > p.inv_off) fail("pre past its region", T, N, D, bytes, n);
    if (p.inv_off + (size_t)n * 4 > room) fail("past the workspace", T, N, D, bytes, n);
  }
}

// the fused forward: no row of sums written twice, none past its region, and
// no more of them than a few for every token that runs share
static void walk_fused(int64_t T, int D, int cus, bool whole_tiles) {
  const PostPrePlan p = post_pre_plan(T, D, cus, whole_tiles);
  const int64_t nst = D / kPPCW, ntiles = (T + kPPTile - 1) / kPPTile, left0 = p.rounds * p.blocks;
  const int64_t total = (ntiles - left0) * nst, regions = (int64_t)(p.ssq_off / (4 * kPPM));
  if (p.heads != (whole_tiles || total == 0)) fail("heads", T, kPPN, D, p.bytes, T);
  if (!p.heads && p.left != T - left0 * kPPTile) fail("left", T, kPPN, D, p.bytes, T);
  int64_t last = left0 * kPPTile < T ? left0 * kPPTile : T, covered = 0;  // rows of the whole tiles
  for (int64_t b = 0; b < p.blocks; ++b) {
    const int64_t u0 = b * p.w, u1 = u0 + p.w < total ? u0 + p.w : total;
    if (u0 < u1) covered += u1 - u0;
    for (int64_t i = u0 / nst; u0 < u1 && i <= (u1 - 1) / nst; ++i) {  // tile left0 + i
      const int64_t slot = b - i * nst / p.w;
      const int64_t n = (left0 + i + 1) * kPPTile < T ? (left0 + i + 1) * kPPTile : T;
      if (slot < 0 || slot >= ((i + 1) * nst - 1) / p.w - i * nst / p.w + 1) fail("slot", T, kPPN, D, p.bytes, T);
      if (p.heads && (i * nst < u0 || (i + 1) * nst > u1)) fail("part of a tile", T, kPPN, D, p.bytes, T);
      if (slot * p.left + n > last) last = slot * p.left + n;
    }
  }
  if (covered != total) fail("stages without a block", T, kPPN, D, p.bytes, T);
  if (!p.heads && (last > regions || p.ssq_off + last * 4 > p.y_off)) fail("sums past their region", T, kPPN, D, p.bytes, T);
  if (p.y_off + fwd_y_ws_bytes(T, kPPN) > p.bytes) fail("pre past the workspace", T, kPPN, D, p.bytes, T);
  if (p.heads && p.bytes > fwd_y_ws_bytes(T, kPPN)) fail("more than pre and inv_rms", T, kPPN, D, p.bytes, T);
  if ((int64_t)p.bytes > (T + 3 * (int64_t)kPPTile * cus) * 100 + 20 * T + 2048) fail("too much", T, kPPN, D, p.bytes, T);
}

int main() {
  // last chunks whose own plan would have shorter runs, and so more slots,
  // than a whole chunk's
  walk(16512, 4, 256, 256, 4326656);
  walk(8297, 4, 512, 256, 3900000);
  walk(16157, 4, 1040, 256, 5170944);
  // rows of a few elements: more tokens than a dispatch has blocks of 1024 threads for
  walk(70000000, 4, 8, 256, gen_ws_bytes(70000000, 4, 8, 256));
  walk(70000000, 8, 3, 256, gen_ws_bytes(70000000, 8, 3, 256) / 3);
  walk((int64_t)2147483647, 4, 1, 256, gen_ws_bytes(2147483647, 4, 1, 256));
  for (int whole = 0; whole < 2; ++whole) {
    walk_fused(65537, 5120, 256, whole);
    walk_fused(131104, 5120, 256, whole);
  }
  std::mt19937_64 rng(1);
  auto uni = [&](double a, double b) { return a + (b - a) * (double)(rng() >> 11) / 9007199254740992.0; };
  auto logu = [&](double a, double b) { return (int64_t)exp2(uni(log2(a), log2(b))); };
  for (int i = 0; i < 20000; ++i) {
    const int N = rng() % 3 ? 4 : 8, D = (int)logu(1, 8192), cus = rng() % 8 ? 256 : (int)logu(1, 304);
    const int64_t T = logu(1, 200000);
    const size_t full = gen_ws_bytes(T, N, D, cus);
    walk(T, N, D, cus, full);
    walk(T, N, D, cus, (size_t)(full * uni(0.02, 1.0)));
    walk_fused(T, (int)(64 * logu(4, 160)), cus, rng() & 1);
    // exactly what some chunk needs
    const int64_t c = gen_chunk(T, N, D, cus, (size_t)(full * uni(0.05, 1.0)));
    if (c > 0) walk(T, N, D, cus, gen_ws_bytes(c, N, D, cus));
  }
  printf("%ld calls in chunks, %ld faults\n", chunked, bad);
  return bad || chunked < 1000;
}
"""


def test_every_chunk_stays_in_the_workspace(tmp_path):
    cxx = shutil.which("g++") or shutil.which("clang++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    src, exe = tmp_path / "walk.cpp", tmp_path / "walk"
    src.write_text("#include <cmath>\nusing std::exp2; using std::log2;\n" + WALK)
    subprocess.run([cxx, "-std=c++17", "-O2", "-Wall", "-Werror", "-I", os.path.join(PKG_DIR, "csrc"), str(src), "-o",
                    str(exe)], check=True)
    p = subprocess.run([str(exe)], capture_output=True, text=True, timeout=100)
    assert p.returncode == 0, p.stdout


@pytest.mark.parametrize("T,D", [(65537, 5120), (65568, 2048), (131104, 5120), (8193, 256)])
def test_fused_workspace_of_a_token_more_than_whole_rounds(T, D):
    """The slots of the runs are those of the tokens left after whole rounds
    (at most 8192 tokens and their sums twice over), not of all tokens."""
    lib = _lib.load()
    most = lib.mhc_pre_fwd_workspace_size(T, 4, D, 1) + 100 * (T + 3 * 8192) + 20 * T
    assert lib.mhc_post_pre_fwd_workspace_size(T, 4, D, 1) <= most
