// Work split and workspace layout of the pre forward's general contraction
// (pre_fwd_gen.hpp) and of the fused post + pre forward (post_pre.hip).  Plain
// host C++ with no HIP in it: a test compiles it alone and walks the layouts of
// many shapes on the CPU.
#pragma once

#include <stddef.h>
#include <stdint.h>

namespace mhc {

inline size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }
inline int64_t round_up(int64_t v, int64_t m) { return (v + m - 1) / m * m; }

// Bytes the pre forward (and the fused post + pre forward) keep per call for
// pre (T, N) and inv_rms (T,) between their contraction and y kernels.
inline size_t fwd_y_ws_bytes(int64_t T, int N) { return align256((size_t)T * N * 4) + align256((size_t)T * 4); }

constexpr size_t kPreFwdWsBase = 256;  // workspace bytes before the sums

constexpr int kGenSmallT = 64;     // tokens up to which the 16-token tiles run
constexpr int kGenFewUnits = 128;  // .. and stages of 128-token tiles below which they do
constexpr int kGenMaxSlots = 128;  // slots of a tile's sums, at most about

// The split of a chunk of T tokens, and where its sums lie in the workspace.
// A call that takes its tokens in chunks has one plan, that of a whole chunk,
// for the shorter last one too: with the run length w fixed, fewer tokens are
// fewer runs and fewer rows of every slot.  (A plan of the last chunk's own
// could need more memory than a whole chunk's: w is a rounded-up quotient, and
// one tile less can halve it and double the slots.)
struct GenPlan {
  bool small = false;
  int nst = 0, tt = 0, slots = 0;
  int64_t w = 0;
  size_t ssq_off = 0, pre_off = 0, inv_off = 0, bytes = 0;  // the sums, at 0, of squares, pre and inv_rms
  // blocks that n <= T tokens take
  int64_t blocks(int64_t n) const { return ((n + tt - 1) / tt * nst + w - 1) / w; }
};

inline GenPlan gen_plan(int64_t T, int N, int D, int cus) {
  GenPlan p;
  if (T <= 0) return p;
  const int M = 2 * N + N * N, cw = N == 8 ? 64 : 128;
  const int64_t K = (int64_t)N * D;
  p.small = T <= kGenSmallT || (T + 127) / 128 * ((K + cw - 1) / cw) < kGenFewUnits;
  const int cws = N == 8 || !p.small ? cw : 256;
  p.tt = p.small ? 16 : 128;
  p.nst = (int)((K + cws - 1) / cws);
  const int64_t total = (T + p.tt - 1) / p.tt * p.nst;
  const int64_t resident = 2 * (int64_t)cus;
  p.w = (total + resident - 1) / resident;
  if (p.w < (p.nst + kGenMaxSlots - 1) / kGenMaxSlots) p.w = (p.nst + kGenMaxSlots - 1) / kGenMaxSlots;
  p.slots = (int)((p.nst + p.w - 1) / p.w) + 1;
  if (p.slots > p.blocks(T)) p.slots = (int)p.blocks(T);
  p.ssq_off = align256((size_t)p.slots * T * M * 4);
  p.pre_off = p.ssq_off + align256((size_t)p.slots * T * 4);
  p.inv_off = p.pre_off + align256((size_t)T * N * 4);
  p.bytes = p.pre_off + fwd_y_ws_bytes(T, N);
  return p;
}

// Tokens a call of the general form takes at a time in `bytes` of workspace:
// all of them, or a multiple of the tile of at least kGenMinChunk (below that
// 0: the caller runs the form that needs no sums in memory).  At most
// kGenMaxChunk: the kernels after the contraction have a block of up to 1024
// threads a token, and a dispatch less than 2^32 threads.
constexpr int64_t kGenMinChunk = 4096, kGenMaxChunk = ((int64_t)1 << 22) - 128;
inline int64_t gen_chunk(int64_t T, int N, int D, int cus, size_t bytes) {
  if (bytes <= kPreFwdWsBase) return 0;
  bytes -= kPreFwdWsBase;
  int64_t c = T < kGenMaxChunk ? T : kGenMaxChunk;
  while (gen_plan(c, N, D, cus).bytes > bytes) {
    c = round_up(c / 2, 128);
    if (c < kGenMinChunk || c >= T) return 0;
  }
  return c;
}

// Workspace of the general form's largest chunk of T tokens.
inline size_t gen_ws_bytes(int64_t T, int N, int D, int cus) {
  return kPreFwdWsBase + gen_plan(T < kGenMaxChunk ? T : kGenMaxChunk, N, D, cus).bytes;
}

// ---- fused post + pre forward ------------------------------------------------
constexpr int kPPN = 4, kPPM = 24;  // streams, and columns of mixes
constexpr int kPPTile = 32;         // tokens of a tile
constexpr int kPPCW = 64;           // columns of a stage

// One block a CU (its LDS).  Whole tiles in rounds over all CUs, in an order
// that keeps the blocks on neighbouring tiles (runs of several tiles a block
// were 10% slower at D = 2048), then runs of equal length over the tiles left;
// at most about 64 slots of sums a tile for the finish kernel to add.  A token
// t of the whole tiles has one row of sums, row t; the `left` after them have
// `slots`, row s * left + t in slot s.  With whole rounds only, or with
// `whole_tiles` (a tile left a block, for a workspace without room for sums),
// the kernel runs the heads itself and keeps none.
struct PostPrePlan {
  int64_t w = 1, blocks = 0, left = 0;
  int rounds = 0, slots = 0;
  bool heads = false;
  size_t ssq_off = 0, y_off = 0, bytes = 0;
};
inline PostPrePlan post_pre_plan(int64_t T, int32_t D, int cus, bool whole_tiles = false) {
  PostPrePlan p;
  if (T <= 0) return p;
  const int64_t nst = D / kPPCW, ntiles = (T + kPPTile - 1) / kPPTile;
  p.rounds = (int)(ntiles / cus);
  const int64_t whole = (int64_t)p.rounds * cus, total = (ntiles - whole) * nst;
  p.heads = whole_tiles || total == 0;
  p.w = p.heads ? nst : (total + cus - 1) / cus;
  if (p.w < (nst + 63) / 64) p.w = (nst + 63) / 64;
  p.blocks = p.rounds ? cus : (total + p.w - 1) / p.w;
  if (!p.heads) {
    p.left = T - whole * kPPTile;
    p.slots = (int)((nst + p.w - 1) / p.w) + 1;
    if (p.slots > p.blocks) p.slots = (int)p.blocks;
    const int64_t rows = T - p.left + p.slots * p.left;
    p.ssq_off = align256((size_t)rows * kPPM * 4);
    p.y_off = p.ssq_off + align256((size_t)rows * 4);
  }
  p.bytes = p.y_off + fwd_y_ws_bytes(T, kPPN);
  return p;
}

}  // namespace mhc
