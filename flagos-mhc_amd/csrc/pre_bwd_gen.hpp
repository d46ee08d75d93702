// The pre backward's general kernel B: any activation dtype, any D and
// alignment, N = 4 or 8 (aligned bf16 rows take the LDS-pipelined kernel).
// Included by pre_bwd.hip.
//
// Columns are those of the flat row k = n D + d: x, grad_x, phi and grad_phi
// all have that layout, so their pieces keep the row's alignment (8 bytes at
// least for 2-byte types, N D being a multiple of 4) whatever D is, and only
// grad_y, a ninth of the bytes, is read at each stream's own alignment.  A
// wave owns 64 columns of a stream (cut at multiples of four flat columns), a
// block's four waves those of four streams, so that they read the same
// grad_y; it walks the 16-token tiles split, split + nsplit, ...  Lane (r, q) holds, for the tile's tokens
// 4 q .. 4 q + 3, the 4 columns k0 + 4 r .. of x and grad_y: one load a row,
// the next tile's rows loaded before this tile's work.
//   * grad_phi += g^T x (MFMA 16x16x32, both planes of g as its k: element
//     (plane, token) of g^T, kernel A's layout, against the token's x twice):
//     column c of the lane's 4 x 4 block, as bf16 planes (1 for bf16, 2 for
//     fp16, exact, and fp32, 2^-17), is the B operand; the instance covers
//     the columns 4 r + c, r = 0..15.
//   * gs = grad_mixes phi (MFMA 16x16x32 over m): A = the tokens' grad_mixes
//     rows, B = phi^T rows kept in registers.  Lane (r, q) of the result holds
//     the tokens and columns that it loaded, so
//     grad_x = grad_y pre + inv gs + scale x (+ grad_x_in) is formed and
//     stored in place.
// gs comes first: its operands arrive first, and grad_phi's conversions of x
// then run between MFMAs (N = 8, one wave a SIMD, T = 8192, D = 1024 fp16: 193
// us the other way round, 164 so; N = 4 equal).
// grad_phi is added in MFMA chains of 64 tiles, which meet in fp32 sums in
// LDS by round-to-nearest adds: one chain over a block's tiles drifts with
// their number (2-norm error against 64 bits, bf16, one chain / so: N = 8, D =
// 8191, T = 32768 4.2e-6 / 2.5e-6; N = 4, D = 8191, T = 65536 4.1e-6 / 2.5e-6).
// No barriers: a wave waits for nothing but its own loads.  It replaces a
// kernel that staged 32 tokens x 256 columns in LDS (element by element for
// unaligned rows) between barriers.  Measured, whole backward on MI355X, eager,
// before -> after (in a replayed graph): fp16, N = 4, T = 8192: D = 1003 291 ->
// 115 us (99), D = 1024 145 -> 80 (66); bf16 T = 16384, D = 907 510 -> 174
// (145); fp32 T = 8192, D = 2048 248 -> 215 (202; this kernel 132: 3.5 TB/s),
// N = 8, D = 1024 449 -> 271 (with gs last; 251 in a graph, 246 with gs first).
// Bound by issue at N = 8 (MFMA, conversions) and by loads in flight at N = 4.
// What the four rows' loads may not meet is a branch or a use before the next
// tile's: a wave that joins two streams' columns at load time took twice as
// long, and the whole grid waits for it.
#pragma once

namespace mhc {

template <int N, typename S> struct GenBwdCfg {
  static constexpr int VC = 4;                                     // columns per lane
  static constexpr int WAVES = 4, THREADS = WAVES * kWave;
  static constexpr int NG = N / WAVES;                             // stream groups in the grid
  static constexpr int DW = 16 * VC;                               // columns of a wave
  static constexpr int NW = VC * (int)sizeof(S) / 4;               // 4-byte words of a lane's row piece
  static constexpr int XP = std::is_same<S, bf16_t>::value ? 1 : 2;  // bf16 planes of x
  static constexpr int BLOCKS_PER_CU = N == 4 ? 2 : 1;
  static_assert(NW == 2 || NW == 4, "8- or 16-byte row pieces");
};

constexpr int kGenBwdStretch = 64;  // tiles of an MFMA chain of grad_phi

template <int NW> struct GenWords { uint32_t w[NW]; };

template <typename S, int NW>
__device__ __forceinline__ GenWords<NW> gen_load_piece(const S* p) {
  GenWords<NW> o;
  if constexpr (NW == 4) {
    const u32x4 v = ld16u(p);
#pragma unroll
    for (int i = 0; i < 4; ++i) o.w[i] = v[i];
  } else {
    const u32x2 v = *reinterpret_cast<const u32x2_a2*>(p);
    o.w[0] = v[0];
    o.w[1] = v[1];
  }
  return o;
}
// a = elements sh .. sh + 3 of the eight (a, b), sh = 0..3
template <typename S, int NW>
__device__ __forceinline__ void gen_join(GenWords<NW>& a, const GenWords<NW>& b, int sh) {
  if constexpr (NW == 2) {
    const uint64_t va = (uint64_t)a.w[1] << 32 | a.w[0], vb = (uint64_t)b.w[1] << 32 | b.w[0];
    const uint64_t v = sh ? va >> (16 * sh) | vb << (64 - 16 * sh) : va;
    a.w[0] = (uint32_t)v;
    a.w[1] = (uint32_t)(v >> 32);
  } else {
    uint32_t t[6];
#pragma unroll
    for (int i = 0; i < 6; ++i) {
      const uint32_t lo = i < 4 ? a.w[i < 4 ? i : 0] : b.w[i < 4 ? 0 : i - 4];
      const uint32_t hi = i < 2 ? a.w[i < 2 ? i + 2 : 0] : b.w[i < 2 ? 0 : i - 2];
      t[i] = sh & 2 ? hi : lo;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) a.w[i] = sh & 1 ? t[i + 1] : t[i];
  }
}
template <typename S, int NW>
__device__ __forceinline__ float gen_elem(const GenWords<NW>& v, int c) {
  if constexpr (sizeof(S) == 4)
    return __uint_as_float(v.w[c]);
  else
    return Store<S>::to_f32((uint16_t)((v.w[c / 2] >> (16 * (c & 1))) & 0xffffu));
}

// JOIN: D is no multiple of the lane's four columns
template <int N, typename S, int P, bool JOIN>
__global__ __launch_bounds__((GenBwdCfg<N, S>::THREADS), (GenBwdCfg<N, S>::BLOCKS_PER_CU)) void pre_bwd_gen_kernel(
    PreBwdStreamArgs a, int64_t ntiles) {
  using C = GenBwdCfg<N, S>;
  using PD = PreDims<N>;
  constexpr int M = PD::M, MT = PD::MT, MK = PD::MK, MP32 = PD::MP32;
  constexpr int VC = C::VC, NW = C::NW, XP = C::XP, TT = kStreamTile;
  typedef GenWords<NW> Row;

  const int lane = threadIdx.x & (kWave - 1);
  const int D = a.D;
  const int64_t K = (int64_t)N * D, T = a.T;
  const int split = (int)blockIdx.y, nsplit = (int)gridDim.y;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, q = lane >> 4;
  // the lane's first column, its stream and its column there
  const int64_t s0 = (int64_t)(blockIdx.x % C::NG * C::WAVES + wave) * D;
  const int64_t kl = s0 / VC * VC + (int64_t)(blockIdx.x / C::NG) * C::DW + VC * r;
  const bool in = kl < (s0 + D) / VC * VC;
  const int n0 = in ? (int)(kl / D) : 0;
  const int d0 = in ? (int)(kl - (int64_t)n0 * D) : 0;
  // A lane whose columns end its stream after cb < 4 of them takes the others
  // from the next one (`cross`: some lane of the wave does; such a wave must
  // not fall far behind the others, which all walk as many tiles).  Rows of
  // less than four columns go element by element.
  const bool tiny = JOIN && D < VC;
  const int cb = JOIN && in && d0 + VC > D ? D - d0 : VC;
  const bool cross = JOIN && !tiny && __ballot(cb < VC) != 0;
  const int n1 = n0 + 1 < N ? n0 + 1 : N - 1;
  const S* __restrict__ x = static_cast<const S*>(a.x);
  const S* __restrict__ gy = static_cast<const S*>(a.gy);
  S* __restrict__ gx = static_cast<S*>(a.gx);
  const int64_t kc = in ? kl : 0;

  u32x4 pb[VC][MK][P];
#pragma unroll
  for (int c = 0; c < VC; ++c)
#pragma unroll
    for (int mk = 0; mk < MK; ++mk)
#pragma unroll
      for (int p = 0; p < P; ++p)
        pb[c][mk][p] = ld16(a.phiT + p * a.phiT_plane_stride + (kc + c) * MP32 + 32 * mk + 8 * q);

  // grad_phi: the tiles of a stretch in ph, those of the stretches before in
  // LDS (a lane's own sums; N = 4 has no registers for them)
  __shared__ floatx4 run[MT * VC][C::THREADS];
  const bool folds = ntiles > (int64_t)kGenBwdStretch * nsplit;
  floatx4 ph[MT][VC];
  auto clear = [&]() {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int c = 0; c < VC; ++c) ph[mt][c] = floatx4{0.f, 0.f, 0.f, 0.f};
  };
  auto fold = [&]() {
#pragma unroll
    for (int i = 0; i < MT * VC; ++i) {
      run[i][threadIdx.x] += ph[i / VC][i % VC];
      if (i % 4 == 3) __builtin_amdgcn_sched_barrier(0);  // not all of them in registers at once
    }
  };
  clear();
  if (folds) {
#pragma unroll
    for (int i = 0; i < MT * VC; ++i) run[i][threadIdx.x] = floatx4{0.f, 0.f, 0.f, 0.f};
  }

  // Rows past T read row T - 1: its x meets zero columns of g (kernel A
  // zero-fills the padding tokens of the last tile) and its grad_x is not
  // stored, like the grad_mixes rows and coefficients of tokens past T.
  auto load_rows = [&](int64_t tile, Row (&xr)[4], Row (&gr)[4]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int64_t t = tile * TT + 4 * q + e, tc = t < T ? t : T - 1;
      xr[e] = gen_load_piece<S, NW>(x + tc * K + kc);
      // the row's last four columns where the lane's own pass its end (rows of
      // less than four: anything, they are read below)
      gr[e] = gen_load_piece<S, NW>(tiny ? x + tc * K : gy + tc * D + (cb < VC ? D - VC : d0));
    }
  };

  Row xn[4], gn[4];
  if (split < ntiles) load_rows(split, xn, gn);
  auto step = [&](int64_t tile) {
    Row xr[4], gr[4];
    const int64_t tb = tile * TT;
    // ---- operands of the tile (L2), then the next tile's rows --------------
    float4 cf[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int64_t t = tb + 4 * q + e;
      cf[e] = a.coef[(t < T ? t : T - 1) * N + n0];  // pre[t, n0], inv[t], scale[t]
    }
    // JOIN: the next stream's first columns of grad_y and its pre gate
    Row gj[JOIN ? 4 : 1];
    float pre1[JOIN ? 4 : 1];
    if constexpr (JOIN) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int64_t t = tb + 4 * q + e, tc = t < T ? t : T - 1;
        pre1[e] = a.coef[tc * N + n1].x;
        if (!tiny) gj[e] = gen_load_piece<S, NW>(gy + tc * D);
      }
    }
    const int64_t ts = tb + r < T ? tb + r : T - 1;  // token of MFMA row r in the gs product
    u32x4 gA[MK][2], ga[MT];
#pragma unroll
    for (int mk = 0; mk < MK; ++mk)
#pragma unroll
      for (int g = 0; g < 2; ++g) gA[mk][g] = ld16(a.gmP + g * a.gmP_plane + ts * MP32 + 32 * mk + 8 * q);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) ga[mt] = ld16(a.gTw + ((tile * MT + mt) * kWave + lane) * 8);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      xr[e] = xn[e];
      gr[e] = gn[e];
    }
    if (tile + nsplit < ntiles) load_rows(tile + nsplit, xn, gn);

    if constexpr (JOIN) {
      if (cross) {
#pragma unroll
        for (int e = 0; e < 4; ++e) gen_join<S, NW>(gr[e], gj[e], VC - cb);
      }
    }
    // ---- gs = grad_mixes phi, then grad_x -----------------------------------
    floatx4 gs[VC];
#pragma unroll
    for (int c = 0; c < VC; ++c) {
      gs[c] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int mk = 0; mk < MK; ++mk) {
        gs[c] = mfma16x16x32(as_bf16x8(gA[mk][0]), as_bf16x8(pb[c][mk][0]), gs[c]);
        gs[c] = mfma16x16x32(as_bf16x8(gA[mk][1]), as_bf16x8(pb[c][mk][0]), gs[c]);
        if constexpr (P > 1) gs[c] = mfma16x16x32(as_bf16x8(gA[mk][0]), as_bf16x8(pb[c][mk][P - 1]), gs[c]);
      }
    }
    // ---- grad_phi partial += g^T x over the tile's 16 tokens --------------
#pragma unroll
    for (int c = 0; c < VC; ++c) {
      u32x4 bx[XP];  // tokens (2w, 2w + 1) in words w and w + 2
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        if constexpr (XP == 1) {
          const uint32_t lo = xr[2 * w].w[c / 2], hi = xr[2 * w + 1].w[c / 2];
          bx[0][w] = (c & 1) ? ((lo >> 16) | (hi & 0xffff0000u)) : ((lo & 0xffffu) | (hi << 16));
        } else {
          const float v0 = gen_elem<S, NW>(xr[2 * w], c), v1 = gen_elem<S, NW>(xr[2 * w + 1], c);
          const uint32_t h = pack_bf16x2(v0, v1);
          bx[0][w] = h;
          bx[XP - 1][w] = pack_bf16x2(v0 - __uint_as_float(h << 16), v1 - __uint_as_float(h & 0xffff0000u));
        }
      }
#pragma unroll
      for (int p = 0; p < XP; ++p) {
        bx[p][2] = bx[p][0];
        bx[p][3] = bx[p][1];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) ph[mt][c] = mfma16x16x32(as_bf16x8(ga[mt]), as_bf16x8(bx[p]), ph[mt][c]);
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int64_t t = tb + 4 * q + e;
      if (t >= T || !in) continue;
      float o[VC];
#pragma unroll
      for (int c = 0; c < VC; ++c) {
        float pre = JOIN && c >= cb ? pre1[JOIN ? e : 0] : cf[e].x, g = gen_elem<S, NW>(gr[e], c);
        if (JOIN && tiny) {
          pre = a.coef[t * N + (kl + c) / D].x;
          g = load_elem(gy, t * D + (kl + c) % D);
        }
        o[c] = fmaf(cf[e].z, gen_elem<S, NW>(xr[e], c), fmaf(cf[e].y, gs[c][e], g * pre));
      }
      if (a.gin) {
        const Row gi = gen_load_piece<S, NW>(static_cast<const S*>(a.gin) + t * K + kl);
#pragma unroll
        for (int c = 0; c < VC; ++c) o[c] += gen_elem<S, NW>(gi, c);
      }
      S* row = gx + t * K + kl;
      if constexpr (sizeof(S) == 4) {
        __builtin_nontemporal_store(Store<float>::pack(o), reinterpret_cast<u32x4_a2*>(row));
      } else {
        u32x2 v;
#pragma unroll
        for (int i = 0; i < 2; ++i)
          v[i] = (uint32_t)Store<S>::from_f32(o[2 * i]) | ((uint32_t)Store<S>::from_f32(o[2 * i + 1]) << 16);
        __builtin_nontemporal_store(v, reinterpret_cast<u32x2_a2*>(row));
      }
    }
  };
  // One loop at N = 4 (two take 20 registers more, and rows of fp32 then
  // spill); two at N = 8, whose accumulators are AGPRs: folded inside the loop
  // over tiles they, or phi^T, move between register files at every tile.
  if constexpr (N == 4) {
    int done = 0;
    for (int64_t tile = split; tile < ntiles; tile += nsplit) {
      step(tile);
      if (folds && ++done == kGenBwdStretch) {
        done = 0;
        fold();
        clear();
      }
    }
  } else {
    const int64_t span = (int64_t)kGenBwdStretch * nsplit;
    int64_t tile = split;
    while (folds && tile + span < ntiles) {
      for (const int64_t end = tile + span; tile < end; tile += nsplit) step(tile);
      fold();
      clear();
    }
    for (; tile < ntiles; tile += nsplit) step(tile);
  }
  if (folds) {
#pragma unroll
    for (int i = 0; i < MT * VC; ++i) ph[i / VC][i % VC] += run[i][threadIdx.x];
  }

  float* part = a.gphi_part + (int64_t)split * M * K + kl;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int m = 16 * mt + 4 * q + v;
      if (m < M && in)
        *reinterpret_cast<float4*>(part + (int64_t)m * K) = float4{ph[mt][0][v], ph[mt][1][v], ph[mt][2][v], ph[mt][3][v]};
    }
}

}  // namespace mhc
