// The pre forward's general contraction: any x and phi dtype, any D and
// alignment, N = 4 or 8.  Included by pre_fwd.hip.
//
//   part[slot][t][m] = sum_k x[t][k] phi[m][k]   part_ssq[slot][t] = sum_k x[t][k]^2
//
// over the columns k of one block's share of token t's tile; the finish
// kernel (pre_fwd_finish_kernel) adds a token's slots in order and forms the
// heads, Sinkhorn and y.
//
// Work split.  A stage is CW columns of a tile of TT tokens.  The
// tiles * nst stages are cut into equal runs of gen_w consecutive stages, one
// block a run, so every CU gets the same number of stages whatever T is (65
// tiles on 512 resident blocks leave no second wave of blocks); a tile's
// stages fall to at most nst / gen_w + 2 blocks, each with a slot of its own.
//
// A block's waves share phi: its threads read a stage's phi in its own dtype
// (rows are read once per 128 tokens), split it into bf16 planes (1 for bf16,
// 2 for fp16, 3 for fp32: residual below 2^-26) and write the planes to one of
// two LDS buffers, so no separate kernel and no memory holds them.  x goes
// from memory to the registers of the one wave that needs it: lane (r, q)
// takes columns 8 q .. 8 q + 7 of each 32-column step of token row r, which is
// the MFMA A operand as it stands for bf16 (fp16 and fp32 are split in
// registers).  Both are loaded one stage ahead; one barrier a stage.
// Unaligned rows take the same 16-byte loads (global memory accesses need no
// alignment on this part); only the last, partial columns are read one by one.
//
// Eight waves of 16 tokens, 128-token tiles; SMALL (few tokens, or a product
// too small to fill the chip): one 16-token tile, the waves splitting each
// stage's 32-column steps, so that a decode step's time is the latency of a
// few loads; the waves' sums meet in LDS at the end of a tile's run.
//
// A stage's products go through a fresh MFMA chain that is added to the
// running sums by round-to-nearest adds (a chain over all of K drifts), and a
// stage's squares through a chain of their own: one over a block's whole run
// loses the small squares, which all round the same way (inv_rms at T = 65536,
// D = 7168, bf16: 3.1e-6 off so, 7e-8 now, at the same time).
//
// Measured (MI355X, the whole operator; before: one block a 64-token tile
// that walked all of K with one wave a SIMD, then y): phi fp32, bf16 x, N =
// 4: D = 7168, T = 1: 177 -> 9.8 us (now in a replayed graph); D = 4096, T =
// 777: 253 -> 23; D = 3584, T = 8193: 250 -> 98 (this kernel 55: 4.2 TB/s of
// x); fp16 x and phi, D = 1003, T = 2049: 312 -> 25; fp32, D = 256, T = 1024:
// 42 -> 11.  At many tokens issue bounds it as much as memory (splitting phi, the
// sum of squares, 24 MFMA and 24 LDS reads per wave and stage); two row
// blocks a wave (half the LDS reads, four waves a block) measured 10% slower,
// streaming loads 8%, 128-byte row pieces per load instruction 2%.
#pragma once

namespace mhc {

template <typename S> struct GenPlanes;
template <> struct GenPlanes<bf16_t> { static constexpr int P = 1; };
template <> struct GenPlanes<f16_t> { static constexpr int P = 2; };
template <> struct GenPlanes<float> { static constexpr int P = 3; };

template <int N, bool SMALL> struct GenCfg {
  static constexpr int M = PreDims<N>::M, MT = PreDims<N>::MT;
  static constexpr int CW = N == 8 ? 64 : (SMALL ? 256 : 128);    // columns of a stage
  static constexpr int KS = CW / 32;                              // 32-column steps of a stage
  static constexpr int WT = SMALL ? 1 : 8;                        // waves over the tokens
  static constexpr int WK = SMALL ? KS : 1;                       // waves over the steps
  static constexpr int STEPS = KS / WK;                           // steps a wave takes
  static constexpr int WAVES = WT * WK, THREADS = WAVES * kWave, TT = 16 * WT;
  static constexpr int CPR = CW / 8;                              // 8-column groups of a row
  static constexpr int NG = (M * CPR + THREADS - 1) / THREADS;    // phi groups a thread stages
  // 16-byte chunk c of LDS row `row` sits at position c ^ swz(row): the 16
  // rows of an MFMA operand read then hit 16 different bank groups
  __device__ static constexpr int swz(int row) { return CW == 64 ? ((row >> 1) & 7) : (row & 15); }
};

template <typename S>
__device__ __forceinline__ void gen_unpack(const Raw8<S>& r, float (&f)[8]) {
  if constexpr (sizeof(S) == 2) {
    Store<S>::unpack(r.v[0], f);
  } else {
    Store<float>::unpack(r.v[0], f);
    Store<float>::unpack(r.v[1], f + 4);
  }
}
// bf16 planes of eight elements (f: their fp32 values)
template <typename S>
__device__ __forceinline__ void gen_planes(const Raw8<S>& r, const float (&f)[8], u32x4 (&pl)[GenPlanes<S>::P]) {
  if constexpr (GenPlanes<S>::P == 1)
    pl[0] = r.v[0];
  else if constexpr (GenPlanes<S>::P == 2)
    split8(f, pl[0], pl[1]);
  else
    split8x3(f, pl[0], pl[1], pl[2]);
}

// A lane's eight elements of a 512-column chunk: columns 8 l .. 8 l + 7, or
// (SPLIT: 4-byte elements are moved) 4 l .. 4 l + 3 and 256 + 4 l .., so that
// every 16-byte access of a wave continues its neighbour's (4-byte elements
// stored as 16-byte pieces at a 32-byte lane stride move at a third of the
// rate).
template <typename S, bool SPLIT>
__device__ __forceinline__ Raw8<S> gen_load_chunk(const S* row, int c0, int lane, int lim) {
  if constexpr (!SPLIT) {
    const int k = c0 + 8 * lane;
    return k + 8 <= lim ? gen_load8(row + k) : gen_load8_tail(row, k, lim);
  } else {
    Raw8<S> r;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int k = c0 + 256 * h + 4 * lane;
      if constexpr (sizeof(S) == 4) {
        r.v[h] = zero4();
        if (k + 4 <= lim) {
          r.v[h] = ld16u(row + k);
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (k + i < lim) r.v[h][i] = reinterpret_cast<const uint32_t*>(row)[k + i];
        }
      } else {
        u32x2 p = {0u, 0u};
        if (k + 4 <= lim) {
          p = *reinterpret_cast<const u32x2_a2*>(row + k);
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (k + i < lim) p[i / 2] |= (uint32_t)reinterpret_cast<const uint16_t*>(row)[k + i] << (16 * (i & 1));
        }
        r.v[0][2 * h] = p[0];
        r.v[0][2 * h + 1] = p[1];
      }
    }
    return r;
  }
}
template <typename S>
__device__ __forceinline__ void gen_store4(S* row, int k, int lim, const float* f) {
  if (k + 4 <= lim) {
    if constexpr (sizeof(S) == 4) {
      __builtin_nontemporal_store(Store<float>::pack(f), reinterpret_cast<u32x4_a2*>(row + k));
    } else {
      u32x2 v;
#pragma unroll
      for (int i = 0; i < 2; ++i)
        v[i] = (uint32_t)Store<S>::from_f32(f[2 * i]) | ((uint32_t)Store<S>::from_f32(f[2 * i + 1]) << 16);
      __builtin_nontemporal_store(v, reinterpret_cast<u32x2_a2*>(row + k));
    }
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (k + i < lim) store_elem(row, k + i, f[i]);
  }
}
template <typename S, bool SPLIT>
__device__ __forceinline__ void gen_store_chunk(S* row, int c0, int lane, int lim, const float (&f)[8]) {
  if constexpr (SPLIT) {
    gen_store4(row, c0 + 4 * lane, lim, f);
    gen_store4(row, c0 + 256 + 4 * lane, lim, f + 4);
  } else {
    static_assert(sizeof(S) == 2, "4-byte elements move in split pieces");
    const int k = c0 + 8 * lane;
    if (k + 8 <= lim) {
      __builtin_nontemporal_store(Store<S>::pack(f), reinterpret_cast<u32x4_a2*>(row + k));
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (k + i < lim) store_elem(row, k + i, f[i]);
    }
  }
}

// Two 8-wave blocks a CU (four waves a SIMD, 128 registers) where that spills
// at most a few of them; N = 8 with fp16 x and bf16 phi spills 148.
template <int N, typename S, typename PT, bool SMALL>
constexpr int gen_min_waves() {
  return SMALL ? 1 : N == 8 && GenPlanes<S>::P == 2 && GenPlanes<PT>::P == 1 ? 2 : 4;
}

template <int N, typename S, typename PT, bool SMALL>
__global__ __launch_bounds__((GenCfg<N, SMALL>::THREADS), (gen_min_waves<N, S, PT, SMALL>())) void pre_fwd_gen_kernel(PreFwdArgs a) {
  using C = GenCfg<N, SMALL>;
  constexpr int M = C::M, MT = C::MT, CW = C::CW, STEPS = C::STEPS, NG = C::NG, P = GenPlanes<PT>::P,
                XP = GenPlanes<S>::P;
  __shared__ u32x4 ph[2][P * M * C::CPR];
  __shared__ floatx4 red[C::WK > 1 ? C::WK - 1 : 1][MT][C::WK > 1 ? kWave : 1];
  __shared__ float red_ssq[C::WK > 1 ? C::WK - 1 : 1][16];

  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wt = wave / C::WK, wk = wave % C::WK;
  const int r = lane & 15, q = lane >> 4;
  const int64_t T = a.T, K = (int64_t)N * a.D;
  const int nst = a.gen_nst;
  const int64_t ntiles = (T + C::TT - 1) / C::TT;
  const int64_t u0 = (int64_t)blockIdx.x * a.gen_w;
  const int64_t total = ntiles * nst;
  const int64_t u1 = u0 + a.gen_w < total ? u0 + a.gen_w : total;
  if (u0 >= u1) return;  // uniform over the block

  const S* __restrict__ x = static_cast<const S*>(a.x);
  const PT* __restrict__ phi = static_cast<const PT*>(a.phi_raw);

  // rows past T read row T - 1 (their sums are not stored)
  auto row_of = [&](int64_t tile) {
    const int64_t t = tile * C::TT + 16 * wt + r;
    return x + (t < T ? t : T - 1) * K;
  };
  auto load_x = [&](Raw8<S>(&X)[STEPS], const S* row, int s) {
    const int64_t k = (int64_t)s * CW + 32 * (wk * STEPS) + 8 * q;
    if ((int64_t)(s + 1) * CW <= K) {
#pragma unroll
      for (int i = 0; i < STEPS; ++i) X[i] = gen_load8(row + k + 32 * i);
    } else {
#pragma unroll
      for (int i = 0; i < STEPS; ++i)
        X[i] = k + 32 * i + 8 <= K ? gen_load8(row + k + 32 * i) : gen_load8_tail(row, k + 32 * i, K);
    }
  };
  // phi group j of this thread: row gr, columns 8 gc .. of a stage
  auto load_phi = [&](Raw8<PT>(&F)[NG], int s) {
#pragma unroll
    for (int j = 0; j < NG; ++j) {
      const int gi = tid + j * C::THREADS;
      if (NG * C::THREADS == M * C::CPR || gi < M * C::CPR) {
        const PT* prow = phi + (int64_t)(gi / C::CPR) * K;
        const int64_t k = (int64_t)s * CW + 8 * (gi % C::CPR);
        F[j] = k + 8 <= K ? gen_load8(prow + k) : gen_load8_tail(prow, k, K);
      }
    }
  };
  auto write_phi = [&](const Raw8<PT>(&F)[NG], int buf) {
#pragma unroll
    for (int j = 0; j < NG; ++j) {
      const int gi = tid + j * C::THREADS;
      if (NG * C::THREADS == M * C::CPR || gi < M * C::CPR) {
        const int gr = gi / C::CPR, gc = gi % C::CPR;
        float f[8];
        u32x4 pl[P];
        gen_unpack(F[j], f);
        gen_planes(F[j], f, pl);
#pragma unroll
        for (int p = 0; p < P; ++p) ph[buf][(p * M + gr) * C::CPR + (gc ^ C::swz(gr))] = pl[p];
      }
    }
  };
  // the block's LDS writes are done; loads in flight stay in flight
  auto sync = [&]() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  floatx4 acc[MT];
  float ssq;
  auto clear = [&]() {
    ssq = 0.f;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[mt] = floatx4{0.f, 0.f, 0.f, 0.f};
  };
  clear();

  // phi rows 16 mt + r; N = 4: rows 24..31 do not exist, their lanes read
  // rows 16..23 again (accumulator columns that are never stored)
  int prow[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) prow[mt] = 16 * mt + r < M ? 16 * mt + r : 16 * mt + (r & 7);

  auto compute = [&](const Raw8<S>(&X)[STEPS], int buf) {
    floatx4 part[MT];
    float sq = 0.f;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) part[mt] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < STEPS; ++i) {
      const int c = 4 * (wk * STEPS + i) + q;
      float f[8];
      u32x4 xp[XP];
      gen_unpack(X[i], f);
      gen_planes(X[i], f, xp);
#pragma unroll
      for (int e = 0; e < 8; ++e) sq = fmaf(f[e], f[e], sq);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int p = 0; p < P; ++p) {
          const u32x4 b = ph[buf][(p * M + prow[mt]) * C::CPR + (c ^ C::swz(prow[mt]))];
#pragma unroll
          for (int xi = 0; xi < XP; ++xi)
            if (xi + p <= 2)  // the dropped products are below 2^-26 relative
              part[mt] = mfma16x16x32(as_bf16x8(xp[xi]), as_bf16x8(b), part[mt]);
        }
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[mt] += part[mt];
    ssq += sq;
  };

  // the block's sums of a tile: lane (r, q) of acc[mt] holds token 16 wt +
  // 4 q + v, m = 16 mt + r; after the adds the lanes of row r hold the sum of
  // squares of token 16 wt + r
  auto flush = [&](int64_t tile) {
    ssq = add_xor32(add_xor16(ssq));
    if constexpr (C::WK > 1) {
      if (wk > 0) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) red[wk - 1][mt][lane] = acc[mt];
        if (q == 0) red_ssq[wk - 1][r] = ssq;
      }
      sync();
      if (wk == 0) {
#pragma unroll
        for (int w = 0; w < C::WK - 1; ++w) {
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) acc[mt] += red[w][mt][lane];
          ssq += red_ssq[w][r];
        }
      }
    }
    if (C::WK == 1 || wk == 0) {
      const int64_t slot = (int64_t)blockIdx.x - tile * nst / a.gen_w;
      const int64_t tb = tile * C::TT + 16 * wt;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int64_t tok = tb + 4 * q + v;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          if (tok < T && 16 * mt + r < M) a.part[(slot * T + tok) * M + 16 * mt + r] = acc[mt][v];
      }
      if (q == 0 && tb + r < T) a.part_ssq[slot * T + tb + r] = ssq;
    }
    clear();
  };

  int64_t tile = u0 / nst;
  int s = (int)(u0 - tile * nst);
  Raw8<S> X0[STEPS], X1[STEPS];
  Raw8<PT> F[NG];
  auto next = [&](int v) { return v + 1 == nst ? 0 : v + 1; };
  const S* row = row_of(tile);
  load_phi(F, s);
  load_x(X0, row, s);
  write_phi(F, 0);
  if (u0 + 1 < u1) load_phi(F, next(s));
  sync();
  // stage u: its x in Xc, its phi in buffer `buf`; F holds phi of stage u + 1
  auto stage = [&](int64_t u, Raw8<S>(&Xc)[STEPS], Raw8<S>(&Xn)[STEPS], int buf) {
    const bool more = u + 1 < u1, last = s == nst - 1;
    const int sn = next(s);
    if (more) {
      if (last) row = row_of(tile + 1);
      load_x(Xn, row, sn);
    }
    compute(Xc, buf);
    if (more) write_phi(F, buf ^ 1);  // every wave left that buffer before the last barrier
    if (u + 2 < u1) load_phi(F, next(sn));
    if (last || !more) flush(tile);
    if (last) ++tile;
    s = sn;
    sync();
  };
  for (int64_t u = u0; u < u1; u += 2) {
    stage(u, X0, X1, 0);
    if (u + 1 < u1) stage(u + 1, X1, X0, 1);
  }
}

// ---------------------------------------------------------------------------
// finish: sums, heads, Sinkhorn and y of one token in one block
// ---------------------------------------------------------------------------
// y (and x_scaled) of a lane's eight columns of the chunk at c0, given the N
// rows' elements there
template <typename S, bool XS> constexpr bool kGenSplit = XS || sizeof(S) == 4;

template <int N, typename S, bool XS>
__device__ __forceinline__ void gen_load_rows(const PreFwdArgs& a, int64_t t, int c0, int lane, Raw8<S> (&X)[N]) {
  const S* x = static_cast<const S*>(a.x) + t * N * a.D;
#pragma unroll
  for (int n = 0; n < N; ++n) X[n] = gen_load_chunk<S, kGenSplit<S, XS>>(x + (int64_t)n * a.D, c0, lane, a.D);
}
template <int N, typename S, bool XS>
__device__ __forceinline__ void gen_y8(const PreFwdArgs& a, int64_t t, int c0, int lane, const Raw8<S> (&X)[N],
                                       const float (&p)[N], float inv) {
  const int D = a.D;
  float o[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] = 0.f;
#pragma unroll
  for (int n = 0; n < N; ++n) {
    float f[8];
    gen_unpack(X[n], f);
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = fmaf(p[n], f[e], o[e]);
    if constexpr (XS) {
#pragma unroll
      for (int e = 0; e < 8; ++e) f[e] *= inv;
      gen_store_chunk<float, true>(a.x_scaled + (t * N + n) * (int64_t)D, c0, lane, D, f);
    }
  }
  // y is an fp32 sum, then rounded: without this the compiler forms fp16 sums
  // with v_fma_mixlo in one of the two layouts only, and y would depend on
  // whether x_scaled is asked for
  if constexpr (sizeof(S) == 2) {
#pragma unroll
    for (int e = 0; e < 8; ++e) asm volatile("" : "+v"(o[e]));
  }
  gen_store_chunk<S, kGenSplit<S, XS>>(static_cast<S*>(a.y) + t * D, c0, lane, D, o);
}

// One block per token, after the general contraction or the LDS-pipelined
// kernels' sums (see finish_applies).  All waves add the slots, wave 0 then
// runs the heads and Sinkhorn while the others form y from rows they began to
// load before the sums were complete; y needs only the pre gates, which every
// wave forms for itself, a gate a lane.
constexpr int kFinishWaves = 16;
template <int N, typename S, bool XS>
__global__ __launch_bounds__(kWave * kFinishWaves) void pre_fwd_finish_kernel(PreFwdArgs a, int nsplit) {
  constexpr int M = PreDims<N>::M, L = N * N, VP = N == 4 ? 32 : 128;  // VP > M: the sums and the sum of squares
  static_assert(M < VP && VP <= 2 * kWave, "a lane for each sum; blocks of at least two waves");
  __shared__ float red[kWave * kFinishWaves / VP][VP];
  __shared__ float tot[VP];
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int groups = blockDim.x / VP, yw = blockDim.x / kWave - 1;
  const int64_t t = blockIdx.x;
  const int ns = fwd_slots(a, t, nsplit);
  {
    const int v = tid % VP, g = tid / VP;
    float sum = 0.f;
    if (v <= M) {
      const float* p = v < M ? a.part + t * M + v : a.part_ssq + t;
      const int64_t rows = fwd_slot_rows(a), stride = v < M ? rows * M : rows;
#pragma unroll 4
      for (int s = g; s < ns; s += groups) sum += p[s * stride];
    }
    if (g < groups) red[g][v] = sum;
  }
  const int first = (wave - 1) * 512;
  Raw8<S> X[N];
  if (wave > 0) gen_load_rows<N, S, XS>(a, t, first, lane, X);
  __syncthreads();
  if (tid < VP) {
    float sum = 0.f;
    for (int g = 0; g < groups; ++g) sum += red[g][tid];
    tot[tid] = sum;
  }
  __syncthreads();
  const float inv = rms_inv(tot[M], (float)(N * (int64_t)a.D), a.norm_eps), a0 = a.alpha[0];
  if (wave > 0) {
    const float p_l = pre_gate(tot[lane % N] * inv, a0, a.base[lane % N], a.hc_eps);
    float p[N];
#pragma unroll
    for (int n = 0; n < N; ++n) p[n] = __shfl(p_l, n, kWave);
    for (int c0 = first; c0 < a.D; c0 += yw * 512) {
      if (c0 != first) gen_load_rows<N, S, XS>(a, t, c0, lane, X);
      gen_y8<N, S, XS>(a, t, c0, lane, X, p, inv);
    }
    return;
  }
  const int e = lane % L;
  const bool ok = lane < L;
  const float mix_l = tot[2 * N + e] * inv;
  const float logit = mix_l * a.alpha[2] + a.base[2 * N + e];
  if (ok) {
    if (a.mixes) a.mixes[t * M + 2 * N + e] = mix_l;
    if (a.logits) a.logits[t * L + e] = logit;
    if (e == 0 && a.inv_rms) a.inv_rms[t] = inv;
    if (e < 2 * N) {
      const float mix_h = tot[e] * inv;
      if (a.mixes) a.mixes[t * M + e] = mix_h;
      if (e < N) {
        if (a.pre) a.pre[t * N + e] = pre_gate(mix_h, a0, a.base[e], a.hc_eps);
      } else {
        a.post_out[t * N + (e - N)] = 2.0f * sigmoidf_(mix_h * a.alpha[1] + a.base[e]);
      }
    }
  }
  const float c = sinkhorn_fwd<N>(clamp_logit(logit, a.apply_clamp, a.cmin, a.cmax), a.hc_eps, a.iters);
  if (ok) a.comb[t * L + e] = c;
}

// y (and x_scaled) after the finalize kernel: a block per token of W waves,
// wave w taking the 512-column chunks w, w + W, ..
template <int N, typename S, bool XS>
__global__ __launch_bounds__(kWave * kFinishWaves) void pre_fwd_gen_y_kernel(PreFwdArgs a) {
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), W = blockDim.x / kWave;
  const int64_t t = blockIdx.x;
  float p[N];
#pragma unroll
  for (int n = 0; n < N; ++n) p[n] = a.pre_ws[t * N + n];
  const float inv = XS ? a.inv_ws[t] : 0.f;
  for (int c0 = wave * 512; c0 < a.D; c0 += W * 512) {
    Raw8<S> X[N];
    gen_load_rows<N, S, XS>(a, t, c0, lane, X);
    gen_y8<N, S, XS>(a, t, c0, lane, X, p, inv);
  }
}

// ---- host side --------------------------------------------------------------
// Whether the finish kernel ends a call, rather than the finalize kernel
// (tokens packed N * N lanes each) and a y kernel.  Its Sinkhorn chain, about
// 5 us a token, hides behind other blocks only while there are few of them or
// each has much y to form; a launch less is what counts at few tokens.
// Measured (bf16, us, finish / finalize + y, whole operator): N = 4: T = 64 D =
// 7168 11.6 / 16.2; T = 512 D = 4096 15.0 / 18.0; T = 2048 D = 4096 37.0 / 37.6,
// D = 256 13.5 / 12.9; T = 16384 D = 256 39 / 26, D = 512 41 / 38, D = 9216 451
// / 438; fp16 T = 8192 D = 1003 59.6 / 50.5.  N = 8: T = 64 D = 2048 13.6 /
// 16.1; T = 16384 D = 2048 253 / 262, D = 256 72 / 57.  Narrow rows at few
// tokens (replayed graphs): N = 4: D = 256, T = 1 8.9 / 10.1, T = 1024 10.0 /
// 11.3, T = 1536 11.9 / 11.8; D = 512, T = 1024 9.8 / 12.7; fp32 phi, D = 256,
// T = 1024 10.0 / 12.4; N = 8: D = 256, T = 1 11.4 / 11.8, T = 1024 13.6 / 15.3,
// T = 1536 15.8 / 15.6; fp32 phi, D = 256, T = 1024 19.0 / 20.7.  Four tokens a block
// (N = 4, one Sinkhorn wave for the four) gained 0 to 6% above 2048 tokens and
// lost as much at wide rows.
static bool finish_applies(int64_t T, int N, int D) { return T <= 1024 || (D >= 512 && (N == 8 || T <= 2048)); }

template <int N, typename S, typename PT>
static int launch_gen_contraction(const PreFwdArgs& a, const GenPlan& p, hipStream_t st) {
  const dim3 grid((unsigned)p.blocks(a.T));
  if (p.small)
    hipLaunchKernelGGL((pre_fwd_gen_kernel<N, S, PT, true>), grid, dim3(GenCfg<N, true>::THREADS), 0, st, a);
  else
    hipLaunchKernelGGL((pre_fwd_gen_kernel<N, S, PT, false>), grid, dim3(GenCfg<N, false>::THREADS), 0, st, a);
  return check_launch("pre_fwd_gen");
}

// One kernel for heads, Sinkhorn and y of `a.T` tokens from the sums of
// `nsplit` slots (or, with gen_w, the general contraction's).
template <int N, typename S>
static int launch_pre_fwd_finish(const PreFwdArgs& a, int nsplit, hipStream_t st) {
  const int chunks = (a.D + 511) / 512;
  int yw = chunks < kFinishWaves - 1 ? chunks : kFinishWaves - 1;
  // N = 8: a group of two waves adds a token's slots (up to 129 of the general
  // form's), one after the other, and at few tokens the call waits for them:
  // two groups at least (fp32 phi, D = 1024: T = 1 18.0 -> 14.3 us, T = 256
  // 26.2 -> 21.3, where finalize + y take 16.6 and 24.6; D = 512, T = 1024 23.4
  // -> 22.8, but T = 2048 23.9 -> 27.2)
  if (N == 8 && a.gen_w && a.T <= 1024 && yw < 3) yw = 3;
  const dim3 grid((unsigned)a.T), block(kWave * (1 + yw));
  if (int rc = check_grid(grid, block, "mhc_pre_fwd")) return rc;
  if (a.x_scaled)
    hipLaunchKernelGGL((pre_fwd_finish_kernel<N, S, true>), grid, block, 0, st, a, nsplit);
  else
    hipLaunchKernelGGL((pre_fwd_finish_kernel<N, S, false>), grid, block, 0, st, a, nsplit);
  return check_launch("pre_fwd_finish");
}

template <int N, typename S>
static int launch_pre_fwd_gen_chunk(PreFwdArgs a, const GenPlan& p, int32_t phi_dtype, char* w, hipStream_t st) {
  a.gen_nst = p.nst;
  a.gen_w = p.w;
  a.gen_tt = p.tt;
  a.part = reinterpret_cast<float*>(w);
  a.part_ssq = reinterpret_cast<float*>(w + p.ssq_off);
  a.pre_ws = reinterpret_cast<float*>(w + p.pre_off);
  a.inv_ws = reinterpret_cast<float*>(w + p.inv_off);
  int rc = phi_dtype == MHC_DTYPE_BF16  ? launch_gen_contraction<N, S, bf16_t>(a, p, st)
           : phi_dtype == MHC_DTYPE_F16 ? launch_gen_contraction<N, S, f16_t>(a, p, st)
                                        : launch_gen_contraction<N, S, float>(a, p, st);
  if (rc) return rc;
  if (finish_applies(a.T, N, a.D)) return launch_pre_fwd_finish<N, S>(a, 0, st);
  constexpr int TPP = kFwdThreads / (N * N);
  hipLaunchKernelGGL((pre_fwd_finalize_kernel<N>), dim3((unsigned)((a.T + TPP - 1) / TPP)), dim3(kFwdThreads), 0, st,
                     a, 0);
  if ((rc = check_launch("pre_fwd_finalize"))) return rc;
  const int chunks = (a.D + 511) / 512;
  const dim3 grid((unsigned)a.T), block(kWave * (chunks < kFinishWaves ? chunks : kFinishWaves));
  if ((rc = check_grid(grid, block, "mhc_pre_fwd"))) return rc;
  if (a.x_scaled)
    hipLaunchKernelGGL((pre_fwd_gen_y_kernel<N, S, true>), grid, block, 0, st, a);
  else
    hipLaunchKernelGGL((pre_fwd_gen_y_kernel<N, S, false>), grid, block, 0, st, a);
  return check_launch("pre_fwd_gen_y");
}

// The general form on `chunk` tokens at a time, all by the plan of a whole
// chunk (the stream orders the chunks' use of the workspace).
template <int N, typename S>
static int launch_pre_fwd_gen(const PreFwdArgs& a, int32_t phi_dtype, int64_t chunk, void* workspace,
                              hipStream_t st) {
  constexpr int M = 2 * N + N * N;
  const GenPlan p = gen_plan(chunk, N, a.D, device_cu_count());
  for (int64_t t0 = 0; t0 < a.T; t0 += chunk) {
    PreFwdArgs c = a;
    c.T = a.T - t0 < chunk ? a.T - t0 : chunk;
    c.x = static_cast<const S*>(a.x) + t0 * N * a.D;
    c.y = static_cast<S*>(a.y) + t0 * a.D;
    c.post_out = a.post_out + t0 * N;
    c.comb = a.comb + t0 * N * N;
    if (a.inv_rms) c.inv_rms = a.inv_rms + t0;
    if (a.mixes) c.mixes = a.mixes + t0 * M;
    if (a.logits) c.logits = a.logits + t0 * N * N;
    if (a.pre) c.pre = a.pre + t0 * N;
    if (a.x_scaled) c.x_scaled = a.x_scaled + t0 * N * a.D;
    const int rc =
        launch_pre_fwd_gen_chunk<N, S>(c, p, phi_dtype, static_cast<char*>(workspace) + kPreFwdWsBase, st);
    if (rc) return rc;
  }
  return MHC_OK;
}

}  // namespace mhc
