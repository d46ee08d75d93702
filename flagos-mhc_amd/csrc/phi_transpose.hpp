// phi^T as bf16 planes [P][K][MP] (zero for m >= M), the operand layout of the
// pre backward's grad_mixes @ phi.
#pragma once

#include "common.hpp"

namespace mhc {

struct PhiTArgs {
  const void* phi;  // (M, K)
  int dtype;        // MHC_DTYPE_*
  int M, MP, P;     // MP: M rounded up to 32; P: planes, 1 or 2
  int64_t K;
  uint16_t* out;
};

constexpr int kPhiTThreads = 256;

// blocks of kPhiTThreads that cover phi^T: a thread per column k and eight m
inline int64_t phiT_blocks(const PhiTArgs& a) { return (a.K * (a.MP / 8) + kPhiTThreads - 1) / kPhiTThreads; }

// Block b of phiT_blocks.  Neighbouring threads take neighbouring k, so each
// of the eight loads is coalesced (a thread per element of phi^T, m fastest,
// read a cache line for every element: 5.9 us at D = 7168 fp32).
__device__ __forceinline__ void phiT_block(const PhiTArgs& a, int64_t b) {
  const int64_t idx = b * kPhiTThreads + threadIdx.x;
  const int64_t mg = idx / a.K, k = idx - mg * a.K;
  if (mg >= a.MP / 8) return;
  float v[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int64_t m = 8 * mg + i, at = (m < a.M ? m : 0) * a.K + k;
    const float f = a.dtype == 0   ? static_cast<const float*>(a.phi)[at]
                    : a.dtype == 1 ? load_elem(static_cast<const bf16_t*>(a.phi), at)
                                   : load_elem(static_cast<const f16_t*>(a.phi), at);
    v[i] = m < a.M ? f : 0.f;
  }
  u32x4 hi, lo;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    hi[i] = pack_bf16x2(v[2 * i], v[2 * i + 1]);
    lo[i] = pack_bf16x2(v[2 * i] - __uint_as_float(hi[i] << 16), v[2 * i + 1] - __uint_as_float(hi[i] & 0xffff0000u));
  }
  uint16_t* dst = a.out + k * a.MP + 8 * mg;
  st16(dst, hi);
  if (a.P > 1) st16(dst + a.K * a.MP, lo);
}

}  // namespace mhc
