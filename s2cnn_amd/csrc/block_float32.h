// Blocks of the block products (so3_mm_real.hip, so3_mm.hip) with the float32 matrix instruction, operands straight from memory: for
// the waves whose sums of bf16 parts are not finite (split_bf16.h).  Infinities and values of any size take part as they are
// here, so overflow, infinities and NaN come out as in any float32 product.
#pragma once
#include "common.h"
#include "split_bf16.h"

namespace s2cnn {
namespace block {

// acc = the NI x NJ blocks of 32 x 32 outputs, STEP apart, of which this lane holds row row0 and column col0 of the first; A, B: the
// operands of the degree, L x L blocks of RI (CI) x KI elements; fa, fb: the float of an element that takes part.
template <typename C_, int NI, int NJ, int STEP, typename E, class FA, class FB>
__device__ __forceinline__ void contract_float32(const E* A, const E* B, int RI, int CI, int KI, v16f (&acc)[NI][NJ], int L, int row0, int col0, int h,
                                                 FA fa, FB fb) {
  const int K = L * KI;
  size_t ao[NI], bo[NJ];
  bool aok[NI], bok[NJ];
  const size_t ablk = (size_t)RI * KI, bblk = (size_t)CI * KI;
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int row = row0 + STEP * i, rb = row / RI, ri = row - rb * RI;
    aok[i] = row < L * RI;
    ao[i] = (C_::A_MNMAJ ? (size_t)rb * L : (size_t)rb) * ablk + (size_t)ri * (C_::A_KC ? KI : 1);
  }
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int col = col0 + STEP * j, cb = col / CI, ci = col - cb * CI;
    bok[j] = col < L * CI;
    bo[j] = (C_::B_MNMAJ ? (size_t)cb * L : (size_t)cb) * bblk + (size_t)ci * (C_::B_KC ? KI : 1);
  }
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
  int kb = h / KI, kin = h - kb * KI;
  for (int k0 = 0; k0 < K; k0 += 2) {
    const bool ok = k0 + h < K;
    const size_t ka = (C_::A_MNMAJ ? (size_t)kb : (size_t)kb * L) * ablk + (size_t)kin * (C_::A_KC ? 1 : RI);
    const size_t kbo = (C_::B_MNMAJ ? (size_t)kb : (size_t)kb * L) * bblk + (size_t)kin * (C_::B_KC ? 1 : CI);
    float a[NI], b[NJ];
#pragma unroll
    for (int i = 0; i < NI; ++i) a[i] = ok && aok[i] ? fa(A[ao[i] + ka]) : 0.f;
#pragma unroll
    for (int j = 0; j < NJ; ++j) b[j] = ok && bok[j] ? fb(B[bo[j] + kbo]) : 0.f;
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[j], acc[i][j], 0, 0, 0);
    kin += 2;
    while (kin >= KI) { kin -= KI; ++kb; }
  }
}

}  // namespace block
}  // namespace s2cnn
