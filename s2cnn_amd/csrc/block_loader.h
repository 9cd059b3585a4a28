// Loads of the block products (so3_mm_real.hip, so3_mm.hip): one operand of a degree, an L x L grid of dense feature blocks in
// which either the contraction index or the free index is the fast one, fetched in octets of contraction steps.
#pragma once
#include "common.h"

namespace s2cnn {
namespace block {

constexpr unsigned OUTSIDE = 0x80000000u;   // a byte offset behind the end of every buffer: such loads return 0

// How the contraction index (the flattened pair block, feature; KI features per block) is walked; ADV = steps per stage:
//   DIVIDES  KI a multiple of 8 and KI, ADV divide one another: an octet of steps never straddles a block and every stage
//            starts at the same place inside a block, so a thread's offsets are fixed and a stage advances by a
//            wave-uniform step
//   WALK     any KI: every thread follows its own position (block, feature), in granules of GR steps (GR = 4, 2 or 1 divides
//            KI, so a granule lies in one block)
//   FAR      the same with 64-bit addresses, for operands whose degrees exceed 32-bit byte offsets.  ms of forward and of both gradients
//            with loads of one element -> of four or two: real, 4 degrees, batch 64, 4096 -> 4096: 13.4, 25.1 -> 8.0, 14.1; complex, 3
//            degrees: 7.3, 14.0 -> 6.5, 12.3
enum Walk { DIVIDES = 0, WALK = 1, FAR = 2 };

// N consecutive elements (float, or float2 for complex numbers) as one access
template <typename E, int N> struct VecT { typedef E type; };
template <> struct VecT<float, 2> { typedef float2 type; };
template <> struct VecT<float, 4> { typedef float4 type; };
template <> struct VecT<float2, 2> { typedef float4 type; };

// One operand's loader.  A thread owns NMN rows (ROWSTEP apart) of 8 contraction steps, starting at step k0 and ADV further on with
// every load(): an octet of a row is what a lane feeds to the matrix instruction, and what one 16-byte LDS store takes,
// whichever index is the fast one in memory.  VEC = elements per global access, along the contraction (K-contiguous) or along
// the rows (MN-contiguous).  Rows outside the matrix and steps behind the last block are loaded from OUTSIDE, that is as
// zeros.
template <typename E, bool KC, bool MNMAJ, int NMN, int ROWSTEP, int VEC, int HOW, int GR, int ADV>
struct Loader {
  static constexpr unsigned ES = sizeof(E);
  static_assert(NMN >= 1 && (KC || VEC == 1 || (VEC <= NMN && ROWSTEP == 1)), "no such loader");
  typedef typename VecT<E, VEC>::type vec_t;

  E reg[NMN][8];
  const E* base;
  __amdgpu_buffer_rsrc_t rsrc;
  unsigned off[NMN];            // offset of the row (DIVIDES: and of the octet): bytes, FAR: elements; OUTSIDE for no row
  int MNI, KI, L, blk_k_stride;
  int kb, kin, adv_b, adv_k;    // WALK, FAR: block and feature of this thread's first step; what a stage adds to them
  unsigned soff, step_in, step_cross;   // DIVIDES: uniform byte offset of the stage and its increments
  int sub, nsub, stage_i, last_ragged;
  bool tail_ok;

  __device__ __forceinline__ void init(const E* base_l, int L_, int MNI_, int KI_, int row0, int k0) {
    base = base_l; MNI = MNI_; KI = KI_; L = L_;
    const int blk_elems = MNI * KI;
    const int blk_mn_stride = (MNMAJ ? L : 1) * blk_elems;
    blk_k_stride = (MNMAJ ? 1 : L) * blk_elems;
    const int unit = KC ? 1 : MNI;                       // stride of one contraction step inside a block
    rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<E*>(base_l), 0, HOW == FAR ? 0 : (int)ES * L * L * MNI * KI, 0x00020000);
    kb = k0 / KI;
    kin = k0 - kb * KI;
    const int K = L * KI, nstage = (K + ADV - 1) / ADV, ktail = K - (nstage - 1) * ADV;
#pragma unroll
    for (int q = 0; q < NMN; ++q) {
      const int row = row0 + q * ROWSTEP;
      const int mb = row / MNI, mi = row - mb * MNI;
      unsigned o = (unsigned)(mb * blk_mn_stride + mi * (KC ? KI : 1));
      if (HOW == DIVIDES) o += (unsigned)((KI >= ADV ? 0 : kb) * blk_k_stride + kin * unit);
      off[q] = row >= L * MNI ? OUTSIDE : HOW == FAR ? o : ES * o;
    }
    if (HOW == DIVIDES) {
      soff = 0; sub = 0; stage_i = 0;
      if (KI >= ADV) { nsub = KI / ADV; step_in = ES * ADV * unit; step_cross = ES * (unsigned)(blk_k_stride - (KI - ADV) * unit); }
      else { nsub = 1; step_in = 0; step_cross = ES * (unsigned)(ADV / KI * blk_k_stride); }
      last_ragged = ktail < ADV ? nstage - 1 : -1;
      tail_ok = k0 < ktail;
    } else {
      adv_b = ADV / KI;
      adv_k = ADV - adv_b * KI;
    }
  }

  __device__ __forceinline__ vec_t fetch(unsigned o, unsigned so) const {
    if constexpr (sizeof(vec_t) == 16) {
      typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
      const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)o, (int)so, 0);
      return make_float4(__uint_as_float(v.x), __uint_as_float(v.y), __uint_as_float(v.z), __uint_as_float(v.w));
    } else if constexpr (sizeof(vec_t) == 8) {
      typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
      const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(rsrc, (int)o, (int)so, 0);
      return make_float2(__uint_as_float(v.x), __uint_as_float(v.y));
    } else {
      return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)o, (int)so, 0));
    }
  }

  // the values of access (row q, step e): K-contiguous VEC steps of one row, MN-contiguous one step of VEC rows
  __device__ __forceinline__ void put(int q, int e, vec_t v) {
    if constexpr (VEC == 1) reg[q][e] = v;
    else if constexpr (sizeof(E) == 8) { reg[q][e] = make_float2(v.x, v.y); reg[KC ? q : q + 1][KC ? e + 1 : e] = make_float2(v.z, v.w); }
    else if constexpr (KC && VEC == 2) { reg[q][e] = v.x; reg[q][e + 1] = v.y; }
    else if constexpr (KC && VEC == 4) { reg[q][e] = v.x; reg[q][e + 1] = v.y; reg[q][e + 2] = v.z; reg[q][e + 3] = v.w; }
    else { reg[q][e] = v.x; reg[q + 1][e] = v.y; }
  }

  // fetches the current stage and steps to the next one
  __device__ __forceinline__ void load() {
    constexpr int QSTEP = KC ? 1 : VEC, ESTEP = KC ? VEC : 1;
    if (HOW == DIVIDES) {
      const bool ok = stage_i != last_ragged || tail_ok;
#pragma unroll
      for (int q = 0; q < NMN; q += QSTEP) {
        const unsigned o = ok ? off[q] : OUTSIDE;
#pragma unroll
        for (int e = 0; e < 8; e += ESTEP)
          put(q, e, KC ? fetch(o + ES * e, soff) : fetch(o, soff + ES * (unsigned)(e * MNI)));
      }
      ++stage_i;
      if (++sub == nsub) { sub = 0; soff += step_cross; }
      else soff += step_in;
      return;
    }
    const unsigned scale = HOW == FAR ? 1u : ES, unit = scale * (unsigned)(KC ? 1 : MNI), bstride = scale * (unsigned)blk_k_stride;
    const unsigned cross = bstride - (unsigned)KI * unit;      // from behind the end of a block to the start of the next
    int k = kin, b = kb;
    unsigned o = (unsigned)b * bstride + (unsigned)k * unit;
#pragma unroll
    for (int g = 0; g < 8; g += GR) {
#pragma unroll
      for (int q = 0; q < NMN; q += QSTEP) {
        if constexpr (HOW == FAR) {
          const bool in = b < L && off[q] != OUTSIDE;
          const E* at = base + (in ? (size_t)off[q] + o : 0);
#pragma unroll
          for (int e = 0; e < GR; e += ESTEP) {
            const vec_t v = *reinterpret_cast<const vec_t*>(in ? at + (size_t)e * unit : base);
            put(q, g + e, in ? v : vec_t{});
          }
        } else {
          const unsigned at = b < L ? off[q] + o : OUTSIDE;                                      // OUTSIDE + o is outside as well
#pragma unroll
          for (int e = 0; e < GR; e += ESTEP)
            put(q, g + e, KC ? fetch(at + scale * e, 0) : fetch(at, e * unit));
        }
      }
      k += GR;
      o += (unsigned)GR * unit;
      if (k >= KI) { k = 0; ++b; o += cross; }                // KI is a multiple of GR
    }
    kin += adv_k;
    kb += adv_b;
    if (kin >= KI) { kin -= KI; ++kb; }
  }
};

}  // namespace block
}  // namespace s2cnn
