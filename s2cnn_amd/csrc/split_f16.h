// float32 products on the f16 matrix cores (v_mfma_f32_32x32x16_f16, the rate of the bf16 instruction), operands in two parts.
//
// A float32 value is EXACTLY the sum of two f16 values where neither leaves the range of f16: h = f16(x) takes 11 of the 24 bits of the
// mantissa, and the rest x - h, at most half a unit of h, is a multiple of 2^-12 units and so has at most 11 bits as well.  Of the
// four products of the parts of two values the smallest (l l) is left out: at most 2^-24 of the product, 2^-26.6 in the mean, and the
// other three are exact in the matrix cores and are added in float32: three matrix instructions where three bf16 parts
// (split_bf16.h) take six.
//
// What f16 lacks is range.  The blocks of the contraction therefore have a scale, a power of two that evens out their sizes in the one operand
// and is taken off the other (StepScales), and then every row of the operands has one that puts the largest of some samples of the
// row at [2^10, 2^11) (RowScales).  Then values up to 32 times that are in range, larger ones make the sums
// infinite or NaN; values from 2^-1 on, 2^-11 of the samples, are cut exactly, and smaller ones (the last bits of l) with an absolute error
// of at most 2^-25.  That is nothing beside the roundings of the sums unless a sum consists of such values: so the sums are
// looked at when they are formed (Trust), and a tile with a row or column of results that are too small for these errors, or
// not finite, is formed again with bf16 parts, which have the range of float32.
#pragma once
#include "common.h"
#include "split_bf16.h"

namespace s2cnn {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));

struct HalfFragment { v8h h, l; };

// the two parts of two values times scale, each a packed pair
__device__ __forceinline__ void split_pair_f16(float x, float y, float scale, unsigned& h, unsigned& l) {
  const float xs = x * scale, ys = y * scale;
  const v2h hh = __builtin_convertvector(v2f{xs, ys}, v2h);
  const v2h ll = {(_Float16)(xs - (float)hh[0]), (_Float16)(ys - (float)hh[1])};
  h = __builtin_bit_cast(unsigned, hh);
  l = __builtin_bit_cast(unsigned, ll);
}

// The parts of EXT rows x TK contraction steps in LDS, as in SplitTile.
template <int EXT, int TK> struct HalfTile {
  static constexpr int LD = EXT + (TK == 16 ? 4 : 2);
  uint4 part[2][TK / 8][LD];

  // the octet of a row, or half of it
  __device__ __forceinline__ void put(int row, int octet, uint4 h, uint4 l) {
    const int s = SplitTile<EXT, TK>::slot(row);
    part[0][octet][s] = h;
    part[1][octet][s] = l;
  }
  __device__ __forceinline__ void put_half(int row, int octet, int half, uint2 h, uint2 l) {
    const int s = SplitTile<EXT, TK>::slot(row);
    reinterpret_cast<uint2*>(&part[0][octet][s])[half] = h;
    reinterpret_cast<uint2*>(&part[1][octet][s])[half] = l;
  }

  __device__ __forceinline__ HalfFragment get(int row, int octet) const {
    const int s = SplitTile<EXT, TK>::slot(row);
    return {__builtin_bit_cast(v8h, part[0][octet][s]), __builtin_bit_cast(v8h, part[1][octet][s])};
  }
};

// The exponents of the scales of EXT rows of an operand.  SAMPLES values per row are looked at, at places of the contraction
// that shift from row to row; a row whose samples lie more than 2^4 below the largest of the tile is taken to be larger than they
// show (a row of few large values).  Also holds which rows there are (in the matrix, and not all zero once that has been looked at).
template <int EXT> struct RowScales {
  static constexpr int SAMPLES = 16, TARGET = 10, FLOOR = 4;
  unsigned largest[EXT];
  unsigned tile;
  int exponent[EXT];
  unsigned present[EXT];

  // all of these with a barrier of the workgroup behind each
  __device__ __forceinline__ void clear(int t) {
    if (t < EXT) { largest[t] = 0u; present[t] = 0u; }
    if (t == 0) tile = 0u;
  }
  __device__ __forceinline__ void note(int row, unsigned bits) {
    atomicMax(&largest[row], bits);
    atomicMax(&tile, bits);
  }
  __device__ __forceinline__ void finish(int t, int rows_inside) {
    if (t >= EXT) return;
    const int top = (int)(tile >> 23) - FLOOR, own = (int)(largest[t] >> 23), e = own > top ? own : top;
    const int k = tile == 0u ? 0 : TARGET + 127 - e;
    exponent[t] = k > 64 ? 64 : k < -64 ? -64 : k;
    present[t] = t < rows_inside ? 1u : 0u;
  }
  __device__ __forceinline__ float scale(int row) const { return __uint_as_float((unsigned)(127 + exponent[row]) << 23); }
};

// Scales along the contraction: operand A is taken times 2^-d, B times 2^d, d <= 0 the size of a block of A beside its largest one.  (The spectra of
// signals that hardly depend on an angle fall off by many powers of two from block to block, and so do those of kernels near the identity:
// without these scales the sums of the small blocks of one would vanish beside the large ones of the other, which they do not meet.)
// Per granule of four steps: the size of the block that it begins in.
template <int BLOCKS, int GRANULES> struct StepScales {
  static constexpr int LOWEST = -60;
  unsigned largest[BLOCKS];
  signed char exponent[GRANULES];

  __device__ __forceinline__ void clear(int t, int threads) {
    for (int i = t; i < BLOCKS; i += threads) largest[i] = 0u;
  }
  __device__ __forceinline__ void note(int block, float v) { atomicMax(&largest[block], __float_as_uint(v) & 0x7fffffffu); }
  __device__ __forceinline__ int top(int L) const {
    unsigned m = 0u;
    for (int i = 0; i < L; ++i) m = largest[i] > m ? largest[i] : m;
    return (int)(m >> 23);
  }
  __device__ __forceinline__ int of_block(int block, int top) const {
    const int d = (int)(largest[block] >> 23) - top;
    return largest[block] == 0u || d < LOWEST ? LOWEST : d;
  }
  __device__ __forceinline__ void finish(int t, int threads, int L, int KI, int granules, int top) {
    for (int g = t; g < granules; g += threads) {
      const int block = 4 * g / KI;
      exponent[g] = (signed char)(block < L ? of_block(block, top) : 0);
    }
  }
};
__device__ __forceinline__ float power_of_two(int e) { return __uint_as_float((unsigned)(127 + e) << 23); }

// What the sums of K products of scaled values are worth.  Cutting leaves absolute errors of at most 2^-25, 2^-26.8 in the mean, on values
// whose partners are around 2^9.5 or below: errors of 2^-16.3 sqrt(K) of a sum, which is 2^-20 of one of TRUST sqrt(K), the rounding that a
// float32 sum of some thousand products has.  Sums of ordinary operands are around 2^19 sqrt(K).
constexpr float TRUST = 16.f;

// largest of the 16 lanes of a row of lanes
__device__ __forceinline__ float max16(float v) {
#define S2CNN_ROR(N) v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x120 + N, 0xf, 0xf, false)));
  S2CNN_ROR(1) S2CNN_ROR(2) S2CNN_ROR(4) S2CNN_ROR(8)
#undef S2CNN_ROR
  return v;
}

// The largest results of the rows (over 16 columns) and of the columns of a block of 32 x 32 as the matrix instruction leaves it:
// register v of lane (r32, h) holds row 8*(v/4) + 4*h + v%4 and column r32.
struct BlockMaxima { float row[16], col; };
__device__ __forceinline__ BlockMaxima block_maxima(v16f acc) {
  BlockMaxima m;
  m.col = 0.f;
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const float a = fabsf(acc[v]);
    m.row[v] = max16(a);
    m.col = fmaxf(m.col, a);
  }
  m.col = fmaxf(m.col, __shfl_xor(m.col, 32));
  return m;
}

// whether all of a block's results are finite and none is below least
__device__ __forceinline__ bool all_large(v16f acc, float least) {
  float low = INFINITY;
#pragma unroll
  for (int v = 0; v < 16; ++v) low = fminf(low, fabsf(acc[v]));
  return low >= least && finite(acc);
}

// whether a row or column of the block that is there has only results below least; row0, col0: the first of the block
template <class RS, class CS>
__device__ __forceinline__ bool too_small(const BlockMaxima& m, float least, const RS& rows, const CS& cols, int row0, int col0, int r32, int h) {
  const bool col_there = cols.present[col0 + r32] != 0u;
  const bool any_col = max16(col_there ? 1.f : 0.f) > 0.f;
  bool bad = false, any_row = false;
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const bool row_there = rows.present[row0 + 8 * (v / 4) + 4 * h + v % 4] != 0u;
    any_row = any_row || row_there;
    bad = bad || (row_there && any_col && !(m.row[v] >= least));
  }
  any_row = any_row || __shfl_xor((int)any_row, 32) != 0;
  return bad || (col_there && any_row && !(m.col >= least));
}

}  // namespace s2cnn
