// float32 products on the bf16 matrix cores (v_mfma_f32_32x32x16_bf16, sixteen times the rate of the float32 instruction).
//
// A float32 value is the sum of three bf16 values: x = h + m + l with h = bf16(x), m = bf16(x - h), l = bf16(x - h - m),
// each difference exact, |m| <= 2^-9 |x| and |l| <= 2^-18 |x| (round to nearest).  Of the nine products of the parts of two
// values the three smallest (m l, l m, l l) are left out: at most 2^-26 of the product, a quarter of what a float32
// multiplication rounds off.  The other six are exact in the matrix cores and are added in float32, six matrix
// instructions per 16 contraction steps where the float32 instruction takes eight of twice the length.
#pragma once
#include "common.h"

namespace s2cnn {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef float v2f __attribute__((ext_vector_type(2)));

__device__ __forceinline__ unsigned pack_bf16(float x, float y) {
  return __builtin_bit_cast(unsigned, __builtin_convertvector(v2f{x, y}, v2bf));
}

// Values are cut times SCALE.  Every float32 value, subnormal ones included, is a multiple of 2^-149, so that its parts are multiples of
// 2^-125: none is subnormal in bf16, and every cut of a finite value below 2^104 is exact.  Sums of products of cut values come
// out times SCALE^2: UNSCALE takes that off (exactly, but for results that are subnormal and rounded once more).
// (Unscaled, parts below 2^-133 are lost: relative errors of products of values around 2^-118 and 1: 9e-6, 2^-124: 5e-4, 2^-140: 1.)
constexpr float SCALE = 0x1p24f, UNSCALE = 0x1p-48f;

// the three parts of two values (SCALED: that are times SCALE already), each a packed pair
template <bool SCALED = false> __device__ __forceinline__ void split_pair(float x, float y, unsigned& h, unsigned& m, unsigned& l) {
  const float xs = SCALED ? x : x * SCALE, ys = SCALED ? y : y * SCALE;
  h = pack_bf16(xs, ys);
  const float xr = xs - __uint_as_float(h << 16), yr = ys - __uint_as_float(h & 0xffff0000u);
  m = pack_bf16(xr, yr);
  l = pack_bf16(xr - __uint_as_float(m << 16), yr - __uint_as_float(m & 0xffff0000u));
}

struct SplitFragment { v8bf h, m, l; };

// Whether all of these sums are finite.  If not they may be none of a float32 product: the parts of an infinity, and of a value that
// rounds to one in bf16, are not its sum, and scaled sums leave the range of float32 from 2^80 on.
template <int N> __device__ __forceinline__ bool finite(const float (&v)[N]) {
  float t = 0.f;
#pragma unroll
  for (int i = 0; i < N; ++i) t = fmaf(v[i], 0.f, t);
  return t == 0.f;
}
__device__ __forceinline__ bool finite(v16f v) {
  struct Row { float f[16]; };
  return finite(__builtin_bit_cast(Row, v).f);
}

template <bool SCALED = false> __device__ __forceinline__ void split_octet(const float (&x)[8], uint4& h, uint4& m, uint4& l) {
  split_pair<SCALED>(x[0], x[1], h.x, m.x, l.x);
  split_pair<SCALED>(x[2], x[3], h.y, m.y, l.y);
  split_pair<SCALED>(x[4], x[5], h.z, m.z, l.z);
  split_pair<SCALED>(x[6], x[7], h.w, m.w, l.w);
}
__device__ __forceinline__ SplitFragment split_octet(const float (&x)[8]) {
  uint4 h, m, l;
  split_octet(x, h, m, l);
  return {__builtin_bit_cast(v8bf, h), __builtin_bit_cast(v8bf, m), __builtin_bit_cast(v8bf, l)};
}

// The parts of EXT rows x TK contraction steps in LDS: per part and octet of steps one 16-byte slot per row.  A lane's operand
// of the matrix instruction is one slot.  Two slots of padding per octet and the exchange of neighbouring slots in every
// other group of eight rows keep the stores (four octets of neighbouring rows, or every other row of one octet) and the
// loads (neighbouring rows of one octet) of eight lanes in different banks; with two octets (TK = 16: four rows of both) four.
template <int EXT, int TK> struct SplitTile {
  static constexpr int LD = EXT + (TK == 16 ? 4 : 2);
  uint4 part[3][TK / 8][LD];

  static __device__ __forceinline__ int slot(int row) { return row ^ ((row >> 3) & 1); }

  template <bool SCALED = false> __device__ __forceinline__ void put(int row, int octet, const float (&x)[8]) {
    uint4 h, m, l;
    split_octet<SCALED>(x, h, m, l);
    const int s = slot(row);
    part[0][octet][s] = h;
    part[1][octet][s] = m;
    part[2][octet][s] = l;
  }

  __device__ __forceinline__ SplitFragment get(int row, int octet) const {
    const int s = slot(row);
    return {__builtin_bit_cast(v8bf, part[0][octet][s]), __builtin_bit_cast(v8bf, part[1][octet][s]), __builtin_bit_cast(v8bf, part[2][octet][s])};
  }
};

// acc += a b, the small products first
__device__ __forceinline__ void split_mma_one(const SplitFragment& a, const SplitFragment& b, v16f& acc) {
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.l, b.h, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.h, b.l, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.m, b.m, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.m, b.h, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.h, b.m, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.h, b.h, acc, 0, 0, 0);
}

// the same for NI x NJ blocks, consecutive instructions on different accumulators
template <int NI, int NJ>
__device__ __forceinline__ void split_mma(const SplitFragment (&a)[NI], const SplitFragment (&b)[NJ], v16f (&acc)[NI][NJ]) {
#define S2CNN_PARTS(PA, PB)                                                                                     \
  _Pragma("unroll") for (int i = 0; i < NI; ++i) _Pragma("unroll") for (int j = 0; j < NJ; ++j)                 \
      acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i].PA, b[j].PB, acc[i][j], 0, 0, 0);
  S2CNN_PARTS(l, h)
  S2CNN_PARTS(h, l)
  S2CNN_PARTS(m, m)
  S2CNN_PARTS(m, h)
  S2CNN_PARTS(h, m)
  S2CNN_PARTS(h, h)
#undef S2CNN_PARTS
}

}  // namespace s2cnn
