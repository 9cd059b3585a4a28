// Kernel spectrum of the SO(3) convolution layer for grids with few distinct beta values.
//
// The reference evaluates  y[l,m,n] = sum_a x_a conj(D^l_{mn}(alpha_a, beta_a, gamma_a))  as one dense product with a
// [len(grid), nspec] matrix (s2cnn/so3_ft.py:8-24).  For the points A_i that share beta_i,
//     conj D^l_{mn} = d^l_{mn}(beta_i) * exp(-i (m alpha_a + n gamma_a)),
// so  y[l,m,n] = sum_i d^l_{mn}(beta_i) G_i[m,n]  with the plane coefficients G_i[m,n] = sum_{a in A_i} x_a e^{-i(m alpha_a + n gamma_a)}:
// a product with a small matrix per beta (planes_kernel, which also serves the kernel spectra of the S^2 layers), then the
// expansion over the degrees, directly in the real basis of so3_real_basis.hip; x is real, so G_i[-m,-n] = conj G_i[m,n] and
// only n >= 0 is stored:
//     G [nbeta][(m + b-1) * b + n][re, im][ld],  m in -(b-1)..b-1,  n in 0..b-1,  ld >= ncols
// With A = y[l,+a,n], C = y[l,-a,n] (a, n >= 0) and s = (-1)^a the real-basis entries are
//     R[+a,+n] = A.re + s C.re    R[+a,-n] = -A.im - s C.im    R[-a,+n] = A.im - s C.im    R[-a,-n] = A.re - s C.re
//     a = 0: sqrt2 A.re, -sqrt2 A.im     n = 0: (A.re + s C.re)/sqrt2, (A.im - s C.im)/sqrt2     a = n = 0: A.re
// The complex form of the same spectrum needs no combination at all: y[l,+a,n] = A, y[l,-a,n] = C and, x being real,
// y[l,-a,-n] = (-1)^(a+n) conj A, y[l,+a,-n] = (-1)^(a+n) conj C (template argument CPLX: y [nspec][ncols][re, im]).
// One thread owns one pair (a, n) and V = four columns or one and walks over the degrees: G stays in registers, the
// d-values are uniform (scalar loads), every access to y is a piece of a contiguous row.  One column per thread where the
// column count is no multiple of four, and where four would leave fewer workgroups than two per CU: what counts then is how many
// loads are in flight (13 degrees, 1 485 columns, three betas: 27 -> 11 us for the adjoint, 14 -> 10 for the expansion).
#include "common.h"
#include "split_bf16.h"

namespace {

constexpr float SQRT2 = 1.41421356237309504880f, RSQRT2 = 0.70710678118654752440f;
constexpr int NBMAX = 4;
constexpr unsigned OUTSIDE = 0x80000000u;   // a byte offset behind the end of every buffer: such loads return 0

__device__ __forceinline__ int lmn_index(int l, int m, int n) { return l * (4 * l * l - 1) / 3 + (l + m) * (2 * l + 1) + (l + n); }
__device__ __forceinline__ float4 fma4(float s, float4 v, float4 acc) {
  return make_float4(fmaf(s, v.x, acc.x), fmaf(s, v.y, acc.y), fmaf(s, v.z, acc.z), fmaf(s, v.w, acc.w));
}
__device__ __forceinline__ float fma4(float s, float v, float acc) { return fmaf(s, v, acc); }
__device__ __forceinline__ float lin4(float p, float u, float q, float v) { return p * u + q * v; }
__device__ __forceinline__ float4 lin4(float p, float4 u, float q, float4 v) {   // p u + q v
  return make_float4(p * u.x + q * v.x, p * u.y + q * v.y, p * u.z + q * v.z, p * u.w + q * v.w);
}

template <int NB, bool CPLX, class V>
__global__ __launch_bounds__(256) void rft_expand_kernel(const float* __restrict__ G, const float* __restrict__ dtab,
                                                         float* __restrict__ y, int b, long ncols, long ld) {
  constexpr int W = sizeof(V) / 4;
  static_assert(W == 4 || !CPLX, "complex output comes in pairs of columns");
  const int a = blockIdx.x / b, n = blockIdx.x - a * b;
  // the thread's four columns: c0 .. c0 + 3, or, for complex output, the pairs c0, c0 + 1 and c1, c1 + 1 half a tile apart,
  // so that the 16 bytes (two complex numbers) a lane stores lie next to its neighbours'
  const long c0 = CPLX ? (long)blockIdx.y * 1024 + 2 * threadIdx.x : ((long)blockIdx.y * 256 + threadIdx.x) * W;
  const long c1 = c0 + 512;
  if (c0 >= ncols) return;
  const bool has1 = !CPLX || c1 < ncols;
  const long nspec = (long)b * (4L * b * b - 1) / 3;
  const size_t R = (size_t)(2 * b - 1) * b * 2;
  const bool stream = (size_t)nspec * (size_t)ncols * (CPLX ? 8 : 4) >= s2cnn::STREAM_BYTES;    // the spectrum is streamed: uniform
  const size_t rp = (size_t)((a + b - 1) * b + n) * 2, rm = (size_t)((-a + b - 1) * b + n) * 2;
  auto columns = [&](const float* row) {      // the thread's four columns of a row of G
    if constexpr (CPLX) {
      const float2 u = *reinterpret_cast<const float2*>(row + c0);
      const float2 v = has1 ? *reinterpret_cast<const float2*>(row + c1) : make_float2(0.f, 0.f);
      return make_float4(u.x, u.y, v.x, v.y);
    } else {
      return *reinterpret_cast<const V*>(row + c0);
    }
  };
  V pr[NB], pi[NB], mr[NB], mi[NB];
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const float* g = G + (size_t)i * R * ld;
    pr[i] = columns(g + rp * ld);
    pi[i] = columns(g + (rp + 1) * ld);
    mr[i] = columns(g + rm * ld);
    mi[i] = columns(g + (rm + 1) * ld);
  }
  const float s = (a & 1) ? -1.f : 1.f;
  const V zero{};
  for (int l = a > n ? a : n; l < b; ++l) {
    const int ip = lmn_index(l, a, n), im = lmn_index(l, -a, n);
    V Ar = zero, Ai = zero, Cr = zero, Ci = zero;
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const float d1 = dtab[i * nspec + ip], d2 = dtab[i * nspec + im];
      Ar = fma4(d1, pr[i], Ar); Ai = fma4(d1, pi[i], Ai);
      Cr = fma4(d2, mr[i], Cr); Ci = fma4(d2, mi[i], Ci);
    }
    if constexpr (CPLX) {
      // the two column pairs of a row, (re, im) interleaved: 16 bytes each
      auto put = [&](int lmn, float4 re, float4 im, float sg) {
        float* d = y + (size_t)lmn * ncols * 2;
        s2cnn::store_policy(make_float4(sg * re.x, im.x, sg * re.y, im.y), reinterpret_cast<float4*>(d + c0 * 2), stream);
        if (has1) s2cnn::store_policy(make_float4(sg * re.z, im.z, sg * re.w, im.w), reinterpret_cast<float4*>(d + c1 * 2), stream);
      };
      const float sg = ((a + n) & 1) ? -1.f : 1.f;
      const float4 nAi = make_float4(-sg * Ai.x, -sg * Ai.y, -sg * Ai.z, -sg * Ai.w);      // sg conj: (sg re, -sg im)
      const float4 nCi = make_float4(-sg * Ci.x, -sg * Ci.y, -sg * Ci.z, -sg * Ci.w);
      put(ip, Ar, Ai, 1.f);
      if (a > 0) put(im, Cr, Ci, 1.f);
      if (n > 0) {
        put(lmn_index(l, -a, -n), Ar, nAi, sg);
        if (a > 0) put(lmn_index(l, a, -n), Cr, nCi, sg);
      }
      continue;
    }
    const auto put_row = [&](V v, int lmn) { s2cnn::store_policy(v, reinterpret_cast<V*>(y + (size_t)lmn * ncols + c0), stream); };
    if (a > 0 && n > 0) {
      put_row(lin4(1.f, Ar, s, Cr), ip);
      put_row(lin4(-1.f, Ai, -s, Ci), lmn_index(l, a, -n));
      put_row(lin4(1.f, Ai, -s, Ci), im);
      put_row(lin4(1.f, Ar, -s, Cr), lmn_index(l, -a, -n));
    } else if (a > 0) {
      put_row(lin4(RSQRT2, Ar, s * RSQRT2, Cr), ip);
      put_row(lin4(RSQRT2, Ai, -s * RSQRT2, Ci), im);
    } else if (n > 0) {
      put_row(lin4(SQRT2, Ar, 0.f, zero), ip);
      put_row(lin4(-SQRT2, Ai, 0.f, zero), lmn_index(l, 0, -n));
    } else {
      put_row(Ar, ip);
    }
  }
}

// adjoint: gG_i[+-a, n] = sum_l d^l_{+-a,n}(beta_i) * (gA, gC)(l), with (gA, gC) the adjoint of the formulas above
template <int NB, class V>
__global__ __launch_bounds__(256) void rft_expand_grad_kernel(const float* __restrict__ gy, const float* __restrict__ dtab,
                                                              float* __restrict__ gG, int b, long ncols, long ld) {
  constexpr int W = sizeof(V) / 4;
  const int a = blockIdx.x / b, n = blockIdx.x - a * b;
  const long c0 = ((long)blockIdx.y * 256 + threadIdx.x) * W;
  if (c0 >= ncols) return;
  const long nspec = (long)b * (4L * b * b - 1) / 3;
  const size_t R = (size_t)(2 * b - 1) * b * 2;
  const bool stream = (size_t)nspec * (size_t)ncols * 4 >= s2cnn::STREAM_BYTES;    // the spectrum is streamed: uniform
  const size_t rp = (size_t)((a + b - 1) * b + n) * 2, rm = (size_t)((-a + b - 1) * b + n) * 2;
  const V zero{};
  V pr[NB], pi[NB], mr[NB], mi[NB];
#pragma unroll
  for (int i = 0; i < NB; ++i) pr[i] = pi[i] = mr[i] = mi[i] = zero;
  const float s = (a & 1) ? -1.f : 1.f;
  for (int l = a > n ? a : n; l < b; ++l) {
    const int ip = lmn_index(l, a, n), im = lmn_index(l, -a, n);
    const auto row = [&](int lmn) { return s2cnn::load_policy(reinterpret_cast<const V*>(gy + (size_t)lmn * ncols + c0), stream); };
    V gAr, gAi, gCr = zero, gCi = zero;
    if (a > 0 && n > 0) {
      const V gpp = row(ip);
      const V gpm = row(lmn_index(l, a, -n));
      const V gmp = row(im);
      const V gmm = row(lmn_index(l, -a, -n));
      gAr = lin4(1.f, gpp, 1.f, gmm); gAi = lin4(-1.f, gpm, 1.f, gmp);
      gCr = lin4(s, gpp, -s, gmm);    gCi = lin4(-s, gpm, -s, gmp);
    } else if (a > 0) {
      const V gpp = row(ip);
      const V gmp = row(im);
      gAr = lin4(RSQRT2, gpp, 0.f, zero);     gAi = lin4(RSQRT2, gmp, 0.f, zero);
      gCr = lin4(s * RSQRT2, gpp, 0.f, zero); gCi = lin4(-s * RSQRT2, gmp, 0.f, zero);
    } else if (n > 0) {
      const V gpp = row(ip);
      const V gpm = row(lmn_index(l, 0, -n));
      gAr = lin4(SQRT2, gpp, 0.f, zero); gAi = lin4(-SQRT2, gpm, 0.f, zero);
    } else {
      gAr = row(ip); gAi = zero;
    }
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const float d1 = dtab[i * nspec + ip], d2 = dtab[i * nspec + im];
      pr[i] = fma4(d1, gAr, pr[i]); pi[i] = fma4(d1, gAi, pi[i]);
      mr[i] = fma4(d2, gCr, mr[i]); mi[i] = fma4(d2, gCi, mi[i]);
    }
  }
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    float* g = gG + (size_t)i * R * ld + c0;
    *reinterpret_cast<V*>(g + rp * ld) = pr[i];
    *reinterpret_cast<V*>(g + (rp + 1) * ld) = pi[i];
    if (a > 0) {   // for a = 0 the (-a) row is the (+a) row
      *reinterpret_cast<V*>(g + rm * ld) = mr[i];
      *reinterpret_cast<V*>(g + (rm + 1) * ld) = mi[i];
    }
  }
}

// ---- products with the small matrix of a grid
// out [i][r][c] = scale sum_p E[i][p][r] x[c][idx[i][p]] and its adjoint gx[c][idx[i][p]] = scale sum_r Et[i][r][p] g[i][r][c], on the
// bf16 matrix cores with operands cut into three parts (split_bf16.h), straight from memory, in blocks of 32 x 32 outputs; the smallest
// with the float32 instruction (planes_chain_kernel).
// fa(k): the lane's row of the first operand at contraction step k < K; fb(k, j): its column of block j of the second.

template <int N, class F>
__device__ __forceinline__ void load_octets(float (&o)[N][8], int K, int k0, int h, F f) {
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int k = k0 + 8 * h + e;
    const bool ok = k < K;
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const float v = f(ok ? k : 0, j);
      o[j][e] = ok ? v : 0.f;
    }
  }
}

// a block again with the float32 instruction (see s2cnn::finite)
template <class FA, class FB> __device__ __forceinline__ s2cnn::v16f block_float32(int K, int h, FA fa, FB fb) {
  s2cnn::v16f acc;
#pragma unroll
  for (int v = 0; v < 16; ++v) acc[v] = 0.f;
  for (int k0 = 0; k0 < K; k0 += 2) {
    const int k = k0 + h;
    const bool ok = k < K;
    const float a = fa(ok ? k : 0), b = fb(ok ? k : 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(ok ? a : 0.f, ok ? b : 0.f, acc, 0, 0, 0);
  }
  return acc;
}

// The NW waves of the workgroup take every NW-th 16 steps of NJ blocks side by side; part: where their sums meet.  store(v, j, x) is
// called by wave v / (16 / NW) for accumulator register v of block j.
template <int NW, int NJ, class FA, class FB, class Store>
__device__ __forceinline__ void split_product(int K, int wave, int lane, FA fa, FB fb, Store store, float (*part)[NJ][16][64]) {
  constexpr int PER = 16 / NW;
  const int h = lane >> 5;
  s2cnn::v16f acc[1][NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[0][j][v] = 0.f;
  float a[1][8], b[NJ][8];
  const auto load = [&](int k0) {
    load_octets(a, K, k0, h, [&](int k, int) { return fa(k); });
    load_octets(b, K, k0, h, fb);
  };
  if (16 * wave < K) load(16 * wave);
  for (int k0 = 16 * wave; k0 < K; k0 += 16 * NW) {
    s2cnn::SplitFragment fra[1], frb[NJ];
    fra[0] = s2cnn::split_octet(a[0]);
#pragma unroll
    for (int j = 0; j < NJ; ++j) frb[j] = s2cnn::split_octet(b[j]);
    if (k0 + 16 * NW < K) load(k0 + 16 * NW);
    s2cnn::split_mma<1, NJ>(fra, frb, acc);
  }
#pragma unroll
  for (int j = 0; j < NJ; ++j)
#pragma unroll
    for (int v = 0; v < 16; ++v) part[wave][j][v][lane] = acc[0][j][v];
  __syncthreads();
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    float sum[PER], unscale = s2cnn::UNSCALE;
#pragma unroll
    for (int v = 0; v < PER; ++v) {
      const int r = PER * wave + v;
      sum[v] = part[0][j][r][lane];
#pragma unroll
      for (int w = 1; w < NW; ++w) sum[v] += part[w][j][r][lane];
    }
    if (!__all(s2cnn::finite(sum))) {
      const s2cnn::v16f again = block_float32(K, h, fa, [&](int k) { return fb(k, j); });
#pragma unroll
      for (int v = 0; v < 16; ++v)
        if (v / PER == wave) sum[v % PER] = again[v];
      unscale = 1.f;
    }
#pragma unroll
    for (int v = 0; v < PER; ++v) store(PER * wave + v, j, unscale * sum[v]);
  }
}

// scale times the sample that group member k of beta i contributes to column col (-1 in idx: no such member), rounded as a product of
// tensors is: what the layer's kernel times its factor gives
struct Samples {
  const float* x;
  const int* idx;
  int npts;
  float scale;
  bool ok;
  __device__ __forceinline__ Samples(const float* x_, const int* idx_, int i, int P, int npts_, long col, long ncols, float scale_)
      : x(x_ + (col < ncols ? col : 0) * npts_), idx(idx_ ? idx_ + (size_t)i * P : nullptr), npts(npts_), scale(scale_), ok(col < ncols) {}
  __device__ __forceinline__ float operator()(int k) const {
    const int q = idx ? idx[k] : k;
    const bool in = ok && (unsigned)q < (unsigned)npts;
    const float v = x[in ? q : 0];
    return in ? scale * v : 0.f;
  }
};

// Up to 16 STEPS points and few outputs, with the float32 matrix instruction: a wave owns 16 x 16 outputs, and a result is one chain
// of fused multiply-adds in the order in which the library's products take the points: groups of points (idx) one after the
// other, a single group by 0 2 4 6 1 3 5 7 within each eight of the whole sixteens and the rest one after the other.  So the spectra of the
// layers of a small network are bit for bit those of the public transforms, as the products behind them are kept (see
// so3_block_mm_real_chain_kernel).  Bound by the latency of two dependent loads, all of them in flight together.
constexpr int STEPS = 4;
template <bool GROUPS>
__global__ __launch_bounds__(256) void planes_chain_kernel(const float* __restrict__ x, const int* __restrict__ idx, const float* __restrict__ E,
                                                           float* __restrict__ out, int P, int R, int npts, long ncols, long ld, float scale) {
  typedef float v4f __attribute__((ext_vector_type(4)));
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r16 = lane & 15, g = lane >> 4;
  const int row0 = (blockIdx.y * 4 + wave) * 16, row = row0 + r16;
  if (row0 >= R) return;
  const long col = (long)blockIdx.x * 16 + r16;
  const bool rok = row < R;
  const float* e = E + (size_t)blockIdx.z * P * R + (rok ? row : 0);
  const Samples s(x, idx, blockIdx.z, P, npts, col, ncols, scale);
  float a[STEPS][4], b[STEPS][4];
#pragma unroll
  for (int q = 0; q < STEPS; ++q) {
    const bool whole = !GROUPS && 16 * q + 16 <= P;
    if (16 * q < P) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int k = 16 * q + (whole ? 8 * (j / 2) + (j & 1) + 2 * g : 4 * j + g), kc = k < P ? k : 0;
        const float av = e[(size_t)kc * R], bv = s(kc);
        a[q][j] = rok && k < P ? av : 0.f;
        b[q][j] = k < P ? bv : 0.f;
      }
    }
  }
  v4f acc{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int q = 0; q < STEPS; ++q)
    if (16 * q < P)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[q][j], b[q][j], acc, 0, 0, 0);
  if (!s.ok) return;
  float* o = out + (size_t)blockIdx.z * R * ld + col;
#pragma unroll
  for (int v = 0; v < 4; ++v) {      // register v of lane (r16, g) holds row 4 g + v and column r16
    const int r = row0 + 4 * g + v;
    if (r < R) o[(size_t)r * ld] = acc[v];
  }
}

// few blocks of many points: the contraction split over the waves
__global__ __launch_bounds__(256) void planes_split_kernel(const float* __restrict__ x, const int* __restrict__ idx, const float* __restrict__ E,
                                                           float* __restrict__ out, int P, int R, int npts, long ncols, long ld, float scale) {
  __shared__ float part[4][1][16][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r32 = lane & 31, h = lane >> 5;
  const long col = (long)blockIdx.x * 32 + r32;
  const int row0 = blockIdx.y * 32, row = row0 + r32;
  const bool rok = row < R;
  const float* e = E + (size_t)blockIdx.z * P * R + (rok ? row : 0);
  const Samples s(x, idx, blockIdx.z, P, npts, col, ncols, scale);
  float* o = out + (size_t)blockIdx.z * R * ld + col;
  split_product<4, 1>(
      P, wave, lane, [&](int k) { return rok ? e[(size_t)k * R] : 0.f; }, [&](int k, int) { return s(k); },
      [&](int v, int, float z) {
        const int r = row0 + 8 * (v / 4) + 4 * h + v % 4;
        if (s.ok && r < R) o[(size_t)r * ld] = z;
      },
      part);
}

// Up to 16 STEPS points and enough outputs: a wave keeps the parts of 32 columns of samples in registers, and the workgroup walks over
// ROW_BLOCKS blocks of 32 rows of E, each cut into parts once (an octet per thread) and read by the four waves from LDS.  Three betas of
// 64 points, 4 032 rows, 4 096 columns (198 MB of results): 98 us (129 with every wave cutting the rows for itself; the gather,
// masking, scaling and library product that this stands for: 131).
constexpr int ROW_BLOCKS = 8, WALK_GRID = 208;
__global__ __launch_bounds__(256) void planes_kernel(const float* __restrict__ x, const int* __restrict__ idx, const float* __restrict__ E,
                                                     float* __restrict__ out, int P, int R, int npts, long ncols, long ld, float scale) {
  static_assert(32 * 2 * STEPS == 256, "an octet of the block per thread");
  __shared__ s2cnn::SplitTile<32, 16 * STEPS> tile[2];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r32 = lane & 31, h = lane >> 5;
  const int trow = threadIdx.x & 31, toct = threadIdx.x >> 5;
  const long col = (long)blockIdx.x * 128 + 32 * wave + r32;
  const Samples s(x, idx, blockIdx.z, P, npts, col, ncols, scale);
  const float* Ei = E + (size_t)blockIdx.z * P * R;
  float* o = out + (size_t)blockIdx.z * R * ld + col;
  const int first = blockIdx.y * ROW_BLOCKS * 32, last = first + ROW_BLOCKS * 32 < R ? first + ROW_BLOCKS * 32 : R;
  float a[8];
  const auto load = [&](int row0) {
    const bool rok = row0 + trow < R;
    const float* e = Ei + (rok ? row0 + trow : 0);
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int k = 8 * toct + q;
      const bool ok = rok && k < P;
      const float v = e[(size_t)(k < P ? k : 0) * R];
      a[q] = ok ? v : 0.f;
    }
  };
  load(first);
  s2cnn::SplitFragment frb[STEPS];
#pragma unroll
  for (int q = 0; q < STEPS; ++q) {
    float b[1][8];
    load_octets(b, P, 16 * q, h, [&](int k, int) { return s(k); });
    frb[q] = s2cnn::split_octet(b[0]);
  }
  tile[0].put(trow, toct, a);
  if (first + 32 < last) load(first + 32);
  __syncthreads();
  int cur = 0;
  for (int row0 = first; row0 < last; row0 += 32, cur ^= 1) {
    s2cnn::v16f acc;
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] = 0.f;
#pragma unroll
    for (int q = 0; q < STEPS; ++q) s2cnn::split_mma_one(tile[cur].get(r32, 2 * q + h), frb[q], acc);
    if (row0 + 32 < last) tile[cur ^ 1].put(trow, toct, a);        // last read in the round before, which every wave has left
    if (row0 + 64 < last) load(row0 + 64);
    float unscale = s2cnn::UNSCALE;
    if (!__all(s2cnn::finite(acc))) {
      const bool rok = row0 + r32 < R;
      acc = block_float32(P, h, [&](int k) { return rok ? Ei[(size_t)k * R + row0 + r32] : 0.f; }, [&](int k) { return s(k); });
      unscale = 1.f;
    }
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int r = row0 + 8 * (v / 4) + 4 * h + v % 4;
      if (s.ok && r < R) o[(size_t)r * ld] = unscale * acc[v];
    }
    __syncthreads();
  }
}

// More points and enough outputs: 128 rows x 128 columns per workgroup, in stages of 32 points.  E is cut once per stage, two octets per thread,
// on its way to LDS; the samples go there as they are, fetched along the points (a wave's load covers two columns; a lane per column
// would touch a line with every value), and each wave cuts those of its 32 columns.  The next stage is in flight meanwhile.
constexpr int TILE_BLOCKS = 4, TILE_STEPS = 32;
__global__ __launch_bounds__(256, 2) void planes_tile_kernel(const float* __restrict__ x, const int* __restrict__ idx, const float* __restrict__ E,
                                                             float* __restrict__ out, int P, int R, int npts, long ncols, long ld, float scale) {
  constexpr int ROWS = 32 * TILE_BLOCKS, COLS = 128, PITCH = TILE_STEPS + 4, NX = COLS / 8;
  static_assert(ROWS * TILE_STEPS == 256 * 16 && TILE_STEPS == 32, "two octets of E per thread, a wave over two columns");
  __shared__ s2cnn::SplitTile<ROWS, TILE_STEPS> tile;
  __shared__ __attribute__((aligned(16))) float samples[COLS][PITCH];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r32 = lane & 31, h = lane >> 5;
  const int trow = threadIdx.x % ROWS, toct = threadIdx.x / ROWS, row0 = blockIdx.y * ROWS;
  const int tpoint = threadIdx.x % TILE_STEPS, tcol = threadIdx.x / TILE_STEPS;
  const long col0 = (long)blockIdx.x * COLS;
  const float* Ei = E + (size_t)blockIdx.z * P * R;
  const int* group = idx ? idx + (size_t)blockIdx.z * P : nullptr;
  // loads behind the end of a buffer are zeros, so that nothing has to be done to a value before it is used
  const long rest = ncols - col0 < COLS ? ncols - col0 : COLS;
  const __amdgpu_buffer_rsrc_t re = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(Ei), 0, 4 * P * R, 0x00020000);
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(x + col0 * npts), 0, (int)(4 * rest * npts), 0x00020000);
  const unsigned eo = row0 + trow < R ? 4u * (unsigned)(8 * toct * R + row0 + trow) : OUTSIDE, xo = 4u * (unsigned)(tcol * npts);
  float a[2][8], xs[NX];
  const auto load = [&](int k0, int place) {
#pragma unroll
    for (int o = 0; o < 2; ++o)
#pragma unroll
      for (int n = 0; n < 8; ++n)
        a[o][n] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(re, (int)(eo + 4u * (unsigned)((k0 + 16 * o + n) * R)), 0, 0));
    const int q = k0 + tpoint < P ? (group ? place : k0 + tpoint) : -1;
    const unsigned at = (unsigned)q < (unsigned)npts ? xo + 4u * (unsigned)q : OUTSIDE;
#pragma unroll
    for (int n = 0; n < NX; ++n) xs[n] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rx, (int)(at + 32u * (unsigned)(n * npts)), 0, 0));
  };
  const auto place = [&](int k0) { return group && k0 + tpoint < P ? group[k0 + tpoint] : 0; };
  s2cnn::v16f acc[TILE_BLOCKS][1];
#pragma unroll
  for (int i = 0; i < TILE_BLOCKS; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[i][0][v] = 0.f;
  load(0, place(0));
  int next = place(TILE_STEPS);
  for (int k0 = 0; k0 < P; k0 += TILE_STEPS) {
#pragma unroll
    for (int o = 0; o < 2; ++o) tile.put(trow, toct + 2 * o, a[o]);
#pragma unroll
    for (int n = 0; n < NX; ++n) samples[tcol + 8 * n][tpoint] = scale * xs[n];
    if (k0 + TILE_STEPS < P) {
      load(k0 + TILE_STEPS, next);
      next = place(k0 + 2 * TILE_STEPS);
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < TILE_STEPS / 16; ++s) {
      s2cnn::SplitFragment fa[TILE_BLOCKS], fb[1];
      const float4* o = reinterpret_cast<const float4*>(&samples[32 * wave + r32][16 * s + 8 * h]);
      const float4 u = o[0], w = o[1];
      const float octet[8] = {u.x, u.y, u.z, u.w, w.x, w.y, w.z, w.w};
      fb[0] = s2cnn::split_octet(octet);
#pragma unroll
      for (int i = 0; i < TILE_BLOCKS; ++i) fa[i] = tile.get(32 * i + r32, 2 * s + h);
      s2cnn::split_mma<TILE_BLOCKS, 1>(fa, fb, acc);
    }
    __syncthreads();
  }
  const long col = col0 + 32 * wave + r32;
  const Samples all(x, idx, blockIdx.z, P, npts, col, ncols, scale);
  float* o = out + (size_t)blockIdx.z * R * ld + col;
#pragma unroll
  for (int i = 0; i < TILE_BLOCKS; ++i) {
    const int first = row0 + 32 * i;
    s2cnn::v16f z = acc[i][0];
    float unscale = s2cnn::UNSCALE;
    if (!__all(s2cnn::finite(z))) {
      const bool ok = first + r32 < R;
      z = block_float32(P, h, [&](int k) { return ok ? Ei[(size_t)k * R + first + r32] : 0.f; }, [&](int k) { return all(k); });
      unscale = 1.f;
    }
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int r = first + 8 * (v / 4) + 4 * h + v % 4;
      if (all.ok && r < R) o[(size_t)r * ld] = unscale * z[v];
    }
  }
}

// rows: columns c of g, columns: points; 32 columns and 64 points per workgroup of NW waves.  The transposed matrix makes both operands
// coalesced; g is read once for up to 64 points.  At the size above 100 us (118 with four waves; 229 in blocks of 32 points with the
// matrix as it lies).
template <int NW>
__global__ __launch_bounds__(64 * NW) void planes_grad_kernel(const float* __restrict__ g, const int* __restrict__ idx, const float* __restrict__ Et,
                                                          float* __restrict__ gx, int P, int R, int npts, long ncols, long ld, float scale) {
  __shared__ float part[NW][2][16][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r32 = lane & 31, h = lane >> 5;
  const long c0 = (long)blockIdx.x * 32, c = c0 + r32;
  const int p0 = blockIdx.y * 64 + r32;
  const bool cok = c < ncols;
  const float* gc = g + (size_t)blockIdx.z * R * ld + (cok ? c : 0);
  const float* e = Et + (size_t)blockIdx.z * P * R;
  int q[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int p = p0 + 32 * j;
    q[j] = p >= P ? -1 : idx ? idx[(size_t)blockIdx.z * P + p] : p;
  }
  split_product<NW, 2>(
      R, wave, lane, [&](int k) { const float v = gc[(size_t)k * ld]; return cok ? v : 0.f; },
      [&](int k, int j) { const int p = p0 + 32 * j; const float v = e[(size_t)k * P + (p < P ? p : 0)]; return p < P ? v : 0.f; },
      [&](int v, int j, float z) {
        const long cc = c0 + 8 * (v / 4) + 4 * h + v % 4;
        if (cc < ncols && (unsigned)q[j] < (unsigned)npts) gx[cc * npts + q[j]] = scale * z;
      },
      part);
}

int check_planes(const void* a, const void* E, const void* o, int nbeta, int P, int R, int npts, long ncols, long ld) {
  if (!a || !E || !o || nbeta < 1 || nbeta > 65535 || P < 1 || R < 1 || npts < 1 || ncols < 1 || ncols >= (1L << 31) || ld < ncols) return S2CNN_EINVAL;
  if ((P + 31) / 32 > 65535 || (R + 31) / 32 > 65535) return S2CNN_EINVAL;
  return S2CNN_OK;
}

// Row blocks in a walk pay once there are workgroups for most CUs and the samples of a column fit the registers.  us split -> walk:
// 158 workgroups (32 points, 760 rows, 10 000 columns) 19 -> 31; 192 (14 points, 182 rows, 24 500 columns) 22 -> 27; 224 (64 points,
// 1 892 rows, 3 500 columns) 43 -> 34; 1 536 (three times 64 points, 4 032 rows, 4 096 columns) 245 -> 98.
// Fewer of both: one chain per result, up to CHAIN_LOADS loads of either operand by its waves.  us split -> chain (with the expansion where
// there are betas): 24 points, 100 rows, 20 columns (70 tiles of 16 x 16) 3.5 -> 3.6; 400 rows, 78 columns (125) 6.2 -> 3.8; 1 024 rows, 600 columns
// (2 432) 7.9 -> 6.0; three times 64 points, 132 rows, 800 columns (1 350) 9.2 -> 11.2; 380 rows, 400 columns (1 800) 10.7 -> 12.9; 650 rows,
// 1 485 columns (11 439) 31 -> 48.
constexpr long CHAIN_LOADS = 96 * 1024;      // 16 x 16 tiles times points
// More of either: tiles of 128 x 128 from TILE_GRID of them on.  us split -> tiles: 128 points, 1 024 rows, 800 columns (56 tiles) 11.5 -> 12.7, 1 200
// columns (80) 14.0 -> 12.8; 100 points, 992 rows, 1 485 columns (96) 12.9 -> 13.5; three times 64 points, 380 rows, 1 485 columns (108) 14.2 -> 9.6;
// 256 points, 400 rows, 1 200 columns (40) 12.5 -> 19.9, 1 024 rows, 4 096 columns (256) 72 -> 24; 128 points, 4 032 rows, 4 096 columns (1 024) 143
// -> 41; three times 256 points, 1 560 rows, 2 048 columns (624) 170 -> 48.
constexpr long TILE_GRID = 100;
int planes(const float* x, const int* idx, const float* E, float* out, int nbeta, int P, int R, int npts, long ncols, long ld, float scale, hipStream_t st) {
  const dim3 wide((unsigned)((ncols + 127) / 128), (R + ROW_BLOCKS * 32 - 1) / (ROW_BLOCKS * 32), nbeta), narrow((unsigned)((ncols + 31) / 32), (R + 31) / 32, nbeta),
      chain((unsigned)((ncols + 15) / 16), (R + 63) / 64, nbeta), tiles((unsigned)((ncols + 127) / 128), (R + 32 * TILE_BLOCKS - 1) / (32 * TILE_BLOCKS), nbeta);
  const bool chains = P <= 16 * STEPS && (long)chain.x * ((R + 15) / 16) * nbeta * P <= CHAIN_LOADS;
  if (P <= 16 * STEPS && (long)wide.x * wide.y * wide.z >= WALK_GRID)
    hipLaunchKernelGGL(planes_kernel, wide, dim3(256), 0, st, x, idx, E, out, P, R, npts, ncols, ld, scale);
  else if (chains && idx)
    hipLaunchKernelGGL(planes_chain_kernel<true>, chain, dim3(256), 0, st, x, idx, E, out, P, R, npts, ncols, ld, scale);
  else if (chains)
    hipLaunchKernelGGL(planes_chain_kernel<false>, chain, dim3(256), 0, st, x, idx, E, out, P, R, npts, ncols, ld, scale);
  else if ((long)tiles.x * tiles.y * tiles.z >= TILE_GRID && (P + 2L * TILE_STEPS) * R < (1L << 29) && npts < (1 << 22))      // 32-bit offsets below OUTSIDE
    hipLaunchKernelGGL(planes_tile_kernel, tiles, dim3(256), 0, st, x, idx, E, out, P, R, npts, ncols, ld, scale);
  else
    hipLaunchKernelGGL(planes_split_kernel, narrow, dim3(256), 0, st, x, idx, E, out, P, R, npts, ncols, ld, scale);
  return s2cnn::launch_status();
}

int planes_grad(const float* g, const int* idx, const float* Et, float* gx, int nbeta, int P, int R, int npts, long ncols, long ld, float scale, hipStream_t st) {
  const dim3 grid((unsigned)((ncols + 31) / 32), (P + 63) / 64, nbeta);
  if ((long)grid.x * grid.y * grid.z < 1024 && R >= 256)       // few workgroups and a long contraction: twice the waves on it
    hipLaunchKernelGGL(planes_grad_kernel<8>, grid, dim3(512), 0, st, g, idx, Et, gx, P, R, npts, ncols, ld, scale);
  else
    hipLaunchKernelGGL(planes_grad_kernel<4>, grid, dim3(256), 0, st, g, idx, Et, gx, P, R, npts, ncols, ld, scale);
  return s2cnn::launch_status();
}

int check(const void* p, const void* q, const void* r, int b, int nbeta, long ncols) {
  if (!p || !q || !r || b < 1 || b > 512 || nbeta < 1 || nbeta > NBMAX || ncols < 4 || ncols % 4 || ncols >= (1L << 31)) return S2CNN_EINVAL;
  if (!s2cnn::aligned16(p) || !s2cnn::aligned16(r)) return S2CNN_EALIGN;
  return S2CNN_OK;
}

}  // namespace

namespace {
template <bool CPLX, class V>
int launch_expand_v(const float* G, const float* dtab, float* y, int b, int nbeta, long ncols, long ld, hipStream_t st) {
  constexpr long WG = 256 * sizeof(V) / 4;
  const dim3 grid((unsigned)(b * b), (unsigned)((ncols + WG - 1) / WG));
  switch (nbeta) {
    case 1: hipLaunchKernelGGL((rft_expand_kernel<1, CPLX, V>), grid, dim3(256), 0, st, G, dtab, y, b, ncols, ld); break;
    case 2: hipLaunchKernelGGL((rft_expand_kernel<2, CPLX, V>), grid, dim3(256), 0, st, G, dtab, y, b, ncols, ld); break;
    case 3: hipLaunchKernelGGL((rft_expand_kernel<3, CPLX, V>), grid, dim3(256), 0, st, G, dtab, y, b, ncols, ld); break;
    default: hipLaunchKernelGGL((rft_expand_kernel<4, CPLX, V>), grid, dim3(256), 0, st, G, dtab, y, b, ncols, ld); break;
  }
  return s2cnn::launch_status();
}
template <class V>
int launch_expand_grad_v(const float* gy, const float* dtab, float* gG, int b, int nbeta, long ncols, long ld, hipStream_t st) {
  constexpr long WG = 256 * sizeof(V) / 4;
  const dim3 grid((unsigned)(b * b), (unsigned)((ncols + WG - 1) / WG));
  switch (nbeta) {
    case 1: hipLaunchKernelGGL((rft_expand_grad_kernel<1, V>), grid, dim3(256), 0, st, gy, dtab, gG, b, ncols, ld); break;
    case 2: hipLaunchKernelGGL((rft_expand_grad_kernel<2, V>), grid, dim3(256), 0, st, gy, dtab, gG, b, ncols, ld); break;
    case 3: hipLaunchKernelGGL((rft_expand_grad_kernel<3, V>), grid, dim3(256), 0, st, gy, dtab, gG, b, ncols, ld); break;
    default: hipLaunchKernelGGL((rft_expand_grad_kernel<4, V>), grid, dim3(256), 0, st, gy, dtab, gG, b, ncols, ld); break;
  }
  return s2cnn::launch_status();
}
// four columns per thread: whole 16-byte pieces of the rows of y (aligned to them), and at least two workgroups per CU; more
// columns than one per thread would put into the grid's second dimension too
bool four_columns(const void* y, int b, long ncols) {
  const bool can = ncols % 4 == 0 && s2cnn::aligned16(y);
  return can && ((long)b * b * ((ncols + 1023) / 1024) >= 512 || ncols > 65535L * 256);
}
int launch_expand(const float* G, const float* dtab, float* y, int b, int nbeta, long ncols, long ld, hipStream_t st) {
  return four_columns(y, b, ncols) ? launch_expand_v<false, float4>(G, dtab, y, b, nbeta, ncols, ld, st) : launch_expand_v<false, float>(G, dtab, y, b, nbeta, ncols, ld, st);
}
int launch_expand_grad(const float* gy, const float* dtab, float* gG, int b, int nbeta, long ncols, long ld, hipStream_t st) {
  return four_columns(gy, b, ncols) ? launch_expand_grad_v<float4>(gy, dtab, gG, b, nbeta, ncols, ld, st) : launch_expand_grad_v<float>(gy, dtab, gG, b, nbeta, ncols, ld, st);
}

template <bool CPLX>
int expand(const float* G, const float* dtab, float* y, int b, int nbeta, long ncols, void* stream) {
  s2cnn::clear_stale_error();
  if (int rc = check(G, dtab, y, b, nbeta, ncols)) return rc;
  if (!CPLX) return launch_expand(G, dtab, y, b, nbeta, ncols, ncols, static_cast<hipStream_t>(stream));
  return launch_expand_v<CPLX, float4>(G, dtab, y, b, nbeta, ncols, ncols, static_cast<hipStream_t>(stream));
}

// columns of the plane coefficients: whole 16-byte pieces
long padded(long ncols) { return (ncols + 3) & ~3L; }
int plane_rows(int b) { return (2 * b - 1) * b * 2; }

int check_rft(const void* x, const void* idx, const void* E, const void* dtab, const void* y, const void* ws, size_t ws_bytes, int b, int nbeta, int P,
              int npts, long ncols) {
  if (!idx || !dtab || b < 1 || b > 512 || nbeta > NBMAX) return S2CNN_EINVAL;
  if (int rc = check_planes(x, E, y, nbeta, P, plane_rows(b), npts, ncols, ncols)) return rc;
  if (!ws || ws_bytes < s2cnn_so3_rft_workspace(b, nbeta, ncols) || !s2cnn::aligned16(ws)) return S2CNN_EWORKSPACE;
  return S2CNN_OK;
}
}  // namespace

extern "C" int s2cnn_so3_rft_expand_real(const float* G, const float* dtab, float* y, int b, int nbeta, long ncols, void* stream) {
  return expand<false>(G, dtab, y, b, nbeta, ncols, stream);
}

extern "C" int s2cnn_so3_rft_expand(const float* G, const float* dtab, float* y, int b, int nbeta, long ncols, void* stream) {
  return expand<true>(G, dtab, y, b, nbeta, ncols, stream);
}

extern "C" int s2cnn_so3_rft_expand_real_grad(const float* gy, const float* dtab, float* gG, int b, int nbeta, long ncols, void* stream) {
  s2cnn::clear_stale_error();
  if (int rc = check(gy, dtab, gG, b, nbeta, ncols)) return rc;
  return launch_expand_grad(gy, dtab, gG, b, nbeta, ncols, ncols, static_cast<hipStream_t>(stream));
}

extern "C" int s2cnn_rft_planes(const float* x, const int* idx, const float* E, float* out, int nbeta, int P, int R, int npts, long ncols, long ld,
                                float scale, void* stream) {
  s2cnn::clear_stale_error();
  if (int rc = check_planes(x, E, out, nbeta, P, R, npts, ncols, ld)) return rc;
  return planes(x, idx, E, out, nbeta, P, R, npts, ncols, ld, scale, static_cast<hipStream_t>(stream));
}

extern "C" int s2cnn_rft_planes_grad(const float* g, const int* idx, const float* Et, float* gx, int nbeta, int P, int R, int npts, long ncols, long ld,
                                     float scale, void* stream) {
  s2cnn::clear_stale_error();
  if (int rc = check_planes(g, Et, gx, nbeta, P, R, npts, ncols, ld)) return rc;
  return planes_grad(g, idx, Et, gx, nbeta, P, R, npts, ncols, ld, scale, static_cast<hipStream_t>(stream));
}

extern "C" size_t s2cnn_so3_rft_workspace(int b, int nbeta, long ncols) {
  if (b < 1 || b > 512 || nbeta < 1 || nbeta > NBMAX || ncols < 1) return 0;
  return (size_t)nbeta * plane_rows(b) * padded(ncols) * sizeof(float);
}

extern "C" int s2cnn_so3_rft(const float* x, const int* idx, const float* E, const float* dtab, float* y, void* workspace, size_t workspace_bytes,
                             int b, int nbeta, int P, int npts, long ncols, float scale, int complex_out, void* stream) {
  s2cnn::clear_stale_error();
  if (int rc = check_rft(x, idx, E, dtab, y, workspace, workspace_bytes, b, nbeta, P, npts, ncols)) return rc;
  if (complex_out && ncols % 4) return S2CNN_EINVAL;
  if (complex_out && !s2cnn::aligned16(y)) return S2CNN_EALIGN;
  const long ld = padded(ncols);
  float* G = static_cast<float*>(workspace);
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (int rc = planes(x, idx, E, G, nbeta, P, plane_rows(b), npts, ncols, ld, scale, st)) return rc;
  return complex_out ? launch_expand_v<true, float4>(G, dtab, y, b, nbeta, ncols, ld, st) : launch_expand(G, dtab, y, b, nbeta, ncols, ld, st);
}

extern "C" int s2cnn_so3_rft_real_grad(const float* gy, const int* idx, const float* Et, const float* dtab, float* gx, void* workspace,
                                       size_t workspace_bytes, int b, int nbeta, int P, int npts, long ncols, float scale, void* stream) {
  s2cnn::clear_stale_error();
  if (int rc = check_rft(gy, idx, Et, dtab, gx, workspace, workspace_bytes, b, nbeta, P, npts, ncols)) return rc;
  const long ld = padded(ncols);
  float* gG = static_cast<float*>(workspace);
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (int rc = launch_expand_grad(gy, dtab, gG, b, nbeta, ncols, ld, st)) return rc;
  return planes_grad(gG, idx, Et, gx, nbeta, P, plane_rows(b), npts, ncols, ld, scale, st);
}
