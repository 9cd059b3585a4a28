// Block-diagonal complex products over the (2l+1)x(2l+1) blocks of an SO(3) spectrum, on the bf16 matrix cores of gfx950 with
// float32 operands and results.
//
// For one degree l (L = 2l+1) each of the three products is a complex GEMM whose three
// index spaces are pairs (spectral index, feature index):
//
//   fwd   : Z[(m,i),(n,j)] = sum_{(p,k)} X [(m,i),(p,k)] * conj(Y[(p,k),(n,j)])
//   gradx : GX[(m,i),(p,k)] = sum_{(n,j)} GZ[(m,i),(n,j)] *      Y[(n,j),(p,k)]
//   grady : GY[(p,k),(n,j)] = sum_{(m,i)} X [(p,k),(m,i)] * conj(GZ[(m,i),(n,j)])
//
// with tensors stored as [l, spectral row, spectral col, feature row, feature col, 2].
// An operand is therefore an L x L grid of dense feature blocks; within a block either the
// contraction index ("K-contiguous") or the free index ("MN-contiguous") is the fast one.
#include "common.h"
#include "split_bf16.h"
#include "block_loader.h"
#include "block_float32.h"

namespace {

using namespace s2cnn::block;
using s2cnn::SplitFragment;
using s2cnn::SplitTile;
using s2cnn::v16f;

constexpr int NB = 2;             // 32 x 32 blocks per wave in each direction
constexpr int TM = 64 * NB;       // tile rows and columns (flattened (spectral, feature) index)
constexpr int BSTR = 64, WSTR = 32;   // a wave's blocks are 64 apart, the two waves of a dimension offset by 32
constexpr int TK = 16;            // complex contraction steps per LDS stage
constexpr int GROUP = 256;        // threads that form one of the three real products
constexpr int NT = 3 * GROUP;
constexpr int BAND = 8;           // tiles are listed in bands of 8 rows of tiles, column after column
constexpr int XCD_RUN = 32;       // consecutive tiles of the list that one XCD takes
constexpr int NTS = 256;          // threads of a workgroup of the kernel for small problems
constexpr int SMALL_TILES = 2048; // fewer 32 x 32 tiles than this: that kernel

enum Mode { FWD = 0, GRADX = 1, GRADY = 2 };
enum Kind { RE = 0, IM = 1, SUM = 2 };

struct MmParams {
  const float2* A;
  const float2* B;
  float2* C;
  int nl;
  int RI;  // feature rows per block of C (and of A)
  int CI;  // feature cols per block of C (and of B)
  int KI;  // contraction features per block
};

template <int MODE> struct Cfg;
// A block (rb,kb) at rb*L+kb (MNMAJOR) or kb*L+rb; same for B with (cb,kb); C (rb,cb) at rb*L+cb or cb*L+rb.
template <> struct Cfg<FWD>   { static constexpr bool A_KC = true,  B_KC = false, A_MNMAJ = true,  B_MNMAJ = true,  C_RMAJ = true,  CONJ = true;  };
template <> struct Cfg<GRADX> { static constexpr bool A_KC = true,  B_KC = true,  A_MNMAJ = true,  B_MNMAJ = false, C_RMAJ = true,  CONJ = false; };
template <> struct Cfg<GRADY> { static constexpr bool A_KC = false, B_KC = false, A_MNMAJ = false, B_MNMAJ = false, C_RMAJ = false, CONJ = true;  };

__host__ __device__ inline int tile_counts(int L, int RI, int CI, int TMV, int TNV, int& tm, int& tn) {
  tm = s2cnn::ceil_div(L * RI, TMV);
  tn = s2cnn::ceil_div(L * CI, TNV);
  return tm * tn;
}

// degree and place in its list of tiles, heaviest degree first
__device__ __forceinline__ int find_degree(const MmParams& p, int TMV, int TNV, int& t, int& tm, int& tn) {
  int l = p.nl - 1;
  for (;; --l) {
    const int slots = tile_counts(2 * l + 1, p.RI, p.CI, TMV, TNV, tm, tn);
    if (t < slots || l == 0) break;
    t -= slots;
  }
  return l;
}

// what one of the three products takes from a complex operand: b carries the sign of the conjugation
__device__ __forceinline__ float part_of(float2 v, int kind) { return kind == RE ? v.x : kind == IM ? v.y : v.x + v.y; }
template <bool CONJ> __device__ __forceinline__ float2 conj_of(float2 v) { return CONJ ? make_float2(v.x, -v.y) : v; }

// One operand's tile in LDS: real parts, imaginary parts (with the sign of the conjugation), their sums, each in bf16 parts.
struct OperandTile {
  SplitTile<TM, TK> kind[3];

  template <bool CONJ> __device__ __forceinline__ void put(int row, int octet, const float2 (&v)[8]) {
    float re[8], im[8], sum[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      re[e] = s2cnn::SCALE * v[e].x;
      im[e] = (CONJ ? -s2cnn::SCALE : s2cnn::SCALE) * v[e].y;
      sum[e] = re[e] + im[e];
    }
    kind[RE].put<true>(row, octet, re);
    kind[IM].put<true>(row, octet, im);
    kind[SUM].put<true>(row, octet, sum);
  }
};

constexpr int CLD = TM;           // row pitch (floats) of the products on their way to the combination
union Smem {
  struct { OperandTile a, b; } stage[2];
  float product[3][64][CLD];
};

// a thread without a share of the loads
struct NoLoader {
  __device__ __forceinline__ void load() {}
};

// The contraction loop of group G.  While the matrix cores take stage s from one buffer, the first two groups cut the operands
// of stage s + 1 (group 0 those of A, group 1 those of B, fetched during stage s - 1) into the other; one barrier per stage.
// Group 0 cuts first and multiplies second, group 1 the other way round: a SIMD holds one wave of each group, and one at most
// has the vector unit to itself while the others feed the matrix cores.
template <int G, bool FULL, bool CONJ, typename LD>
__device__ __forceinline__ void contract(LD& ld, Smem& s, v16f (&acc)[NB][NB], int nstage, int row, int octet, int arow, int bcol, int h, int ni, int nj) {
  auto put = [&](int buf) {
    if constexpr (G == 0) s.stage[buf].a.template put<false>(row, octet, ld.reg[0]);
    if constexpr (G == 1) s.stage[buf].b.template put<CONJ>(row, octet, ld.reg[0]);
  };
  auto mma = [&](int buf) {
    SplitFragment a[NB], b[NB];
#pragma unroll
    for (int i = 0; i < NB; ++i) a[i] = s.stage[buf].a.kind[G].get(arow + BSTR * i, h);
#pragma unroll
    for (int j = 0; j < NB; ++j) b[j] = s.stage[buf].b.kind[G].get(bcol + BSTR * j, h);
    if (FULL) {
      s2cnn::split_mma<NB, NB>(a, b, acc);
    } else {
#pragma unroll
      for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
          if (i < ni && j < nj) s2cnn::split_mma_one(a[i], b[j], acc[i][j]);
    }
  };
  ld.load();
  put(0);
  if (nstage > 1) ld.load();
  __syncthreads();
  for (int stage = 0; stage < nstage; ++stage) {
    const int cur = stage & 1;
    if (G != 0) mma(cur);
    if (stage + 1 < nstage) {                  // the other buffer was last read in stage - 1, which every wave has left
      put(cur ^ 1);
      if (stage + 2 < nstage) ld.load();
    }
    if (G == 0) mma(cur);
    __syncthreads();
  }
}

// Complex arithmetic on a real matrix core, three real products per complex one (Gauss): with
// b = br + i bi' (bi' = -bi where the operand is conjugated)
//     P1 = sum ar br,   P2 = sum ai bi',   P3 = sum (ar + ai)(br + bi')
//     re = P1 - P2,     im = P3 - P1 - P2.
// A workgroup of twelve waves owns 128 x 128 outputs; each of its three groups of four forms one of the real products of the
// tile, operands cut into three bf16 parts once per tile and read by the group that needs them (the sums are formed in
// float32 before they are cut, so the imaginary part carries a rounding error of the size of |a||b| eps rather than of its own
// size: the bound of any float32 complex product).  The products meet in LDS at the end.
//
// Why three groups: a wave that forms all three products of 2 x 2 blocks needs 192 accumulator registers (one wave per SIMD), and
// of 2 x 1 blocks reads 27 KB of LDS for 36 matrix instructions, more clocks than these take; a wave of a group reads 12 KB
// for 24 and holds 64 accumulators, three waves per SIMD.  LDS: 1 728 of the 2 304 clocks of matrix instructions per stage.
// One workgroup per CU (149 KB), tiles listed in bands and dealt to the XCDs in runs as in so3_mm_real.hip.
//
// Measured (us, fwd / gradx / grady; before: v_mfma_f32_32x32x2_f32 in tiles of 128 x 64, at 77 % of its peak):
//   32 degrees, batch 16,  64 ->  64:  6849 / 6839 / 6553 -> 4449 / 4453 / 4527, 1.1 PFLOP/s of bf16 instructions, the rate that
//                                      the real product reaches as well (energy: the clock falls with the power drawn)
//   22 degrees, batch 32, 100 -> 100:  8190 / 8365 / 7246 -> 4888 / 4880 / 4889
//   16 degrees, batch 16,  64 ->  64:   539 /  588 /  465 ->  367 /  371 /  307
//   24 degrees, batch  4,  30 ->  30:   277 /  267 /  503 ->  148 /  150 /  123
// Errors against 64 bits (relative 2-norm) at the first size 1.56e-6 / 1.56e-6 / 7.8e-7 -> 1.33e-6 / 1.33e-6 / 6.6e-7, smaller at all
// sizes measured.
template <int MODE, int VA, int VB, int HOW, int GA, int GB>
__global__ __launch_bounds__(NT, 3) void so3_block_mm_kernel(MmParams p) {
  typedef Cfg<MODE> C_;
  __shared__ __attribute__((aligned(16))) Smem s;

  int t = blockIdx.x;
  constexpr int ROUND = 8 * XCD_RUN;
  if (t < (int)gridDim.x / ROUND * ROUND) t = t / ROUND * ROUND + t % 8 * XCD_RUN + t % ROUND / 8;
  int tm = 0, tn = 0;
  const int l = find_degree(p, TM, TM, t, tm, tn);
  const int L = 2 * l + 1;
  const int band = t / (BAND * tn), bm = tm - band * BAND < BAND ? tm - band * BAND : BAND, tb = t - band * BAND * tn;
  const int tile_m = (band * BAND + tb % bm) * TM;
  const int tile_n = tb / bm * TM;
  const size_t L0 = (size_t)l * (4 * l * l - 1) / 3;
  const int M = L * p.RI, N = L * p.CI;
  const float2* A = p.A + L0 * p.RI * p.KI;
  const float2* B = p.B + L0 * p.CI * p.KI;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int group = wave >> 2;
  const int r32 = lane & 31, h = lane >> 5;
  const int wrow = ((wave >> 1) & 1) * WSTR, wcol = (wave & 1) * WSTR;

  v16f acc[NB][NB];
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  const int remr = M - tile_m - wrow, remc = N - tile_n - wcol;
  int ni = remr <= 0 ? 0 : (remr + BSTR - 1) / BSTR, nj = remc <= 0 ? 0 : (remc + BSTR - 1) / BSTR;
  ni = ni > NB ? NB : ni;
  nj = nj > NB ? NB : nj;
  const bool full = ni == NB && nj == NB;
  const int nstage = s2cnn::ceil_div(L * p.KI, TK);
  const int u = threadIdx.x & (GROUP - 1);
#define S2CNN_GROUP(G, LDR)                                                                                                       \
  do {                                                                                                                            \
    if (full) contract<G, true, C_::CONJ>(LDR, s, acc, nstage, row, octet, wrow + r32, wcol + r32, h, ni, nj);                     \
    else contract<G, false, C_::CONJ>(LDR, s, acc, nstage, row, octet, wrow + r32, wcol + r32, h, ni, nj);                         \
  } while (0)
  if (group == 0) {            // K-contiguous: two threads on a row; MN-contiguous: neighbouring threads on neighbouring rows
    const int row = C_::A_KC ? u >> 1 : u & (TM - 1), octet = C_::A_KC ? u & 1 : u / TM;
    Loader<float2, C_::A_KC, C_::A_MNMAJ, 1, 1, VA, HOW, GA, TK> ld;
    ld.init(A, L, p.RI, p.KI, tile_m + row, 8 * octet);
    S2CNN_GROUP(0, ld);
  } else if (group == 1) {
    const int row = C_::B_KC ? u >> 1 : u & (TM - 1), octet = C_::B_KC ? u & 1 : u / TM;
    Loader<float2, C_::B_KC, C_::B_MNMAJ, 1, 1, VB, HOW, GB, TK> ld;
    ld.init(B, L, p.CI, p.KI, tile_n + row, 8 * octet);
    S2CNN_GROUP(1, ld);
  } else {
    const int row = 0, octet = 0;
    NoLoader ld;
    S2CNN_GROUP(2, ld);
  }
#undef S2CNN_GROUP
  bool finite = true;
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) finite = finite && s2cnn::finite(acc[i][j]);
  float unscale = s2cnn::UNSCALE;
  if (!__all(finite)) {
    contract_float32<C_, NB, NB, BSTR>(A, B, p.RI, p.CI, p.KI, acc, L, tile_m + wrow + r32, tile_n + wcol + r32, h,
                                       [&](float2 v) { return part_of(v, group); }, [&](float2 v) { return part_of(conj_of<C_::CONJ>(v), group); });
    unscale = 1.f;
  }

  // Accumulator register v of lane (r32, h) holds row 8*(v/4) + 4*h + v%4 and column r32 of its 32x32 block.  64 rows of the tile at a
  // time; a thread stores every sixth row of one column.
  float2* Cl = p.C + L0 * p.RI * p.CI;
  const int blk_elems = p.RI * p.CI;
  const int ct = threadIdx.x % TM, col = tile_n + ct;
  const int cb = col / p.CI, ci = col - cb * p.CI;
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    if (i) __syncthreads();
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v)
        s.product[group][wrow + 8 * (v / 4) + 4 * h + v % 4][wcol + BSTR * j + r32] = unscale * acc[i][j][v];
    __syncthreads();
    if (col < N) {
      for (int r = threadIdx.x / TM; r < 64; r += NT / TM) {
        const int row = tile_m + BSTR * i + r;
        if (row >= M) break;
        const int rb = row / p.RI, ri = row - rb * p.RI;
        const int blk = C_::C_RMAJ ? rb * L + cb : cb * L + rb;
        const float p1 = s.product[RE][r][ct], p2 = s.product[IM][r][ct];
        Cl[(size_t)blk * blk_elems + ri * p.CI + ci] = make_float2(p1 - p2, s.product[SUM][r][ct] - p1 - p2);
      }
    }
  }
}

__device__ __forceinline__ uint4 flip_signs(uint4 v) { return make_uint4(v.x ^ 0x80008000u, v.y ^ 0x80008000u, v.z ^ 0x80008000u, v.w ^ 0x80008000u); }
__device__ __forceinline__ s2cnn::v8bf negated(s2cnn::v8bf v) {
  return __builtin_bit_cast(s2cnn::v8bf, flip_signs(__builtin_bit_cast(uint4, v)));
}

// Small problems: too few 128 x 128 tiles to fill the chip.  A workgroup owns 32 x 32 outputs, its four waves take every
// fourth 16 steps of the contraction; a lane loads the octets it feeds to the matrix instruction straight from memory (no LDS,
// no barriers, the next octets in flight meanwhile) and the four partial sums meet in LDS at the end.  What bounds it is the
// cutting of operands that each wave has to itself, so the four products of the direct form take the place of three with
// sums that would have to be cut as well (and the errors halve).
// us of fwd / gradx / grady, float32 kernel before -> tiles of 128 x 128 -> this one: 6 degrees, batch 32, 20 -> 40: 49 / 66 / 49 -> 30 / 48 / 40
// -> 12 / 12 / 11; 13 degrees, batch 11, 33 -> 45: 178 / 151 / 109 -> 96 / 134 / 65 -> 72 / 86 / 62.  The line, in 32 x 32 tiles: 1 792 (32
// degrees, batch 1, 32 -> 32) 190 us in tiles of 128, 144 here; 2 460 (24 degrees, batch 4, 30 -> 30) 154 and 165; 2 720 24.7 and 26;
// 3 174 59 and 69; 4 148 equal; 5 712 366 and 466.
template <int MODE, int VA, int VB, int HOW, int GR>
__global__ __launch_bounds__(NTS) void so3_block_mm_slices_kernel(MmParams p) {
  typedef Cfg<MODE> C_;
  constexpr int NW = NTS / 64, T = 32, ADV = 16 * NW;
  __shared__ float part[NW][2][16][64];

  int t = blockIdx.x, tm = 0, tn = 0;
  const int l = find_degree(p, T, T, t, tm, tn);
  const int L = 2 * l + 1;
  const int tile_m = t % tm * T, tile_n = t / tm * T;
  const size_t L0 = (size_t)l * (4 * l * l - 1) / 3;
  const int M = L * p.RI, N = L * p.CI;
  const float2* A = p.A + L0 * p.RI * p.KI;
  const float2* B = p.B + L0 * p.CI * p.KI;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r32 = lane & 31, h = lane >> 5;

  Loader<float2, C_::A_KC, C_::A_MNMAJ, 1, 1, VA, HOW, GR, ADV> la;
  Loader<float2, C_::B_KC, C_::B_MNMAJ, 1, 1, VB, HOW, GR, ADV> lb;
  la.init(A, L, p.RI, p.KI, tile_m + r32, 16 * wave + 8 * h);
  lb.init(B, L, p.CI, p.KI, tile_n + r32, 16 * wave + 8 * h);

  v16f re, im;
#pragma unroll
  for (int v = 0; v < 16; ++v) { re[v] = 0.f; im[v] = 0.f; }
  const auto split = [](const float2 (&v)[8], SplitFragment& r, SplitFragment& i) {
    float x[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = v[e].x;
    r = s2cnn::split_octet(x);
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = v[e].y;
    i = s2cnn::split_octet(x);
  };
  const int nstep = s2cnn::ceil_div(L * p.KI, ADV);      // the same for all waves: steps behind the end are zeros
  la.load();
  lb.load();
  for (int step = 0; step < nstep; ++step) {
    SplitFragment ar, ai, br, bi;
    split(la.reg[0], ar, ai);
    split(lb.reg[0], br, bi);
    if (step + 1 < nstep) {
      la.load();
      lb.load();
    }
    const SplitFragment bn{negated(bi.h), negated(bi.m), negated(bi.l)};
    // conjugated b: re = ar br + ai bi, im = ai br - ar bi; else re = ar br - ai bi, im = ai br + ar bi
#define S2CNN_PARTS(PA, PB)                                                                                           \
    re = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ar.PA, br.PB, re, 0, 0, 0);                                          \
    im = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ai.PA, br.PB, im, 0, 0, 0);                                          \
    re = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ai.PA, C_::CONJ ? bi.PB : bn.PB, re, 0, 0, 0);                       \
    im = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ar.PA, C_::CONJ ? bn.PB : bi.PB, im, 0, 0, 0);
    S2CNN_PARTS(l, h)
    S2CNN_PARTS(h, l)
    S2CNN_PARTS(m, m)
    S2CNN_PARTS(m, h)
    S2CNN_PARTS(h, m)
    S2CNN_PARTS(h, h)
#undef S2CNN_PARTS
  }

  // Accumulator register v of lane (r32, h) holds row 8*(v/4) + 4*h + v%4 and column r32; wave w adds up and stores v = 4w .. 4w+3.
#pragma unroll
  for (int v = 0; v < 16; ++v) { part[wave][0][v][lane] = re[v]; part[wave][1][v][lane] = im[v]; }
  __syncthreads();
  float2 sum[4];
  float part_sums[8];
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    float2 z = make_float2(part[0][0][4 * wave + v][lane], part[0][1][4 * wave + v][lane]);
#pragma unroll
    for (int w = 1; w < NW; ++w) { z.x += part[w][0][4 * wave + v][lane]; z.y += part[w][1][4 * wave + v][lane]; }
    part_sums[2 * v] = z.x;
    part_sums[2 * v + 1] = z.y;
    sum[v] = make_float2(s2cnn::UNSCALE * z.x, s2cnn::UNSCALE * z.y);
  }
  if (!__all(s2cnn::finite(part_sums))) {
    v16f p1[1][1], p2[1][1], p3[1][1];
    const auto contract_kind = [&](int kind, v16f (&acc)[1][1]) {
      contract_float32<C_, 1, 1, 32>(A, B, p.RI, p.CI, p.KI, acc, L, tile_m + r32, tile_n + r32, h, [&](float2 v) { return part_of(v, kind); },
                                     [&](float2 v) { return part_of(conj_of<C_::CONJ>(v), kind); });
    };
    contract_kind(RE, p1);
    contract_kind(IM, p2);
    contract_kind(SUM, p3);
#pragma unroll
    for (int v = 0; v < 16; ++v)
      if (v / 4 == wave) sum[v % 4] = make_float2(p1[0][0][v] - p2[0][0][v], p3[0][0][v] - p1[0][0][v] - p2[0][0][v]);
  }

  float2* Cl = p.C + L0 * p.RI * p.CI;
  const int col = tile_n + r32;
  if (col >= N) return;
  const int cb = col / p.CI, ci = col - cb * p.CI;
  const int row0 = tile_m + 8 * wave + 4 * h;
  int rb = row0 / p.RI, ri = row0 - rb * p.RI;
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    if (row0 + v < M) {
      const int blk = C_::C_RMAJ ? rb * L + cb : cb * L + rb;
      Cl[(size_t)blk * (p.RI * p.CI) + ri * p.CI + ci] = sum[v];
    }
    if (++ri == p.RI) { ri = 0; ++rb; }
  }
}

long total_slots(int nl, int RI, int CI, int TMV, int TNV) {
  long n = 0;
  for (int l = 0; l < nl; ++l) {
    int tm, tn;
    n += tile_counts(2 * l + 1, RI, CI, TMV, TNV, tm, tn);
  }
  return n > 0x7fffffffL ? -1 : n;
}

template <int MODE>
int run(const float* a, const float* b, float* c, int nl, int RI, int CI, int KI, void* stream) {
  if (!a || !b || !c || nl < 1 || RI < 1 || CI < 1 || KI < 1) return S2CNN_EINVAL;
  if (nl > 512 || (long)RI * KI > (1L << 24) || (long)CI * KI > (1L << 24) || (long)RI * CI > (1L << 24)) return S2CNN_EINVAL;
  // per-degree operand slabs are indexed with 32-bit offsets
  const long Lmax = 2L * nl - 1;
  if (Lmax * Lmax * RI * KI >= (1L << 31) || Lmax * Lmax * CI * KI >= (1L << 31)) return S2CNN_EINVAL;
  if (!s2cnn::aligned8(a) || !s2cnn::aligned8(b) || !s2cnn::aligned8(c)) return S2CNN_EALIGN;
  const long grid = total_slots(nl, RI, CI, TM, TM), small = total_slots(nl, RI, CI, 32, 32);
  if (total_slots(nl, RI, CI, 128, 64) < 1) return S2CNN_EINVAL;      // a grid beyond 2^31 - 1
  MmParams p{reinterpret_cast<const float2*>(a), reinterpret_cast<const float2*>(b),
             reinterpret_cast<float2*>(c), nl, RI, CI, KI};
  typedef Cfg<MODE> C_;
  // two complex numbers per access need a K-contiguous operand of even length and a 16-byte base
  const bool pairs = KI % 2 == 0 && (!C_::A_KC || s2cnn::aligned16(a)) && (!C_::B_KC || s2cnn::aligned16(b));
  const bool near = Lmax * Lmax * RI * KI < (1L << 28) && Lmax * Lmax * CI * KI < (1L << 28);   // byte offsets below OUTSIDE
  const bool divides = near && pairs && KI % 8 == 0 && (KI % TK == 0 || TK % KI == 0);
  hipStream_t st = static_cast<hipStream_t>(stream);
#define S2CNN_LAUNCH(V, HOW, GR) \
  hipLaunchKernelGGL((so3_block_mm_kernel<MODE, (C_::A_KC ? V : 1), (C_::B_KC ? V : 1), HOW, GR, GR>), dim3((unsigned)grid), dim3(NT), 0, st, p)
#define S2CNN_SLICES(V, GR) \
  hipLaunchKernelGGL((so3_block_mm_slices_kernel<MODE, (C_::A_KC ? V : 1), (C_::B_KC ? V : 1), WALK, GR>), dim3((unsigned)small), dim3(NTS), 0, st, p)
  if (near && small > 0 && small < SMALL_TILES) {
    if (pairs && KI % 4 == 0) S2CNN_SLICES(2, 4);
    else if (pairs) S2CNN_SLICES(2, 2);
    else S2CNN_SLICES(1, 1);
    return s2cnn::launch_status();
  }
  if (!near && pairs && KI % 4 == 0) S2CNN_LAUNCH(2, FAR, 4);
  else if (!near) S2CNN_LAUNCH(1, FAR, 1);
  else if (divides) S2CNN_LAUNCH(2, DIVIDES, 8);
  else if (pairs && KI % 4 == 0) S2CNN_LAUNCH(2, WALK, 4);
  else if (pairs) S2CNN_LAUNCH(2, WALK, 2);
  else S2CNN_LAUNCH(1, WALK, 1);
#undef S2CNN_LAUNCH
#undef S2CNN_SLICES
  return s2cnn::launch_status();
}

}  // namespace

extern "C" int s2cnn_so3_mm_fwd(const float* x, const float* y, float* z, int nl, int nbatch, int f_in,
                                int f_out, void* stream) {
  s2cnn::clear_stale_error();
  return run<FWD>(x, y, z, nl, nbatch, f_out, f_in, stream);
}

extern "C" int s2cnn_so3_mm_gradx(const float* gz, const float* y, float* gx, int nl, int nbatch, int f_in,
                                  int f_out, void* stream) {
  s2cnn::clear_stale_error();
  return run<GRADX>(gz, y, gx, nl, nbatch, f_in, f_out, stream);
}

extern "C" int s2cnn_so3_mm_grady(const float* gz, const float* x, float* gy, int nl, int nbatch, int f_in,
                                  int f_out, void* stream) {
  s2cnn::clear_stale_error();
  return run<GRADY>(x, gz, gy, nl, f_in, f_out, nbatch, stream);
}
