// Block-diagonal REAL products over the (2l+1)x(2l+1) blocks of an SO(3) spectrum held in the real
// basis (see so3_real_basis.hip), on the bf16 matrix cores of gfx950 with float32 operands and results.
//
// The spectrum of a real signal on SO(3) obeys x[l,-m,-n] = (-1)^(m-n) conj(x[l,m,n]); a fixed unitary
// change of basis per degree turns every such block into a real matrix, and the complex product
// z = x y^H of two such spectra into the real product z_r = x_r y_r^T: a quarter of the multiply-adds.
//
//   fwd   : Z [(m,i),(n,j)] = sum_{(p,k)} X [(m,i),(p,k)] * Y [(p,k),(n,j)]
//   gradx : GX[(m,i),(p,k)] = sum_{(n,j)} GZ[(m,i),(n,j)] * Y [(n,j),(p,k)]
//   grady : GY[(p,k),(n,j)] = sum_{(m,i)} X [(p,k),(m,i)] * GZ[(m,i),(n,j)]
//
// with tensors stored as [l, spectral row, spectral col, feature row, feature col] (the layout of the
// complex product without the trailing pair).  As there, an operand is an L x L grid of dense feature
// blocks in which either the contraction index ("K-contiguous") or the free index ("MN-contiguous") is
// the fast one.
//
// Arithmetic: every operand value is cut into three bf16 parts and six of the nine part products are summed in float32
// (split_bf16.h).  At nl = 32, batch 16, 64 -> 64 features a product took 2.25 .. 2.35 ms with v_mfma_f32_32x32x2_f32 (77 % of
// the float32 matrix peak) and takes 1.42 / 1.46 / 1.51 ms now (gradx, fwd, grady): 1.1 PFLOP/s of bf16 instructions, the
// rate that a large library product in bf16 reaches on this card (its clock falls with the power the matrix cores draw), so
// what bounds it is energy.  Errors against 64 bits fall as well (relative 2-norm 1.02e-6 -> 8.9e-7 at that size, 3.5e-7 ->
// 2.9e-7 at 6 degrees): the products are exact and six roundings take the place of sixteen.
//
// Tiling.  A workgroup (4 waves) owns 128 x TN = 128 x (64 NCB) outputs (NCB = 2, or 1 when the 128 x 128 tiles
// of a small problem would leave CUs without work); wave (wm, wn) takes row
// blocks wm + 2i and column blocks wn + 2j (interleaved, so ragged tiles still split evenly).  The grid
// lists exactly the tiles of all degrees, heaviest degree first; inside a degree in bands of 8 tile rows, and 32 consecutive
// tiles go to one XCD, so that they share 8 + 4 operand panels in its L2 instead of fetching one panel per tile (22 degrees,
// batch 32, 100 -> 100: 3 to 6 %; 32 degrees, 64 -> 64: 2 %; 16 and 64 tiles measured the same).
//
// Tried and not kept: three workgroups per CU (168 registers): 0 to 2 % slower.
#include "common.h"
#include "split_bf16.h"
#include "block_loader.h"
#include "block_float32.h"

namespace {

using namespace s2cnn::block;
using s2cnn::v16f;
using s2cnn::SplitTile;

constexpr int NRB = 2;            // 32-row blocks per wave
constexpr int TM = 64 * NRB;
constexpr int BSTR = 64, WSTR = 32;
constexpr int TK = 32;            // contraction steps per LDS stage
constexpr int NT = 256;
constexpr int BAND = 8;           // tiles are listed in bands of 8 rows of tiles, column after column
constexpr int XCD_RUN = 32;       // consecutive tiles of the list that one XCD takes
constexpr int SMALL_GRID = 512;   // workgroups that fill the chip (2 per CU)
constexpr int SLICES_GRID = 256;  // fewer 128 x 64 tiles than this: the kernel for small problems
constexpr int SLICES_WIDE = 400;  // as many 32 x 64 tiles: two blocks per wave of it
constexpr int CHAIN_STEPS = 256;  // contractions of the forward product up to this length: the kernel with one chain per result

enum Mode { FWD = 0, GRADX = 1, GRADY = 2 };
struct MmParams {
  const float* A;
  const float* B;
  float* C;
  int nl;
  int RI;  // feature rows per block of C (and of A)
  int CI;  // feature cols per block of C (and of B)
  int KI;  // contraction features per block
};

template <int MODE> struct Cfg;
// A block (rb,kb) at rb*L+kb (MNMAJ) or kb*L+rb; same for B with (cb,kb); C (rb,cb) at rb*L+cb or cb*L+rb.
template <> struct Cfg<FWD>   { static constexpr bool A_KC = true,  B_KC = false, A_MNMAJ = true,  B_MNMAJ = true,  C_RMAJ = true;  };
template <> struct Cfg<GRADX> { static constexpr bool A_KC = true,  B_KC = true,  A_MNMAJ = true,  B_MNMAJ = false, C_RMAJ = true;  };
template <> struct Cfg<GRADY> { static constexpr bool A_KC = false, B_KC = false, A_MNMAJ = false, B_MNMAJ = false, C_RMAJ = false; };

// The loader of a workgroup's tile of EXT rows and TK steps: K-contiguous, TK / 8 threads on a row; MN-contiguous, neighbouring
// threads on neighbouring rows.
template <bool KC, bool MNMAJ, int EXT, int VEC, int HOW, int GR>
struct TileLoader : Loader<float, KC, MNMAJ, EXT * TK / (NT * 8), KC ? NT / (TK / 8) : 1, VEC, HOW, GR, TK> {
  static constexpr int NMN = EXT * TK / (NT * 8), ROWSTEP = KC ? NT / (TK / 8) : 1;
  int row0, octet;

  __device__ __forceinline__ void init(const float* base_l, int L, int MNI, int KI, int tile0) {
    const int t = threadIdx.x;
    octet = KC ? t % (TK / 8) : t / (EXT / NMN);
    row0 = KC ? t / (TK / 8) : (t % (EXT / NMN)) * NMN;
    Loader<float, KC, MNMAJ, NMN, ROWSTEP, VEC, HOW, GR, TK>::init(base_l, L, MNI, KI, tile0 + row0, 8 * octet);
  }

  __device__ __forceinline__ void store(SplitTile<EXT, TK>& tile) const {
#pragma unroll
    for (int q = 0; q < NMN; ++q) tile.put(row0 + q * ROWSTEP, octet, this->reg[q]);
  }
};

__host__ __device__ inline void tile_counts(int L, int RI, int CI, int TM, int TN, int& tm, int& tn, int& slots) {
  tm = s2cnn::ceil_div(L * RI, TM);
  tn = s2cnn::ceil_div(L * CI, TN);
  slots = tm * tn;
}

// One LDS buffer: the operands of a stage are split and written while the loads of the next stage are issued, a barrier,
// the matrix instructions, a barrier.  The other workgroup of the CU fills the matrix cores meanwhile.
template <int NCB, bool FULL, typename LA, typename LB>
__device__ __forceinline__ void contract(LA& la, LB& lb, SplitTile<TM, TK>& As, SplitTile<64 * NCB, TK>& Bs, v16f (&acc)[NRB][NCB],
                                         int nstage, int arow, int bcol, int h, int ni, int nj) {
  la.load();
  lb.load();
  for (int stage = 0; stage < nstage; ++stage) {
    la.store(As);
    lb.store(Bs);
    if (stage + 1 < nstage) {
      la.load();
      lb.load();
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < TK / 16; ++s) {
      s2cnn::SplitFragment a[NRB], b[NCB];
#pragma unroll
      for (int i = 0; i < NRB; ++i) a[i] = As.get(arow + BSTR * i, 2 * s + h);
#pragma unroll
      for (int j = 0; j < NCB; ++j) b[j] = Bs.get(bcol + BSTR * j, 2 * s + h);
      if (FULL) {
        s2cnn::split_mma<NRB, NCB>(a, b, acc);
      } else {
#pragma unroll
        for (int i = 0; i < NRB; ++i)
#pragma unroll
          for (int j = 0; j < NCB; ++j)
            if (i < ni && j < nj) s2cnn::split_mma_one(a[i], b[j], acc[i][j]);
      }
    }
    __syncthreads();
  }
}

template <int MODE, int VA, int VB, int HOW, int GR, int NCB>
__global__ __launch_bounds__(NT, 2) void so3_block_mm_real_kernel(MmParams p) {
  typedef Cfg<MODE> C_;
  constexpr int TN = 64 * NCB;

  __shared__ SplitTile<TM, TK> As;
  __shared__ SplitTile<TN, TK> Bs;

  int t = blockIdx.x;
  constexpr int ROUND = 8 * XCD_RUN;
  if (t < (int)gridDim.x / ROUND * ROUND) t = t / ROUND * ROUND + t % 8 * XCD_RUN + t % ROUND / 8;
  int l = p.nl - 1, tm = 0, tn = 0, slots = 0;
  for (;; --l) {
    tile_counts(2 * l + 1, p.RI, p.CI, TM, TN, tm, tn, slots);
    if (t < slots || l == 0) break;
    t -= slots;
  }
  const int L = 2 * l + 1;
  const int band = t / (BAND * tn), bm = tm - band * BAND < BAND ? tm - band * BAND : BAND, tb = t - band * BAND * tn;
  const int tile_m = (band * BAND + tb % bm) * TM;
  const int tile_n = tb / bm * TN;
  const size_t L0 = (size_t)l * (4 * l * l - 1) / 3;
  const int M = L * p.RI, N = L * p.CI;
  const float* A = p.A + L0 * p.RI * p.KI;
  const float* B = p.B + L0 * p.CI * p.KI;

  TileLoader<C_::A_KC, C_::A_MNMAJ, TM, VA, HOW, GR> la;
  TileLoader<C_::B_KC, C_::B_MNMAJ, TN, VB, HOW, GR> lb;
  la.init(A, L, p.RI, p.KI, tile_m);
  lb.init(B, L, p.CI, p.KI, tile_n);

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r32 = lane & 31, h = lane >> 5;
  const int wrow = (wave >> 1) * WSTR, wcol = (wave & 1) * WSTR;

  v16f acc[NRB][NCB];
#pragma unroll
  for (int i = 0; i < NRB; ++i)
#pragma unroll
    for (int j = 0; j < NCB; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  const int remr = M - tile_m - wrow, remc = N - tile_n - wcol;
  int ni = remr <= 0 ? 0 : (remr + BSTR - 1) / BSTR, nj = remc <= 0 ? 0 : (remc + BSTR - 1) / BSTR;
  ni = ni > NRB ? NRB : ni;
  nj = nj > NCB ? NCB : nj;

  const int nstage = s2cnn::ceil_div(L * p.KI, TK);
  if (ni == NRB && nj == NCB) contract<NCB, true>(la, lb, As, Bs, acc, nstage, wrow + r32, wcol + r32, h, ni, nj);
  else contract<NCB, false>(la, lb, As, Bs, acc, nstage, wrow + r32, wcol + r32, h, ni, nj);

  // Accumulator register v of lane (r32, h) holds row 8*(v/4) + 4*h + v%4 and column r32 of its 32x32 block.
  bool finite = true;
#pragma unroll
  for (int i = 0; i < NRB; ++i)
#pragma unroll
    for (int j = 0; j < NCB; ++j) finite = finite && s2cnn::finite(acc[i][j]);
  const auto same = [](float v) { return v; };
  float unscale = s2cnn::UNSCALE;
  if (!__all(finite)) {
    contract_float32<C_, NRB, NCB, BSTR>(A, B, p.RI, p.CI, p.KI, acc, L, tile_m + wrow + r32, tile_n + wcol + r32, h, same, same);
    unscale = 1.f;
  }

  float* Cl = p.C + L0 * p.RI * p.CI;
  const int blk_elems = p.RI * p.CI;
#pragma unroll
  for (int j = 0; j < NCB; ++j) {
    const int col = tile_n + wcol + BSTR * j + r32;
    if (j >= nj || col >= N) continue;
    const int cb = col / p.CI, ci = col - cb * p.CI;
#pragma unroll
    for (int i = 0; i < NRB; ++i) {
      if (i >= ni) continue;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int row0 = tile_m + wrow + BSTR * i + 8 * g + 4 * h;
        int rb = row0 / p.RI, ri = row0 - rb * p.RI;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          if (row0 + v < M) {
            const int blk = C_::C_RMAJ ? rb * L + cb : cb * L + rb;
            Cl[(size_t)blk * blk_elems + ri * p.CI + ci] = unscale * acc[i][j][4 * g + v];
          }
          if (++ri == p.RI) { ri = 0; ++rb; }
        }
      }
    }
  }
}

// Small problems: too few 128 x 64 tiles to fill the chip, so that what counts is how many loads are in flight and how few
// steps follow one another.  A workgroup owns 32 x (32 NJ) outputs and its four waves take every
// fourth 16 steps of the contraction; a lane loads the octets it feeds to the matrix instruction straight from memory
// (no LDS, no barriers, the next octets in flight meanwhile) and the four partial sums meet in LDS at the end.
// us of fwd / gradx / grady, tiles of the other kernel -> this one (the float32 kernel before): 6 degrees, batch 32, 20 -> 40:
// 14 / 21 / 20 -> 5.7 / 5.8 / 6.4 (15 / 22 / 19); the same with batch 1: 12 / 20 / 6 -> 4.7 / 5.5 / 4.0 (10 / 13 / 8); 8 degrees, batch 2,
// 50 -> 50: 37 / 36 / 8 -> 9 / 9 / 9 (23 / 24 / 9).  From 256 tiles of 128 x 64 on it is the slower one: 24 degrees, batch 4, 30 -> 30
// (440 tiles) 72 / 69 -> 74 / 82; around the line (10 to 40 stages, 230 to 360 tiles) the two are within 10 % of one another.  Two
// blocks per wave pay from 400 tiles of 32 x 64 (422: 30.4 -> 28.4, 794: 47 -> 36; 353: 38 -> 44).
template <int MODE, int VA, int VB, int HOW, int GR, int NJ>
__global__ __launch_bounds__(NT) void so3_block_mm_real_slices_kernel(MmParams p) {
  typedef Cfg<MODE> C_;
  constexpr int NW = NT / 64, TMS = 32, TNS = 32 * NJ, ADV = 16 * NW;
  __shared__ float part[NW][NJ][16][64];

  int t = blockIdx.x;
  int l = p.nl - 1, tm = 0, tn = 0, slots = 0;
  for (;; --l) {
    tile_counts(2 * l + 1, p.RI, p.CI, TMS, TNS, tm, tn, slots);
    if (t < slots || l == 0) break;
    t -= slots;
  }
  const int L = 2 * l + 1;
  const int tile_m = t % tm * TMS, tile_n = t / tm * TNS;
  const size_t L0 = (size_t)l * (4 * l * l - 1) / 3;
  const int M = L * p.RI, N = L * p.CI;
  const float* A = p.A + L0 * p.RI * p.KI;
  const float* B = p.B + L0 * p.CI * p.KI;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r32 = lane & 31, h = lane >> 5;

  Loader<float, C_::A_KC, C_::A_MNMAJ, 1, 1, VA, HOW, GR, ADV> la;
  Loader<float, C_::B_KC, C_::B_MNMAJ, NJ, 32, VB, HOW, GR, ADV> lb;
  la.init(A, L, p.RI, p.KI, tile_m + r32, 16 * wave + 8 * h);
  lb.init(B, L, p.CI, p.KI, tile_n + r32, 16 * wave + 8 * h);

  v16f acc[1][NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[0][j][v] = 0.f;

  const int nstep = s2cnn::ceil_div(L * p.KI, ADV);      // the same for all waves: steps behind the end are zeros
  la.load();
  lb.load();
  for (int step = 0; step < nstep; ++step) {
    s2cnn::SplitFragment a[1], b[NJ];
    a[0] = s2cnn::split_octet(la.reg[0]);
#pragma unroll
    for (int j = 0; j < NJ; ++j) b[j] = s2cnn::split_octet(lb.reg[j]);
    if (step + 1 < nstep) {
      la.load();
      lb.load();
    }
    s2cnn::split_mma<1, NJ>(a, b, acc);
  }

  // Accumulator register v of lane (r32, h) holds row 8*(v/4) + 4*h + v%4 and column r32; wave w adds up and stores v = 4w .. 4w+3.
#pragma unroll
  for (int j = 0; j < NJ; ++j)
#pragma unroll
    for (int v = 0; v < 16; ++v) part[wave][j][v][lane] = acc[0][j][v];
  __syncthreads();
  float sum[NJ][4];
#pragma unroll
  for (int j = 0; j < NJ; ++j)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      float s = part[0][j][4 * wave + v][lane];
#pragma unroll
      for (int w = 1; w < NW; ++w) s += part[w][j][4 * wave + v][lane];
      sum[j][v] = s;
    }
  bool finite = true;
#pragma unroll
  for (int j = 0; j < NJ; ++j) finite = finite && s2cnn::finite(sum[j]);
  float unscale = s2cnn::UNSCALE;
  if (!__all(finite)) {
    const auto same = [](float v) { return v; };
    contract_float32<C_, 1, NJ, 32>(A, B, p.RI, p.CI, p.KI, acc, L, tile_m + r32, tile_n + r32, h, same, same);
    unscale = 1.f;
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v)
        if (v / 4 == wave) sum[j][v % 4] = acc[0][j][v];
  }

  float* Cl = p.C + L0 * p.RI * p.CI;
  const int blk_elems = p.RI * p.CI;
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int col = tile_n + 32 * j + r32;
    if (col >= N) continue;
    const int cb = col / p.CI, ci = col - cb * p.CI;
    const int row0 = tile_m + 8 * wave + 4 * h;
    int rb = row0 / p.RI, ri = row0 - rb * p.RI;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      if (row0 + v < M) {
        const int blk = C_::C_RMAJ ? rb * L + cb : cb * L + rb;
        Cl[(size_t)blk * blk_elems + ri * p.CI + ci] = unscale * sum[j][v];
      }
      if (++ri == p.RI) { ri = 0; ++rb; }
    }
  }
}

// Forward products of small problems with a short contraction, with the float32 matrix instruction: a wave owns 32 x 32 outputs
// and takes the steps 8s + t, 8s + 4 + t (t = 0 .. 3) one pair after the other, so that a result is one chain of fused
// multiply-adds, rounded once per step, in an order that does not depend on the tiling.  These products lie in front of the
// activations of the small networks: a sample next to zero that falls on the other side of a ReLU is worth 5e-5 of a gradient of
// the digit network, so the last bit is kept as it is.  What bounds it is the latency of the chain (64 clocks per pair) and of the
// first loads; operands come straight from memory, 32 steps ahead.  us, slices -> this one: 6 degrees, 20 -> 40, batch 32: 5.6 -> 8.3, batch 1:
// 4.5 -> 7.6, batch 64: 7.5 -> 8.8 (a pass of the digit network takes 200); 5 degrees, batch 16, 28 -> 28: 4.8 -> 8.9.  Features in multiples of four,
// for wide loads (17 features: 14 against 6.5), and up to CHAIN_STEPS steps: from there on the chain costs several times the slices.
__global__ __launch_bounds__(NT) void so3_block_mm_real_chain_kernel(MmParams p, int tiles) {
  constexpr int T = 32, AHEAD = 4;      // groups of eight steps that are loaded together
  typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r32 = lane & 31, h = lane >> 5;
  int t = blockIdx.x * (NT / 64) + wave;
  if (t >= tiles) return;
  int l = p.nl - 1, tm = 0, tn = 0, slots = 0;
  for (;; --l) {
    tile_counts(2 * l + 1, p.RI, p.CI, T, T, tm, tn, slots);
    if (t < slots || l == 0) break;
    t -= slots;
  }
  const int L = 2 * l + 1, M = L * p.RI, N = L * p.CI;
  const int tile_m = t % tm * T, tile_n = t / tm * T;
  const size_t L0 = (size_t)l * (4 * l * l - 1) / 3;
  const int ablk = p.RI * p.KI, bblk = p.CI * p.KI;
  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.A + L0 * ablk), 0, 4 * L * L * ablk, 0x00020000);
  const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.B + L0 * bblk), 0, 4 * L * L * bblk, 0x00020000);
  const int row = tile_m + r32, col = tile_n + r32, cb = col / p.CI, ci = col - cb * p.CI;
  const unsigned ao = row < M ? 4u * (unsigned)(row / p.RI * L * ablk + row % p.RI * p.KI) : OUTSIDE;
  const unsigned bo = col < N ? 4u * (unsigned)(cb * L * bblk + ci) : OUTSIDE;

  // block and feature of the lane's first step of the group, and what they add to the offsets; a block that ends adds the way to the next
  int kb = 4 * h / p.KI, kin = 4 * h - kb * p.KI;
  const int adv_b = 8 / p.KI, adv_k = 8 - adv_b * p.KI;
  const unsigned cross_a = 4u * (unsigned)(ablk - p.KI), cross_b = 4u * (unsigned)(bblk - p.KI * p.CI);
  unsigned oa = ao + 4u * (unsigned)(kb * ablk + kin), ob = bo + 4u * (unsigned)(kb * bblk + kin * p.CI);
  float a[2][AHEAD][4], b[2][AHEAD][4];
  const auto load = [&](float (&av)[AHEAD][4], float (&bv)[AHEAD][4]) {
#pragma unroll
    for (int g = 0; g < AHEAD; ++g) {
      const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(ra, (int)(kb < L ? oa : OUTSIDE), 0, 0);      // four steps never straddle a block
      const unsigned at = kb < L ? ob : OUTSIDE;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        av[g][e] = __uint_as_float(v[e]);
        bv[g][e] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rb, (int)at, 4 * e * p.CI, 0));
      }
      kin += adv_k;
      kb += adv_b;
      oa += 4u * (unsigned)(adv_b * ablk + adv_k);
      ob += 4u * (unsigned)(adv_b * bblk + adv_k * p.CI);
      if (kin >= p.KI) { kin -= p.KI; ++kb; oa += cross_a; ob += cross_b; }
    }
  };

  v16f acc;
#pragma unroll
  for (int v = 0; v < 16; ++v) acc[v] = 0.f;
  const auto multiply = [&](const float (&av)[AHEAD][4], const float (&bv)[AHEAD][4]) {
#pragma unroll
    for (int g = 0; g < AHEAD; ++g)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(av[g][e], bv[g][e], acc, 0, 0, 0);
  };
  const int K = L * p.KI;
  load(a[0], b[0]);
  for (int k0 = 0; k0 < K; k0 += 16 * AHEAD) {      // two rounds; steps behind the end are zeros
    load(a[1], b[1]);
    multiply(a[0], b[0]);
    if (k0 + 8 * AHEAD >= K) break;
    load(a[0], b[0]);
    multiply(a[1], b[1]);
  }

  if (col >= N) return;
  float* Cl = p.C + L0 * p.RI * p.CI;
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const int row0 = tile_m + 8 * g + 4 * h;
    int rb_ = row0 / p.RI, ri = row0 - rb_ * p.RI;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      if (row0 + v < M) Cl[(size_t)(rb_ * L + cb) * (p.RI * p.CI) + ri * p.CI + ci] = acc[4 * g + v];
      if (++ri == p.RI) { ri = 0; ++rb_; }
    }
  }
}

long total_slots(int nl, int RI, int CI, int TM, int TN) {
  long n = 0;
  for (int l = 0; l < nl; ++l) {
    int tm, tn, slots;
    tile_counts(2 * l + 1, RI, CI, TM, TN, tm, tn, slots);
    n += slots;
  }
  return n > 0x7fffffffL ? -1 : n;
}

inline bool aligned4(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 3u) == 0; }

template <int MODE>
int run(const float* a, const float* b, float* c, int nl, int RI, int CI, int KI, void* stream) {
  if (!a || !b || !c || nl < 1 || RI < 1 || CI < 1 || KI < 1) return S2CNN_EINVAL;
  if (nl > 512 || (long)RI * KI > (1L << 24) || (long)CI * KI > (1L << 24) || (long)RI * CI > (1L << 24)) return S2CNN_EINVAL;
  const long Lmax = 2L * nl - 1;
  if (Lmax * Lmax * RI * KI >= (1L << 31) || Lmax * Lmax * CI * KI >= (1L << 31)) return S2CNN_EINVAL;
  if (!aligned4(a) || !aligned4(b) || !aligned4(c)) return S2CNN_EALIGN;
  // beyond the small problems: 128 x 128 tiles unless they are too few to give every CU its two workgroups: then 128 x 64
  const bool narrow = total_slots(nl, RI, CI, TM, 128) < SMALL_GRID;
  const int grid = (int)total_slots(nl, RI, CI, TM, narrow ? 64 : 128);
  if (grid < 1) return S2CNN_EINVAL;
  MmParams p{a, b, c, nl, RI, CI, KI};
  typedef Cfg<MODE> C_;
  // Wide accesses need the fast index of the operand to be a multiple of the width and a base aligned to it.  Along the
  // contraction (K-contiguous operands) the width is also the granule of the walk.
  const auto width = [](int fast, const float* q) { return fast % 4 == 0 && s2cnn::aligned16(q) ? 4 : fast % 2 == 0 && s2cnn::aligned8(q) ? 2 : 1; };
  const int wa = width(C_::A_KC ? KI : RI, a), wb = width(C_::B_KC ? KI : CI, b);
  const bool a2 = wa >= 2, b2 = wb >= 2;
  const bool near = Lmax * Lmax * RI * KI < (1L << 29) && Lmax * Lmax * CI * KI < (1L << 29);   // 32-bit byte offsets below OUTSIDE
  const bool wide = (C_::A_KC ? wa == 4 : a2) && (C_::B_KC ? wb == 4 : b2);
  const bool divides = near && wide && KI % 8 == 0 && (KI % TK == 0 || TK % KI == 0);
  hipStream_t st = static_cast<hipStream_t>(stream);
  const long tiles64 = total_slots(nl, RI, CI, TM, 64);
  if (MODE == FWD && near && tiles64 > 0 && tiles64 < SLICES_GRID && wa == 4 && Lmax * KI <= CHAIN_STEPS) {
    const int tiles = (int)total_slots(nl, RI, CI, 32, 32);
    hipLaunchKernelGGL(so3_block_mm_real_chain_kernel, dim3((unsigned)((tiles + NT / 64 - 1) / (NT / 64))), dim3(NT), 0, st, p, tiles);
    return s2cnn::launch_status();
  }
  if (near && tiles64 > 0 && tiles64 < SLICES_GRID) {
    const long tiles = total_slots(nl, RI, CI, 32, 64);
    const bool two = tiles >= SLICES_WIDE;
    const int g = (int)(two ? tiles : total_slots(nl, RI, CI, 32, 32));
#define S2CNN_SLICES(V, GR)                                                                                                                              \
  do {                                                                                                                                                   \
    if (two) hipLaunchKernelGGL((so3_block_mm_real_slices_kernel<MODE, (C_::A_KC ? V : 1), (C_::B_KC ? V : 1), WALK, GR, 2>), dim3(g), dim3(NT), 0, st, p); \
    else hipLaunchKernelGGL((so3_block_mm_real_slices_kernel<MODE, (C_::A_KC ? V : 1), (C_::B_KC ? V : 1), WALK, GR, 1>), dim3(g), dim3(NT), 0, st, p);     \
  } while (0)
    const int w = !C_::A_KC ? (KI % 4 == 0 ? 4 : 1) : C_::B_KC && wb < wa ? wb : wa;
    if (w == 4) S2CNN_SLICES(4, 4);
    else if (w == 2 && C_::A_KC) S2CNN_SLICES(2, (C_::A_KC ? 2 : 1));
    else S2CNN_SLICES(1, 1);
#undef S2CNN_SLICES
    return s2cnn::launch_status();
  }
  // a 64-column tile of an MN-contiguous operand has one column per thread
#define S2CNN_LAUNCH(VA, VB, HOW, GR)                                                                                                    \
  do {                                                                                                                                   \
    if (narrow) hipLaunchKernelGGL((so3_block_mm_real_kernel<MODE, VA, (C_::B_KC ? VB : 1), HOW, GR, 1>), dim3(grid), dim3(NT), 0, st, p); \
    else hipLaunchKernelGGL((so3_block_mm_real_kernel<MODE, VA, VB, HOW, GR, 2>), dim3(grid), dim3(NT), 0, st, p);                        \
  } while (0)
  if (!near && wide && KI % 4 == 0) S2CNN_LAUNCH((C_::A_KC ? 4 : 2), (C_::B_KC ? 4 : 2), FAR, 4);
  else if (!near && a2 && b2 && KI % 2 == 0) S2CNN_LAUNCH(2, 2, FAR, 2);
  else if (!near) S2CNN_LAUNCH(1, 1, FAR, 1);
  else if (divides) S2CNN_LAUNCH((C_::A_KC ? 4 : 2), (C_::B_KC ? 4 : 2), DIVIDES, 8);
  else if constexpr (MODE == FWD) {
    if (wa == 4) { if (b2) S2CNN_LAUNCH(4, 2, WALK, 4); else S2CNN_LAUNCH(4, 1, WALK, 4); }
    else if (wa == 2) { if (b2) S2CNN_LAUNCH(2, 2, WALK, 2); else S2CNN_LAUNCH(2, 1, WALK, 2); }
    else { if (b2) S2CNN_LAUNCH(1, 2, WALK, 1); else S2CNN_LAUNCH(1, 1, WALK, 1); }
  } else if constexpr (MODE == GRADX) {
    if (wa == 4 && wb == 4) S2CNN_LAUNCH(4, 4, WALK, 4);
    else if (a2 && b2) S2CNN_LAUNCH(2, 2, WALK, 2);
    else S2CNN_LAUNCH(1, 1, WALK, 1);
  } else if (KI % 4 == 0) {
    if (a2 && b2) S2CNN_LAUNCH(2, 2, WALK, 4);
    else if (a2) S2CNN_LAUNCH(2, 1, WALK, 4);
    else if (b2) S2CNN_LAUNCH(1, 2, WALK, 4);
    else S2CNN_LAUNCH(1, 1, WALK, 4);
  } else {
    if (a2 && b2) S2CNN_LAUNCH(2, 2, WALK, 1);
    else if (a2) S2CNN_LAUNCH(2, 1, WALK, 1);
    else if (b2) S2CNN_LAUNCH(1, 2, WALK, 1);
    else S2CNN_LAUNCH(1, 1, WALK, 1);
  }
#undef S2CNN_LAUNCH
  return s2cnn::launch_status();
}

}  // namespace

extern "C" int s2cnn_so3_mm_real_fwd(const float* x, const float* y, float* z, int nl, int nbatch, int f_in,
                                     int f_out, void* stream) {
  s2cnn::clear_stale_error();
  return run<FWD>(x, y, z, nl, nbatch, f_out, f_in, stream);
}

extern "C" int s2cnn_so3_mm_real_gradx(const float* gz, const float* y, float* gx, int nl, int nbatch, int f_in,
                                       int f_out, void* stream) {
  s2cnn::clear_stale_error();
  return run<GRADX>(gz, y, gx, nl, nbatch, f_in, f_out, stream);
}

extern "C" int s2cnn_so3_mm_real_grady(const float* gz, const float* x, float* gy, int nl, int nbatch, int f_in,
                                       int f_out, void* stream) {
  s2cnn::clear_stale_error();
  return run<GRADY>(x, gz, gy, nl, f_in, f_out, nbatch, stream);
}
