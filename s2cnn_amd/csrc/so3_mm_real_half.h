// The forward product of so3_mm_real.hip with a long contraction, on the f16 matrix cores with float32 operands in two parts (split_f16.h);
// included there, inside its namespace.
//
// Three matrix instructions per product of two blocks of 32 x 16 float32 values instead of six.  Tiles of 128 x 128 and their order are those of
// the bf16 kernel.  us of that kernel -> this one: 32 degrees, batch 16, 64 -> 64: 1460 -> 1115; 22 degrees, batch 32, 100 -> 100: 1813 -> 1258;
// 16 degrees, batch 32, 100 -> 100: 579 -> 417.  Relative 2-norm errors against 64 bits 8.9e-7 -> 6.4e-7, 9.3e-7 -> 6.6e-7, 7.9e-7 -> 5.6e-7.
// What bounds it: with its loads left out the first size takes 730 us, with all of them from one cache line 975; the matrix cores are busy
// 44 % of the clocks, and the clock is at 1.7 of 2.4 GHz.
//
// The line: a workgroup looks at samples of its operands first and at all of its sums last, which short contractions do not pay back (188 steps
// 51 -> 85 us, 273 steps 75 -> 97, 688 steps equal, 992 steps 477 -> 419).  Fewer tiles than fill the chip go to the bf16 kernel with tiles of
// 128 x 64, features that are no multiple of four to the bf16 kernel as well (50 -> 70 features: 404 -> 462).  Not the gradients: with random
// operands they gain as much, but behind an activation that passes nearly everything the gradient's spectrum has columns of rounding
// noise beside those of full size, their tiles are formed twice, and the two products of the deep shape network take 4.0 and 3.6 ms instead
// of 1.8 and 1.6.
//
// Tried and not kept: tiles of 256 x 128, one workgroup per CU: 1342 us at the first size (one wave per SIMD); tiles of 256 x 256 in
// eight waves: spilled registers, 1067 where this one took 1052; one LDS buffer, cuts and matrix instructions in turn: 1079.
constexpr int HALF_STEPS = 768;   // contractions from this length on
constexpr int HALF_BLOCKS = 127, HALF_MOST = 1 << 14;      // and up to as many blocks and steps: the scales of the steps are in LDS
typedef s2cnn::StepScales<HALF_BLOCKS, HALF_MOST / 4 + 2 * TK> HalfSteps;

// The loader of a workgroup's tile of EXT rows and TK steps.  Octet o of a stage holds its steps 4o .. 4o+3 and 16 + 4o .. 16 + 4o+3 (of both
// operands).  K-contiguous: four threads on a row, 64 bytes of which they read at once; MN-contiguous: neighbouring threads on
// neighbouring (groups of VEC) rows, and half octets where a thread's share is four rows of four steps.
template <bool KC, int VEC> struct Share {      // rows and steps of a thread
  static constexpr int VALUES = 128 * TK / NT, NMN = !KC && VEC == 4 ? 4 : VALUES / 8, NK = VALUES / NMN;
  static_assert(NK == 8 || NK == 4, "octets or their halves");
};
template <bool KC, bool MNMAJ, int VEC, int HOW, int GR>
struct HalfLoader : Loader<float, KC, MNMAJ, Share<KC, VEC>::NMN, KC ? NT / (TK / 8) : 1, VEC, HOW, GR, TK, Share<KC, VEC>::NK, 16> {
  static constexpr int EXT = 128, NMN = Share<KC, VEC>::NMN, NK = Share<KC, VEC>::NK, ROWSTEP = KC ? NT / (TK / 8) : 1;
  int row0, octet, half, quad;

  __device__ __forceinline__ void init(const float* base_l, int L, int MNI, int KI, int tile0) {
    const int t = threadIdx.x;
    quad = KC ? t % (TK / 8) : t / (EXT / NMN);
    octet = quad % (TK / 8);
    half = quad / (TK / 8);
    row0 = KC ? t / (TK / 8) : t % (EXT / NMN) * NMN;
    Loader<float, KC, MNMAJ, NMN, ROWSTEP, VEC, HOW, GR, TK, NK, 16>::init(base_l, L, MNI, KI, tile0 + row0, 4 * quad);
  }

  __device__ __forceinline__ void store(SplitTile<EXT, TK>& tile) const {
#pragma unroll
    for (int q = 0; q < NMN; ++q) {
      if constexpr (NK == 8) tile.put(row0 + q * ROWSTEP, octet, this->reg[q]);
      else tile.put_half(row0 + q * ROWSTEP, octet, half, this->reg[q]);
    }
  }
  // cuts four of the values, the u-th of UNITS such shares; an octet is stored when its second half has been cut
  static constexpr int UNITS = NMN * NK / 4;
  uint4 high, low;
  float step_scale[NK / 4];       // of the granules in reg
  template <int SIGN> __device__ __forceinline__ void take_scales(const HalfSteps& steps, int stage) {
#pragma unroll
    for (int r = 0; r < NK / 4; ++r) step_scale[r] = s2cnn::power_of_two(SIGN * steps.exponent[stage * (TK / 4) + quad + 4 * r]);
  }
  template <int U> __device__ __forceinline__ void cut(HalfTile<EXT, TK>& tile, const float (&scale)[NMN]) {
    constexpr int q = U / (NK / 4), r = U % (NK / 4), e = 4 * r;
    const float s = scale[q] * step_scale[r];
    uint2 h, l;
    s2cnn::split_pair_f16(this->reg[q][e], this->reg[q][e + 1], s, h.x, l.x);
    s2cnn::split_pair_f16(this->reg[q][e + 2], this->reg[q][e + 3], s, h.y, l.y);
    if constexpr (NK == 4) tile.put_half(row0 + q * ROWSTEP, octet, half, h, l);
    else if (e == 0) { high.x = h.x; high.y = h.y; low.x = l.x; low.y = l.y; }
    else tile.put(row0 + q * ROWSTEP, octet, make_uint4(high.x, high.y, h.x, h.y), make_uint4(low.x, low.y, l.x, l.y));
  }

  // notes the rows of the tile that are not all zero
  __device__ __forceinline__ void find_present(unsigned* present, int nstage) {
    unsigned seen[NMN] = {};
    for (int stage = 0; stage < nstage; ++stage) {
      this->load();
#pragma unroll
      for (int q = 0; q < NMN; ++q)
#pragma unroll
        for (int e = 0; e < NK; ++e) seen[q] |= __float_as_uint(this->reg[q][e]) << 1;
    }
#pragma unroll
    for (int q = 0; q < NMN; ++q)
      if (seen[q]) atomicOr(&present[row0 + q * ROWSTEP], 1u);
  }
};

constexpr int NB = 2;             // 32 x 32 blocks per wave in each direction
struct HalfStage { HalfTile<TM, TK> a, b; };
struct WideStage { SplitTile<TM, TK> a, b; };

__device__ __forceinline__ void clear(v16f (&acc)[NB][NB]) {
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
}

// f(integral_constant<int, I>) for I = 0 .. N-1: indexes of registers stay constants however large the body is
template <int N, int I = 0, class F> __device__ __forceinline__ void unrolled(F f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    unrolled<N, I + 1>(f);
  }
}

// Two LDS buffers: while the matrix cores take stage s from one, the operands of stage s + 1 are cut into the other and those of stage
// s + 2 are loaded; one barrier per stage.  (Loads behind the last stage come from OUTSIDE.)  A wave does all of this side by
// side: the vector instructions of the cuts, four values at a time, stand between the matrix instructions, from the second third of
// these on, so that the loads they wait for have two thirds of a stage to arrive.
template <bool FULL, typename LA, typename LB>
__device__ __forceinline__ void contract(LA& la, LB& lb, HalfStage (&s)[2], const HalfSteps& steps, const float (&sa)[LA::NMN],
                                         const float (&sb)[LB::NMN], v16f (&acc)[NB][NB], int nstage, int arow, int bcol, int h, int ni, int nj) {
  constexpr int BLOCKS = NB * NB, HALVES = TK / 16, MMA = HALVES * 3 * BLOCKS, UNITS = LA::UNITS + LB::UNITS, FIRST = MMA / 3;
  const auto cut = [&](auto unit, HalfStage& to) {
    constexpr int U = decltype(unit)::value;
    if constexpr (U < LA::UNITS) la.template cut<U>(to.a, sa);
    else lb.template cut<U - LA::UNITS>(to.b, sb);
    if constexpr (U == LA::UNITS - 1) la.load();
    if constexpr (U == UNITS - 1) lb.load();
  };
  const auto step = [&](HalfStage& cur, HalfStage& next, int stage) {
    la.template take_scales<-1>(steps, stage + 1);
    lb.template take_scales<1>(steps, stage + 1);
    s2cnn::HalfFragment a[HALVES][NB], b[HALVES][NB];
    const auto get = [&](int k) {
#pragma unroll
      for (int i = 0; i < NB; ++i) a[k][i] = cur.a.get(arow + BSTR * i, 2 * k + h);
#pragma unroll
      for (int j = 0; j < NB; ++j) b[k][j] = cur.b.get(bcol + BSTR * j, 2 * k + h);
    };
    get(0);
    unrolled<MMA>([&](auto at) {
      constexpr int m = decltype(at)::value, k = m / (3 * BLOCKS), part = m / BLOCKS % 3, i = m % BLOCKS / NB, j = m % NB;      // the small products first
      if (FULL || (i < ni && j < nj))
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(part == 0 ? a[k][i].l : a[k][i].h, part == 1 ? b[k][j].l : b[k][j].h, acc[i][j], 0, 0, 0);
      if constexpr (m % (3 * BLOCKS) == BLOCKS && k + 1 < HALVES) get(k + 1);
      constexpr int FROM = m <= FIRST ? 0 : ((m - FIRST) * UNITS + MMA - FIRST - 1) / (MMA - FIRST);
      constexpr int TO = m < FIRST ? 0 : ((m + 1 - FIRST) * UNITS + MMA - FIRST - 1) / (MMA - FIRST);
      unrolled<TO - FROM>([&](auto n) { cut(std::integral_constant<int, FROM + decltype(n)::value>{}, next); });
      __builtin_amdgcn_sched_barrier(0);
    });
    __syncthreads();
  };
  clear(acc);
  la.load();
  lb.load();
  la.template take_scales<-1>(steps, 0);
  lb.template take_scales<1>(steps, 0);
  unrolled<UNITS>([&](auto u) { cut(u, s[0]); });
  __syncthreads();
  for (int stage = 0; stage < nstage; stage += 2) {
    step(s[0], s[1], stage);
    if (stage + 1 == nstage) break;
    step(s[1], s[0], stage + 1);
  }
}

// The same with bf16 parts, for the tiles that come here: one LDS buffer.
template <typename LA, typename LB>
__device__ __forceinline__ void contract(LA& la, LB& lb, WideStage& s, v16f (&acc)[NB][NB], int nstage, int arow, int bcol, int h, int ni, int nj) {
  clear(acc);
  for (int stage = 0; stage < nstage; ++stage) {
    la.load();
    lb.load();
    la.store(s.a);
    lb.store(s.b);
    __syncthreads();
#pragma unroll 1
    for (int k = 0; k < TK / 16; ++k) {
      s2cnn::SplitFragment b[NB];
#pragma unroll
      for (int j = 0; j < NB; ++j) b[j] = s.b.get(bcol + BSTR * j, 2 * k + h);
#pragma unroll
      for (int i = 0; i < NB; ++i) {
        if (i >= ni) continue;
        const s2cnn::SplitFragment a = s.a.get(arow + BSTR * i, 2 * k + h);
#pragma unroll
        for (int j = 0; j < NB; ++j)
          if (j < nj) s2cnn::split_mma_one(a, b[j], acc[i][j]);
      }
    }
    __syncthreads();
  }
}

template <int MODE, int VA, int VB, int HOW, int GR>
__global__ __launch_bounds__(NT, 2) void so3_block_mm_real_half_kernel(MmParams p) {
  typedef Cfg<MODE> C_;

  __shared__ union {
    HalfStage half[2];
    WideStage wide;
  } s;
  __shared__ RowScales<TM> ra, rb;
  __shared__ HalfSteps steps;

  int t = blockIdx.x;
  constexpr int ROUND = 8 * XCD_RUN;
  if (t < (int)gridDim.x / ROUND * ROUND) t = t / ROUND * ROUND + t % 8 * XCD_RUN + t % ROUND / 8;
  int l = p.nl - 1, tm = 0, tn = 0, slots = 0;
  for (;; --l) {
    tile_counts(2 * l + 1, p.RI, p.CI, TM, TM, tm, tn, slots);
    if (t < slots || l == 0) break;
    t -= slots;
  }
  const int L = 2 * l + 1;
  const int band = t / (BAND * tn), bm = tm - band * BAND < BAND ? tm - band * BAND : BAND, tb = t - band * BAND * tn;
  const int tile_m = (band * BAND + tb % bm) * TM;
  const int tile_n = tb / bm * TM;
  const size_t L0 = (size_t)l * (4 * l * l - 1) / 3;
  const int M = L * p.RI, N_ = L * p.CI;
  const float* A = p.A + L0 * p.RI * p.KI;
  const float* B = p.B + L0 * p.CI * p.KI;

  ra.clear(threadIdx.x);
  rb.clear(threadIdx.x);
  steps.clear(threadIdx.x, NT);
  __syncthreads();
  constexpr int N = 16 * TM / NT;
  const int u = threadIdx.x;
  float va[N], vb[N];
  int ka[N], kb[N];
  sample_row<C_::A_KC, C_::A_MNMAJ, N>(A, L, p.RI, p.KI, tile_m + u % TM, u / TM, va, ka);
  sample_row<C_::B_KC, C_::B_MNMAJ, N>(B, L, p.CI, p.KI, tile_n + u % TM, u / TM, vb, kb);
#pragma unroll
  for (int i = 0; i < N; ++i) steps.note(ka[i], va[i]);
  __syncthreads();
  const int nstage = s2cnn::ceil_div(L * p.KI, TK);
  const int top = steps.top(L);
  steps.finish(u, NT, L, p.KI, (nstage + 2) * (TK / 4), top);
  float ma = 0.f, mb = 0.f;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    ma = fmaxf(ma, fabsf(va[i]) * s2cnn::power_of_two(-steps.of_block(ka[i], top)));
    mb = fmaxf(mb, fabsf(vb[i]) * s2cnn::power_of_two(steps.of_block(kb[i], top)));
  }
  ra.note(u % TM, __float_as_uint(ma));
  rb.note(u % TM, __float_as_uint(mb));
  __syncthreads();
  ra.finish(threadIdx.x, M - tile_m);
  rb.finish(threadIdx.x, N_ - tile_n);
  __syncthreads();

  HalfLoader<C_::A_KC, C_::A_MNMAJ, VA, HOW, GR> la;
  HalfLoader<C_::B_KC, C_::B_MNMAJ, VB, HOW, GR> lb;
  la.init(A, L, p.RI, p.KI, tile_m);
  lb.init(B, L, p.CI, p.KI, tile_n);
  float sa[la.NMN], sb[lb.NMN];
#pragma unroll
  for (int q = 0; q < la.NMN; ++q) sa[q] = ra.scale(la.row0 + q * la.ROWSTEP);
#pragma unroll
  for (int q = 0; q < lb.NMN; ++q) sb[q] = rb.scale(lb.row0 + q * lb.ROWSTEP);

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r32 = lane & 31, h = lane >> 5;
  const int wrow = wave / 2 * WSTR, wcol = wave % 2 * WSTR;

  v16f acc[NB][NB];
  const int remr = M - tile_m - wrow, remc = N_ - tile_n - wcol;
  int ni = remr <= 0 ? 0 : (remr + BSTR - 1) / BSTR, nj = remc <= 0 ? 0 : (remc + BSTR - 1) / BSTR;
  ni = ni > NB ? NB : ni;
  nj = nj > NB ? NB : nj;

  if (ni == NB && nj == NB) contract<true>(la, lb, s.half, steps, sa, sb, acc, nstage, wrow + r32, wcol + r32, h, ni, nj);
  else contract<false>(la, lb, s.half, steps, sa, sb, acc, nstage, wrow + r32, wcol + r32, h, ni, nj);

  // Whether all sums can be relied on; rows and columns of zeros count as such once they have been looked for.
  const float least = s2cnn::TRUST * sqrtf((float)(L * p.KI));
  unsigned suspect = 0u;
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
      if (i < ni && j < nj && !__all(s2cnn::all_large(acc[i][j], least))) suspect |= 1u << (i * NB + j);
  bool again = false;
  for (int pass = 0; pass < 2; ++pass) {
    bool bad = false;
    for (unsigned left = suspect; left != 0u; left &= left - 1) {
      const int b = __builtin_ctz(left);
      v16f blk;
#pragma unroll
      for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
          if (b == i * NB + j) blk = acc[i][j];
      bad = s2cnn::too_small(s2cnn::block_maxima(blk), least, ra, rb, wrow + BSTR * (b / NB), wcol + BSTR * (b % NB), r32, h) || !s2cnn::finite(blk) || bad;
    }
    again = __syncthreads_or(bad);
    if (!again || pass == 1) break;
    if (threadIdx.x < TM) ra.present[threadIdx.x] = 0u;
    if (threadIdx.x < TM) rb.present[threadIdx.x] = 0u;
    __syncthreads();
    la.init(A, L, p.RI, p.KI, tile_m);
    lb.init(B, L, p.CI, p.KI, tile_n);
    la.find_present(ra.present, nstage);
    lb.find_present(rb.present, nstage);
    __syncthreads();
  }
  int wave_exponent = 0;             // of the results, beside those of their rows and columns
  if (again) {                       // (the sums of bf16 parts come out times SCALE^2 = 2^48)
    la.init(A, L, p.RI, p.KI, tile_m);
    lb.init(B, L, p.CI, p.KI, tile_n);
    contract(la, lb, s.wide, acc, nstage, wrow + r32, wcol + r32, h, ni, nj);
    wave_exponent = -48;
    bool finite = true;
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) finite = finite && s2cnn::finite(acc[i][j]);
    if (!__all(finite)) {
      const auto same = [](float v) { return v; };
      contract_float32<C_, NB, NB, BSTR, BSTR>(A, B, p.RI, p.CI, p.KI, acc, L, tile_m + wrow + r32, tile_n + wcol + r32, h, same, same);
      wave_exponent = 0;
    }
  }

  // Accumulator register v of lane (r32, h) holds row 8*(v/4) + 4*h + v%4 and column r32 of its 32x32 block.
  float* Cl = p.C + L0 * p.RI * p.CI;
  const int blk_elems = p.RI * p.CI;
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int col = tile_n + wcol + BSTR * j + r32;
    if (j >= nj || col >= N_) continue;
    const int cb = col / p.CI, ci = col - cb * p.CI;
    const int col_exponent = again ? wave_exponent : -rb.exponent[wcol + BSTR * j + r32];
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      if (i >= ni) continue;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int row0 = tile_m + wrow + BSTR * i + 8 * g + 4 * h;
        int rblk = row0 / p.RI, ri = row0 - rblk * p.RI;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          if (row0 + v < M) {
            const int blk = C_::C_RMAJ ? rblk * L + cb : cb * L + rblk;
            Cl[(size_t)blk * blk_elems + ri * p.CI + ci] = ldexpf(acc[i][j][4 * g + v], again ? col_exponent : col_exponent - ra.exponent[row0 - tile_m + v]);
          }
          if (++ri == p.RI) { ri = 0; ++rblk; }
        }
      }
    }
  }
}

