// Products of some tens to many thousands of rows with activations in half form (FORM_HALF; pg_half.h) and W in half
// form beside its stored rows (transposed_dense_projection_into, src/models/cpu.rs:58-75).
//
// f32 inputs and sums on the f16 matrix cores.  An input value times a power of two is two f16 numbers, hi and lo, an
// f32 weight too (its row times a power of two of its own); a bf16 or int8 weight is one f16 number as it is.  So
// x w = hi w + lo w, two v_mfma_f32_32x32x16_f16 with exact products, where three bf16 parts take three instructions
// (pg_gemm_cut.hip); for f32 rows three, hi hi + hi lo + lo hi, where they take six.
//
// What is lost: two f16 hold 23 of a value's 24 significant bits, all 24 of three values in four, so that a product is off by
// 6 10^-8 in the mean, of either sign, and lo lo is 2^-24 and less.  Over a sum of K products that is 7 10^-8 of the result
// (bf16 and int8 rows 4 10^-8), below what its roundings cost: with one f32 sum over K = 1600 2.7 10^-7.  Those are made
// fewer for it: a chain of matrix instructions ends after CH stages, 64 to 128 columns, and is added to a total, and wherever
// there are registers for it the small products are a chain of their own (in one with the others they are cut downward, and
// the error has a mean: a model's logits were off by up to 1.4 times as much), or every second chain has the other sign.  Error against f64 (values N(0, 1) by N(0, 0.02), of
// the result's norm, 512 rows), one part of K, before -> now: 1280 x 1280 f32 rows 2.1 10^-7 -> 1.3, K = 5120 4.5 -> 1.6 (64 x
// 64 a wavefront: 1.4, 2.1); bf16 rows 2.1 -> 1.1, 4.5 -> 1.5; 128 x 256 tiles, one chain, 16384 x 1600 x 1600 4.3 -> 3.6.
// Logits of prompts of 450 to 1000 tokens, all sizes: 0.65 to 0.85 of what they were off by.
//
// The range of f16: every column of the inputs has a power of two of its own, with which none of its values can be past 2^15
// whatever the model is given (k_half_bound: what a LayerNorm, a projection of one, an average of such or a GELU of such can
// reach at most), and W's half form has its inverse in that column.  Below 2^-2 a value is right to 2^-25, 2^-40 of its own column's
// bound, and so is a weight with its column's power to 2^-40 of the largest in its row: of a product that counts, whatever the
// sizes of the gains and of the columns of W are to each other.  f16 subnormals count in these instructions.
//
// How operands travel: a producer cuts a value once, in its epilogue; here all are operands as they lie, whole KB by
// global_load_lds without registers, LDS reads free of conflicts without a permutation, no vector instruction in the loop
// but a chain's end.  1000 x 4800 x 1600 f32 rows 102 us and a reduction of 11 -> 52, 1000 x 6400 x 1600 113 -> 58, 8192 x
// 4800 x 1600 606 -> 337; bf16 16384 x 4800 x 1600 610 -> 436, 16384 x 1600 x 6400 880 -> 606 (1125 TFLOP/s of matrix
// instructions; a plain library product reaches 1354).
//
// The same kernels serve rows in cut form (bf16, three parts) with W in cut form beside its stored rows, six products: what
// pg_gemm_rows.hip and pg_gemm_cut.hip do with W as stored, without the cut of W in every block.  For f32 models narrow enough
// that W's six bytes a weight do not outweigh it (make_half_form): 1024 rows, 768 wide, the four products 28.4, 16.0, 40.0,
// 34.6 -> 26.7, 15.7, 29.7, 34.6 us with the plans fitted to half form, 24.9, 15.7, 29.9, 32.5 the best ones; logits 0.86 to 0.95
// of what they were off by (129 to 1024 tokens: chains as in half form).
#include "pg_gemm_dev.h"
#include "pg_half.h"
#include "pg_wave.h"

#include <type_traits>

namespace pgk {

namespace {

// The products of parts (input, weight) that stand for one in f32, small ones first: half form with one or two parts a weight, cut form.
template <int PX, int PW>
struct Products {
  static constexpr int n = PX == 3 ? 6 : PW + 1;
  static constexpr int x[6] = {PX - 1, 0, PX == 3 ? 1 : 0, 1, 0, 0};
  static constexpr int w[6] = {0, PX == 3 ? 2 : PW - 1, PX == 3 ? 1 : 0, 0, PW > 1 ? 1 : 0, 0};
};

// Planes of W in an octet of columns, and which of them is the second part for the m-th block of input rows (k_half_rows).
template <int PW>
__device__ __forceinline__ int planes_of(const GemmArgs& a) {
  return PW == 2 ? a.w_half_planes : PW;
}
template <int PW>
__device__ __forceinline__ int second_plane(const GemmArgs& a, int m) {
  return PW == 2 ? 1 + (m & (a.w_half_planes - 2)) : 1;
}

// GELU of sum + bias, four columns of a row, in half form with what f32 rounds away on the way, or in cut form.
template <int PX>
__device__ __forceinline__ void store_gelu(void* to, int mp, size_t m, size_t n, f4 sum, f4 bias, f4 scale) {
  const f4 c = bias + sum, b = c - sum, c_rest = (bias - b) + (sum - (c - b));
  f4 y, rest;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float r;
    y[e] = gelu_tanh(c[e], c_rest[e], r);
    rest[e] = r;
  }
  if constexpr (PX == 3) store_cut4(to, mp, m, n, y);
  else store_half4(to, mp, m, n, y, rest, scale);
}

// WM x WN wavefronts, each on MB x NB blocks of 32 x 32.  The operands are turned round: lane (l, half) of the first holds
// columns 8 half .. 8 half + 7 of row l of W, of the second those of input row l, so that the result's lane is a row
// of C and its values four by four neighbouring columns.  PX, PW: parts of an input value (3: cut form, on the bf16 cores; W
// then has three parts too) and of a weight (2: f32 rows in half form).  K runs in stages of KT
// columns in NA buffers, a stage in steps of 16 whose operands are read during the step before.  One barrier per stage, in front of the step that reads the next stage: by then the wavefront has
// waited for its own share of that stage, and has read the stage before it to the end, whose buffer is free for the stage that
// is asked for next.  CH: stages in a chain of matrix instructions (0: one chain).  TWO: the small products of a chain have a
// sum of their own.  TURN: where there are no registers for that, every second chain has W's sign turned, and its sum is taken away
// instead of added: the instructions cut what they add downward, most of all what is small next to the sum, and so the errors of two
// chains cancel, which are of one sign otherwise (bf16 rows, K = 1024, a mean of -0.19 of 2^-23 of the outputs' size -> -0.01).  SPLIT: the stages are cut into gridDim.y parts, raw partial tiles go to a.ws[part][M][N].  OCC:
// wavefronts per SIMD that the registers are kept for.
template <int WM, int WN, int MB, int NB, int PX, int PW, int EPI, int SPLIT, int OCC, int NA, int KT, int CH, bool TWO, bool TURN>
__global__ __launch_bounds__(64 * WM * WN, OCC) void k_gemm_half(GemmArgs a) {
  constexpr int NW = WM * WN, BM = 32 * MB * WM, BN = 32 * NB * WN, NO = KT / 8, NS = KT / 16;
  constexpr int IA = NO * PX * BM / 64 / NW, IB = NO * PW * BN / 64 / NW, IC = IA + IB;
  constexpr int H = NS == 2 && NA > 2 ? (IC + 1) / 2 : IC;  // requests of a stage behind the barrier; the rest in the step before the next
  constexpr int UN = CH ? CH : NA;
  static_assert(!TURN || (!TWO && CH != 0));
  static_assert(UN % NA == 0 && (NS == 2 || UN % 2 == 0) && UN <= 8 && (CH != 0 || !TWO));
  static_assert(NO * PX * BM % (64 * NW) == 0 && NO * PW * BN % (64 * NW) == 0 && BM % 64 == 0 && BN % 64 == 0);
  __shared__ u4v As[NA][NO * PX * BM];
  __shared__ u4v Bs[NA][NO * PW * BN];
  __shared__ f4 Es[3][64];  // of the tile's columns: factors of the sums, bias, GELU's powers

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int half = lane >> 5, l32 = lane & 31;
  const int tiles_m = (a.M + BM - 1) / BM, tiles_n = (a.N + BN - 1) / BN;
  int tile;
  {
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
    const int per_xcd = ((int)gridDim.x + 7) >> 3;
    tile = xcd * per_xcd + slot;
  }
  if (tile >= tiles_m * tiles_n) return;
  int tm, tn;
  tile_coords(tile, tiles_m, tiles_n, a.band_rows, &tm, &tn);
  const int m0 = tm * BM, n0 = tn * BN;
  const int mp = cut_rows(a.M);

  const int T_all = a.K / KT;
  const int kt0 = SPLIT ? (int)(((long)blockIdx.y * T_all) / gridDim.y) : 0;
  const int kt1 = SPLIT ? (int)(((long)(blockIdx.y + 1) * T_all) / gridDim.y) : T_all;
  const int T = kt1 - kt0;

  const int wplanes = planes_of<PW>(a), second = second_plane<PW>(a, tm);
  unsigned aoff[IA], boff[IB];
#pragma unroll
  for (int i = 0; i < IA; ++i) {
    const int at = (wave * IA + i) * 64, plane = at / BM, row = at % BM + lane;
    aoff[i] = ((unsigned)plane * (unsigned)mp + (unsigned)min(m0 + row, a.M - 1)) * 16u;
  }
#pragma unroll
  for (int i = 0; i < IB; ++i) {
    const int at = (wave * IB + i) * 64, part = at / BN % PW, row = at % BN + lane;
    const int plane = at / BN / PW * wplanes + (part == 1 ? second : part);
    boff[i] = ((unsigned)plane * (unsigned)a.N + (unsigned)min(n0 + row, a.N - 1)) * 16u;
  }
  const size_t astage = (size_t)NO * PX * mp * 16, bstage = (size_t)NO * wplanes * a.N * 16;
  const char* Ab = reinterpret_cast<const char*>(a.A) + kt0 * astage;
  const char* Wb = static_cast<const char*>(a.w_half) + kt0 * bstage;
  const unsigned as_lds = (unsigned)(size_t)(lds_ptr)(void*)&As[0][0], bs_lds = (unsigned)(size_t)(lds_ptr)(void*)&Bs[0][0];
  // The i-th of a wavefront's requests for stage t, of which `an` and `bn` are the operands.
  auto request = [&](const char* an, const char* bn, int buf, int i) __attribute__((always_inline)) {
    if (i < IA) lds_dma16(an, aoff[i < IA ? i : 0], as_lds + (unsigned)(buf * NO * PX * BM * 16 + (wave * IA + i) * 1024));
    else lds_dma16(bn, boff[i < IA ? 0 : i - IA], bs_lds + (unsigned)(buf * NO * PW * BN * 16 + (wave * IB + i - IA) * 1024));
  };
  auto requests = [&](int t, int buf, int n) __attribute__((always_inline)) {
    const size_t k = (size_t)min(t, T - 1);
#pragma unroll
    for (int i = 0; i < n; ++i) request(Ab + k * astage, Wb + k * bstage, buf, i);
  };

  f16v acc[MB][NB], tot[CH ? MB : 1][CH ? NB : 1], low[TWO ? MB : 1][TWO ? NB : 1];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        acc[i][j][v] = 0.0f;
        if constexpr (CH != 0) tot[i][j][v] = 0.0f;
      }
  struct Ops { u4v x[MB][PX], w[NB][PW]; };
  constexpr int NR = PX * MB + PW * NB;
  auto read = [&](int buf, int s, Ops& o, int r) __attribute__((always_inline)) {  // the r-th, in the order in which the products need them
    int at = 0;
#pragma unroll
    for (int p = PX - 1; p >= 0; --p) {
#pragma unroll
      for (int i = 0; i < MB; ++i)
        if (at++ == r) o.x[i][p] = As[buf][((2 * s + half) * PX + p) * BM + (wm * MB + i) * 32 + l32];
      const int q = PX - 1 - p;
      if (q < PW) {
#pragma unroll
        for (int j = 0; j < NB; ++j)
          if (at++ == r) o.w[j][q] = Bs[buf][((2 * s + half) * PW + q) * BN + (wn * NB + j) * 32 + l32];
      }
    }
  };
  using P = Products<PX, PW>;
  constexpr int NP = P::n, NM = NP * MB * NB;
  auto multiply = [&](auto first, const Ops& cur, int f) __attribute__((always_inline)) {  // the f-th of a step
    constexpr bool fresh = CH != 0 && decltype(first)::value;
    const int p = f / (MB * NB), j = f / MB % NB, i = f % MB;
    f16v& sum = TWO && p < NP - 1 ? low[TWO ? i : 0][TWO ? j : 0] : acc[i][j];
    if (fresh && (p == 0 || (TWO && p == NP - 1))) {
#pragma unroll
      for (int v = 0; v < 16; ++v) sum[v] = 0.0f;
    }
    const u4v &w = cur.w[j][P::w[p]], &x = cur.x[i][P::x[p]];
    if constexpr (PX == 3)
      sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, w), __builtin_bit_cast(bf16x8, x), sum, 0, 0, 0);
    else
      sum = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8v, w), __builtin_bit_cast(h8v, x), sum, 0, 0, 0);
  };
  // A step: its matrix instructions, the reads of the next step's operands (step s of buffer buf) and requests FROM .. UPTO - 1 of a
  // wavefront for stage t, to buffer `to`, spread over one another: all
  // requests of a stage in one go behind the barrier keep every wavefront of a CU from its matrix instructions until the path to LDS
  // has taken them (32 KB a stage; single products 0 to 7 % longer; a prompt of 1000 against f32 rows 1600 wide, 48 layers, 13.28 ms
  // so and 13.03 spread, 32 prompts of 512 against bf16 rows 105.8 and 104.4).  With two buffers all of them stay behind the barrier:
  // later ones are late (1000 x 6400 x 1600 70.8 and 73.7 us).
  auto step = [&](auto turned, auto first, Ops& cur, Ops& nxt, int buf, int s, int t, int to, auto from, auto upto) __attribute__((always_inline)) {
    constexpr int FROM = decltype(from)::value, N = decltype(upto)::value - FROM, G = N > 0 ? N : NM;
    if constexpr (decltype(turned)::value) {  // (the sign bits of two f16 numbers)
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int p = 0; p < PW; ++p) cur.w[j][p] ^= 0x80008000u;
    }
    const size_t k = (size_t)min(t, T - 1);
    const char *an = Ab + k * astage, *bn = Wb + k * bstage;
#pragma unroll
    for (int g = 0; g < G; ++g) {
#pragma unroll
      for (int r = g * NR / G; r < (g + 1) * NR / G; ++r) read(buf, s, nxt, r);
#pragma unroll
      for (int f = g * NM / G; f < (g + 1) * NM / G; ++f) multiply(first, cur, f);
      __builtin_amdgcn_sched_barrier(0);
      if (N > 0) {
        request(an, bn, to, FROM + g);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };

  if (T > 0) {
    Ops pa, pb;
    // What the write-out needs of the columns is asked for first of all: by then it is there, and takes no registers.
    if (wave == 0) {
      const unsigned off = (unsigned)min(n0 + 4 * lane, a.N - 4) * 4u, es = (unsigned)(size_t)(lds_ptr)(void*)&Es[0][0];
      if constexpr (PX == 2) lds_dma16(a.w_half_mul, off, es);
      if (!SPLIT && a.bias) lds_dma16(a.bias, off, es + 1024);
      if constexpr (EPI == GEMM_GELU && PX == 2) lds_dma16(a.c_scale, off, es + 2048);
    }
#pragma unroll
    for (int t = 0; t < NA - 1; ++t) requests(t, t, IC);
    requests(NA - 1, NA - 1, H);
    vm_wait<(NA - 2) * IC + H>();
    asm volatile("s_barrier" ::: "memory");
#pragma unroll
    for (int r = 0; r < NR; ++r) read(0, 0, pa, r);
    auto stage = [&](auto turned, auto u, int t, Ops& p0, Ops& p1) __attribute__((always_inline)) {
      constexpr int U = decltype(u)::value, ab = U % NA, nb = (U + 1) % NA;
      const std::integral_constant<bool, U == 0> head;
      const std::false_type rest;
      const std::integral_constant<int, 0> none;
      const std::integral_constant<int, H> some;
      const std::integral_constant<int, IC> all;
      if constexpr (NS == 2) step(turned, head, p0, p1, ab, 1, t - 1 + NA, (U + NA - 1) % NA, some, all);
      vm_wait<(NA - 2) * IC>();
      __builtin_amdgcn_sched_barrier(0);
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (NS == 2) step(turned, rest, p1, p0, nb, 0, t + NA, ab, none, some);
      else step(turned, head, p0, p1, nb, 0, t + NA, ab, none, all);
    };
    auto chain = [&](auto turned, int t) __attribute__((always_inline)) {
      auto at = [&](auto u) __attribute__((always_inline)) {
        constexpr int U = decltype(u)::value;
        if (t + U < T) {
          if constexpr (NS == 2 || U % 2 == 0) stage(turned, u, t + U, pa, pb);
          else stage(turned, u, t + U, pb, pa);
        }
      };
      at(std::integral_constant<int, 0>());
      if constexpr (UN > 1) at(std::integral_constant<int, 1 % UN>());
      if constexpr (UN > 2) at(std::integral_constant<int, 2 % UN>());
      if constexpr (UN > 3) at(std::integral_constant<int, 3 % UN>());
      if constexpr (UN > 4) at(std::integral_constant<int, 4 % UN>());
      if constexpr (UN > 5) at(std::integral_constant<int, 5 % UN>());
      if constexpr (UN > 6) at(std::integral_constant<int, 6 % UN>());
      if constexpr (UN > 7) at(std::integral_constant<int, 7 % UN>());
      if constexpr (CH != 0) {
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
          for (int i = 0; i < MB; ++i) {
            if constexpr (TWO) acc[i][j] += low[TWO ? i : 0][TWO ? j : 0];
            if constexpr (decltype(turned)::value) tot[CH ? i : 0][CH ? j : 0] -= acc[i][j];
            else tot[CH ? i : 0][CH ? j : 0] += acc[i][j];
          }
      }
    };
    for (int t = 0; t < T; t += UN) {
      chain(std::false_type(), t);
      if constexpr (TURN) {
        t += UN;
        if (t < T) chain(std::true_type(), t);
      }
    }
    vm_wait<0>();
  }
  // lane: row m of C; value v: column 8 (v / 4) + 4 half + v % 4
#pragma unroll
  for (int j = 0; j < NB; ++j)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int n = n0 + (wn * NB + j) * 32 + 8 * g + 4 * half;
      if (n >= a.N) continue;
      const int e4 = (n - n0) / 4;
      f4 mul = f4{1.f, 1.f, 1.f, 1.f};
      if constexpr (PX == 2) mul = Es[0][e4] * a.a_unscale;
      f4 bias = f4{0.f, 0.f, 0.f, 0.f};
      if (!SPLIT && a.bias) bias = Es[1][e4];
      f4 scale = f4{1.f, 1.f, 1.f, 1.f};
      if constexpr (EPI == GEMM_GELU && PX == 2) scale = Es[2][e4];
#pragma unroll
      for (int i = 0; i < MB; ++i) {
        const int m = m0 + (wm * MB + i) * 32 + l32;
        if (m >= a.M) continue;
        f4 c;
#pragma unroll
        for (int e = 0; e < 4; ++e) c[e] = CH ? tot[CH ? i : 0][CH ? j : 0][4 * g + e] : acc[i][j][4 * g + e];
        c *= mul;
        if constexpr (SPLIT != 0) {
          *reinterpret_cast<f4*>(a.ws + ((size_t)blockIdx.y * a.M + m) * a.N + n) = c;
          continue;
        }
        if constexpr (EPI == GEMM_GELU) {
          store_gelu<PX>(a.C, mp, (size_t)m, (size_t)n, c, bias, scale);
          continue;
        }
        c += bias;
        if (EPI == GEMM_RESID) c += *reinterpret_cast<const f4*>(a.resid + (size_t)m * a.ldc + n);
        *reinterpret_cast<f4*>(a.C + (size_t)m * a.ldc + n) = c;
      }
    }
}

// ---- some tens to some hundreds of rows --------------------------------------------------------
// A block owns 16 MT input rows and up to 16 NG rows of W (a.rows_per_block of them, a multiple of eight); its
// eight wavefronts take the steps of 32 columns in turn, operands from L2 straight to registers, and the eight partial tiles
// are added through LDS.  gridDim.y > 1: K is cut over blocks as well, raw tiles go to a.ws[part][M][N].  As k_gemm_cut_rows
// (pg_gemm_rows.hip), with rows of W that need no turn through LDS and no cut, and in half form 4 bytes per input value for 6.
// PX = PW = 3: both operands in cut form, on the bf16 cores: 1024 x 2304 x 768, us, 28.4 there, 24.9 here (48 rows of W a block).
template <int EPI, int PX, int PW, int MT, int NG>
__global__ __launch_bounds__(512) void k_gemm_half_rows(GemmArgs a) {
  constexpr int CSTR = 16 * NG + 4;  // row stride of the partial tile, floats
  constexpr int PD = MT * NG * 8 + 8 * (NG * PW + MT * PX) <= (PX == 3 ? 140 : 184) ? 2 : 1;  // steps requested ahead
  __shared__ __attribute__((aligned(16))) float slab[8][16 * MT * CSTR];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int i16 = lane & 15, kq = lane >> 4;
  const int part = (int)blockIdx.y, parts = (int)gridDim.y;
  const int n0 = (int)blockIdx.x * a.rows_per_block, n1 = min(n0 + a.rows_per_block, a.N);
  const int m0 = (int)blockIdx.z * 16 * MT;
  const int mp = cut_rows(a.M);
  const int piece = part * 8 + wave, pieces = parts * 8;
  const int steps_all = a.K / 32;
  const int steps = piece < steps_all ? (steps_all - piece + pieces - 1) / pieces : 0;

  const int wplanes = planes_of<PW>(a), second = second_plane<PW>(a, (int)blockIdx.z);
  const char* wp[NG];
#pragma unroll
  for (int g = 0; g < NG; ++g)
    wp[g] = static_cast<const char*>(a.w_half) + ((size_t)kq * wplanes * a.N + min(n0 + 16 * g + i16, n1 - 1)) * 16;
  const char* xp[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
    xp[mt] = reinterpret_cast<const char*>(a.A) + ((size_t)kq * PX * mp + min(m0 + 16 * mt + i16, a.M - 1)) * 16;
  const size_t wpart = (size_t)a.N * 16, wstep = wpart * 4 * wplanes, xpart = (size_t)mp * 16, xstep = xpart * 4 * PX;

  // The write-out takes four columns of a row at a time, neighbouring lanes neighbouring columns, or, into a matrix
  // in half form, neighbouring rows, which lie next to each other there.  What it adds is requested first.
  constexpr int ITEMS = 16 * MT * 4 * NG;
  constexpr int IPT = (ITEMS + 511) / 512;
  const bool c_half = EPI == GEMM_GELU;
  auto row_of = [&](int idx) { return c_half ? idx % (16 * MT) : idx / (4 * NG); };
  auto col_of = [&](int idx) { return 4 * (c_half ? idx / (16 * MT) : idx % (4 * NG)); };
  f4 ebias[IPT], eres[IPT], emul[IPT];
#pragma unroll
  for (int q = 0; q < IPT; ++q) {
    const int idx = tid + 512 * q, m = m0 + row_of(idx), n = n0 + col_of(idx);
    const bool live = idx < ITEMS && m < a.M && n < n1;
    ebias[q] = eres[q] = emul[q] = f4{0.f, 0.f, 0.f, 0.f};
    if (PX == 2 && live) emul[q] = *reinterpret_cast<const f4*>(a.w_half_mul + n) * a.a_unscale;
    if (parts > 1) continue;
    if (live && a.bias) ebias[q] = *reinterpret_cast<const f4*>(a.bias + n);
    if (live && EPI == GEMM_RESID) eres[q] = *reinterpret_cast<const f4*>(a.resid + (size_t)m * a.ldc + n);
  }

  f4 tot[MT][NG];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int g = 0; g < NG; ++g) tot[mt][g] = f4{0.f, 0.f, 0.f, 0.f};

  u4v rw[PD][NG][PW], rx[PD][MT][PX];
  auto load_step = [&](int s, u4v (&w)[NG][PW], u4v (&x)[MT][PX]) {
    const size_t col = (size_t)piece + (size_t)pieces * min(s, steps - 1);
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int p = 0; p < PW; ++p) w[g][p] = *reinterpret_cast<const u4v*>(wp[g] + col * wstep + (p == 1 ? second : p) * wpart);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int p = 0; p < PX; ++p) x[mt][p] = *reinterpret_cast<const u4v*>(xp[mt] + col * xstep + p * xpart);
  };
  auto mul_step = [&](const u4v (&w)[NG][PW], const u4v (&x)[MT][PX]) {
    // a chain of matrix instructions is a step, the small products one of their own; each product over a row of tiles before
    // the next
    auto one = [](const u4v& x, const u4v& w, const f4& c) {
      if constexpr (PX == 3) return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, x), __builtin_bit_cast(bf16x8, w), c, 0, 0, 0);
      else return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8v, x), __builtin_bit_cast(h8v, w), c, 0, 0, 0);
    };
    using P = Products<PX, PW>;
    const f4 zero{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      f4 c[NG], big[NG];
#pragma unroll
      for (int p = 0; p < P::n - 1; ++p)
#pragma unroll
        for (int g = 0; g < NG; ++g) c[g] = one(x[mt][P::x[p]], w[g][P::w[p]], p ? c[g] : zero);
#pragma unroll
      for (int g = 0; g < NG; ++g) big[g] = one(x[mt][0], w[g][0], zero);
#pragma unroll
      for (int g = 0; g < NG; ++g) tot[mt][g] += big[g] + c[g];
    }
  };
  if (steps > 0) {
#pragma unroll
    for (int i = 0; i < PD; ++i) load_step(i, rw[i], rx[i]);
    int s = 0;
    for (; s + 2 * PD <= steps; s += PD) {
#pragma unroll
      for (int i = 0; i < PD; ++i) {
        mul_step(rw[i], rx[i]);
        load_step(s + i + PD, rw[i], rx[i]);
      }
    }
#pragma unroll
    for (int i = 0; i < PD; ++i) {
      if (s + i < steps) mul_step(rw[i], rx[i]);
      if (s + i + PD < steps) load_step(s + i + PD, rw[i], rx[i]);
    }
#pragma unroll
    for (int i = 0; i < PD; ++i)
      if (s + PD + i < steps) mul_step(rw[i], rx[i]);
  }
  // (GELU's column powers: over the loop there are no registers for them)
  if constexpr (EPI == GEMM_GELU && PX == 2) {
#pragma unroll
    for (int q = 0; q < IPT; ++q) {
      const int idx = tid + 512 * q, n = n0 + col_of(idx);
      if (idx < ITEMS && n < n1) eres[q] = *reinterpret_cast<const f4*>(a.c_scale + n);
    }
  }
  // tot[mt][g][r] is row 16 mt + 4 kq + r, column 16 g + i16
  float* mine = slab[wave];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        mine[(16 * mt + 4 * kq + r) * CSTR + 16 * g + i16] = tot[mt][g][r];
  __syncthreads();
#pragma unroll
  for (int q = 0; q < IPT; ++q) {
    const int idx = tid + 512 * q, mr = row_of(idx), nl = col_of(idx);
    const int m = m0 + mr, n = n0 + nl;
    if (idx >= ITEMS || m >= a.M || n >= n1) continue;
    f4 w8[8];
#pragma unroll
    for (int w = 0; w < 8; ++w) w8[w] = *reinterpret_cast<const f4*>(slab[w] + mr * CSTR + nl);
    const f4 sum = (((w8[0] + w8[1]) + (w8[2] + w8[3])) + ((w8[4] + w8[5]) + (w8[6] + w8[7]))) * (PX == 2 ? emul[q] : f4{1.f, 1.f, 1.f, 1.f});
    if (parts > 1) {
      *reinterpret_cast<f4*>(a.ws + ((size_t)part * a.M + m) * a.N + n) = sum;
      continue;
    }
    if (EPI == GEMM_GELU) {
      store_gelu<PX>(a.C, mp, (size_t)m, (size_t)n, sum, ebias[q], eres[q]);
      continue;
    }
    f4 c = ebias[q] + sum;
    if (EPI == GEMM_RESID) c += eres[q];
    *reinterpret_cast<f4*>(a.C + (size_t)m * a.ldc + n) = c;
  }
}

// ---- norms -------------------------------------------------------------------------------------
// A norm's values are worked out past f32 where they are cut: half form drops a bit of a f32 value in four, 4.4 10^-8, as much as
// the roundings of (x - mean) / sigma g + b in f32 cost; so cut, they are as far off as f32 values were.
struct Norm {
  double mean, inv;
  __device__ __forceinline__ Norm(float sum, float squares, int n, float eps)
      : mean((double)sum / n) {
    const double v = (double)squares / n + (double)eps;
    const double y = (double)(1.0f / sqrtf((float)v));
    // (one Newton step of the root; squares that are past f32 leave 0, as they do in f32)
    inv = v < (double)INFINITY ? y * (1.5 - 0.5 * v * y * y) : y;
  }
  // four columns of a row, part by part `stride` bytes apart: half form (PX 2), times scale, or cut form (3)
  template <int PX>
  __device__ __forceinline__ void store(char* at, size_t stride, f4 c, f4 g, f4 b, float scale) const {
    double o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = ((double)c[e] - mean) * inv * (double)g[e] + (double)b[e];
    unsigned ab[3], cd[3];
    if constexpr (PX == 2) {
      halves2(o[0] * (double)scale, o[1] * (double)scale, ab[0], ab[1]);
      halves2(o[2] * (double)scale, o[3] * (double)scale, cd[0], cd[1]);
    } else {
      cut_safe2((float)o[0], (float)o[1], ab);
      cut_safe2((float)o[2], (float)o[3], cd);
    }
#pragma unroll
    for (int p = 0; p < PX; ++p) *reinterpret_cast<u2v*>(at + p * stride) = u2v{ab[p], cd[p]};
  }
};
// Rows of N values to LayerNorm in half form (layer_norm_in_place, cpu.rs:119-143: mean, biased variance in a second pass,
// eps inside the root), a wavefront a row, four rows a block: the 16-byte pieces of four rows lie next to each other in half
// form, and the block writes them so, through LDS.  PARTS: the row is first put together from the parts of a cut K, bias and
// residual, and written to a.C; otherwise it is read from there.  NQ: 256 NQ >= N.
// Pairs of blocks whose rows share cache lines are on one XCD (block % 8).
template <int NQ, bool PARTS, int PX>
__global__ __launch_bounds__(256) void k_norm_rows_half(GemmArgs a, int parts) {
  extern __shared__ __attribute__((aligned(16))) char staged[];
  constexpr int OSTR = PX * 4 * 16 + 16;  // an octet of columns: its parts, four rows; padded
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int b = (int)blockIdx.x / 16 * 16 + (int)blockIdx.x % 8 * 2 + (int)blockIdx.x % 16 / 8;
  const int m0 = 4 * b, m = min(m0 + wave, a.M - 1), n4 = a.N / 4;
  if (m0 >= a.M) return;
  f4 c[NQ], g[NQ], sh[NQ];
  auto col = [&](int q) { return 4 * (size_t)min(lane + 64 * q, n4 - 1); };
#pragma unroll
  for (int q = 0; q < NQ; ++q) c[q] = *reinterpret_cast<const f4*>((PARTS ? a.resid : a.C) + (size_t)m * a.ldc + col(q));
  if constexpr (PARTS) {
    f4 s[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) s[q] = *reinterpret_cast<const f4*>(a.ws + (size_t)m * a.N + col(q));
    for (int p = 1; p < parts; ++p)
#pragma unroll
      for (int q = 0; q < NQ; ++q) s[q] += *reinterpret_cast<const f4*>(a.ws + ((size_t)p * a.M + m) * a.N + col(q));
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      if (a.bias) s[q] = *reinterpret_cast<const f4*>(a.bias + col(q)) + s[q];
      c[q] = c[q] + s[q];
    }
  }
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    g[q] = *reinterpret_cast<const f4*>(a.ln_g + col(q));
    sh[q] = *reinterpret_cast<const f4*>(a.ln_b + col(q));
  }
  float sum = 0.0f;
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    const bool live = lane + 64 * q < n4;
    if (PARTS && live && m0 + wave < a.M) *reinterpret_cast<f4*>(a.C + (size_t)m * a.ldc + col(q)) = c[q];
    if (live) sum += (c[q].x + c[q].y) + (c[q].z + c[q].w);
  }
  sum = wave_sum(sum);
  const float mean = sum / (float)a.N;
  float var = 0.0f;
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    const f4 d = c[q] - mean;
    if (lane + 64 * q < n4) var += (d.x * d.x + d.y * d.y) + (d.z * d.z + d.w * d.w);
  }
  const Norm norm(sum, wave_sum(var), a.N, a.ln_eps);
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    const int i = lane + 64 * q;
    if (i >= n4) continue;
    char* at = staged + (i >> 1) * OSTR + wave * 16 + (i & 1) * 8;
    norm.store<PX>(at, 64, c[q], g[q], sh[q], a.ln_scale);
  }
  __syncthreads();
  const int mp = cut_rows(a.M);
  for (int i = threadIdx.x; i < a.N / 2 * PX; i += 256) {  // (octet, part, row)
    const int row = i & 3;
    if (m0 + row >= a.M) continue;
    *reinterpret_cast<u4v*>(reinterpret_cast<char*>(a.ln_out) + ((size_t)(i >> 2) * mp + m0 + row) * 16) =
        *reinterpret_cast<const u4v*>(staged + i / (4 * PX) * OSTR + i % (4 * PX) * 16);
  }
}

// The same, a block a row, for few rows: everything a thread reads is requested before the first use.  Eight rows share cache
// lines: their blocks are on one XCD (block % 8), whose L2 then writes whole lines back.  NQ: 1024 NQ >= N.
template <int NQ, bool PARTS, int PX, typename Next = Nothing>
__global__ __launch_bounds__(256) void k_norm_row_half(GemmArgs a, int parts, Next next) {
  __shared__ float red[2][4];
  if constexpr (std::is_same_v<Next, Ahead>) {
    if ((int)blockIdx.x >= (a.M + 63) / 64 * 64) {
      read_ahead(next, (int)blockIdx.x - (a.M + 63) / 64 * 64, blockIdx.x, 256);
      return;
    }
  }
  const int m = (int)blockIdx.x / 64 * 64 + (int)blockIdx.x % 8 * 8 + (int)blockIdx.x % 64 / 8;
  if (m >= a.M) return;
  const int n4 = a.N / 4;
  auto col = [&](int q) { return 4 * (size_t)min((int)threadIdx.x + 256 * q, n4 - 1); };
  auto bsum = [&](float v, float (&r)[4]) {
    v = wave_sum(v);
    if ((threadIdx.x & 63) == 0) r[threadIdx.x >> 6] = v;
    __syncthreads();
    return (r[0] + r[1]) + (r[2] + r[3]);
  };
  f4 c[NQ], v[NQ][PARTS ? 8 : 1], bias[NQ], g[NQ], sh[NQ];
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    if constexpr (PARTS) {
#pragma unroll
      for (int p = 0; p < 8; ++p) v[q][p] = *reinterpret_cast<const f4*>(a.ws + ((size_t)min(p, parts - 1) * a.M + m) * a.N + col(q));
      bias[q] = a.bias ? *reinterpret_cast<const f4*>(a.bias + col(q)) : f4{0.f, 0.f, 0.f, 0.f};
    }
    c[q] = *reinterpret_cast<const f4*>((PARTS ? a.resid : a.C) + (size_t)m * a.ldc + col(q));
    g[q] = *reinterpret_cast<const f4*>(a.ln_g + col(q));
    sh[q] = *reinterpret_cast<const f4*>(a.ln_b + col(q));
  }
  float sum = 0.0f;
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    const bool live = (int)threadIdx.x + 256 * q < n4;
    if constexpr (PARTS) {
      f4 t = v[q][0];
#pragma unroll
      for (int p = 1; p < 8; ++p)
        if (p < parts) t += v[q][p];
      c[q] += bias[q] + t;
      if (live) *reinterpret_cast<f4*>(a.C + (size_t)m * a.ldc + col(q)) = c[q];
    }
    if (live) sum += (c[q].x + c[q].y) + (c[q].z + c[q].w);
  }
  sum = bsum(sum, red[0]);
  const float mean = sum / (float)a.N;
  float var = 0.0f;
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    const f4 d = c[q] - mean;
    if ((int)threadIdx.x + 256 * q < n4) var += (d.x * d.x + d.y * d.y) + (d.z * d.z + d.w * d.w);
  }
  const Norm norm(sum, bsum(var, red[1]), a.N, a.ln_eps);
  const size_t mp = cut_rows(a.M);
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    if ((int)threadIdx.x + 256 * q >= n4) continue;
    const size_t k = col(q);
    char* at = reinterpret_cast<char*>(a.ln_out) + (k >> 3) * PX * mp * 16 + (size_t)m * 16 + (k & 4) * 2;
    norm.store<PX>(at, mp * 16, c[q], g[q], sh[q], a.ln_scale);
  }
}

constexpr int kNormRowMax = 256;  // rows up to which a block takes one
template <bool PARTS, int PX>
hipError_t launch_norm(const GemmArgs& a, int parts, hipStream_t s) {
  if (a.N % 8 != 0 || a.N > kNormWidest || a.ldc != a.N) return hipErrorInvalidValue;
  if (a.M <= kNormRowMax) {
    const dim3 rows((unsigned)((a.M + 63) / 64 * 64));
    if constexpr (PARTS && PX == 2) {
      if (a.ahead && a.ahead->blocks > 0 && a.N > 1024 && a.N <= 2048) {  // (narrower models have too few bytes to read ahead here)
        hipLaunchKernelGGL((k_norm_row_half<2, PARTS, PX, Ahead>), dim3(rows.x + a.ahead->blocks), dim3(256), 0, s, a, parts, *a.ahead);
        return hipGetLastError();
      }
    }
    if (a.N <= 1024) hipLaunchKernelGGL((k_norm_row_half<1, PARTS, PX>), rows, dim3(256), 0, s, a, parts, Nothing{});
    else if (a.N <= 2048) hipLaunchKernelGGL((k_norm_row_half<2, PARTS, PX>), rows, dim3(256), 0, s, a, parts, Nothing{});
    else hipLaunchKernelGGL((k_norm_row_half<4, PARTS, PX>), rows, dim3(256), 0, s, a, parts, Nothing{});
    return hipGetLastError();
  }
  const dim3 grid((unsigned)((a.M + 63) / 64 * 16));
  const size_t lds = (size_t)a.N / 8 * (PX * 4 * 16 + 16);
  if (a.N <= 768) hipLaunchKernelGGL((k_norm_rows_half<3, PARTS, PX>), grid, dim3(256), lds, s, a, parts);
  else if (a.N <= 1280) hipLaunchKernelGGL((k_norm_rows_half<5, PARTS, PX>), grid, dim3(256), lds, s, a, parts);
  else if (a.N <= 1792) hipLaunchKernelGGL((k_norm_rows_half<7, PARTS, PX>), grid, dim3(256), lds, s, a, parts);
  else {
    if (lds > 48 * 1024) {  // (from 2731 columns on in half form, 1891 in cut form)
      const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_norm_rows_half<16, PARTS, PX>),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL((k_norm_rows_half<16, PARTS, PX>), grid, dim3(256), lds, s, a, parts);
  }
  return hipGetLastError();
}
template <bool PARTS>
hipError_t launch_norm_rows(const GemmArgs& a, int parts, hipStream_t s) {
  return a.ln_scale > 0.0f ? launch_norm<PARTS, 2>(a, parts, s) : launch_norm<PARTS, 3>(a, parts, s);
}

// ---- weights -----------------------------------------------------------------------------------
// Rows of W as stored (WT as elsewhere: f32, bf16, int8 with their scales) to half form: part p of element (n, k) is the
// (k % 8)-th f16 of the 16 bytes at ((k / 8 * PW + p) * N + n) * 16, times mul[n]^-1: divided by the power of two that column k of the
// inputs is kept times (powers; null: 1), and its row scaled by the one that puts the largest between 2^14 and 2^15.  A bf16 weight is
// then a f16 number as it is down to 2^-32 of the row's largest and right to 2^-40 of that below, as a f32 weight's lo part is (of
// normally distributed weights one in 10^9 is as small: a large model has some).  *refused is set where a value is not finite or a row
// so small or large that its power of two, or an int8 row's scale beside it, would matter.
// A f32 weight in four lies half-way between two values of its second part.  Over the positions of a prompt that is the same error
// every time, and attention adds them up: behind prompts of 300 to 900 tokens the next token's logits were off by 1.02 to 1.04 times
// as much as with W whole, though each position's were off by less.  planes 3: the other of the two values is there as well, and
// every second block of input rows takes it.
template <int WT>
__global__ __launch_bounds__(256) void k_half_rows(const void* W, const float* scales, const float* powers, void* to, float* mul,
                                                   unsigned* refused, int N, int K, int planes) {
  __shared__ float biggest[4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int n = (int)blockIdx.x * 64 + lane, row = min(n, N - 1);
  auto get = [&](int k, float (&x)[8]) {  // columns k .. k + 7
    if constexpr (WT == 0) {
      const f4* w = reinterpret_cast<const f4*>(static_cast<const float*>(W) + (size_t)row * K + k);
      const f4 u = w[0], v = w[1];
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = u[e], x[4 + e] = v[e];
    } else if constexpr (WT == 1) {
      const u4v w = *reinterpret_cast<const u4v*>(static_cast<const unsigned short*>(W) + (size_t)row * K + k);
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = __uint_as_float(e & 1 ? w[e / 2] & 0xffff0000u : w[e / 2] << 16);
    } else {
      const u2v w = *reinterpret_cast<const u2v*>(static_cast<const signed char*>(W) + (size_t)row * K + k);
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = (float)((int)(w[e / 4] << (24 - 8 * (e % 4))) >> 24);
    }
    if (powers)
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] *= 1.0f / powers[k + e];
  };
  float x[8], most = 0.0f, row_scale = 1.0f;
  bool bad = false;
  for (int k = 8 * wave; k < K; k += 32) {
    get(k, x);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      bad |= !(fabsf(x[e]) < INFINITY);
      most = fmaxf(most, fabsf(x[e]));
    }
  }
  biggest[wave][lane] = most;
  __syncthreads();
  most = fmaxf(fmaxf(biggest[0][lane], biggest[1][lane]), fmaxf(biggest[2][lane], biggest[3][lane]));
  int top = 15;
  if (most > 0.0f && most < INFINITY) frexpf(most, &top);
  if constexpr (WT == 2) {
    row_scale = scales[row];
    int e = 0;
    if (most > 0.0f && row_scale != 0.0f) frexpf(row_scale, &e);
    bad |= !(fabsf(row_scale) < INFINITY) || abs(e) > kHalfMostExp;
  }
  bad |= most > 0.0f && abs(15 - top) > kHalfMostExp;
  const float scale = bad ? 1.0f : ldexpf(1.0f, 15 - top);
  if (wave == 0 && n < N) mul[n] = row_scale / scale;
  for (int k = 8 * wave; k < K; k += 32) {
    get(k, x);
    u4v h, l, other;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      unsigned hi, lo;
      halves2(x[2 * e], x[2 * e + 1], scale, hi, lo);
      h[e] = hi, l[e] = lo;
      if (WT == 0) {  // 2 (x - hi) - lo
        const h2v hv = __builtin_bit_cast(h2v, hi), lv = __builtin_bit_cast(h2v, lo);
        const float a = x[2 * e] * scale - (float)hv.x, b = x[2 * e + 1] * scale - (float)hv.y;
        const f2 o{fmaf(2.0f, a, -(float)lv.x), fmaf(2.0f, b, -(float)lv.y)};
        other[e] = __builtin_bit_cast(unsigned, __builtin_convertvector(o, h2v));
      }
    }
    if (n < N) {
      u4v* at = static_cast<u4v*>(to) + (size_t)(k / 8) * planes * N + n;
      at[0] = h;
      if (planes > 1) at[N] = l;
      if (planes > 2) at[2 * (size_t)N] = other;
    }
  }
  if (bad) atomicOr(refused, 1u);
}

// f32 rows to cut form, three bf16 numbers a weight, in the order of k_half_rows.
__global__ __launch_bounds__(256) void k_cut_weights(const float* W, void* to, int N, int K) {
  const int n = (int)blockIdx.x * 64 + (threadIdx.x & 63);
  if (n >= N) return;
  for (int k = 8 * (threadIdx.x >> 6); k < K; k += 32) {
    const f4* w = reinterpret_cast<const f4*>(W + (size_t)n * K + k);
    const Cut c = cut8(w[0], w[1]);
    u4v* at = static_cast<u4v*>(to) + (size_t)(k / 8) * 3 * N + n;
#pragma unroll
    for (int p = 0; p < 3; ++p) at[(size_t)p * N] = c.p[p];
  }
}

// The largest that an output of a projection behind a LayerNorm can be: the norm's values before scale and shift are at most
// sqrt(C) long together, so |W_o . (g z + b) + bias_o| <= sqrt(C) |W_o g| + |W_o . b + bias_o|, the second as fold has it
// (launch_ln_fold).
template <int WT>
__global__ __launch_bounds__(256) void k_half_bound(const void* W, const float* scales, const float* g, const float* fold,
                                                    float* bounds, int N, int K) {
  const int lane = threadIdx.x & 63, row = (int)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= N) return;
  float ss = 0.0f;
  for (int k = lane; k < K; k += 64) {
    const size_t at = (size_t)row * K + k;
    const float w = WT == 0   ? static_cast<const float*>(W)[at]
                    : WT == 1 ? __uint_as_float((unsigned)static_cast<const unsigned short*>(W)[at] << 16)
                              : (float)static_cast<const signed char*>(W)[at] * scales[row];
    ss = fmaf(w * g[k], w * g[k], ss);
  }
  ss = wave_sum(ss);
  if (lane == 0) bounds[row] = sqrtf(ss * (float)K) + fabsf(fold[2 * row + 1]);
}
// The exponent of the power of two that puts values up to `bound` at 2^15 at most; refused where it is out of bounds itself.
__device__ __forceinline__ int half_power(float bound, bool& refused) {
  int e = 15;  // (a bound of 0: a column of zeros)
  if (bound > 0.0f && bound < INFINITY) frexpf(bound, &e);
  refused |= !(bound < INFINITY) || abs(15 - e) > kHalfMostExp;  // (NaN too)
  return 15 - e;
}
__global__ __launch_bounds__(256) void k_half_powers(float* at, unsigned* refused, int n) {
  const int i = (int)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  bool bad = false;
  at[i] = ldexpf(1.0f, half_power(at[i], bad));
  if (bad) atomicOr(refused, 1u);
}
// The norm's own values, sqrt(C) |g_c| + |b_c| at most: their powers, and gains and shifts times them.
__global__ __launch_bounds__(256) void k_half_norm_powers(const float* g, const float* b, float* powers, float* g_out, float* b_out,
                                                          unsigned* refused, int C) {
  const int i = (int)blockIdx.x * 256 + threadIdx.x;
  if (i >= C) return;
  bool bad = false;
  const float p = ldexpf(1.0f, half_power(fabsf(g[i]) * sqrtf((float)C) + fabsf(b[i]), bad));
  powers[i] = p, g_out[i] = g[i] * p, b_out[i] = b[i] * p;
  if (bad) atomicOr(refused, 1u);
}
// Queries and keys, whose products over a head's 64 dims are added: the product of their powers is the same for all of a head's dims,
// score[h].  Queries take the whole range, keys of dim d as much of it as the largest product of d is of the head's largest.  A
// wavefront a head; q and k hold the bounds and get the powers.
__global__ __launch_bounds__(64) void k_half_score_powers(float* q, float* k, float* score, unsigned* refused) {
  const int h = (int)blockIdx.x, i = h * 64 + (int)threadIdx.x;
  const float bq = q[i], bk = k[i];
  bool bad = false;
  const int pq = half_power(bq, bad), pk = half_power(bk, bad);
  const bool counts = bq > 0.0f && bk > 0.0f;  // (otherwise the product is 0 whatever the powers are)
  __shared__ int least[64];
  least[threadIdx.x] = counts ? pq + pk : 1 << 20;
  __syncthreads();
  int both = 1 << 20;
  for (int j = 0; j < 64; ++j) both = min(both, least[j]);
  if (both == 1 << 20) both = 0;
  const int pk_of = counts ? both - pq : pk;
  bad |= abs(pk_of) > 2 * kHalfMostExp;
  q[i] = ldexpf(1.0f, pq), k[i] = ldexpf(1.0f, bad ? 0 : pk_of);
  if (threadIdx.x == 0) score[h] = ldexpf(1.0f, both);
  if (bad) atomicOr(refused, 1u);
}

// ---- launchers ---------------------------------------------------------------------------------
template <int WM, int WN, int MB, int NB, int PX, int PW, int OCC, int NA, int KT, int CH, bool TWO, bool TURN = false>
struct Shape {
  static constexpr int bm = 32 * MB * WM, bn = 32 * NB * WN;
  template <int EPI, int SPLIT>
  static hipError_t start(const GemmArgs& a0, int parts, hipStream_t s) {
    GemmArgs a = a0;
    const int tiles_m = (a.M + bm - 1) / bm, tiles_n = (a.N + bn - 1) / bn, tiles = tiles_m * tiles_n;
    a.band_rows = choose_band(tiles_m, std::max(1, (tiles + 7) / 8), bm, bn);
    const dim3 grid((unsigned)((tiles + 7) / 8 * 8), (unsigned)parts);  // whole rounds over the 8 XCDs
    hipLaunchKernelGGL((k_gemm_half<WM, WN, MB, NB, PX, PW, EPI, SPLIT, OCC, NA, KT, CH, TWO, TURN>), grid, dim3(64 * WM * WN), 0, s, a);
    return hipGetLastError();
  }
  static hipError_t launch(const GemmArgs& a, int epi, int parts, hipStream_t s) {
    if (parts > 1) return start<GEMM_BIAS, 1>(a, parts, s);
    switch (epi) {
      case GEMM_BIAS: return start<GEMM_BIAS, 0>(a, 1, s);
      case GEMM_GELU: return start<GEMM_GELU, 0>(a, 1, s);
      case GEMM_RESID: return start<GEMM_RESID, 0>(a, 1, s);
      default: return hipErrorInvalidValue;
    }
  }
};
hipError_t launch_tile(const GemmArgs& a, int epi, const HalfPlan& p, hipStream_t s) {
  if (a.w_half_parts == 3) {
    switch (p.tile) {
      case HALF_64x128: return Shape<2, 2, 1, 2, 3, 3, 2, 2, 32, 4, true>::launch(a, epi, p.parts, s);
      case HALF_128x128_8: return Shape<4, 2, 1, 2, 3, 3, 2, 3, 32, 3, true>::launch(a, epi, p.parts, s);
      default: return hipErrorInvalidValue;
    }
  }
  if (a.w_half_parts == 2) {
    switch (p.tile) {
      case HALF_64x128: return Shape<2, 2, 1, 2, 2, 2, 3, 2, 32, 4, true>::launch(a, epi, p.parts, s);
      case HALF_128x128: return Shape<2, 2, 2, 2, 2, 2, 2, 2, 32, 4, false, true>::launch(a, epi, p.parts, s);
      case HALF_128x128_8: return Shape<4, 2, 1, 2, 2, 2, 2, 4, 32, 4, true>::launch(a, epi, p.parts, s);
      default: return hipErrorInvalidValue;
    }
  }
  switch (p.tile) {
    case HALF_64x128: return Shape<2, 2, 1, 2, 2, 1, 3, 2, 32, 4, true>::launch(a, epi, p.parts, s);
    case HALF_128x128: return Shape<2, 2, 2, 2, 2, 1, 2, 3, 32, 3, false, true>::launch(a, epi, p.parts, s);
    case HALF_128x128_8: return Shape<4, 2, 1, 2, 2, 1, 2, 4, 32, 4, true>::launch(a, epi, p.parts, s);
    case HALF_128x256: return Shape<2, 2, 2, 4, 2, 1, 2, 4, 16, 0, false>::launch(a, epi, p.parts, s);
    case HALF_128x256_8: return Shape<2, 4, 2, 2, 2, 1, 2, 4, 32, 4, true>::launch(a, epi, p.parts, s);
    default: return hipErrorInvalidValue;
  }
}

template <int EPI, int PX, int PW>
hipError_t launch_rows_form(const GemmArgs& a, const HalfPlan& p, hipStream_t s) {
  const unsigned n_blocks = (unsigned)((a.N + a.rows_per_block - 1) / a.rows_per_block), m_blocks = (unsigned)((a.M + 16 * p.mt - 1) / (16 * p.mt));
  if (m_blocks > 65535u) return hipErrorInvalidValue;
  const dim3 grid(n_blocks, (unsigned)p.parts, m_blocks);
  const int ng = (p.rows + 15) / 16;
#define PG_CASE(MT, NG) \
  if (p.mt == MT && ng == NG) { hipLaunchKernelGGL((k_gemm_half_rows<EPI, PX, PW, MT, NG>), grid, dim3(512), 0, s, a); return hipGetLastError(); }
  PG_CASE(1, 1) PG_CASE(2, 1) PG_CASE(3, 1) PG_CASE(4, 1)
  PG_CASE(1, 2) PG_CASE(2, 2) PG_CASE(3, 2) PG_CASE(4, 2)
  PG_CASE(3, 3) PG_CASE(4, 3)
  if constexpr (PX == 2) { PG_CASE(3, 4) PG_CASE(4, 4) }
#undef PG_CASE
  return hipErrorInvalidValue;
}
template <int PX, int PW>
hipError_t launch_rows(const GemmArgs& a, int epi, const HalfPlan& p, hipStream_t s) {
  if (p.parts > 1) return launch_rows_form<GEMM_BIAS, PX, PW>(a, p, s);
  switch (epi) {
    case GEMM_BIAS: return launch_rows_form<GEMM_BIAS, PX, PW>(a, p, s);
    case GEMM_GELU: return launch_rows_form<GEMM_GELU, PX, PW>(a, p, s);
    case GEMM_RESID: return launch_rows_form<GEMM_RESID, PX, PW>(a, p, s);
    default: return hipErrorInvalidValue;
  }
}

// Time of a product in microseconds.  Tiles: a start, the stages of 32 columns at the pace of the CU with the most items (a stage
// alone, each further item, a partly filled round).  Blocks of rows: rounds of the blocks over the CUs, of a block's steps over
// its wavefronts, and what it costs that blocks of the same rows of W lie on several XCDs (a number of them that eight does not
// divide: 512 x 1280 x 1280 f32 rows, 48 rows of W 19.3 us, 40 rows 14.7).  And what is left to do behind it: the launch that adds
// the parts, with or without a norm, per part and value, or a norm by itself.  Constants of the least regret over the four
// projections of widths 512 to 1600 at 2 to 8192 rows, W from HBM (35000 plans; cut form widths 512 and 768, 33 to 1024 rows): the
// plan of least predicted time is 2 % (f32 rows 1.5 %, cut form 0.6 %) slower than the best measured one in the mean.
struct TilePace {
  float start, stage, more, part;
};
struct Finish {
  float reduce_norm, part, values_norm, reduce, values, norm, norm_values;
};
struct RowsPace {
  float start, turn, step, mt, ng, both, fill_mt, fill_ng, uneven;
};
// [half form of f32 rows, of bf16 and int8 rows, cut form][HalfTile]
constexpr TilePace kTilePace[3][3] = {
    {{5.981f, 0.546f, 0.074f, 0.197f}, {9.04f, 0.604f, 0.329f, 0.111f}, {7.24f, 0.503f, 11.3f, 2.426f}},
    {{5.243f, 0.389f, 0.027f, 0.13f}, {6.453f, 0.422f, 0.178f, 0.125f}, {5.701f, 0.36f, 1.06f, -0.021f}},
    {{3.39f, 0.667f, 0.426f, -0.051f}, {}, {3.014f, 0.924f, 0.685f, 0.149f}}};
// Products of half form with a tile of 128 x 128 for every CU or more: tiles only, and their times are fitted by themselves
// (160 products of widths 768 to 1600, 700 to 16384 rows; 4 to 10 % off, the choice 0.4 to 1.5 % slower than the best tile in the mean).
// HALF_128x256 is for bf16 rows and parts of K up to 2048 only.  Its one chain errs by 3.6 10^-7 at K = 1600 and 7.3 10^-7 at 6400, the chains
// of the eight wavefronts by 1.2 and 1.6 10^-7, at 1.12 to 1.24 of its time (16384 x 4800 x 1600 490 us for 412, x 1600 x 6400 644
// for 588).  With it the logits of int8 models' prompts of 2000 rows were off by 1.2 times as much as three bf16 parts are, those
// of bf16 models with it at K = 4096 too, without at 0.8.
struct FullPace {
  float start, stage, more, part, gelu;  // (gelu: of an item's write-out)
};
constexpr FullPace kFullPace[2][6] = {
    {{5.17f, 0.463f, 0.077f, 0.314f, 0.83f}, {7.13f, 0.602f, 0.388f, 0.319f, 2.21f}, {7.37f, 0.495f, 0.619f, 0.191f, 3.58f}, {}, {}, {}},
    {{5.01f, 0.39f, 0.01f, 0.259f, 1.06f}, {7.24f, 0.412f, 0.252f, 0.267f, 2.23f}, {7.15f, 0.348f, 0.426f, 0.184f, 3.41f},
     {9.13f, 0.629f, 0.61f, 0.247f, 5.74f}, {}, {9.64f, 0.592f, 0.836f, 0.234f, 5.8f}}};
constexpr Finish kFinish[3] = {{2.903f, 2.218f, 0.056f, 5.858f, -3.213f, 2.241f, 2.427f},
                               {4.686f, 1.352f, 0.859f, 18.205f, -0.462f, 3.567f, 1.958f},
                               {3.025f, 1.971f, 0.603f, 0.682f, 0.016f, 1.99f, 5.505f}};
constexpr RowsPace kRowsPace[3] = {{6.051f, 0.928f, -0.147f, 0.191f, 0.302f, 0.003f, -0.07f, 0.019f, 0.077f},
                                   {1.852f, 0.411f, -0.082f, 0.117f, 0.048f, 0.024f, 0.068f, 0.085f, 0.067f},
                                   {3.29f, 1.262f, 0.536f, 0.049f, -0.171f, 0.155f, -0.052f, -0.005f, 0.369f}};

}  // namespace

bool gemm_half_takes(const GemmArgs& a, int epi) {
  const uintptr_t at = reinterpret_cast<uintptr_t>(a.A) | reinterpret_cast<uintptr_t>(a.w_half) | reinterpret_cast<uintptr_t>(a.C) |
                       reinterpret_cast<uintptr_t>(a.w_half_mul) | reinterpret_cast<uintptr_t>(a.bias) |
                       reinterpret_cast<uintptr_t>(a.resid) | reinterpret_cast<uintptr_t>(a.ws) | reinterpret_cast<uintptr_t>(a.ln_out) |
                       reinterpret_cast<uintptr_t>(a.ln_g) | reinterpret_cast<uintptr_t>(a.ln_b);
  return a.w_half && (a.w_half_parts == 3 || (a.w_half_mul && (a.w_half_parts == 1 || (a.w_half_parts == 2 && (a.w_half_planes == 2 || a.w_half_planes == 3))))) && !(at & 15) && a.M >= 1 && a.M < (1 << 23) &&
         a.K >= 64 && a.K % 32 == 0 && a.N >= 64 && a.N % 8 == 0 && a.N < (1 << 24) && a.ldc % 4 == 0 && a.a_unscale > 0.0f &&
         (a.c_scale != nullptr) == (epi == GEMM_GELU && a.w_half_parts != 3) && !(reinterpret_cast<uintptr_t>(a.c_scale) & 15) &&
         (epi == GEMM_BIAS || epi == GEMM_GELU || epi == GEMM_RESID) && (epi != GEMM_GELU || a.ldc == a.N);
}

HalfPlan gemm_half_plan(const GemmArgs& a, int epi, int num_cus) {
  const int kind = a.w_half_parts == 1 ? 1 : a.w_half_parts == 2 ? 0 : 2;
  const int steps = a.K / 32, cus = num_cus;
  const float mn = (float)a.M * (float)a.N * 1e-6f;
  const int most = epi != GEMM_GELU && a.ws ? (int)std::min<size_t>(std::min(8, a.K / 256), a.ws_floats / ((size_t)a.M * a.N)) : 1;
  const Finish& f = kFinish[kind];
  auto finish = [&](int parts) {
    if (parts == 1) return a.ln_out ? f.norm + f.norm_values * mn : 0.0f;
    return (a.ln_out ? f.reduce_norm : f.reduce) + (f.part * (float)parts + (a.ln_out ? f.values_norm : f.values)) * mn;
  };
  HalfPlan best{HALF_128x128, 1, 0, 0};
  float best_us = INFINITY;
  auto take = [&](const HalfPlan& p, float us) {
    if (us < best_us) best = p, best_us = us;
  };
  // (many values: their bytes; 4000 x 1280 values in a norm by itself 10.8 us, with two parts 18.7, three 20.9)
  auto full_finish = [&](int parts) {
    if (parts == 1) return a.ln_out ? 2.0f + 1.65f * mn : 0.0f;
    return 1.0f + ((a.ln_out ? 2.3f : 1.3f) + 0.55f * (float)parts) * mn;
  };
  if (kind != 2 && (long)((a.M + 127) / 128) * ((a.N + 127) / 128) >= cus) {
    for (int t : {HALF_64x128, HALF_128x128, HALF_128x128_8, HALF_128x256, HALF_128x256_8}) {
      if (t >= HALF_128x256 && kind != 1) continue;
      const int bm = t == HALF_64x128 ? 64 : 128, bn = t >= HALF_128x256 ? 256 : 128;
      for (int parts = 1; parts <= std::max(1, most); ++parts) {
        if (t == HALF_128x256 && (a.w_scale || a.K > 2048 * parts)) continue;
        const long items = ((long)((a.M + bm - 1) / bm) * ((a.N + bn - 1) / bn) + 7) / 8 * 8 * parts;
        const float on_cu = (float)((items + cus - 1) / cus), round = std::max(0.0f, (float)items / (float)cus - 1.0f);
        const FullPace& p = kFullPace[kind][t];
        take({t, parts, 0, 0}, p.start + (float)((steps + parts - 1) / parts) * (p.stage + (on_cu - 1.0f) * p.more + round * p.part) +
                                (epi == GEMM_GELU ? on_cu * p.gelu : 0.0f) + full_finish(parts));
      }
    }
    return best;
  }
  for (int t : {HALF_64x128, HALF_128x128, HALF_128x128_8}) {
    if (t == HALF_128x128 && kind == 2) continue;
    const int bm = t == HALF_64x128 ? 64 : 128, bn = 128;
    const long tiles = (long)((a.M + bm - 1) / bm) * ((a.N + bn - 1) / bn);
    for (int parts = 1; parts <= std::max(1, most); ++parts) {
      const long items = (tiles + 7) / 8 * 8 * parts;  // (as many to each XCD as the fullest one has)
      const float on_cu = (float)((items + cus - 1) / cus), round = std::max(0.0f, (float)items / (float)cus - 1.0f);
      const TilePace& p = kTilePace[kind][t];
      take({t, parts, 0, 0}, p.start + (float)((steps + parts - 1) / parts) * (p.stage + (on_cu - 1.0f) * p.more + round * p.part) + finish(parts));
    }
  }
  const int groups = (a.M + 63) / 64, mt = ((a.M + groups - 1) / groups + 15) / 16;
  const int m_blocks = (a.M + 16 * mt - 1) / (16 * mt);
  const RowsPace& p = kRowsPace[kind];
  for (int parts = 1; parts <= std::max(1, most); ++parts)
    for (int rows = 8; rows <= (mt <= 2 ? 32 : kind == 2 ? 48 : 64); rows += 8) {
      const int ng = (rows + 15) / 16;
      const int n_blocks = (a.N + rows - 1) / rows;
      const long blocks = (long)n_blocks * m_blocks * parts;
      const float turns = (float)((blocks + cus - 1) / cus), fill = (float)blocks / (float)cus;
      const float rounds = (float)(((steps + parts - 1) / parts + 7) / 8);
      take({HALF_ROWS, parts, mt, rows},
           p.start + turns * (p.turn + rounds * (p.step + p.mt * mt + p.ng * ng + p.both * mt * ng)) +
               fill * rounds * (p.fill_mt * mt + p.fill_ng * ng + (n_blocks % 8 != 0 && m_blocks > 1 ? p.uneven : 0.0f)) + finish(parts));
    }
  return best;
}

hipError_t launch_gemm_half_plan(const GemmArgs& a0, int epi, const HalfPlan& p, hipStream_t s) {
  GemmArgs a = a0;
  if (!gemm_half_takes(a, epi) || p.parts < 1 || p.parts > 8) return hipErrorInvalidValue;
  if (p.parts > 1 && (epi == GEMM_GELU || !a.ws || a.K / 32 < p.parts || (size_t)p.parts * a.M * a.N > a.ws_floats)) return hipErrorInvalidValue;
  if (p.tile != HALF_ROWS) return launch_tile(a, epi, p, s);
  if (p.rows < 8 || p.rows % 8 != 0 || p.mt < 1) return hipErrorInvalidValue;
  a.rows_per_block = p.rows;
  return a.w_half_parts == 3 ? launch_rows<3, 3>(a, epi, p, s) : a.w_half_parts == 2 ? launch_rows<2, 2>(a, epi, p, s) : launch_rows<2, 1>(a, epi, p, s);
}

void gemm_half_ahead(const GemmArgs& a, int epi, int num_cus, int k, Ahead* to) {
  if (!a.w_half || a.w_half_parts != 1) return;
  const HalfPlan p = gemm_half_plan(a, epi, num_cus);
  if (p.tile == HALF_ROWS && a.M <= 16 * p.mt) to->matrix(k, a.w_half, a.K / 8, (size_t)a.N * 16, (size_t)p.rows * 16);
}

hipError_t launch_gemm_half(const GemmArgs& a, int epi, int num_cus, hipStream_t s) {
  if (!gemm_half_takes(a, epi)) return hipErrorInvalidValue;
  const HalfPlan p = gemm_half_plan(a, epi, num_cus);
  const hipError_t e = launch_gemm_half_plan(a, epi, p, s);
  return e != hipSuccess ? e : finish_gemm_half(a, epi, p, s);
}
hipError_t finish_gemm_half(const GemmArgs& a, int epi, const HalfPlan& p, hipStream_t s) {
  if (p.parts == 1 && !a.ln_out) return hipSuccess;
  if (!a.ln_out || (a.ln_scale == 0.0f && !a.ln_cut)) {  // (a norm of f32 rows: the logits' input)
    if (p.parts == 1) return launch_layer_norm_rows(a.C, a.ln_out, a.M, a.N, a.ln_g, a.ln_b, a.ln_eps, s, a.ln_packed ? FORM_PACKED32 : FORM_ROWS);
    bool ln_done = false;
    const hipError_t e = launch_splitk_reduce(a, epi, p.parts, s, &ln_done);
    return e != hipSuccess || !a.ln_out || ln_done ? e : hipErrorInvalidValue;
  }
  if (p.parts == 1) return launch_norm_rows<false>(a, 0, s);
  return epi == GEMM_RESID ? launch_norm_rows<true>(a, p.parts, s) : hipErrorInvalidValue;
}

hipError_t launch_norm_rows_half(float* src, void* dst, int rows, int cols, const float* g, const float* b, float eps, float scale,
                                 hipStream_t s, int parts, const float* ws, const float* bias, const float* resid) {
  GemmArgs a{};
  a.C = src; a.ln_out = static_cast<float*>(dst); a.M = rows; a.N = a.ldc = cols;
  a.ln_g = g; a.ln_b = b; a.ln_eps = eps; a.ln_scale = scale;
  if (parts < 0 || parts > 8 || rows < 1) return hipErrorInvalidValue;
  if (parts == 0) return launch_norm_rows<false>(a, 0, s);
  a.ws = const_cast<float*>(ws); a.bias = bias; a.resid = resid;
  return launch_norm_rows<true>(a, parts, s);
}

hipError_t launch_half_rows(const void* W, int w_bytes, const float* scales, const float* powers, size_t rows, int cols, void* to,
                            float* mul, unsigned* refused, hipStream_t s, int planes) {
  const dim3 grid((unsigned)((rows + 63) / 64));
  if (cols % 32 != 0 || rows > (1u << 24) || (w_bytes == 4 ? planes != 2 && planes != 3 : planes != 1)) return hipErrorInvalidValue;
  if (w_bytes == 4) hipLaunchKernelGGL(k_half_rows<0>, grid, dim3(256), 0, s, W, scales, powers, to, mul, refused, (int)rows, cols, planes);
  else if (w_bytes == 2) hipLaunchKernelGGL(k_half_rows<1>, grid, dim3(256), 0, s, W, scales, powers, to, mul, refused, (int)rows, cols, planes);
  else hipLaunchKernelGGL(k_half_rows<2>, grid, dim3(256), 0, s, W, scales, powers, to, mul, refused, (int)rows, cols, planes);
  return hipGetLastError();
}
hipError_t launch_cut_weights(const float* W, size_t rows, int cols, void* to, hipStream_t s) {
  if (cols % 32 != 0 || rows > (1u << 24)) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_cut_weights, dim3((unsigned)((rows + 63) / 64)), dim3(256), 0, s, W, to, (int)rows, cols);
  return hipGetLastError();
}
hipError_t launch_half_bound(const void* W, int w_bytes, const float* scales, const float* g, const float* fold, size_t rows, int cols,
                             float* bounds, hipStream_t s) {
  const dim3 grid((unsigned)((rows + 3) / 4));
  if (w_bytes == 4) hipLaunchKernelGGL(k_half_bound<0>, grid, dim3(256), 0, s, W, scales, g, fold, bounds, (int)rows, cols);
  else if (w_bytes == 2) hipLaunchKernelGGL(k_half_bound<1>, grid, dim3(256), 0, s, W, scales, g, fold, bounds, (int)rows, cols);
  else hipLaunchKernelGGL(k_half_bound<2>, grid, dim3(256), 0, s, W, scales, g, fold, bounds, (int)rows, cols);
  return hipGetLastError();
}
hipError_t launch_half_norm_powers(const float* g, const float* b, int cols, float* powers, float* g_out, float* b_out, unsigned* refused,
                                   hipStream_t s) {
  hipLaunchKernelGGL(k_half_norm_powers, dim3((unsigned)((cols + 255) / 256)), dim3(256), 0, s, g, b, powers, g_out, b_out, refused, cols);
  return hipGetLastError();
}
hipError_t launch_half_powers(float* at, int n, unsigned* refused, hipStream_t s) {
  hipLaunchKernelGGL(k_half_powers, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, at, refused, n);
  return hipGetLastError();
}
hipError_t launch_half_score_powers(float* q, float* k, int heads, float* score, unsigned* refused, hipStream_t s) {
  hipLaunchKernelGGL(k_half_score_powers, dim3((unsigned)heads), dim3(64), 0, s, q, k, score, refused);
  return hipGetLastError();
}

}  // namespace pgk
