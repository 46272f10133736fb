// Products of many rows on the bf16 matrix cores, with f32 inputs, f32 sums and W stored as f32, bf16 or
// int8 rows (transposed_dense_projection_into, src/models/cpu.rs:58-75; QuantizedRows, cpu.rs:26-56).
// Stack models' products and those of sampled streams, whose results do not change; the projections of GPT-2 models whose weights
// have a half form go through pg_gemm_half.hip otherwise.
//
// Every f32 operand is cut into three bf16 numbers whose sum is the value: hi = bf16(x), mid =
// bf16(x - hi), lo = bf16(x - hi - mid), rounded to nearest, every difference exact; lo holds all that is
// left of the 24 significant bits.  bf16 and int8 rows are bf16 numbers as they are (the scale of an int8 row
// multiplies the row's sum), so x w = hi w + mid w + lo w: three v_mfma_f32_32x32x16_bf16 with every product
// exact, sums in f32, where the f32 matrix cores take eight instructions of twice the duration.  For f32 rows
// both operands are cut and the six products down to hi lo, mid mid and lo hi are formed.  |mid| <= 2^-8 |x|
// and |lo| <= 2^-17 |x|, the same of w, so the three left out are at most 2^-24 of x w together, one
// rounding of the product to f32; over ordinary values they are of either sign.
//
// How the sums round: the instruction adds two groups of eight products to the accumulator one after the other
// and rounds to f32 each time; before that it cuts off products below 2^-24 of the group's largest, and downward
// the accumulator below the same and the group's sum below 2^-31 of the accumulator.  With all products of K in one
// register the small ones (mid, lo) cost as many roundings at the whole sum's size as hi hi does, the
// error has a mean (-8e-8 of the result at K = 1600), and rows that are alike get the same error from hi lo,
// which is a few units of the sum's last place: keys and values of a whole cache are off the same way,
// which attention does not average out (XL, logits behind 896 tokens: 5.8e-7 with f32-core products, 9.2e-7
// so).  Tiles that have the registers therefore keep two sums, hi hi (bf16 and int8 rows: hi w) and all that
// is smaller, added at the end (TWO): the same logits 4.1e-7; 895 x 4800 x 1600 against f64 2.4e-7 of the
// result for f32 rows (one sum 6.2e-7, f32 cores 7.1e-7) and 2.4e-7 for bf16 rows (one sum 4.3e-7).  The
// 128 x 256 tile has no room for a second sum, and where there are more than two 128 x 128 tiles to a CU the third
// one there is worth more: 4.3e-7, as such products always had.
//
// What bounds it: in large products the clock goes down to 1.9 to 2.1 GHz with the matrix cores at work (a plain bf16
// product of the library reaches 1354 of 2500 TFLOP/s on this card), and what else the CU moves is paid
// for in clock as well as in time; the matrix cores are busy for 0.64 to 0.71 of the clocks in which a CU is, the rest is
// waits and VALU work that no MFMA covers.  In small ones (one tile on 144 to 240 of 256 CUs, 0.44 to 0.49) the clock stays
// and a tile's start and end count.  So the inputs travel as stored: f32 rows of A go straight to LDS
// (global_load_lds, no registers, no VALU), as do bf16 rows of W; a wavefront owns whole rows of the tile and
// cuts its A operands itself, in registers, once for all columns it owns; W, which every wavefront needs,
// is cut once on its way to LDS.  Against the form that cut A for the whole block and kept its planes in
// LDS (128 x 128 tiles, 2 x 2 wavefronts) that is a quarter of the LDS reads and half the VALU
// instructions per MFMA: 8192 x 4800 x 1600 bf16 488 -> 378 us, 8192 x 1600 x 6400 640 -> 470 us, int8
// 643 -> 508 us; f32, nine products -> six, 4096 x 6400 x 1600 680 -> 457 us (one box, W from HBM).
// The dot instruction that could take both subtractions of a cut (v_dot2_f32_bf16) runs on the matrix
// cores' time: 6 % slower.
#include "pg_gemm_dev.h"

#include <type_traits>

namespace pgk {

namespace {

// WM x WN wavefronts, each on MB x NB blocks of 32 x 32 (MFMA operand: lane (l, half) holds columns
// 8 half .. 8 half + 7 of row l; result: lane column l, value v row 8 (v / 4) + 4 half + v % 4).
// K runs in stages of 32 columns (16 for f32 rows), a stage in steps of 16.  While the MFMAs of a step run, the
// operands of the next one are read from LDS and cut, in the registers that the MFMAs have just freed; W of
// the stage after it is cut and stored; A and W further ahead are on their way (A in NA buffers).  One
// barrier per stage, in front of the step that reads the next stage: by then the wavefront has waited for
// its own share of that stage, and has read the stage before it to the end, whose buffer is free for the
// stage that is asked for next.  Every buffer has a fixed place in a turn of the loop, so that LDS
// addresses are constants (no VALU).
// SPLIT: the stages are cut into gridDim.y parts, raw partial tiles go to a.ws[part][M][N].
// GROUPED: see launch_gemm_grouped.  WT: W holds f32 (0), bf16 (1) or int8 rows with a.w_scale (2).
// OCC: wavefronts per SIMD that the registers are kept for.  TWO: small products have a sum of their own.
template <int WM, int WN, int MB, int NB, int WT, int EPI, int SPLIT, bool GROUPED, int OCC, int NA, bool TWO>
__global__ __launch_bounds__(64 * WM * WN, OCC) void k_gemm_cut(GemmArgs a) {
  constexpr int NW = WM * WN, BM = 32 * MB * WM, BN = 32 * NB * WN;
  constexpr int KT = WT == 0 ? 16 : 32, NS = KT / 16;
  constexpr int AP = KT / 4;                          // 16-byte pieces of a row of A in LDS
  constexpr int IA = BM * AP / 64 / NW;               // DMA instructions of A per wavefront and stage
  constexpr int IB = WT == 1 ? BN * 4 / 64 / NW : 0;  // the same of W where it is multiplied as stored
  constexpr int BLD = WT == 0 ? BN * 4 / (64 * NW) : WT == 2 ? BN * 2 / (64 * NW) : 0;  // else 16-byte loads per thread
  constexpr int UN = WT == 1 ? NA : 4;  // stages per turn of the loop: every buffer has a fixed place in it
  constexpr int RS = WT == 1 ? 1 : 4;   // sets of load registers
  constexpr int NPB = WT == 0 ? 3 : 1;  // planes of W in LDS
  constexpr int NBUF = WT == 1 ? NA : 2;
  constexpr int BP = WT == 0 ? 2 : 4;   // 16-byte pieces of a row of a plane
  static_assert(UN % 2 == 0 && UN % NA == 0 && UN <= 4);
  static_assert(IA >= 1 && BM * AP % (64 * NW) == 0);
  static_assert(WT == 1 ? IB >= 1 : BLD >= 1);
  __shared__ u4v As[NA][BM * AP];
  __shared__ u4v Bs[NBUF][NPB][BN * BP];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;
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
  const int group = GROUPED ? a.group_tile[tm] : 0;
  if (GROUPED && group < 0) return;

  const int T_all = a.K / KT;
  const int kt0 = SPLIT ? (int)(((long)blockIdx.y * T_all) / gridDim.y) : 0;
  const int kt1 = SPLIT ? (int)(((long)(blockIdx.y + 1) * T_all) / gridDim.y) : T_all;
  const int T = kt1 - kt0;
  const int half = lane >> 5, l32 = lane & 31;

  // DMA: the lane's piece of each instruction.  A row's pieces lie permuted (`turn`), so that the 16
  // lanes that an LDS read serves in one go, 16 rows at the same piece, are on different banks; the
  // permutation is in the address that a lane loads from, as the instruction stores lane after lane.
  unsigned aoff[GROUPED ? 1 : IA], boff[IB ? IB : 1];
  const char* arow[GROUPED ? IA : 1];  // (a grouped row lies anywhere in A, further than 32 bits reach)
#pragma unroll
  for (int i = 0; i < IA; ++i) {
    const int at = (wave * IA + i) * 64 + lane, row = at / AP, slot = at % AP;
    const int turn = KT == 32 ? (row >> 1) & 7 : (row >> 2) & 3;
    const unsigned piece = (unsigned)(slot ^ turn) * 16u;
    if constexpr (GROUPED) arow[i] = reinterpret_cast<const char*>(a.A + (size_t)group_row(a, m0 + row) * a.lda) + piece;
    else aoff[i] = (unsigned)(min(m0 + row, a.M - 1) - m0) * (unsigned)a.lda * 4u + piece;
  }
  constexpr int WBYTES = WT == 0 ? 4 : WT == 1 ? 2 : 1;
#pragma unroll
  for (int i = 0; i < IB; ++i) {
    const int at = (wave * IB + i) * 64 + lane, row = at / 4, slot = at % 4;
    const int piece = slot ^ ((row >> 2) & 3);
    boff[i] = (unsigned)(min(n0 + row, a.N - 1) - n0) * (unsigned)a.K * WBYTES + (unsigned)piece * 16u;
  }
  const char* Ab = reinterpret_cast<const char*>(a.A + (size_t)m0 * a.lda + (size_t)kt0 * KT);
  const char* Wb = reinterpret_cast<const char*>(a.W) +
                   (((size_t)n0 + (GROUPED ? (size_t)group * a.N : 0)) * a.K + (size_t)kt0 * KT) * WBYTES;
  const unsigned as_lds = (unsigned)(size_t)(lds_ptr)(void*)&As[0][0], bs_lds = (unsigned)(size_t)(lds_ptr)(void*)&Bs[0][0][0];
  auto dma = [&](int t, int buf) __attribute__((always_inline)) {
    const size_t k = (size_t)min(t, T - 1) * KT;
#pragma unroll
    for (int i = 0; i < IA; ++i) {
      const unsigned to = as_lds + (unsigned)(buf * BM * AP * 16 + (wave * IA + i) * 1024);
      if constexpr (GROUPED) lds_dma16_at(arow[i] + k * 4, to);
      else lds_dma16(Ab + k * 4, aoff[i], to);
    }
#pragma unroll
    for (int i = 0; i < IB; ++i)
      lds_dma16(Wb + k * WBYTES, boff[i], bs_lds + (unsigned)(buf * BN * BP * 16 + (wave * IB + i) * 1024));
  };
  // W through registers (f32 to be cut, int8 to be widened), asked for RS stages ahead
  struct Regs { u4v r[BLD ? BLD : 1]; };
  constexpr int LPR = WT == 0 ? 4 : 2;  // lanes per row
  const int lr = tid / LPR, lp = tid % LPR;
  unsigned roff[BLD ? BLD : 1];
#pragma unroll
  for (int i = 0; i < BLD; ++i)
    roff[i] = (unsigned)(min(n0 + lr + i * (64 * NW / LPR), a.N - 1) - n0) * (unsigned)a.K * WBYTES + (unsigned)lp * 16u;
  auto load_b = [&](int t, Regs& g) __attribute__((always_inline)) {
    const char* w = Wb + (size_t)min(t, T - 1) * (KT * WBYTES);
#pragma unroll
    for (int i = 0; i < BLD; ++i) g.r[i] = *reinterpret_cast<const u4v*>(w + roff[i]);
  };
  auto store_b = [&](int buf, const Regs& g) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < BLD; ++i) {
      const int row = lr + i * (64 * NW / LPR);
      if constexpr (WT == 0) {
        const f4 x = __builtin_bit_cast(f4, g.r[i]);
        unsigned h0, d0, l0, h1, d1, l1;
        cut2(x.x, x.y, h0, d0, l0);
        cut2(x.z, x.w, h1, d1, l1);
        const int piece = (lp >> 1) ^ (((row >> 2) ^ (row >> 3)) & 1);
        reinterpret_cast<u2v*>(&Bs[buf][0][row * BP + piece])[lp & 1] = u2v{h0, h1};
        reinterpret_cast<u2v*>(&Bs[buf][1 % NPB][row * BP + piece])[lp & 1] = u2v{d0, d1};
        reinterpret_cast<u2v*>(&Bs[buf][2 % NPB][row * BP + piece])[lp & 1] = u2v{l0, l1};
      } else if constexpr (WT == 2) {
        unsigned w[8];
#pragma unroll
        for (int d = 0; d < 4; ++d)
#pragma unroll
          for (int b = 0; b < 2; ++b)
            w[2 * d + b] = pk_bf16((float)((int)(g.r[i][d] << (24 - 16 * b)) >> 24), (float)((int)(g.r[i][d] << (16 - 16 * b)) >> 24));
        const int turn = (row >> 2) & 3;
        Bs[buf][0][row * BP + ((2 * lp) ^ turn)] = u4v{w[0], w[1], w[2], w[3]};
        Bs[buf][0][row * BP + ((2 * lp + 1) ^ turn)] = u4v{w[4], w[5], w[6], w[7]};
      }
    }
  };

  f16v acc[MB][NB], low[TWO ? MB : 1][TWO ? NB : 1];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        acc[i][j][v] = 0.0f;
        if constexpr (TWO) low[i][j][v] = 0.0f;
      }

  struct Raw { f4 x[MB][2]; };
  struct Planes { Cut c[MB]; };
  u4v bb[NPB][NB];
  auto read_a = [&](int buf, int s, Raw& r) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < MB; ++i) {
      const int row = (wm * MB + i) * 32 + l32;
      const int turn = KT == 32 ? (row >> 1) & 7 : (row >> 2) & 3;
      const int p = 4 * s + 2 * half;
      r.x[i][0] = __builtin_bit_cast(f4, As[buf][row * AP + (p ^ turn)]);
      r.x[i][1] = __builtin_bit_cast(f4, As[buf][row * AP + ((p + 1) ^ turn)]);
    }
  };
  auto read_b = [&](int buf, int s, int j) __attribute__((always_inline)) {
    const int row = (wn * NB + j) * 32 + l32;
    const int piece = WT == 0 ? half ^ (((row >> 2) ^ (row >> 3)) & 1) : (2 * s + half) ^ ((row >> 2) & 3);
#pragma unroll
    for (int pl = 0; pl < NPB; ++pl) bb[pl][j] = Bs[buf][pl][row * BP + piece];
  };
  constexpr int JG = MB == 1 ? 2 : 1;  // column blocks whose sums are taken in turn (a sum waits for its last MFMA)
  static_assert(NB % JG == 0);
  constexpr int NP = WT == 0 ? 6 : 3;
  // one 16-column step: MFMAs of the operands at hand; the next step's operands come in as the
  // registers get free
  auto step = [&](const Planes& cur, Planes& nxt, int abuf, int bbuf, int s) __attribute__((always_inline)) {
    Raw raw;
    read_a(abuf, s, raw);
#pragma unroll
    for (int jg = 0; jg < NB; jg += JG) {
#pragma unroll
      for (int p = 0; p < NP; ++p) {
        constexpr int kPA[6] = {2, 1, 0, 1, 0, 0}, kPB[6] = {0, 1, 2, 0, 1, 0};  // small terms first
        const int pa = WT == 0 ? kPA[p] : 2 - p, pb = WT == 0 ? kPB[p] : 0;
#pragma unroll
        for (int j = jg; j < jg + JG; ++j)
#pragma unroll
          for (int i = 0; i < MB; ++i) {
            f16v& sum = TWO && pa + pb > 0 ? low[TWO ? i : 0][TWO ? j : 0] : acc[i][j];
            sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, cur.c[i].p[pa]),
                                                         __builtin_bit_cast(bf16x8, bb[pb % NPB][j]), sum, 0, 0, 0);
          }
      }
#pragma unroll
      for (int j = jg; j < jg + JG; ++j) read_b(bbuf, s, j);
    }
#pragma unroll
    for (int i = 0; i < MB; ++i) nxt.c[i] = cut8(raw.x[i][0], raw.x[i][1]);
  };
  // the order of what a step does: an MFMA, and in its shadow a share of the other work
  auto interleave = [&](auto with_b) __attribute__((always_inline)) {
    constexpr bool wb = decltype(with_b)::value;
    constexpr int NM = NP * MB * NB;
    constexpr int NV = (MB * 46 + (wb ? BLD * (WT == 0 ? 26 : 32) : 0) + NM - 1) / NM + 1;
    constexpr int NR = (2 * MB + NPB * NB + NM - 1) / NM;
    __builtin_amdgcn_sched_group_barrier(0x100, 2 * MB, 0);
#pragma unroll
    for (int g = 0; g < NM; ++g) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, NR, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, NV, 0);
      if constexpr (wb) {
        __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  if (T > 0) {
    Planes pa, pb;
    Regs r[RS];
#pragma unroll
    for (int t = 0; t < NA; ++t) dma(t, t);
    if constexpr (WT != 1) {
#pragma unroll
      for (int t = 0; t < RS; ++t) load_b(t, r[t]);
      store_b(0, r[0]);
      load_b(RS, r[0]);
      store_b(1, r[1]);
      load_b(RS + 1, r[1]);
    }
    vm_wait<(WT == 1 ? (NA - 2) * (IA + IB) : RS * BLD)>();
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    {
      Raw raw;
      read_a(0, 0, raw);
#pragma unroll
      for (int j = 0; j < NB; ++j) read_b(0, 0, j);
#pragma unroll
      for (int i = 0; i < MB; ++i) pa.c[i] = cut8(raw.x[i][0], raw.x[i][1]);
    }
    const std::true_type yes;
    const std::false_type no;
    // stage t, t % UN == U
    auto stage = [&](auto u, int t, Planes& p0, Planes& p1) __attribute__((always_inline)) {
      constexpr int U = decltype(u)::value, ab = U % NA, nb = (U + 1) % NA, odd = U & 1;
      if constexpr (NS == 2) {
        step(p0, p1, ab, WT == 1 ? ab : odd, 1);
        interleave(no);
      }
      // stage t + 1 has landed once nothing but what was asked for after it is in flight
      vm_wait<(NA - 2) * (IA + IB) + (NA - 1) * BLD>();
      __builtin_amdgcn_sched_barrier(0);
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      dma(t + NA, ab);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (WT != 1) {
        store_b(odd, r[(U + 2) % RS]);
        load_b(t + 2 + RS, r[(U + 2) % RS]);
      }
      if constexpr (NS == 2) step(p1, p0, nb, WT == 1 ? nb : odd ^ 1, 0);
      else step(p0, p1, nb, odd ^ 1, 0);
      interleave(yes);
    };
    for (int t = 0; t < T; t += UN) {
      auto at = [&](auto u) __attribute__((always_inline)) {
        constexpr int U = decltype(u)::value;
        if (t + U < T) {
          if constexpr (NS == 2 || U % 2 == 0) stage(u, t + U, pa, pb);
          else stage(u, t + U, pb, pa);
        }
      };
      at(std::integral_constant<int, 0>());
      if (UN > 1) at(std::integral_constant<int, 1 % UN>());
      if constexpr (UN > 2) {
        at(std::integral_constant<int, 2 % UN>());
        at(std::integral_constant<int, 3 % UN>());
      }
    }
    vm_wait<0>();  // (nothing may land in LDS once the block has left it)
  }

  // an operand that is infinite, or becomes so when it is rounded to bf16, makes the sums it meets
  // NaN (inf - inf): the wavefront's tile once more in plain f32 arithmetic
  float bad = 0.0f;
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        if constexpr (TWO) acc[i][j][v] += low[i][j][v];
        bad = fmaf(acc[i][j][v], 0.0f, bad);
      }
  if (__any(bad != 0.0f)) {
    redo_tile<MB, NB, WT, EPI, SPLIT, GROUPED>(a, m0 + wm * 32 * MB, n0 + wn * 32 * NB, kt0 * KT, kt1 * KT,
                                               (int)blockIdx.y, (size_t)group * a.N);
    return;
  }
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const int n = n0 + (wn * NB + j) * 32 + l32;
      if (n >= a.N) continue;
      const float wscale = WT == 2 ? a.w_scale[n] : 1.0f;
      const float bias = !SPLIT && a.bias ? a.bias[n] : 0.0f;
      float* part = SPLIT ? a.ws + (size_t)blockIdx.y * a.M * a.N : nullptr;
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int m = m0 + (wm * MB + i) * 32 + 8 * (v >> 2) + 4 * half + (v & 3);
        if (m >= a.M) continue;
        float c = WT == 2 ? wscale * acc[i][j][v] : acc[i][j][v];
        if constexpr (SPLIT != 0) {
          part[(size_t)m * a.N + n] = c;
          continue;
        }
        c = bias + c;
        if constexpr (EPI == GEMM_SILU_PAIR) {
          store_silu_pair(a, m, n, c);
          continue;
        }
        if (EPI == GEMM_GELU) c = gelu_tanh(c);
        if (EPI == GEMM_SQRELU) c = sq_relu(c);
        if (kAddsResid<EPI>) c = a.resid[(size_t)m * a.ldc + n] + col_scaled<EPI>(a, n, c);
        a.C[(size_t)m * a.ldc + n] = c;
      }
    }
}

// ---- launchers ---------------------------------------------------------------------------------
template <int WM, int WN, int MB, int NB, int WT, int OCC, int NA, bool TWO>
struct Shape {
  static constexpr int bm = 32 * MB * WM, bn = 32 * NB * WN, threads = 64 * WM * WN;
  static GemmArgs numbered(const GemmArgs& a0, int* grid) {
    GemmArgs a = a0;
    const int tiles_m = (a.M + bm - 1) / bm, tiles_n = (a.N + bn - 1) / bn, tiles = tiles_m * tiles_n;
    a.band_rows = a.plan_band ? std::min(a.plan_band, tiles_m) : choose_band(tiles_m, std::max(1, (tiles + 7) / 8), bm, bn);
    *grid = (tiles + 7) / 8 * 8;  // whole rounds over the 8 XCDs
    return a;
  }
  template <int EPI, int SPLIT>
  static hipError_t start(const GemmArgs& a0, int parts, hipStream_t s) {
    int grid;
    const GemmArgs a = numbered(a0, &grid);
    hipLaunchKernelGGL((k_gemm_cut<WM, WN, MB, NB, WT, EPI, SPLIT, false, OCC, NA, TWO>), dim3(grid, parts), dim3(threads), 0, s, a);
    return hipGetLastError();
  }
  static hipError_t launch(const GemmArgs& a, int epi, int parts, hipStream_t s) {
    if (parts > 1) return start<GEMM_BIAS, 1>(a, parts, s);
    switch (epi) {
      case GEMM_BIAS: return start<GEMM_BIAS, 0>(a, 1, s);
      case GEMM_GELU: return start<GEMM_GELU, 0>(a, 1, s);
      case GEMM_RESID: return start<GEMM_RESID, 0>(a, 1, s);
      case GEMM_RESID_SCALED: return start<GEMM_RESID_SCALED, 0>(a, 1, s);
      case GEMM_SQRELU: return start<GEMM_SQRELU, 0>(a, 1, s);
      default: return hipErrorInvalidValue;
    }
  }
  static hipError_t launch_grouped(const GemmArgs& a0, int epi, hipStream_t s) {
    int grid;
    const GemmArgs a = numbered(a0, &grid);
    if (epi == GEMM_BIAS)
      hipLaunchKernelGGL((k_gemm_cut<WM, WN, MB, NB, WT, GEMM_BIAS, 0, true, OCC, NA, TWO>), dim3(grid), dim3(threads), 0, s, a);
    else
      hipLaunchKernelGGL((k_gemm_cut<WM, WN, MB, NB, WT, GEMM_SILU_PAIR, 0, true, OCC, NA, TWO>), dim3(grid), dim3(threads), 0, s, a);
    return hipGetLastError();
  }
};
// Two wavefronts share an A row block in the smallest tile; in the others a wavefront owns whole rows.  With two
// sums two wavefronts per SIMD fit (128 x 128, f32 rows, one sum, eight wavefronts and four per SIMD:
// 4096 x 6400 x 1600 467 us, here 457; bf16 rows, one sum, three per SIMD: 236 us, here 246).  f32 rows and no more
// than one tile to a CU: eight wavefronts on it, two to a row block (1024 x 2304 x 768 37 us, four wavefronts 42).
// bf16 and int8 rows and more than two 128 x 128 tiles to a CU: one sum, so that three of them are there (3200 x 3840 x
// 1280 85 us, two sums 100; int8 92, 113); so many tiles have always been whole and had one sum.
template <int WT>
using Tile64x128 = Shape<2, 2, 1, 2, WT, 3, WT == 0 ? 4 : 2, true>;
template <int WT>
using Tile128x128 = Shape<4, 1, 1, 4, WT, 2, 2, true>;
using Tile128x128by8 = Shape<4, 2, 1, 2, 0, 2, 4, true>;  // (f32 rows)
using Tile256x128 = Shape<8, 1, 1, 4, 0, 2, 2, true>;  // (f32 rows)
template <int WT>
using Tile128x128by3 = Shape<4, 1, 1, 4, WT, 3, 2, false>;  // (bf16 and int8 rows)
template <int WT>
using Tile128x256 = Shape<4, 1, 1, 8, WT, 2, 2, false>;  // (bf16 and int8 rows)

template <int WT>
hipError_t launch_tile(const GemmArgs& a, int epi, CutPlan p, hipStream_t s) {
  if (p.tile == CUT_64x128) return Tile64x128<WT>::launch(a, epi, p.parts, s);
  if (p.tile == CUT_128x128) return Tile128x128<WT>::launch(a, epi, p.parts, s);
  if constexpr (WT == 0) {
    if (p.tile == CUT_128x128_8) return Tile128x128by8::launch(a, epi, p.parts, s);
    if (p.tile == CUT_256x128) return Tile256x128::launch(a, epi, p.parts, s);
  } else {
    if (p.tile == CUT_128x128_3) return Tile128x128by3<WT>::launch(a, epi, p.parts, s);
    if (p.tile == CUT_128x256) return Tile128x256<WT>::launch(a, epi, p.parts, s);
  }
  return hipErrorInvalidValue;
}

bool takes(const GemmArgs& a) {
  const int kt = !a.w_bf16 && !a.w_scale ? 16 : 32;
  // (offsets within a tile's rows are 32 bits)
  return !(a.w_bf16 && a.w_scale) && a.K % kt == 0 && a.K >= kt && !a.a_packed && !a.c_packed &&
         (size_t)a.lda * 256 * 4 < ((size_t)1 << 31) && (size_t)a.K * 256 * 4 < ((size_t)1 << 31);
}

// Time of a product in microseconds: a start, the stages of K at the pace of the CU with the most items,
// and for a cut K the partial tiles' way through memory.  The constants are those of the
// least regret over the four GPT-2 widths' projections at 66 to 8192 rows (464 shapes a storage, W from HBM) with 1 to 8
// parts each.  f32 rows: timed with the epilogue and norm that each has in the model, the plan of least predicted time
// is 0.3 % slower than the best measured one in the mean, 6 % at most (fitted to bare products 1.0 and 14 %: whole
// 64 x 128 tiles where two parts of 128 x 128 were faster, 420 x 3072 x 768 with GELU 31.4 us against 27.5).  bf16 and int8
// rows: fitted to bare products, 1.7 and 1.8 % with the epilogues.
struct Pace {
  float start, stage, more, part;  // start; a stage alone; each further item on the CU; a partly filled round
};
struct Reduce {
  float start, part, rest;  // a reduction's launch; a part and what is left per 10^6 outputs
};
// [storage][CutTile]
constexpr Pace kPace[3][5] = {
    {{7.79f, 0.496f, 0.171f, 0.167f}, {8.78f, 0.647f, 0.497f, 0.080f}, {9.31f, 1.018f, 0.988f, 0.207f}, {8.69f, 0.612f, 0.0f, 0.0f}, {}},
    {{3.4f, 0.461f, 0.204f, 0.131f}, {9.1f, 0.661f, 0.316f, 0.302f}, {}, {}, {12.3f, 0.403f, 0.404f, 0.311f}},
    {{7.9f, 0.518f, 0.234f, 0.139f}, {12.0f, 0.807f, 0.285f, 0.383f}, {}, {}, {14.0f, 0.101f, 0.630f, 0.288f}}};
constexpr Reduce kReduce[3] = {{0.06f, 1.33f, 0.126f}, {2.0f, 1.20f, 0.2f}, {5.0f, 1.55f, 0.4f}};

}  // namespace

bool gemm_cut_plan(const GemmArgs& a, int num_cus, CutPlan* plan) {
  if (!takes(a) || a.M < kCutMinRows) return false;  // (37 x 5120 x 1280, int8: a tile of 64 rows is half padding)
  const int wt = a.w_scale ? 2 : a.w_bf16 ? 1 : 0;
  const long tiles64 = (long)((a.M + 63) / 64) * ((a.N + 127) / 128);
  if (wt == 0) {
    // Little work: the f32 cores' 64 x 64 tiles are as fast or faster (192 x 2304 x 768: 17.0 against 18.4 us), and so
    // they are where two rows of tiles leave most CUs with one (100 x 3840 x 1280: 23.2 against 28.2 us, 128 x 4800 x
    // 1600 33.9 against 35.0, 128 x 6400 x 1600 35.0 against 35.8); from there on the other way round (134 x 6400 x
    // 1600: 50.3 against 41.1 us, 134 x 4800 x 1600 35.8 against 34.9, 256 x 4096 x 1024 28.8 against 27.7).
    const double mnk = (double)a.M * a.N * a.K;
    if (a.M < a.b9_min_rows || (a.M <= 128 && 2 * tiles64 <= num_cus)) return false;
    if (!(tiles64 >= 20 && mnk >= 0.85e9) && !(tiles64 >= 60 && a.K >= 1280)) return false;
  } else if (tiles64 < (wt == 1 ? 13 : 24)) {
    return false;  // (96 x 768 x 768, bf16: 9.9 against 11.3 us; 100 x 1280 x 1280, int8: 14.2 against 15.5)
  }
  // Many tiles of 128 x 256 (bf16 and int8 rows; 1.75 to a CU): half the cuts of A per MFMA
  // (8192 x 4800 x 1600 bf16: 378 against 388 us, int8 8192 x 1600 x 6400: 508 against 535).
  if (wt != 0 && (long)((a.M + 127) / 128) * ((a.N + 255) / 256) * 4 >= 7L * num_cus) {
    *plan = {CUT_128x256, 1};
    return true;
  }
  const float mn = (float)a.M * (float)a.N * 1e-6f;
  const int stages = a.K / (wt == 0 ? 16 : 32);
  const bool norm = a.ln_out || a.post_x;  // rides on the reduction of a cut K, else a launch of its own
  const int most = a.ws && a.N % 4 == 0 ? (int)std::min<size_t>(std::min(8, a.K / 128), a.ws_floats / ((size_t)a.M * a.N)) : 1;
  const Reduce& red = kReduce[wt];
  float best = 0.0f;
  for (int t = CUT_64x128; t <= CUT_128x128_3; ++t) {
    if (wt == 0 ? t == CUT_128x128_3 || (t == CUT_256x128 && a.M < 512) : t == CUT_256x128 || t == CUT_128x128_8) continue;
    const int bm = t == CUT_64x128 ? 64 : t == CUT_256x128 ? 256 : 128;
    const long tiles = (long)((a.M + bm - 1) / bm) * ((a.N + 127) / 128);
    for (int parts = 1; parts <= std::max(1, most); ++parts) {
      const long items = (tiles + 7) / 8 * 8 * parts;  // (as many to each XCD as the fullest one has)
      if (t == CUT_128x128_8 && items > num_cus) continue;
      if (wt != 0 && t != CUT_64x128 && (t == CUT_128x128_3) != (parts == 1 && items > 2 * num_cus)) continue;
      const float on_cu = (float)((items + num_cus - 1) / num_cus), round = std::max(0.0f, (float)items / (float)num_cus - 1.0f);
      const Pace& p = kPace[wt][t];
      const float us = p.start + (float)((stages + parts - 1) / parts) * (p.stage + (on_cu - 1.0f) * p.more + round * p.part) +
                       (parts > 1 ? red.start + (red.part * (float)parts + red.rest) * mn : norm ? 4.0f + 2.0f * mn : 0.0f);
      if (best == 0.0f || us < best) {
        best = us;
        *plan = {(CutTile)t, parts};
      }
    }
  }
  return true;
}

bool gemm_cut_forced(const GemmArgs& a, CutPlan* plan) {
  const bool f32_rows = !a.w_bf16 && !a.w_scale;
  const int bm = a.plan_bm, bn = a.plan_bn;
  plan->parts = std::max(1, a.plan_parts);
  plan->tile = bn == 256    ? CUT_128x256
               : bm == 256  ? CUT_256x128
               : bm == 64   ? CUT_64x128
               : a.plan_alt ? (f32_rows ? CUT_128x128_8 : CUT_128x128_3)
                            : CUT_128x128;
  if (plan->parts > std::max(1, a.K / 32)) return false;
  if (a.plan_alt && (bm != 128 || bn != 128)) return false;
  return (bn == 128 && (bm == 64 || bm == 128 || (bm == 256 && f32_rows))) || (bn == 256 && bm == 128 && !f32_rows);
}

hipError_t launch_gemm_cut(const GemmArgs& a, int epi, CutPlan plan, hipStream_t s) {
  if (!takes(a) || plan.parts < 1 || plan.parts > 8) return hipErrorInvalidValue;
  if (plan.parts > 1 && (!a.ws || a.N % 4 != 0 || (size_t)plan.parts * a.M * a.N > a.ws_floats)) return hipErrorInvalidValue;
  if (a.w_scale) return launch_tile<2>(a, epi, plan, s);
  return a.w_bf16 ? launch_tile<1>(a, epi, plan, s) : launch_tile<0>(a, epi, plan, s);
}

hipError_t launch_gemm_cut_grouped(const GemmArgs& a, int epi, int tile_rows, hipStream_t s) {
  if (!takes(a) || !a.w_bf16) return hipErrorInvalidValue;
  if (tile_rows == 64) return Tile64x128<1>::launch_grouped(a, epi, s);
  if (tile_rows == 128) return Tile128x128by3<1>::launch_grouped(a, epi, s);  // (many rows: many tiles)
  return hipErrorInvalidValue;
}

}  // namespace pgk
