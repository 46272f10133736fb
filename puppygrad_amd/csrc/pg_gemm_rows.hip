// Products of some tens to some hundreds of rows with activations in cut form (FORM_CUT; pg_cut.h): f32 rows, 33 to 64 of them, from 129
// on those of models wider than 768 (narrower ones keep W in cut form too, pg_gemm_half.hip), and all of a model's whose weights have
// no half form (takes_half_form).
#include "pg_gemm_dev.h"

namespace pgk {
namespace {

// Between the 32-row kernel, whose blocks each cut all of the input (VALU bound from 33 rows on: 37 x 3840 x 1280 against
// int8 rows 12.8 us, a third of it the cut), and the tiles of pg_gemm_cut.hip, which leave most CUs without one and walk K
// at a memory latency a stage (80 x 3840 x 1280, int8 rows: 21 us and 4.5 for the reduction of a cut K).  Here every CU
// has a block, all of a block's loads are operands as they are and nearly all in flight at once: 7.9 and 8.5 us.
// Bound by what a CU takes in from L2, 6 bytes per input value and block (75 to 85 KB/us), behind 3 us of launch and
// first loads.
// A block owns 16 MT input rows (blockIdx.z) and up to 16 NG rows of W (a.rows_per_block of them, a multiple of
// eight); its eight wavefronts take the steps of 32 columns in turn, each with all of the block's rows, and the
// eight partial tiles are added through LDS at the end.  gridDim.y > 1: K is cut over blocks as well, raw tiles go
// to a.ws[part][M][N].
template <int EPI, int WT, int MT, int NG>
__global__ __launch_bounds__(512) void k_gemm_cut_rows(GemmArgs a) {
  constexpr int RB = WT == 0 ? 128 : WT == 1 ? 64 : 32;  // bytes of a row of W in a step
  constexpr int LPR = RB / 16, RPL = 64 / LPR;           // lanes to a row, rows per load
  constexpr int WL = (16 * NG + RPL - 1) / RPL;          // loads of W per step
  constexpr int WSTR = RB + 16;                          // row stride of the W tile in LDS, bytes
  constexpr int CSTR = 16 * NG + 4;                      // row stride of the partial tile, floats
  constexpr int SLAB = RPL * WL * WSTR > 16 * MT * CSTR * 4 ? RPL * WL * WSTR : 16 * MT * CSTR * 4;
  constexpr int PD = MT * NG > 8 ? 1 : 2;                // steps requested ahead
  __shared__ __attribute__((aligned(16))) char slab[8][SLAB];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int i16 = lane & 15, kq = lane >> 4;
  const int n0 = (int)blockIdx.x * a.rows_per_block, n1 = min(n0 + a.rows_per_block, a.N);
  const int m0 = (int)blockIdx.z * 16 * MT;
  const int mp = cut_rows(a.M);
  const int piece = (int)blockIdx.y * 8 + wave, pieces = (int)gridDim.y * 8;
  const int steps_all = a.K / 32;
  const int steps = piece < steps_all ? (steps_all - piece + pieces - 1) / pieces : 0;
  char* wt = slab[wave];

  // W: LPR lanes to a row
  const char* wp[WL];
  const size_t rowbytes = (size_t)a.K * (RB / 32);
#pragma unroll
  for (int j = 0; j < WL; ++j)
    wp[j] = reinterpret_cast<const char*>(a.W) + (size_t)min(n0 + RPL * j + lane / LPR, n1 - 1) * rowbytes + 16 * (lane % LPR);
  // input: operand (tile mt, part p) of a step is 16 bytes a lane, rows next to each other
  const char* xp[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
    xp[mt] = reinterpret_cast<const char*>(a.A) + ((size_t)kq * 3 * mp + min(m0 + 16 * mt + i16, a.M - 1)) * 16;
  const size_t xpart = (size_t)mp * 16, xstep = (size_t)mp * 4 * 3 * 16;

  // The write-out takes four columns of a row at a time, neighbouring lanes neighbouring columns, or, into a matrix
  // in cut form, neighbouring rows, which lie next to each other there.  What it adds is requested first.
  constexpr int ITEMS = 16 * MT * 4 * NG;
  constexpr int IPT = (ITEMS + 511) / 512;
  auto row_of = [&](int idx) { return a.c_cut ? idx % (16 * MT) : idx / (4 * NG); };
  auto col_of = [&](int idx) { return 4 * (a.c_cut ? idx / (16 * MT) : idx % (4 * NG)); };
  f4 ebias[IPT], eres[IPT];
#pragma unroll
  for (int q = 0; q < IPT; ++q) {
    const int idx = tid + 512 * q, m = m0 + row_of(idx), n = n0 + col_of(idx);
    const bool live = gridDim.y == 1 && idx < ITEMS && m < a.M && n < n1;
    ebias[q] = eres[q] = f4{0.f, 0.f, 0.f, 0.f};
    if (live && a.bias) ebias[q] = *reinterpret_cast<const f4*>(a.bias + n);
    if (live && kAddsResid<EPI>) eres[q] = *reinterpret_cast<const f4*>(a.resid + (size_t)m * a.ldc + n);
  }

  f4 big[MT][NG], small[MT][NG];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int g = 0; g < NG; ++g) big[mt][g] = small[mt][g] = f4{0.f, 0.f, 0.f, 0.f};

  u4v rw[PD][WL], rx[PD][MT][3];
  auto load_step = [&](int s, u4v (&w)[WL], u4v (&x)[MT][3]) {
    const size_t col = (size_t)piece + (size_t)pieces * min(s, steps - 1);
#pragma unroll
    for (int j = 0; j < WL; ++j) w[j] = *reinterpret_cast<const u4v*>(wp[j] + col * RB);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int p = 0; p < 3; ++p) x[mt][p] = *reinterpret_cast<const u4v*>(xp[mt] + col * xstep + p * xpart);
  };
  auto mfma = [](const u4v& x, const u4v& w, const f4& c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, x), __builtin_bit_cast(bf16x8, w), c, 0, 0, 0);
  };
  auto mul_step = [&](const u4v (&w)[WL], const u4v (&x)[MT][3]) {
#pragma unroll
    for (int j = 0; j < WL; ++j)
      *reinterpret_cast<u4v*>(wt + (RPL * j + lane / LPR) * WSTR + 16 * (lane % LPR)) = w[j];
    __builtin_amdgcn_wave_barrier();
    u4v wo[NG][WT == 0 ? 3 : 1];
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const char* at = wt + (16 * g + i16) * WSTR;
      if constexpr (WT == 1) {
        wo[g][0] = *reinterpret_cast<const u4v*>(at + 16 * kq);
      } else if constexpr (WT == 2) {
        const u2v raw = *reinterpret_cast<const u2v*>(at + 8 * kq);
#pragma unroll
        for (int e = 0; e < 4; ++e) {  // columns 2 e and 2 e + 1
          const unsigned v = raw[e / 2];
          const unsigned lo = __float_as_uint((float)((int)(v << (24 - 16 * (e % 2))) >> 24));
          const unsigned hi = __float_as_uint((float)((int)(v << (16 - 16 * (e % 2))) >> 24));
          wo[g][0][e] = (lo >> 16) | (hi & 0xffff0000u);
        }
      } else {
        const Cut c = cut8(*reinterpret_cast<const f4*>(at + 32 * kq), *reinterpret_cast<const f4*>(at + 32 * kq + 16));
#pragma unroll
        for (int p = 0; p < 3; ++p) wo[g][p] = c.p[p];
      }
    }
    __builtin_amdgcn_wave_barrier();
    // the small products first, in a sum of their own; each product over all tiles before the next
    auto all = [&](int xpl, int wpl, f4 (&c)[MT][NG]) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int g = 0; g < NG; ++g) c[mt][g] = mfma(x[mt][xpl], wo[g][wpl], c[mt][g]);
    };
    if constexpr (WT == 0) {
      all(2, 0, small);
      all(0, 2, small);
      all(1, 1, small);
      all(1, 0, small);
      all(0, 1, small);
    } else {
      all(2, 0, small);
      all(1, 0, small);
    }
    all(0, 0, big);
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
  // big[mt][g][r] is row 16 mt + 4 kq + r, column 16 g + i16
  float* mine = reinterpret_cast<float*>(slab[wave]);
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        mine[(16 * mt + 4 * kq + r) * CSTR + 16 * g + i16] = big[mt][g][r] + small[mt][g][r];
  __syncthreads();
#pragma unroll
  for (int q = 0; q < IPT; ++q) {
    const int idx = tid + 512 * q, mr = row_of(idx), nl = col_of(idx);
    const int m = m0 + mr, n = n0 + nl;
    if (idx >= ITEMS || m >= a.M || n >= n1) continue;
    f4 sum = *reinterpret_cast<const f4*>(slab[0] + (mr * CSTR + nl) * 4);
#pragma unroll
    for (int w = 1; w < 8; ++w) sum += *reinterpret_cast<const f4*>(slab[w] + (mr * CSTR + nl) * 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (fabsf(sum[e]) < INFINITY) continue;
      // an infinite operand, or a weight whose first part is: the block's columns in f32 arithmetic
      float t = 0.0f;
      for (int k = 0; k < a.K; ++k) {
        const int in_turn = k / 32 % pieces - 8 * (int)blockIdx.y;
        if (in_turn < 0 || in_turn >= 8) continue;
        const size_t at = (size_t)(n + e) * a.K + k;
        const float w = WT == 2 ? (float)reinterpret_cast<const signed char*>(a.W)[at]
                        : WT == 1 ? __uint_as_float((unsigned)reinterpret_cast<const unsigned short*>(a.W)[at] << 16)
                                  : a.W[at];
        t = fmaf(cut_form_value(a.A, mp, (size_t)m, (size_t)k), w, t);
      }
      sum[e] = t;
    }
    if (WT == 2) sum *= *reinterpret_cast<const f4*>(a.w_scale + n);
    if (gridDim.y > 1) {
      *reinterpret_cast<f4*>(a.ws + ((size_t)blockIdx.y * a.M + m) * a.N + n) = sum;
      continue;
    }
    f4 c = ebias[q] + sum;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (EPI == GEMM_GELU) c[e] = gelu_tanh(c[e]);
      if (EPI == GEMM_SQRELU) c[e] = sq_relu(c[e]);
      if (kAddsResid<EPI>) c[e] = eres[q][e] + col_scaled<EPI>(a, n + e, c[e]);
    }
    if (a.c_cut) store_cut4(a.C, mp, (size_t)m, (size_t)n, c);
    else *reinterpret_cast<f4*>(a.C + (size_t)m * a.ldc + n) = c;
  }
}

template <int EPI, int WT>
hipError_t launch_form(const GemmArgs& a, const CutRowsPlan& p, hipStream_t s) {
  const dim3 grid((unsigned)((a.N + a.rows_per_block - 1) / a.rows_per_block), (unsigned)p.parts,
                  (unsigned)((a.M + 16 * p.mt - 1) / (16 * p.mt)));
#define PG_CASE(MT, NG) \
  if (p.mt == MT && p.ng == NG) { hipLaunchKernelGGL((k_gemm_cut_rows<EPI, WT, MT, NG>), grid, dim3(512), 0, s, a); return hipGetLastError(); }
  if constexpr (WT == 2) { PG_CASE(2, 1) PG_CASE(2, 2) }  // (17 to 32 rows, which the other storages leave to the 32-row kernel)
  PG_CASE(3, 1) PG_CASE(4, 1)
  PG_CASE(3, 2) PG_CASE(4, 2)
  PG_CASE(3, 3) PG_CASE(4, 3)
  if constexpr (WT != 0) { PG_CASE(3, 4) PG_CASE(4, 4) }
#undef PG_CASE
  return hipErrorInvalidValue;
}
template <int WT>
hipError_t launch_wt(const GemmArgs& a, int epi, const CutRowsPlan& p, hipStream_t s) {
  if (p.parts > 1) return launch_form<GEMM_BIAS, WT>(a, p, s);
  switch (epi) {
    case GEMM_BIAS: return launch_form<GEMM_BIAS, WT>(a, p, s);
    case GEMM_GELU: return launch_form<GEMM_GELU, WT>(a, p, s);
    case GEMM_RESID: return launch_form<GEMM_RESID, WT>(a, p, s);
    default: return hipErrorInvalidValue;
  }
}
// What a plan of a product costs, in microseconds but for a constant, chosen so that the plan of least cost is close to the
// best measured one, over 24860 plans of the four GPT-2 widths' projections, W from HBM, at rows on both sides of where
// the form ends.  At other rows, and at widths 384, 512 and 2048 too (35054 plans, which the int8 constants have seen), a
// layer's four products are 1.0 % slower than the best plans in the mean for f32 rows, 1.3 bf16, 0.6 int8 (9 % at most;
// constants from times at 24 to 320 rows: 1.9, 2.7 and 2.5 %, 12 % at most).  `most`: a block of 64 x 64, whose registers spill.  `reduce`: the launch that adds the parts; `norm`,
// `norm_values`: that of a norm by itself, and per 10^6 values.
struct RowsPace {
  float round, step, mt, ng, both, most, fill, part, reduce, norm, norm_values;
};
constexpr RowsPace kRowsPace[3] = {{11.237f, -0.786f, 0.179f, 0.891f, -0.013f, 0.0f, 0.203f, 3.578f, 2.545f, 3.175f, 0.731f},
                                   {0.357f, -0.208f, 0.129f, 0.086f, 0.039f, 0.307f, 0.117f, 4.787f, 2.433f, 2.971f, 3.534f},
                                   {0.039f, -0.064f, 0.170f, -0.025f, 0.054f, -0.033f, 0.022f, 4.668f, 3.294f, 2.652f, 7.051f}};

}  // namespace

// The rows up to which a model's four projections take cut form, from whole prompts timed both ways (ms, the tiles of pg_gemm_cut.hip
// first, these kernels second; where half form is had it goes before both for bf16 and int8 rows, and past these rows for f32 ones).  A step in this form's time is a round of blocks (64 rows by 48 rows of W, 64 for int8 rows) over the CUs, so the
// line is a number of rounds of the widest product, past which the tiles of pg_gemm_cut.hip, which read an input row once
// for 128 columns, are the faster ones:
//  - f32 and bf16 rows, two rounds.  f32 at width 1600: 192 rows 7.52 / 6.58, 193 rows 7.79 / 8.15; 1280: 256 rows 4.83 /
//    4.59, 300 rows 5.41 / 5.53; 1024: 320 rows 2.98 / 2.60, 400 rows 3.29 / 3.22, 600 rows 3.93 / 4.09; 33 rows, 1600: 4.03 / 3.43.
//    bf16 at 1600: 131 rows 5.00 / 4.49, 192 rows 5.28 / 5.22, 193 rows 5.76 / 6.36; 1280: 256 rows 3.90 / 3.65, 257 rows
//    3.99 / 4.02; 1024: 320 rows 2.44 / 2.15, 400 rows 2.57 / 2.54; 768: 512 rows 1.08 / 1.01, 560 rows 1.17 / 1.17, 800 rows
//    1.16 / 1.34.
//  - f32 rows up to width 768, where the tiles leave a third of the CUs without one: four rounds and 1024 rows.  768: 512 rows
//    1.41 / 1.26, 700 rows 1.71 / 1.65, 1024 rows 2.01 / 1.93 (8 x 128 1.82 / 1.73), 1026 rows 2.03 / 2.27; 512: 600 rows 1.12 /
//    1.06, 1000 rows 1.39 / 1.38, 1200 rows 1.47 / 1.57.
//  - int8 rows, three rounds.  1600: 448 rows 9.28 / 8.34, 449 rows 9.71 / 9.63, 500 rows 9.96 / 10.2; 1280: 576 rows 6.41 / 5.61,
//    577 rows 6.58 / 6.36; 1024: 768 rows 3.86 / 3.63, 769 rows 4.02 / 3.92; 768: 1024 rows 1.72 / 1.61, 1026 rows 1.68 / 1.71.  Up to
//    32 rows, a step of 20 at 1280 1.89 / 1.85, of 32 2.13 / 2.15, of 32 at 768 0.60 / 0.57.
bool gemm_takes_cut(int M, int K, int N, int w_bf16, int w_int8, int f32_min_rows, int num_cus) {
  if (K < 256 || K % 32 != 0 || N % 32 != 0) return false;  // (narrower: no step for some of the eight wavefronts)
  const int cols = w_int8 ? 64 : 48;  // of a full block, 64 rows
  const long blocks = (long)((std::max(N, 3 * K) + cols - 1) / cols) * ((M + 63) / 64);
  if (w_int8) return M >= 17 && blocks <= 3L * num_cus && (M > 32 || (double)M * N * K <= 0.17e9);
  if (M < kCutFormMinRows) return false;
  if (w_bf16) return blocks <= 2L * num_cus;
  // (65 to 128 rows stay on the f32 cores at the price of 3.88 ms for 100 rows at 1280 that take 2.95 in this form: models
  // tuned with gemm_b9_min_rows get the same results there at every setting)
  if (M > 64 && M <= 128) return false;
  return M >= f32_min_rows && (K <= 768 ? blocks <= 4L * num_cus && M <= 4 * num_cus : blocks <= 2L * num_cus);
}

bool gemm_cut_rows_plan(const GemmArgs& a, int num_cus, CutRowsPlan* plan) {
  if (a.M < 1 || a.K < 32 || a.K % 32 != 0 || a.N < 8 || a.N % 8 != 0 || (a.w_bf16 && a.w_scale) || a.a_packed ||
      a.c_packed || a.ln_packed || a.ldc % 4 != 0 || a.rms_cols || a.post_x || (a.c_cut && a.ldc != a.N))
    return false;
  const int wt = a.w_scale ? 2 : a.w_bf16 ? 1 : 0;
  const int groups = (a.M + 63) / 64, mt = std::max(wt == 2 ? 2 : 3, ((a.M + groups - 1) / groups + 15) / 16);
  const int m_blocks = (a.M + 16 * mt - 1) / (16 * mt), steps = a.K / 32;
  const float mn = (float)a.M * (float)a.N * 1e-6f;
  const RowsPace& p = kRowsPace[wt];
  // (a part: a step at least for each wavefront)
  const int most = a.ws && !a.c_cut ? (int)std::min<size_t>(std::min(8, steps / 8), a.ws_floats / ((size_t)a.M * a.N)) : 1;
  float best = -1.0f;
  for (int parts = 1; parts <= std::max(1, most); ++parts)
    for (int rows = 8; rows <= 64; rows += 8) {
      const int ng = (rows + 15) / 16;
      if ((mt == 2 && ng > 2) || (wt == 0 && ng > 3)) continue;
      const long blocks = (long)((a.N + rows - 1) / rows) * m_blocks * parts;
      const float turns = (float)((blocks + num_cus - 1) / num_cus);
      const float rounds = (float)(((steps + parts - 1) / parts + 7) / 8);
      const float us = turns * (p.round + rounds * (p.step + p.mt * mt + p.ng * ng + p.both * mt * ng + (mt * ng == 16 ? p.most : 0.0f))) +
                       p.fill * (float)blocks / (float)num_cus * rounds * mt +
                       (parts > 1 ? p.reduce + p.part * parts * mn : a.ln_out ? p.norm + p.norm_values * mn : 0.0f);
      if (best < 0.0f || us < best) {
        best = us;
        *plan = {mt, ng, rows, parts};
      }
    }
  return true;
}

hipError_t launch_gemm_cut_rows(const GemmArgs& a0, int epi, const CutRowsPlan& p, hipStream_t s) {
  GemmArgs a = a0;
  const uintptr_t at = reinterpret_cast<uintptr_t>(a.A) | reinterpret_cast<uintptr_t>(a.W) | reinterpret_cast<uintptr_t>(a.C) |
                       reinterpret_cast<uintptr_t>(a.bias) | reinterpret_cast<uintptr_t>(a.w_scale) | reinterpret_cast<uintptr_t>(a.ws);
  if (at & 15 || p.rows < 8 || p.rows % 8 != 0 || p.rows > 16 * p.ng || p.parts < 1 ||
      (p.parts > 1 && (!a.ws || (size_t)p.parts * a.M * a.N > a.ws_floats)) || (a.M + 16 * p.mt - 1) / (16 * p.mt) > 65535)
    return hipErrorInvalidValue;
  a.rows_per_block = p.rows;
  if (a.w_scale) return launch_wt<2>(a, epi, p, s);
  return a.w_bf16 ? launch_wt<1>(a, epi, p, s) : launch_wt<0>(a, epi, p, s);
}

}  // namespace pgk
