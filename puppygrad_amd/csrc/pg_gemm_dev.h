// What the product kernels of pg_prefill.hip and pg_gemm_cut.hip share.
#pragma once
#include <math.h>

#include <algorithm>

#include "pg_cut.h"
#include "pg_kernels.h"
#include "pg_math.h"

namespace pgk {

// A product on the bf16 matrix cores (pg_gemm_cut.hip): the tile and the number of parts that K is
// cut into (1: whole tiles; otherwise raw partial tiles to GemmArgs::ws, for a reduce kernel).
// (CUT_128x128_8: by eight wavefronts; CUT_128x128_3: three of them on a CU)
enum CutTile : int { CUT_64x128 = 0, CUT_128x128 = 1, CUT_256x128 = 2, CUT_128x128_8 = 3, CUT_128x128_3 = 4, CUT_128x256 = 5 };
struct CutPlan {
  CutTile tile;
  int parts;
};
// False where these kernels do not take the product, or are not the faster ones for it.
bool gemm_cut_plan(const GemmArgs& a, int num_cus, CutPlan* plan);
// The plan that GemmArgs::plan_bm, plan_bn and plan_parts ask for; false where there is none such.
bool gemm_cut_forced(const GemmArgs& a, CutPlan* plan);
hipError_t launch_gemm_cut(const GemmArgs& a, int epi, CutPlan plan, hipStream_t s);
// A product of an activation matrix in cut form (pg_gemm_rows.hip): input rows per block (16 mt), rows of W per block
// (at most 16 ng, a multiple of eight) and parts of K.
struct CutRowsPlan {
  int mt, ng, rows, parts;
};
bool gemm_cut_rows_plan(const GemmArgs& a, int num_cus, CutRowsPlan* plan);
hipError_t launch_gemm_cut_rows(const GemmArgs& a, int epi, const CutRowsPlan& p, hipStream_t s);
// (bf16 rows; tiles of tile_rows = 64 or 128 rows)
hipError_t launch_gemm_cut_grouped(const GemmArgs& a, int epi, int tile_rows, hipStream_t s);

// A product with activations and W in half form (pg_gemm_half.hip): the tile, or blocks of 16 mt input rows and `rows` rows of W
// (HALF_ROWS), and parts of K (1: whole tiles; otherwise raw partial tiles to GemmArgs::ws).
// (_8: by eight wavefronts; HALF_128x256: one chain of matrix instructions, its sums are the less precise ones)
enum HalfTile : int { HALF_64x128 = 0, HALF_128x128 = 1, HALF_128x128_8 = 2, HALF_128x256 = 3, HALF_ROWS = 4, HALF_128x256_8 = 5 };
struct HalfPlan {
  int tile, parts, mt, rows;
};
bool gemm_half_takes(const GemmArgs& a, int epi);
HalfPlan gemm_half_plan(const GemmArgs& a, int epi, int num_cus);
hipError_t launch_gemm_half_plan(const GemmArgs& a, int epi, const HalfPlan& p, hipStream_t s);
// Reduction and norm behind it, and all of it.
hipError_t finish_gemm_half(const GemmArgs& a, int epi, const HalfPlan& p, hipStream_t s);
hipError_t launch_gemm_half(const GemmArgs& a, int epi, int num_cus, hipStream_t s);
// Adds the parts of a cut K (GemmArgs::ws) with bias and epilogue; *ln_done: and the norm.
hipError_t launch_splitk_reduce(const GemmArgs& a, int epi, int parts, hipStream_t s, bool* ln_done);

namespace {

typedef float f16v __attribute__((ext_vector_type(16)));

typedef __attribute__((address_space(3))) char* lds_ptr;

// 16 bytes per lane from base + byte_off (per lane) to lds + 16 lane (LDS address, wavefront-uniform).
// Inline assembly, so that the compiler's count of loads in flight does not know it: it would wait for all
// of them at every LDS read.  vm_wait is the wait that belongs to it; a wait that the compiler places for a
// load of its own is at worst too long (loads return in order).
__device__ __forceinline__ void lds_dma16(const void* base, unsigned byte_off, unsigned lds) {
  asm volatile(
      "s_mov_b32 m0, %0\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %1, %2"
      :
      : "s"(lds), "v"(byte_off), "s"(base)
      : "memory", "m0");
}
// The same from an address per lane.
__device__ __forceinline__ void lds_dma16_at(const void* from, unsigned lds) {
  asm volatile(
      "s_mov_b32 m0, %0\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %1, off"
      :
      : "s"(lds), "v"(from)
      : "memory", "m0");
}
// At most N loads of the wavefront in flight.
template <int N>
__device__ __forceinline__ void vm_wait() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

typedef unsigned u4v __attribute__((ext_vector_type(4)));
// Eight columns of a row as three MFMA operands.
struct Cut {
  u4v p[3];
};
__device__ __forceinline__ Cut cut8(f4 a, f4 b) {
  Cut c;
  unsigned h, m, l;
  cut2(a.x, a.y, h, m, l);
  c.p[0].x = h, c.p[1].x = m, c.p[2].x = l;
  cut2(a.z, a.w, h, m, l);
  c.p[0].y = h, c.p[1].y = m, c.p[2].y = l;
  cut2(b.x, b.y, h, m, l);
  c.p[0].z = h, c.p[1].z = m, c.p[2].z = l;
  cut2(b.z, b.w, h, m, l);
  c.p[0].w = h, c.p[1].w = m, c.p[2].w = l;
  return c;
}

// Epilogues that add to the residual, and what column n of the product adds
// (GEMM_RESID_SCALED: GemmArgs::col_scale).
template <int EPI>
constexpr bool kAddsResid = EPI == GEMM_RESID || EPI == GEMM_RESID_SCALED;
template <int EPI>
__device__ __forceinline__ float col_scaled(const GemmArgs& a, int n, float c) {
  if constexpr (EPI == GEMM_RESID_SCALED) return a.col_scale[n] * c;
  return c;
}

__device__ __forceinline__ float sq_relu(float x) {
  const float p = fmaxf(x, 0.0f);
  return p * p;
}
// Grouped products: the row of A that row m takes.
__device__ __forceinline__ int group_row(const GemmArgs& a, int m) {
  return a.group_rows ? max(a.group_rows[m], 0) : m;
}
// GEMM_SILU_PAIR: column n of the product with its partner column in the neighbouring lane; even
// columns write.
__device__ __forceinline__ void store_silu_pair(const GemmArgs& a, int m, int n, float c) {
  const float up = __shfl_xor(c, 1, 64);
  if ((n & 1) == 0) a.C[(size_t)m * a.ldc + (n >> 1)] = c / (1.0f + expf(-c)) * up;
}

// Tile number -> tile coordinates.  Tiles are numbered band by band (a band is `band` tile
// rows high), down the columns of a band, so that a run of consecutive numbers, which is
// what one XCD computes, is a compact block of C: its tiles share few rows of A and of W,
// which that XCD's L2 then fetches once.  (Row-major numbering makes every XCD read all of
// W.)
__device__ __forceinline__ void tile_coords(int tile, int tiles_m, int tiles_n, int band, int* tm, int* tn) {
  const int per_band = band * tiles_n;
  const int b = tile / per_band, rem = tile - b * per_band;
  const int bh = min(band, tiles_m - b * band);
  const int col = rem / bh;
  *tn = col;
  *tm = b * band + (rem - col * bh);
}

// A wavefront's tile once more in plain f32 arithmetic, sums over columns [k0, k1), finished and
// written out as the kernel's own epilogue would (SPLIT: the raw partial tile of part `part`):
// where an operand is infinite, or so large that its first part is, the cut values give NaN (inf - inf)
// and f32 arithmetic gives the reference's result.  The tile is MB x NB blocks of 32 x 32 at (mbase,
// nbase), a lane's values those of its accumulators.  WT: W holds f32 (0), bf16 (1) or int8 (2) rows;
// `wrow` is the row of W that column 0 meets, `rows` (may be null) the rows of A as group_row gives
// them.  It keeps no more than a dozen sums at a time, so that its registers stay below what the
// kernel's own loop needs; slow, and next to never run.
template <int MB, int NB, int WT, int EPI, int SPLIT, bool GROUPED>
__device__ __forceinline__ void redo_tile(const GemmArgs& a, int mbase, int nbase, int k0, int k1, int part, size_t wrow) {
  const int lane = threadIdx.x & 63, half = lane >> 5, l32 = lane & 31;
  auto w_at = [&](int n, int k) -> float {
    const size_t at = (wrow + n) * a.K + k;
    if (WT == 1) return __uint_as_float((unsigned)reinterpret_cast<const unsigned short*>(a.W)[at] << 16);
    if (WT == 2) return (float)reinterpret_cast<const signed char*>(a.W)[at];
    return a.W[at];
  };
  for (int i = 0; i < MB; ++i)
    for (int g = 0; g < 4; ++g) {  // four consecutive rows at a time
      const int mrow = mbase + 32 * i + 8 * g + 4 * half;
      float sum[4][NB];
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int j = 0; j < NB; ++j) sum[r][j] = 0.0f;
      for (int k = k0; k < k1; ++k) {
        float wv[NB], av[4];
#pragma unroll
        for (int j = 0; j < NB; ++j) wv[j] = w_at(min(nbase + 32 * j + l32, a.N - 1), k);
#pragma unroll
        for (int r = 0; r < 4; ++r) av[r] = a.A[(size_t)(GROUPED ? group_row(a, mrow + r) : min(mrow + r, a.M - 1)) * a.lda + k];
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int j = 0; j < NB; ++j) sum[r][j] = fmaf(av[r], wv[j], sum[r][j]);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int j = 0; j < NB; ++j) {
          const int m = mrow + r, n = nbase + 32 * j + l32;
          if (m >= a.M || n >= a.N) continue;
          float c = WT == 2 ? a.w_scale[n] * sum[r][j] : sum[r][j];
          if (SPLIT) {
            a.ws[((size_t)part * a.M + m) * a.N + n] = c;
            continue;
          }
          c = (a.bias ? a.bias[n] : 0.0f) + c;
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

// Band height for tile_coords: a run of `run` consecutive tiles (one XCD's share) should
// touch as few rows of A and W as it can: hb tile rows and run / hb tile columns.
inline int choose_band(int tiles_m, int run, int bm, int bn) {
  int best = 1;
  long best_cost = -1;
  for (int hb = 1; hb <= tiles_m; ++hb) {
    const int bands = (tiles_m + hb - 1) / hb;
    const int last = tiles_m - (bands - 1) * hb;  // a short last band makes short, wide runs
    const long cost = (long)hb * bm + (long)((run + hb - 1) / hb) * bn + (last < hb ? (long)(hb - last) * bm / 2 : 0);
    if (best_cost < 0 || cost < best_cost) {
      best_cost = cost;
      best = hb;
    }
  }
  return best;
}

}  // namespace
}  // namespace pgk
