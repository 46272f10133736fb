// Causal attention of prompts on the f16 matrix cores, in and out of half form (pg_half.h).
#include "pg_gemm_dev.h"
#include "pg_half.h"
#include "pg_wave.h"

namespace pgk {
namespace {

__device__ __forceinline__ f16v mfma16(const u4v& a, const u4v& b, const f16v& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8v, a), __builtin_bit_cast(h8v, b), c, 0, 0, 0);
}
__device__ __forceinline__ void halves8(f4 a, f4 b, u4v (&part)[2]) {
  const float x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    unsigned h, l;
    halves2(x[2 * e], x[2 * e + 1], 1.0f, h, l);
    part[0][e] = h, part[1][e] = l;
  }
}

// causal_self_attention (src/models/gpt2/rust.rs:1580-1659) for head_dim 64 over qkv[T][3C], as k_attn_prefill_cut
// (pg_attn_cut.hip) with two f16 numbers a value for three bf16 numbers: three products of the parts for six, half of the
// cutting.  Every dim of Q, K and V of a head is kept times a power of two (HalfScales) with which none of its values can be past
// 2^15; the weights, whose largest is 1, times 2^7.  FORM: out is in half form times V's, or in cut form, as the projection behind it wants it.  Scores, maxima, weights
// and sums are f32.  A tile's products are chains of their own that are added to the output: over 1000 keys one chain of f32
// roundings is off by more than all else in here.
// A block holds QG x 32 queries: the QG wavefronts of a key group share a tile of 32 keys that they have cut once, in operand
// order, in LDS.  KG key groups take the tiles in turn, each wavefront with its own running (max, sum, O), added at the
// end through LDS in the order of the groups.
//   S^T (keys x queries) = K . Q^T      lane (l, half) holds dims 16 s + 8 half .. + 7 of key l / query l
//   online softmax per query            a lane holds 16 keys of one query
//   O^T (dims x queries) += V^T . P^T   a lane's own weights are the operand; V's keys are in LDS in that order
// It appends K and V to the cache panels.  512 tokens x 32, 25 heads 231 us (k_attn_prefill_cut) -> 177; 1000 tokens 42 -> 33.5; 1024
// tokens, 12 heads 29.5 (k_attn_prefill64) -> 27 (with one power of two for all of Q, of K and of V 32 and 25).  Error against f64,
// values N(0, 1), 1.4 to 1.85 10^-7: 0.95 to 1.1 of the f32 cores' (queries three times as large 0.83 to 0.93), 1.5 of k_attn_prefill_cut's (1.2).
// What bounds it: per tile and wavefront 768 clocks of matrix instructions and about 1100 of vector ones.  Grid: x = head, y = block of queries, longest rows first, z = sequence.
template <int QG, int KG, int FORM, typename Next = Nothing>
__global__ __launch_bounds__(64 * QG * KG, 2) void k_attn_prefill_half(const float* __restrict__ qkv, int T, int C, int P,
                                                                      float* __restrict__ kcache,
                                                                      float* __restrict__ vcache,
                                                                      void* __restrict__ out, size_t kv_stride, HalfScales scales, Next next) {
  constexpr int NW = QG * KG;
  constexpr int KSTR = 32 * 16 + 16;            // bytes of an octet of dims of 32 keys, padded
  constexpr int KPART = 8 * KSTR, VPART = 4 * 64 * 16;
  constexpr int TILE = 2 * (KPART + VPART);     // a key group's tile
  constexpr int MERGE = 64 * 33 * 4;            // O^T of a wavefront
  constexpr int LDS = KG * TILE > NW * MERGE ? KG * TILE : NW * MERGE;
  __shared__ __attribute__((aligned(16))) char lds[LDS];
  __shared__ float Ms[NW][32], Ls[NW][32];
  __shared__ __attribute__((aligned(16))) float Ks[2][QG == 1 ? 64 : 1];  // K's and V's powers where there are no registers for them
  if constexpr (std::is_same_v<Next, Ahead>) {  // one sequence: the rows of blocks behind those of queries (attention of 37 tokens by
    // 20 heads is 20 blocks and 6.7 us; c_fc behind it, 13 MB from HBM, 9.7)
    const int first = (T + 32 * QG - 1) / (32 * QG) * (int)gridDim.x, id = (int)(blockIdx.x + gridDim.x * blockIdx.y);
    if (id >= first) {
      if (id - first < next.blocks) read_ahead(next, id - first, (unsigned)id, 64 * NW);
      return;
    }
  }
  qkv += (size_t)blockIdx.z * T * 3 * C;
  kcache += (size_t)blockIdx.z * kv_stride;
  vcache += (size_t)blockIdx.z * kv_stride;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int half = lane >> 5, l32 = lane & 31;
  const int qg = wave % QG, kg = wave / QG;
  const int h = blockIdx.x;
  const int nqb = (T + 32 * QG - 1) / (32 * QG);
  const int qb = nqb - 1 - (int)blockIdx.y;  // the longest rows first
  const int q0 = qb * 32 * QG + 32 * qg;     // the wavefront's queries
  const int qi = q0 + l32;
  const int C3 = 3 * C;
  const float* qbase = qkv + h * 64;
  const float* kbase = qkv + C + h * 64;
  const float* vbase = qkv + 2 * C + h * 64;
  const float* sq = scales.q + h * 64;
  // (a power of two; uniform, and no register to spare)
  const float kC = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(0.125f * 1.44269504088896341f / scales.score[h])));
  constexpr float kLag = 8.0f;  // a weight is at most 2^15, half form's most
  char* kt = lds + kg * TILE;
  char* vt = kt + 2 * KPART;

  // Everything the first tile needs is requested before any of it is waited for.  Q^T operands: step s holds dims 16 s + 8 half .. + 7
  // of query l32.
  f4 q_raw[8], q_pow[8];
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    const int at = 8 * half + 16 * (s >> 1) + 4 * (s & 1);
    q_raw[s] = *reinterpret_cast<const f4*>(qbase + (size_t)min(qi, T - 1) * C3 + at);
    q_pow[s] = *reinterpret_cast<const f4*>(sq + at);
  }
  f4 sk0, sk1;
  float sv = scales.v[h * 64 + lane];
  if constexpr (QG == 1) {
    sk0.x = scales.k[h * 64 + lane];
  } else {
    const f4* k = reinterpret_cast<const f4*>(scales.k + h * 64 + 8 * (lane & 7));
    sk0 = k[0], sk1 = k[1];
  }
  f16v o0, o1;  // O^T rows 0..31 and 32..63
#pragma unroll
  for (int v = 0; v < 16; ++v) o0[v] = o1[v] = 0.0f;
  float m_run = -INFINITY, l_run = 0.0f;

  const int last = (min(qb * 32 * QG + 32 * QG, T) - 1) / 32;  // the block's last key tile
  const int mine = q0 / 32;                                    // the wavefront's
  const int turns = last / KG + 1;
  // Raw rows of the group's next tile: KI pieces of (key, eight dims) and VI of (eight keys, dim) per lane.  A unit of V
  // is the eight keys of an operand: unit u = 2 s + half is keys 16 s + 8 (j / 4) + 4 half + j % 4.
  constexpr int KI = 4 / QG, VI = 4 / QG;
  f4 kr[KI][2];
  float vr[VI][8];
  auto key_of = [](int u, int j) { return 16 * (u >> 1) + 8 * (j >> 2) + 4 * (u & 1) + (j & 3); };
  // (rows of V, and the first of a piece's eight rows of K, are the same for the wavefront: scalar addresses)
  auto fetch = [&](int tile) {
    const int left = T - 1 - tile * 32;  // the last row of the tile that there is
#pragma unroll
    for (int i = 0; i < KI; ++i) {
      const float* k = kbase + (size_t)tile * 32 * C3;
      const unsigned at = (unsigned)min(8 * (qg * KI + i) + (lane >> 3), left) * (unsigned)C3 + 8 * (lane & 7);
      kr[i][0] = *reinterpret_cast<const f4*>(k + at);
      kr[i][1] = *reinterpret_cast<const f4*>(k + at + 4);
    }
#pragma unroll
    for (int i = 0; i < VI; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j)
        vr[i][j] = (vbase + (size_t)(tile * 32 + min(key_of(qg * VI + i, j), left)) * C3)[lane];
  };
  auto meet = [&] {
    if constexpr (QG == 1) __builtin_amdgcn_wave_barrier();
    else __syncthreads();
  };
  if (kg <= last) fetch(kg);
  u4v qp[4][2];
#pragma unroll
  for (int s = 0; s < 4; ++s) halves8(q_raw[2 * s] * q_pow[2 * s], q_raw[2 * s + 1] * q_pow[2 * s + 1], qp[s]);
  if constexpr (QG == 1) Ks[0][lane] = sk0.x, Ks[1][lane] = sv;  // (every wavefront the same)
  for (int turn = 0; turn < turns; ++turn) {
    const int tile = kg + KG * turn;
    meet();  // the last tile has been read
    if (tile <= last) {
      const bool append = tile >= qb * QG;  // the block's own positions go to the cache
      if constexpr (QG == 1) {
        asm volatile("" ::: "memory");  // (not before the loop)
        sk0 = *reinterpret_cast<const f4*>(Ks[0] + 8 * (lane & 7)), sk1 = *reinterpret_cast<const f4*>(Ks[0] + 8 * (lane & 7) + 4);
        sv = Ks[1][lane];
      }
#pragma unroll
      for (int i = 0; i < KI; ++i) {
        const int id = lane + 64 * (qg * KI + i), key = id >> 3, o = id & 7;
        u4v c[2];
        halves8(kr[i][0] * sk0, kr[i][1] * sk1, c);
#pragma unroll
        for (int p = 0; p < 2; ++p) *reinterpret_cast<u4v*>(kt + p * KPART + o * KSTR + key * 16) = c[p];
        if (append && tile * 32 + key < T) {
          float* to = kcache + ((size_t)h * P + tile * 32 + key) * 64 + 8 * o;
          *reinterpret_cast<f4*>(to) = kr[i][0];
          *reinterpret_cast<f4*>(to + 4) = kr[i][1];
        }
      }
#pragma unroll
      for (int i = 0; i < VI; ++i) {
        const int u = qg * VI + i;
        u4v c[2];
        halves8(f4{vr[i][0], vr[i][1], vr[i][2], vr[i][3]} * sv, f4{vr[i][4], vr[i][5], vr[i][6], vr[i][7]} * sv, c);
#pragma unroll
        for (int p = 0; p < 2; ++p) *reinterpret_cast<u4v*>(vt + p * VPART + (u * 64 + lane) * 16) = c[p];
        if (append) {
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const int key = tile * 32 + key_of(u, j);
            if (key < T) vcache[((size_t)h * P + key) * 64 + lane] = vr[i][j];
          }
        }
      }
    }
    meet();
    if (tile + KG <= last) fetch(tile + KG);
    if (tile > mine) continue;  // (wavefront-uniform) later than all of its queries

    // S^T = K . Q^T
    f16v sb, ss;
#pragma unroll
    for (int v = 0; v < 16; ++v) sb[v] = ss[v] = 0.0f;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      u4v k[2];
#pragma unroll
      for (int p = 0; p < 2; ++p) k[p] = *reinterpret_cast<const u4v*>(kt + p * KPART + (2 * s + half) * KSTR + l32 * 16);
      ss = mfma16(k[1], qp[s][0], ss);
      sb = mfma16(k[0], qp[s][0], sb);
      ss = mfma16(k[0], qp[s][1], ss);
    }
    sb += ss;
    if (tile == mine) {
#pragma unroll
      for (int v = 0; v < 16; ++v)
        if (tile * 32 + 8 * (v >> 2) + 4 * half + (v & 3) > qi) sb[v] = -INFINITY;
    }
    float mx = fmaxf(fmaxf(sb[0], sb[1]), sb[2]);
#pragma unroll
    for (int v = 3; v < 15; v += 2) mx = fmaxf(fmaxf(mx, sb[v]), sb[v + 1]);
    mx = fmaxf(mx, sb[15]);
    mx = fmaxf(mx, other_half(mx));
    // the running maximum moves when a score is past it by 2^kLag only: the sums are scaled anew in the first tile and seldom
    // after it
    if (__builtin_amdgcn_ballot_w64((mx - m_run) * kC > kLag) != 0) {
      const float m_new = fmaxf(m_run, mx);
      const float corr = __builtin_amdgcn_exp2f((m_run - m_new) * kC);
      l_run *= corr;
      m_run = m_new;
#pragma unroll
      for (int v = 0; v < 16; ++v) o0[v] *= corr, o1[v] *= corr;
    }
    const float mc = m_run * kC - (15.0f - kLag);
    float psum = 0.0f;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      sb[v] = __builtin_amdgcn_exp2f(fmaf(sb[v], kC, -mc));
      psum += sb[v];
    }
    l_run += psum + other_half(psum);
    // O^T += V^T . P^T, sixteen keys a step; a tile's products are chains of their own
    f16v b0, b1, s0, s1;
#pragma unroll
    for (int v = 0; v < 16; ++v) b0[v] = b1[v] = s0[v] = s1[v] = 0.0f;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      u4v pp[2], va[2], vb[2];
      halves8(f4{sb[8 * s], sb[8 * s + 1], sb[8 * s + 2], sb[8 * s + 3]}, f4{sb[8 * s + 4], sb[8 * s + 5], sb[8 * s + 6], sb[8 * s + 7]}, pp);
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const char* at = vt + p * VPART + ((2 * s + half) * 64 + l32) * 16;
        va[p] = *reinterpret_cast<const u4v*>(at);
        vb[p] = *reinterpret_cast<const u4v*>(at + 32 * 16);
      }
      s0 = mfma16(va[1], pp[0], s0);
      s1 = mfma16(vb[1], pp[0], s1);
      b0 = mfma16(va[0], pp[0], b0);
      b1 = mfma16(vb[0], pp[0], b1);
      s0 = mfma16(va[0], pp[1], s0);
      s1 = mfma16(vb[0], pp[1], s1);
    }
    o0 += b0 + s0;
    o1 += b1 + s1;
  }
  // ---- the key groups' results, added in their order
  if (half == 0) {
    Ms[wave][l32] = m_run;
    Ls[wave][l32] = l_run;
  }
  __syncthreads();
  float M = Ms[qg][l32];
#pragma unroll
  for (int g = 1; g < KG; ++g) M = fmaxf(M, Ms[g * QG + qg][l32]);
  float L = 0.0f;
#pragma unroll
  for (int g = 0; g < KG; ++g) {
    const float mw = Ms[g * QG + qg][l32];
    L += (mw == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f((mw - M) * kC)) * Ls[g * QG + qg][l32];
  }
  const float share = m_run == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f((m_run - M) * kC);
  float (*ob)[33] = reinterpret_cast<float (*)[33]>(lds + wave * MERGE);
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const int d = 8 * (v >> 2) + 4 * half + (v & 3);
    ob[d][l32] = o0[v] * share;
    ob[32 + d][l32] = o1[v] * share;
  }
  __syncthreads();
  if (qi >= T) return;
  // the wavefronts of a query group share its 64 dims; lane: query l32, half of the wavefront's share
  const float inv = 1.0f / L, inv_rest = fmaf(-L, inv, 1.0f);
  const size_t row = (size_t)blockIdx.z * T + qi;
  constexpr int ND = 64 / KG / 2;
#pragma unroll
  for (int j = 0; j < ND; j += 4) {
    const int d = 2 * ND * kg + ND * half + j;
    f4 r, rest;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float sum = 0.0f;
#pragma unroll
      for (int g = 0; g < KG; ++g) sum += reinterpret_cast<float (*)[33]>(lds + (g * QG + qg) * MERGE)[d + e][l32];
      r[e] = sum * inv;
      rest[e] = fmaf(sum, inv, -r[e]) + r[e] * inv_rest;  // (what f32 rounds away: half form keeps some of it)
    }
    // (times V's powers, as the values were)
    if constexpr (FORM == FORM_HALF) store_half4(out, cut_rows((int)gridDim.z * T), row, (size_t)h * 64 + d, r, rest, f4{1.f, 1.f, 1.f, 1.f});
    else {
      const u4v p = *reinterpret_cast<const u4v*>(scales.v + h * 64 + d);  // (one over a power of two)
      store_cut4(out, cut_rows((int)gridDim.z * T), row, (size_t)h * 64 + d, r * __builtin_bit_cast(f4, (254u << 23) - p));
    }
  }
}

template <int QG, int KG>
hipError_t start(const float* qkv, int T, int C, int H, int P, float* kcache, float* vcache, void* out, hipStream_t s, int nseq,
                 size_t kv_stride, const HalfScales& f, int out_form) {
  const dim3 grid(H, (T + 32 * QG - 1) / (32 * QG), nseq), block(64 * QG * KG);
  if (out_form == FORM_HALF)
    hipLaunchKernelGGL((k_attn_prefill_half<QG, KG, FORM_HALF>), grid, block, 0, s, qkv, T, C, P, kcache, vcache, out, kv_stride, f, Nothing{});
  else
    hipLaunchKernelGGL((k_attn_prefill_half<QG, KG, FORM_CUT>), grid, block, 0, s, qkv, T, C, P, kcache, vcache, out, kv_stride, f, Nothing{});
  return hipGetLastError();
}
}  // namespace

// Which block shape is the fastest (queries groups, key groups), by the blocks that there are to a CU; us, 25 heads or as said:
//  - one tile or two of keys: 64 queries, two key groups (64 tokens 6.1; 41 7.2, 14 6.9; 32 x 33 14.2; 41 16.8, 24 23.6);
//  - 32 queries a block where that is a block to a CU or, for long rows, one and a half, their keys in eight shares (300 tokens
//    11.6; 24 12.1; 1024 tokens, 12 heads 23.6; 24 26.1, k_attn_prefill64 29.6), of short rows in four (100 tokens, 16 heads 7.0; 18 8.1;
//    200 x 4, 12 heads 10.5 with 24, 16.8 with 18);
//  - 64 queries and four shares up to a block and a half to a CU (1000 tokens 31.8; 22 34.6, k_attn_prefill_cut 42);
//  - 64 and two shares up to eleven (16 x 400, 12 heads 44.9; 41 49.9; 8 x 1024, 16 heads 106; 41 108, 24 128);
//  - 128 queries, all keys (32 x 512 177; 22 229, k_attn_prefill_cut 231).
int attn_half_shape(int T, int H, int nseq, int num_cus) {
  auto blocks = [&](int queries) { return (double)H * nseq * ((T + queries - 1) / queries) * 256.0 / num_cus; };
  const double b32 = blocks(32), b64 = blocks(64);
  if (T <= 64) return 22;
  if (b32 <= 256 || (b32 <= 400 && T >= 500)) return T >= 256 ? 18 : T < 160 ? 14 : 24;
  if (b64 <= 400) return T <= 128 ? 22 : 24;
  return b64 <= 2800 ? 22 : 41;
}

hipError_t launch_attn_prefill_half(const float* qkv, int T, int C, int H, int P, float* kcache, float* vcache, void* out,
                                    hipStream_t s, int nseq, size_t kv_stride, const HalfScales& f, int shape, int out_form, const Ahead* next) {
  if ((out_form != FORM_HALF && out_form != FORM_CUT) || nseq < 1 || nseq > 65535 || (reinterpret_cast<uintptr_t>(out) & 15)) return hipErrorInvalidValue;
  if (next && next->blocks > 0 && nseq == 1 && shape == 22 && out_form == FORM_HALF) {
    const dim3 grid(H, (T + 63) / 64 + (next->blocks + H - 1) / H);
    hipLaunchKernelGGL((k_attn_prefill_half<2, 2, FORM_HALF, Ahead>), grid, dim3(256), 0, s, qkv, T, C, P, kcache, vcache, out, kv_stride, f, *next);
    return hipGetLastError();
  }
  switch (shape) {
    case 41: return start<4, 1>(qkv, T, C, H, P, kcache, vcache, out, s, nseq, kv_stride, f, out_form);
    case 22: return start<2, 2>(qkv, T, C, H, P, kcache, vcache, out, s, nseq, kv_stride, f, out_form);
    case 24: return start<2, 4>(qkv, T, C, H, P, kcache, vcache, out, s, nseq, kv_stride, f, out_form);
    case 18: return start<1, 8>(qkv, T, C, H, P, kcache, vcache, out, s, nseq, kv_stride, f, out_form);
    case 14: return start<1, 4>(qkv, T, C, H, P, kcache, vcache, out, s, nseq, kv_stride, f, out_form);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace pgk
