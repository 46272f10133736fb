// Causal attention of prompts on the bf16 matrix cores, for models without half form (pg_attn_half.hip has the others').
#include "pg_gemm_dev.h"
#include "pg_wave.h"

namespace pgk {
namespace {

__device__ __forceinline__ f16v mfma16(const u4v& a, const u4v& b, const f16v& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// causal_self_attention (src/models/gpt2/rust.rs:1580-1659) for head_dim 64 over qkv[T][3C], as k_attn_prefill64, with
// the two products on the bf16 matrix cores: K, V, Q and the weights are cut into three bf16 numbers each (cut8), six
// products of the parts stand for one in f32, hi . hi in a sum of its own and everything smaller in another.
// A matrix instruction takes a third of the f32 form's time, but the cut is vector work, and a CU's vector and matrix
// instructions add up.  So a block holds QG x 32 queries: the QG wavefronts of a key group share a tile of 32 keys
// that they have cut once, in operand order, in LDS.  KG key groups take the tiles in turn, each wavefront with its own
// running (max, sum, O), added at the end through LDS in the order of the groups.
//   S^T (keys x queries) = K . Q^T      lane (l, half) holds dims 16 s + 8 half .. + 7 of key l / query l
//   online softmax per query            a lane holds 16 keys of one query
//   O^T (dims x queries) += V^T . P^T   a lane's own weights are the operand; V's keys are in LDS in that order
// It appends K and V to the cache panels.  Grid: x = head, y = block of queries, longest rows first, z = sequence.
// 512 tokens x 32, 25 heads: 490 us by k_attn_prefill64, here 265; error against f64 3.9 and 3.6 10^-7.  What is left: per tile
// and wavefront 1536 clocks of matrix and about 1500 of vector instructions (128 queries a block), and two barriers.
template <int QG, int KG, bool CUT>
__global__ __launch_bounds__(64 * QG * KG, 2) void k_attn_prefill_cut(const float* __restrict__ qkv, int T, int C, int P,
                                                                      float* __restrict__ kcache,
                                                                      float* __restrict__ vcache,
                                                                      float* __restrict__ out, size_t kv_stride) {
  constexpr int NW = QG * KG;
  constexpr int KSTR = 32 * 16 + 16;            // bytes of an octet of dims of 32 keys, padded
  constexpr int KPART = 8 * KSTR, VPART = 4 * 64 * 16;
  constexpr int TILE = 3 * (KPART + VPART);     // a key group's tile
  constexpr int MERGE = 64 * 33 * 4;            // O^T of a wavefront
  constexpr int LDS = KG * TILE > NW * MERGE ? KG * TILE : NW * MERGE;
  __shared__ __attribute__((aligned(16))) char lds[LDS];
  __shared__ float Ms[NW][32], Ls[NW][32];
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
  char* kt = lds + kg * TILE;
  char* vt = kt + 3 * KPART;

  // Q^T operands: step s holds dims 16 s + 8 half .. + 7 of query l32
  u4v qp[4][3];
  {
    const float* q = qbase + (size_t)min(qi, T - 1) * C3 + 8 * half;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const Cut c = cut8(*reinterpret_cast<const f4*>(q + 16 * s), *reinterpret_cast<const f4*>(q + 16 * s + 4));
#pragma unroll
      for (int p = 0; p < 3; ++p) qp[s][p] = c.p[p];
    }
  }
  f16v ob0, ob1, os0, os1;  // O^T rows 0..31 and 32..63: first products, all others
#pragma unroll
  for (int v = 0; v < 16; ++v) ob0[v] = ob1[v] = os0[v] = os1[v] = 0.0f;
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
  for (int turn = 0; turn < turns; ++turn) {
    const int tile = kg + KG * turn;
    meet();  // the last tile has been read
    if (tile <= last) {
      const bool append = tile >= qb * QG;  // the block's own positions go to the cache
#pragma unroll
      for (int i = 0; i < KI; ++i) {
        const int id = lane + 64 * (qg * KI + i), key = id >> 3, o = id & 7;
        const Cut c = cut8(kr[i][0], kr[i][1]);
#pragma unroll
        for (int p = 0; p < 3; ++p) *reinterpret_cast<u4v*>(kt + p * KPART + o * KSTR + key * 16) = c.p[p];
        if (append && tile * 32 + key < T) {
          float* to = kcache + ((size_t)h * P + tile * 32 + key) * 64 + 8 * o;
          *reinterpret_cast<f4*>(to) = kr[i][0];
          *reinterpret_cast<f4*>(to + 4) = kr[i][1];
        }
      }
#pragma unroll
      for (int i = 0; i < VI; ++i) {
        const int u = qg * VI + i;
        const Cut c = cut8(f4{vr[i][0], vr[i][1], vr[i][2], vr[i][3]}, f4{vr[i][4], vr[i][5], vr[i][6], vr[i][7]});
#pragma unroll
        for (int p = 0; p < 3; ++p) *reinterpret_cast<u4v*>(vt + p * VPART + (u * 64 + lane) * 16) = c.p[p];
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
      u4v k[3];
#pragma unroll
      for (int p = 0; p < 3; ++p) k[p] = *reinterpret_cast<const u4v*>(kt + p * KPART + (2 * s + half) * KSTR + l32 * 16);
      ss = mfma16(k[2], qp[s][0], ss);
      sb = mfma16(k[0], qp[s][0], sb);
      ss = mfma16(k[0], qp[s][2], ss);
      ss = mfma16(k[1], qp[s][1], ss);
      ss = mfma16(k[1], qp[s][0], ss);
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
    constexpr float kC = 0.125f * 1.44269504088896341f;
    // the running maximum moves when a score is past it by 2^8 only: the weights stay below that, and the sums are
    // scaled anew in the first tile and seldom after it
    if (__builtin_amdgcn_ballot_w64((mx - m_run) * kC > 8.0f) != 0) {
      const float m_new = fmaxf(m_run, mx);
      const float corr = __builtin_amdgcn_exp2f((m_run - m_new) * kC);
      l_run *= corr;
      m_run = m_new;
#pragma unroll
      for (int v = 0; v < 16; ++v) ob0[v] *= corr, ob1[v] *= corr, os0[v] *= corr, os1[v] *= corr;
    }
    const float mc = m_run * kC;
    float psum = 0.0f;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      sb[v] = __builtin_amdgcn_exp2f(fmaf(sb[v], kC, -mc));
      psum += sb[v];
    }
    l_run += psum + other_half(psum);
    // O^T += V^T . P^T, sixteen keys a step
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const Cut pp = cut8(f4{sb[8 * s], sb[8 * s + 1], sb[8 * s + 2], sb[8 * s + 3]},
                          f4{sb[8 * s + 4], sb[8 * s + 5], sb[8 * s + 6], sb[8 * s + 7]});
      u4v va[3], vb[3];
#pragma unroll
      for (int p = 0; p < 3; ++p) {
        const char* at = vt + p * VPART + ((2 * s + half) * 64 + l32) * 16;
        va[p] = *reinterpret_cast<const u4v*>(at);
        vb[p] = *reinterpret_cast<const u4v*>(at + 32 * 16);
      }
      os0 = mfma16(va[2], pp.p[0], os0);
      os1 = mfma16(vb[2], pp.p[0], os1);
      ob0 = mfma16(va[0], pp.p[0], ob0);
      ob1 = mfma16(vb[0], pp.p[0], ob1);
      os0 = mfma16(va[0], pp.p[2], os0);
      os1 = mfma16(vb[0], pp.p[2], os1);
      os0 = mfma16(va[1], pp.p[1], os0);
      os1 = mfma16(vb[1], pp.p[1], os1);
      os0 = mfma16(va[1], pp.p[0], os0);
      os1 = mfma16(vb[1], pp.p[0], os1);
      os0 = mfma16(va[0], pp.p[1], os0);
      os1 = mfma16(vb[0], pp.p[1], os1);
    }
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
    L += (mw == -INFINITY ? 0.0f : expf((mw - M) * 0.125f)) * Ls[g * QG + qg][l32];
  }
  const float share = m_run == -INFINITY ? 0.0f : expf((m_run - M) * 0.125f);
  float (*ob)[33] = reinterpret_cast<float (*)[33]>(lds + wave * MERGE);
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const int d = 8 * (v >> 2) + 4 * half + (v & 3);
    ob[d][l32] = (ob0[v] + os0[v]) * share;
    ob[32 + d][l32] = (ob1[v] + os1[v]) * share;
  }
  __syncthreads();
  if (qi >= T) return;
  // the wavefronts of a query group share its 64 dims; lane: query l32, half of the wavefront's share
  const float inv = 1.0f / L;
  const size_t row = (size_t)blockIdx.z * T + qi;
  constexpr int ND = 64 / KG / 2;
#pragma unroll
  for (int j = 0; j < ND; j += 4) {
    const int d = 2 * ND * kg + ND * half + j;
    f4 r;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float sum = 0.0f;
#pragma unroll
      for (int g = 0; g < KG; ++g) sum += reinterpret_cast<float (*)[33]>(lds + (g * QG + qg) * MERGE)[d + e][l32];
      r[e] = sum * inv;
    }
    bool finite = true;
#pragma unroll
    for (int e = 0; e < 4; ++e) finite &= fabsf(r[e]) < INFINITY;
    if (!finite) {
      // a value that is infinite, or as bf16: the parts of it are not numbers; the row in plain f32 arithmetic
      const f4* q = reinterpret_cast<const f4*>(qbase + (size_t)qi * C3);
      float m = -INFINITY, l = 0.0f;
      f4 t{0.f, 0.f, 0.f, 0.f};
      for (int key = 0; key <= qi; ++key) {
        const f4* k = reinterpret_cast<const f4*>(kbase + (size_t)key * C3);
        float z = 0.0f;
#pragma unroll
        for (int i = 0; i < 16; ++i) z = fmaf(q[i].w, k[i].w, fmaf(q[i].z, k[i].z, fmaf(q[i].y, k[i].y, fmaf(q[i].x, k[i].x, z))));
        z *= 0.125f;
        if (z == -INFINITY) continue;  // (no weight; a row of nothing else ends as 0 / 0)
        const float m_new = fmaxf(m, z), keep = expf(m - m_new), w = expf(z - m_new);
        l = l * keep + w;
        t = t * keep + w * *reinterpret_cast<const f4*>(vbase + (size_t)key * C3 + d);
        m = m_new;
      }
      r = t / l;
    }
    if constexpr (CUT) store_cut4(out, cut_rows((int)gridDim.z * T), row, (size_t)h * 64 + d, r);
    else *reinterpret_cast<f4*>(out + row * C + h * 64 + d) = r;
  }
}

template <int QG, int KG>
void start(const float* qkv, int T, int C, int H, int P, float* kcache, float* vcache, float* out, hipStream_t s, int nseq,
           size_t kv_stride, int out_form) {
  const dim3 grid(H, (T + 32 * QG - 1) / (32 * QG), nseq), block(64 * QG * KG);
  if (out_form == FORM_CUT)
    hipLaunchKernelGGL((k_attn_prefill_cut<QG, KG, true>), grid, block, 0, s, qkv, T, C, P, kcache, vcache, out, kv_stride);
  else
    hipLaunchKernelGGL((k_attn_prefill_cut<QG, KG, false>), grid, block, 0, s, qkv, T, C, P, kcache, vcache, out, kv_stride);
}
}  // namespace

// Which block shape is the fastest, or 0 where k_attn_prefill64 is: by the blocks that there are to a CU, us of k_attn_prefill64
// and of the shape that is taken, on 256 CUs (whose blocks the lines below count; a part of the chip has its share).
//  - up to 32 positions it is one tile a sequence: equal or slower here (32 x 20, 25 heads 13.5 / 15.3);
//  - 128 queries a block where that fills the chip: 32 x 200, 25 heads 131 / 80; 32 x 512, 25 heads 490 / 265.  64 for sequences
//    that short (32 x 60, 25 heads 30.7 / 22.4), and where the longer blocks of fewer queries even out the CUs (4 x 700, 20
//    heads 97 / 66; 16 x 400, 12 heads 87 / 64, and 70 with 128);
//  - eight wavefronts a block, the keys in two or four shares, with fewer blocks: 16 x 100, 12 heads 19.9 / 14.6; 1000, 25
//    heads 62 / 43; 1024, 20 heads 49 / 39; 4 x 200, 12 heads 17.3 / 12.7;
//  - fewer still: k_attn_prefill64's blocks of 32 queries (1024, 12 heads 31 / 35; 200, 20 heads 10.4 / 11.6).
int attn_cut_shape(int T, int H, int nseq, int num_cus) {
  if (T <= 32) return 0;
  auto blocks = [&](int queries) { return (double)H * nseq * ((T + queries - 1) / queries) * 256.0 / num_cus; };
  const double nb128 = blocks(128), nb64 = blocks(64);
  if (T <= 64) return nb64 >= 192 ? 22 : 0;
  if (nb128 >= 320) return T > 256 && nb64 <= (T <= 512 ? 2800 : 1024) ? 22 : 41;
  if (nb128 >= 192) return T <= 400 ? 42 : 24;
  return nb64 >= (nseq > 1 ? 180 : 250) ? 24 : 0;
}

hipError_t launch_attn_prefill_cut(const float* qkv, int T, int C, int H, int P, float* kcache, float* vcache, float* out,
                                   hipStream_t s, int nseq, size_t kv_stride, int out_form, int shape) {
  if (shape == 41) start<4, 1>(qkv, T, C, H, P, kcache, vcache, out, s, nseq, kv_stride, out_form);
  else if (shape == 22) start<2, 2>(qkv, T, C, H, P, kcache, vcache, out, s, nseq, kv_stride, out_form);
  else if (shape == 42) start<4, 2>(qkv, T, C, H, P, kcache, vcache, out, s, nseq, kv_stride, out_form);
  else if (shape == 24) start<2, 4>(qkv, T, C, H, P, kcache, vcache, out, s, nseq, kv_stride, out_form);
  else return hipErrorInvalidValue;
  return hipGetLastError();
}

}  // namespace pgk
