// Weights on their way while a launch leaves most of the chip idle: its spare blocks read a word of every cache line that the
// next product will read, each on the die whose blocks will, and the product finds them in that die's cache.
#pragma once
#include <stddef.h>

#ifdef __HIPCC__
#include <hip/hip_runtime.h>
#define PG_HOST_DEVICE __host__ __device__ __forceinline__
#else
#define PG_HOST_DEVICE inline
#endif

namespace pgk {

// No weights to read ahead (a branch for them in the launches that have none cost 0.2 to 0.7 us each).
struct Nothing {};

constexpr unsigned kDies = 8;  // block i of a launch runs on die i % kDies, and each die has a cache (4 MB) of its own
constexpr unsigned kAheadLine = 128;

// Up to two matrices of `slabs` slabs of slab_bytes bytes, a multiple of 4 (whole matrices below 4 GB); block i of the product
// reads bytes [i * group_bytes, (i + 1) * group_bytes) of every slab.  (Rows one after the other: one slab.)  lines, words: cache
// lines of a group; a die's words of a slab.  blocks: spare blocks of the launch, a multiple of kDies (0: none).
struct Ahead {
  const void* at[2] = {nullptr, nullptr};
  unsigned slabs[2] = {0, 0}, slab_bytes[2] = {0, 0}, group_bytes[2] = {0, 0}, lines[2] = {1, 1}, words[2] = {1, 1};
  int blocks = 0;
  size_t total() const { return (size_t)slabs[0] * slab_bytes[0] + (size_t)slabs[1] * slab_bytes[1]; }
  void matrix(int k, const void* from, size_t n_slabs, size_t slab, size_t group) {
    at[k] = from;
    slabs[k] = (unsigned)n_slabs, slab_bytes[k] = (unsigned)slab, group_bytes[k] = (unsigned)group;
    lines[k] = (unsigned)((group + kAheadLine - 1) / kAheadLine);
    words[k] = (unsigned)(((slab + group - 1) / group + kDies - 1) / kDies) * lines[k];
  }
};

// Whether reading ahead pays, by the bytes of the product; us of a step, without and with.  Too few, and the product gains no more
// than the launch in front of it loses: 3.5 to 8 MB (c_attn and c_fc of width 768, bf16 rows, 16 sequences) 465 and 474, (1024)
// 953 and 958, 10 to 13 MB (1280) 1 % either way, a stack model 768 wide (5 MB) 173 and 180, 1280 (13 MB) 216 and 215.  15 to 20 MB (width
// 1600, bf16 rows, 16 sequences of 700 tokens) 3123 and 3083, stack model 1600 wide (20 MB) 248 and 239.  Too many for the eight
// caches: f32 rows, 31 to 41 MB (1600) 2796 and 2930.  Part of the columns or of the rows read ahead gave nothing: the product waits for
// the others.
constexpr size_t kAheadLeast = 14000000, kAheadMost = 24000000;
inline bool ahead_pays(size_t bytes) { return bytes >= kAheadLeast && bytes <= kAheadMost; }

// Where word w < a.words[k] of die `die` lies in a slab of matrix k, unless it would be behind the slab's end.
PG_HOST_DEVICE bool ahead_word(const Ahead& a, int k, unsigned die, unsigned w, unsigned* at) {
  const unsigned group = w / a.lines[k];
  *at = (group * kDies + die) * a.group_bytes[k] + (w - group * a.lines[k]) * kAheadLine;
  return *at + 4 <= a.slab_bytes[k];
}

#ifdef __HIPCC__
// Spare block `block` of a.blocks, `threads` threads; id: its number in the launch.
__device__ __forceinline__ void read_ahead(const Ahead& a, int block, unsigned id, unsigned threads) {
  constexpr int kAtOnce = 4;  // words of a thread in flight
  const unsigned die = id % kDies, all = (unsigned)a.blocks / kDies * threads;  // threads of a die
  const unsigned me = (unsigned)block / kDies * threads + threadIdx.x;
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    if (a.slabs[k] == 0) continue;
    const char* p = static_cast<const char*>(a.at[k]);
    unsigned v[kAtOnce];
    auto take = [&](unsigned slab, unsigned w, int q) __attribute__((always_inline)) {
      unsigned at;
      v[q] = 0;
      if (slab < a.slabs[k] && w < a.words[k] && ahead_word(a, k, die, w, &at)) v[q] = *reinterpret_cast<const unsigned*>(p + (slab * a.slab_bytes[k] + at));
    };
    auto wait = [&] __attribute__((always_inline)) {
#pragma unroll
      for (int q = 0; q < kAtOnce; ++q) asm volatile("" ::"v"(v[q]));
    };
    if (a.words[k] >= all) {
      for (unsigned slab = 0; slab < a.slabs[k]; ++slab)
        for (unsigned w = me; w < a.words[k]; w += kAtOnce * all) {
#pragma unroll
          for (int q = 0; q < kAtOnce; ++q) take(slab, w + q * all, q);
          wait();
        }
    } else {  // as many slabs side by side as there are threads for
      const unsigned beside = all / a.words[k], mine = me / a.words[k], w = me - mine * a.words[k];
      if (mine >= beside) continue;
      for (unsigned slab = mine; slab < a.slabs[k]; slab += kAtOnce * beside) {
#pragma unroll
        for (int q = 0; q < kAtOnce; ++q) take(slab + q * beside, w, q);
        wait();
      }
    }
  }
}
#endif

}  // namespace pgk
