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

// No weights to read ahead (a branch for them cost the reductions that have none 0.2 to 0.7 us each; beside mixers, which have blocks of
// several kinds anyway, it cost nothing: stack models 768 and 1280 wide, 24 tokens, 4512 and 4503 us, 5590 and 5590).
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

// Whether reading ahead behind a sum or beside mixers pays, by the bytes of the product; us of a step, or ms of 13 of them (*), without and with.
//  - Too few, and the product gains no more than the launch in front of it loses: 3.5 to 8 MB (c_attn and c_fc of width 768, bf16 rows, 16
//    sequences) 465 and 474, (1024) 953 and 958, a stack model 768 wide (5 MB) 173 and 180, 1280 (13 MB) 216 and 215, c_attn and c_fc of
//    1280 (9.8 and 13.1 MB), bf16 rows, 3 sequences 18.65* and 18.60, 16 20.24* and 19.99.
//  - 15 to 20 MB: width 1600, bf16 rows, 16 sequences of 700 tokens 3123 and 3083, a stack model 1600 wide (20 MB) 248 and 239; 1280, f32 rows
//    (c_attn, 19.7 MB), 16 sequences 23.2* and 22.8; 1728, bf16 rows (17.9 and 23.9 MB), 16 sequences, 12 layers, 8.84* and 8.48.
//  - Too many: f32 rows, 26.2 MB (1280) 22.91* and 23.07, 28.9 (1344) 8.66* and 8.78, 31 to 41 (1600) 2796 and 2930; bf16 rows, 27.6
//    (1856) 8.95* and 8.85.
// Part of the columns or of the rows read ahead gave nothing: the product waits for the others.
constexpr size_t kAheadLeast = 14000000, kAheadMost = 24000000;
inline bool ahead_pays(size_t bytes) { return bytes >= kAheadLeast && bytes <= kAheadMost; }

// Where word w < a.words[k] of die `die` lies in a slab of matrix k, unless it would be behind the slab's end.
PG_HOST_DEVICE bool ahead_word(const Ahead& a, int k, unsigned die, unsigned w, unsigned* at) {
  const unsigned group = w / a.lines[k];
  *at = (group * kDies + die) * a.group_bytes[k] + (w - group * a.lines[k]) * kAheadLine;
  return *at + 4 <= a.slab_bytes[k];
}

// What thread `tid` (of `threads`) of spare block `block` reads of matrix k; id: the block's number in the launch.  kAheadAtOnce times
// load(place in the matrix), then wait(what they gave), and so on.
constexpr int kAheadAtOnce = 4;  // words of a thread in flight
template <typename Load, typename Wait>
PG_HOST_DEVICE void ahead_words(const Ahead& a, int k, int block, unsigned id, unsigned tid, unsigned threads, Load load, Wait wait) {
  const unsigned die = id % kDies, all = (unsigned)a.blocks / kDies * threads;  // threads of a die
  const unsigned me = (unsigned)block / kDies * threads + tid;
  unsigned v[kAheadAtOnce];
  // (the load stands inside the condition: with the condition handed to it, every load was waited for before the next)
  auto take = [&](unsigned slab, unsigned w, int q) __attribute__((always_inline)) {
    unsigned at;
    v[q] = 0;
    if (slab < a.slabs[k] && w < a.words[k] && ahead_word(a, k, die, w, &at)) v[q] = load(slab * a.slab_bytes[k] + at);
  };
  if (a.words[k] >= all) {
    for (unsigned slab = 0; slab < a.slabs[k]; ++slab)
      for (unsigned w = me; w < a.words[k]; w += kAheadAtOnce * all) {
#pragma unroll
        for (int q = 0; q < kAheadAtOnce; ++q) take(slab, w + q * all, q);
        wait(v);
      }
  } else {  // as many slabs side by side as there are threads for
    const unsigned beside = all / a.words[k], mine = me / a.words[k], w = me - mine * a.words[k];
    if (mine >= beside) return;
    for (unsigned slab = mine; slab < a.slabs[k]; slab += kAheadAtOnce * beside) {
#pragma unroll
      for (int q = 0; q < kAheadAtOnce; ++q) take(slab + q * beside, w, q);
      wait(v);
    }
  }
}

#ifdef __HIPCC__
// Spare block `block` of a.blocks, `threads` threads; id: its number in the launch.
__device__ __forceinline__ void read_ahead(const Ahead& a, int block, unsigned id, unsigned threads) {
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    if (a.slabs[k] == 0) continue;
    const char* p = static_cast<const char*>(a.at[k]);
    auto load = [&](unsigned at) __attribute__((always_inline)) { return *reinterpret_cast<const unsigned*>(p + at); };
    auto wait = [](const unsigned (&v)[kAheadAtOnce]) __attribute__((always_inline)) {
#pragma unroll
      for (int q = 0; q < kAheadAtOnce; ++q) asm volatile("" ::"v"(v[q]));
    };
    ahead_words(a, k, block, id, threadIdx.x, threads, load, wait);
  }
}
#endif

}  // namespace pgk
