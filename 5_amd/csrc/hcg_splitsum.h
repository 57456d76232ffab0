// hcg_splitsum.h -- K splits summed by the last workgroup of an output block
// (device code).
//
// A second launch that sums partials costs 3 to 6 us of GPU time, most of it
// the gap between launches, and 2.5 us of host time.  Where a block's partials
// are small the workgroup that finishes last sums them faster: each workgroup
// writes its partial through to the point that all XCDs' L2s share, waits for
// those stores (0.4 to 0.8 us), counts its arrival (0.4 us), and the last one
// loads the others' (about 1 us, plus 1 us per 100 KB).  It waits for nobody.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "hcg_tile.h"

namespace hcg {

typedef float split_f32x4 __attribute__((ext_vector_type(4)));

// Counters (32-bit, one per output block, zero between launches) lie 64 bytes
// apart, so that the blocks' atomics do not queue on one line (512 x 512 x
// 16384 in 32 tiles and 8 splits: 19.4 -> 18.6 us).
constexpr int kSplitCounterStride = 16;
constexpr int kMaxSummedSplits = 16;

// v: this thread's P pieces of split `split`'s partial of block `block` (of
// `blocks`).  The workspace holds [splits][blocks][P][THREADS] pieces: writer
// and reader are the same thread index, so any layout of v will do.  True in
// the last workgroup of the block to arrive, with v summed over the splits in
// the order 0, 1, ...; false in the others.  flag: an LDS word that no wave
// still uses when all have reached the first barrier here.  splits <=
// kMaxSummedSplits; the workspace stays below 2^31 bytes.
template <int P, int THREADS>
__device__ __forceinline__ bool sum_splits(split_f32x4 (&v)[P], __amdgpu_buffer_rsrc_t ws, int blocks, int block,
                                           int splits, int split, unsigned* counters, unsigned* flag) {
  constexpr int kAgent = 16;  // SC1: the cache policy of an agent-scope access
  const int tid = threadIdx.x;
  auto at = [&](int sp, int p) { return (((sp * blocks + block) * P + p) * THREADS + tid) * 16; };
#pragma unroll
  for (int p = 0; p < P; ++p)
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v[p]), ws, at(split, p), 0, kAgent);
  // Visible at agent scope once the stores have completed; only then is the
  // arrival counted.
  __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
  __syncthreads();
  unsigned* word = counters + block * kSplitCounterStride;
  if (tid == 0) *flag = __hip_atomic_fetch_add(word, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  if (*flag != (unsigned)(splits - 1)) return false;
  if (tid == 0) __hip_atomic_store(word, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  split_f32x4 own[P];
#pragma unroll
  for (int p = 0; p < P; ++p) own[p] = v[p];
  // Splits whose loads are in flight together (at most 32 of 16 bytes a thread).
  constexpr int kBatch = P >= 4 ? 32 / P : 8;
  for (int s0 = 0; s0 < splits; s0 += kBatch) {
    u32x4 part[kBatch][P];
#pragma unroll
    for (int q = 0; q < kBatch; ++q)
      if (s0 + q < splits && s0 + q != split) {
#pragma unroll
        for (int p = 0; p < P; ++p) part[q][p] = __builtin_amdgcn_raw_buffer_load_b128(ws, at(s0 + q, p), 0, kAgent);
      }
#pragma unroll
    for (int q = 0; q < kBatch; ++q)
      if (s0 + q < splits) {
#pragma unroll
        for (int p = 0; p < P; ++p) {
          const split_f32x4 x = s0 + q == split ? own[p] : __builtin_bit_cast(split_f32x4, part[q][p]);
          v[p] = s0 + q == 0 ? x : v[p] + x;
        }
      }
  }
  return true;
}

}  // namespace hcg
