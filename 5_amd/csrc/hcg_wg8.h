// hcg_wg8.h -- the eight-wave tiled GEMM kernel of gfx950 (device code).
//
// C tile of TM x TN by one 512-thread workgroup: WM x WN waves over the
// tile and WK = 8 / (WM * WN) groups of waves over K, each wave
// (TM/WM) x (TN/WN) of v_mfma_f32_32x32x16 accumulators.  K advances KS
// (64 or 32) at a time through a STAGES-deep LDS ring filled by
// buffer_load_dwordx4 ... lds; group kg of the WK multiplies k rows
// [kg * KS/WK, (kg + 1) * KS/WK) of every stage and the groups' sums are
// added once, in the epilogue, in the order kg = 0, 1, ...
//
// For shapes whose 256-row tiles would leave most CUs idle.  There one
// workgroup per CU of four waves (gemm_dma_kernel's 128x128 tile, two 32-wide
// K tiles ahead) waited on its loads and on LDS: four waves read LDS at 125
// of the 239 bytes per cycle that eight reach, and 64x64 of accumulators per
// wave need 128 per cycle of MFMA issue.  Eight waves (two per SIMD) and 96
// KB in flight per CU took 2048^3 bf16 from 23.9 to 18.8 us; per-workgroup
// timestamps: K loop 12.0 us (14.0 on a slower board), 693 (670) cycles per
// 64-wide step against 512 of MFMA issue, at 1.95 (1.69) GHz, prologue 1.7,
// epilogue 2.0 (16 MiB of C); 128x256 tiles on 4096 x 2048 x 2048 24.8 us, 1380
// cycles against 1024.  Two K groups (WK = 2) keep the wave tile square at 64x64
// where the workgroup's is 128x128: 64 KB of LDS reads per 64-wide step, against
// 96 KB for eight 64x32 wave tiles.  Small tiles are bound by the DMA (64 bytes
// per cycle per CU): 64x64 takes 344 to 396 cycles per step, 256 of them DMA and
// 128 MFMA, and wins by filling CUs: 1024^3 12.3 -> 6.5 us, 512^3 6.7 -> 4.2.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "hcg_gemm.h"
#include "hcg_splitsum.h"
#include "hcg_tile.h"

namespace hcg {
namespace wg8 {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

constexpr int kThreads = 512;
constexpr int kWaves = 8;
struct Args {
  const uint16_t* A;
  const uint16_t* B;
  float* C;
  int lda, ldb;  // elements between consecutive rows as stored
  int64_t ldc;
  int M, N, K;
  int tiles_m, tiles_n;
  int a_bytes, b_bytes;  // buffer extents for the hardware range check
  bool c_vec;            // C rows are 16-byte aligned at every 4th column
  // Split-K (splits > 1): split s of a tile covers k [s * kchunk,
  // (s + 1) * kchunk).  With counters (one per tile, all zero between
  // launches) the workgroups of a tile sum their partials themselves, in the
  // order of s, through ws [splits][tiles][TM * TN] of ws_bytes < 2^31;
  // without, split s writes ws + s * M * N (row stride N) and a second
  // launch sums.
  int splits, kchunk;
  float* ws;
  bool ws_vec;  // N is a multiple of 4 (16-byte partial rows)
  unsigned* counters;
  int ws_bytes;
#ifdef HCG_STAMPS
  int stamp_slot;
#endif
};

// Tiles whose split partials the workgroups sum themselves (hcg_splitsum.h): a
// thread holds its own pieces and a batch of others' in registers (128x256
// would spill).
constexpr bool can_fuse(int tm, int tn) { return tm * tn <= 128 * 128; }

template <int N>
__device__ __forceinline__ void wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt(0x0f70 | (N & 15) | ((N >> 4) << 14));
}
__device__ __forceinline__ void wait_lgkm() { __builtin_amdgcn_s_waitcnt(0xc07f); }

template <int DT>
__device__ __forceinline__ f32x16 mfma(u32x4 a, u32x4 b, f32x16 c) {
  if constexpr (DT == HCG_F16)
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0,
                                                  0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                   0, 0);
}

// Each stage of a ring is an LDS object of its own and every access names
// its stage at compile time, so the compiler can tell a DMA into one stage
// from reads of another and does not serialize them.
template <int BYTES, int S>
__device__ __forceinline__ unsigned char* ring_stage() {
  __shared__ __attribute__((aligned(1024))) unsigned char buf[BYTES];
  return buf;
}

// blockIdx -> (K split, output tile): each XCD (id % 8) takes a contiguous
// run of units, split by split and within a split by tile in groups of 4
// tile rows, so that the workgroups sharing an L2 share A rows and B columns
// of the same K range (512 x 512 x 16384 in 64x128 tiles and 8 splits: 13.1
// us this way, 17.9 with every XCD taking the same tiles of each split, which
// reads A and B through 8 L2s instead of one).
__device__ __forceinline__ void unit_of(int tiles_m, int tiles_n, int splits, int wg, int& split, int& tm, int& tn) {
  const int nt = tiles_m * tiles_n, n = nt * splits;
  const int per = n >> 3, rem = n & 7, xcd = wg & 7, idx = wg >> 3;
  const int unit = xcd < rem ? xcd * (per + 1) + idx : rem * (per + 1) + (xcd - rem) * per + idx;
  split = unit / nt;
  const int logical = unit - split * nt;
  const int span = 4 * tiles_n;
  const int group = logical / span, first = group * 4;
  const int size = min(tiles_m - first, 4);
  const int in_group = logical - group * span;
  tm = first + in_group % size;
  tn = in_group / size;
}

// One operand's part of a stage: T rows of the output's M (A) or N (B) by
// KS of K.  KC (K-contiguous: A as stored, B stored transposed): LDS rows
// of KS elements, one per output row; fragments are one ds_read_b128.
// Otherwise (K rows of T contiguous output columns: B as stored, A stored
// transposed): LDS rows of T elements, one per k; fragments are two
// ds_read_b64_tr_b16, which hand lane i of a 16-lane group element i%4 of
// source lanes 4j + i/4.  Either way a lane's fragment holds 8 consecutive
// k of one output row, the MFMA operand layout.  The 16-byte chunks of an
// LDS row are XOR-swizzled so that the 16 lanes that an LDS cycle serves
// cover all 64 banks.
template <int T, int KS, bool KC>
struct Operand {
  static constexpr int kBytes = T * KS * 2;
  static constexpr int kInst = kBytes / 1024 / kWaves;  // DMA instructions per wave per stage
  static constexpr int kRowBytes = KC ? KS * 2 : T * 2;
  static constexpr int kChunks = kRowBytes / 16;        // chunks per LDS row
  static constexpr int kRowsPerInst = 64 / kChunks;
  static_assert(kInst >= 1, "a stage is at least one DMA instruction per wave");
  static_assert(KS == 64 || KS == 32, "K step");

  static __device__ __forceinline__ int swz(int row, int c) {
    if constexpr (KC) {
      if constexpr (KS == 64) return c ^ ((row >> 1) & 7);
      return c ^ ((row >> 1) & 3) ^ ((row >> 3) & 1);
    } else {
      const int m = row & 3;
      if constexpr (T == 64) return c ^ ((m >> 1) * 4);
      return c ^ ((m >> 1) * 10 + (m & 1) * 4);
    }
  }

  int off[kInst];  // byte offset of the lane's chunk at k = 0
  int key[kInst];  // KC: the chunk's first k; else its k row (never below K: a dead lane)

  // base: the tile's first output row; extent: output rows; ld, bytes: the
  // stored matrix.  Lanes past the extent read zeros (offset at the end of
  // the buffer whatever the K advance).
  __device__ __forceinline__ void init(int wave, int lane, int base, int extent, int ld, int bytes) {
#pragma unroll
    for (int i = 0; i < kInst; ++i) {
      const int row = (wave * kInst + i) * kRowsPerInst + lane / kChunks;
      const int c = swz(row, lane % kChunks);
      if constexpr (KC) {
        const bool live = base + row < extent;
        off[i] = live ? ((base + row) * ld + c * 8) * 2 : bytes;
        key[i] = live ? c * 8 : 0x3fffffff;
      } else {
        const bool live = base + c * 8 < extent;
        off[i] = live ? (row * ld + base + c * 8) * 2 : bytes;
        key[i] = live ? row : 0x3fffffff;
      }
    }
  }

  // Stage rows k0 .. k0 + KS - 1 into st.  full: the tile lies inside K.
  template <bool FULL>
  __device__ __forceinline__ void issue(__amdgpu_buffer_rsrc_t r, unsigned char* st, int wave, int k0, int K,
                                        int ld) const {
    const int adv = KC ? k0 * 2 : (int)((uint32_t)k0 * (uint32_t)ld * 2u);
#pragma unroll
    for (int i = 0; i < kInst; ++i) {
      lds_void* dst = (lds_void*)(st + (wave * kInst + i) * 1024);
      if constexpr (FULL)
        dma16(r, dst, off[i], adv);
      else
        dma16(r, dst, dma_offset(k0 + key[i] < K, (int)((uint32_t)off[i] + (uint32_t)adv)));
    }
  }

  // Fragment addresses: 32-row block b (of the wave's first row `first`) and
  // 16-wide K step s (from the wave's first k `k0`).
  int fa;
  int fb[2];
  __device__ __forceinline__ void frag_init(int lane, int first, int k0) {
    if constexpr (KC) {
      const int row = first + (lane & 31);
      fa = row * kRowBytes + swz(row, k0 / 8 + (lane >> 5)) * 16;
    } else {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int sl = lane & 15, grp = lane >> 4;
        const int krow = k0 + 8 * (grp >> 1) + 4 * h + (sl >> 2);
        const int col = first + 16 * (grp & 1) + 4 * (sl & 3);
        fb[h] = krow * kRowBytes + swz(krow, col >> 3) * 16 + (col & 7) * 2;
      }
    }
  }
  // (The K step and the block index are disjoint bits of the chunk index, so
  // they commute with the swizzle's XOR.)
  __device__ __forceinline__ u32x4 frag(const unsigned char* st, int b, int s) const {
    if constexpr (KC) {
      return *reinterpret_cast<const u32x4*>(st + (fa ^ (s * 32)) + b * 32 * kRowBytes);
    } else {
      const int x = s * 16 * kRowBytes;
      const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (__attribute__((address_space(3))) s16x4*)(st + (fb[0] ^ (b * 64)) + x));
      const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (__attribute__((address_space(3))) s16x4*)(st + (fb[1] ^ (b * 64)) + x));
      const uint64_t l = __builtin_bit_cast(uint64_t, lo), h = __builtin_bit_cast(uint64_t, hi);
      return u32x4{(uint32_t)l, (uint32_t)(l >> 32), (uint32_t)h, (uint32_t)(h >> 32)};
    }
  }
};

template <int S>
using StageC = std::integral_constant<int, S>;

// AKC: A is stored with K contiguous (row-major M x K), else as K x M.
// BKC: B is stored transposed (N x K), else as K x N.  KT: K is not a
// multiple of 8 and an operand is K-contiguous; its chunk holding k = K - 1
// also brings elements past K (the next row, or padding that may hold NaN),
// which are cleared in the fragments of the last stage.
template <int DT, int TM, int TN, int WM, int WN, int KS, int STAGES, bool AKC, bool BKC, bool KT>
__global__ __launch_bounds__(kThreads, 1) void gemm_wg8_kernel(Args g) {
  constexpr int WK = kWaves / (WM * WN);
  static_assert(WM * WN * WK == kWaves, "eight waves");
  constexpr int MI = TM / WM / 32, NI = TN / WN / 32;
  static_assert(MI >= 1 && NI >= 1, "wave tile");
  constexpr int KW = KS / WK;     // k per wave per stage
  constexpr int NSUB = KW / 16;   // 16-wide K steps per wave per stage
  static_assert(NSUB == 2 || NSUB == 4, "K steps");
  static_assert(STAGES == 3 || STAGES == 4, "stages");
  using OpA = Operand<TM, KS, AKC>;
  using OpB = Operand<TN, KS, BKC>;
  constexpr int kStageBytes = OpA::kBytes + OpB::kBytes;
  constexpr int kDma = OpA::kInst + OpB::kInst;

  WgStamps stamps(HCG_STAMP_SLOT(g));
  stamps.mark(0);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = wave / (WM * WN), wm = (wave / WN) % WM, wn = wave % WN;

  int split, tm, tn;
  unit_of(g.tiles_m, g.tiles_n, g.splits, blockIdx.x, split, tm, tn);
  if (g.splits > 1) {
    const int kbeg = split * g.kchunk;
    const int64_t ka = AKC ? (int64_t)kbeg : (int64_t)kbeg * g.lda, kb = BKC ? (int64_t)kbeg : (int64_t)kbeg * g.ldb;
    g.A += ka;
    g.B += kb;
    g.a_bytes -= (int)(ka * 2);
    g.b_bytes -= (int)(kb * 2);
    g.K = min(g.K - kbeg, g.kchunk);
    if (!can_fuse(TM, TN) || g.counters == nullptr) {
      g.C = g.ws + (int64_t)split * g.M * g.N;
      g.ldc = g.N;
      g.c_vec = g.ws_vec;
    }
  }
  const int m0 = tm * TM, n0 = tn * TN;
  const int nk = (g.K + KS - 1) / KS;

  const __amdgpu_buffer_rsrc_t ra = make_rsrc(g.A, g.a_bytes), rb = make_rsrc(g.B, g.b_bytes);
  OpA a;
  OpB b;
  a.init(wave, lane, m0, g.M, g.lda, g.a_bytes);
  b.init(wave, lane, n0, g.N, g.ldb, g.b_bytes);
  a.frag_init(lane, wm * (TM / WM), kg * KW);
  b.frag_init(lane, wn * (TN / WN), kg * KW);

  f32x16 acc[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) acc[i][j] = f32x16{};

  u32x4 fa[2][MI], fb[2][NI];
  auto issue_a = [&](auto sc, auto full, int kt) {
    a.template issue<decltype(full)::value>(ra, ring_stage<kStageBytes, decltype(sc)::value>(), wave, kt * KS, g.K,
                                            g.lda);
  };
  auto issue_b = [&](auto sc, auto full, int kt) {
    b.template issue<decltype(full)::value>(rb, ring_stage<kStageBytes, decltype(sc)::value>() + OpA::kBytes, wave,
                                            kt * KS, g.K, g.ldb);
  };
  auto read = [&](auto sc, int s, auto mask, int kt) {
    constexpr int S = decltype(sc)::value;
    const unsigned char* st = ring_stage<kStageBytes, S>();
#pragma unroll
    for (int i = 0; i < MI; ++i) fa[s & 1][i] = a.frag(st, i, s);
#pragma unroll
    for (int j = 0; j < NI; ++j) fb[s & 1][j] = b.frag(st + OpA::kBytes, j, s);
    if constexpr (decltype(mask)::value) {
      const int v = min(max(g.K - (kt * KS + kg * KW + s * 16 + (lane >> 5) * 8), 0), 8);
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const uint32_t m = (2 * w < v ? 0x0000ffffu : 0u) | (2 * w + 1 < v ? 0xffff0000u : 0u);
        if constexpr (AKC) {
#pragma unroll
          for (int i = 0; i < MI; ++i) fa[s & 1][i][w] &= m;
        }
        if constexpr (BKC) {
#pragma unroll
          for (int j = 0; j < NI; ++j) fb[s & 1][j][w] &= m;
        }
      }
    }
  };
  auto multiply = [&](int s) {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NI; ++j) acc[i][j] = mfma<DT>(fa[s & 1][i], fb[s & 1][j], acc[i][j]);
  };
  // Instruction order of one 16-wide K step: fragment reads behind the first
  // MFMAs, the step's DMA loads spread over the rest.
  constexpr int kReads = MI * (AKC ? 1 : 2) + NI * (BKC ? 1 : 2);
  constexpr int kMfmas = MI * NI;
  auto schedule = [&](auto nv_c) {
    constexpr int nv = decltype(nv_c)::value;
    constexpr int per = (kReads + kMfmas - 1) / kMfmas > 2 ? (kReads + kMfmas - 1) / kMfmas : 2;
#pragma unroll
    for (int m = 0; m < kMfmas; ++m) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      if (per * m < kReads) __builtin_amdgcn_sched_group_barrier(0x100, per, 0);
      int loads = 0;
#pragma unroll
      for (int v = 0; v < nv; ++v) loads += (v * kMfmas / (nv > 0 ? nv : 1) == m) ? 1 : 0;
      if (loads == 1) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
      if (loads == 2) __builtin_amdgcn_sched_group_barrier(0x020, 2, 0);
      if (loads == 4) __builtin_amdgcn_sched_group_barrier(0x020, 4, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  // One stage.  On entry fa[0] / fb[0] hold its first K step, on exit the
  // next stage's.  Before the barrier the B part of stage kt + STAGES - 1 is
  // requested, after it (every wave is past its reads of stage kt) the A
  // part of kt + STAGES into the stage just freed.
  auto iteration = [&](auto sc, auto full, int kt) {
    constexpr int S = decltype(sc)::value;
    using Mask = std::integral_constant<bool, KT && !decltype(full)::value>;
    constexpr int kPre = NSUB - 1;  // K steps before the barrier
#pragma unroll
    for (int s = 0; s < kPre; ++s) {
      read(sc, s + 1, Mask{}, kt);
      if (s == 0) issue_b(StageC<(S + STAGES - 1) % STAGES>{}, full, kt + STAGES - 1);
      multiply(s);
      if (s == 0)
        schedule(std::integral_constant<int, OpB::kInst>{});
      else
        schedule(std::integral_constant<int, 0>{});
    }
    wait_vm<(STAGES - 2) * kDma>();
    wait_lgkm();
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    read(StageC<(S + 1) % STAGES>{}, 0, Mask{}, kt + 1);
    issue_a(sc, full, kt + STAGES);
    multiply(NSUB - 1);
    schedule(std::integral_constant<int, OpA::kInst>{});
  };

  using Full = std::true_type;
  using Checked = std::false_type;
  issue_a(StageC<0>{}, Checked{}, 0);
  issue_b(StageC<0>{}, Checked{}, 0);
  issue_a(StageC<1>{}, Checked{}, 1);
  issue_b(StageC<1>{}, Checked{}, 1);
  if constexpr (STAGES > 3) {
    issue_a(StageC<2>{}, Checked{}, 2);
    issue_b(StageC<2>{}, Checked{}, 2);
  }
  issue_a(StageC<STAGES - 1>{}, Checked{}, STAGES - 1);
  wait_vm<(STAGES - 2) * kDma + OpA::kInst>();
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  stamps.mark(1);
  read(StageC<0>{}, 0, std::integral_constant<bool, KT>{}, 0);

  int kt = 0;
  const int nfull = g.K / KS;
  for (; kt + 2 * STAGES <= nfull; kt += STAGES) {
    iteration(StageC<0>{}, Full{}, kt);
    iteration(StageC<1>{}, Full{}, kt + 1);
    iteration(StageC<2>{}, Full{}, kt + 2);
    if constexpr (STAGES > 3) iteration(StageC<3 % STAGES>{}, Full{}, kt + 3);
  }
  for (; kt + STAGES <= nk; kt += STAGES) {
    iteration(StageC<0>{}, Checked{}, kt);
    iteration(StageC<1>{}, Checked{}, kt + 1);
    iteration(StageC<2>{}, Checked{}, kt + 2);
    if constexpr (STAGES > 3) iteration(StageC<3 % STAGES>{}, Checked{}, kt + 3);
  }
  if (kt < nk) iteration(StageC<0>{}, Checked{}, kt++);
  if (kt < nk) iteration(StageC<1>{}, Checked{}, kt++);
  if constexpr (STAGES > 3)
    if (kt < nk) iteration(StageC<2>{}, Checked{}, kt++);
  wait_vm<0>();  // no DMA may still be writing LDS
  stamps.mark(2);
  __builtin_amdgcn_s_barrier();  // every wave is done reading the stages

  // Epilogue: 16 rows of every wave row at a time (WM * 16 x TN floats) go
  // through LDS, one copy per K group, and are summed and stored by all
  // threads in whole 16-byte pieces.  Accumulator layout: register r of lane
  // l holds row 8 (r/4) + 4 (l/32) + r%4, column l%32.  Columns are XORed
  // with 32 in rows whose bit 2 is set, so the two halves of a wave's write
  // cover different banks.
  constexpr int kEpBytes = WM * 16 * TN * 4;
  static_assert(kEpBytes <= kStageBytes && WK <= STAGES, "epilogue staging");
  constexpr bool kTwo = 2 * WK <= STAGES;  // alternate staging: one barrier per block
  constexpr int kPieces = WM * 16 * TN / 4 / kThreads;
  static_assert(kPieces >= 1, "epilogue pieces");
  constexpr int kMine = 2 * MI * kPieces;  // pieces per thread
  const bool full_tile = g.c_vec && m0 + TM <= g.M && n0 + TN <= g.N;
  const bool vec_edge = g.c_vec && (g.N & 3) == 0;
  const bool fused = can_fuse(TM, TN) && g.splits > 1 && g.counters != nullptr;
  auto store_piece = [&](f32x4 v, int piece) {
    const int idx = piece % kPieces * kThreads + tid, block = piece / kPieces;
    const int row = idx / (TN / 4), col = (idx % (TN / 4)) * 4;
    const int grow = m0 + (row >> 4) * (TM / WM) + block * 16 + (row & 15), gcol = n0 + col;
    float* dst = g.C + (int64_t)grow * g.ldc + gcol;
    if (full_tile) {
      __builtin_nontemporal_store(v, reinterpret_cast<f32x4*>(dst));
    } else if (vec_edge) {
      if (grow < g.M && gcol < g.N) __builtin_nontemporal_store(v, reinterpret_cast<f32x4*>(dst));
    } else if (grow < g.M) {
      if (gcol + 3 < g.N) {
        *reinterpret_cast<f32x4u*>(dst) = v;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (gcol + e < g.N) dst[e] = v[e];
      }
    }
  };
  f32x4 mine[kMine];
  auto ep_block = [&](auto ic) {
    constexpr int I = decltype(ic)::value;
    constexpr int mi = I / 2, hh = I % 2;
    constexpr int s0 = kTwo ? (I & 1) * WK : 0;
    auto stage_of = [&](int q) -> float* {
      if (WK > 1 && q == 1) return reinterpret_cast<float*>(ring_stage<kStageBytes, (s0 + 1) % STAGES>());
      return reinterpret_cast<float*>(ring_stage<kStageBytes, s0>());
    };
    static_assert(WK <= 2, "K groups");
    if (!kTwo && I > 0) __syncthreads();
    float* ep = stage_of(kg);
#pragma unroll
    for (int ni = 0; ni < NI; ++ni)
#pragma unroll
      for (int r = 8 * hh; r < 8 * hh + 8; ++r) {
        const int row = wm * 16 + ((r >> 2) & 1) * 8 + (lane >> 5) * 4 + (r & 3);
        const int col = wn * (TN / WN) + ni * 32 + (lane & 31);
        ep[row * TN + (col ^ ((lane >> 5) * 32))] = acc[mi][ni][r];
      }
    __syncthreads();
#pragma unroll
    for (int p = 0; p < kPieces; ++p) {
      const int idx = p * kThreads + tid;
      const int row = idx / (TN / 4), col = (idx % (TN / 4)) * 4;
      const int at = row * TN + (col ^ ((row & 4) * 8));
      f32x4 v = *reinterpret_cast<const f32x4*>(stage_of(0) + at);
      if constexpr (WK > 1) v += *reinterpret_cast<const f32x4*>(stage_of(1) + at);
      mine[I * kPieces + p] = v;
    }
    if (!fused) {
#pragma unroll
      for (int p = 0; p < kPieces; ++p) store_piece(mine[I * kPieces + p], I * kPieces + p);
    }
  };
  ep_block(StageC<0>{});
  ep_block(StageC<1>{});
  if constexpr (MI > 1) {
    ep_block(StageC<2>{});
    ep_block(StageC<3>{});
  }
  if constexpr (MI > 2) {
    ep_block(StageC<4>{});
    ep_block(StageC<5>{});
  }
  if constexpr (MI > 3) {
    ep_block(StageC<6>{});
    ep_block(StageC<7>{});
  }
  if constexpr (can_fuse(TM, TN)) {
    if (fused && sum_splits<kMine, kThreads>(mine, make_rsrc(g.ws, g.ws_bytes), g.tiles_m * g.tiles_n,
                                             tm * g.tiles_n + tn, g.splits, split, g.counters,
                                             reinterpret_cast<unsigned*>(ring_stage<kStageBytes, STAGES - 1>()))) {
#pragma unroll
      for (int p = 0; p < kMine; ++p) store_piece(mine[p], p);
    }
  }
  stamps.write();
}

}  // namespace wg8
}  // namespace hcg
