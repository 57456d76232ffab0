// hcg_tile.hip -- masked tile gather / scatter on gfx950: the hc DSL's
// group.load(view, shape=) / group.load(view, mask=), with_inactive(fill),
// .mask and group.store(view, tile) over batches of tiles, built on the
// primitives of hcg_tile.h (the tail machinery of the GEMM kernels).
//
// Reference semantics: hc/simulator.py:1304-1357 (_load_value,
// _load_masked, _copy_loaded_value: the in-bounds overlap is copied, the
// rest of the tile is inactive), hc/simulator.py:1416-1458 (_store_value,
// _store_from_value: only active elements inside the target view are
// written), doc/langref.md:530-596 (masking, with_inactive, .mask).
//
// Bound: HBM (copies).  One thread moves one chunk of 16 bytes of one tile
// row (8, 4 or 2 elements): a chunk wholly inside the view moves as one
// vector access at the elements' own alignment (rows of a view need not be
// 16-byte aligned, and gfx950 takes unaligned global accesses), its activity
// as one word; edge chunks go element by element, and elements outside the
// view are never read or written.  Per-element accesses for rows that are not
// 16-byte aligned, byte stores of the activity and 64-bit divisions per chunk
// made the form before this one instruction-bound: the 64x64 tiles of a tight
// 4095 x 3001 f16 matrix (61 MB each way) gather in 21.0 -> 14.8 us and scatter
// in 29.6 -> 16.4, and in 11.4 and 15.0 with each XCD on neighbouring tiles
// (block_of).  Four chunks per thread, all loads first, did not help (16.0 and
// 17.4 without the mapping): latency is covered by the waves in flight.

#include <hip/hip_runtime.h>

#include <stdint.h>

#include <type_traits>

#include "hcg_runtime.h"
#include "hcg_tile.h"
#include "hcg_tile_ops.h"

namespace {

struct TileJob {
  const void* src;  // load: source view; store: unused
  void* dst;        // store: target view; load: unused
  int64_t ld;       // view row stride, elements
  int64_t rows, cols;
  const int64_t* origins;  // [ntiles][2] = (row0, col0)
  int64_t ntiles, th, tw;
  int64_t chunks_per_row;  // ceil(tw / elements per chunk)
  int64_t total_chunks;    // ntiles * th * chunks_per_row
  const uint8_t* mask_in;  // load: mask= operand; store: the tile's activity (NULL: all active)
  const void* tiles_in;    // store: the tiles
  void* tiles_out;         // load: the tiles
  uint8_t* mask_out;       // load: the tiles' activity (may be NULL)
  uint64_t fill_bits;      // load: with_inactive value, low sizeof(T) bytes
};

// Chunk index -> tile, row and first column in the tile.  I: uint32_t when
// every index fits (a 64-bit division costs about as much as the rest of a
// chunk's work), else int64_t.
template <typename T, typename I>
__device__ __forceinline__ void decompose(const TileJob& j, I idx, int64_t& t, int64_t& r, int64_t& c0) {
  const I per = (I)j.chunks_per_row, th = (I)j.th;
  const I row_id = idx / per;  // t * th + r
  const I tile = row_id / th;
  c0 = (int64_t)(idx - row_id * per) * (16 / (int64_t)sizeof(T));
  t = (int64_t)tile;
  r = (int64_t)(row_id - tile * th);
}

// 16 bytes, and one byte per element of a chunk, at element alignment.
template <typename T>
struct Chunk {
  static constexpr int kN = 16 / sizeof(T);
  union {
    hcg::u32x4 v;
    T e[kN];
  };
  // Activity bytes of a chunk (kN of 8, 4 or 2 bytes).
  typedef std::conditional_t<kN == 8, uint64_t, std::conditional_t<kN == 4, uint32_t, uint16_t>> Bytes;

  __device__ __forceinline__ void load(const T* p) { __builtin_memcpy(&v, p, 16); }
  __device__ __forceinline__ void store(T* p) const { __builtin_memcpy(p, &v, 16); }
};

// Bits of the elements whose activity byte is nonzero.
template <typename T>
__device__ __forceinline__ uint32_t mask_bits(const uint8_t* m, int n) {
  constexpr int kN = Chunk<T>::kN;
  uint32_t bits = 0;
  if (n == kN) {
    typename Chunk<T>::Bytes b;
    __builtin_memcpy(&b, m, sizeof b);
    const uint64_t w = b;
#pragma unroll
    for (int e = 0; e < kN; ++e) bits |= ((w >> (8 * e)) & 0xff) ? 1u << e : 0u;
  } else {
#pragma unroll
    for (int e = 0; e < kN; ++e)
      if (e < n && m[e]) bits |= 1u << e;
  }
  return bits;
}

// Workgroup -> block of 256 chunks: workgroups go round-robin over the 8 XCDs
// (id % 8), so each XCD takes a contiguous run of blocks -- with rows that are
// not line-aligned, neighbouring tiles share lines of the view, and one L2
// then merges them.
__device__ __forceinline__ int64_t block_of(unsigned wg, unsigned grid) {
  const unsigned per = grid >> 3, rem = grid & 7, x = wg & 7, i = wg >> 3;
  return x < rem ? (int64_t)x * (per + 1) + i : (int64_t)rem * (per + 1) + (int64_t)(x - rem) * per + i;
}

template <typename T, typename I>
__global__ __launch_bounds__(256) void tile_load_kernel(TileJob j) {
  constexpr int kN = Chunk<T>::kN;
  constexpr uint32_t kAll = (1u << kN) - 1u;
  T fill;
  __builtin_memcpy(&fill, &j.fill_bits, sizeof(T));
  for (int64_t at = block_of(blockIdx.x, gridDim.x) * 256 + threadIdx.x; at < j.total_chunks;
       at += (int64_t)gridDim.x * 256) {
    int64_t t, r, c0;
    decompose<T, I>(j, (I)at, t, r, c0);
    const int n = (int)min((int64_t)kN, j.tw - c0);
    const int64_t row = hcg::tile_coord(j.origins[2 * t], r);
    const int64_t col = hcg::tile_coord(j.origins[2 * t + 1], c0);
    const int64_t out_off = (t * j.th + r) * j.tw + c0;
    const bool whole = n == kN && hcg::chunk_inside(row, j.rows, col, j.cols, kN);
    uint32_t active = whole ? kAll : hcg::chunk_active_bits(row, j.rows, col, j.cols, n);
    if (j.mask_in) active &= mask_bits<T>(j.mask_in + out_off, n);
    // Rows outside the view are never addressed (active is 0 for them).
    const T* p = static_cast<const T*>(j.src) + (active ? row * j.ld + col : 0);
    Chunk<T> c;
    if (whole && active) {
      c.load(p);
      if (active != kAll) {
#pragma unroll
        for (int e = 0; e < kN; ++e)
          if (!((active >> e) & 1u)) c.e[e] = fill;
      }
    } else {
#pragma unroll
      for (int e = 0; e < kN; ++e) c.e[e] = ((active >> e) & 1u) ? p[e] : fill;
    }
    T* out = static_cast<T*>(j.tiles_out) + out_off;
    uint8_t* om = j.mask_out ? j.mask_out + out_off : nullptr;
    if (n == kN) {
      c.store(out);
      if (om) {
        uint64_t w = 0;
#pragma unroll
        for (int e = 0; e < kN; ++e) w |= (uint64_t)((active >> e) & 1u) << (8 * e);
        const typename Chunk<T>::Bytes b = (typename Chunk<T>::Bytes)w;
        __builtin_memcpy(om, &b, sizeof b);
      }
    } else {
#pragma unroll
      for (int e = 0; e < kN; ++e)
        if (e < n) {
          out[e] = c.e[e];
          if (om) om[e] = (active >> e) & 1u;
        }
    }
  }
}

template <typename T, typename I>
__global__ __launch_bounds__(256) void tile_store_kernel(TileJob j) {
  constexpr int kN = Chunk<T>::kN;
  constexpr uint32_t kAll = (1u << kN) - 1u;
  for (int64_t at = block_of(blockIdx.x, gridDim.x) * 256 + threadIdx.x; at < j.total_chunks;
       at += (int64_t)gridDim.x * 256) {
    int64_t t, r, c0;
    decompose<T, I>(j, (I)at, t, r, c0);
    const int n = (int)min((int64_t)kN, j.tw - c0);
    const int64_t row = hcg::tile_coord(j.origins[2 * t], r);
    const int64_t col = hcg::tile_coord(j.origins[2 * t + 1], c0);
    const int64_t in_off = (t * j.th + r) * j.tw + c0;
    const bool whole = n == kN && hcg::chunk_inside(row, j.rows, col, j.cols, kN);
    uint32_t write = whole ? kAll : hcg::chunk_active_bits(row, j.rows, col, j.cols, n);
    if (write == 0) continue;
    const T* in = static_cast<const T*>(j.tiles_in) + in_off;
    Chunk<T> c;
    if (n == kN) {
      c.load(in);  // beside the mask's load: a tile's chunk is always readable
    } else {
#pragma unroll
      for (int e = 0; e < kN; ++e)
        if (e < n) c.e[e] = in[e];
    }
    if (j.mask_in) write &= mask_bits<T>(j.mask_in + in_off, n);
    if (write == 0) continue;
    T* p = static_cast<T*>(j.dst) + row * j.ld + col;
    if (write == kAll) {
      c.store(p);
    } else {
#pragma unroll
      for (int e = 0; e < kN; ++e)
        if ((write >> e) & 1u) p[e] = c.e[e];
    }
  }
}

template <typename T>
void run_load(const TileJob& j, unsigned grid, hipStream_t s) {
  if (j.total_chunks <= 0x7fffffff)
    tile_load_kernel<T, uint32_t><<<grid, 256, 0, s>>>(j);
  else
    tile_load_kernel<T, int64_t><<<grid, 256, 0, s>>>(j);
}
template <typename T>
void run_store(const TileJob& j, unsigned grid, hipStream_t s) {
  if (j.total_chunks <= 0x7fffffff)
    tile_store_kernel<T, uint32_t><<<grid, 256, 0, s>>>(j);
  else
    tile_store_kernel<T, int64_t><<<grid, 256, 0, s>>>(j);
}

// Argument checks shared by both entry points; fills the geometry of j.
int prepare(int elem_bytes, int64_t ld, int64_t rows, int64_t cols, const void* view, const int64_t* origins,
            int64_t ntiles, int64_t th, int64_t tw, const char* what, TileJob& j) {
  if (elem_bytes != 2 && elem_bytes != 4 && elem_bytes != 8)
    return hcg::set_error(HCG_EINVAL, "%s: elem_bytes must be 2, 4 or 8, got %d", what, elem_bytes);
  if (rows < 0 || cols < 0 || ntiles < 0 || th < 0 || tw < 0)
    return hcg::set_error(HCG_EINVAL, "%s: negative extent (rows=%lld cols=%lld ntiles=%lld th=%lld tw=%lld)",
                          what, (long long)rows, (long long)cols, (long long)ntiles, (long long)th,
                          (long long)tw);
  if (rows > 0 && cols > 0) {
    if (view == nullptr) return hcg::set_error(HCG_EINVAL, "%s: view pointer is NULL", what);
    if (ld < cols) return hcg::set_error(HCG_EINVAL, "%s: ld (%lld) < cols (%lld)", what, (long long)ld,
                                         (long long)cols);
  }
  if (ntiles > 0 && origins == nullptr) return hcg::set_error(HCG_EINVAL, "%s: origins is NULL", what);
  const int64_t n = 16 / elem_bytes;
  j.ld = ld;
  j.rows = rows;
  j.cols = cols;
  j.origins = origins;
  j.ntiles = ntiles;
  j.th = th;
  j.tw = tw;
  j.chunks_per_row = (tw + n - 1) / n;
  j.total_chunks = ntiles * th * j.chunks_per_row;
  return HCG_OK;
}

unsigned grid_for(int64_t chunks) {
  const int64_t blocks = (chunks + 255) / 256;
  return (unsigned)(blocks < 65536 ? blocks : 65536);
}

}  // namespace

extern "C" {

int hcg_tile_load(int elem_bytes, const void* src, int64_t ld, int64_t rows, int64_t cols, const int64_t* origins,
                  int64_t ntiles, int64_t th, int64_t tw, const uint8_t* in_mask, uint64_t fill_bits, void* out,
                  uint8_t* out_mask, void* stream) {
  TileJob j{};
  int rc = prepare(elem_bytes, ld, rows, cols, src, origins, ntiles, th, tw, "hcg_tile_load", j);
  if (rc != HCG_OK) return rc;
  if (j.total_chunks == 0) {
    hcg::t_last_error.clear();
    return HCG_OK;
  }
  if (out == nullptr) return hcg::set_error(HCG_EINVAL, "hcg_tile_load: out is NULL");
  j.src = src;
  j.mask_in = in_mask;
  j.tiles_out = out;
  j.mask_out = out_mask;
  j.fill_bits = fill_bits;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  const unsigned grid = grid_for(j.total_chunks);
  if (elem_bytes == 2)
    run_load<uint16_t>(j, grid, s);
  else if (elem_bytes == 4)
    run_load<uint32_t>(j, grid, s);
  else
    run_load<uint64_t>(j, grid, s);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return hcg::set_error(HCG_EHIP, "tile_load_kernel launch failed: %s", hipGetErrorString(e));
  hcg::t_last_error.clear();
  return HCG_OK;
}

int hcg_tile_store(int elem_bytes, void* dst, int64_t ld, int64_t rows, int64_t cols, const int64_t* origins,
                   int64_t ntiles, int64_t th, int64_t tw, const void* tiles, const uint8_t* tile_mask,
                   void* stream) {
  TileJob j{};
  int rc = prepare(elem_bytes, ld, rows, cols, dst, origins, ntiles, th, tw, "hcg_tile_store", j);
  if (rc != HCG_OK) return rc;
  if (j.total_chunks == 0 || rows == 0 || cols == 0) {
    hcg::t_last_error.clear();
    return HCG_OK;
  }
  if (tiles == nullptr) return hcg::set_error(HCG_EINVAL, "hcg_tile_store: tiles is NULL");
  j.dst = dst;
  j.tiles_in = tiles;
  j.mask_in = tile_mask;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  const unsigned grid = grid_for(j.total_chunks);
  if (elem_bytes == 2)
    run_store<uint16_t>(j, grid, s);
  else if (elem_bytes == 4)
    run_store<uint32_t>(j, grid, s);
  else
    run_store<uint64_t>(j, grid, s);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return hcg::set_error(HCG_EHIP, "tile_store_kernel launch failed: %s", hipGetErrorString(e));
  hcg::t_last_error.clear();
  return HCG_OK;
}

}  // extern "C"
