// spk_tri.hpp -- triangular sweeps in tiles: the layout, its construction
// on the device and the sweep kernel's launch.
//
// A triangle of an n-row factor is cut into tiles of kTileRows consecutive
// rows, one wavefront each, and kGroupTiles tiles make a block.  A tile's
// rows are sorted by dependency level and cut into steps of at most 64 rows
// of one level and similar length; a lane takes a row of the step.  Values
// pass between a block's rows through LDS in a few hundred cycles; only a
// dependency on another block's rows waits for the published value (2-3 us
// of memory round trips).  The chain of a stencil's sweep then crosses
// memory once per block boundary instead of once per level.
//
// Progress: blocks take their tiles by a ticket in the triangle's order
// (ascending rows below the diagonal, descending above it), so every
// dependency lies in a block that is running or has ended; within a tile the
// steps ascend by level, and a row waits only for rows of lower levels.  The
// wait of an unfinished row of the lowest level therefore always ends.  Waits
// are bounded all the same, by the time in which no tile gets on.
#pragma once

#include "spk_csr.hpp"

namespace spk {

constexpr int kTileRows = 2048;
static_assert((kTileRows & (kTileRows - 1)) == 0, "sorted as a power of two");
constexpr int kGroupTiles = 4;  // LDS: 64 KB of FP64 values; a SIMD each
constexpr int kGroupRows = kTileRows * kGroupTiles;
constexpr int64_t kMaxTileSweepRows = int64_t(1) << 29;  // 32-bit byte offsets
constexpr int kBatch = 4;  // entries of a row that lie and are loaded together

// Entries of a row: column code >= 0, a row of the block; < 0, ~row of another
// block; kGroupRows: none (the value is +0 and so is what the code names, so
// the subtraction changes nothing).  Batch j of lane l of a step is group
// entries + j * rows + l.
template <typename T>
struct TriView {
  int64_t n;
  int tiles;
  const int32_t* __restrict__ rows;    // [n] rows in tile, step, lane order
  const int32_t* __restrict__ first;   // [tiles + 1] first step of each tile
  const int4* __restrict__ steps;      // {position of its first row, rows,
                                       //  first group, batches of a row,
                                       //  negative: no other block's values}
  const int4* __restrict__ cols;
  const T* __restrict__ v;             // kBatch a group
  const T* __restrict__ d;             // [n] diagonal by position (upper)
};

// One triangle of a factor.
struct TriTiles {
  int64_t n = 0, groups = 0;
  int tiles = 0, nsteps = 0;
  DevBuf<int32_t> rows, first;
  DevBuf<int4> steps, cols;
  DevBuf<double> v64, d64;
  DevBuf<float> v32, d32;
  bool has32 = false;
  template <typename T>
  TriView<T> view();
};

// The pattern both triangles come from, in device memory: CSR rows with the
// diagonal at dpos.
struct TriPattern {
  int64_t n;
  const int32_t* rp;
  const int32_t* ci;
  const int32_t* dpos;
};

// How long a wait may see no tile of its launch get on, in ticks of the 100
// MHz clock (0: the default, 10 s, of the construction 1 s; 1: every wait that lasts is given up, tiles
// that get on or not); for tests.
void set_tri_wait(unsigned long long ticks);
// Words of what is `ticket` below, zero before the first launch.
constexpr int kTriTicketWords = 4;
// Dependency levels of the rows of both triangles (lvl[0..n-1] below the
// diagonal, lvl[n..2n-1] above), and the number of levels of each; false if a
// bounded wait expired.
bool tri_levels(const TriPattern& P, DevBuf<int32_t>& lvl, int levels[2]);
// Order and steps of both triangles from their levels.  (What is freed here and
// below while kernels that use it are queued is handed out again only after
// them, see DevBuf.)
void tri_layouts(const TriPattern& P, const int32_t* lvl, TriTiles& lower, TriTiles& upper);
// Fills both triangles' values from w (one per entry of the pattern).
void tri_values(const TriPattern& P, const double* w, TriTiles& lower, TriTiles& upper);
// The IKJ factorization (ilu.hpp:72-115) of the values `in` into f (one per
// entry of the pattern), rows in the lower triangle's tile order.  max_len:
// the longest row, at most kTriFactorLen; max_side: the most entries a row
// has on one side of its diagonal.  No column is repeated in a row.  A wait
// that expired leaves 4 in *error, and f without meaning.
constexpr int kTriFactorLen = 32;
void tri_factor(const TriPattern& P, const TriTiles& lower, const double* in,
                DevBuf<double>& f, bool modified, int max_len, int max_side, int* ticket,
                int* error);

// x = L^-1 b or U^-1 b.  x must hold the ready sentinel; reset_b returns b's
// entries to it once read; else mark (may be null, may be b itself) is
// filled with it, every entry after b's entry has been read.
template <typename T, bool LOWER>
void tri_sweep(TriTiles& A, T* b, T* x, bool reset_b, T* mark, int* ticket, int* error,
               hipStream_t s);

// ------------------------------------------------------------- readiness
// A value doubles as its own ready flag: the output starts filled with a NaN
// sentinel that arithmetic never produces, a finished row stores its value
// with one agent-scope atomic store, and a row that needs it spins on an
// agent-scope load.
template <typename T>
struct Sentinel;
template <>
struct Sentinel<double> {
  typedef unsigned long long U;
  static constexpr U bits = 0xFFF8DEADBEEFCAFEull;
};
template <>
struct Sentinel<float> {
  typedef unsigned int U;
  static constexpr U bits = 0xFFC0DEADu;
};

template <typename T>
__device__ __forceinline__ bool load_ready(const T* p, T* out) {
  typedef typename Sentinel<T>::U U;
  U u = __hip_atomic_load(reinterpret_cast<const U*>(p), __ATOMIC_RELAXED,
                          __HIP_MEMORY_SCOPE_AGENT);
  T v;
  __builtin_memcpy(&v, &u, sizeof(T));
  *out = v;
  return u != Sentinel<T>::bits;
}

template <typename T>
__device__ __forceinline__ void store_ready(T* p, T v) {
  typedef typename Sentinel<T>::U U;
  U u;
  __builtin_memcpy(&u, &v, sizeof(T));
  // a NaN result carrying the sentinel's payload (propagated from a NaN
  // input) must not read as "not ready": publish it with another payload
  if (u == Sentinel<T>::bits) u ^= (U)1;
  __hip_atomic_store(reinterpret_cast<U*>(p), u, __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}

template <typename T>
__device__ __forceinline__ T sentinel_value() {
  typedef typename Sentinel<T>::U U;
  U u = Sentinel<T>::bits;
  T v;
  __builtin_memcpy(&v, &u, sizeof(T));
  return v;
}

}  // namespace spk
