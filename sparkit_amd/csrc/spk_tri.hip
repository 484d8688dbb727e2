// spk_tri.hip -- triangular sweeps in tiles (layout and progress argument:
// spk_tri.hpp).
#include "spk_tri.hpp"

#include <algorithm>
#include <type_traits>

namespace spk {
namespace {

// The block's ticket (ticket[0] counts those taken, ticket[1] the tiles done:
// the last returns both to zero for the next launch) and the launch's beat
// (ticket[2]), a number that changes while any tile gets on: a healthy chain
// of dependencies may take longer than any limit on a single wait.
static_assert(kTriTicketWords > 2, "ticket");
__device__ __forceinline__ void beat(int* ticket) {
  if ((threadIdx.x & 63) == 0)
    (void)__hip_atomic_fetch_add(ticket + 2, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A bounded wait, for a whole wavefront: false once the beat has stood still
// for `ticks` of the 100 MHz clock (looked at every kLook polls).  With kSleep a
// wait that lasts sleeps between its polls, up to 3 us: 20 addresses a lane of
// every waiting wavefront keep the memory from those that work.  The sweeps
// poll what is missing only, in LDS where they can, and do not sleep: a tile
// of a narrow grid follows the one before it by 30 us (40 x 20,000 rows: 14.9
// ms an application, 18.7 with the sleep and a look every 256 polls).
template <unsigned kLook, bool kSleep>
struct Wait {
  unsigned polls = 0;
  int seen = 0;
  unsigned long long since = 0;
  __device__ bool again(const int* ticket, unsigned long long ticks) {
    ++polls;
    if (kSleep)
      for (unsigned k = polls >> 6 < 16u ? polls >> 6 : 16u; k > 0; --k)
        __builtin_amdgcn_s_sleep(8);
    if ((polls & (kLook - 1)) != 0) return true;
    const int b =
        __hip_atomic_load(ticket + 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const unsigned long long now = wall_clock64();
    if (since == 0 || (b != seen && ticks > 1)) {
      since = now;
      seen = b;
    }
    return now - since < ticks;
  }
};
using BuildWait = Wait<256, true>;
using SweepWait = Wait<4096, false>;
constexpr unsigned long long kWaitTicks = 1000000000ull;  // 10 s
constexpr unsigned long long kBuildTicks = 100000000ull;  // the construction: 1 s,
                                                          // it goes on without waits
unsigned long long g_wait_ticks = 0;  // 0: these
unsigned long long sweep_ticks() { return g_wait_ticks ? g_wait_ticks : kWaitTicks; }
unsigned long long build_ticks() { return g_wait_ticks ? g_wait_ticks : kBuildTicks; }
__device__ __forceinline__ int take_tile(int* ticket) {
  int t = 0;
  if ((threadIdx.x & 63) == 0)
    t = __hip_atomic_fetch_add(ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return __builtin_amdgcn_readfirstlane(t);
}
__device__ __forceinline__ void tile_done(int* ticket, int tiles) {
  beat(ticket);
  if ((threadIdx.x & 63) != 0) return;
  if (__hip_atomic_fetch_add(ticket + 1, 1, __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT) == tiles - 1) {
    __hip_atomic_store(ticket, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(ticket + 1, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// Batch j of lane l of a step (unsigned: a triangle may hold more than 2^31
// groups).
__device__ __forceinline__ unsigned group_at(const int4& h, int j, int lane) {
  return (unsigned)h.z + (unsigned)(j * h.y + lane);
}

// ------------------------------------------------------------- levels

// One block per tile of either triangle (blocks [0, tiles): lower).  A thread
// has kLevelRows of the tile's rows; in a pass it looks up one dependency of
// each of them (in LDS within the tile, by an agent-scope load beyond), all
// looked up before the first is used, and a row whose dependencies are
// through publishes its level.  The rows finish in whatever order their
// dependencies do.  lvl starts at -1.
constexpr int kLevelSleep = 16;
constexpr int kLevelBlock = 256;
constexpr int kLevelRows = kTileRows / kLevelBlock;
__global__ __launch_bounds__(kLevelBlock) void tri_level_kernel(
    TriPattern P, int tiles, int32_t* lvl, int* ticket, int* maxlvl, int* error,
    unsigned long long ticks) {
  __shared__ int32_t mine[kTileRows];
  __shared__ int shared_tile;
  const bool lower = blockIdx.x < (unsigned)tiles;
  int* tk = ticket + (lower ? 0 : kTriTicketWords);
  int32_t* out = lvl + (lower ? 0 : P.n);
  if (threadIdx.x < 64) {
    const int t = take_tile(tk);
    if (threadIdx.x == 0) shared_tile = t;
  }
  for (int k = threadIdx.x; k < kTileRows; k += kLevelBlock) mine[k] = -1;
  __syncthreads();
  const int tile = lower ? shared_tile : tiles - 1 - shared_tile;
  const int base = tile * kTileRows;
  const int rows = (int)(P.n - base < kTileRows ? P.n - base : kTileRows);
  int p[kLevelRows], pe[kLevelRows], c[kLevelRows], level[kLevelRows];
  int left = 0, top = 0;
#pragma unroll
  for (int u = 0; u < kLevelRows; ++u) {
    const int loc = (int)threadIdx.x + u * kLevelBlock;
    p[u] = pe[u] = c[u] = 0;
    level[u] = -1;  // not a row, or published
    if (loc < rows) {
      const int i = base + loc, dp = P.dpos[i];
      p[u] = lower ? P.rp[i] : dp + 1;
      pe[u] = lower ? dp : P.rp[i + 1];
      level[u] = 0;
      ++left;
    }
  }
#pragma unroll
  for (int u = 0; u < kLevelRows; ++u)
    if (p[u] < pe[u]) c[u] = P.ci[p[u]];
  BuildWait w;
  unsigned moves = 0;
  while (__any(left > 0)) {
    int l[kLevelRows];
#pragma unroll
    for (int u = 0; u < kLevelRows; ++u) {
      l[u] = -1;
      const bool ask = level[u] >= 0 && p[u] < pe[u];
      const int j = c[u] - base;
      if (ask && (unsigned)j >= (unsigned)kTileRows)
        l[u] = __hip_atomic_load(out + c[u], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      else if (ask)
        l[u] = __hip_atomic_load(&mine[j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
#pragma unroll
    for (int u = 0; u < kLevelRows; ++u)
      if (l[u] >= 0) {
        level[u] = l[u] + 1 > level[u] ? l[u] + 1 : level[u];
        if (++p[u] < pe[u]) c[u] = P.ci[p[u]];
      }
#pragma unroll
    for (int u = 0; u < kLevelRows; ++u)
      if (level[u] >= 0 && p[u] >= pe[u]) {
        const int loc = (int)threadIdx.x + u * kLevelBlock;
        __hip_atomic_store(&mine[loc], level[u], __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_WORKGROUP);
        __hip_atomic_store(out + base + loc, level[u], __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
        top = level[u] + 1 > top ? level[u] + 1 : top;
        level[u] = -1;
        --left;
      }
    // a wavefront nothing has reached yet leaves the memory to the others
    bool moved = false;
#pragma unroll
    for (int u = 0; u < kLevelRows; ++u) moved = moved || l[u] >= 0;
    if (__any(moved)) {
      w = BuildWait{};
      if ((++moves & 255u) == 0) beat(tk);
      continue;
    }
    __builtin_amdgcn_s_sleep(kLevelSleep);
    if (!w.again(tk, ticks)) {
      if ((threadIdx.x & 63) == 0) atomicOr(error, 4);
      break;
    }
  }
  for (int o = 32; o > 0; o >>= 1) {
    const int other = __shfl_xor(top, o, 64);
    top = other > top ? other : top;
  }
  if ((threadIdx.x & 63) == 0) atomicMax(maxlvl + (lower ? 0 : 1), top);
  if (threadIdx.x < 64) tile_done(tk, tiles);
}

// ------------------------------------------------------------- order

// rows of similar length share a step: its lanes' entries are padded to the
// longest (at most twice a row's own length) and to whole batches
__device__ __forceinline__ int length_class(int len) {
  return len <= 4 ? 0 : 30 - __clz(len - 1);
}

// What the construction of both triangles works on (0: lower, 1: upper).
struct TriBuild {
  int tiles;
  const int32_t* lvl[2];
  int32_t* rows[2];
  int2* step[2];
  int* first[2];  // [tiles + 1]
  int* ent[2];    // [tiles + 1]
  int4* steps[2];
  int4* cols[2];
};

// One block per tile of either triangle (blocks [0, tiles): lower): its rows
// sorted by (level, length, row), the steps' {position, batches} and their
// number and groups.
__global__ __launch_bounds__(256) void tri_order_kernel(TriPattern P, TriBuild B) {
  __shared__ unsigned long long key[kTileRows];
  const bool lower = blockIdx.x < (unsigned)B.tiles;
  const int k2 = lower ? 0 : 1, tile = (int)blockIdx.x - k2 * B.tiles, base = tile * kTileRows;
  const int32_t* lvl = B.lvl[k2];
  int32_t* order = B.rows[k2];
  int2* step = B.step[k2];
  const int rows = (int)(P.n - base < kTileRows ? P.n - base : kTileRows);
  for (int k = threadIdx.x; k < kTileRows; k += 256) {
    unsigned long long q = ~0ull;
    if (k < rows) {
      const int i = base + k, dp = P.dpos[i];
      int len = lower ? dp - P.rp[i] : P.rp[i + 1] - dp - 1;
      len = len < 65535 ? len : 65535;
      q = ((unsigned long long)(unsigned)lvl[i] << 32) | ((unsigned)len << 16) | (unsigned)k;
    }
    key[k] = q;
  }
  __syncthreads();
  for (int size = 2; size <= kTileRows; size *= 2)
    for (int st = size / 2; st > 0; st /= 2) {
      for (int k = threadIdx.x; k < kTileRows / 2; k += 256) {
        const int a = 2 * k - (k & (st - 1)), b = a + st;
        const bool up = (a & size) == 0;
        const unsigned long long x = key[a], y = key[b];
        if ((x > y) == up) {
          key[a] = y;
          key[b] = x;
        }
      }
      __syncthreads();
    }
  for (int k = threadIdx.x; k < rows; k += 256)
    order[base + k] = base + (int)(key[k] & 0xFFFF);
  if (threadIdx.x >= 64) return;
  // runs of one level and length class, cut every 64 rows
  const int lane = threadIdx.x;
  int run = 0, count = 0;
  for (int g = 0; g < rows; g += 64) {
    const int k = g + lane;
    bool head = false;
    if (k < rows) {
      const unsigned long long q = key[k];
      if (k == 0) head = true;
      else {
        const unsigned long long o = key[k - 1];
        head = (q >> 32) != (o >> 32) ||
               length_class((int)(q >> 16) & 0xFFFF) != length_class((int)(o >> 16) & 0xFFFF);
      }
    }
    const unsigned long long heads = __ballot(head);
    const unsigned long long upto = heads & (~0ull >> (63 - lane));
    const int start = upto ? g + 63 - __clzll(upto) : run;
    const bool cut = k < rows && ((k - start) & 63) == 0;
    const unsigned long long cuts = __ballot(cut);
    if (cut) step[base + count + __popcll(cuts & ((1ull << lane) - 1))].x = base + k;
    count += __popcll(cuts);
    if (heads) run = g + 63 - __clzll(heads);
  }
  __threadfence_block();
  int ent = 0;
  for (int q = lane; q < count; q += 64) {
    const int a = step[base + q].x - base;
    const int b = q + 1 < count ? step[base + q + 1].x - base : rows;
    // lengths ascend within a step (65535 stands for that and longer)
    int width = (int)(key[b - 1] >> 16) & 0xFFFF;
    if (width == 65535)
      for (int k = a; k < b; ++k) {
        const int r = base + (int)(key[k] & 0xFFFF), d = P.dpos[r];
        const int len = lower ? d - P.rp[r] : P.rp[r + 1] - d - 1;
        width = len > width ? len : width;
      }
    const int batches = width > kBatch ? (width + kBatch - 1) / kBatch : 1;
    step[base + q].y = batches;
    ent += batches * (b - a);
  }
  for (int o = 32; o > 0; o >>= 1) ent += __shfl_xor(ent, o, 64);
  if (lane == 0) {
    B.first[k2][tile] = count;
    B.ent[k2][tile] = ent;
  }
}

// exclusive sums of each triangle's steps and groups in place, the totals
// behind them and in total[4]; one block a triangle
__global__ __launch_bounds__(1024) void tri_scan_kernel(TriBuild B, int* total) {
  __shared__ int sa[1024], sb[1024];
  const int m = B.tiles;
  int *a = B.first[blockIdx.x], *b = B.ent[blockIdx.x];
  int ca = 0, cb = 0;
  for (int g = 0; g < m; g += 1024) {
    const int k = g + (int)threadIdx.x;
    const int va = k < m ? a[k] : 0, vb = k < m ? b[k] : 0;
    sa[threadIdx.x] = va;
    sb[threadIdx.x] = vb;
    __syncthreads();
    for (int o = 1; o < 1024; o *= 2) {
      const int xa = (int)threadIdx.x >= o ? sa[threadIdx.x - o] : 0;
      const int xb = (int)threadIdx.x >= o ? sb[threadIdx.x - o] : 0;
      __syncthreads();
      sa[threadIdx.x] += xa;
      sb[threadIdx.x] += xb;
      __syncthreads();
    }
    if (k < m) {
      a[k] = ca + sa[threadIdx.x] - va;
      b[k] = cb + sb[threadIdx.x] - vb;
    }
    ca += sa[1023];
    cb += sb[1023];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    a[m] = total[2 * blockIdx.x] = ca;
    b[m] = total[2 * blockIdx.x + 1] = cb;
  }
}

// One block per tile of either triangle: the step headers and the column
// codes.
__global__ __launch_bounds__(256) void tri_fill_kernel(TriPattern P, TriBuild B) {
  const bool lower = blockIdx.x < (unsigned)B.tiles;
  const int k2 = lower ? 0 : 1, tile = (int)blockIdx.x - k2 * B.tiles, base = tile * kTileRows;
  const int32_t* order = B.rows[k2];
  const int2* step = B.step[k2];
  const int *first = B.first[k2], *ent = B.ent[k2];
  int4 *steps = B.steps[k2], *cols = B.cols[k2];
  const int gbase = tile / kGroupTiles * kGroupRows;
  const int rows = (int)(P.n - base < kTileRows ? P.n - base : kTileRows);
  const int s0 = first[tile], count = first[tile + 1] - s0;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (wave == 0) {
    int at = ent[tile];
    for (int g = 0; g < count; g += 64) {
      const int q = g + lane;
      int4 h{0, 0, 0, 0};
      if (q < count) {
        h.x = step[base + q].x;
        h.w = step[base + q].y;
        h.y = (q + 1 < count ? step[base + q + 1].x : base + rows) - h.x;
      }
      int sum = h.y * h.w;
      for (int o = 1; o < 64; o *= 2) {
        const int up = __shfl_up(sum, o, 64);
        if (lane >= o) sum += up;
      }
      h.z = at + sum - h.y * h.w;
      if (q < count) steps[s0 + q] = h;
      at += __shfl(sum, 63, 64);
    }
  }
  __syncthreads();  // the block's own global writes, read below
  for (int q = wave; q < count; q += 4) {
    const int4 h = steps[s0 + q];
    const bool in = lane < h.y;
    int p0 = 0, pe = 0;
    if (in) {
      const int i = order[h.x + lane], dp = P.dpos[i];
      p0 = lower ? P.rp[i] : dp + 1;
      pe = lower ? dp : P.rp[i + 1];
    }
    bool beyond = false;
    for (int j = 0; j < h.w; ++j) {
      int code[kBatch];
#pragma unroll
      for (int k = 0; k < kBatch; ++k) {
        code[k] = kGroupRows;
        const int p = p0 + j * kBatch + k;
        if (p < pe) {
          const int c = P.ci[p];
          code[k] = (unsigned)(c - gbase) < (unsigned)kGroupRows ? c - gbase : ~c;
          beyond = beyond || code[k] < 0;
        }
      }
      if (in) cols[group_at(h, j, lane)] = int4{code[0], code[1], code[2], code[3]};
    }
    // the sign of w: no value of another block in the step
    if (!__any(beyond) && lane == 0) steps[s0 + q].w = -h.w;
  }
}

// One wavefront per step of either triangle: the values in the layout's order.
struct TriValues {
  int nsteps[2];
  const int32_t* rows[2];
  const int4* steps[2];
  double* v[2];
  double* d;
};
__global__ __launch_bounds__(256) void tri_value_kernel(TriPattern P, TriValues B,
                                                        const double* __restrict__ w) {
  const int at = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  const bool lower = at < B.nsteps[0];
  const int k2 = lower ? 0 : 1, q = at - k2 * B.nsteps[0];
  if (q >= B.nsteps[k2]) return;
  const int32_t* order = B.rows[k2];
  const int4* steps = B.steps[k2];
  double *v = B.v[k2], *d = B.d;
  const int4 h = steps[q];
  if (lane >= h.y) return;
  const int i = order[h.x + lane], dp = P.dpos[i];
  const int p0 = lower ? P.rp[i] : dp + 1, pe = lower ? dp : P.rp[i + 1];
  const int batches = h.w < 0 ? -h.w : h.w;
  for (int j = 0; j < batches; ++j) {
    double* o = v + (size_t)group_at(h, j, lane) * kBatch;
#pragma unroll
    for (int k = 0; k < kBatch; ++k) {
      const int p = p0 + j * kBatch + k;
      o[k] = p < pe ? w[p] : 0.0;
    }
  }
  if (!lower) d[h.x + lane] = w[dp];
}

__global__ void tri_cast_kernel(const double* __restrict__ in, float* __restrict__ out,
                                int64_t n) {
  for (int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; k < n;
       k += (int64_t)gridDim.x * blockDim.x)
    out[k] = (float)in[k];
}

// ------------------------------------------------------------- sweep

constexpr int kRing = 8;  // steps in flight
// How many steps ahead of its solution a step's rows and entries, its
// right-hand side and its other blocks' values are loaded.  Polls 3 or 4
// steps ahead must find values that are older still (128^3 sweep, one tile a
// block: 0.55 ms at 2, 0.62 at 3, 0.60 at 4), 1 ahead waits for each poll
// (a chain of 2,048 rows 0.80 ms against 0.64).
constexpr int kAheadEntries = 6, kAheadRhs = 3, kAheadPoll = 2;

// Four values of a group, loaded with 16-byte loads.
template <typename T>
struct alignas(16) Group {
  T v[kBatch];
};

// What a lane holds of its row of a step.
template <typename T>
struct Stage {
  int rows, row;  // the step's rows, the lane's row
  int batches;    // of its rows; negative: all values are the block's own
  unsigned group;
  T b, d;
  int4 c;
  Group<T> v;
  T u[kBatch];
};

template <typename T>
__device__ __forceinline__ T raw_load(const T* p) {
  T v;
  (void)load_ready(p, &v);
  return v;
}
template <typename T>
__device__ __forceinline__ void raw_store(T* p, T v) {
  typename Sentinel<T>::U u;
  __builtin_memcpy(&u, &v, sizeof(T));
  __hip_atomic_store(reinterpret_cast<typename Sentinel<T>::U*>(p), u, __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}
// LDS words other wavefronts of the block write
template <typename T>
__device__ __forceinline__ T lds_load(const T* p) {
  typename Sentinel<T>::U u = __hip_atomic_load(
      reinterpret_cast<const typename Sentinel<T>::U*>(p), __ATOMIC_RELAXED,
      __HIP_MEMORY_SCOPE_WORKGROUP);
  T v;
  __builtin_memcpy(&v, &u, sizeof(T));
  return v;
}
template <typename T>
__device__ __forceinline__ void lds_store(T* p, T v) {
  typename Sentinel<T>::U u;
  __builtin_memcpy(&u, &v, sizeof(T));
  __hip_atomic_store(reinterpret_cast<typename Sentinel<T>::U*>(p), u, __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_WORKGROUP);
}
// p + i with a 32-bit byte offset, which a load adds by itself
// (kMaxTileSweepRows rows at most)
template <typename T>
__device__ __forceinline__ T* at(T* p, int i) {
  return (T*)((char*)p + (unsigned)i * (unsigned)sizeof(T));
}
// a NaN that is the sentinel by accident, with another payload
template <typename T>
__device__ __forceinline__ T other_nan(T v) {
  typename Sentinel<T>::U u;
  __builtin_memcpy(&u, &v, sizeof(T));
  u ^= 1;
  __builtin_memcpy(&v, &u, sizeof(T));
  return v;
}
template <typename T>
__device__ __forceinline__ bool is_ready(T v) {
  typename Sentinel<T>::U u;
  __builtin_memcpy(&u, &v, sizeof(T));
  return u != Sentinel<T>::bits;
}

// How a sweep leaves b: as it is, filled with the sentinel elsewhere (mark),
// or returned to it.
enum { kPlain = 0, kMark = 1, kReset = 2 };

// One wavefront per tile.  A lone wavefront issues an instruction every few
// cycles, so the step's code has no branches for single entries: lanes past
// the step's rows repeat its last row (and store the same values), absent
// entries name a zero, and every entry's value is both read from LDS and
// loaded from x, at the tile's first row where it is not another block's.
// Bound: the chain of steps, 0.31 us each, and about 2.5 us from a value's
// store to its use per block boundary the dependency chain crosses.  One
// application (both triangles, FP64), a launch per level -> this: 64^3 7-point
// 1.95 -> 0.35 ms, 128^3 4.6 -> 1.25 ms, 256^2 5-point 3.6 -> 0.49 ms, 512^2
// 9-point 12.5 -> 1.47 ms (the sweep that gave every row of a window of
// levels a thread: 1.23 ms at 64^3, 2.98 at 128^3).  Blocks of 1 / 4 / 8
// tiles took 0.46 / 0.35 / 0.41 ms at 64^3 and 1.13 / 1.25 / 1.44 at 128^3;
// tiles of 1,024 rows 0.47 and 1.29.
template <typename T, bool LOWER, int MODE>
__global__ __launch_bounds__(64 * kGroupTiles) void tri_sweep_kernel(
    TriView<T> A, T* b, T* x, T* mark, int* ticket, int* error, unsigned long long ticks) {
#pragma clang fp contract(off)
  __shared__ T val[kGroupRows + 1];
  __shared__ int taken;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (wave == 0) {
    const int t = take_tile(ticket);
    if (lane == 0) taken = t;
  }
  for (int k = threadIdx.x; k <= kGroupRows; k += 64 * kGroupTiles)
    val[k] = k < kGroupRows ? sentinel_value<T>() : T(0);
  __syncthreads();
  const int groups = (A.tiles + kGroupTiles - 1) / kGroupTiles;
  const int group = LOWER ? taken : groups - 1 - taken;
  const int tile = __builtin_amdgcn_readfirstlane(group * kGroupTiles + wave);
  if (tile >= A.tiles) return;
  const int base = tile * kTileRows, gbase = group * kGroupRows;
  const int s0 = __builtin_amdgcn_readfirstlane(A.first[tile]);
  const int count = __builtin_amdgcn_readfirstlane(A.first[tile + 1]) - s0;
  bool dead = false;
  // step at + lane's; past the last, the last one's again (loaded, not run)
  auto headers = [&](int at) {
    const int q = at + lane < count ? at + lane : count - 1;
    return A.steps[s0 + q];
  };
  // headers come 64 at a time into the lanes and are read from there: scalar
  // loads would share their counter with the LDS reads of the chain
  int4 hnow = headers(0), hnext = headers(64);
  Stage<T> ring[kRing];

  // rows, entries and diagonal of step f, in order
  auto load_entries = [&](Stage<T>& g, int f) {
    const int nth = f & 63;
    if (nth == 0 && f > 0) {
      hnow = hnext;
      hnext = headers(f + 64);
      beat(ticket);
    }
    const int pos = __builtin_amdgcn_readlane(hnow.x, nth);
    g.rows = __builtin_amdgcn_readlane(hnow.y, nth);
    g.group = (unsigned)__builtin_amdgcn_readlane(hnow.z, nth);
    g.batches = __builtin_amdgcn_readlane(hnow.w, nth);
    const unsigned l = (unsigned)(lane < g.rows ? lane : g.rows - 1);
    g.row = (A.rows + pos)[l];
    if (!LOWER) g.d = (A.d + pos)[l];
    g.c = (A.cols + g.group)[l];
    g.v = ((const Group<T>*)A.v + g.group)[l];
  };
  auto load_rhs = [&](Stage<T>& g) { g.b = *at(b, g.row); };
  auto poll = [&](int batches, const int4& c, T* u) {
    if (batches < 0) return;
    const int q[kBatch] = {c.x, c.y, c.z, c.w};
#pragma unroll
    for (int k = 0; k < kBatch; ++k) u[k] = raw_load(at(x, q[k] < 0 ? ~q[k] : base));
  };
  // s -= v * x over the batch, in storage order, multiply-adds not
  // contracted (triangular_solve.hpp:42-53, 82-96: bit-identical to the
  // sequential reference), once every value in it is ready
  auto solve = [&](const int4& c, const Group<T>& v, T* u, T s) {
    const int q[kBatch] = {c.x, c.y, c.z, c.w};
    T xv[kBatch];
    bool all = true;
#pragma unroll
    for (int k = 0; k < kBatch; ++k) {
      const unsigned own = (unsigned)q[k] < (unsigned)kGroupRows ? (unsigned)q[k]
                                                                 : (unsigned)kGroupRows;
      const T in = lds_load(val + own);  // by every lane
      xv[k] = q[k] < 0 ? u[k] : in;
      all = all && is_ready(xv[k]);
    }
    if (!__all(all)) {
      SweepWait w;
      while (!dead && !__all(all)) {
        all = true;
#pragma unroll
        for (int k = 0; k < kBatch; ++k) {
          if (!is_ready(xv[k])) xv[k] = q[k] < 0 ? raw_load(at(x, ~q[k])) : lds_load(val + q[k]);
          all = all && is_ready(xv[k]);
        }
        if (!w.again(ticket, ticks)) {
          dead = true;
          if (lane == 0) atomicOr(error, LOWER ? 1 : 2);
        }
      }
    }
#pragma unroll
    for (int k = 0; k < kBatch; ++k) s = s - v.v[k] * xv[k];
    return s;
  };
  auto step = [&](auto slot, int q) {
    constexpr int J = decltype(slot)::value;
    Stage<T>& g = ring[J];
    T s = solve(g.c, g.v, g.u, g.b);
    const int batches = g.batches < 0 ? -g.batches : g.batches;
    for (int j = 1; j < batches; ++j) {  // wider rows
      if ((j & 255) == 0) beat(ticket);
      const int l = lane < g.rows ? lane : g.rows - 1;
      const unsigned e = g.group + (unsigned)(j * g.rows + l);
      const int4 c = A.cols[e];
      const Group<T> v = ((const Group<T>*)A.v)[e];
      T u[kBatch];
      poll(g.batches, c, u);
      s = solve(c, v, u, s);
    }
    // L's diagonal is 1: s / 1 is s
    T xi = LOWER ? s : s / g.d;
    if (!is_ready(xi)) xi = other_nan(xi);
    lds_store(val + (g.row - gbase), xi);
    raw_store(at(x, g.row), xi);
    if (MODE == kReset) *at(b, g.row) = sentinel_value<T>();
    if (MODE == kMark) *at(mark, g.row) = sentinel_value<T>();
    __builtin_amdgcn_wave_barrier();
    Stage<T>& gp = ring[(J + kAheadPoll) % kRing];
    poll(gp.batches, gp.c, gp.u);
    load_rhs(ring[(J + kAheadRhs) % kRing]);
    load_entries(ring[(J + kAheadEntries) % kRing], q + kAheadEntries);
  };
#pragma unroll
  for (int f = 0; f < kAheadEntries; ++f) load_entries(ring[f], f);
#pragma unroll
  for (int f = 0; f < kAheadRhs; ++f) load_rhs(ring[f]);
#pragma unroll
  for (int f = 0; f < kAheadPoll; ++f) poll(ring[f].batches, ring[f].c, ring[f].u);
  for (int q = 0;; q += kRing) {
    step(std::integral_constant<int, 0>{}, q);
    if (q + 1 >= count) break;
    step(std::integral_constant<int, 1>{}, q + 1);
    if (q + 2 >= count) break;
    step(std::integral_constant<int, 2>{}, q + 2);
    if (q + 3 >= count) break;
    step(std::integral_constant<int, 3>{}, q + 3);
    if (q + 4 >= count) break;
    step(std::integral_constant<int, 4>{}, q + 4);
    if (q + 5 >= count) break;
    step(std::integral_constant<int, 5>{}, q + 5);
    if (q + 6 >= count) break;
    step(std::integral_constant<int, 6>{}, q + 6);
    if (q + 7 >= count) break;
    step(std::integral_constant<int, 7>{}, q + 7);
    if (q + 8 >= count) break;
  }
  tile_done(ticket, A.tiles);
}

// ------------------------------------------------------------- factorization

// One IKJ row of ilu0_impl (ilu.hpp:72-115) per lane, the rows of a step
// together, tiles and steps as the lower sweep, one wavefront a tile.
// Multiply-adds are not contracted, so every update rounds exactly as the
// reference's w[pos] -= l_ik * w[q].

// Rows of any length up to max_len: the row is worked on in LDS (entry e of
// lane l at e * 64 + l).  A finished row's entries are stored first and its
// pivot, whose sentinel is the ready flag, once they have reached memory.
__global__ __launch_bounds__(64) void tri_factor_kernel(TriPattern P, TriView<double> A,
                                                        double* w, double* pivot,
                                                        int max_len, int modified,
                                                        int* ticket, int* error,
                                                        unsigned long long ticks) {
#pragma clang fp contract(off)
  extern __shared__ double buf[];
  int* cbuf = (int*)(buf + max_len * 64);
  const int tile = take_tile(ticket), lane = threadIdx.x;
  const int s0 = A.first[tile], s1 = A.first[tile + 1];
  bool dead = false;
  for (int q = s0; q < s1; ++q) {
    if ((q & 15) == 0) beat(ticket);
    const int4 h = A.steps[q];
    const bool in = lane < h.y;
    int i = 0, p0 = 0, len = 0, nl = 0;
    if (in) {
      i = A.rows[h.x + lane];
      p0 = P.rp[i];
      len = P.rp[i + 1] - p0;
      nl = P.dpos[i] - p0;
      for (int e = 0; e < len; ++e) {
        buf[e * 64 + lane] = w[p0 + e];
        cbuf[e * 64 + lane] = P.ci[p0 + e];
      }
    }
    double dropped = 0.0;
    for (int e = 0; __any(e < nl); ++e) {
      const bool has = e < nl;
      const int k = has ? cbuf[e * 64 + lane] : 0;
      const int z0 = has ? P.dpos[k] + 1 : 0, z1 = has ? P.rp[k + 1] : 0;
      double d = 1.0;
      bool ok = !has;
      BuildWait wt;
      for (;;) {
        if (!ok) ok = load_ready(pivot + k, &d);
        if (__all(ok)) break;
        if (dead || !wt.again(ticket, ticks)) {
          if (!dead && lane == 0) atomicOr(error, 4);
          dead = true;
          break;
        }
      }
      if (!has) continue;
      double* t = buf + e * 64 + lane;
      const double l = *t / d;
      *t = l;
      int at = e + 1;
      for (int z = z0; z < z1; ++z) {
        const int j = P.ci[z];
        const double wz = raw_load(w + z);
        while (at < len && cbuf[at * 64 + lane] < j) ++at;
        if (at < len && cbuf[at * 64 + lane] == j) {
          double* x = buf + at * 64 + lane;
          *x = *x - l * wz;
        } else if (modified) {
          dropped = dropped + l * wz;
        }
      }
    }
    if (in) {
      double* t = buf + nl * 64 + lane;
      if (modified) *t = *t - dropped;
      for (int e = 0; e < len; ++e) raw_store(w + p0 + e, buf[e * 64 + lane]);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (in) store_ready(pivot + i, buf[nl * 64 + lane]);
    __builtin_amdgcn_wave_barrier();
  }
  tile_done(ticket, A.tiles);
}

// Rows of at most kBatch entries on each side of the diagonal (stencils): a
// row's elimination is written down beforehand, all rows at once, in the
// order the factorization takes them.
struct RowProgram {
  int4 row;  // first entry, entries, pivots, -
  int4 z;    // the pivots' positions (absent: the row's first entry)
  int4 use;  // which entry each pivot row's upper entry t updates: byte t of
             // its word, kDrop none, kNone no such entry
};
constexpr int kShort = 2 * kBatch + 1;  // entries of a row, at most
constexpr unsigned kDrop = 0xFE, kNone = 0xFF;

__global__ __launch_bounds__(256) void tri_program_kernel(TriPattern P,
                                                          const int32_t* __restrict__ order,
                                                          RowProgram* __restrict__ prog) {
  const int64_t pos = blockIdx.x * (int64_t)256 + threadIdx.x;
  if (pos >= P.n) return;
  const int i = order[pos], p0 = P.rp[i], len = P.rp[i + 1] - p0, nl = P.dpos[i] - p0;
  int c[kShort];
#pragma unroll
  for (int e = 0; e < kShort; ++e) c[e] = e < len ? P.ci[p0 + e] : -1;
  int z[kBatch];
  unsigned use[kBatch];
#pragma unroll
  for (int u = 0; u < kBatch; ++u) {
    z[u] = p0;
    use[u] = ~0u;
    if (u < nl) {
      const int k = c[u], z0 = P.dpos[k], cnt = P.rp[k + 1] - z0 - 1;
      z[u] = z0;
#pragma unroll
      for (int t = 0; t < kBatch; ++t)
        if (t < cnt) {
          const int j = P.ci[z0 + 1 + t];
          unsigned m = kDrop;
#pragma unroll
          for (int e = 1; e < kShort; ++e)
            if (e > u && c[e] == j) m = (unsigned)e;
          use[u] = (use[u] & ~(0xFFu << (8 * t))) | (m << (8 * t));
        }
    }
  }
  prog[pos] = RowProgram{int4{p0, len, nl, 0}, int4{z[0], z[1], z[2], z[3]},
                         int4{(int)use[0], (int)use[1], (int)use[2], (int)use[3]}};
}

// The entries go to f, which starts filled with the ready sentinel: a row
// polls the pivots and upper entries it needs themselves, all together, and
// a step costs that one round trip.  Programs are loaded two steps ahead,
// the rows' values one.  128^3 7-point: 2.2 ms (a flag behind each finished
// row and no programs 3.3; a launch per level about 5).
struct ProgramStage {
  RowProgram r;
  double v[kShort];
};
__global__ __launch_bounds__(64) void tri_factor_short_kernel(
    int tiles, const int32_t* __restrict__ first, const int4* __restrict__ steps,
    const RowProgram* __restrict__ prog, const double* __restrict__ in, double* f,
    int modified, int* ticket, int* error, unsigned long long ticks) {
#pragma clang fp contract(off)
  // the row's entries; kShort: what updates of no entry write to
  __shared__ double buf[(kShort + 1) * 64];
  const int tile = take_tile(ticket), lane = threadIdx.x;
  const int s0 = __builtin_amdgcn_readfirstlane(first[tile]);
  const int count = __builtin_amdgcn_readfirstlane(first[tile + 1]) - s0;
  auto headers = [&](int at) {
    const int q = at + lane < count ? at + lane : count - 1;
    return steps[s0 + q];
  };
  int4 hnow = headers(0), hnext = headers(64);
  bool dead = false;
  ProgramStage ring[4];
  // lanes past the step's rows repeat its last row
  auto load_program = [&](ProgramStage& g, int q) {
    const int nth = q & 63;
    if (nth == 0 && q > 0) {
      hnow = hnext;
      hnext = headers(q + 64);
      beat(ticket);
    }
    const int pos = __builtin_amdgcn_readlane(hnow.x, nth);
    const int rows = __builtin_amdgcn_readlane(hnow.y, nth);
    g.r = (prog + pos)[(unsigned)(lane < rows ? lane : rows - 1)];
  };
  auto load_values = [&](ProgramStage& g) {
#pragma unroll
    for (int e = 0; e < kShort; ++e) g.v[e] = in[g.r.row.x + (e < g.r.row.y ? e : 0)];
  };
  auto step = [&](auto slot, int q) {
    ProgramStage& g = ring[decltype(slot)::value];
    const int p0 = g.r.row.x, len = g.r.row.y, nl = g.r.row.z;
    const int z[kBatch] = {g.r.z.x, g.r.z.y, g.r.z.z, g.r.z.w};
    const unsigned use[kBatch] = {(unsigned)g.r.use.x, (unsigned)g.r.use.y,
                                  (unsigned)g.r.use.z, (unsigned)g.r.use.w};
    double d[kBatch], w[kBatch][kBatch];
    auto ask = [&]() {
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        d[u] = raw_load(f + z[u]);
#pragma unroll
        for (int t = 0; t < kBatch; ++t)  // absent: the pivot once more
          w[u][t] = raw_load(f + z[u] + ((use[u] >> (8 * t) & 0xFF) == kNone ? 0 : t + 1));
      }
    };
    ask();
#pragma unroll
    for (int e = 0; e < kShort; ++e) buf[e * 64 + lane] = g.v[e];
    load_values(ring[(decltype(slot)::value + 1) % 4]);
    load_program(ring[(decltype(slot)::value + 2) % 4], q + 2);
    BuildWait wt;
    for (;;) {
      bool all = true;
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        bool ok = is_ready(d[u]);
#pragma unroll
        for (int t = 0; t < kBatch; ++t) ok = ok && is_ready(w[u][t]);
        all = all && (u >= nl || ok);
      }
      if (__all(all)) break;
      if (dead || !wt.again(ticket, ticks)) {
        if (!dead && lane == 0) atomicOr(error, 4);
        dead = true;
        break;
      }
      ask();
    }
    double dropped = 0.0;
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      if (!__any(u < nl)) break;
      const bool has = u < nl;
      const double l = buf[u * 64 + lane] / d[u];
      if (has) buf[u * 64 + lane] = l;
      double x[kBatch];
      unsigned at[kBatch];
#pragma unroll
      for (int t = 0; t < kBatch; ++t) {
        const unsigned m = use[u] >> (8 * t) & 0xFF;
        at[t] = (has && m < (unsigned)kShort ? m : (unsigned)kShort) * 64 + lane;
        x[t] = buf[at[t]];
      }
#pragma unroll
      for (int t = 0; t < kBatch; ++t) {
        const double p = l * w[u][t];
        buf[at[t]] = x[t] - p;
        if (modified && has && (use[u] >> (8 * t) & 0xFF) == kDrop) dropped = dropped + p;
      }
    }
    if (modified) buf[nl * 64 + lane] = buf[nl * 64 + lane] - dropped;
#pragma unroll
    for (int e = 0; e < kShort; ++e)
      if (e < len) store_ready(f + p0 + e, buf[e * 64 + lane]);
    __builtin_amdgcn_wave_barrier();
  };
  load_program(ring[0], 0);
  load_program(ring[1], 1);
  load_values(ring[0]);
  for (int q = 0;; q += 4) {
    step(std::integral_constant<int, 0>{}, q);
    if (q + 1 >= count) break;
    step(std::integral_constant<int, 1>{}, q + 1);
    if (q + 2 >= count) break;
    step(std::integral_constant<int, 2>{}, q + 2);
    if (q + 3 >= count) break;
    step(std::integral_constant<int, 3>{}, q + 3);
    if (q + 4 >= count) break;
  }
  tile_done(ticket, tiles);
}

__global__ void tri_fill_words_kernel(unsigned long long* p, unsigned long long v,
                                      int64_t n) {
  for (int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; k < n;
       k += (int64_t)gridDim.x * blockDim.x)
    p[k] = v;
}

template <typename K>
void fill_words(DevBuf<K>& b, unsigned long long v, hipStream_t s) {
  const int64_t words = (int64_t)(b.n * sizeof(K) / 8);
  hipLaunchKernelGGL(tri_fill_words_kernel,
                     dim3((unsigned)std::min<int64_t>((words + 255) / 256, 4096)), dim3(256),
                     0, s, (unsigned long long*)b.p, v, words);
  SPK_HIP_TRY(hipGetLastError());
}

int tile_count(int64_t n) { return (int)((n + kTileRows - 1) / kTileRows); }

}  // namespace

template <>
TriView<double> TriTiles::view<double>() {
  return {n, tiles, rows.p, first.p, steps.p, cols.p, v64.p, d64.p};
}
template <>
TriView<float> TriTiles::view<float>() {
  if (!has32) {
    auto cast = [](DevBuf<double>& in, DevBuf<float>& out) {
      if (!in.p) return;
      out.alloc(in.n);
      hipLaunchKernelGGL(tri_cast_kernel,
                         dim3((unsigned)std::min<size_t>((in.n + 255) / 256, 16384)),
                         dim3(256), 0, stream(), in.p, out.p, (int64_t)in.n);
      SPK_HIP_TRY(hipGetLastError());
    };
    cast(v64, v32);
    cast(d64, d32);
    has32 = true;
  }
  return {n, tiles, rows.p, first.p, steps.p, cols.p, v32.p, d32.p};
}

void set_tri_wait(unsigned long long ticks) { g_wait_ticks = ticks; }

bool tri_levels(const TriPattern& P, DevBuf<int32_t>& lvl, int levels[2]) {
  levels[0] = levels[1] = 0;
  lvl.alloc((size_t)(2 * P.n + (P.n ? 0 : 1)));
  if (P.n == 0) return true;
  hipStream_t s = stream();
  constexpr int kMax = 2 * kTriTicketWords;
  // two tickets, two maxima, the error word
  DevBuf<int> st(kMax + 4);
  fill_words(st, 0, s);
  fill_words(lvl, ~0ull, s);
  const int tiles = tile_count(P.n);
  hipLaunchKernelGGL(tri_level_kernel, dim3(2 * tiles), dim3(kLevelBlock), 0, s, P, tiles,
                     lvl.p, st.p, st.p + kMax, st.p + kMax + 2, build_ticks());
  SPK_HIP_TRY(hipGetLastError());
  int h[3];
  SPK_HIP_TRY(hipMemcpyAsync(h, st.p + kMax, sizeof(h), hipMemcpyDeviceToHost, s));
  SPK_HIP_TRY(hipStreamSynchronize(s));
  levels[0] = h[0];
  levels[1] = h[1];
  return h[2] == 0;
}

void tri_layouts(const TriPattern& P, const int32_t* lvl, TriTiles& lower, TriTiles& upper) {
  hipStream_t s = stream();
  const size_t m = (size_t)tile_count(P.n);
  TriTiles* T[2] = {&lower, &upper};
  for (TriTiles* t : T) {
    t->n = P.n;
    t->tiles = (int)m;
  }
  if (P.n == 0) return;
  DevBuf<int> ent(2 * (m + 1) + 4);  // and the totals
  DevBuf<int2> step((size_t)(2 * P.n));
  int* total = ent.p + 2 * (m + 1);
  TriBuild B{};
  B.tiles = (int)m;
  for (int k = 0; k < 2; ++k) {
    T[k]->v64.release();  // of another layout
    T[k]->rows.alloc((size_t)P.n);
    T[k]->first.alloc(m + 1);
    B.lvl[k] = lvl + k * P.n;
    B.rows[k] = T[k]->rows.p;
    B.step[k] = step.p + k * P.n;
    B.first[k] = T[k]->first.p;
    B.ent[k] = ent.p + k * (m + 1);
  }
  hipLaunchKernelGGL(tri_order_kernel, dim3(2 * (unsigned)m), dim3(256), 0, s, P, B);
  hipLaunchKernelGGL(tri_scan_kernel, dim3(2), dim3(1024), 0, s, B, total);
  SPK_HIP_TRY(hipGetLastError());
  int h[4];
  SPK_HIP_TRY(hipMemcpyAsync(h, total, sizeof(h), hipMemcpyDeviceToHost, s));
  SPK_HIP_TRY(hipStreamSynchronize(s));
  for (int k = 0; k < 2; ++k) {
    T[k]->nsteps = h[2 * k];
    T[k]->groups = (int64_t)(unsigned)h[2 * k + 1];
    T[k]->steps.alloc((size_t)T[k]->nsteps);
    T[k]->cols.alloc((size_t)T[k]->groups);
    B.steps[k] = T[k]->steps.p;
    B.cols[k] = T[k]->cols.p;
  }
  hipLaunchKernelGGL(tri_fill_kernel, dim3(2 * (unsigned)m), dim3(256), 0, s, P, B);
  SPK_HIP_TRY(hipGetLastError());
}

void tri_values(const TriPattern& P, const double* w, TriTiles& lower, TriTiles& upper) {
  if (P.n == 0) return;
  TriTiles* T[2] = {&lower, &upper};
  TriValues B{};
  if (!upper.d64.p) upper.d64.alloc((size_t)P.n);
  for (int k = 0; k < 2; ++k) {
    if (!T[k]->v64.p) T[k]->v64.alloc((size_t)T[k]->groups * kBatch);
    B.nsteps[k] = T[k]->nsteps;
    B.rows[k] = T[k]->rows.p;
    B.steps[k] = T[k]->steps.p;
    B.v[k] = T[k]->v64.p;
  }
  B.d = upper.d64.p;
  const int64_t waves = (int64_t)lower.nsteps + upper.nsteps;
  hipLaunchKernelGGL(tri_value_kernel, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0,
                     stream(), P, B, w);
  SPK_HIP_TRY(hipGetLastError());
}

void tri_factor(const TriPattern& P, const TriTiles& lower, const double* in, DevBuf<double>& f,
                bool modified, int max_len, int max_side, int* ticket, int* error) {
  if (P.n == 0) return;
  hipStream_t s = stream();
  if (max_side <= kBatch) {
    DevBuf<RowProgram> prog((size_t)P.n);
    fill_words(f, Sentinel<double>::bits, s);
    hipLaunchKernelGGL(tri_program_kernel, dim3((unsigned)((P.n + 255) / 256)), dim3(256), 0,
                       s, P, (const int32_t*)lower.rows.p, prog.p);
    hipLaunchKernelGGL(tri_factor_short_kernel, dim3(lower.tiles), dim3(64), 0, s,
                       lower.tiles, (const int32_t*)lower.first.p, (const int4*)lower.steps.p,
                       (const RowProgram*)prog.p, in, f.p, modified ? 1 : 0, ticket, error,
                       build_ticks());
    SPK_HIP_TRY(hipGetLastError());
    return;
  }
  DevBuf<double> pivot((size_t)P.n);
  fill_words(pivot, Sentinel<double>::bits, s);
  SPK_HIP_TRY(hipMemcpyAsync(f.p, in, f.n * sizeof(double), hipMemcpyDeviceToDevice, s));
  TriView<double> v{P.n, lower.tiles, lower.rows.p, lower.first.p, lower.steps.p,
                    nullptr, nullptr, nullptr};
  hipLaunchKernelGGL(tri_factor_kernel, dim3(lower.tiles), dim3(64),
                     (size_t)max_len * 64 * (sizeof(double) + sizeof(int)), s, P, v, f.p,
                     pivot.p, max_len, modified ? 1 : 0, ticket, error, build_ticks());
  SPK_HIP_TRY(hipGetLastError());
}

template <typename T, bool LOWER>
void tri_sweep(TriTiles& A, T* b, T* x, bool reset_b, T* mark, int* ticket, int* error,
               hipStream_t s) {
  if (A.n == 0) return;
  const dim3 grid((A.tiles + kGroupTiles - 1) / kGroupTiles), block(64 * kGroupTiles);
  if (reset_b)
    hipLaunchKernelGGL((tri_sweep_kernel<T, LOWER, kReset>), grid, block, 0, s,
                       A.view<T>(), b, x, mark, ticket, error, sweep_ticks());
  else if (mark)
    hipLaunchKernelGGL((tri_sweep_kernel<T, LOWER, kMark>), grid, block, 0, s, A.view<T>(),
                       b, x, mark, ticket, error, sweep_ticks());
  else
    hipLaunchKernelGGL((tri_sweep_kernel<T, LOWER, kPlain>), grid, block, 0, s,
                       A.view<T>(), b, x, mark, ticket, error, sweep_ticks());
  SPK_HIP_TRY(hipGetLastError());
}
template void tri_sweep<double, true>(TriTiles&, double*, double*, bool, double*, int*, int*, hipStream_t);
template void tri_sweep<double, false>(TriTiles&, double*, double*, bool, double*, int*, int*, hipStream_t);
template void tri_sweep<float, true>(TriTiles&, float*, float*, bool, float*, int*, int*, hipStream_t);
template void tri_sweep<float, false>(TriTiles&, float*, float*, bool, float*, int*, int*, hipStream_t);

}  // namespace spk
