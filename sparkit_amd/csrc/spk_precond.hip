// spk_precond.hip -- Jacobi, ILU(0)/MILU(0) and SpMV preconditioners.
#include "spk_precond.hpp"

#include <algorithm>
#include <cstring>
#include <type_traits>
#include <utility>

#include "spk_vec.hpp"

namespace spk {
namespace {

// jacobi(A): d = extract_diagonal(A); zero -> error; d = 1/d (jacobi.hpp:27-35)
__global__ void invert_diag_kernel(const int32_t* rp, const int32_t* ci,
                                   const double* v, int64_t len, double* d,
                                   int* zero) {
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= len) return;
  int lo = rp[i], hi = rp[i + 1], e = hi;
  while (lo < hi) {
    int mid = lo + (hi - lo) / 2;
    if (ci[mid] < i) lo = mid + 1; else hi = mid;
  }
  double di = (lo < e && ci[lo] == i) ? v[lo] : 0.0;
  if (di == 0.0) {
    atomicOr(zero, 1);
    d[i] = 0.0;
  } else {
    d[i] = 1.0 / di;
  }
}

__global__ void to_f32_kernel(const double* in, float* out, int64_t n) {
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) out[i] = (float)in[i];
}

// One IKJ row of ilu0_impl (ilu.hpp:72-115) per thread, for the rows of one
// dependency level.  Multiply-adds are not contracted so that every update
// rounds exactly as the reference's w[pos] -= l_ik * w[q].
__global__ void ilu_factor_level_kernel(const int32_t* __restrict__ rows,
                                        int count,
                                        const int32_t* __restrict__ rp,
                                        const int32_t* __restrict__ ci,
                                        const int32_t* __restrict__ diag_pos,
                                        double* __restrict__ w, int modified) {
#pragma clang fp contract(off)
  int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= count) return;
  const int i = rows[t];
  const int pe = rp[i + 1];
  double dropped = 0.0;
  for (int p = rp[i]; p < pe; ++p) {
    const int k = ci[p];
    if (k >= i) break;
    w[p] = w[p] / w[diag_pos[k]];
    const double l_ik = w[p];
    int pi = p + 1;  // row i positions with column > k
    const int qe = rp[k + 1];
    for (int q = diag_pos[k] + 1; q < qe; ++q) {
      const int j = ci[q];
      while (pi < pe && ci[pi] < j) ++pi;
      if (pi < pe && ci[pi] == j) {
        w[pi] = w[pi] - l_ik * w[q];
      } else if (modified) {
        dropped = dropped + l_ik * w[q];
      }
    }
  }
  if (modified) w[diag_pos[i]] = w[diag_pos[i]] - dropped;
}

// Split the factored rows into L (unit diagonal last) and U (diagonal
// first): ilu.hpp:123-141.
__global__ void ilu_split_kernel(TriPattern P, const double* __restrict__ w,
                                 const int32_t* __restrict__ lrp,
                                 int32_t* __restrict__ lci, double* __restrict__ lv,
                                 const int32_t* __restrict__ urp,
                                 int32_t* __restrict__ uci, double* __restrict__ uv) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= P.n) return;
  const int dp = P.dpos[i];
  int lk = lrp[i], uk = urp[i];
  for (int p = P.rp[i]; p < dp; ++p, ++lk) {
    lci[lk] = P.ci[p];
    lv[lk] = w[p];
  }
  lci[lk] = (int32_t)i;
  lv[lk] = 1.0;
  for (int p = dp; p < P.rp[i + 1]; ++p, ++uk) {
    uci[uk] = P.ci[p];
    uv[uk] = w[p];
  }
}

// Each row's diagonal position (ilu.hpp:54-66); out[0] |= 1 a missing
// diagonal, 2 columns that do not ascend, 4 a repeated diagonal, 8 another
// repeated column; out[1] the longest row; out[4] the most entries on one
// side of the diagonal; out[5] how far the farthest column is from its row;
// *lower: the strictly lower entries.
__global__ void ilu_rows_kernel(int64_t n, const int32_t* __restrict__ rp,
                                const int32_t* __restrict__ ci, int32_t* __restrict__ dpos,
                                int* out, unsigned long long* lower) {
  __shared__ unsigned long long red[256 / 64];
  unsigned long long below = 0;
  int bad = 0, len = 0, side = 0, reach = 0;
  for (int64_t i = blockIdx.x * (int64_t)256 + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * 256) {
    const int p0 = rp[i], pe = rp[i + 1];
    int d = -1, last = -1;
    for (int p = p0; p < pe; ++p) {
      const int c = ci[p];
      if (c < last) bad |= 2;
      if (c == last && c != i) bad |= 8;
      if (c == i) {
        if (d >= 0) bad |= 4;
        else d = p;
      }
      last = c;
    }
    if (d < 0) {
      bad |= 1;
      d = p0;
    }
    dpos[i] = d;
    below += (unsigned long long)(d - p0);
    if (pe > p0) {  // ascending, or to be sorted
      const int lo = (int)i - ci[p0], hi = ci[pe - 1] - (int)i;
      reach = lo > reach ? lo : reach;
      reach = hi > reach ? hi : reach;
    }
    len = pe - p0 > len ? pe - p0 : len;
    side = d - p0 > side ? d - p0 : side;
    side = pe - d - 1 > side ? pe - d - 1 : side;
  }
  below = block_reduce_sum<unsigned long long, 256>(below, red);
  for (int o = 32; o > 0; o >>= 1) {
    const int other = __shfl_xor(len, o, 64);
    len = other > len ? other : len;
    const int os = __shfl_xor(side, o, 64);
    side = os > side ? os : side;
    const int far = __shfl_xor(reach, o, 64);
    reach = far > reach ? far : reach;
    bad |= __shfl_xor(bad, o, 64);
  }
  if (threadIdx.x == 0) atomicAdd(lower, below);
  if ((threadIdx.x & 63) == 0) {
    if (bad) atomicOr(out, bad);
    atomicMax(out + 1, len);
    atomicMax(out + 4, side);
    atomicMax(out + 5, reach);
  }
}

__global__ void clear_words_kernel(int* p, int n) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) p[k] = 0;
}

constexpr int kErrorWords = 64;  // sweep status word + guard words
// Few levels: from 65,536 rows on one launch per level, below a window.
constexpr int64_t kLevelLaunchRows = 65536;
constexpr int64_t kLevelLaunchMaxLevels = 4096;

// A triangular sweep of few, wide levels in one launch: one thread per row in
// padded level order (a wavefront holds rows of one level, which do not wait
// for each other).  A small persistent grid walks the order, W threads at a
// time, so only a window of a few levels waits; a row's dependencies are polled
// kSweepBatch at a time and consumed in storage order, multiply-adds not
// contracted: bit-identical to the sequential reference
// (triangular_solve.hpp:42-53, 82-96).  Workgroups are dispatched in order, so
// the earliest unfinished wavefront always has its dependencies resident or
// finished.  reset_b returns b[i] to the sentinel after reading it; mark[i] is
// filled with it (the next sweep's output).
constexpr unsigned kSpinLimit = 1u << 22;
constexpr int kSweepBatch = 4;
template <typename T, bool LOWER>
__global__ __launch_bounds__(256) void window_sweep_kernel(
    const int32_t* __restrict__ rows, int n, const int32_t* __restrict__ rp,
    const int32_t* __restrict__ ci, const T* __restrict__ v, T* b, T* x, bool reset_b,
    T* mark, int* error) {
#pragma clang fp contract(off)
  const int W = gridDim.x * blockDim.x;
  for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < n; t += W) {
    const int i = rows[t];
    if (i < 0) continue;  // level padding
    const int p0 = rp[i], p1 = rp[i + 1];
    const int q1 = LOWER ? p1 - 1 : p1;
    const int pd = LOWER ? p1 - 1 : p0;
    T s = b[i];
    if (reset_b) b[i] = sentinel_value<T>();
    if (mark) mark[i] = sentinel_value<T>();
    int p = LOWER ? p0 : p0 + 1;
    unsigned spins = 0;
    while (p < q1) {
      const int cnt = q1 - p < kSweepBatch ? q1 - p : kSweepBatch;
      int c[kSweepBatch];
      T xv[kSweepBatch];
      bool ok[kSweepBatch];
#pragma unroll
      for (int k = 0; k < kSweepBatch; ++k) {
        ok[k] = k >= cnt;
        c[k] = k < cnt ? ci[p + k] : 0;
      }
      bool all = false;
      while (!all) {
        all = true;
#pragma unroll
        for (int k = 0; k < kSweepBatch; ++k) {
          if (!ok[k]) ok[k] = load_ready(x + c[k], &xv[k]);
          all = all && ok[k];
        }
        if (!all) {
          if (++spins > kSpinLimit) {
            atomicOr(error, LOWER ? 1 : 2);
            break;
          }
          __builtin_amdgcn_s_sleep(2);  // back off: fewer polls in flight
        }
      }
      if (!all) {  // expired wait: publish what there is (reported)
        p = q1;
        break;
      }
#pragma unroll
      for (int k = 0; k < kSweepBatch; ++k)
        if (k < cnt) s = s - v[p + k] * xv[k];
      p += cnt;
    }
    store_ready(x + i, s / v[pd]);
    // keep this row's publication ahead of the next row's waits
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
  }
}

// One dependency level of a triangular sweep: every row of the level reads
// only rows of earlier levels (final, previous launches), so plain loads
// suffice.  Same operation order as the sweeps in tiles.
template <typename T, bool LOWER>
__global__ __launch_bounds__(256) void level_sweep_kernel(
    const int32_t* __restrict__ rows, int count, const int32_t* __restrict__ rp,
    const int32_t* __restrict__ ci, const T* __restrict__ v, const T* b, T* x) {
#pragma clang fp contract(off)
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= count) return;
  const int i = rows[t];
  const int p0 = rp[i], p1 = rp[i + 1];
  const int q1 = LOWER ? p1 - 1 : p1;
  const int pd = LOWER ? p1 - 1 : p0;
  T s = b[i];
  for (int p = LOWER ? p0 : p0 + 1; p < q1; ++p) s = s - v[p] * x[ci[p]];
  x[i] = s / v[pd];
}

template <typename T>
__global__ void fill_sentinel_kernel(T* x, int64_t n) {
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) x[i] = sentinel_value<T>();
}

// group rows by level (counting sort); returns level pointer array
std::vector<int32_t> group_levels(const std::vector<int32_t>& lvl,
                                  std::vector<int32_t>& rows_out) {
  int32_t nl = 0;
  for (int32_t l : lvl) nl = std::max(nl, l + 1);
  std::vector<int32_t> ptr((size_t)nl + 1, 0);
  for (int32_t l : lvl) ptr[l + 1]++;
  for (int32_t l = 0; l < nl; ++l) ptr[l + 1] += ptr[l];
  std::vector<int32_t> fill(ptr.begin(), ptr.end() - 1);
  rows_out.resize(lvl.size());
  for (size_t i = 0; i < lvl.size(); ++i) rows_out[fill[lvl[i]]++] = (int32_t)i;
  return ptr;
}

// rows grouped by level, each level padded with -1 to a multiple of 64
std::vector<int32_t> pad_levels(const std::vector<int32_t>& rows,
                                const std::vector<int32_t>& ptr) {
  std::vector<int32_t> out;
  out.reserve(rows.size() + 64 * (ptr.size() - 1));
  for (size_t l = 0; l + 1 < ptr.size(); ++l) {
    out.insert(out.end(), rows.begin() + ptr[l], rows.begin() + ptr[l + 1]);
    out.resize((out.size() + 63) / 64 * 64, -1);
  }
  return out;
}

// an n x n store with the given row offsets, columns and values not set
spk_csr_s* make_store(int64_t n, std::vector<int32_t>&& rp) {
  auto* S = new spk_csr_s();
  try {
    S->allocate(n, n, rp[(size_t)n]);
    SPK_HIP_TRY(hipMemcpyAsync(S->rp.p, rp.data(), rp.size() * 4, hipMemcpyHostToDevice,
                               stream()));
    SPK_HIP_TRY(hipStreamSynchronize(stream()));
    S->h_rp = std::move(rp);
    upload_plan(*S, build_spmv_plan(S->h_rp.data(), n, &S->nlong));
  } catch (...) {
    delete S;
    throw;
  }
  return S;
}

inline unsigned blocks_for(int64_t n) { return (unsigned)((n + 255) / 256); }

}  // namespace
}  // namespace spk

using namespace spk;

spk_precond_s::~spk_precond_s() {
  delete L;
  delete U;
  delete Ls;
  delete Us;
}

const float* spk_precond_s::inv_diag32() {
  if (!has32) {
    inv_d32.alloc((size_t)n);
    if (n > 0)
      hipLaunchKernelGGL(to_f32_kernel, dim3(blocks_for(n)), dim3(256), 0,
                         stream(), inv_d64.p, inv_d32.p, n);
    SPK_HIP_TRY(hipGetLastError());
    has32 = true;
  }
  return inv_d32.p;
}

// Where a tile's chain of steps (2,048 rows: 32 and more) is longer than the
// levels, and its rows wait for other tiles': up to 4 levels anywhere; beyond,
// from three tiles to 2^20 rows, up to 32 levels (24 of long rows), 64 where
// they are launched one by one; not where rows reach less far than a tile.  One
// application (both
// triangles, FP64) in tiles / as below: two colours of a 5-point stencil 100^2
// 0.077 / 0.030 ms, 1000^2 0.093 / 0.058; four of a 9-point one 100^2 0.146 /
// 0.042, 700^2 0.239 / 0.078; stencils in random order 3,600 rows (12 levels)
// 0.065 / 0.072, 62,500 0.217 / 0.088, 512,000 (20) 0.399 / 0.322, 4.1M (22)
// 1.03 / 1.44; 10 random entries a row, 30,000 rows (31) 0.48 / 0.34; up to 60,
// 30,000 (26) 0.67 / 1.27;
// 27 points 8,000 (49) 0.45 / 0.92, 216,000 (54) 1.94 / 1.77;
// dense blocks of 30 rows, 150,000 (30, within the blocks) 0.29 / 0.72.
bool spk_precond_s::few_levels() const {
  const int levels = std::max(levels_l, levels_u);
  if (n <= kTileRows) return levels <= 4;
  if (reach < kTileRows) return false;
  return levels <= 4 || (n > 2 * kTileRows && n <= (1 << 20) &&
                         levels <= (n >= kLevelLaunchRows    ? 64
                                    : max_len <= kTriFactorLen ? 32
                                                               : 24));
}

void spk_precond_s::choose_sweep(int schedule) {
  const bool launch =
      n >= kLevelLaunchRows && std::max(levels_l, levels_u) <= kLevelLaunchMaxLevels;
  sweep = schedule == SPK_ILU_LEVELS || twice ? kLevels
          : !few_levels() && n < kMaxTileSweepRows ? kTiles
          : schedule == SPK_ILU_SYNC_FREE || !launch ? kWindow
                                                     : kLevels;
}

void spk_precond_s::set_schedule(int schedule, const int32_t* lvl) {
  choose_sweep(schedule);
  if (sweep == kTiles) return;
  build_factors();
  build_levels(lvl);
  if (sweep == kWindow) build_windows();
}

// ilu0_impl (ilu.hpp:35-141): the pattern, both triangles' layouts and the
// numeric factorization, all on the device; the host reads back a few
// counters in between.
void spk_precond_s::factor(const spk_csr_s& A, bool modified) {
  hipStream_t s = stream();
  n = A.nrows;
  nnz = A.nnz;
  rp.alloc((size_t)n + 1);
  ci.alloc((size_t)nnz);
  w.alloc((size_t)nnz);
  dpos.alloc((size_t)n);
  sweep_error.alloc(kErrorWords);
  constexpr int kCount = 2 * kTriTicketWords;  // counters of the construction
  ticket.alloc(kCount + 6);
  SPK_HIP_TRY(hipMemcpyAsync(rp.p, A.rp.p, (n + 1) * 4, hipMemcpyDeviceToDevice, s));
  if (nnz) SPK_HIP_TRY(hipMemcpyAsync(ci.p, A.ci.p, nnz * 4, hipMemcpyDeviceToDevice, s));
  DevBuf<double> ordered;  // the values, where the rows had to be sorted
  hipLaunchKernelGGL(clear_words_kernel, dim3(1), dim3(256), 0, s, sweep_error.p, kErrorWords);
  int h[6];
  for (bool sorted = false;;) {
    hipLaunchKernelGGL(clear_words_kernel, dim3(1), dim3(256), 0, s, ticket.p,
                       kCount + 6);
    hipLaunchKernelGGL(ilu_rows_kernel, dim3(std::min(blocks_for(n), 1024u)), dim3(256), 0, s, n,
                       (const int32_t*)rp.p, (const int32_t*)ci.p, dpos.p,
                       ticket.p + kCount, (unsigned long long*)(ticket.p + kCount + 2));
    SPK_HIP_TRY(hipGetLastError());
    SPK_HIP_TRY(hipMemcpyAsync(h, ticket.p + kCount, sizeof(h), hipMemcpyDeviceToHost, s));
    SPK_HIP_TRY(hipStreamSynchronize(s));
    SPK_REQUIRE((h[0] & 1) == 0, SPK_INVALID_ARGUMENT, "ilu0: missing diagonal entry");
    if ((h[0] & 2) == 0 || sorted) break;
    sort_rows(A, ordered);  // a caller's CSR rows in another order than ascending
    sorted = true;
  }
  unsigned long long below;
  std::memcpy(&below, h + 2, sizeof(below));
  nnz_l = (int64_t)below + n;
  nnz_u = nnz - (int64_t)below;
  reach = h[5];
  const TriPattern P = pattern();
  max_len = h[1];
  twice = (h[0] & 4) != 0;
  // Long rows, or a column twice: the factorization by levels.  Their levels
  // come from the host, and those of small factors with more than four entries
  // on a side: a dependency takes the device a round trip, the host a few
  // nanoseconds (a chain of 100,000 rows with two of 4,096 entries 80 / 1 ms,
  // 27 points 20^3 1.84 / 0.4).
  const bool long_rows = max_len > kTriFactorLen || (h[0] & 12) != 0;
  DevBuf<int32_t> lvl;
  bool on_host = long_rows || (h[4] > kBatch && nnz <= (1 << 20)), tiles, tiled;
  auto lay_out = [&] {
    int count[2];
    find_levels(lvl, count, on_host);
    levels_l = count[0];
    levels_u = count[1];
    choose_sweep(SPK_ILU_AUTO);
    tiles = sweep == kTiles;
    if (tiles) tri_layouts(P, lvl.p, lower, upper);
  };
  lay_out();
  const double* in = ordered.p ? ordered.p : A.v64.p;
  // A tile works on one step at a time, the launches on a whole level: rows of
  // more than four entries on a side, a row's elimination being hundreds of
  // loads one after the other, take the tiles where those have fewer steps by
  // a third.  Set-up in tiles / by levels: 20 random entries a row, 20,000 rows
  // (54 levels) 28.8 / 13.1 ms, 27 points 20^3 natural 15.3 / 13.4, 40^3
  // natural 29 / 39, 64^3 natural 47 / 79.
  tiled = tiles && !long_rows &&
          (h[4] <= kBatch || 2 * (int64_t)levels_l * lower.tiles > 3 * (int64_t)lower.nsteps);
  for (;;) {
    if (tiled)
      tri_factor(P, lower, in, w, modified, h[1], h[4], ticket.p, sweep_error.p);
    else
      factor_by_levels(in, modified, lvl.p);
    if (tiles) tri_values(P, w.p, lower, upper);
    if (!tiled || !sweep_errors()) break;
    // a wait expired: again, without waits and with nothing that came of them
    tiled = false;
    on_host = true;
    lay_out();
  }
  set_schedule(SPK_ILU_AUTO, lvl.p);
  SPK_HIP_TRY(hipStreamSynchronize(s));
}

// One launch per dependency level, a thread per row.
void spk_precond_s::factor_by_levels(const double* in, bool modified, const int32_t* lvl) {
  hipStream_t s = stream();
  SPK_HIP_TRY(hipMemcpyAsync(w.p, in, nnz * 8, hipMemcpyDeviceToDevice, s));
  build_levels(lvl);
  for (size_t l = 0; l + 1 < lvl_ptr_l.size(); ++l) {
    const int cnt = lvl_ptr_l[l + 1] - lvl_ptr_l[l];
    hipLaunchKernelGGL(ilu_factor_level_kernel, dim3(blocks_for(cnt)), dim3(256), 0, s,
                       lvl_rows_l.p + lvl_ptr_l[l], cnt, rp.p, ci.p, dpos.p, w.p,
                       modified ? 1 : 0);
  }
  SPK_HIP_TRY(hipGetLastError());
}

// tri_levels, or the same on the host (also where a wait of it expired, or where
// a row would wait for itself)
void spk_precond_s::find_levels(DevBuf<int32_t>& lvl, int count[2], bool host) {
  if (!host && !twice && tri_levels(pattern(), lvl, count)) return;
  hipStream_t s = stream();
  lvl.reserve((size_t)(2 * n));
  std::vector<int32_t> hrp((size_t)n + 1), hd((size_t)n), hc((size_t)nnz), l((size_t)(2 * n));
  SPK_HIP_TRY(hipMemcpyAsync(hrp.data(), rp.p, (n + 1) * 4, hipMemcpyDeviceToHost, s));
  SPK_HIP_TRY(hipMemcpyAsync(hd.data(), dpos.p, n * 4, hipMemcpyDeviceToHost, s));
  SPK_HIP_TRY(hipMemcpyAsync(hc.data(), ci.p, nnz * 4, hipMemcpyDeviceToHost, s));
  SPK_HIP_TRY(hipStreamSynchronize(s));
  count[0] = count[1] = 0;
  auto row = [&](int64_t i, int64_t p, int64_t pe, int32_t* out, int* most) {
    int32_t v = 0;
    for (; p < pe; ++p)
      if (hc[(size_t)p] != i) v = std::max(v, out[hc[(size_t)p]] + 1);
    out[i] = v;
    *most = std::max(*most, v + 1);
  };
  for (int64_t i = 0; i < n; ++i) row(i, hrp[i], hd[i], l.data(), count);
  for (int64_t i = n - 1; i >= 0; --i)
    row(i, hd[i] + 1, hrp[i + 1], l.data() + n, count + 1);
  SPK_HIP_TRY(hipMemcpyAsync(lvl.p, l.data(), 8 * n, hipMemcpyHostToDevice, s));
  SPK_HIP_TRY(hipStreamSynchronize(s));
}

void spk_precond_s::sort_rows(const spk_csr_s& A, DevBuf<double>& values) {
  hipStream_t s = stream();
  std::vector<int32_t> c((size_t)nnz);
  std::vector<double> v((size_t)nnz);
  SPK_HIP_TRY(hipMemcpyAsync(c.data(), ci.p, nnz * 4, hipMemcpyDeviceToHost, s));
  SPK_HIP_TRY(hipMemcpyAsync(v.data(), A.v64.p, nnz * 8, hipMemcpyDeviceToHost, s));
  SPK_HIP_TRY(hipStreamSynchronize(s));
  std::vector<std::pair<int32_t, double>> row;
  for (int64_t i = 0; i < n; ++i) {
    const size_t a = (size_t)A.h_rp[(size_t)i], b = (size_t)A.h_rp[(size_t)i + 1];
    row.clear();
    for (size_t k = a; k < b; ++k) row.emplace_back(c[k], v[k]);
    std::stable_sort(row.begin(), row.end(),
                     [](const auto& x, const auto& y) { return x.first < y.first; });
    for (size_t k = a; k < b; ++k) {
      c[k] = row[k - a].first;
      v[k] = row[k - a].second;
    }
  }
  SPK_HIP_TRY(hipMemcpyAsync(ci.p, c.data(), nnz * 4, hipMemcpyHostToDevice, s));
  values.alloc((size_t)nnz);
  SPK_HIP_TRY(hipMemcpyAsync(values.p, v.data(), nnz * 8, hipMemcpyHostToDevice, s));
  SPK_HIP_TRY(hipStreamSynchronize(s));
}

template <typename T>
static T* sentinel_buffer(DevBuf<T>& buf, int64_t n) {
  if (buf.p == nullptr || buf.n < (size_t)n) {
    buf.alloc((size_t)n);
    hipLaunchKernelGGL((fill_sentinel_kernel<T>), dim3(blocks_for(n)),
                       dim3(256), 0, stream(), buf.p, n);
    SPK_HIP_TRY(hipGetLastError());
  }
  return buf.p;
}

template <>
double* spk_precond_s::tmp<double>() {
  return sentinel_buffer(tmp64, n);
}
template <>
float* spk_precond_s::tmp<float>() {
  return sentinel_buffer(tmp32, n);
}

void spk_precond_s::reset_sentinels() {
  if (tmp64.p)
    hipLaunchKernelGGL((fill_sentinel_kernel<double>), dim3(blocks_for(n)),
                       dim3(256), 0, stream(), tmp64.p, n);
  if (tmp32.p)
    hipLaunchKernelGGL((fill_sentinel_kernel<float>), dim3(blocks_for(n)),
                       dim3(256), 0, stream(), tmp32.p, n);
  SPK_HIP_TRY(hipGetLastError());
}

int spk_precond_s::sweep_errors() {
  // word 0: 1 = a forward, 2 = a backward sweep's bounded wait expired, 4 =
  // the factorization's;
  // words 1..kErrorWords-1 must stay zero (a guard against stray writes)
  int h[kErrorWords];
  SPK_HIP_TRY(hipMemcpyAsync(h, sweep_error.p, sizeof(h), hipMemcpyDeviceToHost,
                             stream()));
  SPK_HIP_TRY(hipStreamSynchronize(stream()));
  bool guard_ok = true;
  for (int k = 1; k < kErrorWords; ++k) guard_ok = guard_ok && h[k] == 0;
  if (h[0] == 0 && guard_ok) return 0;
  SPK_HIP_TRY(hipMemsetAsync(sweep_error.p, 0, sizeof(h), stream()));
  SPK_HIP_TRY(hipStreamSynchronize(stream()));
  SPK_REQUIRE(guard_ok, SPK_HIP_ERROR,
              "ILU sweep status words overwritten (a stray device write)");
  return h[0];
}

void spk_precond_s::check_sweeps() {
  if (kind != kIlu) return;
  const int e = sweep_errors();
  SPK_REQUIRE(e == 0, SPK_HIP_ERROR,
              std::string("ILU triangular sweep: bounded wait expired in the ") +
                  (e & 1 ? "forward" : "") + (e == 3 ? " and " : "") +
                  (e & 2 ? "backward" : "") + " sweep (results invalid)");
}

template <typename T, bool LOWER>
void spk_precond_s::level_sweep(const T* b, T* x) {
  hipStream_t s = stream();
  CsrView<T> v = (LOWER ? L : U)->view<T>();
  const std::vector<int32_t>& ptr = LOWER ? lvl_ptr_l : lvl_ptr_u;
  const int32_t* rows = LOWER ? lvl_rows_l.p : lvl_rows_u.p;
  for (size_t l = 0; l + 1 < ptr.size(); ++l) {
    const int cnt = ptr[l + 1] - ptr[l];
    hipLaunchKernelGGL((level_sweep_kernel<T, LOWER>), dim3(blocks_for(cnt)),
                       dim3(256), 0, s, rows + ptr[l], cnt, v.rp, v.ci, v.v, b, x);
  }
  SPK_HIP_TRY(hipGetLastError());
}

template <typename T, bool LOWER>
void spk_precond_s::one_launch(T* b, T* x, bool reset_b, T* mark) {
  hipStream_t s = stream();
  if (sweep == kTiles) {
    tri_sweep<T, LOWER>(LOWER ? lower : upper, b, x, reset_b, mark,
                        ticket.p + (LOWER ? 0 : kTriTicketWords), sweep_error.p, s);
    return;
  }
  const CsrView<T> v = (LOWER ? L : U)->view<T>();
  hipLaunchKernelGGL((window_sweep_kernel<T, LOWER>),
                     dim3(LOWER ? sweep_grid_l : sweep_grid_u), dim3(256), 0, s,
                     (const int32_t*)(LOWER ? sweep_rows_l : sweep_rows_u).p,
                     (int)(LOWER ? sweep_len_l : sweep_len_u), v.rp, v.ci, v.v, b, x, reset_b,
                     mark, sweep_error.p);
  SPK_HIP_TRY(hipGetLastError());
}

template <typename T>
void spk_precond_s::forward(const T* b, T* x) {
  if (sweep == kLevels) {
    level_sweep<T, true>(b, x);
    return;
  }
  hipLaunchKernelGGL((fill_sentinel_kernel<T>), dim3(blocks_for(n)), dim3(256), 0, stream(),
                     x, n);
  SPK_HIP_TRY(hipGetLastError());
  one_launch<T, true>((T*)b, x, false, nullptr);
}

void spk_precond_s::require_backward() const {
  SPK_REQUIRE(!twice, SPK_INVALID_ARGUMENT,
              "ilu0: a row repeats its diagonal entry, its backward solve would read its "
              "own result");
}

template <typename T>
void spk_precond_s::backward(const T* b, T* x) {
  require_backward();
  if (sweep == kLevels) {
    level_sweep<T, false>(b, x);
    return;
  }
  hipLaunchKernelGGL((fill_sentinel_kernel<T>), dim3(blocks_for(n)), dim3(256), 0, stream(),
                     x, n);
  SPK_HIP_TRY(hipGetLastError());
  one_launch<T, false>((T*)b, x, false, nullptr);
}

void spk_precond_s::build_factors() {
  if (L) return;
  hipStream_t s = stream();
  std::vector<int32_t> hrp((size_t)n + 1), hd((size_t)n), lrp((size_t)n + 1),
      urp((size_t)n + 1);
  SPK_HIP_TRY(hipMemcpyAsync(hrp.data(), rp.p, (n + 1) * 4, hipMemcpyDeviceToHost, s));
  SPK_HIP_TRY(hipMemcpyAsync(hd.data(), dpos.p, n * 4, hipMemcpyDeviceToHost, s));
  SPK_HIP_TRY(hipStreamSynchronize(s));
  for (size_t i = 0; i < (size_t)n; ++i) {
    lrp[i + 1] = lrp[i] + hd[i] - hrp[i] + 1;
    urp[i + 1] = urp[i] + hrp[i + 1] - hd[i];
  }
  spk_csr_s* l = make_store(n, std::move(lrp));
  try {
    U = make_store(n, std::move(urp));
  } catch (...) {
    delete l;
    throw;
  }
  L = l;
  hipLaunchKernelGGL(ilu_split_kernel, dim3(blocks_for(n)), dim3(256), 0, s, pattern(),
                     (const double*)w.p, (const int32_t*)L->rp.p, L->ci.p, L->v64.p,
                     (const int32_t*)U->rp.p, U->ci.p, U->v64.p);
  SPK_HIP_TRY(hipGetLastError());
}

void spk_precond_s::build_levels(const int32_t* lvl) {
  if (lvl_rows_l.p) return;
  hipStream_t s = stream();
  DevBuf<int32_t> own;
  if (!lvl) {
    int count[2];
    find_levels(own, count, false);
    lvl = own.p;
  }
  std::vector<int32_t> h((size_t)(2 * n));
  SPK_HIP_TRY(hipMemcpyAsync(h.data(), lvl, 8 * n, hipMemcpyDeviceToHost, s));
  SPK_HIP_TRY(hipStreamSynchronize(s));
  std::vector<int32_t> rows_l, rows_u;
  lvl_ptr_l = group_levels({h.begin(), h.begin() + n}, rows_l);
  lvl_ptr_u = group_levels({h.begin() + n, h.end()}, rows_u);
  DevBuf<int32_t> l((size_t)n), u((size_t)n);
  SPK_HIP_TRY(hipMemcpyAsync(l.p, rows_l.data(), n * 4, hipMemcpyHostToDevice, s));
  SPK_HIP_TRY(hipMemcpyAsync(u.p, rows_u.data(), n * 4, hipMemcpyHostToDevice, s));
  SPK_HIP_TRY(hipStreamSynchronize(s));
  if (sweep == kWindow) {
    pad_order(rows_u, lvl_ptr_u, sweep_rows_u, &sweep_len_u, &sweep_grid_u);
    pad_order(rows_l, lvl_ptr_l, sweep_rows_l, &sweep_len_l, &sweep_grid_l);
  }
  lvl_rows_l = std::move(l);
  lvl_rows_u = std::move(u);
}

// a padded order, and a grid of about four levels of threads
void spk_precond_s::pad_order(const std::vector<int32_t>& rows,
                              const std::vector<int32_t>& ptr, DevBuf<int32_t>& out,
                              int64_t* len, unsigned* grid) {
  hipStream_t s = stream();
  const std::vector<int32_t> padded = pad_levels(rows, ptr);
  SPK_REQUIRE(padded.size() < (size_t)INT32_MAX, SPK_INVALID_ARGUMENT,
              "too many rows for the sweep order");
  DevBuf<int32_t> d(padded.size());
  SPK_HIP_TRY(hipMemcpyAsync(d.p, padded.data(), padded.size() * 4, hipMemcpyHostToDevice, s));
  SPK_HIP_TRY(hipStreamSynchronize(s));
  *len = (int64_t)padded.size();
  const int64_t levels = (int64_t)ptr.size() - 1;
  const int64_t w = levels > 0 ? *len / levels : 64;
  const int64_t cap = std::max<int64_t>(4, 4 * ctx().num_cus);
  const int64_t g = std::max<int64_t>(4, std::min((4 * w + 255) / 256, cap));
  *grid = (unsigned)std::min<int64_t>(g, blocks_for(std::max<int64_t>(*len, 1)));
  out = std::move(d);
}

void spk_precond_s::build_windows() {
  if (sweep_rows_l.p) return;
  hipStream_t s = stream();
  std::vector<int32_t> l((size_t)n), u((size_t)n);
  SPK_HIP_TRY(hipMemcpyAsync(l.data(), lvl_rows_l.p, n * 4, hipMemcpyDeviceToHost, s));
  SPK_HIP_TRY(hipMemcpyAsync(u.data(), lvl_rows_u.p, n * 4, hipMemcpyDeviceToHost, s));
  SPK_HIP_TRY(hipStreamSynchronize(s));
  pad_order(u, lvl_ptr_u, sweep_rows_u, &sweep_len_u, &sweep_grid_u);
  pad_order(l, lvl_ptr_l, sweep_rows_l, &sweep_len_l, &sweep_grid_l);
}

// strict part of one factor row: L drops its last entry (the unit
// diagonal), U its first (the diagonal, kept in d)
__global__ void strict_copy_kernel(int64_t n, const int32_t* __restrict__ rp,
                                   const int32_t* __restrict__ ci,
                                   const double* __restrict__ v, bool lower,
                                   int32_t* __restrict__ sci,
                                   double* __restrict__ sv,
                                   double* __restrict__ d) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int a = rp[i], b = rp[i + 1];
  if (lower) {
    for (int k = a; k < b - 1; ++k) { sci[k - i] = ci[k]; sv[k - i] = v[k]; }
  } else {
    d[i] = v[a];
    for (int k = a + 1; k < b; ++k) { sci[k - i - 1] = ci[k]; sv[k - i - 1] = v[k]; }
  }
}

void spk_precond_s::build_strict() {
  if (Ls) return;
  build_factors();
  hipStream_t s = stream();
  du64.alloc((size_t)(n > 0 ? n : 1));
  for (int f = 0; f < 2; ++f) {
    spk_csr_s* F = f == 0 ? L : U;
    std::vector<int32_t> hrp((size_t)n + 1);
    for (int64_t i = 0; i <= n; ++i) hrp[(size_t)i] = F->h_rp[(size_t)i] - (int32_t)i;
    auto* S = new spk_csr_s();
    try {
      S->allocate(n, n, F->nnz - n);
      SPK_HIP_TRY(hipMemcpyAsync(S->rp.p, hrp.data(), (n + 1) * sizeof(int32_t),
                                 hipMemcpyHostToDevice, s));
      if (n > 0)
        hipLaunchKernelGGL(strict_copy_kernel, dim3(blocks_for(n)), dim3(256), 0,
                           s, n, (const int32_t*)F->rp.p, (const int32_t*)F->ci.p,
                           (const double*)F->v64.p, f == 0, S->ci.p, S->v64.p,
                           du64.p);
      SPK_HIP_TRY(hipGetLastError());
      SPK_HIP_TRY(hipStreamSynchronize(s));
      finish_store(*S, false);
    } catch (...) {
      delete S;
      throw;
    }
    (f == 0 ? Ls : Us) = S;
  }
}

template <typename T>
struct EpiJacLastForward {  // y = r - L_s y_old; z_0 = y / d (z may alias r)
  static constexpr bool kReduce = false;
  const T* r;
  T* __restrict__ y;
  const T* __restrict__ d;
  T* z;
  const int* done = nullptr;
  __device__ double row(int i, T s) const {
    const T yi = r[i] - s;
    y[i] = yi;
    z[i] = yi / d[i];
    return 0.0;
  }
  __device__ void finalize(double) const {}
};

template <typename T>
struct EpiJacBackward {  // z = (y - U_s z_old) / d
  static constexpr bool kReduce = false;
  const T* __restrict__ y;
  const T* __restrict__ d;
  T* __restrict__ z;
  const int* done = nullptr;
  __device__ double row(int i, T s) const {
    z[i] = (y[i] - s) / d[i];
    return 0.0;
  }
  __device__ void finalize(double) const {}
};

template <typename T>
static T* scratch_vec(DevBuf<T>& b, int64_t n) {
  if (b.n < (size_t)n) b.alloc((size_t)(n > 0 ? n : 1));
  return b.p;
}

template <typename T>
static void jac_buffers(spk_precond_s& P, T** a, T** b);
template <>
void jac_buffers<double>(spk_precond_s& P, double** a, double** b) {
  *a = scratch_vec(P.jb64a, P.n);
  *b = scratch_vec(P.jb64b, P.n);
}
template <>
void jac_buffers<float>(spk_precond_s& P, float** a, float** b) {
  *a = scratch_vec(P.jb32a, P.n);
  *b = scratch_vec(P.jb32b, P.n);
}
// a third buffer: z_0 for an odd sweep count >= 3, whose last forward pass
// gathers from b
template <typename T>
static T* jac_buffer_c(spk_precond_s& P);
template <>
double* jac_buffer_c<double>(spk_precond_s& P) { return scratch_vec(P.jb64c, P.n); }
template <>
float* jac_buffer_c<float>(spk_precond_s& P) { return scratch_vec(P.jb32c, P.n); }

template <typename T>
static const T* diag_u(spk_precond_s& P);
template <>
const double* diag_u<double>(spk_precond_s& P) { return P.du64.p; }
template <>
const float* diag_u<float>(spk_precond_s& P) {
  if (!P.du_has32) {
    P.du32.alloc((size_t)(P.n > 0 ? P.n : 1));
    if (P.n > 0)
      hipLaunchKernelGGL(to_f32_kernel, dim3(blocks_for(P.n)), dim3(256), 0,
                         stream(), (const double*)P.du64.p, P.du32.p, P.n);
    SPK_HIP_TRY(hipGetLastError());
    P.du_has32 = true;
  }
  return P.du32.p;
}

template <typename T>
void spk_precond_s::jacobi_apply(const T* in, T* out) {
  hipStream_t s = stream();
  const int k = jac_sweeps;
  T *a, *b;
  jac_buffers<T>(*this, &a, &b);
  const T* d = diag_u<T>(*this);
  // forward: y_0 = r, y_j = r - L_s y_{j-1}; y_k ends in a
  // backward: z_0 = y / d, z_j = (y - U_s z_{j-1}) / d; z_k ends in out
  // z_0 is written by the last forward pass: into out for an even k (in
  // may alias out: that pass reads in[i] only for its own row, before
  // writing z_0[i], and gathers from b), into b for k = 1 (its one pass
  // gathers in), into a third buffer for an odd k >= 3 (its last pass
  // gathers from b)
  T* z0 = k % 2 == 0 ? out : (k == 1 ? b : jac_buffer_c<T>(*this));
  const T* y = in;
  for (int j = 0; j < k; ++j) {
    T* dst = (k - j) % 2 == 1 ? a : b;
    if (j == k - 1)
      launch_spmv(*Ls, y, EpiJacLastForward<T>{in, dst, d, z0}, s);
    else
      launch_spmv(*Ls, y, EpiResidual<T>{in, dst}, s);
    y = dst;
  }
  if (k == 0) launch_map(n, [=] __device__(int64_t i) { z0[i] = y[i] / d[i]; });
  const T* z = z0;
  for (int j = 0; j < k; ++j) {
    T* dst = (k - j) % 2 == 1 ? out : b;
    launch_spmv(*Us, z, EpiJacBackward<T>{y, d, dst}, s);
    z = dst;
  }
}

template <typename T>
void spk_precond_s::apply(const T* in, T* out) {
  switch (kind) {
    case kIdentity:
      if (in != out)
        SPK_HIP_TRY(hipMemcpyAsync(out, in, (size_t)n * sizeof(T),
                                   hipMemcpyDeviceToDevice, stream()));
      break;
    case kJacobi: {
      const T* d = inv_diag<T>();
      launch_map(n, [=] __device__(int64_t i) { out[i] = d[i] * in[i]; });
      break;
    }
    case kIlu: {
      // ilu_apply: y = forward_solve(L, r); z = backward_solve(U, y).
      // Two launches: the forward sweep marks `out` with the sentinel after
      // reading in[i] (in may alias out), the backward sweep returns y to
      // the sentinel as it consumes it.
      if (jac_sweeps > 0) {
        jacobi_apply(in, out);
        break;
      }
      require_backward();
      T* y = tmp<T>();
      if (sweep == kLevels) {  // no waiting
        level_sweep<T, true>(in, y);
        level_sweep<T, false>((const T*)y, out);
        break;
      }
      one_launch<T, true>((T*)in, y, false, out);
      one_launch<T, false>(y, out, true, nullptr);
      break;
    }
    case kSpmv:
      launch_spmv(*M, in, EpiStore<T>{out}, stream());
      break;
    case kInnerCg:
      inner_cg_apply(in, out);
      break;
    case kInnerIr:
      inner_ir_apply(in, out);
      break;
  }
}

// z = up to inner_iters PCG steps on A z = r from z = 0 (the inner solve's
// vectors in inner_precision; r and z converted at the boundary)
template <typename U, typename T>
static void inner_cg_run(spk_precond_s& P, const T* in, T* out,
                         spk::DevBuf<U>& bb, spk::DevBuf<U>& zb) {
  const int64_t n = P.n;
  const U* b;
  U* z;
  if constexpr (std::is_same<U, T>::value) {
    b = in;
    z = out;
    if (in == out) {  // the solve reads b while it writes z
      bb.reserve((size_t)(n > 0 ? n : 1));
      SPK_HIP_TRY(hipMemcpyAsync(bb.p, in, (size_t)n * sizeof(U),
                                 hipMemcpyDeviceToDevice, stream()));
      b = bb.p;
    }
  } else {
    bb.reserve((size_t)(n > 0 ? n : 1));
    zb.reserve((size_t)(n > 0 ? n : 1));
    U* bp = bb.p;
    launch_map(n, [=] __device__(int64_t i) { bp[i] = (U)in[i]; });
    b = bp;
    z = zb.p;
  }
  launch_map(n, [=] __device__(int64_t i) { z[i] = U(0); });
  spk_solver_config c{P.inner_tol, P.inner_iters, P.inner_iters, 0,
                      P.inner_precision, 0, 0};
  spk_summary sum{};
  const spk_status st = spk_cg_solve(P.inner_A, P.inner_M, nullptr, &c, b, z,
                                     &sum, nullptr);
  if (st != SPK_OK && st != SPK_BREAKDOWN)
    throw Error{st, std::string("inner PCG: ") + spk_last_error()};
  P.inner_total += sum.computed_iterations;
  if constexpr (!std::is_same<U, T>::value) {
    const U* zp = z;
    launch_map(n, [=] __device__(int64_t i) { out[i] = (T)zp[i]; });
  }
}

template <typename T>
void spk_precond_s::inner_cg_apply(const T* in, T* out) {
  if (inner_precision == SPK_F32)
    inner_cg_run<float, T>(*this, in, out, ib32, iz32);
  else
    inner_cg_run<double, T>(*this, in, out, ib64, iz64);
}

// z = spk_ir_solve(inner_A z = r) from z = 0 with inner_M and inner_ir (the
// solve's right-hand side and result are FP64: converted at the boundary
// when the caller's vectors are FP32)
template <typename T>
void spk_precond_s::inner_ir_apply(const T* in, T* out) {
  const double* b;
  double* z;
  const size_t m = (size_t)(n > 0 ? n : 1);
  if constexpr (std::is_same<T, double>::value) {
    b = in;
    z = out;
    if (in == out) {  // the solve reads b while it writes z
      ib64.reserve(m);
      SPK_HIP_TRY(hipMemcpyAsync(ib64.p, in, (size_t)n * sizeof(double),
                                 hipMemcpyDeviceToDevice, stream()));
      b = ib64.p;
    }
  } else {
    ib64.reserve(m);
    iz64.reserve(m);
    double* bp = ib64.p;
    launch_map(n, [=] __device__(int64_t i) { bp[i] = (double)in[i]; });
    b = bp;
    z = iz64.p;
  }
  launch_map(n, [=] __device__(int64_t i) { z[i] = 0.0; });
  spk_ir_summary sum{};
  const spk_status st = spk_ir_solve(inner_A, inner_M, &inner_ir, b, z, &sum,
                                     nullptr);
  if (st != SPK_OK && st != SPK_BREAKDOWN)
    throw Error{st, std::string("inner mixed-precision solve: ") + spk_last_error()};
  inner_total += sum.inner_iterations;
  if constexpr (!std::is_same<T, double>::value) {
    const double* zp = z;
    launch_map(n, [=] __device__(int64_t i) { out[i] = (T)zp[i]; });
  }
}

template void spk_precond_s::apply<double>(const double*, double*);
template void spk_precond_s::apply<float>(const float*, float*);
template void spk_precond_s::forward<double>(const double*, double*);
template void spk_precond_s::forward<float>(const float*, float*);
template void spk_precond_s::backward<double>(const double*, double*);
template void spk_precond_s::backward<float>(const float*, float*);

extern "C" {

spk_status spk_precond_create_jacobi(spk_csr A, spk_precond* out) {
  return guarded([&] {
    SPK_REQUIRE(A && out, SPK_INVALID_ARGUMENT, "null argument");
    auto* M = new spk_precond_s();
    try {
      M->kind = spk_precond_s::kJacobi;
      M->n = std::min(A->nrows, A->ncols);
      M->inv_d64.alloc((size_t)M->n);
      DevBuf<int> zero(1);
      hipStream_t s = stream();
      SPK_HIP_TRY(hipMemsetAsync(zero.p, 0, sizeof(int), s));
      if (M->n > 0)
        hipLaunchKernelGGL(invert_diag_kernel, dim3(blocks_for(M->n)),
                           dim3(256), 0, s, A->rp.p, A->ci.p, A->v64.p, M->n,
                           M->inv_d64.p, zero.p);
      int hz = 0;
      SPK_HIP_TRY(hipMemcpyAsync(&hz, zero.p, sizeof(int),
                                 hipMemcpyDeviceToHost, s));
      SPK_HIP_TRY(hipStreamSynchronize(s));
      SPK_REQUIRE(!hz, SPK_INVALID_ARGUMENT, "jacobi: zero diagonal entry");
    } catch (...) {
      delete M;
      throw;
    }
    *out = M;
  });
}

spk_status spk_precond_create_identity(int64_t n, spk_precond* out) {
  return guarded([&] {
    SPK_REQUIRE(out && n >= 0, SPK_INVALID_ARGUMENT, "bad argument");
    auto* M = new spk_precond_s();
    M->kind = spk_precond_s::kIdentity;
    M->n = n;
    *out = M;
  });
}

spk_status spk_ilu0_set_schedule(spk_precond M, int schedule) {
  return guarded([&] {
    SPK_REQUIRE(M && M->kind == spk_precond_s::kIlu, SPK_INVALID_ARGUMENT,
                "not an ILU(0) preconditioner");
    SPK_REQUIRE(schedule >= 0 && schedule <= 2, SPK_INVALID_ARGUMENT,
                "bad schedule");
    SPK_HIP_TRY(hipStreamSynchronize(stream()));
    M->set_schedule(schedule);
    // the per-level schedule leaves ordinary values in the scratch vector;
    // the others need it filled with the ready sentinel
    if (M->sweep != spk_precond_s::kLevels) M->reset_sentinels();
  });
}

spk_status spk_ilu0_set_jacobi_sweeps(spk_precond M, int sweeps) {
  return guarded([&] {
    SPK_REQUIRE(M && M->kind == spk_precond_s::kIlu, SPK_INVALID_ARGUMENT,
                "not an ILU(0) preconditioner");
    SPK_REQUIRE(sweeps >= 0 && sweeps <= 1024, SPK_INVALID_ARGUMENT,
                "sweeps must be in [0, 1024]");
    SPK_HIP_TRY(hipStreamSynchronize(stream()));
    if (sweeps > 0) M->build_strict();
    M->jac_sweeps = sweeps;
  });
}

spk_status spk_ilu0_set_half_factors(spk_precond M, int enable) {
  return guarded([&] {
    SPK_REQUIRE(M && M->kind == spk_precond_s::kIlu, SPK_INVALID_ARGUMENT,
                "not an ILU(0) preconditioner");
    SPK_HIP_TRY(hipStreamSynchronize(stream()));
    M->build_strict();
    for (spk_csr_s* S : {M->Ls, M->Us}) {
      const spk_status st = spk_csr_set_half_values(S, enable);
      if (st != SPK_OK)
        throw Error{st, std::string("ILU(0) strict factors: ") + spk_last_error()};
    }
  });
}

spk_status spk_ilu0_get_half_factors(spk_precond M, int* enabled) {
  return guarded([&] {
    SPK_REQUIRE(M && enabled && M->kind == spk_precond_s::kIlu,
                SPK_INVALID_ARGUMENT, "not an ILU(0) preconditioner");
    *enabled = M->Ls && M->Ls->half32 ? 1 : 0;
  });
}

spk_status spk_ilu0_get_jacobi_sweeps(spk_precond M, int* sweeps) {
  return guarded([&] {
    SPK_REQUIRE(M && sweeps && M->kind == spk_precond_s::kIlu,
                SPK_INVALID_ARGUMENT, "not an ILU(0) preconditioner");
    *sweeps = M->jac_sweeps;
  });
}

spk_status spk_ilu0_get_schedule(spk_precond M, int* schedule) {
  return guarded([&] {
    SPK_REQUIRE(M && schedule && M->kind == spk_precond_s::kIlu,
                SPK_INVALID_ARGUMENT, "not an ILU(0) preconditioner");
    *schedule = M->sweep == spk_precond_s::kLevels ? SPK_ILU_LEVELS : SPK_ILU_SYNC_FREE;
  });
}

spk_status spk_precond_create_spmv(spk_csr Mst, spk_precond* out) {
  return guarded([&] {
    SPK_REQUIRE(Mst && out, SPK_INVALID_ARGUMENT, "null argument");
    SPK_REQUIRE(Mst->nrows == Mst->ncols, SPK_INVALID_ARGUMENT,
                "approximate inverse must be square");
    auto* M = new spk_precond_s();
    M->kind = spk_precond_s::kSpmv;
    M->n = Mst->nrows;
    M->M = Mst;
    *out = M;
  });
}

spk_status spk_precond_create_inner_cg(spk_csr A, spk_precond M_inner,
                                       int64_t iterations, double tolerance,
                                       int precision, spk_precond* out) {
  return guarded([&] {
    SPK_REQUIRE(A && out, SPK_INVALID_ARGUMENT, "null argument");
    SPK_REQUIRE(A->nrows == A->ncols, SPK_INVALID_ARGUMENT,
                "inner PCG requires a square matrix");
    SPK_REQUIRE(!M_inner || M_inner->n == A->nrows, SPK_INVALID_ARGUMENT,
                "inner preconditioner size mismatch");
    SPK_REQUIRE(!M_inner || !M_inner->runs_solve(), SPK_INVALID_ARGUMENT,
                "inner PCG cannot nest another inner solve");
    SPK_REQUIRE(iterations >= 1 && tolerance >= 0.0, SPK_INVALID_ARGUMENT,
                "iterations >= 1, tolerance >= 0");
    SPK_REQUIRE(precision == SPK_F32 || precision == SPK_F64,
                SPK_INVALID_ARGUMENT, "precision must be SPK_F32 or SPK_F64");
    auto* P = new spk_precond_s();
    P->kind = spk_precond_s::kInnerCg;
    P->n = A->nrows;
    P->inner_A = A;
    P->inner_M = M_inner;
    P->inner_iters = iterations;
    P->inner_tol = tolerance;
    P->inner_precision = precision;
    *out = P;
  });
}

spk_status spk_precond_create_inner_ir(spk_csr A, spk_precond M_inner,
                                       const spk_ir_config* cfg,
                                       spk_precond* out) {
  return guarded([&] {
    SPK_REQUIRE(A && cfg && out, SPK_INVALID_ARGUMENT, "null argument");
    SPK_REQUIRE(A->nrows == A->ncols, SPK_INVALID_ARGUMENT,
                "inner solve requires a square matrix");
    SPK_REQUIRE(!M_inner || M_inner->n == A->nrows, SPK_INVALID_ARGUMENT,
                "inner preconditioner size mismatch");
    SPK_REQUIRE(!M_inner || !M_inner->runs_solve(), SPK_INVALID_ARGUMENT,
                "an inner solve cannot nest another inner solve");
    // the (F)GMRES this preconditioner serves keeps its basis in the GMRES
    // work vectors, which an inner (F)GMRES would reuse
    SPK_REQUIRE(cfg->inner_method == SPK_IR_CG ||
                    cfg->inner_method == SPK_IR_CG_RELIABLE ||
                    cfg->inner_method == SPK_IR_BICGSTAB,
                SPK_INVALID_ARGUMENT,
                "inner solve: inner_method must be SPK_IR_CG, "
                "SPK_IR_CG_RELIABLE or SPK_IR_BICGSTAB");
    SPK_REQUIRE(cfg->tolerance > 0.0 && cfg->max_outer >= 1 && cfg->max_inner >= 1,
                SPK_INVALID_ARGUMENT,
                "inner solve: tolerance > 0, max_outer >= 1, max_inner >= 1");
    auto* P = new spk_precond_s();
    P->kind = spk_precond_s::kInnerIr;
    P->n = A->nrows;
    P->inner_A = A;
    P->inner_M = M_inner;
    P->inner_ir = *cfg;
    *out = P;
  });
}

spk_status spk_precond_inner_cg_iterations(spk_precond M, int64_t* total) {
  return guarded([&] {
    SPK_REQUIRE(M && total && M->runs_solve(), SPK_INVALID_ARGUMENT,
                "not an inner-solve preconditioner");
    *total = M->inner_total;
  });
}

spk_status spk_precond_create_ilu0(spk_csr A, int modified, spk_precond* out) {
  return guarded([&] {
    TraceRange trace_("spk_precond_create_ilu0");
    SPK_REQUIRE(A && out, SPK_INVALID_ARGUMENT, "null argument");
    SPK_REQUIRE(A->nrows == A->ncols, SPK_INVALID_ARGUMENT,
                "ilu0 requires a square matrix");
    auto* M = new spk_precond_s();
    try {
      M->kind = spk_precond_s::kIlu;
      M->factor(*A, modified != 0);
    } catch (...) {
      delete M;
      throw;
    }
    *out = M;
  });
}

spk_status spk_precond_destroy(spk_precond M) {
  return guarded([&] {
    if (!M) return;
    SPK_HIP_TRY(hipStreamSynchronize(stream()));
    delete M;
  });
}

spk_status spk_precond_apply(spk_precond M, int dtype, const void* d_in,
                             void* d_out) {
  return guarded([&] {
    TraceRange trace_("spk_precond_apply");
    SPK_REQUIRE(M && d_in && d_out, SPK_INVALID_ARGUMENT, "null argument");
    if (dtype == SPK_F32) M->apply((const float*)d_in, (float*)d_out);
    else M->apply((const double*)d_in, (double*)d_out);
    M->check_sweeps();
  });
}

spk_status spk_ilu0_factor_nnz(spk_precond M, int64_t* nnz_l, int64_t* nnz_u) {
  return guarded([&] {
    SPK_REQUIRE(M && M->kind == spk_precond_s::kIlu, SPK_INVALID_ARGUMENT,
                "not an ILU preconditioner");
    if (nnz_l) *nnz_l = M->nnz_l;
    if (nnz_u) *nnz_u = M->nnz_u;
  });
}

spk_status spk_ilu0_download(spk_precond M, int64_t* l_row_ptr,
                             int64_t* l_col_ind, double* l_vals,
                             int64_t* u_row_ptr, int64_t* u_col_ind,
                             double* u_vals) {
  spk_status st = SPK_OK;
  if (!M || M->kind != spk_precond_s::kIlu) {
    set_error("not an ILU preconditioner");
    return SPK_INVALID_ARGUMENT;
  }
  st = guarded([&] { M->build_factors(); });
  if (st) return st;
  st = spk_csr_download(M->L, l_row_ptr, l_col_ind, l_vals);
  if (st) return st;
  return spk_csr_download(M->U, u_row_ptr, u_col_ind, u_vals);
}

spk_status spk_ilu0_levels(spk_precond M, int64_t* levels_l,
                           int64_t* levels_u) {
  return guarded([&] {
    SPK_REQUIRE(M && M->kind == spk_precond_s::kIlu, SPK_INVALID_ARGUMENT,
                "not an ILU preconditioner");
    if (levels_l) *levels_l = M->levels_l;
    if (levels_u) *levels_u = M->levels_u;
  });
}

// The sync-free sweeps mark x with a sentinel before they read b, so an
// input that overlaps the output would be overwritten first.
static bool vectors_overlap(const void* b, const void* x, int64_t n, int dtype) {
  const size_t bytes = (size_t)(n > 0 ? n : 0) * (dtype == SPK_F32 ? 4 : 8);
  const uintptr_t pb = (uintptr_t)b, px = (uintptr_t)x;
  return pb == px || (pb < px + bytes && px < pb + bytes);
}

spk_status spk_ilu0_forward(spk_precond M, int dtype, const void* d_b,
                            void* d_x) {
  return guarded([&] {
    SPK_REQUIRE(M && M->kind == spk_precond_s::kIlu && d_b && d_x,
                SPK_INVALID_ARGUMENT, "bad argument");
    SPK_REQUIRE(dtype == SPK_F32 || dtype == SPK_F64, SPK_INVALID_ARGUMENT,
                "dtype must be SPK_F32 or SPK_F64");
    SPK_REQUIRE(!vectors_overlap(d_b, d_x, M->n, dtype), SPK_INVALID_ARGUMENT,
                "ilu0 triangular sweep: b and x must not overlap");
    if (dtype == SPK_F32) M->forward((const float*)d_b, (float*)d_x);
    else M->forward((const double*)d_b, (double*)d_x);
    M->check_sweeps();
  });
}

spk_status spk_ilu0_backward(spk_precond M, int dtype, const void* d_b,
                             void* d_x) {
  return guarded([&] {
    SPK_REQUIRE(M && M->kind == spk_precond_s::kIlu && d_b && d_x,
                SPK_INVALID_ARGUMENT, "bad argument");
    SPK_REQUIRE(dtype == SPK_F32 || dtype == SPK_F64, SPK_INVALID_ARGUMENT,
                "dtype must be SPK_F32 or SPK_F64");
    SPK_REQUIRE(!vectors_overlap(d_b, d_x, M->n, dtype), SPK_INVALID_ARGUMENT,
                "ilu0 triangular sweep: b and x must not overlap");
    if (dtype == SPK_F32) M->backward((const float*)d_b, (float*)d_x);
    else M->backward((const double*)d_b, (double*)d_x);
    M->check_sweeps();
  });
}

}  // extern "C"
