// spk_cgstep.hpp -- many steps of diagonally preconditioned CG in one launch,
// for matrices whose entries fit the registers of the chip.
//
// Three kernels a step cost three kernel boundaries, about 13 us however
// small the matrix.  Here every thread keeps R rows for the whole launch:
// their x, r and p, their entries' values, and a copy of p for every entry.
// A step is
//   q = A p from the registers;              exchange <p, q>
//   x += a p; r -= a q; z = D^-1 r to memory; exchange |r|^2, <r, z>
//   p = z + b p, for the row and for every entry's copy, whose z is loaded.
// The copies are computed from the same z and b by the same operation as the
// row's own p, so they are the same bits, and p itself is never exchanged.
// z needs no second buffer: a block stores the next one only after the next
// <p, q> exchange, which every block enters after its loads.
// The row sums run in storage order with the products rounded separately, as
// the SpMV's; only the dot products' summation order differs from the
// kernels this replaces.
// Bound: two exchanges (1.9 us each), the wait for z's stores and z's loads.
// FP64 Jacobi-PCG, a step by three kernels -> this: 1,024 rows 5-point 17.0 ->
// 3.2 us, 65,536 rows 16.6 -> 6.9, 455,000 rows 25.2 -> 9.0; 262,144 rows
// 7-point 21.5 -> 9.2; 302,500 rows 9-point 24.7 -> 10.5, FP32 19.9 -> 8.0.
#pragma once

#include "spk_csr.hpp"
#include "spk_link.hpp"

namespace spk {

// 448 threads with rows and the link's wavefront: two wavefronts a SIMD, 256
// registers each.
constexpr int kCgBlock = 448;

__device__ __forceinline__ double fma_t(double a, double b, double c) {
  return __builtin_fma(a, b, c);
}
__device__ __forceinline__ float fma_t(float a, float b, float c) {
  return __builtin_fmaf(a, b, c);
}

// What a thread's entries take of its registers: value, p and z's address.
template <typename T>
constexpr int cg_entry_regs = 2 * (int)(sizeof(T) / 4) + 1;

// Rows per thread: the fewest that leave at most `blocks` blocks; 0: the rows'
// entries do not fit (four rows of nine FP64 entries would need 180 registers
// for the entries alone).  K: entries a row holds (padded).
template <typename T>
inline int cg_rows_per_thread(int64_t n, int K, int blocks) {
  const int64_t r = (n + (int64_t)blocks * kCgBlock - 1) / ((int64_t)blocks * kCgBlock);
  const int limit = K * cg_entry_regs<T> * 4 <= 160 ? 4 : 3;
  return r <= limit ? (int)r : 0;
}
inline int cg_row_entries(const spk_csr_s& A) {
  return A.max_len <= 5 ? 5 : A.max_len <= 7 ? 7 : A.max_len <= 9 ? 9 : 0;
}
// One block, whose exchanges stay in LDS, holds the rows.
template <typename T>
bool cg_one_block(const spk_csr_s& A) {
  const int limit = cg_row_entries(A) * cg_entry_regs<T> * 4 <= 160 ? 4 : 3;
  return A.nrows <= (int64_t)kCgBlock * limit;
}
// the plain layout with short rows, few enough of them
template <typename T>
bool cg_steps_fit(const spk_csr_s& A, const GridLink& link) {
  const int K = cg_row_entries(A);
  return K > 0 && A.nrows == A.ncols && A.panels.empty() && A.xt_groups == 0 &&
         !(std::is_same<T, float>::value && A.half32) &&
         cg_rows_per_thread<T>(A.nrows, K, link.blocks) > 0;
}

// Ctl::skip(): the launch is a no-op.  Ctl::rz(): <r, z> at the start.
// Ctl::ends(rr): whether the step with |r|^2 = rr is the last of the solve
// (p is then left as it is).  Ctl::record(step, rr) after every step and
// Ctl::finish(steps, rr, rz before the last step, rz after it, ended) run in
// one thread of block 0 and touch only what no block reads again.
// Ctl::expire(): an exchange did not go through; x, r and p are then parts of
// several steps' and the launch, with those queued after it, is to be undone.
template <typename T, int K, int R, typename Ctl>
__global__ __launch_bounds__(kCgBlock + 64) void cg_steps_kernel(
    unsigned n, const int32_t* __restrict__ rp, const int32_t* __restrict__ ci,
    const T* __restrict__ v, const T* __restrict__ invd, T* __restrict__ x,
    T* __restrict__ r, T* __restrict__ p, T* __restrict__ z, int steps, Ctl ctl,
    GridLink link) {
  __shared__ double red[link_lds(kCgBlock)];
  if (ctl.skip()) return;  // set only after every block has been here
  const int stale = link_open<kCgBlock>(link);
  unsigned tag = *link.tag;
  double rz = ctl.rz();
  const unsigned i0 =
      threadIdx.x < kCgBlock ? blockIdx.x * (kCgBlock * R) + threadIdx.x : n;
  T xv[R], rv[R], pv[R], dv[R], val[R][K], pe[R][K];
  unsigned at[R][K];
#pragma unroll
  for (int u = 0; u < R; ++u) {
    const unsigned i = i0 + u * kCgBlock;
    xv[u] = rv[u] = pv[u] = T(0);
    dv[u] = T(1);
    // absent entries: value 0, at the row itself (no row: row 0)
#pragma unroll
    for (int k = 0; k < K; ++k) {
      val[u][k] = pe[u][k] = T(0);
      at[u][k] = i < n ? i : 0;
    }
    if (i < n) {
      xv[u] = x[i];
      rv[u] = r[i];
      pv[u] = p[i];
      if (invd) dv[u] = invd[i];
      const int b = rp[i], len = rp[i + 1] - b;
#pragma unroll
      for (int k = 0; k < K; ++k)
        if (k < len) {
          at[u][k] = (unsigned)ci[b + k];
          val[u][k] = v[b + k];
        }
#pragma unroll
      for (int k = 0; k < K; ++k) pe[u][k] = p[at[u][k]];
    }
  }
  double rr = 0.0, rz0 = rz;
  bool ended = false;
  int done = 0;
  while (done < steps && !ended) {
    T q[R];
    double s1[1] = {0.0};
#pragma unroll
    for (int u = 0; u < R; ++u) {
#pragma clang fp contract(off)
      T s = T(0);
#pragma unroll
      for (int k = 0; k < K; ++k) s += val[u][k] * pe[u][k];
      q[u] = s;
      s1[0] += (double)pv[u] * (double)s;
    }
    if (!link_sum<1, kCgBlock>(link, stale, ++tag, s1, red)) break;
    const T a = (T)(rz / s1[0]);
    double s2[2] = {0.0, 0.0};
    T zv[R];
#pragma unroll
    for (int u = 0; u < R; ++u) {
      const unsigned i = i0 + u * kCgBlock;
      xv[u] = a * pv[u] + xv[u];
      rv[u] = rv[u] - a * q[u];
      zv[u] = invd ? dv[u] * rv[u] : rv[u];
      if (i < n)
        __hip_atomic_store(z + i, zv[u], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      s2[0] += (double)rv[u] * (double)rv[u];
      s2[1] += (double)rv[u] * (double)zv[u];
    }
    // z has reached memory before this block's sums say so
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (!link_sum<2, kCgBlock>(link, stale, ++tag, s2, red)) break;
    rr = s2[0];
    rz0 = rz;
    ended = ctl.ends(rr);
    if (blockIdx.x == 0 && threadIdx.x == 0) ctl.record(done, rr);
    ++done;
    if (!ended) {
      const T b = (T)(s2[1] / rz);
      rz = s2[1];
      T ze[R][K];
#pragma unroll
      for (int u = 0; u < R; ++u)
#pragma unroll
        for (int k = 0; k < K; ++k)
          ze[u][k] = __hip_atomic_load(z + at[u][k], __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
      for (int u = 0; u < R; ++u) {
        pv[u] = fma_t(b, pv[u], zv[u]);
#pragma unroll
        for (int k = 0; k < K; ++k) pe[u][k] = fma_t(b, pe[u][k], ze[u][k]);
      }
    }
  }
  if (done < steps && !ended) {  // an exchange did not go through
    if (threadIdx.x == 0) ctl.expire();
    return;
  }
#pragma unroll
  for (int u = 0; u < R; ++u) {
    const unsigned i = i0 + u * kCgBlock;
    if (i < n) {
      x[i] = xv[u];
      r[i] = rv[u];
      p[i] = pv[u];
    }
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    link_close(link, tag);
    ctl.finish(done, rr, rz0, rz, ended);
  }
}

// up to `steps` steps; x, r, p in and out, z scratch
template <typename T, typename Ctl>
void launch_cg_steps(spk_csr_s& A, const T* invd, T* x, T* r, T* p, T* z, int steps,
                     const Ctl& ctl, const GridLink& link) {
  const int K = cg_row_entries(A);
  const int rows = cg_one_block<T>(A) ? (int)((A.nrows + kCgBlock - 1) / kCgBlock)
                                      : cg_rows_per_thread<T>(A.nrows, K, link.blocks);
  const CsrView<T> m = A.view<T>();
  auto run = [&](auto kk, auto rr) {
    constexpr int KK = decltype(kk)::value, RR = decltype(rr)::value;
    const int g = (int)((A.nrows + kCgBlock * RR - 1) / (kCgBlock * RR));
    hipLaunchKernelGGL((cg_steps_kernel<T, KK, RR, Ctl>), dim3(g), dim3(kCgBlock + 64), 0,
                       stream(), (unsigned)A.nrows, m.rp, m.ci, m.v, invd, x, r, p, z,
                       steps, ctl, link);
    SPK_HIP_TRY(hipGetLastError());
  };
  auto pick = [&](auto kk) {
    constexpr int KK = decltype(kk)::value;
    if (rows == 1) run(kk, std::integral_constant<int, 1>{});
    else if (rows == 2) run(kk, std::integral_constant<int, 2>{});
    else if (rows == 3) run(kk, std::integral_constant<int, 3>{});
    else if constexpr (KK * cg_entry_regs<T> * 4 <= 160)
      run(kk, std::integral_constant<int, 4>{});
  };
  if (K == 5) pick(std::integral_constant<int, 5>{});
  else if (K == 7) pick(std::integral_constant<int, 7>{});
  else pick(std::integral_constant<int, 9>{});
}

}  // namespace spk
