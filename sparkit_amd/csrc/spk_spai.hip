// spk_spai.hip -- learned sparse approximate inverse: a small MLP predicts
// the rows of M on A's sparsity pattern from per-row features; M is then
// applied as one SpMV (a spk_precond of kind "spmv").  The network is trained
// on the device with hand-written BF16 MFMA forward/backward kernels and an
// Adam update, minimising (1/n) ||I - M A||_F^2.
//
// Row slots.  Row i must hold its diagonal, a_ii > 0, and at most 4 entries
// on each side of it.  Slot 4 is the diagonal; the entries left of it, from
// the nearest outwards, take slots 3, 2, 1, 0; those right of it 5..8 (for
// an interior row of a 9-point stencil: SW S SE W C E NW N NE).
// Features (24, computed in double, stored as float) for the off-diagonal
// slots k = 0..7 (slots 0 1 2 3 5 6 7 8) with column j, zero when empty:
//   x[k] = a_ij / a_ii,  x[8+k] = (a_jj - a_ii) / (a_jj + a_ii),
//   x[16+k] = rowsum_j / a_jj   (rowsum in storage order).
// Network: y = W3^T relu(W2^T relu(W1^T x + b1) + b2) + b3, 24 -> 64 -> 64
// -> 9; GEMM operands (features, weights, activations, backward deltas) are
// bfloat16 (round to nearest even), accumulation and bias/elementwise work
// fp32.  M_i,slot = (delta_{slot,4} + y_slot) / a_ii: zero output weights
// give the Jacobi preconditioner.
//
// Kernel layout.  The matrices of a batch go through each pass together, up
// to kGroupMats matrices or kGroupRows rows at a time (a larger matrix goes
// alone):
//   prepare   a row per thread: diagonal and row sum
//   features  a row per thread: the row's 24 features in bfloat16
//   forward   a wavefront per 64 rows: Y = H2 W3 + b3, H2 = relu(H1 W2 + b2),
//             H1 = relu(X W1 + b1)
//   rows      a row per thread: m from Y, (M A)_i by a merge of the slot
//             rows, the row's loss and dL/dy
//   backward  one workgroup of 4 wavefronts a compute unit, 64 rows per
//             wavefront at a time: H1 and H2 again, then dW3 += H2^T dY;
//             dH2 = dY W3^T * [H2 > 0]; dW2 += H1^T dH2;
//             dH1 = dH2 W2^T * [H1 > 0]; dW1 += X^T dH1
// The per-row passes wait for dependent loads and run at the occupancy their
// registers allow; only the two passes of products need LDS.  Every product
// is a sequence of v_mfma_f32_16x16x32_bf16 on 16x16 output tiles.  The
// weights' fragments stay in registers; an activation or delta is kept in
// LDS by rows where its columns are summed over and by columns where its
// rows are, so that every fragment is one 16-byte read (rows of 72 elements:
// no bank conflicts).  Weight gradients stay in the MFMA accumulators across
// a wavefront's tiles of a matrix, are summed over the workgroup's
// wavefronts in LDS in a fixed order and added to one partial per workgroup;
// the update kernel sums the partials in workgroup order (deterministic) and
// applies Adam to the fp32 master weights, then refreshes the bf16 copy.
//
// Measured on a batch of 4 matrices of 65,536 9-point rows: prepare 20 us,
// features 13, forward 14, rows 57 (issue bound: about 25 columns a row, nine
// lists compared for each), backward 57 (one wavefront per SIMD, bound by
// what its LDS holds; 14 us a matrix, 5 of them the workgroup's sums), update
// 8.  One fused kernel for all of it, a matrix at a time, took 105 us a
// matrix and the update 74 us: its per-row parts ran at one wavefront per
// SIMD, and its fragments were read from LDS two bytes at a time.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <utility>
#include <vector>

#include "spk_csr.hpp"
#include "spk_vec.hpp"

namespace spk {
namespace {

typedef __bf16 bf16;
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int kF = 24, kH = 64, kO = 9;
// canonical parameter layout: W1[24][64] b1 W2[64][64] b2 W3[64][9] b3
constexpr int kW1 = 0, kB1 = kW1 + kF * kH, kW2 = kB1 + kH, kB2 = kW2 + kH * kH,
              kW3 = kB2 + kH, kB3 = kW3 + kH * kO, kNP = kB3 + kO;
static_assert(kNP == SPK_SPAI_NPARAM, "parameter count");
// padded device shapes
constexpr int kFp = 32;  // X columns / W1 rows
constexpr int kOk = 32;  // dY columns / W3 columns (K of dY W3^T)
constexpr int kOn = 16;  // Y columns (one output tile)
// gradient partial layout (floats)
constexpr int gW1 = 0, gW2 = gW1 + kFp * kH, gW3 = gW2 + kH * kH,
              gB1 = gW3 + kH * kOn, gB2 = gB1 + kH, gB3 = gB2 + kH,
              kGradLen = gB3 + kOn;
constexpr int kTile = 64;   // rows per wavefront tile
constexpr int kWaves = 4;   // wavefronts per workgroup
// LDS row length, in bf16 elements, of 64-wide operands and of dY by rows
constexpr int kLd = 72, kLdY = 24;
// what a training launch takes together, at most (or one larger matrix)
constexpr int kGroupMats = 16;
constexpr int64_t kGroupRows = 1 << 20;
constexpr int kRowBlock = 256;

// bf16 weights, those a product reads by columns in a transposed copy, and
// fp32 biases
struct Packed {
  bf16 w1t[kH * kFp];  // [hidden][feature]
  bf16 w2[kH * kH];
  bf16 w2t[kH * kH];
  bf16 w3[kH * kOk];
  bf16 w3t[kOn * kH];
  float b1[kH], b2[kH], b3[kOn];
};

// round to nearest even: v_cvt_pk_bf16_f32
__device__ __forceinline__ bf16 to_bf16(float x) { return (bf16)x; }
// of a value that relu gave (not negative, but -0 may be)
__device__ __forceinline__ bool positive(bf16 h) {
  return (__builtin_bit_cast(uint16_t, h) & 0x7FFF) != 0;
}

// C += A[16 x 32] B[32 x 16].  Lane l's fragment is row (of A) or column (of
// B) l % 16, the eight k from 8 (l / 16) on; acc[i] is C(4 (l / 16) + i, l % 16).
__device__ __forceinline__ floatx4 mma(bf16x8 a, bf16x8 b, floatx4 acc) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc, 0, 0, 0);
}
__device__ __forceinline__ bf16x8 frag(const bf16* p) {  // 16-byte aligned
  return *(const bf16x8*)p;
}
// LDS traffic between the lanes of a wavefront, which is in order
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ floatx4 splat(float v) { return floatx4{v, v, v, v}; }

// Rows [first, last) of a matrix of n rows: row i's diagonal and row sum are
// at dbase + i, its features and outputs at xbase + i - first.  xbase is a
// multiple of kRowBlock.
struct RowSpan {
  const int32_t* __restrict__ rp;
  const int32_t* __restrict__ ci;
  const double* __restrict__ v;
  int64_t n, first, last, dbase, xbase;
};

struct Group {
  RowSpan mat[kGroupMats];
  int count;
  double* __restrict__ diag;
  double* __restrict__ rsum;
  bf16* __restrict__ x;            // [rows][kFp]
  float* __restrict__ y;           // [rows][kO]: outputs, then dL/dy
  // train: the matrices' entries by scratch row, see EntryRows
  int32_t* __restrict__ ecol;
  double* __restrict__ eval;
  double* __restrict__ rowloss;    // [rows]
  const Packed* __restrict__ pk;
  double* __restrict__ mvals;      // predict: M values on A's pattern
  double scale;                    // train: 1 / rows of the batch
  // train, symmetric objective (one matrix): dL/dm per entry of A's pattern
  // and each row's loss, computed beforehand
  const double* __restrict__ gm;
  const double* __restrict__ rl;
};

// the span that scratch row x (of a whole workgroup) lies in
__device__ __forceinline__ int span_of(const Group& G, int64_t x) {
  int k = 0;
  while (k + 1 < G.count && x >= G.mat[k + 1].xbase) ++k;
  return k;
}

// A row's entries, kEntries places 64 rows at a time: place k of scratch row x
// at entry_at(x) + 64 k, the columns ascending and INT32_MAX behind them, so
// that lanes on neighbouring rows read neighbouring words (from the CSR rows
// the merge of the slot rows took three times as long: a lane's rows lie 36
// and 72 bytes from the next lane's).
constexpr int kEntries = kO + 1;
__device__ __forceinline__ int64_t entry_at(int64_t x) {
  return (x >> 6) * (64 * kEntries) + (x & 63);
}

// diagonal, row sums; with err the slot-rule check; the entries if G has
// room for them
__global__ void spai_prepare_kernel(Group G, int* err) {
  const int64_t x = blockIdx.x * (int64_t)blockDim.x;
  const RowSpan& A = G.mat[span_of(G, x)];
  const int64_t i = x + threadIdx.x - A.xbase;
  if (i >= A.n) return;
  const int p0 = A.rp[i], p1 = A.rp[i + 1];
  int dpos = -1;
  double s = 0.0;
  for (int p = p0; p < p1; ++p) {
    if (A.ci[p] == i) dpos = p;
    s += A.v[p];
  }
  const bool bad = dpos < 0 || !(A.v[dpos] > 0.0) || dpos - p0 > 4 ||
                   p1 - dpos - 1 > 4;
  if (bad && err) atomicOr(err, 1);
  G.diag[A.dbase + i] = bad ? 1.0 : A.v[dpos];
  G.rsum[A.dbase + i] = s;
  if (!G.ecol) return;
  const int64_t o = entry_at(A.xbase + i);
  int c[kO];
  double v[kO];
#pragma unroll
  for (int k = 0; k < kO; ++k) {
    const bool in = p0 + k < p1;
    c[k] = in ? A.ci[p0 + k] : INT32_MAX;
    v[k] = in ? A.v[p0 + k] : 0.0;
  }
#pragma unroll
  for (int k = 0; k < kO; ++k) {
    G.ecol[o + 64 * k] = c[k];
    G.eval[o + 64 * k] = v[k];
  }
  G.ecol[o + 64 * kO] = INT32_MAX;
  G.eval[o + 64 * kO] = 0.0;
}

// Two forms of a matrix's rows.  slots(): the places of row i's slots (and
// their columns, INT32_MAX for none), pos[4] its diagonal, pos[3..0] the entries left of it from the nearest outwards,
// pos[5..8] those right of it (-1 unused).  cursor(j): where row j's first
// entry is (col() and val() there, INT32_MAX behind the last; none(i): behind
// the last), step() to the next.
struct CsrRows {
  const int32_t* __restrict__ rp;
  const int32_t* __restrict__ ci;
  const double* __restrict__ v;
  struct Cursor {
    int p, e;
  };
  __device__ __forceinline__ void slots(int64_t i, int* pos, int* j) const {
    const int p0 = rp[i], p1 = rp[i + 1];
    int d = p0;
    while (ci[d] != (int32_t)i) ++d;  // present: checked by the prepare pass
    pos[4] = d;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      pos[3 - k] = (d - 1 - k >= p0) ? d - 1 - k : -1;
      pos[5 + k] = (d + 1 + k < p1) ? d + 1 + k : -1;
    }
#pragma unroll
    for (int s = 0; s < kO; ++s) j[s] = pos[s] >= 0 ? ci[pos[s]] : INT32_MAX;
  }
  __device__ __forceinline__ double val_at(int64_t, int p) const { return v[p]; }
  __device__ __forceinline__ Cursor cursor(int64_t j) const {
    return Cursor{rp[j], rp[j + 1]};
  }
  __device__ __forceinline__ Cursor none(int64_t) const { return Cursor{0, 0}; }
  __device__ __forceinline__ void step(Cursor& c) const { ++c.p; }
  __device__ __forceinline__ int col(const Cursor& c) const {
    return c.p < c.e ? ci[c.p] : INT32_MAX;
  }
  __device__ __forceinline__ double val(const Cursor& c) const {
    return c.p < c.e ? v[c.p] : 0.0;
  }
};
struct EntryRows {
  const int32_t* __restrict__ c;
  const double* __restrict__ v;
  int64_t base;  // scratch row of row 0
  using Cursor = int64_t;
  __device__ __forceinline__ void slots(int64_t i, int* pos, int* j) const {
    const int32_t* row = c + entry_at(base + i);
    int d = 0, own[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) own[k] = row[64 * k];
#pragma unroll
    for (int k = 4; k >= 0; --k) d = own[k] == (int32_t)i ? k : d;  // the first
#pragma unroll
    for (int s = 0; s < kO; ++s) {
      const int k = s - 4 + d;  // at most 8
      j[s] = row[64 * (k < 0 ? kO : k)];
      pos[s] = j[s] != INT32_MAX ? k : -1;
    }
  }
  __device__ __forceinline__ double val_at(int64_t i, int p) const {
    return v[entry_at(base + i) + 64 * p];
  }
  __device__ __forceinline__ Cursor cursor(int64_t j) const { return entry_at(base + j); }
  __device__ __forceinline__ Cursor none(int64_t i) const {
    return entry_at(base + i) + 64 * kO;  // the word behind row i
  }
  __device__ __forceinline__ void step(Cursor& q) const { q += 64; }
  __device__ __forceinline__ int col(const Cursor& q) const { return c[q]; }
  __device__ __forceinline__ double val(const Cursor& q) const { return v[q]; }
};

// Row i's residual e_i - sum_s m_s A_{j_s,:} by a merge of the slot rows
// (their columns ascend): returns ||.||^2 and adds dL/dm_s to gs[s].
template <typename Rows>
__device__ __forceinline__ double row_residual(const Rows& A, int64_t i, const int* j,
                                               const double* m, double* gs) {
#pragma clang fp contract(off)
  typename Rows::Cursor hp[kO];
  int hc[kO];
  double hv[kO];
#pragma unroll
  for (int s = 0; s < kO; ++s)
    hp[s] = j[s] != INT32_MAX ? A.cursor(j[s]) : A.none(i);
#pragma unroll
  for (int s = 0; s < kO; ++s) {
    hc[s] = A.col(hp[s]);
    hv[s] = A.val(hp[s]);
  }
  double lrow = 0.0;
  for (;;) {
    int c = INT32_MAX;
#pragma unroll
    for (int s = 0; s < kO; ++s) c = hc[s] < c ? hc[s] : c;
    if (c == INT32_MAX) break;
    double tsum = 0.0;
#pragma unroll
    for (int s = 0; s < kO; ++s)
      if (hc[s] == c) tsum += m[s] * hv[s];
    const double res = ((int64_t)c == i ? 1.0 : 0.0) - tsum;
    lrow += res * res;
#pragma unroll
    for (int s = 0; s < kO; ++s)
      if (hc[s] == c) {
        gs[s] += -2.0 * res * hv[s];
        // hv is read before its load goes out: the load then writes its
        // register, and the wait for it comes once, before the next column
        __builtin_amdgcn_sched_barrier(0);
        A.step(hp[s]);
        hc[s] = A.col(hp[s]);
        hv[s] = A.val(hp[s]);
      }
  }
  return lrow;
}

// row i's features
template <typename Rows>
__device__ __forceinline__ void row_features(const Rows& A,
                                             const double* __restrict__ diag,
                                             const double* __restrict__ rsum,
                                             int64_t i, float* x) {
#pragma clang fp contract(off)
  int pos[kO], js[kO];
  A.slots(i, pos, js);
  const double di = diag[i];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const int p = pos[k < 4 ? k : k + 1], j = js[k < 4 ? k : k + 1];
    x[k] = x[8 + k] = x[16 + k] = 0.f;
    if (p >= 0) {
      const double dj = diag[j];
      x[k] = (float)(A.val_at(i, p) / di);
      x[8 + k] = (float)((dj - di) / (dj + di));
      x[16 + k] = (float)(rsum[j] / dj);
    }
  }
}

// Features of every scratch row (zero past a span's end).
__global__ __launch_bounds__(kRowBlock) void spai_features_kernel(Group G) {
  const int64_t xb = blockIdx.x * (int64_t)kRowBlock;
  const RowSpan& A = G.mat[span_of(G, xb)];
  const int64_t xr = xb + threadIdx.x, i = xr - A.xbase + A.first;
  float x[kFp];
#pragma unroll
  for (int f = 0; f < kFp; ++f) x[f] = 0.f;
  const double* diag = G.diag + A.dbase;
  const double* rsum = G.rsum + A.dbase;
  if (i < A.last) {
    if (G.ecol) row_features(EntryRows{G.ecol, G.eval, A.xbase}, diag, rsum, i, x);
    else row_features(CsrRows{A.rp, A.ci, A.v}, diag, rsum, i, x);
  }
  bf16x8* out = (bf16x8*)(G.x + xr * kFp);
#pragma unroll
  for (int q = 0; q < kFp / 8; ++q) {
    bf16x8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = to_bf16(x[8 * q + j]);
    out[q] = o;
  }
}

// Y of every scratch row, a tile per wavefront.
__global__ __launch_bounds__(kWaves * 64) void spai_forward_kernel(Group G) {
#pragma clang fp contract(off)
  __shared__ __attribute__((aligned(16))) bf16 pool[kWaves * kTile * kLd];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const Packed& w = *G.pk;
  bf16* H = pool + wave * kTile * kLd;  // H1, then H2, by rows
  const int64_t row = (blockIdx.x * (int64_t)kWaves + wave) * kTile;
  bf16x8 xf[4], wf[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    xf[q] = frag(G.x + (row + q * 16 + r) * kFp + 8 * g);
    wf[q] = frag(w.w1t + (q * 16 + r) * kFp + 8 * g);
  }
#pragma unroll
  for (int mt = 0; mt < 4; ++mt)
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
      const floatx4 acc = mma(xf[mt], wf[nt], splat(w.b1[nt * 16 + r]));
#pragma unroll
      for (int e = 0; e < 4; ++e)
        H[(mt * 16 + 4 * g + e) * kLd + nt * 16 + r] = to_bf16(fmaxf(acc[e], 0.f));
    }
  wave_sync();
  bf16x8 hf[4][2], w2[4][2];
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      hf[q][kb] = frag(H + (q * 16 + r) * kLd + kb * 32 + 8 * g);
      w2[q][kb] = frag(w.w2t + (q * 16 + r) * kH + kb * 32 + 8 * g);
    }
  wave_sync();
#pragma unroll
  for (int mt = 0; mt < 4; ++mt)
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
      floatx4 acc = splat(w.b2[nt * 16 + r]);
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) acc = mma(hf[mt][kb], w2[nt][kb], acc);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        H[(mt * 16 + 4 * g + e) * kLd + nt * 16 + r] = to_bf16(fmaxf(acc[e], 0.f));
    }
  wave_sync();
  bf16x8 w3[2];
#pragma unroll
  for (int kb = 0; kb < 2; ++kb) w3[kb] = frag(w.w3t + r * kH + kb * 32 + 8 * g);
#pragma unroll
  for (int mt = 0; mt < 4; ++mt) {
    floatx4 acc = splat(w.b3[r]);
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
      acc = mma(frag(H + (mt * 16 + r) * kLd + kb * 32 + 8 * g), w3[kb], acc);
    if (r < kO) {
#pragma unroll
      for (int e = 0; e < 4; ++e) G.y[(row + mt * 16 + 4 * g + e) * kO + r] = acc[e];
    }
  }
}

enum { kPredict, kMerge, kGiven };  // what the row pass does

// Per row: M's values from Y (kPredict); or the row's loss and dL/dy, in Y's
// place, from the merge of the slot rows (kMerge) or from G.gm and G.rl.
template <int MODE>
__global__ __launch_bounds__(kRowBlock) void spai_rows_kernel(Group G) {
#pragma clang fp contract(off)
  const int64_t xb = blockIdx.x * (int64_t)kRowBlock;
  const RowSpan& A = G.mat[span_of(G, xb)];
  const int64_t xr = xb + threadIdx.x, i = xr - A.xbase + A.first;
  float* y = G.y + xr * kO;
  if (i >= A.last) {
    if (MODE != kPredict) {
#pragma unroll
      for (int s = 0; s < kO; ++s) y[s] = 0.f;
      G.rowloss[xr] = 0.0;
    }
    return;
  }
  const CsrRows C{A.rp, A.ci, A.v};
  const EntryRows E{G.ecol, G.eval, A.xbase};
  int pos[kO], js[kO];
  if (MODE == kMerge) E.slots(i, pos, js);
  else C.slots(i, pos, js);
  const double di = G.diag[A.dbase + i];
  double m[kO], gs[kO];
  float out[kO];
#pragma unroll
  for (int s = 0; s < kO; ++s) out[s] = MODE == kGiven ? 0.f : y[s];
#pragma unroll
  for (int s = 0; s < kO; ++s) {
    gs[s] = 0.0;
    m[s] = MODE == kGiven || pos[s] < 0
               ? 0.0
               : ((s == 4 ? 1.0 : 0.0) + (double)out[s]) / di;
  }
  if (MODE == kPredict) {
#pragma unroll
    for (int s = 0; s < kO; ++s)
      if (pos[s] >= 0) G.mvals[pos[s]] = m[s];
    return;
  }
  if (MODE == kGiven) {
#pragma unroll
    for (int s = 0; s < kO; ++s) gs[s] = pos[s] >= 0 ? G.gm[pos[s]] : 0.0;
    G.rowloss[xr] = G.rl[i];
  } else {
    G.rowloss[xr] = row_residual(E, i, js, m, gs);
  }
#pragma unroll
  for (int s = 0; s < kO; ++s)
    y[s] = (float)(G.scale * gs[s] / di);  // 0 for a slot without an entry
}

// The backward pass's LDS, in bf16 elements per wavefront.  R1: H1, then dH2,
// by rows; C1: H1, then dH1, by columns; C2: H2, then dH2, by columns.
constexpr int oR1 = 0, oC1 = oR1 + kTile * kLd, oC2 = oC1 + kH * kLd,
              oX = oC2 + kH * kLd, oYr = oX + kFp * kLd, oYc = oYr + kTile * kLdY,
              kPool = oYc + kOn * kLd;
// its use for the workgroup's sums: the matrices' gradients of each
// wavefront, the bias gradients of each lane group, dL/dy and loss per lane
constexpr int kMats = gB1;  // floats of the three matrices
constexpr int fB = kWaves * kMats, fB3 = fB + kWaves * 4 * 2 * kH,
              fLoss = fB3 + kWaves * kTile * kO;
static_assert(fLoss % 2 == 0 && (size_t)fLoss * 4 + kWaves * kTile * 8 <=
                                    (size_t)kWaves * kPool * sizeof(bf16),
              "the sums fit the tiles' LDS");
static_assert(gB2 == gB1 + kH && gB3 == gB2 + kH, "bias order");

// Gradient and loss partials of a group, workgroup b's at index b; those of
// workgroups below `started` are added to.
__global__ __launch_bounds__(kWaves * 64, 1) void spai_backward_kernel(
    Group G, float* __restrict__ partials, double* __restrict__ loss_part,
    int started) {
#pragma clang fp contract(off)
  __shared__ __attribute__((aligned(16))) bf16 pool[kWaves * kPool];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  bf16* R1 = pool + wave * kPool + oR1;
  bf16* C1 = pool + wave * kPool + oC1;
  bf16* C2 = pool + wave * kPool + oC2;
  bf16* Xc = pool + wave * kPool + oX;
  bf16* Yr = pool + wave * kPool + oYr;
  bf16* Yc = pool + wave * kPool + oYc;
  const Packed& w = *G.pk;
  bf16x8 w1t[4], w2t[4][2], w2[4][2], w3[4];
  float b1[4], b2[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int c = q * 16 + r;
    w1t[q] = frag(w.w1t + c * kFp + 8 * g);
    w3[q] = frag(w.w3 + c * kOk + 8 * g);
    b1[q] = w.b1[c];
    b2[q] = w.b2[c];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      w2t[q][kb] = frag(w.w2t + c * kH + kb * 32 + 8 * g);
      w2[q][kb] = frag(w.w2 + c * kH + kb * 32 + 8 * g);
    }
  }
  bool add = (int)blockIdx.x < started;

  for (int k = 0; k < G.count; ++k) {
    const int64_t ntiles = (G.mat[k].n + kTile - 1) / kTile;
    if ((int64_t)blockIdx.x * kWaves >= ntiles && add) continue;  // + 0
    floatx4 aW1[2][4], aW2[4][4], aW3[4];
    float ab1[4], ab2[4], ab3[kO];
    double lsum = 0.0;
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      aW3[a] = splat(0.f);
      ab1[a] = ab2[a] = 0.f;
#pragma unroll
      for (int b = 0; b < 4; ++b) aW2[a][b] = splat(0.f);
    }
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 4; ++b) aW1[a][b] = splat(0.f);
#pragma unroll
    for (int s = 0; s < kO; ++s) ab3[s] = 0.f;

    for (int64_t t = (int64_t)blockIdx.x * kWaves + wave; t < ntiles;
         t += (int64_t)gridDim.x * kWaves) {
      const int64_t row = G.mat[k].xbase + t * kTile;
      bf16x8 xf[4];
#pragma unroll
      for (int mt = 0; mt < 4; ++mt)
        xf[mt] = frag(G.x + (row + mt * 16 + r) * kFp + 8 * g);
      float dy[kO];
#pragma unroll
      for (int s = 0; s < kO; ++s) dy[s] = G.y[(row + lane) * kO + s];
      lsum += G.rowloss[row + lane];
      {  // dL/dy by rows and by columns, X by columns
        bf16x8 lo, hi;
#pragma unroll
        for (int s = 0; s < kOn; ++s) {
          const bf16 d = to_bf16(s < kO ? dy[s] : 0.f);
          if (s < kO) ab3[s] += dy[s];
          if (s < 8) lo[s] = d;
          else hi[s - 8] = d;
          Yc[s * kLd + lane] = d;
        }
        *(bf16x8*)(Yr + lane * kLdY) = lo;
        *(bf16x8*)(Yr + lane * kLdY + 8) = hi;
#pragma unroll
        for (int mt = 0; mt < 4; ++mt)
#pragma unroll
          for (int j = 0; j < 8; ++j) Xc[(8 * g + j) * kLd + mt * 16 + r] = xf[mt][j];
      }
      // H1 and H2 again
#pragma unroll
      for (int mt = 0; mt < 4; ++mt)
#pragma unroll
        for (int nt = 0; nt < 4; ++nt) {
          const floatx4 acc = mma(xf[mt], w1t[nt], splat(b1[nt]));
          bf16x4 h;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            h[e] = to_bf16(fmaxf(acc[e], 0.f));
            R1[(mt * 16 + 4 * g + e) * kLd + nt * 16 + r] = h[e];
          }
          *(bf16x4*)(C1 + (nt * 16 + r) * kLd + mt * 16 + 4 * g) = h;
        }
      wave_sync();
      {
        bf16x8 hf[4][2];
#pragma unroll
        for (int mt = 0; mt < 4; ++mt)
#pragma unroll
          for (int kb = 0; kb < 2; ++kb)
            hf[mt][kb] = frag(R1 + (mt * 16 + r) * kLd + kb * 32 + 8 * g);
#pragma unroll
        for (int mt = 0; mt < 4; ++mt)
#pragma unroll
          for (int nt = 0; nt < 4; ++nt) {
            floatx4 acc = splat(b2[nt]);
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) acc = mma(hf[mt][kb], w2t[nt][kb], acc);
            bf16x4 h;
#pragma unroll
            for (int e = 0; e < 4; ++e) h[e] = to_bf16(fmaxf(acc[e], 0.f));
            *(bf16x4*)(C2 + (nt * 16 + r) * kLd + mt * 16 + 4 * g) = h;
          }
      }
      wave_sync();
      // dW3[64 hid][16 out] += H2^T dY
      {
        bf16x8 yf[2];
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) yf[kb] = frag(Yc + r * kLd + kb * 32 + 8 * g);
#pragma unroll
        for (int mt = 0; mt < 4; ++mt)
#pragma unroll
          for (int kb = 0; kb < 2; ++kb)
            aW3[mt] = mma(frag(C2 + (mt * 16 + r) * kLd + kb * 32 + 8 * g), yf[kb],
                          aW3[mt]);
      }
      wave_sync();
      // dH2 = dY W3^T * [H2 > 0]; outputs from 16 on are zero
#pragma unroll
      for (int mt = 0; mt < 4; ++mt) {
        bf16x8 yf;
#pragma unroll
        for (int j = 0; j < 8; ++j) yf[j] = (bf16)0.f;
        if (g < 2) yf = frag(Yr + (mt * 16 + r) * kLdY + 8 * g);
#pragma unroll
        for (int nt = 0; nt < 4; ++nt) {
          const floatx4 acc = mma(yf, w3[nt], splat(0.f));
          bf16x4* own = (bf16x4*)(C2 + (nt * 16 + r) * kLd + mt * 16 + 4 * g);
          const bf16x4 h = *own;
          bf16x4 d;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float vv = positive(h[e]) ? acc[e] : 0.f;
            ab2[nt] += vv;
            d[e] = to_bf16(vv);
            R1[(mt * 16 + 4 * g + e) * kLd + nt * 16 + r] = d[e];
          }
          *own = d;
        }
      }
      wave_sync();
      // dW2[64 in][64 out] += H1^T dH2
      {
        bf16x8 df[4][2];
#pragma unroll
        for (int nt = 0; nt < 4; ++nt)
#pragma unroll
          for (int kb = 0; kb < 2; ++kb)
            df[nt][kb] = frag(C2 + (nt * 16 + r) * kLd + kb * 32 + 8 * g);
#pragma unroll
        for (int mt = 0; mt < 4; ++mt)
#pragma unroll
          for (int kb = 0; kb < 2; ++kb) {
            const bf16x8 hf = frag(C1 + (mt * 16 + r) * kLd + kb * 32 + 8 * g);
#pragma unroll
            for (int nt = 0; nt < 4; ++nt)
              aW2[mt][nt] = mma(hf, df[nt][kb], aW2[mt][nt]);
          }
      }
      wave_sync();
      // dH1 = dH2 W2^T * [H1 > 0]
#pragma unroll
      for (int mt = 0; mt < 4; ++mt) {
        bf16x8 df[2];
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
          df[kb] = frag(R1 + (mt * 16 + r) * kLd + kb * 32 + 8 * g);
#pragma unroll
        for (int nt = 0; nt < 4; ++nt) {
          floatx4 acc = splat(0.f);
#pragma unroll
          for (int kb = 0; kb < 2; ++kb) acc = mma(df[kb], w2[nt][kb], acc);
          bf16x4* own = (bf16x4*)(C1 + (nt * 16 + r) * kLd + mt * 16 + 4 * g);
          const bf16x4 h = *own;
          bf16x4 d;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float vv = positive(h[e]) ? acc[e] : 0.f;
            ab1[nt] += vv;
            d[e] = to_bf16(vv);
          }
          *own = d;
        }
      }
      wave_sync();
      // dW1[32 feat][64 hid] += X^T dH1
      {
        bf16x8 df[4][2];
#pragma unroll
        for (int nt = 0; nt < 4; ++nt)
#pragma unroll
          for (int kb = 0; kb < 2; ++kb)
            df[nt][kb] = frag(C1 + (nt * 16 + r) * kLd + kb * 32 + 8 * g);
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
#pragma unroll
          for (int kb = 0; kb < 2; ++kb) {
            const bf16x8 xt = frag(Xc + (mt * 16 + r) * kLd + kb * 32 + 8 * g);
#pragma unroll
            for (int nt = 0; nt < 4; ++nt)
              aW1[mt][nt] = mma(xt, df[nt][kb], aW1[mt][nt]);
          }
      }
      wave_sync();
    }

    // ---- workgroup sum of the wavefronts' gradients, in a fixed order:
    // wavefront by wavefront, and for values several lanes of one wavefront
    // hold, lane group by lane group (dL/dy and loss: lane by lane)
    __syncthreads();
    float* red = (float*)pool;
    double* lt = (double*)(red + fLoss);
    float* mine = red + wave * kMats;
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
#pragma unroll
      for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          mine[gW1 + (mt * 16 + 4 * g + e) * kH + nt * 16 + r] = aW1[mt][nt][e];
#pragma unroll
      for (int mt = 0; mt < 4; ++mt)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          mine[gW2 + (mt * 16 + 4 * g + e) * kH + nt * 16 + r] = aW2[mt][nt][e];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        mine[gW3 + (nt * 16 + 4 * g + e) * kOn + r] = aW3[nt][e];
      red[fB + ((wave * 4 + g) * 2 + 0) * kH + nt * 16 + r] = ab1[nt];
      red[fB + ((wave * 4 + g) * 2 + 1) * kH + nt * 16 + r] = ab2[nt];
    }
#pragma unroll
    for (int s = 0; s < kO; ++s) red[fB3 + threadIdx.x * kO + s] = ab3[s];
    lt[threadIdx.x] = lsum;
    __syncthreads();
    float* dst = partials + (size_t)blockIdx.x * kGradLen;
    constexpr int kQuads = kMats / 4 / (kWaves * 64);
    static_assert(kQuads * 4 * kWaves * 64 == kMats && kGradLen % 4 == 0, "quads");
    floatx4 old[kQuads];
#pragma unroll
    for (int q = 0; q < kQuads; ++q)
      old[q] = add ? ((floatx4*)dst)[q * kWaves * 64 + threadIdx.x] : splat(0.f);
#pragma unroll
    for (int q = 0; q < kQuads; ++q) {
      const int at = q * kWaves * 64 + threadIdx.x;
      floatx4 v = ((floatx4*)red)[at];
#pragma unroll
      for (int u = 1; u < kWaves; ++u) v += ((floatx4*)(red + u * kMats))[at];
      ((floatx4*)dst)[at] = old[q] + v;
    }
    if (threadIdx.x < 2 * kH) {
      float v = 0.f;
#pragma unroll
      for (int u = 0; u < 4 * kWaves; ++u) v += red[fB + u * 2 * kH + threadIdx.x];
      dst[gB1 + threadIdx.x] = (add ? dst[gB1 + threadIdx.x] : 0.f) + v;
    } else if (threadIdx.x < 2 * kH + kOn) {
      const int s = threadIdx.x - 2 * kH;
      float v = 0.f;
      if (s < kO) {
#pragma unroll 16
        for (int u = 0; u < kWaves * kTile; ++u) v += red[fB3 + u * kO + s];
      }
      dst[gB3 + s] = (add ? dst[gB3 + s] : 0.f) + v;
    } else if (threadIdx.x == 3 * kTile) {
      double l = 0.0;
#pragma unroll 16
      for (int u = 0; u < kWaves * kTile; ++u) l += lt[u];
      loss_part[blockIdx.x] = (add ? loss_part[blockIdx.x] : 0.0) + G.scale * l;
    }
    add = true;
    __syncthreads();
  }
}

// ---- the symmetric objective (1/n) ||I - S A||_F^2, S = (M + M^T) / 2:
// with mirror(p) the position of entry (j, i) for entry p = (i, j),
// S_p = (m_p + m_mirror(p)) / 2, each row's residual and g_p = dL/dS_p come
// from row_residual over S's values, and dL/dm_p = (g_p + g_mirror(p)) / 2
// (an entry of M enters S twice, at p and at its mirror).

// mirror positions, one thread per row; a missing mirror (a pattern that
// is not structurally symmetric) sets *err
__global__ void spai_mirror_kernel(int64_t n, const int32_t* __restrict__ rp,
                                   const int32_t* __restrict__ ci,
                                   int32_t* __restrict__ mirror, int* err) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  for (int p = rp[i]; p < rp[i + 1]; ++p) {
    const int j = ci[p];
    int lo = rp[j], hi = rp[j + 1];
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (ci[mid] < (int32_t)i) lo = mid + 1;
      else hi = mid;
    }
    const bool ok = lo < rp[j + 1] && ci[lo] == (int32_t)i;
    if (!ok) atomicOr(err, 1);
    mirror[p] = ok ? lo : p;
  }
}

// out_p = (in_p + in_mirror(p)) / 2 over the entries
__global__ void spai_mirror_mean_kernel(int64_t nnz, const double* __restrict__ in,
                                        const int32_t* __restrict__ mirror,
                                        double* __restrict__ out) {
#pragma clang fp contract(off)
  for (int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; p < nnz;
       p += (int64_t)gridDim.x * blockDim.x)
    out[p] = 0.5 * (in[p] + in[mirror[p]]);
}

// each row's residual under S's values: the row's loss and g_p = dL/dS_p
__global__ __launch_bounds__(kRowBlock) void spai_row_loss_kernel(int64_t n, const int32_t* __restrict__ rp,
                                     const int32_t* __restrict__ ci,
                                     const double* __restrict__ v,
                                     const double* __restrict__ svals,
                                     double* __restrict__ g,
                                     double* __restrict__ rowloss) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n) return;
  const CsrRows A{rp, ci, v};
  int pos[kO], js[kO];
  A.slots(i, pos, js);
  double m[kO], gs[kO];
#pragma unroll
  for (int s = 0; s < kO; ++s) {
    m[s] = pos[s] >= 0 ? svals[pos[s]] : 0.0;
    gs[s] = 0.0;
  }
  rowloss[i] = row_residual(A, i, js, m, gs);
#pragma unroll
  for (int s = 0; s < kO; ++s)
    if (pos[s] >= 0) g[pos[s]] = gs[s];
}

// canonical parameter k -> (gradient partial index, packed slot)
__device__ __forceinline__ int partial_index(int k) {
  if (k < kB1) return gW1 + k;  // [f][o], same row length 64
  if (k < kW2) return gB1 + (k - kB1);
  if (k < kB2) return gW2 + (k - kW2);
  if (k < kW3) return gB2 + (k - kB2);
  if (k < kB3) return gW3 + ((k - kW3) / kO) * kOn + (k - kW3) % kO;
  return gB3 + (k - kB3);
}

__device__ __forceinline__ void store_packed(Packed* pk, int k, float w) {
  const bf16 b = to_bf16(w);
  if (k < kB1) {
    pk->w1t[(k % kH) * kFp + k / kH] = b;
  } else if (k < kW2) {
    pk->b1[k - kB1] = w;
  } else if (k < kB2) {
    const int q = k - kW2;
    pk->w2[q] = b;
    pk->w2t[(q % kH) * kH + q / kH] = b;
  } else if (k < kW3) {
    pk->b2[k - kB2] = w;
  } else if (k < kB3) {
    const int q = k - kW3;
    pk->w3[(q / kO) * kOk + q % kO] = b;
    pk->w3t[(q % kO) * kH + q / kO] = b;
  } else {
    pk->b3[k - kB3] = w;
  }
}

struct AdamStep {
  float lr, beta1, beta2, eps, bc1, bc2;  // bc = 1 - beta^t
};

// sum the workgroup partials (in workgroup order); either write the
// gradient (grad != null) or take an Adam step on the master weights.  A
// chain of nparts additions: the loads of 64 go out together (one at a time
// it took 74 us at 256 partials).
constexpr int kUpdateBlock = 64;
__global__ __launch_bounds__(kUpdateBlock) void spai_update_kernel(int nparts, const float* __restrict__ partials,
                                   const double* __restrict__ loss_part,
                                   float* __restrict__ master, float* __restrict__ m1,
                                   float* __restrict__ m2, Packed* __restrict__ pk,
                                   double* __restrict__ loss_out,
                                   float* __restrict__ grad, AdamStep st) {
#pragma clang fp contract(off)
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (blockIdx.x == gridDim.x - 1) {  // a workgroup for the loss
    if (threadIdx.x > 0) return;
    double l = 0.0;
#pragma unroll 64
    for (int b = 0; b < nparts; ++b) l += loss_part[b];
    *loss_out = l;
    return;
  }
  if (k >= kNP) return;
  const int pi = partial_index(k);
  float gsum = 0.f;
#pragma unroll 64
  for (int b = 0; b < nparts; ++b) gsum += partials[(size_t)b * kGradLen + pi];
  if (grad) {
    grad[k] = gsum;
    return;
  }
  const float a = st.beta1 * m1[k] + (1.f - st.beta1) * gsum;
  const float b = st.beta2 * m2[k] + (1.f - st.beta2) * (gsum * gsum);
  m1[k] = a;
  m2[k] = b;
  const float w = master[k] - st.lr * (a / st.bc1) / (sqrtf(b / st.bc2) + st.eps);
  master[k] = w;
  store_packed(pk, k, w);
}

__global__ void spai_pack_kernel(const float* __restrict__ master,
                                 Packed* __restrict__ pk) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < kNP) store_packed(pk, k, master[k]);
}

}  // namespace
}  // namespace spk

using namespace spk;

struct spk_spai_model_s {
  DevBuf<float> master, m1, m2;
  DevBuf<Packed> pk;
  DevBuf<float> partials;
  DevBuf<double> loss_part, loss_hist;
  DevBuf<float> grad;
  DevBuf<double> diag, rsum;  // per row of what is prepared
  DevBuf<bf16> x;             // the passes' scratch, see Group
  DevBuf<float> y;
  DevBuf<double> rowloss, eval;
  DevBuf<int32_t> ecol;
  DevBuf<int> err;
  int64_t step = 0;
  int nparts = 0;
  // training objective: SPK_SPAI_LOSS_INVERSE (||I - M A||) or
  // SPK_SPAI_LOSS_SYMMETRIC (||I - S A||, S = (M + M^T) / 2), with the
  // latter's per-matrix scratch on A's pattern
  int objective = SPK_SPAI_LOSS_INVERSE;
  DevBuf<int32_t> mirror;
  DevBuf<double> mv, sv, gsv, gmv, rowl;

  void reset_optimizer() {
    hipStream_t s = stream();
    SPK_HIP_TRY(hipMemsetAsync(m1.p, 0, kNP * 4, s));
    SPK_HIP_TRY(hipMemsetAsync(m2.p, 0, kNP * 4, s));
    step = 0;
  }
  void upload(const float* host) {
    hipStream_t s = stream();
    SPK_HIP_TRY(hipMemcpyAsync(master.p, host, kNP * 4, hipMemcpyHostToDevice, s));
    SPK_HIP_TRY(hipMemsetAsync(pk.p, 0, sizeof(Packed), s));
    hipLaunchKernelGGL(spai_pack_kernel, dim3((kNP + 255) / 256), dim3(256), 0, s,
                       (const float*)master.p, pk.p);
    SPK_HIP_TRY(hipGetLastError());
    reset_optimizer();
    SPK_HIP_TRY(hipStreamSynchronize(s));
  }
  static int64_t padded(int64_t rows) {
    return (rows + kRowBlock - 1) / kRowBlock * kRowBlock;
  }
  Group group() {
    Group G{};
    G.diag = diag.p;
    G.rsum = rsum.p;
    G.x = x.p;
    G.y = y.p;
    G.rowloss = rowloss.p;
    G.pk = pk.p;
    return G;
  }
  static RowSpan span(const spk_csr_s& A, int64_t first, int64_t last, int64_t dbase,
                      int64_t xbase) {
    return RowSpan{A.rp.p, A.ci.p, A.v64.p, A.nrows, first, last, dbase, xbase};
  }
  void need_rows(int64_t rows) {
    if (diag.n < (size_t)rows) {
      diag.alloc((size_t)rows);
      rsum.alloc((size_t)rows);
    }
  }
  void need_scratch(int64_t rows, bool train) {
    if (x.n < (size_t)rows * kFp) x.alloc((size_t)rows * kFp);
    if (y.n < (size_t)rows * kO) y.alloc((size_t)rows * kO);
    if (train && rowloss.n < (size_t)rows) rowloss.alloc((size_t)rows);
  }
  void need_entries(int64_t rows) {
    if (ecol.n < (size_t)rows * kEntries) ecol.alloc((size_t)rows * kEntries);
    if (eval.n < (size_t)rows * kEntries) eval.alloc((size_t)rows * kEntries);
  }
  void launch_prepare(const Group& G, int64_t rows, int* e) {
    hipLaunchKernelGGL(spai_prepare_kernel, dim3(ceil_div(rows, kRowBlock)),
                       dim3(kRowBlock), 0, stream(), G, e);
    SPK_HIP_TRY(hipGetLastError());
  }
  // diagonal / row sums of A into the model's scratch; *e is set for a
  // matrix the slot rules reject
  void prepare(spk_csr_s& A, int* e) {
    need_rows(padded(A.nrows));
    Group G = group();
    G.count = 1;
    G.mat[0] = span(A, 0, A.nrows, 0, 0);
    launch_prepare(G, A.nrows, e);
  }
  // Prepares matrix by matrix, with mirrors for the symmetric objective;
  // throws what the first rejected one is rejected for.
  void check(const spk_csr* mats, int64_t count) {
    const bool sym = objective == SPK_SPAI_LOSS_SYMMETRIC;
    if (err.n < (size_t)(2 * count)) err.alloc((size_t)(2 * count));
    hipStream_t s = stream();
    SPK_HIP_TRY(hipMemsetAsync(err.p, 0, (size_t)(2 * count) * sizeof(int), s));
    int64_t k = 0;
    for (; k < count; ++k) {
      if (!mats[k] || mats[k]->nrows != mats[k]->ncols) break;
      prepare(*mats[k], err.p + 2 * k);
      if (sym) mirrors(*mats[k], err.p + 2 * k + 1);
    }
    std::vector<int> h((size_t)(2 * count), 0);
    SPK_HIP_TRY(hipMemcpyAsync(h.data(), err.p, h.size() * sizeof(int),
                               hipMemcpyDeviceToHost, s));
    SPK_HIP_TRY(hipStreamSynchronize(s));
    for (int64_t q = 0; q < k; ++q) {
      SPK_REQUIRE(!h[(size_t)(2 * q)], SPK_INVALID_ARGUMENT,
                  "learned SPAI needs a positive diagonal and at most 4 "
                  "entries on each side of it in every row");
      SPK_REQUIRE(!h[(size_t)(2 * q + 1)], SPK_INVALID_ARGUMENT,
                  "the symmetric objective needs a structurally symmetric pattern");
    }
    if (k == count) return;
    SPK_REQUIRE(mats[k], SPK_INVALID_ARGUMENT, "null matrix");
    SPK_REQUIRE(false, SPK_INVALID_ARGUMENT, "learned SPAI needs a square matrix");
  }
  void launch_features(const Group& G, int64_t rows) {
    hipLaunchKernelGGL(spai_features_kernel, dim3((int)(rows / kRowBlock)),
                       dim3(kRowBlock), 0, stream(), G);
    SPK_HIP_TRY(hipGetLastError());
  }
  void launch_forward(const Group& G, int64_t rows) {
    static_assert(kRowBlock % (kWaves * kTile) == 0, "whole workgroups");
    hipLaunchKernelGGL(spai_forward_kernel, dim3((int)(rows / (kWaves * kTile))),
                       dim3(kWaves * 64), 0, stream(), G);
    SPK_HIP_TRY(hipGetLastError());
  }
  template <int MODE>
  void launch_rows(const Group& G, int64_t rows) {
    hipLaunchKernelGGL(spai_rows_kernel<MODE>, dim3((int)(rows / kRowBlock)),
                       dim3(kRowBlock), 0, stream(), G);
    SPK_HIP_TRY(hipGetLastError());
  }
  // M's values on the prepared A's pattern (every entry is a slot: prepare
  // checked), kGroupRows rows at a time
  void predict_into(spk_csr_s& A, double* mvals) {
    need_scratch(padded(std::min(A.nrows, kGroupRows)), false);
    for (int64_t first = 0; first < A.nrows; first += kGroupRows) {
      const int64_t last = std::min(A.nrows, first + kGroupRows);
      Group G = group();
      G.count = 1;
      G.mat[0] = span(A, first, last, 0, 0);
      G.mvals = mvals;
      const int64_t rows = padded(last - first);
      launch_features(G, rows);
      launch_forward(G, rows);
      launch_rows<kPredict>(G, rows);
    }
  }
  // The symmetric objective's passes before the backward one: M, the
  // mirrors, S, each row's loss and dL/dS, then dL/dm (into gmv / rowl).
  // check: report a pattern that is not structurally symmetric.
  void symmetric_scratch(const spk_csr_s& A) {
    const size_t nz = (size_t)(A.nnz > 0 ? A.nnz : 1), n = (size_t)A.nrows;
    if (mirror.n < nz) {
      mirror.alloc(nz);
      mv.alloc(nz);
      sv.alloc(nz);
      gsv.alloc(nz);
      gmv.alloc(nz);
    }
    if (rowl.n < n) rowl.alloc(n);
  }
  // the mirror positions of A's entries; *e is set for a pattern that is not
  // structurally symmetric
  void mirrors(const spk_csr_s& A, int* e) {
    symmetric_scratch(A);
    hipStream_t s = stream();
    hipLaunchKernelGGL(spai_mirror_kernel, dim3((int)ceil_div(A.nrows, 256)),
                       dim3(256), 0, s, A.nrows, (const int32_t*)A.rp.p,
                       (const int32_t*)A.ci.p, mirror.p, e);
    SPK_HIP_TRY(hipGetLastError());
  }
  void symmetric_grad(spk_csr_s& A) {
    hipStream_t s = stream();
    predict_into(A, mv.p);
    mirrors(A, err.p);  // checked before
    const int gr = (int)ceil_div(A.nrows, 256);
    const int ge = (int)std::min<int64_t>(ceil_div(A.nnz > 0 ? A.nnz : 1, 256), 65536);
    hipLaunchKernelGGL(spai_mirror_mean_kernel, dim3(ge), dim3(256), 0, s, A.nnz,
                       (const double*)mv.p, (const int32_t*)mirror.p, sv.p);
    hipLaunchKernelGGL(spai_row_loss_kernel, dim3(gr), dim3(256), 0, s, A.nrows,
                       (const int32_t*)A.rp.p, (const int32_t*)A.ci.p,
                       (const double*)A.v64.p, (const double*)sv.p, gsv.p, rowl.p);
    hipLaunchKernelGGL(spai_mirror_mean_kernel, dim3(ge), dim3(256), 0, s, A.nnz,
                       (const double*)gsv.p, (const int32_t*)mirror.p, gmv.p);
    SPK_HIP_TRY(hipGetLastError());
  }
  // The gradient and loss partials of a batch (its matrices checked);
  // returns the number of workgroups that have one.
  int train_batch(const std::vector<spk_csr_s*>& batch, double scale) {
    const bool sym = objective == SPK_SPAI_LOSS_SYMMETRIC;
    int started = 0;
    for (size_t k = 0; k < batch.size();) {
      size_t e = k;
      int64_t rows = 0;
      while (e < batch.size() &&
             (e == k || (!sym && e - k < (size_t)kGroupMats &&
                         rows + padded(batch[e]->nrows) <= kGroupRows)))
        rows += padded(batch[e++]->nrows);
      need_rows(rows);
      need_scratch(rows, true);
      if (!sym) need_entries(rows);
      Group G = group();
      if (!sym) {
        G.ecol = ecol.p;
        G.eval = eval.p;
      }
      G.scale = scale;
      int64_t most = 0, base = 0;
      for (size_t q = k; q < e; ++q) {
        const spk_csr_s& A = *batch[q];
        G.mat[G.count++] = span(A, 0, A.nrows, base, base);
        base += padded(A.nrows);
        most = std::max<int64_t>(most, ceil_div(A.nrows, kTile * kWaves));
      }
      launch_prepare(G, rows, nullptr);
      if (sym) {
        symmetric_grad(*batch[k]);
        G.gm = gmv.p;
        G.rl = rowl.p;
      }
      launch_features(G, rows);
      if (sym) {
        launch_rows<kGiven>(G, rows);
      } else {
        launch_forward(G, rows);
        launch_rows<kMerge>(G, rows);
      }
      const int blocks = (int)std::max<int64_t>(1, std::min<int64_t>(most, nparts));
      hipLaunchKernelGGL(spai_backward_kernel, dim3(blocks), dim3(kWaves * 64), 0,
                         stream(), G, partials.p, loss_part.p, started);
      SPK_HIP_TRY(hipGetLastError());
      started = std::max(started, blocks);
      k = e;
    }
    return started;
  }
  // sums the batch's partials into loss_hist[at], and into grad or the
  // weights
  void update(int parts, int64_t at, float* gradient, const AdamStep& st) {
    hipLaunchKernelGGL(spai_update_kernel, dim3((kNP + kUpdateBlock - 1) / kUpdateBlock + 1),
                       dim3(kUpdateBlock), 0, stream(), parts,
                       (const float*)partials.p, (const double*)loss_part.p, master.p,
                       m1.p, m2.p, pk.p, loss_hist.p + at, gradient, st);
    SPK_HIP_TRY(hipGetLastError());
  }
};

namespace {

uint64_t host_mix(uint64_t seed, uint64_t k) {
  uint64_t z = seed + (k + 1) * 0x9E3779B97F4A7C15ULL;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
  return z ^ (z >> 31);
}

double host_u01(uint64_t z) {
  return (double)(z >> 11) * (1.0 / 9007199254740992.0);
}

// a store with A's pattern and plan, values uninitialised
spk_csr_s* clone_pattern(const spk_csr_s& A) {
  auto* M = new spk_csr_s();
  try {
    M->allocate(A.nrows, A.ncols, A.nnz);
    hipStream_t s = stream();
    SPK_HIP_TRY(hipMemcpyAsync(M->rp.p, A.rp.p, (A.nrows + 1) * 4,
                               hipMemcpyDeviceToDevice, s));
    if (A.nnz)
      SPK_HIP_TRY(hipMemcpyAsync(M->ci.p, A.ci.p, A.nnz * 4,
                                 hipMemcpyDeviceToDevice, s));
    M->h_rp = A.h_rp;
    M->plan.alloc((size_t)A.nblocks + 1);
    SPK_HIP_TRY(hipMemcpyAsync(M->plan.p, A.plan.p, (A.nblocks + 1) * sizeof(int2),
                               hipMemcpyDeviceToDevice, s));
    M->nblocks = A.nblocks;
    M->nlong = A.nlong;
    M->max_len = A.max_len;
  } catch (...) {
    delete M;
    throw;
  }
  return M;
}

}  // namespace

extern "C" {

spk_status spk_spai_model_create(uint64_t seed, spk_spai_model* out) {
  return guarded([&] {
    SPK_REQUIRE(out, SPK_INVALID_ARGUMENT, "null argument");
    auto* m = new spk_spai_model_s();
    try {
      m->master.alloc(kNP);
      m->m1.alloc(kNP);
      m->m2.alloc(kNP);
      m->grad.alloc(kNP);
      m->pk.alloc(1);
      m->nparts = ctx().num_cus > 0 ? ctx().num_cus : 256;
      m->partials.alloc((size_t)m->nparts * kGradLen);
      m->loss_part.alloc((size_t)m->nparts);
      m->loss_hist.alloc(1);
      m->err.alloc(1);
      // He-uniform hidden layers, zero output layer (M starts as Jacobi)
      std::vector<float> p(kNP, 0.f);
      const uint64_t s = seed ^ 0x4D4C50ULL;
      for (int k = kW1; k < kB1; ++k)
        p[k] = (float)((2.0 * host_u01(host_mix(s, (uint64_t)k)) - 1.0) *
                       std::sqrt(6.0 / kF));
      for (int k = kW2; k < kB2; ++k)
        p[k] = (float)((2.0 * host_u01(host_mix(s, (uint64_t)k)) - 1.0) *
                       std::sqrt(6.0 / kH));
      m->upload(p.data());
    } catch (...) {
      delete m;
      throw;
    }
    *out = m;
  });
}

spk_status spk_spai_model_destroy(spk_spai_model m) {
  return guarded([&] {
    if (!m) return;
    SPK_HIP_TRY(hipStreamSynchronize(stream()));
    delete m;
  });
}

spk_status spk_spai_model_get_params(spk_spai_model m, float* params) {
  return guarded([&] {
    SPK_REQUIRE(m && params, SPK_INVALID_ARGUMENT, "null argument");
    SPK_HIP_TRY(hipMemcpyAsync(params, m->master.p, kNP * 4,
                               hipMemcpyDeviceToHost, stream()));
    SPK_HIP_TRY(hipStreamSynchronize(stream()));
  });
}

spk_status spk_spai_model_set_params(spk_spai_model m, const float* params) {
  return guarded([&] {
    SPK_REQUIRE(m && params, SPK_INVALID_ARGUMENT, "null argument");
    m->upload(params);
  });
}

// Checkpoint file (little-endian): "SPKSPAI" + NUL, uint32 version (1),
// uint32 parameter count, int64 Adam step, then the FP32 master weights,
// Adam's first and second moments (SPK_SPAI_NPARAM floats each, canonical
// order), then a 64-bit FNV-1a hash of everything before it.
namespace {
constexpr char kCkptMagic[8] = {'S', 'P', 'K', 'S', 'P', 'A', 'I', '\0'};
constexpr uint32_t kCkptVersion = 1;
constexpr size_t kCkptHead = 8 + 4 + 4 + 8;
constexpr size_t kCkptBytes = kCkptHead + 3 * (size_t)kNP * 4 + 8;

uint64_t fnv1a(const unsigned char* p, size_t n) {
  uint64_t h = 0xcbf29ce484222325ull;
  for (size_t i = 0; i < n; ++i) h = (h ^ p[i]) * 0x100000001b3ull;
  return h;
}
}  // namespace

spk_status spk_spai_model_save(spk_spai_model m, const char* path) {
  return guarded([&] {
    SPK_REQUIRE(m && path, SPK_INVALID_ARGUMENT, "null argument");
    std::vector<unsigned char> buf(kCkptBytes);
    unsigned char* q = buf.data();
    std::memcpy(q, kCkptMagic, 8);
    std::memcpy(q + 8, &kCkptVersion, 4);
    const uint32_t np = (uint32_t)kNP;
    std::memcpy(q + 12, &np, 4);
    std::memcpy(q + 16, &m->step, 8);
    hipStream_t s = stream();
    const DevBuf<float>* parts[3] = {&m->master, &m->m1, &m->m2};
    for (int k = 0; k < 3; ++k)
      SPK_HIP_TRY(hipMemcpyAsync(q + kCkptHead + (size_t)k * kNP * 4, parts[k]->p,
                                 (size_t)kNP * 4, hipMemcpyDeviceToHost, s));
    SPK_HIP_TRY(hipStreamSynchronize(s));
    const uint64_t h = fnv1a(q, kCkptBytes - 8);
    std::memcpy(q + kCkptBytes - 8, &h, 8);
    FILE* f = std::fopen(path, "wb");
    SPK_REQUIRE(f, SPK_RUNTIME_ERROR, std::string("cannot open ") + path);
    const size_t w = std::fwrite(q, 1, kCkptBytes, f);
    const int c = std::fclose(f);
    SPK_REQUIRE(w == kCkptBytes && c == 0, SPK_RUNTIME_ERROR,
                std::string("cannot write ") + path);
  });
}

spk_status spk_spai_model_load(spk_spai_model m, const char* path) {
  return guarded([&] {
    SPK_REQUIRE(m && path, SPK_INVALID_ARGUMENT, "null argument");
    FILE* f = std::fopen(path, "rb");
    SPK_REQUIRE(f, SPK_RUNTIME_ERROR, std::string("cannot open ") + path);
    std::vector<unsigned char> buf(kCkptBytes + 1);
    const size_t r = std::fread(buf.data(), 1, buf.size(), f);
    std::fclose(f);
    const unsigned char* q = buf.data();
    SPK_REQUIRE(r >= 16 && std::memcmp(q, kCkptMagic, 8) == 0, SPK_RUNTIME_ERROR,
                std::string(path) + " is not a learned-SPAI checkpoint");
    uint32_t ver = 0, np = 0;
    std::memcpy(&ver, q + 8, 4);
    std::memcpy(&np, q + 12, 4);
    SPK_REQUIRE(ver == kCkptVersion && np == (uint32_t)kNP, SPK_RUNTIME_ERROR,
                std::string(path) + ": unsupported checkpoint version or size");
    SPK_REQUIRE(r == kCkptBytes, SPK_RUNTIME_ERROR,
                std::string(path) + ": checkpoint has the wrong length");
    uint64_t h = 0;
    std::memcpy(&h, q + kCkptBytes - 8, 8);
    SPK_REQUIRE(h == fnv1a(q, kCkptBytes - 8), SPK_RUNTIME_ERROR,
                std::string(path) + ": checkpoint checksum mismatch");
    int64_t step = 0;
    std::memcpy(&step, q + 16, 8);
    SPK_REQUIRE(step >= 0, SPK_RUNTIME_ERROR, std::string(path) + ": bad step");
    // weights (and their packed copy) first, then the optimiser state that
    // upload() resets
    m->upload(reinterpret_cast<const float*>(q + kCkptHead));
    hipStream_t s = stream();
    SPK_HIP_TRY(hipMemcpyAsync(m->m1.p, q + kCkptHead + (size_t)kNP * 4,
                               (size_t)kNP * 4, hipMemcpyHostToDevice, s));
    SPK_HIP_TRY(hipMemcpyAsync(m->m2.p, q + kCkptHead + 2 * (size_t)kNP * 4,
                               (size_t)kNP * 4, hipMemcpyHostToDevice, s));
    SPK_HIP_TRY(hipStreamSynchronize(s));
    m->step = step;
  });
}

spk_status spk_spai_model_set_objective(spk_spai_model m, int objective) {
  return guarded([&] {
    SPK_REQUIRE(m, SPK_INVALID_ARGUMENT, "null argument");
    SPK_REQUIRE(objective == SPK_SPAI_LOSS_INVERSE ||
                    objective == SPK_SPAI_LOSS_SYMMETRIC,
                SPK_INVALID_ARGUMENT, "unknown objective");
    m->objective = objective;
  });
}

spk_status spk_spai_model_get_objective(spk_spai_model m, int* objective) {
  return guarded([&] {
    SPK_REQUIRE(m && objective, SPK_INVALID_ARGUMENT, "null argument");
    *objective = m->objective;
  });
}

spk_status spk_spai_features(spk_csr A, float* d_features) {
  return guarded([&] {
    SPK_REQUIRE(A && d_features, SPK_INVALID_ARGUMENT, "null argument");
    // computed by the same per-row code as the features pass, through a
    // model that holds only its scratch
    spk_spai_model_s tmp;
    tmp.err.alloc(1);
    tmp.check(&A, 1);
    const CsrRows R{A->rp.p, A->ci.p, A->v64.p};
    const double* diag = tmp.diag.p;
    const double* rsum = tmp.rsum.p;
    float* X = d_features;
    launch_map(A->nrows, [=] __device__(int64_t i) {
      float x[kF];
      row_features(R, diag, rsum, i, x);
#pragma unroll
      for (int f = 0; f < kF; ++f) X[i * kF + f] = x[f];
    });
    SPK_HIP_TRY(hipStreamSynchronize(stream()));
  });
}

spk_status spk_spai_loss_grad(spk_spai_model m, spk_csr A, double* loss,
                              float* grad) {
  return guarded([&] {
    SPK_REQUIRE(m && A && loss, SPK_INVALID_ARGUMENT, "null argument");
    m->check(&A, 1);
    const int parts = m->train_batch({A}, 1.0 / (double)A->nrows);
    hipStream_t s = stream();
    m->update(parts, 0, m->grad.p, AdamStep{});
    SPK_HIP_TRY(hipMemcpyAsync(loss, m->loss_hist.p, 8, hipMemcpyDeviceToHost, s));
    if (grad)
      SPK_HIP_TRY(hipMemcpyAsync(grad, m->grad.p, kNP * 4, hipMemcpyDeviceToHost, s));
    SPK_HIP_TRY(hipStreamSynchronize(s));
  });
}

spk_status spk_spai_train(spk_spai_model m, const spk_csr* mats, int64_t count,
                          const spk_spai_train_config* cfg,
                          double* loss_history) {
  return guarded([&] {
    TraceRange trace_("spk_spai_train");
    SPK_REQUIRE(m && mats && cfg && count > 0, SPK_INVALID_ARGUMENT,
                "null argument");
    SPK_REQUIRE(cfg->epochs >= 0 && cfg->batch_matrices > 0 &&
                    cfg->learning_rate > 0.0,
                SPK_INVALID_ARGUMENT, "bad training configuration");
    m->check(mats, count);
    const int64_t per_epoch = (count + cfg->batch_matrices - 1) / cfg->batch_matrices;
    const int64_t total = cfg->epochs * per_epoch;
    if (m->loss_hist.n < (size_t)(total > 0 ? total : 1))
      m->loss_hist.alloc((size_t)(total > 0 ? total : 1));
    hipStream_t s = stream();
    std::vector<int64_t> order((size_t)count);
    const float b1 = 0.9f, b2 = 0.999f;
    int64_t h = 0;
    for (int64_t e = 0; e < cfg->epochs; ++e) {
      for (int64_t k = 0; k < count; ++k) order[(size_t)k] = k;
      for (int64_t k = count - 1; k > 0; --k) {  // Fisher-Yates
        uint64_t z = host_mix(cfg->shuffle_seed, (uint64_t)(e * count + k));
        std::swap(order[(size_t)k], order[(size_t)(z % (uint64_t)(k + 1))]);
      }
      for (int64_t b0 = 0; b0 < count; b0 += cfg->batch_matrices) {
        const int64_t b1e = std::min(count, b0 + cfg->batch_matrices);
        int64_t rows = 0;
        std::vector<spk_csr_s*> batch;
        for (int64_t k = b0; k < b1e; ++k) {
          batch.push_back(mats[order[(size_t)k]]);
          rows += batch.back()->nrows;
        }
        const int parts = m->train_batch(batch, 1.0 / (double)rows);
        m->step += 1;
        AdamStep st;
        st.lr = (float)cfg->learning_rate;
        st.beta1 = b1;
        st.beta2 = b2;
        st.eps = 1e-8f;
        st.bc1 = (float)(1.0 - std::pow((double)b1, (double)m->step));
        st.bc2 = (float)(1.0 - std::pow((double)b2, (double)m->step));
        m->update(parts, h, nullptr, st);
        ++h;
      }
    }
    if (loss_history && total > 0)
      SPK_HIP_TRY(hipMemcpyAsync(loss_history, m->loss_hist.p, total * 8,
                                 hipMemcpyDeviceToHost, s));
    SPK_HIP_TRY(hipStreamSynchronize(s));
  });
}

spk_status spk_spai_predict(spk_spai_model m, spk_csr A, spk_csr* M_out) {
  return guarded([&] {
    TraceRange trace_("spk_spai_predict");
    SPK_REQUIRE(m && A && M_out, SPK_INVALID_ARGUMENT, "null argument");
    m->check(&A, 1);
    spk_csr_s* M = clone_pattern(*A);
    try {
      m->predict_into(*A, M->v64.p);
      SPK_HIP_TRY(hipStreamSynchronize(stream()));
    } catch (...) {
      delete M;
      throw;
    }
    *M_out = M;
  });
}

}  // extern "C"
