// spk_link.hpp -- sums over a whole grid inside one kernel.
//
// A persistent kernel of at most GridLink::blocks blocks (one per CU, so that
// all of them are resident) adds numbers over its blocks without ending: every
// block publishes its sum in a slot of its own and reads everybody's.  A
// kernel boundary plus a one-block finisher costs about 4.5 us on this
// chip; one exchange costs about 2 us and leaves each block's data in its
// registers.
//
// A slot carries its own readiness: the double is published as two 64-bit
// words, each half of it beside the exchange's number (the tag), so a reader
// that sees both tags has the whole value.  Nothing is ever reset and no
// store has to be ordered against another.  Two slot sets alternate: a block
// writes a set again only after the exchange in between, which it leaves
// when every block has entered it, that is, has read the set.  Tags grow
// over the launches (the first tag is kept in device memory, advanced by
// block 0 at the end of a kernel), so the words of an earlier launch never
// match.  All blocks add the slots in the same order: the totals are
// bit-identical everywhere.
//
// Other work on the GPU can keep a block from starting for as long as it
// likes.  A wait therefore gives up after GridLink::polls polls: its block
// leaves the kernel with nothing written, the link is marked for renewal, and
// so are the state of the solve and of every later kernel that finds the link
// so.  The host then renews the link, goes back to the state before those
// launches and takes the kernels that need no exchange.
#pragma once

#include "spk_internal.hpp"

namespace spk {

constexpr int kLinkBlocks = 256;
constexpr int kLinkWidth = 2;  // sums per exchange, at most

struct GridLink {
  unsigned long long* slots;  // [2][kLinkWidth][kLinkBlocks][2]
  unsigned* tag;              // the last tag used by an earlier launch
  int* expired;               // set: to be renewed before its next use
  int blocks;                 // of a launch, at most
  unsigned polls;             // of a wait, at most
};
constexpr size_t kLinkSlotWords = (size_t)2 * kLinkWidth * kLinkBlocks * 2;
constexpr size_t kLinkWords = kLinkSlotWords + 2;

// The library's link (its device memory is made and cleared with the library)
// for launches on the library stream.  On a stream that is masked to some of
// the CUs it allows one block, which waits for nobody.
GridLink grid_link();
// Clears the slots, the tag and the flag, in stream order.
void renew_link(const GridLink& l);

// A poll is a round trip through memory, 0.5 us and more: 0.1 s or so, during
// which a process that is swapped out polls nothing.  An exchange takes a few
// polls, and giving up costs no more than that and the steps since.
constexpr unsigned kLinkPolls = 1u << 17;
// Beyond this tag the link is renewed, so that tags never come round to those
// that unused slots still hold; a launch uses fewer than are left.
constexpr unsigned kLinkLastTag = 0xF0000000u;

// What link_sum has to know of the link's state at the start of the kernel; the
// load is under way beside the data's (DATA threads hold data).
template <int DATA>
__device__ __forceinline__ int link_open(const GridLink& l) {
  int e = 0;
  if (threadIdx.x >= DATA && gridDim.x > 1) e = *l.expired;
  return __builtin_amdgcn_readfirstlane(e);
}
// the end of a kernel whose exchanges all went through; one thread of block 0
__device__ __forceinline__ void link_close(const GridLink& l, unsigned tag) {
  if (gridDim.x == 1) return;
  *l.tag = tag;
  if (tag >= kLinkLastTag) *l.expired = 1;
}

__device__ __forceinline__ unsigned long long link_word(unsigned tag, unsigned half) {
  return ((unsigned long long)tag << 32) | half;
}

// Sums v[0..W-1] over the threads of the grid; every thread gets the totals.
// A block has DATA threads that hold data and one more wavefront, the link's,
// which publishes and polls: loads return in order, so a wavefront with data
// loads in flight would wait for all of them before it saw a slot.  The
// link's wavefront adds nothing (its v is ignored).  red: link_lds(DATA)
// doubles of LDS.  tag: the exchange's number, the same in every block and
// one more than the last.  stale: link_open's answer.  false, in every thread:
// the link is to be renewed or the wait expired, v holds nothing and the block
// has to leave.
constexpr int link_lds(int data) {
  return 2 * kLinkWidth * (data / 64) + kLinkWidth + 1;
}

template <int W, int DATA>
__device__ __forceinline__ bool link_sum(const GridLink& l, int stale, unsigned tag,
                                         double (&v)[W], double* red) {
  constexpr int NW = DATA / 64, NS = kLinkBlocks / 64;
  static_assert(W <= kLinkWidth && NW <= 64, "slots");
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, G = gridDim.x;
  const bool linker = wid == NW;
  double* part = red + (tag & 1) * kLinkWidth * NW;
  double* tot = red + 2 * kLinkWidth * NW;
  if (!linker) {
#pragma unroll
    for (int k = 0; k < W; ++k) {
      const double t = wave_sum_dpp(v[k]);
      if (lane == 0) part[k * NW + wid] = t;
    }
  }
  __syncthreads();
  if (G == 1) {
#pragma unroll
    for (int k = 0; k < W; ++k) {
      double t = part[k * NW];
#pragma unroll
      for (int w = 1; w < NW; ++w) t += part[k * NW + w];
      v[k] = t;
    }
    return true;
  }
  if (linker) {
    unsigned long long* set = l.slots + (size_t)(tag & 1) * kLinkWidth * kLinkBlocks * 2;
#pragma unroll
    for (int k = 0; k < W; ++k) {
      const double t = wave_sum_dpp(lane < NW ? part[k * NW + lane] : 0.0);
      // lane 0 stores the low word, lane 1 the high one
      const unsigned half = (unsigned)(lane == 0 ? __double2loint(t) : __double2hiint(t));
      if (lane < 2 && !stale)
        __hip_atomic_store(set + ((size_t)k * kLinkBlocks + blockIdx.x) * 2 + lane,
                           link_word(tag, half), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    }
    unsigned long long lo[W][NS], hi[W][NS];
    bool ok = true;
    unsigned polls = stale ? l.polls : 0;
    for (;;) {
      bool all = true;
#pragma unroll
      for (int k = 0; k < W; ++k)
#pragma unroll
        for (int q = 0; q < NS; ++q) {
          const int b = lane + q * 64;
          const unsigned long long* s = set + ((size_t)k * kLinkBlocks + b) * 2;
          lo[k][q] = hi[k][q] = link_word(tag, 0);
          if (b < G) {
            lo[k][q] = __hip_atomic_load(s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            hi[k][q] = __hip_atomic_load(s + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          }
        }
#pragma unroll
      for (int k = 0; k < W; ++k)
#pragma unroll
        for (int q = 0; q < NS; ++q)
          all = all && (unsigned)(lo[k][q] >> 32) == tag && (unsigned)(hi[k][q] >> 32) == tag;
      if (__all(all) && !stale) break;
      if (++polls >= l.polls) {
        ok = false;
        break;
      }
    }
#pragma unroll
    for (int k = 0; k < W; ++k) {
      double t = 0.0;
#pragma unroll
      for (int q = 0; q < NS; ++q)
        t += __hiloint2double((int)(unsigned)hi[k][q], (int)(unsigned)lo[k][q]);
      t = wave_sum_dpp(t);
      if (lane == 0) tot[k] = t;
    }
    if (lane == 0) {
      tot[kLinkWidth] = ok ? 0.0 : 1.0;
      if (!ok)
        __hip_atomic_store(l.expired, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < W; ++k) v[k] = tot[k];
  // one answer for the wavefront: its branches are scalar
  return __builtin_amdgcn_readfirstlane(__double2hiint(tot[kLinkWidth])) == 0;
}

}  // namespace spk
