// tq_units.h -- the division of a trellis GEMM launch's work among its workgroups, shared by the prefill kernel
// (trellis_m256.hip) and the 17..64-row kernel (trellis_mid.hip).
#pragma once
#include "r4d_dev.h"

namespace {

// The work of a launch is U = (N / 128) * SKG units -- unit u = group * SKG + y is K slice y of column group u / SKG
// -- of nst steps each, taken in unit order. Data-parallel (P = 0): workgroup (group, y) takes one unit. Balanced
// (P > 0 workgroups, used when U exceeds the CUs and is not a multiple of them): workgroup c takes the steps
// an even share (T / P, one more for the first T % P) of the T = U nst, P <= U so that a range spans at most the end of one unit, whole units
// and the start of one more. A unit cut by a range boundary stays one fold from 0.f in k order: the workgroup that
// holds its start runs that part FIRST and publishes its fp32 accumulators through ws (then its flag),
// the workgroup that holds the rest runs it LAST, starting from those accumulators (so every element is the same
// sum, bit for bit). Workgroups are dispatched in index order and the publisher's part is its first work, so the
// wait cannot deadlock; it is bounded anyway, and a wait that runs out poisons its results with NaN.
constexpr int kSegWhole = 0, kSegPublish = 1, kSegContinue = 2;
constexpr int kFlagStride = 4;            // words between two workgroups' flags
// Workgroup c's flag is word kFlagStride c + 1 of the ticket buffer: never word 32 g, the counter of 128-column group g
// that the M <= 64 kernel's split hand-over takes tickets on, so a flag left set can never be read as a ticket count.
__device__ __forceinline__ unsigned* m2_flag(unsigned* flags, unsigned c) { return flags + (size_t)c * kFlagStride + 1; }

// A workgroup's share: steps [beg, end) of the launch's units in order (unit u = group * SKG + y, nst steps each).
struct M2Share {
  int ub, sb, ue, se, whole0, nseg;
};
__device__ __forceinline__ M2Share m2_share(int N, int SKG, int nst, int P) {
  // T = (N / 128) * SKG * nst <= (N / 128) * K / 64 steps fits 32 bits; workgroup c gets T / P steps, one more for the
  // first T % P workgroups
  int beg, end;
  if (P > 0) {
    const unsigned T = (unsigned)(N / 128) * (unsigned)SKG * (unsigned)nst, q = T / (unsigned)P, r = T % (unsigned)P;
    const unsigned c = blockIdx.x;
    beg = (int)(c * q + (c < r ? c : r));
    end = beg + (int)q + (c < r ? 1 : 0);
  } else {
    beg = (blockIdx.x * SKG + blockIdx.y) * nst;
    end = beg + nst;
  }
  M2Share sh;
  sh.ub = beg / nst; sh.sb = beg - sh.ub * nst; sh.ue = end / nst; sh.se = end - sh.ue * nst;
  sh.whole0 = sh.sb ? sh.ub + 1 : sh.ub;
  sh.nseg = (sh.se ? 1 : 0) + (sh.ue - sh.whole0) + (sh.sb ? 1 : 0);
  return sh;
}
// Segment si in run order: the start of unit ue (published), the whole units, the rest of unit ub (continued).
struct M2Seg {
  int u, s0, s1, kind;
};
__device__ __forceinline__ M2Seg m2_seg(const M2Share& sh, int si, int nst) {
  M2Seg g;
  if (sh.se && si == 0) { g.u = sh.ue; g.s0 = 0; g.s1 = sh.se; g.kind = kSegPublish; }
  else if (sh.sb && si == sh.nseg - 1) { g.u = sh.ub; g.s0 = sh.sb; g.s1 = nst; g.kind = kSegContinue; }
  else { g.u = sh.whole0 + si - (sh.se ? 1 : 0); g.s0 = 0; g.s1 = nst; g.kind = kSegWhole; }
  return g;
}

// The reader's side of a cut unit: one thread waits (bounded) for the previous workgroup's flag and clears it for the next
// launch. Returns whether the wait ran out. `word` is an LDS word free for this; the workgroup meets two barriers.
__device__ __forceinline__ bool r4_wait_published(unsigned* flags, int* word) {
  if (threadIdx.x == 0) {
    unsigned* f = m2_flag(flags, blockIdx.x - 1);
    int spin = 0;
    while (__hip_atomic_load(f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0u && spin < (1 << 24)) {
      __builtin_amdgcn_s_sleep(8);
      ++spin;
    }
    __hip_atomic_store(f, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *(volatile int*)word = spin < (1 << 24) ? 0 : 1;
  }
  __syncthreads();
  const bool late = *(volatile int*)word != 0;
  __syncthreads();
  return late;
}

// The device's compute units (cached per device).
inline int r4_cus() {
  static int cache[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (cache[dev] == 0) {
    int n = 0;
    cache[dev] = hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0 ? n : 256;
  }
  return cache[dev];
}
// Workgroups of the balanced form for a launch of U units (0: data-parallel): used when U exceeds the compute units and
// is not a multiple of them, and ws (for the published accumulators) and the tickets (for the flags) are there.
inline int r4_balanced_p(int N, int SKG, bool have_ws, bool have_tickets) {
  const int G = N / 128, U = G * SKG, cus = r4_cus();
  if (!have_ws || !have_tickets || U <= cus || U % cus == 0) return 0;
  if ((long long)cus * kFlagStride + 1 > (long long)G * R4_TICKET_WORDS) return 0;   // the flags fit the ticket buffer
  return cus;
}

}  // namespace
