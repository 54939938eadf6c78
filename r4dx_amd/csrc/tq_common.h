// tq_common.h -- what the M <= 64 trellis kernels (trellis_gemv.hip: a K slice of A staged whole, and the fused transform;
// trellis_mid.hip: in chunks) share: the weight words' loads, the K-part combine, the split hand-over with its fixed-order
// slice sum, and the FWHT-128 epilogue. A linear's bits depend on (K, N, KB, SKG, SK) only, so both kernels run these very sums.
#pragma once
#include "r4d_dev.h"

#include <type_traits>

namespace {

template <int KB>
struct Words {
  unsigned w[KB + 1];   // [0] history, [1..KB] own words
};

#define R4_RSRC_FLAGS 0x00020000
typedef __amdgpu_buffer_rsrc_t r4_rsrc;
__device__ __forceinline__ r4_rsrc r4_make_rsrc(const void* p, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)p, (short)0, (int)bytes, R4_RSRC_FLAGS);
}

// Byte offsets, inside a (pair, k-tile) block, of the lane's own words (KB c .. KB c + KB - 1 of tile t)
// and history word (KB c - 1 mod 8 KB); block q of a step sits q * 64 KB bytes further.
template <int KB>
struct LaneWords {
  unsigned own, hist;
  __device__ __forceinline__ LaneWords(int q, int t, int c) {
    const unsigned tile = (unsigned)(q * 16 * KB + t * 8 * KB);
    own = (tile + KB * c) * 4u;
    hist = (tile + (KB * c - 1 + 8 * KB) % (8 * KB)) * 4u;
  }
};

// Cache policy of the weight loads: nontemporal (each word is read once per launch; measured ~2 % faster
// per step than the default policy).
constexpr int kWeightPolicy = 2;

// One step's words of this lane from the slice buffer at step byte offset so (out of range -> 0).
template <int KB, bool HIST = true>
__device__ __forceinline__ void load_words(Words<KB>& s, r4_rsrc r, const LaneWords<KB>& lw, unsigned so) {
  // one wide load per lane where the KB words allow it (buffer loads need dword alignment only): KB 4 one dwordx4,
  // KB 5 a dwordx4 and a dword, KB 3 a dwordx3 -- not KB dword loads, each of which would touch every line of the step
  if constexpr (KB == 4 || KB == 5) {
    const r4u4 v = __builtin_bit_cast(r4u4, __builtin_amdgcn_raw_buffer_load_b128(r, lw.own + so, 0, kWeightPolicy));
    s.w[1] = v[0]; s.w[2] = v[1]; s.w[3] = v[2]; s.w[4] = v[3];
    if constexpr (KB == 5) s.w[5] = __builtin_amdgcn_raw_buffer_load_b32(r, lw.own + so + 16, 0, kWeightPolicy);
  } else if constexpr (KB == 3) {
    const auto v = __builtin_amdgcn_raw_buffer_load_b96(r, lw.own + so, 0, kWeightPolicy);
    s.w[1] = v[0]; s.w[2] = v[1]; s.w[3] = v[2];
  } else {
#pragma unroll
    for (int i = 0; i < KB; ++i) s.w[1 + i] = __builtin_amdgcn_raw_buffer_load_b32(r, lw.own + so + 4 * i, 0, kWeightPolicy);
  }
  if constexpr (HIST) s.w[0] = __builtin_amdgcn_raw_buffer_load_b32(r, lw.hist + so, 0, kWeightPolicy);
}

// n / d for the staging loops' row split (d = M <= 64, n below 2^20): one high multiply by the launch-uniform
// floor(2^32 / d) + 1, exact whenever n d < 2^32 (the error term n e / (d 2^32), 0 < e <= d, stays below 1 / d);
// d = 1 (whose multiplier would need 33 bits) is marked by 0 and returns n.
// The multipliers for d = 0..64 as a constant table (d = 0 unused): a scalar load of the launch's M instead of a 64-bit
// division formed with VALU ops in every wave.
struct R4DivMagic {
  unsigned m[65];
  constexpr R4DivMagic() : m() {
    for (unsigned d = 1; d <= 64; ++d) m[d] = d == 1u ? 0u : (unsigned)(0x100000000ull / d) + 1u;
  }
};
__constant__ constexpr R4DivMagic kR4DivMagic{};
__device__ __forceinline__ unsigned r4_div_magic(unsigned d) { return kR4DivMagic.m[d]; }
__device__ __forceinline__ int r4_div_by(int n, unsigned magic) {
  return magic ? (int)__umulhi((unsigned)n, magic) : n;
}


// The K-part combine: the SK waves of a pair (wave ks holds part ks) added in k order through LDS into wave ks = 0.
// part_acc holds [(SK - 1) NPW][8 MT][64] floats and is free again after the caller's next barrier.
template <int MT, int NPW, int SK>
__device__ __forceinline__ void tq_combine(r4f4 (&acc)[MT][2], float* part_acc, int pl, int ks, int lane) {
  if constexpr (SK > 1) {
    if (ks > 0) {
      float* dst = part_acc + ((size_t)((ks - 1) * NPW + pl) * 8 * MT) * 64;
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int f = 0; f < 2; ++f)
#pragma unroll
          for (int j = 0; j < 4; ++j) dst[((i * 2 + f) * 4 + j) * 64 + lane] = acc[i][f][j];
    }
    __syncthreads();
    if (ks == 0) {
#pragma unroll
      for (int s = 1; s < SK; ++s) {
        const float* src = part_acc + ((size_t)((s - 1) * NPW + pl) * 8 * MT) * 64;
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int f = 0; f < 2; ++f)
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[i][f][j] += src[((i * 2 + f) * 4 + j) * 64 + lane];
      }
    }
  }
}

// What one unit's end needs (tq_finish).
struct TqOut {
  const float* svh;
  void* C;
  float* ws;
  unsigned* tickets;
  int M, N, SKG, full;
  float out_scale;
};

// LDS bytes of a unit's end: the part accumulators (dead before the group's sums are formed in the same bytes), then
// the ticket flag.
constexpr size_t tq_end_lds_flag(int MT, int NPW, int SK, int M) {
  const size_t parts = (size_t)(SK - 1) * NPW * 8 * MT * 64 * 4;
  const size_t sums = MT > 1 || NPW >= 2 ? (size_t)M * NPW * 32 * 4 : 0;
  return parts > sums ? parts : sums;
}
constexpr size_t tq_end_lds(int MT, int NPW, int SK, int M) { return tq_end_lds_flag(MT, NPW, SK, M) + 16; }

// A unit's end, after tq_combine. Lane l of wave (pl, ks = 0) holds rows 16 i + 4 (l >> 4) + j of column slot nb = l & 15
// of fragment cs: true column 32 pair + 16 (nb >> 3) + (nb & 7) + 8 cs.
//   * SKG = 1, raw: the sums are C.
//   * SKG = 1 in a workgroup that holds its whole group (NPW = 4): the sums meet in LDS and are finished from there.
//   * else the partials go to ws -- above one row tile through LDS, as 16-byte row pieces (the accumulators' own 4-byte
//     stores cost 3 to 5 us a launch at 49 and 64 rows) -- and the last of the group's SKG 4 / NPW contributors (ticket)
//     sums the slices: run p (0..7) is 0.f + slices p, p + 8, ... in order, then the runs in order 0..7 (an absent slice
//     adds +0.f, which changes nothing) -- the same arithmetic for every element whatever M is. The loads are coherent
//     (sc1) 16-byte buffer loads, every slice of a batch of 8 requested before any is added.
// Each 32-lane half of a wave then owns one row's 128 sums, 4 adjacent columns per lane, from the slice sum to the
// store (r4_fwht128_rows): no LDS copy of the slice sums, no stage through the LDS crossbar and one 8-byte store per lane.
// STAGE: also one row tile above 8 rows goes through LDS.
template <int MT, int NPW, int SK, bool STAGE = false>
__device__ __forceinline__ void tq_finish(const r4f4 (&acc)[MT][2], unsigned char* lds, const TqOut& o, int group, int pair,
                                          int ks, int ky) {
  constexpr int NT = 64 * NPW * SK;
  const int lane = threadIdx.x & 63;
  const int M = o.M, N = o.N, SKG = o.SKG, full = o.full;
  const int nb = lane & 15, rq = lane >> 4;
  const int gcol0 = (pair & 3) * 32 + 16 * (nb >> 3) + (nb & 7);   // inside the group
  float* Cf = (float*)o.C;
  unsigned short* Cb = (unsigned short*)o.C;
  const int n0 = group * 128;
  float* red = (float*)lds;                     // [M][128]
  if (SKG == 1 && !full) {
    if (ks == 0) {
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int r = 16 * i + 4 * rq + j;
          if (r < M) {
            Cf[(size_t)r * N + n0 + gcol0] = acc[i][0][j];
            Cf[(size_t)r * N + n0 + gcol0 + 8] = acc[i][1][j];
          }
        }
    }
    return;
  }
  const int c0 = 4 * (lane & 31);               // the 4 columns this lane finishes
  if constexpr (NPW == 4 && SK == 1) {
    // The workgroup holds its whole group. A path of its own, short and in line with the k loop: run through the split's
    // code below, with svh asked for behind the barrier, an unsplit launch took 0.2 us more at 1 row, whatever K, and up to
    // 1.3 us at 64 (128 x 1024, 17 / 64 rows 5.0 / 7.5 -> 4.3 / 6.2 us; 5120 x 34816, 64 rows 68.9 -> 67.9).
    if (SKG == 1) {
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int r = 16 * i + 4 * rq + j;
          if (r < M) {
            red[r * 128 + gcol0] = acc[i][0][j];
            red[r * 128 + gcol0 + 8] = acc[i][1][j];
          }
        }
      float sv[4];
      r4_load_f32<4>(o.svh + n0 + c0, sv);      // in flight over the barrier
      __syncthreads();
      for (int r = (int)threadIdx.x >> 5; r < M; r += NT / 32) {
        float v[4];
        r4_load_f32<4>(red + r * 128 + c0, v);
        r4_fwht128_rows<4>(v, lane);
        unsigned h[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) h[e] = r4_bf16_rn_sel((v[e] * sv[e]) * o.out_scale);
        r4_store_u16<4>(Cb + (size_t)r * N + n0 + c0, h);
      }
      return;
    }
  }
  // the partials pass through LDS and leave as whole 16-byte row pieces (up to 8 rows their few 4-byte stores are as fast)
  const bool staged = MT > 1 || (STAGE && M > 8);
  constexpr int kCols = 32 * NPW;               // the workgroup's columns
  const unsigned sy4 = (unsigned)M * (unsigned)N * 4u;
  const r4_rsrc wsr = r4_make_rsrc(o.ws, (unsigned)SKG * sy4);
  if (staged) {
    if constexpr (SK > 1) __syncthreads();      // the part accumulators have been read
    const int lcol0 = gcol0 & (kCols - 1);
    if (ks == 0) {
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int r = 16 * i + 4 * rq + j;
          if (r < M) {
            red[r * kCols + lcol0] = acc[i][0][j];
            red[r * kCols + lcol0 + 8] = acc[i][1][j];
          }
        }
    }
    __syncthreads();
    const unsigned base = (unsigned)ky * sy4 + (unsigned)(n0 + (kCols == 128 ? 0 : (pair * 32) & (128 - kCols))) * 4u;
    for (int it = (int)threadIdx.x; it < M * (kCols / 4); it += NT) {
      const int r = it / (kCols / 4), cq = it & (kCols / 4 - 1);
      __builtin_amdgcn_raw_buffer_store_b128(*(const r4u4*)(red + r * kCols + 4 * cq), wsr,
                                             base + (unsigned)r * (unsigned)N * 4u + 16u * cq, 0, 16);
    }
  } else if (ks == 0) {
    float* wsy = o.ws + (size_t)ky * M * N;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int r = 16 * i + 4 * rq + j;
        if (r < M) {
          r4_store_coherent(&wsy[(size_t)r * N + n0 + gcol0], acc[i][0][j]);
          r4_store_coherent(&wsy[(size_t)r * N + n0 + gcol0 + 8], acc[i][1][j]);
        }
      }
  }
  if (!r4_ticket_last(&o.tickets[group * R4_TICKET_WORDS], (unsigned)(SKG * (4 / NPW)),
                      (int*)(lds + tq_end_lds_flag(MT, NPW, SK, M))))
    return;
  float sv[4] = {0.f, 0.f, 0.f, 0.f};
  if (full) r4_load_f32<4>(o.svh + n0 + c0, sv);
  // rows per thread and pass, all their slices requested at once (one row at a time, a workgroup at 49 rows made seven
  // memory round trips one after the other)
  constexpr int kU = MT == 1 || (MT == 4 && SK == 4) ? 1 : 2;
  for (int it0 = (int)threadIdx.x; it0 < M * 32; it0 += kU * NT) {
    float v[kU][4];
    unsigned off[kU];
#pragma unroll
    for (int u = 0; u < kU; ++u)
      off[u] = ((unsigned)min((it0 + u * NT) >> 5, M - 1) * (unsigned)N + (unsigned)(n0 + c0)) * 4u;
    auto slice = [&](int u, unsigned sy) {
      return __builtin_bit_cast(r4f4, __builtin_amdgcn_raw_buffer_load_b128(wsr, off[u] + sy, 0, 16));
    };
    // at most one slice per run (every planned split): branch-free, a slice past SKG reads past the buffer and gives the
    // +0.f of an empty run (a load under a branch would also keep its registers live around the caller's loop)
    auto few = [&](auto n) {
      constexpr int kN = decltype(n)::value;
      r4f4 t[kU][kN];
#pragma unroll
      for (int u = 0; u < kU; ++u)
#pragma unroll
        for (int p = 0; p < kN; ++p) t[u][p] = slice(u, p < SKG ? (unsigned)p * sy4 : 0x80000000u);
#pragma unroll
      for (int u = 0; u < kU; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[u][e] = 0.f + t[u][0][e];
#pragma unroll
          for (int p = 1; p < kN; ++p) v[u][e] += 0.f + t[u][p][e];
          if (kN < 8) v[u][e] += 0.f;
        }
    };
    if (SKG <= 4) {
      few(std::integral_constant<int, 4>());
    } else if (SKG <= 8) {
      few(std::integral_constant<int, 8>());
    } else {
#pragma unroll
      for (int u = 0; u < kU; ++u) {
#pragma unroll 1
        for (int p = 0; p < 8; ++p) {
          float run[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
          for (int y = p; y < SKG; y += 8) {
            const r4f4 t = slice(u, (unsigned)y * sy4);
#pragma unroll
            for (int e = 0; e < 4; ++e) run[e] += t[e];
          }
#pragma unroll
          for (int e = 0; e < 4; ++e) v[u][e] = p == 0 ? run[e] : v[u][e] + run[e];
        }
      }
    }
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int it = it0 + u * NT, r = it >> 5;
      if (full) r4_fwht128_rows<4>(v[u], lane);
      if (it >= M * 32) break;
      if (!full) {
        *(r4f4_a4*)(Cf + (size_t)r * N + n0 + c0) = (r4f4){v[u][0], v[u][1], v[u][2], v[u][3]};
        continue;
      }
      unsigned h[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) h[e] = r4_bf16_rn_sel((v[u][e] * sv[e]) * o.out_scale);
      r4_store_u16<4>(Cb + (size_t)r * N + n0 + c0, h);
    }
  }
}

}  // namespace
