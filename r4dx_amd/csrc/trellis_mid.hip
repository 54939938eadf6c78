// trellis_mid.hip -- the trellis linear where a K slice of A does not fit the LDS whole, and for most of 17..64 rows, on gfx950
// (r4d_gemm_trellis_nt_m64 and its _raw, _wq, _parts and no-allocation forms; trellis_gemv.hip has the rule): the batch, and the
// tail of a prompt.
//
// DESIGN (MI355X): the decode (about 4 VALU lane-ops per weight) bounds this range, as it does for fewer rows; the MFMAs
// (2 to 4 row tiles) take a quarter to a half of its time. So the decode stays the GEMV's -- each wave decodes one tile pair
// straight into MFMA B fragments, nothing of it passes through LDS -- and only A is shared: the workgroup stages it in
// LDS, in MFMA operand order, a chunk of CS 64-k steps at a time in two buffers, so a row is read from L2 once per
// workgroup and not once per wave. (Each wave reading its own A fragments from L2, which this replaces, waited for them:
// MT x 2 KiB of scattered 32-byte pieces per 1 KiB of weights. Before -> now, 29 rows: 5120 x 34816 95 -> 49 us, 17408 x
// 5120 52 -> 33; 64 rows: 171 -> 68 and 97 -> 47; 49 rows, KB 5: 5120 x 16384 60 -> 34, 6144 x 5120 52 -> 26. What is left
// over the decode's own time is one wave per SIMD's latencies (0.5 us a step at two row tiles, 0.25 of it decode issue) and
// 9 to 15 us of launch, first loads and split hand-over.)
//
// The sums are the M <= 16 kernel's, bit for bit: SK = 1 -- a wave runs its pair's whole K slice, the workgroup holds a
// 128-column group; SK = 4 -- four waves split each pair's slice into contiguous parts added in k order, the workgroup
// holds two pairs. An SK = 1 launch has only N / 32 SKG waves, one per SIMD or less over most shapes, so a launch whose
// units (column groups x SKG) exceed the CUs without being a multiple of them runs balanced (tq_units.h): one workgroup
// per CU over an even share of the steps; a cut unit's accumulators are handed on through its own place in ws.
#include "r4d_host.h"
#include "tq_common.h"
#include "tq_units.h"
#include "r4d_mi355x.h"

namespace {

// 64-k steps per staged chunk: 8 to 16 KiB of A per buffer at SK = 1, 16 to 32 KiB over the four parts at SK = 4
__host__ __device__ constexpr int mid_cs(int MT, int SK) { return SK == 1 ? (MT <= 2 ? 4 : 2) : (MT <= 2 ? 2 : 1); }
__host__ __device__ constexpr int mid_stage(int MT, int SK) { return SK * mid_cs(MT, SK) * MT * 2048; }
constexpr int mid_pairs(int SK) { return SK == 1 ? 4 : 2; }

template <int KB, int MT, int SK, bool WQ>
__global__ __launch_bounds__(64 * mid_pairs(SK) * SK, WQ ? 1 : SK == 1 ? 2 : 4) void tq_mid_kernel(
    const R4AParts ap, const unsigned* __restrict__ W, const TqOut out0, int K, const float* __restrict__ wsc, int wq_gsh,
    unsigned long long* __restrict__ clk, int P) {
  constexpr int NPW = mid_pairs(SK), NT = 64 * NPW * SK;
  constexpr int BLK = 16 * KB;                   // words per (pair, k-tile) block
  constexpr unsigned kStepBytes = 4 * BLK * 4;
  constexpr int CS = mid_cs(MT, SK), kStage = mid_stage(MT, SK);
  constexpr int MR = 16 * MT, RP = NT / 8;       // staged rows; rows (of 64 k) per pass of the workgroup
  constexpr int AU = SK * CS * MR / RP;          // 16-byte A loads per thread and chunk
  static_assert(SK * CS * MR % RP == 0, "whole staging passes");
  constexpr int PF = SK == 4 || MT == 4 ? 2 : 4;  // weight steps in flight per wave
  // the history word of a lane's run: loaded, but at KB 5 with 4 row tiles taken from the neighbour lane (three VALU ops a
  // step), whose ring slots and address would not fit the registers
  constexpr bool kHist = !(KB == 5 && MT == 4);
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int pl = wave % NPW, ks = wave / NPW;
  const int SKG = out0.SKG;
  const int KT = K >> 4, ktw = KT / SKG;
  const int steps = (ktw + 3) >> 2;              // steps of a K slice
  const int nsw = (steps + SK - 1) / SK;         // ... of a part
  const bool probe = clk != nullptr && blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0;
  if (probe) {
    clk[0] = __builtin_amdgcn_s_memtime();
    clk[1] = __builtin_amdgcn_s_memrealtime();
  }

  // SK = 1: this workgroup's segments of the launch's units (tq_units.h); SK = 4: its column half-group and slice
  M2Share sh;
  if constexpr (SK == 1) sh = m2_share(out0.N, SKG, steps, P);
  else { sh.ub = sh.sb = sh.ue = sh.se = sh.whole0 = 0; sh.nseg = 1; }
#pragma unroll 1
  for (int si = 0; si < sh.nseg; ++si) {
    // the thread index and the sizes pass through an empty asm at every segment, so the addresses and row masks derived
    // from them are formed per segment instead of being hoisted out of the segment loop (live through the k loop, they
    // overflow the scalar registers)
    TqOut out = out0;
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid), "+s"(out.M), "+s"(out.N));
    const int lane = tid & 63, M = out.M, N = out.N;
    const int q = lane >> 4, t = (lane >> 3) & 1, c = lane & 7;
    M2Seg sg;
    int pair, group, ky;
    if constexpr (SK == 1) {
      sg = m2_seg(sh, si, steps);
      group = sg.u / SKG;
      ky = sg.u - group * SKG;
      pair = group * 4 + pl;
    } else {
      sg.s0 = 0; sg.s1 = nsw; sg.kind = kSegWhole;
      pair = blockIdx.x * NPW + pl;
      group = blockIdx.x >> 1;
      ky = blockIdx.y;
    }
    const int kt0 = ky * ktw + 4 * sg.s0, ktv = ktw - 4 * sg.s0;      // first k-tile; the slice's k-tiles from it
    const int nmax = sg.s1 - sg.s0;                                   // steps of the longest part
    const int st_beg = ks * nsw;                                      // (0 at SK = 1)
    const int nst = SK == 1 ? nmax : max(0, min(nsw, steps - st_beg));
    const int nch = (nmax + CS - 1) / CS;
    const unsigned short* __restrict__ A = r4_part_a(ap, group * 128);
    __syncthreads();                             // the LDS of the previous segment's end is free
    bool late = false;
    if (sg.kind == kSegContinue) late = r4_wait_published(out.tickets, (int*)lds);

    // ---- weights: PF steps in flight per wave
    const r4_rsrc wr = r4_make_rsrc(W + ((size_t)pair * KT + kt0) * BLK, (unsigned)ktv * BLK * 4u);
    const LaneWords<KB> lw(q, t, c);
    Words<KB> ring[PF];
    auto load_w = [&](Words<KB>& w, int s) {
      load_words<KB, kHist>(w, wr, lw, (unsigned)(st_beg + min(s, nst - 1)) * kStepBytes);
    };

    // ---- A: thread item u of a chunk is 8 k of one row of one (part, step): a 16-byte load, coalesced over 128-byte row
    // segments, and two 8-byte LDS writes (its halves of the fragments h = 0, 1). A step's rows sit as [h][row tile][slot]
    // 16-byte fragments, slot = 16 g + (row ^ 8 (g & 1)) for k-tile g: a fragment read is a permutation of its 16 bank
    // slots, and the writes of a half wave (8 rows x 8 chunks) meet each bank twice, their minimum. Rows past M and
    // k-tiles of the last step past the slice read past the buffer and are 0 (a whole step past a part is staged as it
    // comes and never multiplied).
    const r4_rsrc ar = r4_make_rsrc(A, (unsigned)((size_t)M * K * 2));
    const int k8 = tid & 7, g8 = k8 >> 1;
    // item u is item 0 moved by whole rows and steps, the same for every thread, unless the rows wrap inside a pass (MT 3)
    constexpr bool kEven = MR % RP == 0 || RP % MR == 0;
    unsigned aoff[kEven ? 1 : AU];
    auto a_row = [&](int u) { return ((tid >> 3) + u * RP) % MR; };
    auto a_step = [&](int t8, int u) {           // of the slice; t8 = tid >> 3
      const int ps = (t8 + u * RP) / MR, part = ps / CS;
      return part * nsw + ps - part * CS;
    };
#pragma unroll
    for (int u = 0; u < (kEven ? 1 : AU); ++u)
      aoff[u] = (unsigned)(((size_t)a_row(u) * K + 16 * (kt0 + 4 * a_step(tid >> 3, u) + g8) + 8 * (k8 & 1)) * 2);
    auto a_delta = [&](int u) -> unsigned {      // kEven: item u's bytes from item 0
      constexpr int kRows = MR >= RP ? MR / RP : 1, kSteps = RP >= MR ? RP / MR : 1;
      const int ps = u / kRows * kSteps, part = ps / CS;
      return (unsigned)(((size_t)(u % kRows) * RP * K + 64 * (part * nsw + ps - part * CS)) * 2);
    };
    r4u4 areg[AU];
    auto load_a = [&](int ch) {
      const int dk = 4 * CS * ch;
      unsigned off[AU];
#pragma unroll
      for (int u = 0; u < AU; ++u) off[u] = (kEven ? aoff[0] + a_delta(u) : aoff[kEven ? 0 : u]) + 32u * dk;
      if (ktw & 3) {                             // the slice's last step has k-tiles past its end
        int t8 = tid >> 3;
        asm volatile("" : "+v"(t8));             // formed here, not kept through the k loop
#pragma unroll
        for (int u = 0; u < AU; ++u)
          if (4 * a_step(t8, u) + g8 + dk >= ktv) off[u] = 0xFFFFFFF0u;
      }
#pragma unroll
      for (int u = 0; u < AU; ++u)
        areg[u] = __builtin_bit_cast(r4u4, __builtin_amdgcn_raw_buffer_load_b128(ar, off[u], 0, 0));
    };
    auto put_a = [&](int ch) {
      unsigned char* stg = lds + (ch & 1) * kStage;
#pragma unroll
      for (int u = 0; u < AU; ++u) {
        const int row = a_row(u), ps = ((tid >> 3) + u * RP) / MR;
        unsigned char* p = stg + (ps * 2 * MT + (row >> 4)) * 1024 + (16 * g8 + ((row & 15) ^ (8 * (g8 & 1)))) * 16 + 8 * (k8 & 1);
        *(r4u2*)p = (r4u2){areg[u][0], areg[u][1]};
        *(r4u2*)(p + MT * 1024) = (r4u2){areg[u][2], areg[u][3]};
      }
    };
    const unsigned frag0 = (unsigned)(ks * CS * 2 * MT * 1024 + (16 * q + ((lane & 15) ^ (8 * (q & 1)))) * 16);

    load_a(0);
#pragma unroll
    for (int i = 0; i < PF; ++i) load_w(ring[i], i);

    // Lane l of the pair's wave holds rows 16 i + 4 (l >> 4) + j, column slot l & 15 of fragment cs (tq_finish). A cut
    // unit's accumulators travel through the unit's own elements of ws (its slice; SKG = 1: slice 0)
    // byte offset in ws of row 16 i + 4 rq + j, fragment f of this lane; a row past M is past the buffer
    const r4_rsrc fr = r4_make_rsrc(out.ws + (size_t)ky * M * N, (unsigned)((size_t)M * N * 4));
    auto fix_off = [&](unsigned n, int i, int f, int j) {
      const unsigned r = (unsigned)(16 * i + 4 * (lane >> 4) + j);
      const unsigned col = (unsigned)(group * 128 + (pair & 3) * 32 + 16 * ((lane >> 3) & 1) + (lane & 7) + 8 * f);
      return r < (unsigned)M ? (r * n + col) * 4u : 0xFFFFFFF0u;
    };
    r4f4 acc[MT][2];
    if (sg.kind == kSegContinue) {
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int f = 0; f < 2; ++f)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const float v = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(fr, fix_off(N, i, f, j), 0, 16));
            acc[i][f][j] = late ? __builtin_nanf("") : v;
          }
    } else {
#pragma unroll
      for (int i = 0; i < MT; ++i) acc[i][0] = acc[i][1] = (r4f4){0.f, 0.f, 0.f, 0.f};
    }

    // A step's operands: its A fragments (LDS) and its decoded B fragments, d[cs][h].
    struct Ops {
      r4h8 a[MT][2];
      unsigned d[2][2][4];
    };
    auto operands = [&](Ops& o, const Words<KB>& w, int s, unsigned frag) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < MT; ++i) o.a[i][h] = *(const r4h8*)(lds + frag + (h * MT + i) * 1024);
      unsigned wl[KB + 1];
      wl[0] = kHist ? w.w[0] : r4_hist_word(w.w[KB], lane);
#pragma unroll
      for (int i = 1; i <= KB; ++i) wl[i] = w.w[i];
      r4_decode<KB>(wl, o.d);
      if constexpr (WQ) {
        // the _wq measurement: this lane's k-tile and two columns under their group scales
        const int kt = kt0 + (st_beg + s) * 4 + q;
        float sc[2] = {1.0f, 1.0f};
        if (kt < KT) {
          const size_t row = (size_t)(kt >> wq_gsh) * N + (size_t)pair * 32 + 16 * t + c;
          sc[0] = wsc[row];
          sc[1] = wsc[row + 8];
        }
        r4_wq_apply(o.d, sc);
      }
    };
    auto multiply = [&](const Ops& o) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const r4h8 b0 = r4_frag(o.d[0][h]), b1 = r4_frag(o.d[1][h]);
#pragma unroll
        for (int i = 0; i < MT; ++i) {
          acc[i][0] = r4_mfma16(o.a[i][h], b0, acc[i][0]);
          acc[i][1] = r4_mfma16(o.a[i][h], b1, acc[i][1]);
        }
      }
    };
    // Chunk ch starts: its stage is complete and the other one free once every wave is here; the next chunk goes into
    // that one, and the loads of the one after are issued (a chunk's time ahead of their use).
    unsigned frag = frag0;
    auto chunk = [&](int ch) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      if (ch + 1 < nch) {
        put_a(ch + 1);
        load_a(ch + 2);
      }
      frag = frag0 + (ch & 1) * kStage;
    };

    put_a(0);
    load_a(1);
    int st = 0;
    if constexpr (SK == 1) {
      // One wave per SIMD: nothing else hides this wave's LDS reads and MFMA latencies, so a step's operands are formed a
      // step ahead of its MFMAs.
      Ops cur, nxt;
      chunk(0);
      operands(cur, ring[0], 0, frag);
      nxt = cur;   // defined on every path (left undefined on one, its registers would stay live around the segment loop)
      load_w(ring[0], PF);
      __builtin_amdgcn_sched_barrier(0);
      for (; st + PF < nst; st += PF) {
#pragma unroll
        for (int i = 0; i < PF; ++i) {
          if ((i + 1) % CS == 0) chunk((st + i + 1) / CS);
          __builtin_amdgcn_sched_barrier(0);
          operands(nxt, ring[(i + 1) % PF], st + i + 1, frag + ((i + 1) % CS) * 2 * MT * 1024);
          multiply(cur);
          __builtin_amdgcn_sched_barrier(0);
          load_w(ring[(i + 1) % PF], st + i + 1 + PF);
          cur = nxt;
        }
      }
#pragma unroll
      for (int i = 0; i < PF; ++i) {
        if (st + i >= nst) break;
        if (st + i + 1 < nst) {
          if ((i + 1) % CS == 0) chunk((st + i + 1) / CS);
          operands(nxt, ring[(i + 1) % PF], st + i + 1, frag + ((i + 1) % CS) * 2 * MT * 1024);
        }
        multiply(cur);
        cur = nxt;
      }
    } else {
      for (; st + PF <= nst; st += PF) {
#pragma unroll
        for (int i = 0; i < PF; ++i) {
          if (i % CS == 0) chunk((st + i) / CS);
          Ops o;
          operands(o, ring[i], st + i, frag + (i % CS) * 2 * MT * 1024);
          multiply(o);
          load_w(ring[i], st + i + PF);
          __builtin_amdgcn_sched_barrier(0);   // one step at a time: no decode hoisted across the reload
        }
      }
      // the last steps; a part with fewer steps than the longest still meets the chunks' barriers
      for (; st < nmax; st += PF) {
#pragma unroll
        for (int i = 0; i < PF; ++i) {
          if (i % CS == 0 && (st + i) / CS < nch) chunk((st + i) / CS);
          if (st + i < nst) {
            Ops o;
            operands(o, ring[i], st + i, frag + (i % CS) * 2 * MT * 1024);
            multiply(o);
          }
        }
      }
    }
    __syncthreads();                         // the stages are dead: the unit's end reuses their bytes

    tq_combine<MT, NPW, SK>(acc, (float*)lds, pl, ks, lane);
    if (probe && si == 0) {
      clk[2] = __builtin_amdgcn_s_memtime();
      clk[3] = __builtin_amdgcn_s_memrealtime();
    }
    if (sg.kind == kSegPublish) {
      unsigned n = (unsigned)N;
      asm volatile("" : "+v"(n));              // the offsets are formed here, not kept from the segment's start
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int f = 0; f < 2; ++f)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(acc[i][f][j]), fr, fix_off(n, i, f, j), 0, 16);
      // every store acknowledged before the barrier, then one thread raises the flag
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
      __syncthreads();
      if (threadIdx.x == 0)
        __hip_atomic_store(m2_flag(out.tickets, blockIdx.x), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      continue;
    }
    tq_finish<MT, NPW, SK, true>(acc, lds, out, group, pair, ks, ky);
  }
}

template <int KB, int MT, int SK, bool WQ>
void mid_launch(const r4d_gemv_args& a) {
  const size_t stage = 2 * (size_t)mid_stage(MT, SK), end = tq_end_lds(MT, mid_pairs(SK), SK, a.M);
  const size_t smem = stage > end ? stage : end;
  static std::atomic<unsigned long long> lds_set{0};
  if (smem > 64 * 1024) r4d::allow_lds((const void*)tq_mid_kernel<KB, MT, SK, WQ>, lds_set, "gemm_trellis_nt_m64");
  const R4AParts ap = r4_parts((const void*)a.a0, (const void*)a.a1, a.n_split, (const void*)a.a2, a.n_end1,
                               (const void*)a.a3, a.n_end2);
  const TqOut out{(const float*)a.svh, (void*)a.c, (float*)a.ws, (unsigned*)a.tickets, a.M, a.N, a.SKG, a.full, a.out_scale};
  // Balanced where a unit is long: the hand-over and a second start cost about as much as 10 steps. Data-parallel against
  // balanced, 29 rows: 5120 x 34816 SKG 1 (80 steps a unit, 272 units) 62.4 / 51.8 us; 24 rows: 5120 x 17408 SKG 2 (40
  // steps) 35.4 / 33.1; 29 rows: 17408 x 5120 SKG 8 (34 steps, 320 units) 33.2 / 36.4.
  const int steps = (a.K / 16 / a.SKG + 3) / 4;
  const int P = SK == 1 && steps >= 40 ? r4_balanced_p(a.N, a.SKG, a.ws != 0, a.tickets != 0) : 0;
  const dim3 grid = P > 0 ? dim3(P) : dim3(a.N / 32 / mid_pairs(SK), a.SKG);
  hipLaunchKernelGGL((tq_mid_kernel<KB, MT, SK, WQ>), grid, dim3(64 * mid_pairs(SK) * SK), smem, (hipStream_t)a.stream, ap,
                     (const unsigned*)a.w, out, a.K, (const float*)a.wsc, a.wq_gsh, (unsigned long long*)a.clk, P);
}
template <int KB, int SK, bool WQ>
void mid_launch_mt(const r4d_gemv_args& a) {
  if (a.M <= 16) mid_launch<KB, 1, SK, WQ>(a);
  else if (a.M <= 32) mid_launch<KB, 2, SK, WQ>(a);
  else if (a.M <= 48) mid_launch<KB, 3, SK, WQ>(a);
  else mid_launch<KB, 4, SK, WQ>(a);
}
template <int KB>
void mid_launch_kb(const r4d_gemv_args& a, bool sk1, const char* entry) {
  if (a.wsc) {
    if constexpr (KB == 3) r4d::fail(entry, "KB must be 4 or 5");
    else if (sk1) mid_launch_mt<KB, 1, true>(a);
    else mid_launch_mt<KB, 4, true>(a);
  } else if (sk1) {
    mid_launch_mt<KB, 1, false>(a);
  } else {
    mid_launch_mt<KB, 4, false>(a);
  }
}

}  // namespace

void r4d::gemv_mid(const r4d_gemv_args& a, bool sk1, const char* entry) {
  if (a.KB == 4) mid_launch_kb<4>(a, sk1, entry);
  else if (a.KB == 5) mid_launch_kb<5>(a, sk1, entry);
  else mid_launch_kb<3>(a, sk1, entry);
}
