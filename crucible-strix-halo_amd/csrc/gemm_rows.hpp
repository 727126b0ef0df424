// EXL3 linear over many rows (a prompt chunk): fused decode + MFMA GEMM with the output
// transform in its epilogue.  The few-row path (gemm.hpp) splits K over waves and writes
// partial sums; here every wave runs the whole of K for its own column pair and a workgroup's
// rows, so no partial sum leaves the wave and each weight is decoded once per 16 NRB rows.
//
// Workgroup: 4 waves x one column pair each (128 columns, one output Hadamard block) x up to
// 16 NRB rows.  Two workgroups per CU (2 waves per SIMD, 256 registers each), so one's
// epilogue runs beside the other's main loop.  Activations (chunks of 64 k) and the waves' weights
// are copied from memory straight into LDS two chunks ahead, no registers; one barrier per
// chunk (two steps).  Every wave reads every row's fragments there and keeps its decoded B
// fragments in registers.
//
// Bound by issue: a step of a wave (32 k x 32 columns) is 62 VALU of decode (289 cycles at 4
// bpw) and 2 NRB MFMAs of 17 cycles, which leave the VALU about half of their time: ~440 cycles
// for 8 row blocks.  2048 -> 4096 at 4 bpw, 2,047 rows: 52 us (657 TFLOP/s) with settled clocks.  Parts
// taken out, in shorter runs where the whole took 56: without its epilogue 50, its sums 45, its
// decode 41, its MFMAs 35; the few-row path's GEMM took 158 us there and its output transform 15.
// With the activations and weights staged through registers instead the loop ran as long (56.7 us)
// but spilled at 7 and 8 bpw and in the mcg and 3inst codebooks; reading the windows a step earlier
// gained nothing (60 us).
//
// Sums: K in the few-row path's splits (4 S of them, LinearPlan), added in its order, so a
// row's result is bitwise the same in either path.  Three levels: the split's MFMA
// accumulators, the K segment's sum (registers), and with S > 1 the sum of the segments before
// (parked in the workspace, in the wave's own layout).
#pragma once

#include "gemm.hpp"
#include "rows_rule.hpp"

namespace cx {

// LDS of the row loop below, for workgroups of 4 waves: activation chunks of 16 NRB rows x 64
// halves (NXB buffers: one read, the others on their way), then per wave a ring of 4 weight chunks
// (two steps each: two read, two on their way).
template <int K2, int NRB, int NXB>
struct RowsLds {
  static constexpr int kChunk = 16 * NRB * 128;
  static constexpr int kWeights = 2 * 4 * TileDwords(K2) * 4;
  static constexpr int kBytes = NXB * kChunk + 4 * 4 * kWeights;
};

// Main loop of a wave (one of 4 of its workgroup): its column pair (rw: the pair's tiles) times NA
// 16-row blocks (rx: the rows, ldx_bytes apart; past them zeros), all `steps` steps of 32 k (a
// multiple of 4), MFMA sums into acc.  step_end(s) runs after step s's MFMAs.  On return no copy is
// in flight, but other waves may still read the LDS.  All four waves call it together.
template <int K2, int CB, int NA, int NRB, int NXB, typename StepEnd>
__device__ __forceinline__ void RowsLoop(u32x4_t rw, u32x4_t rx, int ldx_bytes, int steps, char* smem,
                                         float4_t (&acc)[NA][2], StepEnd&& step_end) {
  // In an SGPR also where the compiler cannot tell (the copies' offsets are scalar operands).
  const int ldx = __builtin_amdgcn_readfirstlane(ldx_bytes);
  using L = RowsLds<K2, NRB, NXB>;
  constexpr int T = TileDwords(K2), SD = 4 * T, ND = WindowDwords(K2);
  constexpr int CBYTES = L::kChunk, WBYTES = L::kWeights;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const LaneRun<K2> lr(lane);
  char* const wslot = smem + NXB * CBYTES + wave * 4 * WBYTES;
  const uint32_t xlds = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(uintptr_t)(LdsChar*)smem);
  const uint32_t wlds = xlds + NXB * CBYTES + wave * 4 * WBYTES;
  uint32_t woff[2][ND];
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int i = 0; i < ND; ++i) woff[j][i] = (uint32_t)(((2 * j + lr.tile) * T + (lr.d0 + i) % T) * 4);
  // Activation chunk c (16 NA rows x 128 bytes): copy i of wave w moves rows 8 (4 i + w) .. + 7
  // (1 KB, whole 128-byte lines), lane l the 16-byte piece (l & 7) ^ (l >> 3) of row l >> 3, so
  // piece p of row r lies at piece p ^ (r & 7) of its 128 bytes: the 8 rows of a fragment read
  // then cover all banks.  Rows past the entry read as zeros.
  constexpr int XL = (NA + 1) / 2;
  const uint32_t xoff = (uint32_t)((wave * 8 + (lane >> 3)) * ldx + 16 * ((lane & 7) ^ (lane >> 3)));
  auto load_x = [&](int c, int buf) __attribute__((always_inline)) {
    CopyToLds<4, XL, 4096>(rx, xoff, (uint32_t)(c * 128), xlds + buf * CBYTES + wave * 1024, 32u * (uint32_t)ldx);
  };
  uint32_t xrd[2];  // the lane's fragment of the chunk's step j, row block 0
#pragma unroll
  for (int j = 0; j < 2; ++j) xrd[j] = (uint32_t)((lane & 15) * 128 + 16 * ((4 * j + (lane >> 4)) ^ (lane & 7)));
  // Weight chunk c (steps 2 c, 2 c + 1 of the wave's column pair, contiguous): K2 / 2 dwords per
  // lane at even rates; at odd ones (half-bit rates) K2 dwords per lane every second chunk.
  constexpr bool PAIRED = K2 & 1;
  constexpr int WD = PAIRED ? K2 : K2 / 2;  // dwords per lane of a copy
  constexpr int NW = WD / 4 + WD % 4;       // its instructions: 4 dwords per lane, then single ones
  auto load_w = [&](int c, int buf) __attribute__((always_inline)) {  // PAIRED: c and buf even
    const uint32_t so = (uint32_t)(c * WBYTES), l = wlds + buf * WBYTES;
    if constexpr (WD / 4 > 0) CopyToLds<4, WD / 4, 1024>(rw, (uint32_t)lane * 16, so, l, 1024u);
    if constexpr (WD % 4 > 0) CopyToLds<1, WD % 4, 256>(rw, (uint32_t)lane * 4, so + 1024 * (WD / 4), l + 1024 * (WD / 4), 256u);
  };
  auto read_windows = [&](uint32_t (&v)[2][3], int buf, int j) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
#pragma unroll
      for (int i = 0; i < ND; ++i)
        v[k][i] = *reinterpret_cast<const uint32_t*>(wslot + buf * WBYTES + j * SD * 4 + woff[k][i]);
      if constexpr (ND == 2) v[k][2] = 0u;
    }
  };
  auto decode = [&](const uint32_t (&v)[2][3], half8_t (&b)[2]) __attribute__((always_inline)) {
    half4_t lo0, hi0, lo1, hi1;
    DecodeRun<K2, CB>(v[0][0], v[0][1], v[0][2], lr.shift, lo0, hi0);
    DecodeRun<K2, CB>(v[1][0], v[1][1], v[1][2], lr.shift, lo1, hi1);
    b[0] = half8_t{lo0[0], lo0[1], lo0[2], lo0[3], lo1[0], lo1[1], lo1[2], lo1[3]};
    b[1] = half8_t{hi0[0], hi0[1], hi0[2], hi0[3], hi1[0], hi1[1], hi1[2], hi1[3]};
  };

  // Chunk c is multiplied while activation chunks up to c + NXB - 1 and weight chunks up to c + 3
  // (decoded a step ahead) are copied.  Copies past the last chunk are unconditional (zeros, or
  // other columns of the rows).
  static_assert(NXB == 2 || NXB == 3, "one or two activation chunks ahead");
  load_w(0, 0);
  if constexpr (!PAIRED) load_w(1, 1);
  load_x(0, 0);
  if constexpr (NXB == 3) load_x(1, 1);
  if constexpr (!PAIRED) load_w(2, 2);
  // Copies that may stay in flight at a chunk's start: those of the chunk before, but for what the
  // chunk itself needs (NXB = 2: its activations; PAIRED: its weights).
  constexpr int NLEFT = NXB == 3 ? (PAIRED ? XL : XL + NW) : (PAIRED ? 0 : NW);
  half8_t b[2];
  {
    WaitLoadsBarrier<NLEFT>();  // chunk 0, weight chunks 0 and 1
    uint32_t v[2][3];
    read_windows(v, 0, 0);
    decode(v, b);
  }
  int rbuf = 0, wbuf = 0;  // buffers of activation chunk s / 2 and, at s0, of weight chunk s0 / 2
  for (int s0 = 0; s0 < steps; s0 += 4) {  // steps is a multiple of 4
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int s = s0 + q, j = q & 1;
      if (j == 0) {
        // Activation chunk s / 2 was asked for NXB - 1 chunks ago, weight chunk s / 2 + 1 two chunks
        // ago.  After the barrier every wave's copies are there, and the buffers of the chunk
        // before are free.  PAIRED: two weight chunks at even chunks, before the activations, one
        // chunk before their first use.
        WaitLoadsBarrier<NLEFT>();
        if (PAIRED && q == 0) load_w((s >> 1) + 2, wbuf ^ 2);
        load_x((s >> 1) + NXB - 1, rbuf == 0 ? NXB - 1 : rbuf - 1);
        if (!PAIRED) load_w((s >> 1) + 3, (wbuf + (q >> 1) + 3) & 3);
      }
      uint32_t v[2][3];
      read_windows(v, (wbuf + ((q + 1) >> 1)) & 3, (q + 1) & 1);  // step s + 1
      half8_t av[NA];
#pragma unroll
      for (int i = 0; i < NA; ++i)
        av[i] = __builtin_bit_cast(half8_t, *reinterpret_cast<const u32x4_t*>(smem + rbuf * CBYTES + i * 2048 + xrd[j]));
      half8_t nb[2];
      decode(v, nb);
#pragma unroll
      for (int i = 0; i < NA; ++i) {
        acc[i][0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av[i], b[0], acc[i][0], 0, 0, 0);
        acc[i][1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av[i], b[1], acc[i][1], 0, 0, 0);
      }
      // Decoded here, a few VALU after each MFMA, and not after the fold's branch (the compiler
      // sinks the decode past it otherwise, and nothing runs under the MFMAs).
      asm volatile("" : "+v"(nb[0]), "+v"(nb[1]));
      __builtin_amdgcn_sched_group_barrier(0x100, 2 * ND + NA, 0);
#pragma unroll
      for (int i = 0; i < 2 * NA; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, (72 + 2 * NA - 1) / (2 * NA), 0);
      }
      __builtin_amdgcn_sched_barrier(0);
      b[0] = nb[0];
      b[1] = nb[1];
      if (j == 1) rbuf = rbuf == NXB - 1 ? 0 : rbuf + 1;
      step_end(s);
    }
    wbuf ^= 2;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the last copies: the caller reuses their LDS
}

struct RowsJob {
  const uint32_t* tiles;
  const __half* svh;
  const __half* xp;  // [M][16 A] fp16, MFMA row order
  // S > 1: [entries][ncp][nrb][2][64][4]; the few-row path's S M O floats hold it, since the rows
  // padded to whole entries are fewer than 2 M (nrb at most ceil(M / 16)).
  float* part;
  void* y;           // row r at y + r * ldy (fp32 or fp16)
  int ldy, f16;
  int M, A, ncp, S;
  int nrb;      // 16-row blocks of an entry
  int entries;  // row entries
};
struct RowsMulti {
  int n;
  int start[kMaxMultiJobs + 1];  // first workgroup of each job
  RowsJob job[kMaxMultiJobs];
};

template <int K2, int CB>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) Exl3GemmRowsKernel(RowsMulti gm) {
  constexpr int NRB = kRowsMaxBlocks;
  constexpr int T = TileDwords(K2);
  constexpr int NXB = 3;
  constexpr int ER = 32;  // rows of an epilogue slab
  __shared__ __align__(16) char smem[RowsLds<K2, NRB, NXB>::kBytes];
  static_assert(ER * 132 * 4 <= RowsLds<K2, NRB, NXB>::kBytes, "the epilogue slab reuses the loop's LDS");

  const int L = (int)blockIdx.x;
  int jb = 0;
  while (jb + 1 < gm.n && L >= gm.start[jb + 1]) ++jb;  // uniform
  const RowsJob& J = gm.job[jb];
  const int loc = L - gm.start[jb], ncb = J.ncp / 4;
  int e, cb;
  if (J.entries < 16) {
    e = loc / ncb;
    cb = loc % ncb;
  } else {
    const int k = loc >> 3;
    e = 8 * (k / ncb) + (loc & 7);
    cb = k % ncb;
  }
  if (e >= J.entries) return;
  const int row0 = e * J.nrb * 16, nrows = min(J.nrb * 16, J.M - row0);
  const int nrb = (nrows + 15) / 16;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int steps = J.A / 2, nsplit = 4 * J.S;
  const int cp = cb * 4 + wave, I = J.A * 16;
  const u32x4_t rw = MakeRsrcWords(J.tiles + (size_t)cp * J.A * 2 * T, (uint32_t)steps * 16 * T);
  const u32x4_t rx = MakeRsrcWords(J.xp + (size_t)row0 * I, (uint32_t)nrows * I * 2);

  // always_inline: past the inliner's limit the body would become a called function (its
  // registers and LDS reached through a stack frame).
  auto main_loop = [&](auto nac) __attribute__((always_inline)) {
    constexpr int NA = decltype(nac)::value;
    float4_t acc[NA][2], sum[NA][2];  // the split's accumulators, the K segment's sum
#pragma unroll
    for (int i = 0; i < NA; ++i)
#pragma unroll
      for (int f = 0; f < 2; ++f) acc[i][f] = sum[i][f] = float4_t{0.f, 0.f, 0.f, 0.f};
    // The parked sums of the wave: 16 bytes per lane, fragment and row block.
    float4_t* park = reinterpret_cast<float4_t*>(J.part) + (((size_t)e * J.ncp + cp) * J.nrb * 2) * 64 + lane;
    int split = 0, next = steps / nsplit;  // first step of the next split
    // A segment's sum starts at +0 where the few-row path starts at its first split: the same
    // value, but for the sign of a zero that the last addition below (0 + ...) makes + in both.
    auto fold = [&]() __attribute__((always_inline)) {
      ++split;
      next = steps * (split + 1) / nsplit;
#pragma unroll
      for (int i = 0; i < NA; ++i)
#pragma unroll
        for (int f = 0; f < 2; ++f) {
          sum[i][f] += acc[i][f];
          acc[i][f] = float4_t{0.f, 0.f, 0.f, 0.f};
        }
      if ((split & 3) == 0 && split < nsplit) {  // the segment ends, another follows
        const bool first = split == 4;
#pragma unroll
        for (int i = 0; i < NA; ++i)
#pragma unroll
          for (int f = 0; f < 2; ++f) {
            float4_t* p = park + (i * 2 + f) * 64;
            const float4_t before = first ? float4_t{0.f, 0.f, 0.f, 0.f} : *p;
            *p = before + sum[i][f];
            sum[i][f] = float4_t{0.f, 0.f, 0.f, 0.f};
          }
      }
    };
    RowsLoop<K2, CB, NA, NRB, NXB>(rw, rx, I * 2, steps, smem, acc, [&](int s) __attribute__((always_inline)) {
      if (s + 1 == next) fold();  // uniform
    });
    // v = (0 + the segments before) + the last segment, then the output transform in the
    // rounding of OutputTransformKernel, 32 rows at a time through LDS.
#pragma unroll
    for (int i = 0; i < NA; ++i)
#pragma unroll
      for (int f = 0; f < 2; ++f) {
        const float4_t before = J.S > 1 ? park[(i * 2 + f) * 64] : float4_t{0.f, 0.f, 0.f, 0.f};
        sum[i][f] = before + sum[i][f];
      }
    __syncthreads();
    float(*eb)[132] = reinterpret_cast<float(*)[132]>(smem);
    const int cl = wave * 32 + ((lane & 15) >> 3) * 16 + (lane & 7);
    const int j16 = threadIdx.x & 15, c0 = cb * 128 + 8 * j16;
    float sv[8];
    LoadH8(J.svh + c0, sv);
    const float sg = WhtLaneSign();
    for (int i0 = 0; i0 < NA; i0 += 2) {
#pragma unroll
      for (int i = 0; i < NA; ++i) {
        if (i < i0 || i >= i0 + 2) continue;  // uniform
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          float* r = eb[16 * (i & 1) + 4 * (lane >> 4) + k];
          r[cl] = sum[i][0][k];
          r[cl + 8] = sum[i][1][k];
        }
      }
      __syncthreads();
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int rr = (int)(threadIdx.x >> 4) + 16 * h, r = 16 * i0 + rr;
        if (r < nrows) {  // uniform over the row's 16 lanes
          float v[8];
#pragma unroll
          for (int k = 0; k < 8; ++k) v[k] = eb[rr][8 * j16 + k];
          OutputTransformStore(v, sv, sg, J.f16, J.y, (size_t)(row0 + r) * J.ldy + c0);
        }
      }
      __syncthreads();
    }
  };
  using std::integral_constant;
  [&]<int... Is>(std::integer_sequence<int, Is...>) __attribute__((always_inline)) {
    (void)((nrb <= Is + 1 ? (main_loop(integral_constant<int, Is + 1>{}), true) : false) || ...);
  }(std::make_integer_sequence<int, NRB>{});
}

// Tall prefill GEMM for long entries of the MoE layer: a workgroup of 4 waves owns 128 columns (4
// column pairs) x up to 64 NRBW rows of one entry, full K, with the row loop above (each wave its
// column pair and all the rows), so every tile is decoded once per entry.  Two workgroups per CU
// (two activation chunks each: 160 KB of LDS at 8 bpw), so one's epilogue runs beside the other's loop.
//
// tall_seq_mid (gate/up): the workgroup runs the gate plane and parks its raw sums in plane 0's y,
// then runs the up plane over the same entry and columns and computes the mid in the epilogue
// (grid z = 1).
//
// 8,192 rows of 160 an expert, 3 / 5 bpw, settled clocks: gate/up with the mid 640 -> 547-566 us, down
// 397 -> 380-392 (the first launches after a pause, clocks unsettled: ~640 and ~450), against
// a form that passed the decoded fragments between the waves through LDS and loaded activation
// fragments straight from memory (16 bytes from each of 16 rows per load).  A gate/up workgroup's
// two loops take 88 us (0.69 us a step of two waves per SIMD: ~0.45 is the MFMAs' and the decode's
// issue), its epilogues 22; 2,220 workgroups leave the last of 4.3 rounds mostly empty (16%).
// Reading the windows before the rows or a step ahead, or leaving the order to the compiler,
// changed nothing.
template <int K2, int CB, int NRBW>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
Exl3GemmTallKernel(GemmArgs g) {
  constexpr int NRB = 4 * NRBW, NXB = 2;
  constexpr int T = TileDwords(K2);
  constexpr int ER = 32;  // rows of an epilogue slab
  __shared__ __align__(16) char smem[RowsLds<K2, NRB, NXB>::kBytes];
  static_assert(ER * 132 * 4 <= RowsLds<K2, NRB, NXB>::kBytes, "the epilogue slab reuses the loop's LDS");
  const int n_entries = g.n_entries ? *g.n_entries : g.n_entries_host;
  const GridPos gp = XcdEntryMajor();
  const int ei = gp.y + g.entry_base;
  if (ei >= n_entries) return;
  const int4 ent = EntryOf(g, ei);
  const bool seq = g.tall_seq_mid != 0;  // both planes in this workgroup, the mid fused
  const int cpg = gp.x;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int steps = g.A / 2;
  const int row0 = ent.y, nrows = ent.z;
  if (nrows <= 0) return;
  const int nrb = (nrows + 15) / 16;
  const int cp = cpg * 4 + wave, O = g.ncp * 32;
  const int j = threadIdx.x & 15, c0 = cpg * 128 + 8 * j;  // the thread's columns in the epilogue
  float(*eb)[132] = reinterpret_cast<float(*)[132]>(smem);

  // always_inline: past the inliner's limit the body would become a called function.
  auto main_loop = [&](auto nac) __attribute__((always_inline)) {
    constexpr int NA = decltype(nac)::value;
    for (int pz = seq ? 0 : gp.z;; ++pz) {  // one plane, or gate then up (seq)
      const GemmPlane& pl = g.plane[pz];
      const MatPtr m = MatOf(g, pl, ent.x);
      const u32x4_t rw = MakeRsrcWords(m.tiles + (size_t)cp * g.A * 2 * T, (uint32_t)steps * 16 * T);
      const u32x4_t rx = MakeRsrcWords(pl.x + (size_t)row0 * pl.ldx, (uint32_t)nrows * pl.ldx * 2);
      float4_t acc[NA][2];
#pragma unroll
      for (int i = 0; i < NA; ++i) acc[i][0] = acc[i][1] = float4_t{0.f, 0.f, 0.f, 0.f};
      RowsLoop<K2, CB, NA, NRB, NXB>(rw, rx, pl.ldx * 2, steps, smem, acc, [](int) {});
      __syncthreads();  // every wave is done with the loop's LDS: the slabs reuse it
      const bool mid = seq && pz == 1;
      float sv[8];
      if (pl.epi >= 1) LoadH8(m.svh + c0, sv);
      const MatPtr mg = mid ? MatOf(g, g.plane[0], ent.x) : m;
      const int cl = wave * 32 + ((lane & 15) >> 3) * 16 + (lane & 7);
      for (int i0 = 0; i0 < NA; i0 += 2) {  // slabs of 32 rows: two row blocks
        // The mid's gate sums are asked for before the slab is staged.
        float gv[2][8];
        if (mid) {
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const int r = min(16 * i0 + (int)(threadIdx.x >> 4) + 16 * h, nrows - 1);
            LoadF8(g.plane[0].y + (size_t)(row0 + r) * g.plane[0].ldy + c0, gv[h]);
          }
        }
#pragma unroll
        for (int i = 0; i < NA; ++i) {
          if (i < i0 || i >= i0 + 2) continue;  // uniform
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            float* r = eb[16 * (i & 1) + 4 * (lane >> 4) + k];
            r[cl] = acc[i][0][k];
            r[cl + 8] = acc[i][1][k];
          }
        }
        __syncthreads();
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int rr = (int)(threadIdx.x >> 4) + 16 * h, r = 16 * i0 + rr;
          if (r >= nrows) continue;  // uniform over the row's 16 lanes
          const size_t p = (size_t)(row0 + r);
          float v[8];
#pragma unroll
          for (int k = 0; k < 8; ++k) v[k] = eb[rr][8 * j + k];
          if (mid) {
            MidBlock(gv[h], v, mg.svh + c0, m.svh + c0, g.mid_suh + (size_t)ent.x * O + c0, g.mid_xd + p * O + cpg * 128);
          } else if (pl.epi >= 1) {
#pragma unroll
            for (int k = 0; k < 8; ++k) v[k] = 0.f + v[k];
            Wht128x8Signed(v);
#pragma unroll
            for (int k = 0; k < 8; ++k) v[k] *= WhtLaneSign() * (kHadNorm * sv[k]);
            StoreBlockRow(pl, p, c0, O, v);
          } else {
            StoreF8(pl.y + p * pl.ldy + c0, v);
          }
        }
        __syncthreads();
      }
      if (!seq || pz == 1) return;
    }
  };
  using std::integral_constant;
  [&]<int... Is>(std::integer_sequence<int, Is...>) __attribute__((always_inline)) {
    (void)((nrb <= Is + 1 ? (main_loop(integral_constant<int, Is + 1>{}), true) : false) || ...);
  }(std::make_integer_sequence<int, NRB>{});
}

}  // namespace cx
