// Dense NT GEMM main loop for gfx950: C[M,N] = alpha * A[M,K] . B[N,K]^T with
// both operands K-contiguous fp16 and fp32 accumulation on
// v_mfma_f32_32x32x16_f16.  This is the hot loop of the decode-first NF4
// projections (X . Wdec^T forward, dY . (Wdec^T)^T backward) and of the dense
// NT products; the epilogues (bias, LoRA add, rank-16 update, beta) are the
// ones of gemm.hip.
//
// Operand layouts, configurations and the epilogue: nt_core.h.
//
// Two main loops: NtStream (4 waves, 64-deep stages) and the ping-pong loop of eight
// waves with 32-deep stages, which stays ahead for short K (nt_plan) and where A lies
// K-major (the cross-entropy's dW, 151936 x 1536 x 576: 320 us against 336 us on 128x128
// stream tiles).
//
// The DMA is issued from inline asm.  The compiler does not know which LDS
// buffer an outstanding LDS DMA writes, and would wait for all of them
// (vmcnt(0)) before every LDS read, draining the pipeline; the waits are
// explicit instead.

#include "tuning.h"

#include "nt_core.h"

namespace ss {
namespace {

// Operand sources of one workgroup's tile (both main loops): per-lane DMA
// sources as 32-bit byte offsets from the per-stage operand base, and the
// per-stage advance of that base.  Rows past M / N (row-major operands) or
// chunks past M / N (K-major operands, L bits 0 / 1) are clamped to the last
// valid ones: they only feed accumulator rows / columns that are never stored.
template <class C, int L>
struct NtSources {
  static constexpr bool AT = (L & 1) != 0, BT = (L & 2) != 0;
  uint32_t a_off[C::kDmaA];
  uint32_t b_off[C::kDmaB];
  const half_t* a_base;
  const half_t* b_base;
  int64_t a_step, b_step;  // elements per stage

  __device__ __forceinline__ NtSources(const GemmParams& p, int64_t m0, int64_t n0, int64_t kbeg,
                                       int wave, int lane) {
    a_base = AT ? p.A + kbeg * p.lda : p.A + kbeg;
    b_base = BT ? p.B + kbeg * p.ldb : p.B + kbeg;
    a_step = AT ? (int64_t)C::BK * p.lda : C::BK;
    b_step = BT ? (int64_t)C::BK * p.ldb : C::BK;
#pragma unroll
    for (int j = 0; j < C::kDmaA; ++j) {
      int row, chunk;
      if constexpr (AT) {
        dma_source_t<C::BM>(wave * C::kDmaA + j, lane, row, chunk);
        const int64_t col = m0 + 8 * chunk <= p.M - 8 ? m0 + 8 * chunk : p.M - 8;
        a_off[j] = (uint32_t)((row * p.lda + col) * 2);
      } else {
        dma_source<C::BK>(wave * C::kDmaA + j, lane, row, chunk);
        const int64_t gr = m0 + row < p.M ? m0 + row : p.M - 1;
        a_off[j] = (uint32_t)((gr * p.lda + chunk * 8) * 2);
      }
    }
#pragma unroll
    for (int j = 0; j < C::kDmaB; ++j) {
      int row, chunk;
      if constexpr (BT) {
        dma_source_t<C::BN>(wave * C::kDmaB + j, lane, row, chunk);
        const int64_t col = n0 + 8 * chunk <= p.N - 8 ? n0 + 8 * chunk : p.N - 8;
        b_off[j] = (uint32_t)((row * p.ldb + col) * 2);
      } else {
        dma_source<C::BK>(wave * C::kDmaB + j, lane, row, chunk);
        const int64_t gr = n0 + row < p.N ? n0 + row : p.N - 1;
        b_off[j] = (uint32_t)((gr * p.ldb + chunk * 8) * 2);
      }
    }
  }
};

// Fragment offsets of one wave (both main loops): for a row-major operand the
// lane's offset per k-step plus the 32-row group stride; for a K-major one the
// offset of every (k-step, block) pair, read with read_frag_t.
template <class C, int L>
struct NtFrags {
  static constexpr bool AT = (L & 1) != 0, BT = (L & 2) != 0;
  static constexpr int kGroupBytes = 32 * C::BK * 2;
  int row_off[C::KK];
  int a_off[AT ? C::KK : 1][AT ? C::FM : 1];
  int b_off[BT ? C::KK : 1][BT ? C::FN : 1];
  int a_base, b_base;

  __device__ __forceinline__ NtFrags(int lane, int wm, int wn) {
#pragma unroll
    for (int kk = 0; kk < C::KK; ++kk) row_off[kk] = frag_offset<C::BK>(lane, kk);
    a_base = (wm * C::WM / 32) * kGroupBytes;
    b_base = C::kTileA + (wn * C::WN / 32) * kGroupBytes;
    if constexpr (AT) {
#pragma unroll
      for (int kk = 0; kk < C::KK; ++kk)
#pragma unroll
        for (int i = 0; i < C::FM; ++i)
          a_off[kk][i] = frag_offset_t<C::BM>(lane, kk, wm * C::WM + 32 * i);
    }
    if constexpr (BT) {
#pragma unroll
      for (int kk = 0; kk < C::KK; ++kk)
#pragma unroll
        for (int j = 0; j < C::FN; ++j)
          b_off[kk][j] = C::kTileA + frag_offset_t<C::BN>(lane, kk, wn * C::WN + 32 * j);
    }
  }
  __device__ __forceinline__ half8 a(const unsigned char* stage, int kk, int i) const {
    if constexpr (AT)
      return read_frag_t(stage + a_off[kk][i], C::BM * 2);
    else
      return *reinterpret_cast<const half8*>(stage + a_base + row_off[kk] + i * kGroupBytes);
  }
  __device__ __forceinline__ half8 b(const unsigned char* stage, int kk, int j) const {
    if constexpr (BT)
      return read_frag_t(stage + b_off[kk][j], C::BN * 2);
    else
      return *reinterpret_cast<const half8*>(stage + b_base + row_off[kk] + j * kGroupBytes);
  }
};

// Ping-pong main loop of the 8-wave configurations (two waves per SIMD:
// wave w and w + 4).  Run in lockstep, the two waves of a SIMD issue their
// MFMAs, LDS reads and barrier waits at the same time, and the MFMA pipe
// idles while both wait.  Here every wave runs the same body per stage kt,
//   read the fragments of stage kt, issue its DMAs of stage kt - 1 + STAGES,
//   wait for its DMAs of stage kt + 1, barrier, the 16 MFMAs of stage kt,
//   barrier,
// but waves 4-7 pass one extra barrier before the first stage and waves 0-3
// one after the last.  The barrier instances then pair each MFMA phase of
// one group with a read phase of the other: on every SIMD one wave computes
// while the other loads.  Stage kt's buffer is read by waves 0-3 in phase 2kt
// and by waves 4-7 in phase 2kt + 1, and refilled (stage kt + STAGES) in read
// phases from 2kt + 2 on; each wave's wait for its DMAs of stage kt + 1
// precedes a barrier that ends before either group reads that stage.  The
// MFMAs of every accumulator run in k order, as in NtStream: the same bits.
template <class C, int L = 0>
__device__ __forceinline__ void nt_mainloop_pp(const GemmParams& p, int64_t m0, int64_t n0,
                                               int64_t kbeg, int64_t klen, unsigned char* smem,
                                               NtAcc<C>& acc) {
  static_assert(C::kWaves == 8 && C::KK == 2, "ping-pong: 8 waves, two k-steps per stage");
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);  // uniform: scalar branches
  const int wm = wave / C::kWavesN;
  const int wn = wave % C::kWavesN;
  const bool late = wave >= 4;  // SIMD partner of wave - 4
  const uint32_t lds0 = lds_address(smem);
  const NtSources<C, L> src(p, m0, n0, kbeg, wave, lane);
  const uint32_t lds_a = __builtin_amdgcn_readfirstlane(lds0 + wave * C::kDmaA * 1024);
  const uint32_t lds_b = __builtin_amdgcn_readfirstlane(lds0 + C::kTileA + wave * C::kDmaB * 1024);
  const NtFrags<C, L> frags(lane, wm, wn);

  constexpr int kS = C::STAGES;
  const int64_t ktiles = klen / C::BK;
  auto issue_stage = [&](int64_t kt) {
    if (kt >= ktiles) return;
    const int stage = (int)(kt % kS);
#pragma unroll
    for (int j = 0; j < C::kDmaA; ++j)
      dma16(src.a_off[j], src.a_base + kt * src.a_step, lds_a + stage * C::kStageBytes + j * 1024);
#pragma unroll
    for (int j = 0; j < C::kDmaB; ++j)
      dma16(src.b_off[j], src.b_base + kt * src.b_step, lds_b + stage * C::kStageBytes + j * 1024);
  };
  auto barrier = [&]() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };

#pragma unroll
  for (int st = 0; st < kS; ++st) issue_stage(st);
  if (ktiles <= 0) return;
  wait_stages<C::kDma, kS - 1>((ktiles < kS ? ktiles : kS) - 1);
  barrier();  // stage 0 is in LDS
  if (late) barrier();
  for (int64_t kt = 0; kt < ktiles; ++kt) {
    half8 fa[2][C::FM], fb[2][C::FN];
    const unsigned char* base = smem + (kt % kS) * C::kStageBytes;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
      for (int i = 0; i < C::FM; ++i) fa[kk][i] = frags.a(base, kk, i);
#pragma unroll
      for (int j = 0; j < C::FN; ++j) fb[kk][j] = frags.b(base, kk, j);
    }
    if (kt >= 1) issue_stage(kt - 1 + kS);
    {
      // Stages this wave has issued: up to min(kt + kS - 1, ktiles - 1);
      // stage kt + 1 must have landed.
      const int64_t last = kt + kS - 1 < ktiles - 1 ? kt + kS - 1 : ktiles - 1;
      wait_stages<C::kDma, kS - 2>(last - (kt + 1));
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the fragments are in
    barrier();
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int i = 0; i < C::FM; ++i)
#pragma unroll
        for (int j = 0; j < C::FN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[kk][i], fb[kk][j], acc[i][j], 0,
                                                             0, 0);
    __builtin_amdgcn_s_setprio(0);
    barrier();
  }
  if (!late) barrier();
}

// Main loop of the 4-wave configurations with 64-deep stages (BK = 64): the DMAs fetch
// 128-byte row pieces (64-byte pieces, as the 32-deep stages have, reach 25 B/clk/CU into
// LDS; 256x128 tiles need 48), and the loop overlaps within a wave, not between waves:
// every memory instruction has a slot between two MFMAs, spread evenly (bursts stall:
// 16384 x 18944 x 3584 in 1771 us against 1803 us with the eight DMAs of a half stage
// back to back, 1840 us with fourteen).  Per stage kt of four k-steps,
//   k-steps 0 .. 2: the fragments of the next k-step;
//   k-step 3: after kB MFMAs the wait for stage kt + 1 and the barrier, then the
//   fragments of its k-step 0.
// Stage kt's buffer was last read in k-step 2 (fragments of k-step 3), before the
// barrier of k-step 3; the DMAs of stage kt + STAGES into it start after that barrier
// and end before the next one.  Every accumulator adds its products in k order.
template <class C, int L>
struct NtStream {
  static constexpr int kS = C::STAGES, kMf = C::FM * C::FN, kFr = C::FM + C::FN;
  static constexpr int kB = kMf >= 8 ? 2 : kMf >= 2 ? 1 : 0;  // MFMAs of the last k-step before its barrier
  static constexpr int kPart = kMf - kB;       // slots after it, in that k-step
  // DMA d of a stage goes to slot at(d), counted from the barrier: spread over about
  // half a stage when the next barrier waits for it (two buffers), else a whole one.
  static constexpr int kSpan = kS == 2 ? 2 * kMf : 4 * kMf - (kMf >= 2 ? 2 : 0);
  static constexpr int at(int d) { return (2 * d + 1) * kSpan / (2 * C::kDma); }
  static constexpr int first_of(int slot) {  // DMAs before this slot
    int n = 0;
    while (n < C::kDma && at(n) < slot) ++n;
    return n;
  }
  static constexpr int kEarly = first_of(kPart);  // DMAs issued within the barrier's k-step
  static_assert(C::KK == 4 && (kS == 2 || kS == 3) && kSpan <= 4 * kMf, "stages");
  const NtSources<C, L> src;
  const NtFrags<C, L> frags;
  const unsigned char* smem;
  uint32_t lds_a, lds_b;

  __device__ __forceinline__ NtStream(const GemmParams& p, int64_t m0, int64_t n0, int64_t kbeg,
                                      unsigned char* lds, int wave, int lane)
      : src(p, m0, n0, kbeg, wave, lane),
        frags(lane, wave / C::kWavesN, wave % C::kWavesN),
        smem(lds) {
    const uint32_t lds0 = lds_address(lds);
    lds_a = __builtin_amdgcn_readfirstlane(lds0 + wave * C::kDmaA * 1024);
    lds_b = __builtin_amdgcn_readfirstlane(lds0 + C::kTileA + wave * C::kDmaB * 1024);
  }
  // buf: the stage's buffer.
  __device__ __forceinline__ void dma(int64_t kt, int buf, int idx) const {
    if (idx < C::kDmaA)
      dma16(src.a_off[idx], src.a_base + kt * src.a_step, lds_a + buf * C::kStageBytes + idx * 1024);
    else
      dma16(src.b_off[idx - C::kDmaA], src.b_base + kt * src.b_step,
            lds_b + buf * C::kStageBytes + (idx - C::kDmaA) * 1024);
  }
  __device__ __forceinline__ half8 frag(int buf, int kk, int f) const {
    const unsigned char* base = smem + buf * C::kStageBytes;
    return f < C::FN ? frags.b(base, kk, f) : frags.a(base, kk, f - C::FN);
  }
  static __device__ __forceinline__ int next_buf(int buf) { return buf + 1 == kS ? 0 : buf + 1; }
  // Fragment read r of a k-step, in the order the MFMAs need them (B fragments and the
  // first A fragment for the first row of blocks, then a row's A fragment each).
  static constexpr int order(int r) { return r == 0 ? 0 : r == 1 ? C::FN : r <= C::FN ? r - 1 : r; }

  // AHEAD: stages in flight beyond kt + 1 at its wait; REFILL / CONT: stage kt + kS (its
  // first DMAs) / kt + kS - 1 (its other ones) exists; MORE: stage kt + 1 does.
  template <int AHEAD, bool REFILL, bool CONT, bool MORE>
  __device__ __forceinline__ void stage(int64_t kt, int buf, half8 (&f)[2][kFr],
                                        NtAcc<C>& acc) const {
    const int after = next_buf(buf);
    const int before = buf == 0 ? kS - 1 : buf - 1;  // buffer of stages kt - 1 and kt + kS - 1
#pragma unroll
    for (int kk = 0; kk < C::KK; ++kk) {
#pragma unroll
      for (int s = 0; s < kMf; ++s) {
        half8(&now)[kFr] = f[kk & 1];
        half8(&next)[kFr] = f[(kk + 1) & 1];
        const bool last = kk == C::KK - 1;
        if (MORE && last && s == kB) {
          wait_vm<AHEAD * C::kDma>();
          __builtin_amdgcn_s_waitcnt(0xC07F);
          asm volatile("s_barrier" ::: "memory");
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int r = 0; r < kFr; ++r) {
          if (!last && s == r * kMf / kFr) next[order(r)] = frag(buf, kk + 1, order(r));
          if (MORE && last && s == kB + r * kPart / kFr) next[order(r)] = frag(after, 0, order(r));
        }
        const int slot = last ? s - kB : kPart + kk * kMf + s;  // from the barrier
#pragma unroll
        for (int d = 0; d < C::kDma; ++d) {
          if (at(d) != slot) continue;
          if (last && s >= kB) {
            if (REFILL) dma(kt + kS, buf, d);
          } else if (!last) {
            if (CONT) dma(kt + kS - 1, before, d);
          }
        }
        const int i = s / C::FN, j = s % C::FN;
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(now[C::FN + i], now[j], acc[i][j], 0,
                                                           0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  __device__ __forceinline__ void run(int64_t ktiles, NtAcc<C>& acc) const {
    if (ktiles <= 0) return;
#pragma unroll
    for (int st = 0; st < kS - 1; ++st)
      if (st < ktiles)
#pragma unroll
        for (int idx = 0; idx < C::kDma; ++idx) dma(st, st, idx);
    if (ktiles >= kS) {
#pragma unroll
      for (int idx = 0; idx < kEarly; ++idx) dma(kS - 1, kS - 1, idx);
      wait_vm<(kS - 2) * C::kDma + kEarly>();
    } else {
      wait_vm<0>();
    }
    asm volatile("s_barrier" ::: "memory");
    half8 f[2][kFr];
#pragma unroll
    for (int i = 0; i < kFr; ++i) f[0][order(i)] = frag(0, 0, order(i));
    __builtin_amdgcn_sched_barrier(0);
    int64_t kt = 0;
    int buf = 0;
    for (; kt < ktiles - kS; ++kt, buf = next_buf(buf))
      stage<kS - 2, true, true, true>(kt, buf, f, acc);
    if (kt == ktiles - kS) {
      stage<kS - 2, false, true, true>(kt++, buf, f, acc);
      buf = next_buf(buf);
    }
    if (kS == 3 && kt == ktiles - 2) {
      stage<0, false, false, true>(kt++, buf, f, acc);
      buf = next_buf(buf);
    }
    stage<0, false, false, false>(kt, buf, f, acc);
  }
};

// LDS of a GEMM workgroup: the stage ring; for the dX epilogue (rank-16
// update) also room for a rank-16 grad tail block.
template <class C, int EPI>
constexpr int nt_smem_bytes() {
  constexpr int ring = C::STAGES * C::kStageBytes;
  return EPI == EPI_RANK && kRankGradSmem > ring ? kRankGradSmem : ring;
}

// Data-parallel / split-K kernel: workgroup = one output tile (blockIdx.x,
// XCD-remapped) or, split over K, one (tile, split) pair (split_tile;
// EPI_PARTIAL stores its fp32 accumulator to split plane `split`).  Workgroups past the tiles run the
// optional rank-16 grad tail (p.tail; rank-16 epilogue, unsplit launches)
// after the GEMM tiles, filling CUs the GEMM leaves idle.
template <class C, int CT, int EPI, int L = 0>
__global__ __launch_bounds__(C::kThreads, C::MINW) void gemm_nt_kernel(GemmParams p) {
  __shared__ __attribute__((aligned(1024))) unsigned char smem[nt_smem_bytes<C, EPI>()];
  if (EPI == EPI_PLAIN && p.alpha_dev) p.alpha *= *p.alpha_dev;
  const int64_t tiles = gridDim.x - p.tail_blocks - p.tail2_blocks;
  if constexpr (EPI == EPI_RANK) {
    if ((int64_t)blockIdx.x >= tiles) {
      run_tail_block(p, blockIdx.x - tiles, smem);
      return;
    }
  }
  int64_t tile, split = 0;
  if constexpr (EPI == EPI_PARTIAL)
    split_tile(p.remap, tiles, tile, split);
  else
    tile = p.remap ? xcd_remap(blockIdx.x, tiles) : (int64_t)blockIdx.x;
  int64_t m0, n0;
  tile_origin<C>(p, tile, m0, n0);
  int64_t kbeg = 0, klen = p.K;
  if constexpr (EPI == EPI_PARTIAL) {
    kbeg = split * p.k_split;
    klen = p.K - kbeg < p.k_split ? p.K - kbeg : p.k_split;
  }
  NtAcc<C> acc;
#pragma unroll
  for (int i = 0; i < C::FM; ++i)
#pragma unroll
    for (int j = 0; j < C::FN; ++j) acc[i][j] = float16v{};
  if constexpr (C::kWaves == 4 && C::BK == 64) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    NtStream<C, L>(p, m0, n0, kbeg, smem, wave, threadIdx.x & (kWave - 1))
        .run(klen / C::BK, acc);
  } else {
    nt_mainloop_pp<C, L>(p, m0, n0, kbeg, klen, smem, acc);
  }
  nt_epilogue<C, CT, EPI, sizeof(smem)>(p, m0, n0, acc, smem, split);
}

// Split-K reduction: out[row][col] = epilogue(sum over splits s = 0.. of
// part[s][row][col]), four columns per thread.  The epilogues are those of the
// GEMM kernel with the same rounding order; the rank-16 terms are summed in
// fp32 in rank order.
// TAIL: the first p.tail_blocks + p.tail2_blocks workgroups run the rank-16
// grads p.tail / p.tail2 (run_tail_block, vector loads) instead, overlapping
// the reduce: used for split-K dX products, whose dA and dB would otherwise
// need launches of their own.
template <int CT, int EPI, bool TAIL = false>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(GemmParams p, int splits) {
  if (EPI == EPI_PLAIN && p.alpha_dev) p.alpha *= *p.alpha_dev;
  int64_t block = blockIdx.x;
  if constexpr (TAIL) {
    __shared__ __attribute__((aligned(16))) unsigned char smem[kRankGradSmem];
    if (block < p.tail_blocks + p.tail2_blocks) {
      run_tail_block(p, block, smem);
      return;
    }
    block -= p.tail_blocks + p.tail2_blocks;
  }
  const int64_t groups = cdiv(p.N, 4);
  const int64_t g = block * 256 + threadIdx.x;
  if (g >= p.M * groups) return;
  const int64_t row = g / groups;
  const int64_t c0 = (g % groups) * 4;
  const int64_t plane = p.M * p.N;
  // Every load of the thread -- the epilogue's operands (Z row, lora_B rows or
  // lora_A columns, bias, gate / up) and then up to eight partials -- is
  // issued before the first add, so the thread waits for memory once.
  // Rank-16 operands use 16-byte (Z, lora_B rows) and 8-byte (four lora_A
  // columns) loads where aligned.
  half8 z8[2];
  if (EPI == EPI_RANK || (EPI == EPI_LORA && !p.lora_plane)) {
    const half_t* zr = p.lz + row * 16;
    if (reinterpret_cast<uintptr_t>(p.lz) % 16 == 0) {
      z8[0] = *reinterpret_cast<const half8*>(zr);
      z8[1] = *reinterpret_cast<const half8*>(zr + 8);
    } else {
#pragma unroll
      for (int r = 0; r < 16; ++r) z8[r / 8][r % 8] = zr[r];
    }
  }
  half4 a4[16];  // EPI_RANK: lora_A[r][c0 .. c0 + 3]
  if constexpr (EPI == EPI_RANK) {
    if (c0 + 4 <= p.N && p.ldlb % 4 == 0 && reinterpret_cast<uintptr_t>(p.lb) % 8 == 0) {
#pragma unroll
      for (int r = 0; r < 16; ++r) a4[r] = *reinterpret_cast<const half4*>(p.lb + r * p.ldlb + c0);
    } else {
#pragma unroll
      for (int r = 0; r < 16; ++r)
#pragma unroll
        for (int e = 0; e < 4; ++e) a4[r][e] = c0 + e < p.N ? p.lb[r * p.ldlb + c0 + e] : (half_t)0;
    }
  }
  half8 b8[4][2];  // EPI_LORA: lora_B rows of the four columns (no lora_plane)
  half_t lp[4];    // EPI_LORA: the rounded LoRA terms (lora_plane)
  if constexpr (EPI == EPI_LORA) {
    if (p.lora_plane) {
      const half_t* src = p.lora_plane + row * p.N + c0;
      if (p.N % 4 == 0) {
        const half4 v4 = *reinterpret_cast<const half4*>(src);
#pragma unroll
        for (int e = 0; e < 4; ++e) lp[e] = v4[e];
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) lp[e] = c0 + e < p.N ? src[e] : (half_t)0;
      }
    }
#pragma unroll
    for (int e = 0; e < 4 && !p.lora_plane; ++e) {
      const int64_t col = c0 + e < p.N ? c0 + e : p.N - 1;
      const half_t* br = p.lb + col * 16;
      if (reinterpret_cast<uintptr_t>(p.lb) % 16 == 0) {
        b8[e][0] = *reinterpret_cast<const half8*>(br);
        b8[e][1] = *reinterpret_cast<const half8*>(br + 8);
      } else {
#pragma unroll
        for (int r = 0; r < 16; ++r) b8[e][r / 8][r % 8] = br[r];
      }
    }
  }
  float bias[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) bias[e] = p.bias && c0 + e < p.N ? (float)p.bias[c0 + e] : 0.0f;
  half_t gg[4], uu[4];  // EPI_GLU: gate / up of the four columns, loaded before any store
  if constexpr (EPI == EPI_GLU) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const bool in = c0 + e < p.N;
      gg[e] = in ? p.glu_gate[row * p.ldgate + c0 + e] : (half_t)0;
      uu[e] = in && p.glu == 2 ? p.glu_up[row * p.ldup + c0 + e] : (half_t)0;
    }
  }
  // Sum of the splits in split order.
  float v[4] = {0.f, 0.f, 0.f, 0.f};
  if (p.N % 4 == 0) {
    constexpr int kAhead = 8;
    float4v t[kAhead];
#pragma unroll
    for (int s = 0; s < kAhead; ++s)
      if (s < splits) t[s] = *reinterpret_cast<const float4v*>(p.part + s * plane + row * p.N + c0);
#pragma unroll
    for (int s = 0; s < kAhead; ++s)
      if (s < splits)
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] += t[s][e];
    for (int s = kAhead; s < splits; ++s) {
      const float4v u = *reinterpret_cast<const float4v*>(p.part + s * plane + row * p.N + c0);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += u[e];
    }
  } else {
    for (int s = 0; s < splits; ++s)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (c0 + e < p.N) v[e] += p.part[s * plane + row * p.N + c0 + e];
  }
  float z[16];
  if constexpr (EPI == EPI_LORA || EPI == EPI_RANK) {
#pragma unroll
    for (int r = 0; r < 16; ++r) z[r] = (float)z8[r / 8][r % 8];
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int64_t col = c0 + e;
    if (col >= p.N) break;
    const int64_t idx = row * p.ldc + col;
    if constexpr (EPI == EPI_LORA) {
      const float y = (float)f32_to_f16(v[e] * p.alpha + bias[e]);
      float scaled;
      if (p.lora_plane) {
        scaled = (float)lp[e];
      } else {
        float l = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; ++r) l += z[r] * (float)b8[e][r / 8][r % 8];
        scaled = (float)f32_to_f16((float)f32_to_f16(l) * p.lscale);
      }
      reinterpret_cast<half_t*>(p.C)[idx] = f32_to_f16(y + scaled);
    } else if constexpr (EPI == EPI_RANK) {
      float l = 0.0f;
#pragma unroll
      for (int r = 0; r < 16; ++r) l += z[r] * (float)a4[r][e];
      store_c<CT>(p.C, idx, v[e] + l, p.beta);
    } else {
      if constexpr (EPI == EPI_GLU)
        glu_apply(p, row, col, idx, v[e] * p.alpha + bias[e], gg[e], uu[e]);
      else
        store_c<CT>(p.C, idx, v[e] * p.alpha + bias[e], p.beta);
    }
  }
}

// The rank-16 grad tails on their own.
__global__ __launch_bounds__(256) void rank_tail_kernel(GemmParams p) {
  __shared__ __attribute__((aligned(16))) unsigned char smem[kRankGradSmem];
  run_tail_block(p, blockIdx.x, smem);
}

// Tile configurations: <BM, BN, waves M, waves N, BK, stages, min waves/SIMD>.
using Nt64 = NtCfg<64, 64, 2, 2, 64, 3, 2>;         // 1: 4 waves of 32x32, 48 KiB LDS
using Nt128x64 = NtCfg<128, 64, 2, 2, 64, 3, 2>;    // 2: 64x32, 72 KiB
using Nt128 = NtCfg<128, 128, 2, 2, 64, 3, 1>;      // 3: 64x64, 96 KiB
using Nt128x256 = NtCfg<128, 256, 2, 2, 64, 3, 1>;  // 4: 64x128, 144 KiB
using Nt256x160 = NtCfg<256, 160, 4, 1, 64, 3, 1>;  // 5: 64x160, 156 KiB
using Nt256x192 = NtCfg<256, 192, 2, 2, 64, 2, 1>;  // 6: 128x96, 112 KiB
using Nt256 = NtCfg<256, 256, 2, 2, 64, 2, 1>;      // 7: 128x128, 128 KiB
using NtPingPong = NtCfg<256, 256, 2, 4, 32, 4, 2>; // 8: 8 waves of 128x64, 128 KiB

template <class C, int CT, int EPI, int L = 0>
int launch_nt(const GemmParams& p, int64_t splits, hipStream_t stream) {
  const dim3 grid((unsigned)(cdiv(p.M, C::BM) * cdiv(p.N, C::BN) + p.tail_blocks +
                             p.tail2_blocks),
                  (unsigned)splits);
  hipLaunchKernelGGL((gemm_nt_kernel<C, CT, EPI, L>), grid, dim3(C::kThreads), 0, stream, p);
  SS_CHECK_LAUNCH("gemm_nt_kernel");
  if (EPI == EPI_GLU && p.glu_done) *p.glu_done = 1;
  return SS_OK;
}

// K-major operands (L != 0): configurations 1, 3, 4 and 8 (nt_plan's mask).
template <int CT, int EPI, int L>
int dispatch_nt_t(const GemmParams& p, int cfg, int64_t splits, hipStream_t stream) {
  switch (cfg) {
    case 1: return launch_nt<Nt64, CT, EPI, L>(p, splits, stream);
    case 3: return launch_nt<Nt128, CT, EPI, L>(p, splits, stream);
    case 4: return launch_nt<Nt128x256, CT, EPI, L>(p, splits, stream);
    case 8: return launch_nt<NtPingPong, CT, EPI, L>(p, splits, stream);
    default: return SS_ERR_UNSUPPORTED;
  }
}

template <int CT, int EPI>
int dispatch_nt(const GemmParams& p, int cfg, int64_t splits, hipStream_t stream) {
  const int layout = (p.a_t ? 1 : 0) | (p.b_t ? 2 : 0);
  if constexpr (EPI == EPI_PLAIN || EPI == EPI_PARTIAL) {
    if (layout == 1) return dispatch_nt_t<CT, EPI, 1>(p, cfg, splits, stream);
    if (layout == 2) return dispatch_nt_t<CT, EPI, 2>(p, cfg, splits, stream);
    if (layout == 3) return dispatch_nt_t<CT, EPI, 3>(p, cfg, splits, stream);
  } else {
    if (layout) return SS_ERR_UNSUPPORTED;
  }
  if constexpr (EPI == EPI_GLU) {
    switch (cfg) {
      case 1: return launch_nt<Nt64, CT, EPI>(p, splits, stream);
      case 2: return launch_nt<Nt128x64, CT, EPI>(p, splits, stream);
      case 3: return launch_nt<Nt128, CT, EPI>(p, splits, stream);
      case 8: return launch_nt<NtPingPong, CT, EPI>(p, splits, stream);
      default: return SS_ERR_UNSUPPORTED;
    }
  } else switch (cfg) {
    case 1: return launch_nt<Nt64, CT, EPI>(p, splits, stream);
    case 2: return launch_nt<Nt128x64, CT, EPI>(p, splits, stream);
    case 3: return launch_nt<Nt128, CT, EPI>(p, splits, stream);
    case 4: return launch_nt<Nt128x256, CT, EPI>(p, splits, stream);
    case 5: return launch_nt<Nt256x160, CT, EPI>(p, splits, stream);
    case 6: return launch_nt<Nt256x192, CT, EPI>(p, splits, stream);
    case 7: return launch_nt<Nt256, CT, EPI>(p, splits, stream);
    case 8:
      if constexpr (EPI != EPI_PARTIAL) return launch_nt<NtPingPong, CT, EPI>(p, splits, stream);
    default: return SS_ERR_UNSUPPORTED;
  }
}

template <int CT, int EPI, bool TAIL = false>
int reduce_nt(const GemmParams& p, int64_t splits, hipStream_t stream) {
  const int64_t threads = p.M * cdiv(p.N, 4);
  const int64_t blocks = cdiv(threads, 256) + (TAIL ? p.tail_blocks + p.tail2_blocks : 0);
  hipLaunchKernelGGL((splitk_reduce_kernel<CT, EPI, TAIL>), dim3((unsigned)blocks), dim3(256), 0,
                     stream, p, (int)splits);
  SS_CHECK_LAUNCH("splitk_reduce_kernel");
  if (EPI == EPI_GLU && p.glu_done) *p.glu_done = 1;
  return SS_OK;
}

bool aligned16(const void* ptr) { return reinterpret_cast<uintptr_t>(ptr) % 16 == 0; }

}  // namespace

// Split-K scratch: the fp32 partial planes, then (256-byte aligned) the fp16
// LoRA plane of a split LoRA forward.
static size_t nt_plane_offset(int64_t m, int64_t n, int64_t splits) {
  return ((size_t)(splits * m * n) * sizeof(float) + 255) / 256 * 256;
}
static size_t nt_split_bytes(int64_t m, int64_t n, int64_t splits) {
  return nt_plane_offset(m, n, splits) + (size_t)(m * n) * sizeof(half_t);
}

// Configuration and split-K plan for an M x N x K product: the cheapest by a cost model
// of the time a launch takes,
//   start + q tile + stages (q stage + ceil(q / 2) pair + w load),
//   w = workgroups / CUs, q = ceil(w),
// with a configuration's start, epilogue and 64-deep stage times in us (load: the part that
// grows with the busy share of the chip, clock and caches; pair: the part that two
// workgroups on a CU overlap), plus a split's reduce.  A long K (8192 or more walked by more
// than one workgroup per CU in turn; 3584 on 64-column tiles) adds `drift` to a stage: the
// workgroups fall out of step along K and share less of the caches (16384 x 3584 x 18944 on
// 256x192 tiles 2097 us, 1923 on 128x256).  K is split only where the tiles leave CUs idle.
// The constants are least-squares fits to 4500 products of these kernels measured on
// MI355X (M 260 .. 16384, N 256 .. 18944, K 64 .. 18944, every configuration, and up to 8
// splits of the long K); the model's choice takes 1.005 times the best measured one on
// average, 1.03 at the 95th percentile.  Against the kernels before the 64-deep stages
// (thresholds on the tile count), us before -> now: 990 x 1536 x 1536 16.5 -> 10.5, 990 x 8960 x
// 1536 37 -> 31, 990 x 1536 x 8960 45 -> 42, 2048 x 3584 x 3584 63 -> 50, 16384 x 18944 x 3584
// 1898 -> 1771.  The ping-pong tile stays ahead for short K, where it fills the chip: 3500
// x 3584 x 512 19.4 us (128x256 stream tiles 22.4), 2700 x 4864 x 896 29.3 (31.4), 1350 x 8960 x
// 1536 43.3 (44.8), 16384 x 8960 x 256 116 (131).
struct TileCost {
  int cfg, bm, bn;
  float start, tile, stage, pair, load, drift;
};
constexpr TileCost kTileCosts[] = {
    {1, 64, 64, 3.47f, 0.44f, 0.037f, 0.139f, 0.055f, 0.023f},
    {2, 128, 64, 3.47f, 0.99f, 0.225f, 0.0f, 0.043f, 0.032f},
    {3, 128, 128, 2.68f, 2.79f, 0.279f, 0.0f, 0.165f, 0.047f},
    {4, 128, 256, 2.52f, 4.85f, 0.451f, 0.0f, 0.338f, 0.069f},
    {5, 256, 160, 2.71f, 6.18f, 0.534f, 0.0f, 0.407f, 0.088f},
    {6, 256, 192, 2.23f, 6.85f, 0.712f, 0.0f, 0.404f, 0.184f},
    {7, 256, 256, 2.53f, 11.76f, 0.848f, 0.0f, 0.575f, 0.130f},
    {8, 256, 256, 1.69f, 6.70f, 0.846f, 0.0f, 0.738f, 0.222f},
};

// layout: bit 0 / 1 for K-major A / B (GemmParams::a_t, b_t).  scratch: what the planes of
// a split may take; without room for them the tile is the best one for an unsplit product
// (990 x 1536 x 8960: 45 us on 128x64 tiles, 77 us on the 128x256 tiles of the 5-way split).
NtPlan nt_plan(int64_t m, int64_t n, int64_t k, int layout, size_t scratch) {
  const int64_t cus = device_cu_count();
  NtPlan plan{1, 1, k};
  if ((layout & 1) && cdiv(m, 256) * cdiv(n, 256) >= cus / 2) {
    plan.cfg = 8;
    return plan;
  }
  // Splits: at least 512 deep; more than 8 only where each still has 4096.
  int64_t most = k / 512 < 8 ? k / 512 : (k / 4096 > 8 ? k / 4096 : 8);
  if (most > 64) most = 64;
  if (most < 1) most = 1;
  float best = 0.0f;
  for (const TileCost& c : kTileCosts) {
    // K-major operands: the tiles of dispatch_nt_t, of them the ping-pong one where only B is
    // K-major (the cross-entropy's dX over the vocabulary, 1500 x 1536 x 151936: 605 us in 7
    // splits, 684 on 128x256 tiles; 3000 x 3584 x 151936 2761 and 3142), and not the 64-column
    // one over a long K, whose short rows stream at half the rate (64 x 1536 x 151936: 139 us,
    // 98 on 128x128 tiles in 21 splits).
    if (layout && c.cfg != 1 && c.cfg != 3 && c.cfg != 4 && !(c.cfg == 8 && layout == 2)) continue;
    if (layout && c.cfg == 1 && k >= 16384) continue;
    const int64_t tiles = cdiv(m, c.bm) * cdiv(n, c.bn);
    const int64_t splits = tiles > cus || (c.cfg == 8 && layout != 2) ? 1 : most;
    for (int64_t s = 1; s <= splits; ++s) {
      const int64_t k_split = cdiv(cdiv(k, s), 64) * 64;
      if (cdiv(k, k_split) != s) continue;
      if (s > 1 && nt_split_bytes(m, n, s) > scratch) break;
      const float w = (float)(tiles * s) / (float)cus;
      const int64_t turns = cdiv(tiles * s, cus);
      const float q = (float)turns, pairs = (float)cdiv(turns, 2);
      const bool drifts = c.bn == 64 ? k >= 3584 : k >= 8192 && turns > 1;
      float stage = c.stage + (drifts ? c.drift : 0.0f);
      // (a long K of K-major operands slows the narrower tiles: 1500 x 896 x 151936 509 us on
      // 128x128 tiles in 3 splits, 408 on 256x256 ones in 10; 2048 x 3584 x 151936 2038 us on
      // 128x256 tiles, 1884 on 256x256 ones in 2)
      if (layout && k >= 16384) stage += c.cfg == 3 ? 0.10f : c.cfg == 4 ? 0.06f : 0.0f;
      const float stages = (float)(k_split / 64);
      float us = c.start + q * c.tile + stages * (q * stage + pairs * c.pair + c.load * w);
      // (a split has to win by 3 %: ties go to the plan without planes)
      if (s > 1) us = 1.03f * (us + 4.6f + (float)s * 1.05f * (float)m * (float)n * 1e-6f);
      if (best == 0.0f || us < best) {
        best = us;
        plan = NtPlan{c.cfg, s, k_split};
      }
    }
  }
  if (plan.splits == 1) plan.k_split = k;
  return plan;
}

int splitk_reduce(const GemmParams& p, int splits, int ct, int epi, hipStream_t stream) {
  if (ct == SS_F32) {
    if (epi != EPI_PLAIN) return SS_ERR_UNSUPPORTED;
    return reduce_nt<SS_F32, EPI_PLAIN>(p, splits, stream);
  }
  if (epi == EPI_LORA) return reduce_nt<SS_F16, EPI_LORA>(p, splits, stream);
  if (epi == EPI_RANK) return reduce_nt<SS_F16, EPI_RANK>(p, splits, stream);
  if (p.glu) return reduce_nt<SS_F16, EPI_GLU>(p, splits, stream);
  return reduce_nt<SS_F16, EPI_PLAIN>(p, splits, stream);
}

size_t nt_partial_bytes(int64_t m, int64_t n, int64_t k, int layout) {
  if (m <= 0 || n <= 0 || k <= 0 || k % 64 != 0) return 0;
  const NtPlan plan = nt_plan(m, n, k, layout);
  return plan.splits > 1 ? nt_split_bytes(m, n, plan.splits) : 0;
}

// SS_TUNE_NT_STAGED = 0 keeps fp16 epilogues on direct 2-byte stores.
bool staged_epilogue_enabled() { return SS_TUNE_NT_STAGED != 0; }

int gemm_nt(const GemmParams& p0, int ct, int epi, hipStream_t stream, void* partials,
            size_t partial_bytes) {
  GemmParams p = p0;
  p.c_vec = staged_epilogue_enabled() && ct == SS_F16 && !p.beta && p.N % 8 == 0 &&
            p.ldc % 8 == 0 && aligned16(p.C);
  if (p.M <= 0 || p.N <= 0 || p.K <= 0 || p.K % 64 != 0) return SS_ERR_UNSUPPORTED;  // K % 64
  if (!aligned16(p.A) || !aligned16(p.B) || p.lda % 8 != 0 || p.ldb % 8 != 0)
    return SS_ERR_UNSUPPORTED;
  // K-major operands: whole 16-byte chunks along M / N, plain or split-K
  // epilogues only.
  if ((p.a_t && p.M % 8 != 0) || (p.b_t && p.N % 8 != 0)) return SS_ERR_UNSUPPORTED;
  if ((p.a_t || p.b_t) && (epi != EPI_PLAIN || p.glu)) return SS_ERR_UNSUPPORTED;
  // The DMA addresses operands with 32-bit byte offsets from their base (per
  // stage for K-major operands, whose base moves BK rows a stage).
  const int64_t kMaxOff = (int64_t)1 << 32;
  const int64_t a_span = p.a_t ? 64 * p.lda + p.M : (p.M - 1) * p.lda + p.K;
  const int64_t b_span = p.b_t ? 64 * p.ldb + p.N : (p.N - 1) * p.ldb + p.K;
  if (a_span * 2 >= kMaxOff || b_span * 2 >= kMaxOff) return SS_ERR_UNSUPPORTED;
  if (epi != EPI_PLAIN && (!aligned16(p.lz) || (epi == EPI_LORA && !aligned16(p.lb))))
    return SS_ERR_UNSUPPORTED;
  if (ct != SS_F16 && epi != EPI_PLAIN) return SS_ERR_UNSUPPORTED;
  const NtPlan plan = nt_plan(p.M, p.N, p.K, (p.a_t ? 1 : 0) | (p.b_t ? 2 : 0),
                              partials && aligned16(partials) ? partial_bytes : 0);
  // The rank-16 grad tail rides on unsplit dX products (rank-16 epilogue) after the GEMM
  // tiles where the tile's LDS lets two or more workgroups share a CU (64 columns: it
  // fills CUs that the GEMM leaves idle; q / o / k / v backward 6-11 us faster).  Behind
  // the larger tiles, one workgroup per CU, it gets a launch of its own (990 x 8960 x 1536
  // with 656 tail blocks: 50 us together, 34 + 7 us apart).  On the split-K launches of
  // the long-K dX it slowed the GEMM more than a launch costs; there it leads the reduce.
  if (epi != EPI_RANK) p.tail_blocks = p.tail2_blocks = 0;
  if (p.tail_blocks + p.tail2_blocks > 0 && p.tail_ran) *p.tail_ran = 1;
  if (plan.splits > 1) {
    p.part = reinterpret_cast<float*>(partials);
    p.k_split = plan.k_split;
    // The rank-16 update is folded into split 0's partial (the reduce then
    // only sums: its lora_A column loads dominated its load count); the
    // forward's rounded LoRA term goes from split 0 to a plane of its own
    // (its lora_B row loads doubled the reduce's load count: 990 x 1536 x
    // 8960 reduce 11.7 us against 6.9 us without the LoRA term).
    p.fold_rank = epi == EPI_RANK;
    p.lora_plane = epi == EPI_LORA
                       ? reinterpret_cast<half_t*>(static_cast<char*>(partials) +
                                                   nt_plane_offset(p.M, p.N, plan.splits))
                       : nullptr;
    const int64_t tail = p.tail_blocks, tail2 = p.tail2_blocks;
    p.tail_blocks = p.tail2_blocks = 0;
    const int rc = dispatch_nt<SS_F32, EPI_PARTIAL>(p, plan.cfg, plan.splits, stream);
    if (rc) return rc;
    p.tail_blocks = tail;
    p.tail2_blocks = tail2;
    if (ct == SS_F32) return reduce_nt<SS_F32, EPI_PLAIN>(p, plan.splits, stream);
    if (epi == EPI_LORA) return reduce_nt<SS_F16, EPI_LORA>(p, plan.splits, stream);
    if (epi == EPI_RANK) {
      GemmParams q = p;
      q.alpha = 1.0f;
      q.bias = nullptr;
      if (q.tail_blocks + q.tail2_blocks > 0)
        return reduce_nt<SS_F16, EPI_PLAIN, true>(q, plan.splits, stream);
      return reduce_nt<SS_F16, EPI_PLAIN>(q, plan.splits, stream);
    }
    if (p.glu) return reduce_nt<SS_F16, EPI_GLU>(p, plan.splits, stream);
    return reduce_nt<SS_F16, EPI_PLAIN>(p, plan.splits, stream);
  }
  if (ct == SS_F16) {
    if (epi == EPI_LORA) return dispatch_nt<SS_F16, EPI_LORA>(p, plan.cfg, 1, stream);
    if (epi == EPI_RANK) {
      const int64_t tails = p.tail_blocks + p.tail2_blocks;
      if (tails == 0 || plan.cfg <= 2) return dispatch_nt<SS_F16, EPI_RANK>(p, plan.cfg, 1, stream);
      GemmParams q = p;
      q.tail_blocks = q.tail2_blocks = 0;
      const int rc = dispatch_nt<SS_F16, EPI_RANK>(q, plan.cfg, 1, stream);
      if (rc) return rc;
      hipLaunchKernelGGL(rank_tail_kernel, dim3((unsigned)tails), dim3(256), 0, stream, p);
      SS_CHECK_LAUNCH("rank_tail_kernel");
      return SS_OK;
    }
    // The SwiGLU epilogue moves three more planes through the tile's waves: on the four
    // waves of the wide tiles it outlasts what their loop gains (frozen MLP at T = 990,
    // 1536 x 8960, both activations in epilogues: 435 us on 256 x 160 tiles, 326 us so; 302 us
    // with kernels of their own), so the eight waves of the ping-pong tile do it there, or 128
    // x 128 tiles where few would run.
    if (p.glu) {
      int cfg = plan.cfg;
      if (cfg > 3) cfg = cdiv(p.M, 256) * cdiv(p.N, 256) >= device_cu_count() / 2 ? 8 : 3;
      return dispatch_nt<SS_F16, EPI_GLU>(p, cfg, 1, stream);
    }
    return dispatch_nt<SS_F16, EPI_PLAIN>(p, plan.cfg, 1, stream);
  }
  return dispatch_nt<SS_F32, EPI_PLAIN>(p, plan.cfg, 1, stream);
}

}  // namespace ss
