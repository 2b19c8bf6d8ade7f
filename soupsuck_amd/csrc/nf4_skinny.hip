// Skinny NF4 forward GEMM for small T: Y[T, N] = X[T, K] . Wdec^T (+ epilogue).
//
// Reference: the bnb fused small-M path behind matmul_4bit (solution/
// nf4_patch.py:108-120, solution/kernels/nf4_gemm.py:127-151).  For T <= 128
// the product is bound by reading the NF4 weight once from HBM (0.5 B codes +
// 1/64 B qabs per weight), not by MFMA: this kernel streams the codes
// straight into registers, decodes them there bit-exactly (the standalone
// decoder's arithmetic) into MFMA B fragments, and never stages the weight in
// LDS or writes it back.
//
// Mapping (v_mfma_f32_16x16x32_f16, fp32 accumulate): a wave owns NB blocks of
// 16 weight rows; per iteration it covers 128 k.  Lane l (r = l % 16,
// g = l / 16) loads the 16 bytes = 32 codes of row n0 + r, k 32 g .. 32 g + 31
// (one load, one NF4 64-block, one scale).  Those 32 k feed four MFMA
// k-steps: k-step j takes k 32 g + 8 j .. + 7 from every lane group g.  The
// MFMA sums over its 32 k in any order, so X is read with the same
// permutation: lane (r, g) supplies X[m + r][32 g + 8 j .. + 7].
// Up to 32 rows (nf4_skinny_fwd_kernel): every load an iteration consumes --
// weight runs and X -- is issued PF iterations ahead into a register ring
// (statically indexed by unrolling), and each lane loads its 64-byte X fragment
// runs directly (no LDS, no barrier: the waves of a workgroup run
// independently).
//
// 33 .. 128 rows (nf4_skinny_lds_kernel): X is shared through a double-buffered
// LDS tile whose 272-byte row pitch keeps the 16-row fragment reads
// bank-conflict-free.  Decoding a k-step takes as many VALU cycles as its MFMAs
// take matrix cycles, so the two are software-pipelined within the wave: while
// k-step j multiplies, j + 1 is scaled and rounded and the table reads of j + 2
// are in flight (decode first, multiply after left each pipe idle in turn).
// One instance per 16 rows: 101 rows multiply 7 tiles, not 8.
//
// K is split over grid.y; every split writes fp32 partials [split][T][N] and
// the split-K reduce applies the epilogue (bias, LoRA add) with the GEMM's
// rounding order.  Above 32 rows a split is mostly at least four 128-deep iterations long:
// shorter ones fill the chip but write and reduce an fp32 plane for every 256 k (skinny_plan).
//
// Kernel and reduce on MI355X, us, before (one instance for 65 .. 128 rows, decode ahead
// of the MFMAs, splits of two iterations) -> after, [N, K] at T = 40, 64, 101, 128:
// [3584, 18944] 30.7, 29.9, 38.1, 39.2 -> 26.9, 27.8, 35.0, 37.9; [3584, 3584] 16.1, 18.8,
// 22.8, 23.0 -> 11.9, 13.6, 17.5, 19.9; [1536, 8960] 21.7, 23.7, 27.3, 27.3 -> 13.7, 15.4,
// 18.7, 19.5; [8960, 1536] 15.8, 17.8, 22.9, 24.2 -> 12.3, 14.1, 18.3, 20.4.  At least 3 or
// 6 iterations: [1536, 8960] at 101 rows 20.2 or 19.3.  A bank-conflict-free table (one
// copy of the 16 values per lane, one read per code) costs 5% more than the pair table.

#include "gemm.h"

namespace ss {
namespace {

constexpr int kSkK = 128;          // k per iteration
constexpr int kSkPitch = kSkK + 8; // LDS row pitch of the X tile (halves)
constexpr int kSkNB = 2;           // 16-row weight blocks per wave
constexpr int kSkRowsPerWG = 4 * kSkNB * 16;

// Everything one iteration consumes, loaded PF iterations ahead: the weight
// runs (codes, qabs byte, absmax2) and the lane's 64-byte X fragment run per M tile.
// Because no load is consumed soon after it is issued, the in-order load
// counter never forces the ring's newer loads to complete early.
template <int MT>
struct Slot {
  static constexpr int kX = MT * 4;
  u32x4 codes[kSkNB];
  uint32_t q[kSkNB];
  float a2[kSkNB];
  u32x4 x[kX];
};

template <int MT, int PF>
__global__ __launch_bounds__(256, 2) void nf4_skinny_fwd_kernel(
    const half_t* __restrict__ x, int64_t ldx, int64_t t, Nf4View w, int64_t n, int64_t k,
    int64_t k_split, float* __restrict__ part) {
  using SlotT = Slot<MT>;
  __shared__ float s_code2[256];
  // Both NF4 values of a code byte in one LDS read: {NF4[e >> 4], NF4[e & 15]}.
  __shared__ __attribute__((aligned(8))) float2 s_pair[256];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int r16 = lane & 15;
  const int g = lane >> 4;
  s_code2[tid] = w.code2[tid];
  s_pair[tid] = float2{kNF4[tid >> 4], kNF4[tid & 15]};
  const float offset = w.offset[0];

  const int64_t kbeg = (int64_t)blockIdx.y * k_split;
  const int64_t klen = k - kbeg < k_split ? k - kbeg : k_split;
  const int iters = (int)(klen / kSkK);
  const int64_t wrow0 = (int64_t)blockIdx.x * kSkRowsPerWG + wave * kSkNB * 16;

  // Sources.  Weight rows past N and X rows past T are clamped (their outputs
  // are never stored).
  int64_t code_elem[kSkNB];  // element index of the lane's run at iteration 0
#pragma unroll
  for (int nb = 0; nb < kSkNB; ++nb) {
    int64_t row = wrow0 + nb * 16 + r16;
    row = row < n ? row : n - 1;
    code_elem[nb] = row * k + kbeg + 32 * g;
  }
  const half_t* xsrc[SlotT::kX];
#pragma unroll
  for (int i = 0; i < SlotT::kX; ++i) {
    const int mt = i >> 2, j = i & 3;  // lane's run X[mt*16 + r][32 g + 8 j ..]
    int64_t row = mt * 16 + r16;
    row = row < t ? row : t - 1;
    xsrc[i] = x + row * ldx + kbeg + 32 * g + 8 * j;
  }
  auto fetch = [&](int it, SlotT& sl) {
#pragma unroll
    for (int nb = 0; nb < kSkNB; ++nb) {
      const int64_t e = code_elem[nb] + (int64_t)it * kSkK;
      const int64_t block = e >> 6;
      sl.codes[nb] = *reinterpret_cast<const u32x4*>(w.packed + (e >> 1));
      sl.q[nb] = w.qabs[block];
      sl.a2[nb] = w.absmax2[block >> 8];
    }
#pragma unroll
    for (int i = 0; i < SlotT::kX; ++i)
      sl.x[i] = *reinterpret_cast<const u32x4*>(xsrc[i] + (int64_t)it * kSkK);
  };

  float4v acc[MT][kSkNB];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nb = 0; nb < kSkNB; ++nb) acc[mt][nb] = float4v{0.f, 0.f, 0.f, 0.f};

  SlotT ring[PF];
  const int last = iters > 0 ? iters - 1 : 0;
  // Slot fills stay in program order (sched_barrier): the ring's depth is
  // only real if slot s is never among the newest outstanding loads when
  // step s reads it.
#pragma unroll
  for (int s = 0; s < PF; ++s) {
    fetch(s < last ? s : last, ring[s]);
    __builtin_amdgcn_sched_barrier(0);
  }
  __syncthreads();  // code tables visible

  auto step = [&](int it, SlotT& sl, bool refill) {
    half8 bfrag[kSkNB][4];
#pragma unroll
    for (int nb = 0; nb < kSkNB; ++nb) {
      const float scale = s_code2[sl.q[nb]] * sl.a2[nb] + offset;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          const uint32_t byte = (sl.codes[nb][j] >> (8 * b)) & 0xffu;
          const float2 pr = s_pair[byte];
          bfrag[nb][j][2 * b] = f32_to_f16(pr.x * scale);
          bfrag[nb][j][2 * b + 1] = f32_to_f16(pr.y * scale);
        }
      }
    }
    // k-step j outermost: the MT x NB MFMAs of one k-step update distinct
    // accumulators, so each MFMA's dependency on the previous update of its
    // accumulator is MT x NB instructions back (m-tile outermost left only
    // NB = 2 independent chains and stalled on every other MFMA).  The X
    // fragments of a k-step are read before its MFMAs.
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      half8 af[MT];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        af[mt] = __builtin_bit_cast(half8, sl.x[mt * 4 + j]);
      }
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nb = 0; nb < kSkNB; ++nb)
          acc[mt][nb] =
              __builtin_amdgcn_mfma_f32_16x16x32_f16(af[mt], bfrag[nb][j], acc[mt][nb], 0, 0, 0);
    }
    // Refill with iteration it + PF, clamped to a valid iteration so that the
    // loads are always issued (the load counts stay the same every
    // iteration).
    __builtin_amdgcn_sched_barrier(0);
    if (refill) fetch(it + PF < last ? it + PF : last, sl);
    __builtin_amdgcn_sched_barrier(0);
  };

  // Main loop: whole groups of PF iterations, straight-line; tail after it.
  const int full = iters / PF * PF;
  for (int it0 = 0; it0 < full; it0 += PF) {
#pragma unroll
    for (int s = 0; s < PF; ++s) step(it0 + s, ring[s], true);
  }
#pragma unroll
  for (int s = 0; s < PF; ++s)
    if (full + s < iters) step(full + s, ring[s], false);

  // Partials: lane holds D[4 g + r][r16] of each 16x16 (rows = X rows, cols =
  // weight rows).
  float* out = part + (int64_t)blockIdx.y * t * n;
#pragma unroll
  for (int nb = 0; nb < kSkNB; ++nb) {
    const int64_t col = wrow0 + nb * 16 + r16;
    if (col >= n) continue;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t row = mt * 16 + 4 * g + r;
        if (row < t) out[row * n + col] = acc[mt][nb][r];
      }
  }
}

// 33 .. 128 rows: X shared by the workgroup's waves through LDS.
template <int MT>
__global__ __launch_bounds__(256, 2) void nf4_skinny_lds_kernel(
    const half_t* __restrict__ x, int64_t ldx, int64_t t, Nf4View w, int64_t n, int64_t k,
    int64_t k_split, float* __restrict__ part) {
  constexpr int kSkRing = MT == 8 ? 2 : 3;  // iterations of codes in flight (registers)
  struct Codes {
    u32x4 codes[kSkNB];
    uint32_t q[kSkNB];
    float a2[kSkNB];
  };
  __shared__ __attribute__((aligned(16))) half_t sx[2][MT * 16 * kSkPitch];
  __shared__ float s_code2[256];
  // Both NF4 values of a code byte in one LDS read: {NF4[e >> 4], NF4[e & 15]}.
  __shared__ __attribute__((aligned(8))) float2 s_pair[256];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int r16 = lane & 15;
  const int g = lane >> 4;
  const int64_t kbeg = (int64_t)blockIdx.y * k_split;
  const int64_t klen = k - kbeg < k_split ? k - kbeg : k_split;
  const int iters = (int)(klen / kSkK);
  const int last = iters - 1;
  const int64_t wrow0 = (int64_t)blockIdx.x * kSkRowsPerWG + wave * kSkNB * 16;

  // Weight rows past N and X rows past T are clamped (their outputs are never stored).
  int64_t code_elem[kSkNB];
#pragma unroll
  for (int nb = 0; nb < kSkNB; ++nb) {
    int64_t row = wrow0 + nb * 16 + r16;
    row = row < n ? row : n - 1;
    code_elem[nb] = row * k + kbeg + 32 * g;
  }
  // X tile chunk c = tid + 256 i: row c / 16, 16-byte chunk c % 16.  Only the last 16-row
  // tile can reach past T.
  const int64_t tail_row = (tid >> 4) + 16 * (MT - 1) < t ? (tid >> 4) + 16 * (MT - 1) : t - 1;
  const half_t* const x_first = x + (tid >> 4) * ldx + kbeg + (tid & 15) * 8;
  const half_t* const x_tail = x + tail_row * ldx + kbeg + (tid & 15) * 8;
  Codes ring[kSkRing];
  u32x4 xr[MT];
  auto fetch_codes = [&](int it, Codes& sl) {
    it = it < last ? it : last;
#pragma unroll
    for (int nb = 0; nb < kSkNB; ++nb) {
      const int64_t e = code_elem[nb] + (int64_t)it * kSkK;
      const int64_t block = e >> 6;
      sl.codes[nb] = *reinterpret_cast<const u32x4*>(w.packed + (e >> 1));
      sl.q[nb] = w.qabs[block];
      sl.a2[nb] = w.absmax2[block >> 8];
    }
  };
  auto fetch_x = [&](int it) {
    const int64_t at = (int64_t)(it < last ? it : last) * kSkK;
#pragma unroll
    for (int i = 0; i < MT; ++i)
      xr[i] = *reinterpret_cast<const u32x4*>((i < MT - 1 ? x_first + i * 16 * ldx : x_tail) + at);
  };

  const float c2 = w.code2[tid];
  const float offset = w.offset[0];
  fetch_codes(0, ring[0]);
  fetch_x(0);
#pragma unroll
  for (int s = 1; s < kSkRing; ++s) fetch_codes(s, ring[s]);
  s_code2[tid] = c2;
  s_pair[tid] = float2{kNF4[tid >> 4], kNF4[tid & 15]};
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
  asm volatile("s_barrier" ::: "memory");

  float2 pr[kSkNB][4];
  half8 bc[kSkNB];
  float sc[kSkNB];
  auto lookup = [&](const Codes& sl, int j) {
#pragma unroll
    for (int nb = 0; nb < kSkNB; ++nb)
#pragma unroll
      for (int b = 0; b < 4; ++b) pr[nb][b] = s_pair[(sl.codes[nb][j] >> (8 * b)) & 0xffu];
  };
  auto convert = [&](half8 (&b8)[kSkNB]) {
#pragma unroll
    for (int nb = 0; nb < kSkNB; ++nb)
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        b8[nb][2 * b] = f32_to_f16(pr[nb][b].x * sc[nb]);
        b8[nb][2 * b + 1] = f32_to_f16(pr[nb][b].y * sc[nb]);
      }
  };
  auto scales = [&](const Codes& sl) {
#pragma unroll
    for (int nb = 0; nb < kSkNB; ++nb) sc[nb] = s_code2[sl.q[nb]] * sl.a2[nb] + offset;
  };

  float4v acc[MT][kSkNB];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nb = 0; nb < kSkNB; ++nb) acc[mt][nb] = float4v{0.f, 0.f, 0.f, 0.f};

  // Pipeline over k-steps: while the MFMAs of one run, the next one's weights are scaled
  // and rounded and the table reads of the one after are in flight.
  scales(ring[0]);
  lookup(ring[0], 0);
  convert(bc);
  lookup(ring[0], 1);
  auto step = [&](int it, Codes& cur, const Codes& next) {
    const int buf = it & 1;
#pragma unroll
    for (int i = 0; i < MT; ++i)
      *reinterpret_cast<u32x4*>(&sx[buf][((tid >> 4) + 16 * i) * kSkPitch + (tid & 15) * 8]) =
          xr[i];
    // LDS-only barrier: __syncthreads() would drain the loads in flight.  The barrier of
    // the previous iteration ordered every wave's reads of this buffer before the writes.
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): this thread's LDS writes done
    asm volatile("s_barrier" ::: "memory");
    fetch_x(it + 1);
    const half_t* const tile = &sx[buf][r16 * kSkPitch + 32 * g];
    half8 af[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
      af[mt] = *reinterpret_cast<const half8*>(tile + mt * 16 * kSkPitch);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      half8 bn[kSkNB];
      if (j == 3) scales(next);
      convert(bn);
      lookup(j < 2 ? cur : next, j < 2 ? j + 2 : j - 2);
      if (j == 1) fetch_codes(it + kSkRing, cur);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
        for (int nb = 0; nb < kSkNB; ++nb)
          acc[mt][nb] =
              __builtin_amdgcn_mfma_f32_16x16x32_f16(af[mt], bc[nb], acc[mt][nb], 0, 0, 0);
        if (j < 3)
          af[mt] = *reinterpret_cast<const half8*>(tile + mt * 16 * kSkPitch + 8 * (j + 1));
      }
#pragma unroll
      for (int i = 0; i < MT * kSkNB; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                     // MFMA
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);                     // LDS read
        __builtin_amdgcn_sched_group_barrier(0x002, 80 / (MT * kSkNB), 0);     // VALU
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int nb = 0; nb < kSkNB; ++nb) bc[nb] = bn[nb];
    }
  };
  int it0 = 0;
  for (; it0 + kSkRing <= iters; it0 += kSkRing) {
#pragma unroll
    for (int s = 0; s < kSkRing; ++s) step(it0 + s, ring[s], ring[(s + 1) % kSkRing]);
  }
#pragma unroll
  for (int s = 0; s < kSkRing - 1; ++s)
    if (it0 + s < iters) step(it0 + s, ring[s], ring[s + 1]);

  // Partials: lane holds D[4 g + r][r16] of each 16x16 (rows = X rows, cols = weight rows).
  float* out = part + (int64_t)blockIdx.y * t * n;
#pragma unroll
  for (int nb = 0; nb < kSkNB; ++nb) {
    const int64_t col = wrow0 + nb * 16 + r16;
    if (col >= n) continue;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t row = mt * 16 + 4 * g + r;
        if (row < t) out[row * n + col] = acc[mt][nb][r];
      }
  }
}

}  // namespace

SkinnyPlan skinny_plan(int64_t t, int64_t n, int64_t k) {
  SkinnyPlan plan{0, 0, 0};
  if (t <= 0 || t > kSkinnyMaxT || n <= 0 || k <= 0 || k % kSkK != 0) return plan;
  plan.mt = (int)cdiv(t, 16);
  // About two workgroups per CU, each split at least two iterations long.  Four above 32
  // rows, where the partial planes are tall (measured at the top of the file), unless that
  // leaves a short K's chain to few workgroups: K of at most 2560, half the CUs idle and
  // planes of at most 8 MB.  Kernel and reduce, us, [N, K] with two / four iterations at T = 33,
  // 64, 128: [256, 1536] 7.2 / 9.0, 7.9 / 9.8, 10.3 / 12.7; [896, 2304] 8.0 / 9.7, 9.1 / 10.8, 12.3 /
  // 14.4; [4096, 1536] 8.9 / 9.6, 11.0 / 11.4, 16.5 / 15.8; [8192, 1024] 9.5 / 10.2, 12.4 / 11.9, 20.2 /
  // 17.1; [18944, 512] 11.4 / 10.5, 15.1 / 12.8, 22.3 / 18.4; [1024, 4096] 10.6 / 9.8, 12.3 / 11.0,
  // 15.8 / 14.6.
  const int64_t cols = cdiv(n, kSkRowsPerWG);
  int64_t s = 512 / cols;
  int64_t least = 2;
  if (plan.mt > 2 && (k > 20 * kSkK || cols * (k / (4 * kSkK)) > 128 ||
                      k / (2 * kSkK) * n * t > 2 << 20))
    least = 4;
  if (s > k / (least * kSkK)) s = k / (least * kSkK);
  if (s < 1) s = 1;
  plan.k_split = cdiv(cdiv(k, s), kSkK) * kSkK;
  plan.splits = cdiv(k, plan.k_split);
  return plan;
}

size_t skinny_partial_bytes(int64_t t, int64_t n, int64_t k) {
  const SkinnyPlan plan = skinny_plan(t, n, k);
  return plan.mt ? (size_t)(plan.splits * t * n) * sizeof(float) : 0;
}

int nf4_skinny_fwd(const GemmParams& p, int epi, void* partials, size_t partial_bytes,
                   hipStream_t stream) {
  const SkinnyPlan plan = skinny_plan(p.M, p.N, p.K);
  if (!plan.mt || !partials || partial_bytes < skinny_partial_bytes(p.M, p.N, p.K) ||
      reinterpret_cast<uintptr_t>(partials) % 16 != 0 ||
      reinterpret_cast<uintptr_t>(p.A) % 16 != 0 || p.lda % 8 != 0 ||
      reinterpret_cast<uintptr_t>(p.w.packed) % 16 != 0)
    return SS_ERR_UNSUPPORTED;
  if (epi != EPI_PLAIN && (reinterpret_cast<uintptr_t>(p.lz) % 16 != 0))
    return SS_ERR_UNSUPPORTED;
  float* part = reinterpret_cast<float*>(partials);
  const dim3 grid((unsigned)cdiv(p.N, kSkRowsPerWG), (unsigned)plan.splits);
  switch (plan.mt) {
    case 1:
      hipLaunchKernelGGL((nf4_skinny_fwd_kernel<1, 4>), grid, dim3(256), 0, stream, p.A,
                         p.lda, p.M, p.w, p.N, p.K, plan.k_split, part);
      break;
    case 2:
      hipLaunchKernelGGL((nf4_skinny_fwd_kernel<2, 3>), grid, dim3(256), 0, stream, p.A,
                         p.lda, p.M, p.w, p.N, p.K, plan.k_split, part);
      break;
#define SS_SKINNY(MT)                                                                        \
  case MT:                                                                                   \
    hipLaunchKernelGGL((nf4_skinny_lds_kernel<MT>), grid, dim3(256), 0, stream, p.A, p.lda,  \
                       p.M, p.w, p.N, p.K, plan.k_split, part);                              \
    break;
    SS_SKINNY(3)
    SS_SKINNY(4)
    SS_SKINNY(5)
    SS_SKINNY(6)
    SS_SKINNY(7)
    SS_SKINNY(8)
#undef SS_SKINNY
    default:
      return SS_ERR_UNSUPPORTED;
  }
  SS_CHECK_LAUNCH("nf4_skinny_fwd_kernel");
  GemmParams q = p;
  q.part = part;
  return splitk_reduce(q, (int)plan.splits, SS_F16, epi, stream);
}

}  // namespace ss
