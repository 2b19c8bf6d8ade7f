// Causal attention over packed rows (varlen), forward and backward, head_dim 128.
//
// Replaces the reference's per-row SDPA loop over a packed batch
// (solution/unpad.py:359-410: each real row of length L attends causally to
// itself only; GQA by repeating the KV heads; scale 1/sqrt(head_dim)).  Rows
// are given by cu_seqlens (int32 [rows + 1], offsets into the packed token
// axis); a query attends to the keys of its own row at positions <= its own.
//
// Layout (HBM): q [T, Hq, 128], k / v [T, Hk, 128] with any token and head
// strides (unit last stride), o [T, Hq, 128] likewise, fp16; lse2 fp32 [Hq, T]
// holds m + log2(l) of the base-2 scaled scores (the backward's softmax
// statistic).  Scores are s = (q . k) * scale in fp32 (MFMA accumulate),
// softmax in fp32 with an online maximum, P rounded to fp16 for the P.V MFMA,
// O accumulated in fp32 and rounded once.
//
// What bounds it: LDS reads and MFMA together.  Every product has one operand
// in registers (32 queries or 32 keys of a wave) and reads the other from a
// 64-token LDS tile shared by the workgroup, so a v_mfma_f32_32x32x16_f16 (32
// clocks) needs 1 KiB from LDS.  With 16 queries or keys per wave
// (v_mfma_f32_16x16x32_f16) the same read fed half the work and LDS was the limit.  At
// 6041 tokens in rows of 128 .. 2048, 28 q / 4 kv heads, 16-row against 32-row waves:
// forward 293 -> 93 us (63 GFLOP causal), dQ 319 -> 118 us, dK / dV 619 -> 205 us; at 990
// tokens in rows of 158 .. 382, 12 q / 2 kv heads: 15 -> 10, 17 -> 15, 21 -> 14 us.  A
// forward tile (64 keys) now takes a CU 0.93 us against 0.49 us of MFMA issue; the rest
// is the softmax (about as many vector as MFMA clocks) and the barrier per tile.
//
// MFMA operand order: lane l supplies k 8 (l / 32) .. + 7 of row / column l %
// 32; the accumulator gives lane l rows 8 (r / 4) + 4 (l / 32) + r % 4 of column
// l % 32 in register r.  The k order inside one MFMA is free as long as both
// operands use it, so the accumulator of a score tile (keys down, one query per
// lane) is the operand P^T of O^T += V^T . P^T as it stands: registers 8 u .. 8 u
// + 7 are slots 8 (l / 32) .. + 7 of step u, i.e. keys 16 u + 4 (l / 32) + i and
// 16 u + 8 + 4 (l / 32) + i, and V^T supplies the same keys in the same slots.
//
// LDS tiles hold 64 token rows of 256 B, written by the loads themselves
// (global_load_lds, one wave-wide DMA is four rows; no staging registers) into
// two buffers: tile t + 1 lands while tile t is used, one barrier per tile.
// 16-byte chunk c of row r sits at c ^ (((r & 3) << 2) | ((r >> 2) & 3)): the 16
// rows that one pass of a 128-bit read covers take 16 different chunks, and the
// four rows x 64 B of a transposed read (ds_read_b64_tr_b16, for operands that
// run along the token axis) take different banks too.
//
// Workgroups: 4 waves on 128 queries (keys) of one head, 32 per wave; batches too small
// to fill the chip that way take 64, two waves for each 32 (short_batch).  Batches of short
// rows take 16-row waves (attention_rows16.h).
//
// Backward: a dQ kernel per (row, query block, q head), which also writes
// delta = rowsum(dO . O); then a dK / dV kernel per (row, key block, q head)
// over the causal query tiles; with GQA each q head writes fp32 partials that
// a reduce kernel adds in head order (no atomics, deterministic).
#include <type_traits>
#include <utility>

#include "gemm.h"

namespace ss {
namespace {

typedef float float16v __attribute__((ext_vector_type(16)));

constexpr int kD = 128;                     // head dimension
constexpr int kWaves = 4;                   // per workgroup
constexpr int kTile = 64;                   // token rows of an LDS tile
constexpr int kTileBytes = kTile * kD * 2;  // 16 KiB
constexpr float kLog2e = 1.4426950408889634f;
// The running maximum is raised (and O rescaled: 64 multiplies per lane) only when
// a score exceeds it by more than this many powers of two; until then P stays below
// 2.  A larger bound saves few rescales more and costs accuracy: P of the leading keys
// is best just below 1, where its fp16 rounding is smallest (error of O against 64
// bits over 1536 random keys: 2.50e-4 with 0, 2.52e-4 with 1, 2.61e-4 with 8; 2.53e-4
// with 0 and 64 keys a step, O divided by the unrounded sum, as before).
constexpr float kDefer = 1.0f;

struct AttnArgs {
  const half_t* q; int64_t q_tok, q_head;
  const half_t* k; int64_t k_tok, k_head;
  const half_t* v; int64_t v_tok, v_head;
  const half_t* o; int64_t o_tok, o_head;     // forward output / backward input
  const half_t* dout; int64_t do_tok, do_head;
  half_t* out; int64_t out_tok, out_head;     // forward O, or backward dQ
  half_t* dk; int64_t dk_tok, dk_head;
  half_t* dv; int64_t dv_tok, dv_head;
  float* lse2;      // [hq][total]
  float* delta;     // [hq][total], holds -rowsum(dO . O)
  const int* cu;    // [rows + 1]
  int64_t total;
  int rows, blocks, span;  // packed rows; blocks of the longest row; tokens of a block
  int hq, hk;
  float scale;      // softmax scale (1/sqrt(128) for Qwen2)
};

__device__ __forceinline__ float16v mfma(half8 a, half8 b, float16v c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ half8 ld8(const half_t* p) { return *reinterpret_cast<const half8*>(p); }
__device__ __forceinline__ float exp2_hw(float x) { return __builtin_amdgcn_exp2f(x); }

// The value of lane l ^ 32 combined with this lane's.
__device__ __forceinline__ float2v both_halves(float v) {
  const uint32_t b = __builtin_bit_cast(uint32_t, v);
  const auto r = __builtin_amdgcn_permlane32_swap(b, b, false, false);
  return float2v{__builtin_bit_cast(float, (uint32_t)r[0]),
                 __builtin_bit_cast(float, (uint32_t)r[1])};
}
__device__ __forceinline__ float half_max(float v) {
  const float2v p = both_halves(v);
  return fmaxf(p[0], p[1]);
}
__device__ __forceinline__ float half_sum(float v) {
  const float2v p = both_halves(v);
  return p[0] + p[1];
}

// Scores want a positive base-2 scale (the online maximum, and a mask of -inf before
// the scaling): a negative one is moved into the register operand of the score product
// (exact), a zero one zeroes it.
__device__ __forceinline__ float positive_scale(float sl2, half8 (&f)[8]) {
  if (sl2 > 0.f || sl2 != sl2) return sl2;
  const half_t sign = sl2 < 0.f ? (half_t)-1.f : (half_t)0.f;
#pragma unroll
  for (int ks = 0; ks < 8; ++ks) f[ks] *= sign;
  return sl2 < 0.f ? -sl2 : 1.f;
}

// Eight fp16 values of one MFMA operand, built two at a time.
typedef u32x4 Packed8;
__device__ __forceinline__ half8 operand(const Packed8& p) { return __builtin_bit_cast(half8, p); }

// Two fp32 values rounded into elements 2 (k % 4), + 1 of h.  The tie keeps the
// conversion in its step (it would sink to the operand's use).
__device__ __forceinline__ half2_t round2(Packed8& h, int k, float a, float b) {
  uint32_t v = __builtin_bit_cast(uint32_t, half2_t{f32_to_f16(a), f32_to_f16(b)});
  tie(v);
  h[k & 3] = v;
  return __builtin_bit_cast(half2_t, v);
}

// N MFMA operands streamed from LDS: use(i, operand i) in order, each read issued
// kAhead operands before its use and held there by the fences (the compiler otherwise
// reads one operand ahead of each MFMA, and every MFMA waits for an LDS round trip:
// forward 100 us, dK / dV 224 us in the example above).
// The position is a compile-time value (of type Pos<i>).
template <int I>
using Pos = std::integral_constant<int, I>;

template <int N, int kAhead, int I, class Load, class Use>
__device__ __forceinline__ void stream_from(Load& load, Use& use, half8 (&ring)[kAhead]) {
  if constexpr (I < N) {
    use(Pos<I>{}, ring[I % kAhead]);
    if constexpr (I + kAhead < N) ring[I % kAhead] = load(Pos<I + kAhead>{});
    __builtin_amdgcn_sched_barrier(0);
    stream_from<N, kAhead, I + 1>(load, use, ring);
  }
}
template <int N, int kAhead, class Load, class Use, int... I>
__device__ __forceinline__ void stream_first(Load& load, half8 (&ring)[kAhead],
                                             std::integer_sequence<int, I...>) {
  ((ring[I] = load(Pos<I>{})), ...);
}
template <int N, int kAhead, class Load, class Use>
__device__ __forceinline__ void stream_operands(Load load, Use use) {
  half8 ring[kAhead];
  stream_first<N, kAhead, Load, Use>(load, ring, std::make_integer_sequence<int, kAhead>{});
  __builtin_amdgcn_sched_barrier(0);
  stream_from<N, kAhead, 0>(load, use, ring);
}

// LDS DMA of one lane's 16 (4) bytes at p to lds + 16 (4) x lane.
__device__ __forceinline__ void dma16_at(const void* p, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
               :
               : "v"(p), "s"(lds)
               : "memory", "m0");
}
__device__ __forceinline__ void dma4_at(const void* p, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off"
               :
               : "v"(p), "s"(lds)
               : "memory", "m0");
}

// Loads of one operand's tiles: DMA g (of 16) brings rows 4 g .. 4 g + 3, a wave
// issues four of them.  A whole tile takes wave-uniform row addresses and four
// lane offsets kept in registers; a tile past the packed row's end (or a token
// stride that is negative or whose offsets need 64 bits: they are unsigned 32-bit bytes)
// takes an address per lane, rows past the end re-reading the last row (their scores are
// masked, or their results not stored).
struct TileLoader {
  static constexpr int kPer = 16 / kWaves;  // DMAs per wave and tile
  const half_t* base;  // first token of the row, this head
  int64_t tok;
  int len;
  uint32_t off[4];  // lane's row of a DMA and its chunk ((j & 3) swizzle)

  __device__ __forceinline__ TileLoader(const half_t* p, int64_t tok_stride, int row_len, int lane)
      : base(p), tok(tok_stride), len(row_len) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      off[j] = (uint32_t)(lane >> 4) * (uint32_t)tok * 2 + chunk(lane, j) * 16;
  }
  static __device__ __forceinline__ uint32_t chunk(int lane, int j) {
    return (lane & 15) ^ ((lane >> 4) << 2) ^ j;
  }
  __device__ __forceinline__ void issue(int t0, uint32_t lds, int wave) const {
    if (t0 + kTile <= len && tok >= 0 && tok < (1 << 28)) {
      const half_t* rows = base + (int64_t)(t0 + 4 * wave * kPer) * tok;
#pragma unroll
      for (int j = 0; j < kPer; ++j)
        dma16(off[j & 3], rows + 4 * j * tok, lds + (wave * kPer + j) * 1024);
    } else {
      const int lane = threadIdx.x & 63;
#pragma unroll 1
      for (int j = 0; j < kPer; ++j) {
        const int t = min(t0 + 4 * (wave * kPer + j) + (lane >> 4), len - 1);
        dma16_at(base + (int64_t)t * tok + chunk(lane, j & 3) * 8,
                 lds + (wave * kPer + j) * 1024);
      }
    }
  }
};

// Operand reads of a tile (byte offsets within it).  row(ks): rows l % 32, k =
// 16 ks + 8 (l / 32) .. + 7 of a row-major operand; rows 32 .. 63 are 8 KiB on.
// tr(u, dt): columns d = 32 dt + l % 32, tokens in the slots of step u (16 u + 4 (l
// / 32) + i, then + 8): two ds_read_b64_tr_b16.  In each 16-lane group the lanes'
// 8-byte reads form a 16 x 4 matrix M (row = reading lane) and lane i receives M[4
// j + i / 4][i % 4] (measured on gfx950), so lane r of a group points at token r /
// 4, columns 4 (r % 4) .. + 3.
typedef short attn_short4 __attribute__((ext_vector_type(4)));
typedef short attn_short8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) attn_short4 attn_lds_short4;

struct TileReader {
  int row_off[8];
  int tr_off[4][2];
  __device__ __forceinline__ explicit TileReader(int lane) {
    const int r = lane & 31, h = lane >> 5;
    const int f = ((r & 3) << 2) | ((r >> 2) & 3);
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) row_off[ks] = r * 256 + (((2 * ks + h) ^ f) << 4);
    const int a = (lane & 15) >> 2;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const int c = 4 * dt + 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
        tr_off[dt][s] = (4 * h + a + 8 * s) * 256 + ((c ^ ((a << 2) | h | (s << 1))) << 4) +
                        ((lane & 1) << 3);
      }
  }
  __device__ __forceinline__ half8 row(const unsigned char* tile, int half, int ks) const {
    return *reinterpret_cast<const half8*>(tile + row_off[ks] + half * 8192);
  }
  __device__ __forceinline__ half8 tr(const unsigned char* tile, int u, int dt) const {
    const attn_short4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (attn_lds_short4*)(tile + tr_off[dt][0] + u * 4096));
    const attn_short4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (attn_lds_short4*)(tile + tr_off[dt][1] + u * 4096));
    return __builtin_bit_cast(half8, attn_short8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2],
                                                 hi[3]});
  }
};

// Scores whose register row (8 (r / 4) + r % 4) is below lo or from hi on become -inf (and
// their statistics, if given, 0).
// Called under a rarely true uniform branch; the ties keep the compares and selects
// inside it (hoisted, they were 32 of the ~90 vector instructions of every half tile).
template <class... Stats>
__device__ __forceinline__ void mask_rows(float16v& s, int lo, int hi, Stats&... stats) {
  tie(lo);
  tie(hi);
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    float x = s[r];
    tie(x);
    const int row = 8 * (r >> 2) + (r & 3);
    const bool masked = row < lo || row >= hi;
    s[r] = masked ? -INFINITY : x;
    ((stats[r] = masked ? 0.f : stats[r]), ...);
  }
}

// Every DMA of this wave has landed and its LDS reads are done; after the barrier
// that holds for the workgroup.
__device__ __forceinline__ void tile_barrier() {
  wait_vm<0>();
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// Work item of a workgroup.  Workgroups go round-robin over the 8 XCDs whatever their
// load.  A unit is the q heads of one kv head over one block of one packed row: they
// run one after another on one XCD, whose L2 then serves K and V to the whole group.
// Units are dealt to the XCDs in rounds of eight, each round starting at another XCD
// (dealt straight, 6 rows x 4 kv heads put every long row on the same four XCDs: 110
// against 100 us forward), the blocks with the most tiles first.  With at most 64 rows
// only blocks that exist get workgroups: an empty one still waits for LDS to be free
// before it can leave (half of them empty: 106 against 93 us).
struct Item {
  int block, row, start, len, head, kv_head;
  bool valid;
  __device__ __forceinline__ Item(const AttnArgs& a, bool last_first) {
    const int64_t l = (int64_t)blockIdx.y * gridDim.x + blockIdx.x;
    const int group = a.hq / a.hk;
    int64_t pos;
    const int64_t round = (l >> 3) / group;
    const int64_t unit = round * 8 + ((l + round + (round >> 3) * 3 + (round >> 6) * 5) & 7);
    pos = unit / a.hk;
    kv_head = (int)(unit - pos * a.hk);
    head = kv_head * group + (int)((l >> 3) - round * group);
    if (a.rows <= 64) {
      // Position -> (block, row) with the blocks of the highest index first, rows in
      // order: walk the levels down (up), counting the rows that have a block there.
      const int lane = threadIdx.x & 63;
      const int r = min(lane, a.rows - 1);
      const int c0 = a.cu[r], c1 = a.cu[r + 1];
      const int have = lane < a.rows ? (c1 - c0 + a.span - 1) / a.span : 0;
      int64_t left = pos;
      int k = last_first ? a.blocks - 1 : 0;
      uint64_t rows = 0;
      for (int t = 0; t < a.blocks; ++t) {
        rows = __ballot(have > k);
        const int n = __popcll(rows);
        if (left < n) break;
        left -= n;
        rows = 0;
        k += last_first ? -1 : 1;
      }
      valid = rows != 0;
      const bool mine = (rows >> lane & 1) &&
                        __popcll(rows & (((uint64_t)1 << lane) - 1)) == left;
      const uint64_t pick = __ballot(mine);
      row = pick ? __ffsll((unsigned long long)pick) - 1 : 0;
      block = k;
      start = __builtin_amdgcn_readlane(c0, row);
      len = __builtin_amdgcn_readlane(c1, row) - start;
    } else {
      block = (int)(pos / a.rows);
      row = (int)(pos - (int64_t)block * a.rows);
      valid = block < a.blocks;
      if (last_first) block = a.blocks - 1 - block;
      start = a.cu[row];
      len = a.cu[row + 1] - start;
      valid = valid && block * a.span < len;
    }
  }
};

// Row of 128 outputs held as [d][query] accumulators (scaled, rounded), 16 bytes
// per store: lanes l and l + 32 exchange so that each owns 8 consecutive d.
__device__ __forceinline__ void store_row(half_t* p, const float16v (&acc)[4], float scale,
                                          int h, bool live) {
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int jj = 0; jj < 2; ++jj) {
      half4 even, odd;  // d = 16 jj + 4 h + i and + 8
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        even[i] = f32_to_f16(acc[dt][8 * jj + i] * scale);
        odd[i] = f32_to_f16(acc[dt][8 * jj + 4 + i] * scale);
      }
      const u32x2 e = __builtin_bit_cast(u32x2, even), o = __builtin_bit_cast(u32x2, odd);
      const auto s0 = __builtin_amdgcn_permlane32_swap(e[0], o[0], false, false);
      const auto s1 = __builtin_amdgcn_permlane32_swap(e[1], o[1], false, false);
      const u32x4 v = {(uint32_t)s0[0], (uint32_t)s1[0], (uint32_t)s0[1], (uint32_t)s1[1]};
      if (live) *reinterpret_cast<u32x4*>(p + 32 * dt + 16 * jj + 8 * h) = v;
    }
}

// Exchange of a wave's accumulators with its partner part through 16 KiB of LDS:
// put, and acc = a0 acc + a1 (the partner's).
__device__ __forceinline__ void put_acc(unsigned char* lds, const float16v (&acc)[4], int lane) {
  float4v* to = reinterpret_cast<float4v*>(lds) + lane;
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int j = 0; j < 4; ++j)
      to[(4 * dt + j) * 64] = float4v{acc[dt][4 * j], acc[dt][4 * j + 1], acc[dt][4 * j + 2],
                                      acc[dt][4 * j + 3]};
}
__device__ __forceinline__ void add_acc(const unsigned char* lds, float16v (&acc)[4], float a0,
                                        float a1, int lane) {
  const float4v* from = reinterpret_cast<const float4v*>(lds) + lane;
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float4v o = from[(4 * dt + j) * 64];
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[dt][4 * j + i] = acc[dt][4 * j + i] * a0 + o[i] * a1;
    }
}

// Kernels: G groups of 32 queries (keys) per workgroup, PARTS waves for each.  <4, 1>:
// a wave per group takes whole tiles.  <2, 2>: the two waves of a group take the two
// 32-token halves of every tile and add their results at the end.

// ------------------------------------------------------------------ forward

template <int G, int PARTS>
__global__ __launch_bounds__(64 * kWaves, 2) void attn_fwd_kernel(AttnArgs a) {
  const Item item(a, true);
  if (!item.valid) return;
  const int start = item.start, len = item.len;
  const int q0 = item.block * 32 * G;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = lane >> 5;
  const int q0w = q0 + (wave % G) * 32, part = wave / G;
  const int myq = q0w + (lane & 31);  // the query of this lane's column
  __shared__ __align__(1024) unsigned char smem[4 * kTileBytes];  // K, V of two tiles

  const TileLoader kl(a.k + (int64_t)start * a.k_tok + (int64_t)item.kv_head * a.k_head,
                          a.k_tok, len, lane);
  const TileLoader vl(a.v + (int64_t)start * a.v_tok + (int64_t)item.kv_head * a.v_head,
                          a.v_tok, len, lane);
  const uint32_t lds = __builtin_amdgcn_readfirstlane(lds_address(smem));
  kl.issue(0, lds, wave);
  vl.issue(0, lds + kTileBytes, wave);

  // S^T = K . Q^T: Q[myq][16 ks + 8 h + j].
  half8 qf[8];
  {
    const half_t* qp = a.q + (int64_t)(start + min(myq, len - 1)) * a.q_tok +
                       (int64_t)item.head * a.q_head + 8 * h;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) qf[ks] = ld8(qp + 16 * ks);
  }
  const float sl2 = positive_scale(a.scale * kLog2e, qf);
  const TileReader rd(lane);
  float16v acc[4];  // O^T: [d = 32 dt + ..][q = myq]
#pragma unroll
  for (int dt = 0; dt < 4; ++dt) acc[dt] = float16v{};
  // This lane's keys only, until the end: l sums P in fp32 (the softmax statistic of
  // the backward), lp the rounded P of the P.V product, which O is divided by (the
  // rounding of P then cancels where one key dominates).
  float m = -INFINITY, l = 0.f, lp = 0.f;

  constexpr int kSub = 2 / PARTS;  // 32-key halves of a tile for this wave
  auto compute = [&](int kb, const unsigned char* sK, const unsigned char* sV) {
    const int k0 = PARTS == 2 ? part : 0;
    const int kw = kb + 32 * k0;
    float16v s[kSub];  // S^T[key = kw + 32 kt + 8 (r / 4) + 4 h + r % 4][q = myq]
    Packed8 p[2 * kSub];
    auto softmax = [&]() {
      if (kw + 32 * kSub - 1 > q0w) {  // the diagonal
#pragma unroll
        for (int kt = 0; kt < kSub; ++kt) mask_rows(s[kt], 0, myq - kw - 32 * kt - 4 * h + 1);
      }
      float mx = s[0][0];
#pragma unroll
      for (int kt = 0; kt < kSub; ++kt)
#pragma unroll
        for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[kt][r]);
      mx *= sl2;
      if (__any(mx > m + kDefer)) {
        const float top = fmaxf(m, half_max(mx));
        const float alpha = exp2_hw(m - top);
        m = top;
        l *= alpha;
        lp *= alpha;
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) acc[dt] *= alpha;
      }
#pragma unroll
      for (int kt = 0; kt < kSub; ++kt)
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const float e0 = exp2_hw(__builtin_fmaf(s[kt][2 * k], sl2, -m));
          const float e1 = exp2_hw(__builtin_fmaf(s[kt][2 * k + 1], sl2, -m));
          l += e0;
          l += e1;
          lp = __builtin_amdgcn_fdot2(round2(p[2 * kt + (k >> 2)], k, e0, e1),
                                      half2_t{(half_t)1.f, (half_t)1.f}, lp, false);
        }
    };
    // Operands: K (k step, half), then V (step of 16 keys, 32 columns).
    constexpr int kS = 8 * kSub;
    stream_operands<2 * kS, 6>(
        [&](auto pos) {
          constexpr int i = pos;
          if constexpr (i < kS)
            return rd.row(sK, k0 + i % kSub, i / kSub);
          else
            return rd.tr(sV, 2 * k0 + (i - kS) / 4, (i - kS) % 4);
        },
        [&](auto pos, half8 f) {
          constexpr int i = pos;
          if constexpr (i < kS) {
            s[i % kSub] = mfma(f, qf[i / kSub], i < kSub ? float16v{} : s[i % kSub]);
            if constexpr (i == kS - 1) softmax();
          } else {
            acc[(i - kS) % 4] = mfma(f, operand(p[(i - kS) / 4]), acc[(i - kS) % 4]);
          }
        });
  };

  const int kend = min(len, q0 + 32 * G);  // causal: later keys unused
  auto step = [&](int kb, int buf) {
    tile_barrier();
    if (kb + kTile < kend) {
      kl.issue(kb + kTile, lds + (buf ^ 1) * 2 * kTileBytes, wave);
      vl.issue(kb + kTile, lds + (buf ^ 1) * 2 * kTileBytes + kTileBytes, wave);
    }
    const unsigned char* sK = smem + buf * 2 * kTileBytes;
    const unsigned char* sV = sK + kTileBytes;
    if (kb + (PARTS == 2 ? 32 * part : 0) <= q0w && q0w < len) compute(kb, sK, sV);
  };
  for (int kb = 0; kb < kend; kb += 2 * kTile) {
    step(kb, 0);
    if (kb + kTile < kend) step(kb + kTile, 1);
  }
  l = half_sum(l);
  lp = half_sum(lp);
  if constexpr (PARTS == 2) {
    // The parts' (O, m, l) merge as online-softmax states; a part without a key has m
    // = -inf and weight 0.
    float* stats = reinterpret_cast<float*>(smem + 3 * kTileBytes) + (wave % G) * 192 + lane;
    tile_barrier();
    if (part) {
      put_acc(smem + (wave % G) * kTileBytes, acc, lane);
      stats[0] = m;
      stats[64] = l;
      stats[128] = lp;
    }
    __syncthreads();
    if (part) return;
    const float m1 = stats[0], top = fmaxf(m, m1);
    const float a0 = exp2_hw(m - top), a1 = exp2_hw(m1 - top);
    l = l * a0 + stats[64] * a1;
    lp = lp * a0 + stats[128] * a1;
    m = top;
    add_acc(smem + (wave % G) * kTileBytes, acc, a0, a1, lane);
  }
  store_row(a.out + (int64_t)(start + min(myq, len - 1)) * a.out_tok +
                (int64_t)item.head * a.out_head, acc, 1.0f / lp, h, myq < len);
  if (myq < len && h == 0) a.lse2[(int64_t)item.head * a.total + start + myq] = m + __log2f(l);
}

// --------------------------------------------------------------- backward dQ

template <int G, int PARTS>
__global__ __launch_bounds__(64 * kWaves, 2) void attn_bwd_dq_kernel(AttnArgs a) {
  const Item item(a, true);
  if (!item.valid) return;
  const int start = item.start, len = item.len;
  const int q0 = item.block * 32 * G;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = lane >> 5;
  const int q0w = q0 + (wave % G) * 32, part = wave / G;
  const int myq = q0w + (lane & 31);
  const int64_t qrow = start + min(myq, len - 1);
  __shared__ __align__(1024) unsigned char smem[4 * kTileBytes];  // K, V of two tiles

  const TileLoader kl(a.k + (int64_t)start * a.k_tok + (int64_t)item.kv_head * a.k_head,
                          a.k_tok, len, lane);
  const TileLoader vl(a.v + (int64_t)start * a.v_tok + (int64_t)item.kv_head * a.v_head,
                          a.v_tok, len, lane);
  const uint32_t lds = __builtin_amdgcn_readfirstlane(lds_address(smem));
  kl.issue(0, lds, wave);
  vl.issue(0, lds + kTileBytes, wave);

  half8 qf[8], df[8];  // Q[myq][16 ks + 8 h + j], dO[myq][...]
  float dsum = 0.f;    // this lane's part of rowsum(dO . O)
  {
    const half_t* qp = a.q + qrow * a.q_tok + (int64_t)item.head * a.q_head + 8 * h;
    const half_t* dp = a.dout + qrow * a.do_tok + (int64_t)item.head * a.do_head + 8 * h;
    const half_t* op = a.o + qrow * a.o_tok + (int64_t)item.head * a.o_head + 8 * h;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
      qf[ks] = ld8(qp + 16 * ks);
      df[ks] = ld8(dp + 16 * ks);
      const half8 ov = ld8(op + 16 * ks);
#pragma unroll
      for (int j = 0; j < 8; ++j) dsum += (float)df[ks][j] * (float)ov[j];
    }
  }
  const float sl2 = positive_scale(a.scale * kLog2e, qf);
  const float delta = half_sum(dsum);
  const float lse = a.lse2[(int64_t)item.head * a.total + qrow];
  if (myq < len && h == 0) a.delta[(int64_t)item.head * a.total + qrow] = -delta;
  const TileReader rd(lane);
  float16v dq[4];  // dQ^T: [d = 32 dt + ..][q = myq]
#pragma unroll
  for (int dt = 0; dt < 4; ++dt) dq[dt] = float16v{};

  auto compute = [&](int kb, const unsigned char* sK, const unsigned char* sV) {
    const int k0 = PARTS == 2 ? part : 0;
    float16v s, e;  // S^T and dP^T - delta of a half tile, [key][q = myq]
    Packed8 ds[2];
    auto elements = [&](int k32) {
      if (k32 + 31 > q0w) mask_rows(s, 0, myq - k32 - 4 * h + 1);  // the diagonal
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const float p0 = exp2_hw(__builtin_fmaf(s[2 * k], sl2, -lse));
        const float p1 = exp2_hw(__builtin_fmaf(s[2 * k + 1], sl2, -lse));
        round2(ds[k >> 2], k, p0 * e[2 * k], p1 * e[2 * k + 1]);
      }
    };
    // Operands of a half: K and V rows (8 k steps), then K along the keys.
    stream_operands<48 / PARTS, 6>(
        [&](auto pos) {
          constexpr int i = pos, o = i % 24;
          if constexpr (o >= 16)
            return rd.tr(sK, 2 * (k0 + i / 24) + (o - 16) / 4, o % 4);
          else
            return rd.row(o & 1 ? sV : sK, k0 + i / 24, o / 2);
        },
        [&](auto pos, half8 f) {
          constexpr int i = pos, o = i % 24;
          if constexpr (o >= 16) {
            dq[o % 4] = mfma(f, operand(ds[(o - 16) / 4]), dq[o % 4]);
          } else if constexpr (o & 1) {
            if constexpr (o == 1) {
#pragma unroll
              for (int r = 0; r < 16; ++r) e[r] = -delta;
            }
            e = mfma(f, df[o / 2], e);
            if constexpr (o == 15) elements(kb + 32 * (k0 + i / 24));
          } else {
            s = mfma(f, qf[o / 2], o == 0 ? float16v{} : s);
          }
        });
  };

  const int kend = min(len, q0 + 32 * G);
  auto step = [&](int kb, int buf) {
    tile_barrier();
    if (kb + kTile < kend) {
      kl.issue(kb + kTile, lds + (buf ^ 1) * 2 * kTileBytes, wave);
      vl.issue(kb + kTile, lds + (buf ^ 1) * 2 * kTileBytes + kTileBytes, wave);
    }
    const unsigned char* sK = smem + buf * 2 * kTileBytes;
    const unsigned char* sV = sK + kTileBytes;
    if (kb + (PARTS == 2 ? 32 * part : 0) <= q0w && q0w < len) compute(kb, sK, sV);
  };
  for (int kb = 0; kb < kend; kb += 2 * kTile) {
    step(kb, 0);
    if (kb + kTile < kend) step(kb + kTile, 1);
  }
  if constexpr (PARTS == 2) {
    tile_barrier();
    if (part) put_acc(smem + (wave % G) * kTileBytes, dq, lane);
    __syncthreads();
    if (part) return;
    add_acc(smem + (wave % G) * kTileBytes, dq, 1.f, 1.f, lane);
  }
  store_row(a.out + qrow * a.out_tok + (int64_t)item.head * a.out_head, dq, a.scale, h,
            myq < len);
}

// ------------------------------------------------------------ backward dK/dV

// One workgroup per (row, key block, q head): waves of 32 keys walk the row's
// causal query tiles.  With GQA (hq > hk) the q heads of a group write fp32
// partial dK / dV planes that attn_bwd_reduce_kernel adds in head order;
// without it dK / dV are written directly.
template <int G, int PARTS>
__global__ __launch_bounds__(64 * kWaves, 1) void attn_bwd_dkdv_kernel(AttnArgs a, float* part_k,
                                                                       float* part_v) {
  const Item item(a, false);
  if (!item.valid) return;
  const int start = item.start, len = item.len;
  const int k0 = item.block * 32 * G;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = lane >> 5, col = lane & 31;
  const int k0w = k0 + (wave % G) * 32, part = wave / G;
  const int mykey = k0w + col;
  // Q, dO, lse2 and -delta of two 64-query tiles.
  constexpr int kBuf = 2 * kTileBytes + 1024;
  __shared__ __align__(1024) unsigned char smem[2 * kBuf];

  const TileLoader ql(a.q + (int64_t)start * a.q_tok + (int64_t)item.head * a.q_head, a.q_tok,
                          len, lane);
  const TileLoader ol(a.dout + (int64_t)start * a.do_tok + (int64_t)item.head * a.do_head,
                          a.do_tok, len, lane);
  const float* stats = (wave == 0 ? a.lse2 : a.delta) + (int64_t)item.head * a.total + start;
  const uint32_t lds = __builtin_amdgcn_readfirstlane(lds_address(smem));
  auto issue = [&](int qt, int buf) {
    const uint32_t at = lds + buf * kBuf;
    ql.issue(qt, at, wave);
    ol.issue(qt, at + kTileBytes, wave);
    if (wave < 2) dma4_at(stats + min(qt + lane, len - 1), at + 2 * kTileBytes + wave * 256);
  };
  issue(k0, 0);

  half8 kf[8], vf[8];  // K[mykey][16 ks + 8 h + j], V[mykey][...]
  {
    const int64_t krow = start + min(mykey, len - 1);
    const half_t* kp = a.k + krow * a.k_tok + (int64_t)item.kv_head * a.k_head + 8 * h;
    const half_t* vp = a.v + krow * a.v_tok + (int64_t)item.kv_head * a.v_head + 8 * h;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
      kf[ks] = ld8(kp + 16 * ks);
      vf[ks] = ld8(vp + 16 * ks);
    }
  }
  const float sl2 = positive_scale(a.scale * kLog2e, kf);
  const TileReader rd(lane);
  float16v dk[4], dv[4];  // [key = k0w + 8 (r / 4) + 4 h + r % 4][d = 32 dt + col]
#pragma unroll
  for (int dt = 0; dt < 4; ++dt) {
    dk[dt] = float16v{};
    dv[dt] = float16v{};
  }

  // A masked entry is P = 0 whatever its query's statistic is: a query with a NaN score has
  // a NaN lse, which keys that it does not attend to must not see (exp2(-inf - 0) instead).
  auto mask = [&](float16v& s, float (&lse)[16], int qs) {
    if (qs < k0w + 31 || qs + 32 > len)  // the diagonal or the row's end
      mask_rows(s, mykey - qs - 4 * h, len - qs - 4 * h, lse);
  };
  // P and dS of elements 2 k and 2 k + 1.
  auto elements = [&](const float16v& s, const float16v& dp, const float (&lse)[16],
                      Packed8 (&p)[2], Packed8 (&ds)[2], int k) {
    const float p0 = exp2_hw(__builtin_fmaf(s[2 * k], sl2, -lse[2 * k]));
    const float p1 = exp2_hw(__builtin_fmaf(s[2 * k + 1], sl2, -lse[2 * k + 1]));
    round2(p[k >> 2], k, p0, p1);
    round2(ds[k >> 2], k, p0 * dp[2 * k], p1 * dp[2 * k + 1]);
  };
  // S and dP - delta of 32 queries, [q][key = mykey]; then dV += P^T . dO and dK += dS^T .
  // Q.  Whole tiles run one half's products over the other's element-wise step (the forward
  // and dQ have theirs in one piece between the products).
  auto compute = [&](int qt, const unsigned char* buf) {
    const unsigned char* sQ = buf;
    const unsigned char* sO = buf + kTileBytes;
    const float* sL = reinterpret_cast<const float*>(buf + 2 * kTileBytes);
    const int h0 = PARTS == 2 ? part : 0;
    auto stats = [&](int half, float (&lse)[16], float16v& dp) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float4v l4 = *reinterpret_cast<const float4v*>(sL + 32 * half + 8 * j + 4 * h);
        const float4v d4 = *reinterpret_cast<const float4v*>(sL + 64 + 32 * half + 8 * j + 4 * h);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          lse[4 * j + i] = l4[i];
          dp[4 * j + i] = d4[i];
        }
      }
    };
    Packed8 p[2][2], ds[2][2];
    float lse[2][16];
    float16v s[2], e[2];
    stats(h0, lse[0], e[0]);
    if (PARTS == 1) stats(1, lse[1], e[1]);
    // Operands of a half: Q and dO rows (8 k steps), then dO and Q along the queries.
    // Whole tiles run the scores of both halves first, then the sums: the element-wise
    // step of one half runs between the MFMAs of the other.
    constexpr int kN = 64 / PARTS, kHalf = kN / 2;
    stream_operands<kN, 8>(
        [&](auto pos) {
          constexpr int i = pos, st = (i % 16) / 2;
          const int half = h0 + (i % kHalf) / 16;
          if constexpr (i >= kHalf)
            return rd.tr(i & 1 ? sQ : sO, 2 * half + st / 4, st % 4);
          else
            return rd.row(i & 1 ? sO : sQ, half, st);
        },
        [&](auto pos, half8 f) {
          constexpr int i = pos, b = (i % kHalf) / 16, st = (i % 16) / 2;
          if constexpr (i >= kHalf) {
            if constexpr (i & 1)
              dk[st % 4] = mfma(operand(ds[b][st / 4]), f, dk[st % 4]);
            else
              dv[st % 4] = mfma(operand(p[b][st / 4]), f, dv[st % 4]);
          } else if constexpr (i & 1) {
            e[b] = mfma(f, vf[st], e[b]);
            if constexpr (st == 7) mask(s[b], lse[b], qt + 32 * (h0 + b));
          } else {
            s[b] = mfma(f, kf[st], st == 0 ? float16v{} : s[b]);
          }
          if constexpr (PARTS == 1 && (i & 1)) {
            if constexpr (i >= 16 && i < 32) elements(s[0], e[0], lse[0], p[0], ds[0], st);
            if constexpr (i >= 32 && i < 48) elements(s[1], e[1], lse[1], p[1], ds[1], st);
          }
          if constexpr (PARTS == 2 && i == 15) {
#pragma unroll
            for (int k = 0; k < 8; ++k) elements(s[0], e[0], lse[0], p[0], ds[0], k);
          }
        });
  };

  auto step = [&](int qt, int buf) {
    tile_barrier();
    if (qt + kTile < len) issue(qt + kTile, buf ^ 1);
    // Not when every query is before this wave's keys or past the row's end.
    const int first = qt + (PARTS == 2 ? 32 * part : 0), past = qt + (PARTS == 2 ? 32 * part + 32 : 64);
    if (past > k0w && first < len) compute(qt, smem + buf * kBuf);
  };
  for (int qt = k0; qt < len; qt += 2 * kTile) {
    step(qt, 0);
    if (qt + kTile < len) step(qt + kTile, 1);
  }
  if constexpr (PARTS == 2) {
    static_assert(G * 2 * kTileBytes <= 2 * kBuf, "exchange");
    unsigned char* at = smem + (wave % G) * 2 * kTileBytes;
    tile_barrier();
    if (part) {
      put_acc(at, dk, lane);
      put_acc(at + kTileBytes, dv, lane);
    }
    __syncthreads();
    if (part) return;
    add_acc(at, dk, 1.f, 1.f, lane);
    add_acc(at + kTileBytes, dv, 1.f, 1.f, lane);
  }
  const bool direct = a.hq == a.hk;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int key = k0w + 8 * (r >> 2) + 4 * h + (r & 3);
    if (key >= len) continue;
    if (direct) {
      half_t* kb = a.dk + (int64_t)item.kv_head * a.dk_head + (int64_t)(start + key) * a.dk_tok;
      half_t* vb = a.dv + (int64_t)item.kv_head * a.dv_head + (int64_t)(start + key) * a.dv_tok;
#pragma unroll
      for (int dt = 0; dt < 4; ++dt) {
        kb[dt * 32 + col] = f32_to_f16(dk[dt][r] * a.scale);
        vb[dt * 32 + col] = f32_to_f16(dv[dt][r]);
      }
    } else {
      float* kp = part_k + ((int64_t)item.head * a.total + start + key) * kD;
      float* vp = part_v + ((int64_t)item.head * a.total + start + key) * kD;
#pragma unroll
      for (int dt = 0; dt < 4; ++dt) {
        kp[dt * 32 + col] = dk[dt][r];
        vp[dt * 32 + col] = dv[dt][r];
      }
    }
  }
}

}  // namespace
}  // namespace ss

#include "attention_rows16.h"

namespace ss {
namespace {

// dK / dV of a GQA group: the q heads' fp32 partials added in head order
// (deterministic), dK scaled; four consecutive d per thread.
__global__ __launch_bounds__(256) void attn_bwd_reduce_kernel(AttnArgs a, const float* part_k,
                                                              const float* part_v) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;  // (token, kv head, d / 4)
  const int64_t per_tok = (int64_t)a.hk * (kD / 4);
  if (i >= a.total * per_tok) return;
  const int64_t t = i / per_tok;
  const int kvh = (int)((i % per_tok) / (kD / 4));
  const int d = (int)(i % (kD / 4)) * 4;
  const int group = a.hq / a.hk;
  float4v sk = float4v{0.f, 0.f, 0.f, 0.f}, sv = float4v{0.f, 0.f, 0.f, 0.f};
  for (int hh = 0; hh < group; ++hh) {
    const int64_t off = ((int64_t)(kvh * group + hh) * a.total + t) * kD + d;
    sk += *reinterpret_cast<const float4v*>(part_k + off);
    sv += *reinterpret_cast<const float4v*>(part_v + off);
  }
  half4 ok, ov;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    ok[j] = f32_to_f16(sk[j] * a.scale);
    ov[j] = f32_to_f16(sv[j]);
  }
  *reinterpret_cast<half4*>(a.dk + t * a.dk_tok + (int64_t)kvh * a.dk_head + d) = ok;
  *reinterpret_cast<half4*>(a.dv + t * a.dv_tok + (int64_t)kvh * a.dv_head + d) = ov;
}

// Batches that the 16-row waves (attention_rows16.h) run faster, per step, by their longest
// row; us on 16-row against the better 32-row kernel, 12 q / 2 kv heads:
//   forward, 48: 4000 tokens in rows of 16 23.7 / 28.3, of 32 15.9 / 16.4, 2000 in rows of 48 7.4 /
//     10.5 (4000 14.0 / 12.7), 4000 in rows of 64 13.9 / 12.1;
//   dQ, 64: rows of 16 31.0 / 37.2, of 48 17.4 / 17.9, of 64 16.5 / 16.4 (16 / 16 heads 19.8 /
//     22.5), of 100 19.8 / 15.7;
//   dK / dV, 192: rows of 16 32.6 / 65, of 64 20.2 / 26.6, of 100 28.2 / 25.3 (at 1000 tokens 12.5 /
//     14.4), of 158 29.0 / 30.4 (7900 tokens 47.4 / 56.5), of 300 38.1 / 32.5;
// and rows up to 128 while 64-token blocks are at most 5/4 of the CUs, where the time is
// one workgroup's latency (300 tokens in rows of 100: forward 6.8 / 7.1, dQ 7.3 / 8.2; 1000 in
// rows of 100: dQ 7.6 / 9.9; 2000 11.8 / 12.3).
bool few_blocks(int64_t total, int hq) {
  return cdiv(total, kBlk) * hq * 4 <= 5 * (int64_t)device_cu_count();
}
bool rows16_fwd(int max_len, int64_t total, int hq) {
  return max_len <= 48 || (max_len <= 128 && few_blocks(total, hq));
}
bool rows16_dq(int max_len, int64_t total, int hq) {
  return max_len <= 64 || (max_len <= 128 && few_blocks(total, hq));
}
bool rows16_dkdv(int max_len) { return max_len <= 192; }

// Grid of the 16-row kernels.
dim3 rows16_grid(const AttnArgs& a, int max_len) {
  return dim3((unsigned)cdiv(max_len, kBlk), (unsigned)a.hq, (unsigned)a.rows);
}

// Blocks of 64 queries / keys with two waves for each 32 (<2, 2>) while such blocks (a row's
// last one half full) number at most 3/2 of the CUs, 2 of them for long rows, whose blocks
// are long chains of tiles; beyond that the chip is full and 128-token blocks read each
// tile for twice the rows.  Forward + backward, us, <2, 2> against <4, 1>: 12 q / 2 kv heads, rows
// of 300: 1500 tokens 50.0 / 49.8, 3000 80.1 / 64.4; rows of 1000: 2000 tokens 82.8 / 96.3, 3000
// 107.4 / 105.9, 4000 134.5 / 117.4; 16 / 16 heads, rows of 300: 1500 tokens 52.0 / 46.0, 3000 94.1 /
// 72.9, 3900 117.3 / 92.4; 28 / 4 heads, 1000 in rows of 500 66.4 / 67.6, one row of 1000 88.5 / 96.9.
bool short_batch(int64_t total, int rows, int max_len, int hq) {
  const int64_t blocks = (total / 64 + rows / 2) * hq;
  return blocks * 2 <= (max_len < 768 ? 3 : 4) * (int64_t)device_cu_count();
}

// Grid of the items (Item): all (block, row) positions, or with few rows as many as
// rows of these lengths can have; in two dimensions so that any number fits.
dim3 item_grid(const AttnArgs& a) {
  int64_t positions = (int64_t)a.blocks * a.rows;
  if (a.rows <= 64 && a.total / a.span + a.rows < positions)
    positions = a.total / a.span + a.rows;
  const int64_t items = cdiv(positions * a.hk, 8) * 8 * (a.hq / a.hk);
  const int64_t kWide = (int64_t)1 << 20;  // a multiple of 8: keeps the XCD numbering
  if (items <= kWide) return dim3((unsigned)items);
  return dim3((unsigned)kWide, (unsigned)cdiv(items, kWide));
}

bool al8(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

int check_common(const char* fn, int rows, int max_len, int hq, int hk, int head_dim,
                 int64_t total, const int* cu) {
  SS_CHECK_ARG(rows >= 0 && max_len >= 0 && total >= 0, "%s: negative sizes", fn);
  SS_CHECK_ARG(head_dim == kD, "%s: head_dim %d unsupported (only %d)", fn, head_dim, kD);
  SS_CHECK_ARG(hq > 0 && hk > 0 && hq % hk == 0, "%s: hq=%d must be a positive multiple of hk=%d",
               fn, hq, hk);
  SS_CHECK_ARG(rows <= 65535 && hq <= 65535, "%s: rows / heads exceed the grid", fn);
  SS_CHECK_ARG(rows == 0 || cu, "%s: null cu_seqlens", fn);
  return SS_OK;
}

// Token / head strides (elements) of a tensor must keep every 16-byte load aligned.
bool strides_ok(const void* p, int64_t tok, int64_t head) {
  return p && al8(p) && tok % 8 == 0 && head % 8 == 0;
}

}  // namespace
}  // namespace ss

using namespace ss;

extern "C" int ss_attn_varlen_fwd(const void* q, int64_t q_tok, int64_t q_head, const void* k,
                                  int64_t k_tok, int64_t k_head, const void* v, int64_t v_tok,
                                  int64_t v_head, const int* cu_seqlens, int rows, int max_len,
                                  int64_t total, int hq, int hk, int head_dim, float scale,
                                  void* o, int64_t o_tok, int64_t o_head, float* lse2,
                                  void* stream) {
  const char* fn = "ss_attn_varlen_fwd";
  int rc = check_common(fn, rows, max_len, hq, hk, head_dim, total, cu_seqlens);
  if (rc) return rc;
  if (rows == 0 || max_len == 0) return SS_OK;
  SS_CHECK_ARG(strides_ok(q, q_tok, q_head) && strides_ok(k, k_tok, k_head) &&
                   strides_ok(v, v_tok, v_head) && strides_ok(o, o_tok, o_head) && lse2,
               "%s: q/k/v/o need 16-byte aligned bases and strides that are multiples of 8", fn);
  AttnArgs a{};
  a.q = (const half_t*)q; a.q_tok = q_tok; a.q_head = q_head;
  a.k = (const half_t*)k; a.k_tok = k_tok; a.k_head = k_head;
  a.v = (const half_t*)v; a.v_tok = v_tok; a.v_head = v_head;
  a.out = (half_t*)o; a.out_tok = o_tok; a.out_head = o_head;
  a.lse2 = lse2; a.cu = cu_seqlens; a.total = total; a.hq = hq; a.hk = hk; a.scale = scale;
  a.rows = rows;
  const bool small = short_batch(total, rows, max_len, hq);
  a.span = small ? 64 : 128;
  a.blocks = (int)cdiv(max_len, a.span);
  hipStream_t st = (hipStream_t)stream;
  if (rows16_fwd(max_len, total, hq))
    hipLaunchKernelGGL(attn_fwd_rows16_kernel, rows16_grid(a, max_len), dim3(256), 0, st, a);
  else if (small)
    hipLaunchKernelGGL((attn_fwd_kernel<2, 2>), item_grid(a), dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL((attn_fwd_kernel<4, 1>), item_grid(a), dim3(256), 0, st, a);
  SS_CHECK_LAUNCH("attn_fwd_kernel");
  return SS_OK;
}

static size_t round256(size_t b) { return (b + 255) / 256 * 256; }

extern "C" size_t ss_attn_varlen_bwd_workspace_size(int hq, int hk, int64_t total) {
  if (hq <= 0 || hk <= 0 || total <= 0) return 0;
  const size_t delta = round256((size_t)hq * total * sizeof(float));
  const size_t part = hq == hk ? 0 : round256((size_t)hq * total * kD * sizeof(float));
  return delta + 2 * part;
}

extern "C" int ss_attn_varlen_bwd(const void* q, int64_t q_tok, int64_t q_head, const void* k,
                                  int64_t k_tok, int64_t k_head, const void* v, int64_t v_tok,
                                  int64_t v_head, const void* o, int64_t o_tok, int64_t o_head,
                                  const void* dout, int64_t do_tok, int64_t do_head,
                                  const float* lse2, const int* cu_seqlens, int rows, int max_len,
                                  int64_t total, int hq, int hk, int head_dim, float scale,
                                  void* dq, int64_t dq_tok, int64_t dq_head, void* dk,
                                  int64_t dk_tok, int64_t dk_head, void* dv, int64_t dv_tok,
                                  int64_t dv_head, void* workspace, size_t workspace_bytes,
                                  void* stream) {
  const char* fn = "ss_attn_varlen_bwd";
  int rc = check_common(fn, rows, max_len, hq, hk, head_dim, total, cu_seqlens);
  if (rc) return rc;
  if (rows == 0 || max_len == 0) return SS_OK;
  SS_CHECK_ARG(strides_ok(q, q_tok, q_head) && strides_ok(k, k_tok, k_head) &&
                   strides_ok(v, v_tok, v_head) && strides_ok(o, o_tok, o_head) &&
                   strides_ok(dout, do_tok, do_head) && strides_ok(dq, dq_tok, dq_head) &&
                   strides_ok(dk, dk_tok, dk_head) && strides_ok(dv, dv_tok, dv_head) && lse2,
               "%s: q/k/v/o/dO/dq/dk/dv need 16-byte aligned bases and strides that are "
               "multiples of 8", fn);
  const size_t need = ss_attn_varlen_bwd_workspace_size(hq, hk, total);
  SS_CHECK_ARG(workspace && workspace_bytes >= need && al8(workspace),
               "%s: workspace of %zu bytes (16-byte aligned) needed, %zu given", fn, need,
               workspace_bytes);
  AttnArgs a{};
  a.q = (const half_t*)q; a.q_tok = q_tok; a.q_head = q_head;
  a.k = (const half_t*)k; a.k_tok = k_tok; a.k_head = k_head;
  a.v = (const half_t*)v; a.v_tok = v_tok; a.v_head = v_head;
  a.o = (const half_t*)o; a.o_tok = o_tok; a.o_head = o_head;
  a.dout = (const half_t*)dout; a.do_tok = do_tok; a.do_head = do_head;
  a.out = (half_t*)dq; a.out_tok = dq_tok; a.out_head = dq_head;
  a.dk = (half_t*)dk; a.dk_tok = dk_tok; a.dk_head = dk_head;
  a.dv = (half_t*)dv; a.dv_tok = dv_tok; a.dv_head = dv_head;
  a.lse2 = const_cast<float*>(lse2);
  a.delta = static_cast<float*>(workspace);
  a.cu = cu_seqlens; a.total = total; a.hq = hq; a.hk = hk; a.scale = scale;
  char* base = static_cast<char*>(workspace) + round256((size_t)hq * total * sizeof(float));
  const size_t part = round256((size_t)hq * total * kD * sizeof(float));
  float* part_k = hq == hk ? nullptr : reinterpret_cast<float*>(base);
  float* part_v = hq == hk ? nullptr : reinterpret_cast<float*>(base + part);
  a.rows = rows;
  const bool small = short_batch(total, rows, max_len, hq);
  a.span = small ? 64 : 128;
  a.blocks = (int)cdiv(max_len, a.span);
  hipStream_t st = (hipStream_t)stream;
  if (rows16_dq(max_len, total, hq))
    hipLaunchKernelGGL(attn_bwd_dq_rows16_kernel, rows16_grid(a, max_len), dim3(256), 0, st, a);
  else if (small)
    hipLaunchKernelGGL((attn_bwd_dq_kernel<2, 2>), item_grid(a), dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL((attn_bwd_dq_kernel<4, 1>), item_grid(a), dim3(256), 0, st, a);
  SS_CHECK_LAUNCH("attn_bwd_dq_kernel");
  if (rows16_dkdv(max_len))
    hipLaunchKernelGGL(attn_bwd_dkdv_rows16_kernel, rows16_grid(a, max_len), dim3(256), 0, st, a,
                       part_k, part_v);
  else if (small)
    hipLaunchKernelGGL((attn_bwd_dkdv_kernel<2, 2>), item_grid(a), dim3(256), 0, st, a, part_k,
                       part_v);
  else
    hipLaunchKernelGGL((attn_bwd_dkdv_kernel<4, 1>), item_grid(a), dim3(256), 0, st, a, part_k,
                       part_v);
  SS_CHECK_LAUNCH("attn_bwd_dkdv_kernel");
  if (hq != hk) {
    const int64_t work = total * hk * (kD / 4);
    hipLaunchKernelGGL(attn_bwd_reduce_kernel, dim3((unsigned)cdiv(work, 256)), dim3(256), 0, st,
                       a, part_k, part_v);
    SS_CHECK_LAUNCH("attn_bwd_reduce_kernel");
  }
  return SS_OK;
}
