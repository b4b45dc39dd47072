// GEMM2 for a few rows per expert (64 < T <= kStreamT): C resident in LDS, W2 streamed past it.
//
// O = C W2_e^T (main.py:234-238) with at most a few dozen rows per expert is the time it takes to read W2
// once.  A plain DMA stream of the 32 experts' W2 (470 MB, this kernel's order, non-temporal) takes 71 us;
// the LDS-staged units of gemm_large.hip, which meet at a barrier every 64 K and drain their pipeline at
// each of their 3-4 units per CU, take 108 / 115 / 120 us at T = 128 / 333 / 512, these ones 83 / 88 / 100 us; with
// log-normal tokens, many of whose blocks take two terms, 166 against 100 us at T = 250 and 172 against 121 at T = 512.
//
// With many rows per expert the staged units are the better ones: past 32 rows a block's C does not fit LDS over all of
// K, past 64 W2 is streamed again.  What decides is how the pairs fall on the experts, which only the device
// knows: gemm2_short_kernel runs either (stream_plan has the rule).  Here
//
// * a workgroup (8 wavefronts, one per CU) takes a contiguous share of all (block, 128 output columns) units, block
//   by block (stream_plan);
// * a block's C (up to 64 rows x as much of K as fits 128 KB: all of it up to 32 rows, f16 hi term, both terms
//   if a row needs them) is copied to LDS once for all of the workgroup's units of the block;
// * each wavefront then streams its own 16 W2 rows of every unit through a register ring, whole 128-byte
//   lines with the non-temporal hint, transposed through its own LDS buffer: no barrier, and the ring runs on
//   from one unit into the next.
//
// Blocks whose rows do not fit LDS over all of K take several passes over it; a pass adds its sums to the fp32
// ones that the pass before it left in O.
//
// Two terms of C (see moefp8_device.h): a block takes both where a row took exact GEMM1 products or has a
// measured bound that asks for both (with by_estimate also where the row is of magnitude class 1, the rule of
// the grouped kernels): at least every row that the 128-row path gives both.
#pragma once
#include "moefp8_device.h"
#include "moefp8_launch.h"

namespace moefp8 {

constexpr int kStWaves = 8;
constexpr int kStThreads = 64 * kStWaves;
constexpr int kStCols = 16 * kStWaves;            // output columns per unit
constexpr int kStRows = 64;                       // rows per block
constexpr int kStDepth = 8;                       // K-blocks of W2 in flight per wavefront (64 VGPRs)
constexpr int kStShortDepth = 4;                  // the same where a pass holds only four
constexpr int kStCBytes = 128 * 1024;             // C in LDS
constexpr int kStPad = 16;                        // bytes between LDS rows of C, so that an MFMA operand read
                                                  // (16 rows, 64 bytes per lane group) has no bank conflicts

// K-blocks of `planes` = m-tiles x terms planes of 16 rows that fit LDS, a multiple of the ring depth.
__host__ __device__ constexpr int stream_depth(int planes) { return planes <= 4 ? kStDepth : kStShortDepth; }
__host__ __device__ constexpr int stream_kc(int planes) {
  const int fit = kStCBytes / (planes * 16 * 2 * kBlock);
  return fit - fit % stream_depth(planes);
}
static_assert(stream_kc(8) == kStShortDepth && stream_kc(4) == kStDepth, "a pass fills the ring");

struct StreamLds {
  uint8_t c[kStCBytes + 2 * kStRows * kStPad];
  uint8_t wtr[kStWaves][16 * kBlock];             // transpose buffers
  float sa[32 * 16];                              // row scales of C, [K-block of the pass][16 nt rows]
  int off[kEGlobal + 1];                          // rows before each expert
  int first[kEGlobal + 1];                        // cost per column, or chunks, before each expert
  int budget;                                     // of a chunk (0: shares by cost)
  int staged;                                     // the LDS-staged units do better
};

// One pass (K-blocks [kb0, kb0 + n)) over the units [u0, u1) of one block: rows row0 .. row0 + rows - 1 in NT
// m-tiles, unit u being output columns 128 u.  `first` and `last`: whether the pass starts and ends its sums.
template <bool kTwo, int NT>
__device__ __forceinline__ void stream_pass(const Problem& pb, const Plan& pl, const CHalf8& ch, StreamLds& sh, int e,
                                            int row0, int rows, int u0, int u1, int kb0, int n, bool first, bool last,
                                            float* __restrict__ obuf) {
  constexpr int kTerms = kTwo ? 2 : 1;
  const int H = pb.H, I = pb.I, KB = I / kBlock, HB = H / kBlock;
  int lane = lane_id();
  asm volatile("" : "+v"(lane));   // (addresses formed per pass, not kept across passes)
  const int wave = wave_index(), lr = lane & 15, kg = lane >> 4;
  const int stride = n * 2 * kBlock + kStPad, term = NT * 16 * stride;

  // W2: lane l loads 16-byte chunk l % 8 of rows l / 8 and 8 + l / 8 of the wavefront's 16.  The ring
  // takes the K-blocks of each unit padded to a multiple of its depth (a padding slot repeats the last
  // K-block and counts with weight scale 0), unit after unit; past the last unit it repeats that one.
  constexpr int D = stream_depth(NT * kTerms);
  const int np = (n + D - 1) / D * D;
  const int wr = lane >> 3, wc = lane & 7;
  const uint32_t woff = (uint32_t)wr * (uint32_t)I + (uint32_t)wc * 16u, wrow8 = 8u * (uint32_t)I;
  const uint8_t* wu = pb.w2 + ((size_t)e * H + (size_t)u0 * kStCols + 16 * wave) * I + (size_t)kb0 * kBlock;
  v4i B0[D], B1[D];
  int lk = 0, left = u1 - 1 - u0;   // next K-block to load, units after its own
  auto load = [&](int d) {
    const uint8_t* p = wu + (size_t)min(lk, n - 1) * kBlock;
    B0[d] = __builtin_nontemporal_load(reinterpret_cast<const v4i*>(p + woff));
    B1[d] = __builtin_nontemporal_load(reinterpret_cast<const v4i*>(p + (woff + wrow8)));
    const bool end = lk + 1 == np, more = end && left > 0;
    lk = end ? 0 : lk + 1;
    wu += more ? (size_t)kStCols * I : 0;
    left -= more ? 1 : 0;
  };
#pragma unroll
  for (int d = 0; d < D; d++) load(d);
  const float* s2p = pb.s2 + ((size_t)e * HB + u0) * KB + kb0 + min(lane, n - 1);
  float sw_next = lane < n ? *s2p : 0.f;

  // C and its scales: [term][row][K], 16-byte chunks, each row by whole lines
  {
    const int per_row = n * (2 * kBlock / 16), total = kTerms * rows * per_row;
    constexpr int kBatch = 8;
    for (int i0 = 0; i0 < total; i0 += kBatch * kStThreads) {
      v4i v[kBatch];
      int at[kBatch];
#pragma unroll
      for (int q = 0; q < kBatch; q++) {
        const int i = min(i0 + q * kStThreads + (int)threadIdx.x, total - 1);
        const int tr = i / per_row, c = i - tr * per_row, t = kTwo ? tr / rows : 0, r = tr - t * rows;
        const _Float16* src = (kTwo && t ? ch.lo16 : ch.hi) + (size_t)clamp_index(row0 + r, pl.pair_rows) * I +
                              (size_t)kb0 * kBlock + c * 8;
        v[q] = *reinterpret_cast<const v4i*>(src);
        at[q] = t * term + r * stride + c * 16;
      }
#pragma unroll
      for (int q = 0; q < kBatch; q++)
        if (i0 + q * kStThreads + (int)threadIdx.x < total) *reinterpret_cast<v4i*>(sh.c + at[q]) = v[q];
    }
    for (int i = threadIdx.x; i < rows * n; i += kStThreads) {
      const int r = i / n, k = i - r * n;
      sh.sa[k * (16 * NT) + r] = ch.scale[(size_t)clamp_index(row0 + r, pl.pair_rows) * KB + kb0 + k];
    }
  }
  // each m-tile's row of this lane (rows past the block's last repeat it: computed, never stored)
  int rt[NT];
  float w[NT];
#pragma unroll
  for (int i = 0; i < NT; i++) {
    rt[i] = min(16 * i + lr, rows - 1);
    w[i] = last ? pl.perm_w[clamp_index(row0 + rt[i], pl.pair_rows)] : 1.0f;
  }
  // (waited for here, once, and not by every unit's first step)
  asm volatile("" : "+v"(sw_next));
  __syncthreads();

  uint8_t* const tb = sh.wtr[wave];
  uint8_t* const tw0 = tb + wr * kBlock + (wc ^ slot_key8(wr)) * 16;
  uint8_t* const tw1 = tb + (wr + 8) * kBlock + (wc ^ slot_key8(wr + 8)) * 16;
  const uint8_t* const trx = tb + lr * kBlock + ((2 * kg) ^ slot_key8(lr)) * 16;
  const uint8_t* const try_ = tb + lr * kBlock + ((2 * kg + 1) ^ slot_key8(lr)) * 16;
  v4i bx, by;
  auto transpose = [&](int d) {
    *reinterpret_cast<v4i*>(tw0) = B0[d];
    *reinterpret_cast<v4i*>(tw1) = B1[d];
    bx = *reinterpret_cast<const v4i*>(trx);
    by = *reinterpret_cast<const v4i*>(try_);
  };
  constexpr bool kAhead = NT * kTerms <= 2;
  v8h a_next[kAhead ? NT : 1][kAhead ? 4 * kTerms : 1];
  auto c_at = [&](int i, int kc) { return sh.c + rt[i] * stride + kc * (2 * kBlock) + kg * 64; };
  auto read_c = [&](int k) {
#pragma unroll
    for (int i = 0; i < (kAhead ? NT : 0); i++)
#pragma unroll
      for (int t = 0; t < 4 * kTerms; t++)
        a_next[i][t] = *reinterpret_cast<const v8h*>(c_at(i, min(k, n - 1)) + 16 * (t & 3) + (t >> 2) * term);
  };
  transpose(0);
  load(0);
  read_c(0);
  for (int u = u0; u < u1; u++) {
    const float sw_v = sw_next;
    s2p += u + 1 < u1 ? KB : 0;
    sw_next = lane < n ? *s2p : 0.f;
    float* const orow = obuf + (size_t)u * kStCols + 16 * wave + 4 * kg;
    v4f acc[NT], part[NT];
#pragma unroll
    for (int i = 0; i < NT; i++) acc[i] = v4f{0.f, 0.f, 0.f, 0.f};
    if (!first) {
#pragma unroll
      for (int i = 0; i < NT; i++)
        part[i] = *reinterpret_cast<const v4f*>(orow + (size_t)clamp_index(row0 + rt[i], pl.pair_rows) * H);
    }
    // K-block k from the transposed W2 in (bx, by); the next one's (ring slot d) is transposed meanwhile, and
    // its C read where registers allow (kAhead), so that a step waits for no LDS round trip of its own
    auto step = [&](int d, int k) {
      const int kc = min(k, n - 1);
      const float sw = readlane_f32(sw_v, k);
      v8h b16[4];
      widen_fp8_operand(__builtin_shufflevector(bx, by, 0, 1, 2, 3, 4, 5, 6, 7), b16);
      v8h a[kAhead ? NT : 1][kAhead ? 4 * kTerms : 1];
      if constexpr (kAhead) {
#pragma unroll
        for (int i = 0; i < NT; i++)
#pragma unroll
          for (int t = 0; t < 4 * kTerms; t++) a[i][t] = a_next[i][t];
      }
      transpose(d);
      load(d);
      if constexpr (kAhead) read_c(k + 1 == np ? 0 : k + 1);
      // (m-tiles inside: consecutive MFMAs are independent)
      v4f p[NT];
#pragma unroll
      for (int t = 0; t < 4 * kTerms; t++) {
#pragma unroll
        for (int i = 0; i < NT; i++) {
          v8h x;
          if constexpr (kAhead) x = a[i][t];
          else x = *reinterpret_cast<const v8h*>(c_at(i, kc) + 16 * (t & 3) + (t >> 2) * term);
          p[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b16[t & 3], x, t == 0 ? v4f{0.f, 0.f, 0.f, 0.f} : p[i], 0, 0, 0);
        }
      }
#pragma unroll
      for (int i = 0; i < NT; i++) {
        const float s = sh.sa[kc * (16 * NT) + rt[i]] * sw;
#pragma unroll
        for (int r = 0; r < 4; r++) acc[i][r] += p[i][r] * s;
      }
    };
    for (int k = 0; k < np; k += D) {
#pragma unroll
      for (int d = 0; d < D; d++) {
        step((d + 1) % D, k + d);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (!first) {
#pragma unroll
      for (int i = 0; i < NT; i++) acc[i] += part[i];
    }
    // (rows past the last store its values again)
#pragma unroll
    for (int i = 0; i < NT; i++)
      *reinterpret_cast<v4f*>(orow + (size_t)clamp_index(row0 + rt[i], pl.pair_rows) * H) =
          v4f{acc[i][0] * w[i], acc[i][1] * w[i], acc[i][2] * w[i], acc[i][3] * w[i]};
  }
  // the next pass or block restages only after every wavefront has read this one's rows (and its sums in O
  // are written)
  __syncthreads();
}

// Blocks of an expert's n rows: the fewest of at most kStRows rows, of about equal height (steps of 16).
struct StreamBlocks {
  int n, q, r;
  StreamBlocks() = default;
  __device__ __forceinline__ explicit StreamBlocks(int rows) {
    const int tiles = (rows + 15) / 16;
    n = (tiles + kStRows / 16 - 1) / (kStRows / 16);
    q = n > 0 ? (int)((float)tiles * __builtin_amdgcn_rcpf((float)n) + 0.001f) : 0;   // (tiles <= 256, n <= 64)
    r = tiles - n * q;
  }
  __device__ __forceinline__ int first(int j) const { return 16 * (j * q + min(j, r)); }
  // Time of a unit of nt m-tiles, one for which W2's stream sets it being 2: taller ones stage more C per unit
  // and run longer MFMA chains (equal shares instead took a call of T = 300 at zipf routing 159 us, not 146).
  static __device__ __forceinline__ int cost(int nt) { return nt <= 1 ? 2 : 2 * nt - 1; }
  __device__ __forceinline__ int total() const { return r * cost(q + 1) + (n - r) * cost(q); }
  // The block that cost `at` (of a column) falls in, and the cost before it.
  __device__ __forceinline__ int block_at(int at, int* before) const {
    const int tall = r * cost(q + 1);
    const int j = at < tall ? at / cost(q + 1) : r + (at - tall) / cost(q);
    *before = j < r ? j * cost(q + 1) : tall + (j - r) * cost(q);
    return j;
  }
};

// How the workgroups share the units (block, 128 columns).
//
// By cost (budget 0): each takes the units that start in its equal part of the cost line, columns innermost, so that
// it meets one or two blocks and every CU the same work to within one unit.
//
// By chunks (budget > 0): each takes one run of units of one block, of at most `budget` cost.  A second block costs a
// workgroup another start (the decision on C's terms, C's copy to LDS, the first W2 lines: ~4 us, about
// kStartCost / KB of the cost scale), which a call of a few units per workgroup does not earn back: chosen where the
// smallest budget whose chunks the grid holds is within one start of the equal part.  Calls by cost alone and so, 32
// experts, H = 2048, I = 768: T = 65 / 80 / 127 with 8 / 4 / 4 local pairs per token 66.4 -> 61.9, 64.2 -> 58.7, 65.3
// -> 60.3 us; H = 7168, I = 2048: T = 333 with 1 pair 258.4 -> 257.6.
constexpr int kStartCost = 13;
struct StreamChunks {
  int tall, low;              // units per chunk of the expert's blocks of q + 1 and of q m-tiles
  int per_tall, per_low, n;   // chunks per block of each height, and of the expert
  __device__ __forceinline__ StreamChunks(const StreamBlocks& sb, int budget, int NC) {
    // (quotients of integers below 2^12 in fp32, the offset above the rounding and below the least remainder)
    auto units = [&](int nt) {
      return max(1, min(NC, (int)((float)budget * __builtin_amdgcn_rcpf((float)StreamBlocks::cost(nt)) + 0.01f)));
    };
    auto chunks = [&](int len) { return (int)((float)(NC + len - 1) * __builtin_amdgcn_rcpf((float)len) + 0.001f); };
    tall = units(sb.q + 1);
    low = units(sb.q);
    per_tall = chunks(tall);
    per_low = chunks(low);
    n = sb.r * per_tall + (sb.n - sb.r) * per_low;
  }
};

// Fills sh.off and, from the experts' row counts, sh.staged (with staged_ok) and for the stream sh.first and sh.budget
// (all threads; ends with a barrier).
//
// The staged units are taken where their rounds over the grid, (5 KB + 20) of 128-K steps each (KB K-blocks and what a
// unit costs besides), are no more than the stream's equal share of cost in its padded K-blocks, a quarter more
// for an expert with rows of two-term C, and 8 for its start and 32 for each further pass over K of its tallest block: a
// fit to both kernels' times over 418 calls (1 to 256 local experts, H 512 to 8192, I 256 to 4096, T = 128 to 512, 1 to
// 8 local pairs per token, normal and log-normal tokens, zipf; the weights not in a cache), on average 0.3% above the
// better of the two.  Calls of one round lean to the stream: 16 experts, H = 2048, I = 1024, T = 512 61 us against 65,
// zipf T = 256, 6 pairs 48 and 53; 8 experts, H = 2048, I = 2048, T = 512 76 and 82.  H = 7168, I = 2048,
// 32 experts, calls by the stream and by the staged units: T = 128, 1 pair 245 and 275 us; 256, 3 pairs 284 and 298;
// 333, 2 pairs 283 and 295; 333, 4 pairs 325 and 317; 512, 4 pairs 400 and 347; 512, 8 pairs 546 and 436; zipf T = 512,
// 1501 pairs 288 and 243.  256 experts, I = 256, log-normal, T = 256 391 and 488 (each expert has blocks of both kinds);
// 16 experts of H = 8192, I = 4096, log-normal, T = 128, 4 pairs 463 and 405.
__device__ __forceinline__ void stream_plan(const Problem& pb, const Plan& pl, StreamLds& sh, bool staged_ok) {
  const int KB = pb.I / kBlock, NC = pb.H / kStCols, E = pb.E_local, G = (int)gridDim.x;
  constexpr int kPer = kEGlobal / kWave;   // experts per lane
  int2 ctl[kPer];                          // one- and two-term rows of each
  if (staged_ok) {
#pragma unroll
    for (int i = 0; i < kPer; i++) ctl[i] = reinterpret_cast<const int2*>(pl.g2_ctl)[min(i * kWave + lane_id(), E - 1)];
  }
  for (int i = threadIdx.x; i <= E; i += kStThreads) sh.off[i] = pl.expert_offsets[i];
  __syncthreads();
  if (threadIdx.x < kWave) {
    const int lane = (int)threadIdx.x;
    StreamBlocks sb[kPer];
#pragma unroll
    for (int i = 0; i < kPer; i++) {
      const int e = min(i * kWave + lane, E - 1);
      if (i * kWave < E) sb[i] = StreamBlocks(i * kWave + lane < E ? sh.off[e + 1] - sh.off[e] : 0);
    }
    // sum over the experts of a whole number below 2^24 in all
    auto sum = [&](auto&& value) {
      int v = 0;
#pragma unroll
      for (int i = 0; i < kPer; i++)
        if (i * kWave < E) v += value(sb[i]);
      return (int)wave_sum_f32((float)v);
    };
    const int cost = sum([](const StreamBlocks& b) { return b.total(); });
    int staged = 0;
    if (staged_ok && cost > 0) {
      // of this lane's experts: the staged units' blocks; four times the cost, five with two-term rows; and the most
      // planes of C in a block
      int blocks = 0, weighted = 0, planes = 0;
#pragma unroll
      for (int i = 0; i < kPer; i++) {
        if (i * kWave >= E || sb[i].n == 0) continue;
        const bool two = ctl[i].y > 0;
        blocks += (ctl[i].x + kGemm2Rows - 1) / kGemm2Rows + (ctl[i].y + kGemm2Rows - 1) / kGemm2Rows;
        weighted += (two ? 5 : 4) * sb[i].total();
        planes = max(planes, (two ? 2 : 1) * (sb[i].r > 0 ? sb[i].q + 1 : sb[i].q));
      }
      const int units = (int)wave_sum_f32((float)blocks) * (pb.H / 256);
      const int rounds = (int)((uint32_t)(units + G - 1) / (uint32_t)G);   // of the staged units over the grid
      const int padded = (KB + kStDepth - 1) / kStDepth * kStDepth, share = (int)wave_sum_f32((float)weighted) * NC;
      const uint32_t kc = (uint32_t)stream_kc((int)wave_max_u32((uint32_t)planes));
      const int again = (int)(((uint32_t)KB + kc - 1) / kc) - 1;   // passes over K after the first
      staged = share * padded + 4 * (8 + 32 * again) * G >= 4 * rounds * (5 * KB + 20) * G ? 1 : 0;
    }
    int budget = 0;
    if (!staged) {
      const int most = (int)((uint32_t)(cost * NC * KB + kStartCost * G) / (uint32_t)(G * KB));
      for (int b = max(1, (int)((uint32_t)(cost * NC + G - 1) / (uint32_t)G)); b <= most; b++) {
        if (sum([&](const StreamBlocks& x) { return StreamChunks(x, b, NC).n; }) <= G) {
          budget = b;
          break;
        }
      }
      int carry = 0;
#pragma unroll
      for (int i = 0; i < kPer; i++) {
        if (i * kWave >= E) continue;
        const int c = budget > 0 ? StreamChunks(sb[i], budget, NC).n : sb[i].total();
        const int f = carry + wave_exclusive_sum(c);
        if (i * kWave + lane < E) sh.first[i * kWave + lane] = f;
        carry = __builtin_amdgcn_readlane(f + c, kWave - 1);
      }
      if (lane == 0) sh.first[E] = carry;
    }
    if (lane == 0) {
      sh.budget = budget;
      sh.staged = staged;
    }
  }
  __syncthreads();
}

// This workgroup's units (all threads).
__device__ __forceinline__ void gemm2_stream_units(const Problem& pb, const Plan& pl, const CHalf8& ch, StreamLds& sh,
                                                   float* __restrict__ obuf, int by_estimate) {
  const int I = pb.I, KB = I / kBlock, NC = pb.H / kStCols, E = pb.E_local;
  // Consecutive shares run on one XCD, so that the blocks of an expert share its W2 through that XCD's L2.
  const int G = (int)gridDim.x, nx = G % 8 == 0 ? 8 : 1;
  const int share = ((int)blockIdx.x % nx) * (G / nx) + (int)blockIdx.x / nx;
  // by cost, the units that start in [v, v1) of the cost line; by chunks, the chunk in [v, v1) if any (no more than
  // workgroups, spread over all XCDs)
  const int budget = uniform(sh.budget), width = budget > 0 ? 1 : NC;
  // (at most 512 m-tiles of cost 2 in 64 columns: 32 bits hold the products)
  const uint32_t total = (uint32_t)sh.first[E] * width;
  const int v1 = (int)(total * (share + 1) / (uint32_t)G);
  int v = (int)(total * share / (uint32_t)G);
  while (v < v1) {
    // the expert of v (the last that starts at or before it; empty ones share their successor's start), its
    // block there and the block's units in the share
    int lo = 0, hi = E;
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (sh.first[mid] * width <= v) lo = mid;
      else hi = mid;
    }
    const int e = uniform(lo), n_rows = sh.off[e + 1] - sh.off[e];
    const StreamBlocks sb(n_rows);
    int j, u0, u1;
    if (budget > 0) {
      const StreamChunks sc(sb, budget, NC);
      const int at = v - sh.first[e], tall = sb.r * sc.per_tall;
      const int per = at < tall ? sc.per_tall : sc.per_low, len = at < tall ? sc.tall : sc.low;
      const int jj = (at < tall ? at : at - tall) / per, piece = (at < tall ? at : at - tall) - jj * per;
      j = at < tall ? jj : sb.r + jj;
      u0 = uniform(piece * len);
      u1 = uniform(min(NC, piece * len + len));
      v = v1;
    } else {
      int before;
      j = sb.block_at((v - sh.first[e] * NC) / NC, &before);
      const int cost = StreamBlocks::cost(j < sb.r ? sb.q + 1 : sb.q), start = (sh.first[e] + before) * NC;
      u0 = uniform((v - start + cost - 1) / cost);
      u1 = uniform(min(NC, (v1 - start + cost - 1) / cost));
      v = start + cost * NC;
    }
    const int r0 = sb.first(j);
    const int row0 = uniform(sh.off[e] + r0), rows = uniform(min(sb.first(j + 1), n_rows) - r0);
    if (u0 >= u1) continue;
    // both terms of C where a row of the block needs them
    bool need = row0 + rows > pl.xrow[e];
    {
      const float sigma13 = pl.esig[2 * e], sigma2 = pl.esig[2 * e + 1], sqrt_i = sqrtf((float)I);
      if (by_estimate && (int)threadIdx.x < rows) {
        const int p = clamp_index(row0 + (int)threadIdx.x, pl.pair_rows), t = clamp_index(pl.perm_token[p], pb.T);
        need |= predicted_output_rms(pl.tok_a2[t], pl.perm_w[p], sigma13, sigma2, sqrt_i) > kOneTermRms;
      }
      for (int i = threadIdx.x; i < rows * KB; i += kStThreads) {
        const int p = clamp_index(row0 + i / KB, pl.pair_rows);
        need |= needs_two_terms(pl.perm_w[p], sigma2, 448.0f * ch.scale[(size_t)p * KB + i % KB], sqrt_i);
      }
    }
    const bool two = uniform(__syncthreads_or(need)) != 0;
    const int nt = uniform((rows + 15) / 16), kc = stream_kc(nt * (two ? 2 : 1));
    for (int kb0 = 0; kb0 < KB; kb0 += kc) {
      const int n = min(kc, KB - kb0);
#define MOEFP8_STREAM(TWO, NT) \
  stream_pass<TWO, NT>(pb, pl, ch, sh, e, row0, rows, u0, u1, kb0, n, kb0 == 0, kb0 + n == KB, obuf)
      if (two) {
        if (nt == 1) MOEFP8_STREAM(true, 1);
        else if (nt == 2) MOEFP8_STREAM(true, 2);
        else if (nt == 3) MOEFP8_STREAM(true, 3);
        else MOEFP8_STREAM(true, 4);
      } else {
        if (nt == 1) MOEFP8_STREAM(false, 1);
        else if (nt == 2) MOEFP8_STREAM(false, 2);
        else if (nt == 3) MOEFP8_STREAM(false, 3);
        else MOEFP8_STREAM(false, 4);
      }
#undef MOEFP8_STREAM
    }
  }
}

}  // namespace moefp8
