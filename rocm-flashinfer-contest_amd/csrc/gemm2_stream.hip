// GEMM2 for a few rows per expert (64 < T <= kStreamT): C resident in LDS, W2 streamed past it.
//
// O = C W2_e^T (main.py:234-238) with at most a few dozen rows per expert is the time it takes to read W2
// once.  A plain DMA stream of the 32 experts' W2 (470 MB, this kernel's order, non-temporal) takes 71 us;
// the LDS-staged kernel of gemm_large.hip, which meets at a barrier every 64 K and drains its pipeline at
// each of its 3-4 units per CU, takes 108 / 115 / 120 us at T = 128 / 333 / 512 (with the row
// table's launch, 7 us, before it), this one 83 / 88 / 100 us; with log-normal tokens, many of whose blocks take
// two terms, 166 against 100 us at T = 250 and 172 against 121 at T = 512.  Past kStreamT = 512 the blocks of hot
// experts need several passes over K, each restaging 128 KB of C: at zipf routing calls of T = 400 / 512 take 182 /
// 205 us against 188 / 207, and would take 230 against 217 at T = 700.  Here
//
// * a workgroup (8 wavefronts, one per CU) takes an equal, contiguous share of all (block, 128 output columns)
//   units, block by block, so that it meets one or two blocks in all and every CU the same work to within
//   one of about seven units;
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
  __device__ __forceinline__ explicit StreamBlocks(int rows) {
    const int tiles = (rows + 15) / 16;
    n = (tiles + kStRows / 16 - 1) / (kStRows / 16);
    q = n > 0 ? tiles / n : 0;
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

__global__ __launch_bounds__(kStThreads, 1) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm2_stream_kernel(
    Problem pb, Plan pl, CHalf8 ch, float* __restrict__ obuf, int by_estimate) {
  __shared__ __attribute__((aligned(16))) StreamLds sh;
  __shared__ int off_s[kEGlobal + 1], first_s[kEGlobal + 1];   // rows, and cost per column, before each expert
  const int I = pb.I, KB = I / kBlock, NC = pb.H / kStCols, E = pb.E_local;
  for (int i = threadIdx.x; i <= E; i += kStThreads) off_s[i] = pl.expert_offsets[i];
  __syncthreads();
  if (threadIdx.x < kWave) {
    int carry = 0;
    for (int e0 = 0; e0 < E; e0 += kWave) {
      const int e = e0 + (int)threadIdx.x;
      const int c = e < E ? StreamBlocks(off_s[e + 1] - off_s[e]).total() : 0;
      const int f = carry + wave_exclusive_sum(c);
      if (e < E) first_s[e] = f;
      carry = __builtin_amdgcn_readlane(f + c, kWave - 1);
    }
    if (threadIdx.x == 0) first_s[E] = carry;
  }
  __syncthreads();
  // this workgroup's share of the units (block, 128 columns), columns innermost, by cost: the units that
  // start in [v, v1) of the cost line.  Consecutive shares run on one XCD, so that the blocks of an expert share
  // its W2 through that XCD's L2.
  const int G = (int)gridDim.x, nx = G % 8 == 0 ? 8 : 1;
  const int share = ((int)blockIdx.x % nx) * (G / nx) + (int)blockIdx.x / nx;
  const int64_t total = (int64_t)first_s[E] * NC;
  const int v1 = (int)(total * (share + 1) / G);
  int v = (int)(total * share / G);
  while (v < v1) {
    // the expert of cost v (the last that starts at or before it; empty ones share their successor's start),
    // its block there and the block's units in the share
    int lo = 0, hi = E;
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (first_s[mid] * NC <= v) lo = mid;
      else hi = mid;
    }
    const int e = uniform(lo), n_rows = off_s[e + 1] - off_s[e];
    const StreamBlocks sb(n_rows);
    int before;
    const int j = sb.block_at((v - first_s[e] * NC) / NC, &before);
    const int r0 = sb.first(j);
    const int row0 = uniform(off_s[e] + r0), rows = uniform(min(sb.first(j + 1), n_rows) - r0);
    const int cost = StreamBlocks::cost(j < sb.r ? sb.q + 1 : sb.q), start = (first_s[e] + before) * NC;
    const int u0 = uniform((v - start + cost - 1) / cost), u1 = uniform(min(NC, (v1 - start + cost - 1) / cost));
    v = start + cost * NC;
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

void launch_gemm2_stream(const Problem& pb, const Plan& pl, const CHalf8& ch, float* obuf, bool by_estimate,
                         hipStream_t stream) {
  hipLaunchKernelGGL(gemm2_stream_kernel, dim3(num_compute_units()), dim3(kStThreads), 0, stream, pb, pl, ch, obuf,
                     by_estimate ? 1 : 0);
}

}  // namespace moefp8
