// The cell list's entries grouped by cell, for the adjoint: a stable radix
// sort of digits up to 11 bits whose first pass reads the ILCell list itself
// (no key or value array is written for it) and whose last pass writes keys
// and values apart.
//
// A pass counts the digits of every tile of 8,192 entries (one row of 2^bits
// counters per tile), turns the counters into the tiles' output offsets by a
// scan down the columns, and scatters: each wavefront ranks 64 entries at a
// time among equal digits (ballots) over its own counters in LDS, the
// block's wavefronts are chained per digit, the tile's entries go into digit
// order in LDS and from there out, so that a digit's entries leave side by
// side. No tile waits on another. Cells of up to 22 bits take two passes.
//
// What bounds it is memory: about 8 bytes in and 8 out per entry and pass
// (2.9-3.3 TB/s in the scatters). 5.8e8 entries over 22 bits: scatters 3.3 +
// 2.8 ms, counts 1.9, scans 0.7, against 3 x 3.8 ms for the library's
// onesweep sort of 8-bit digits behind 2.1 ms that wrote its keys and
// values. Writing each entry straight from its lane, without the order in
// LDS, took 2.8 + 7.7 ms: neighbouring lanes then store to different digits.
// 16 entries per lane (one block per CU) instead of 8 (two) 4% slower.
#pragma once
#include "common.h"

namespace cgpu {

constexpr int kTrBlock = 1024;
constexpr int kTrWaves = kTrBlock / kWave;
constexpr int kTrRounds = 8;                       // entries per lane
constexpr int kTrTile = kTrBlock * kTrRounds;       // entries per tile (places fit 16 bits)
static_assert(kTrTile <= 1 << 16, "places");
constexpr int kTrWaveTile = kWave * kTrRounds;      // of which a wavefront takes this many in a row
constexpr int kTrMaxBits = 11;
constexpr int kTrMaxDigits = 1 << kTrMaxBits;
constexpr int kTrRows = 512;  // rows the column scan takes at once; more tiles are summed in rows

// value of an entry: bucket << kBucketShift | offsetID bits 31..22 (replica
// and softened flag; bits 21..0 carry no information for a cell entry)
constexpr int kBucketShift = 10;

struct TrSource {
  const ILCell* cells;  // first pass: the list and its bucket marks
  const int* marks;
  int nb;
  const uint2* packed;  // later passes: (key, value)
};

// Tiles go to the XCDs in contiguous ranges (xcd_bucket): a digit's runs of
// neighbouring tiles are neighbours in memory, and lines that one L2 holds
// are written back whole.
// Digit counts of a tile into its row of counts.
template <bool FIRST>
__global__ __launch_bounds__(kTrBlock) void tr_count_kernel(TrSource src, int n, int shift,
                                                            int bits, int* counts) {
  __shared__ int cnt[kTrMaxDigits];
  const int nd = 1 << bits;
  for (int d = threadIdx.x; d < nd; d += kTrBlock) cnt[d] = 0;
  __syncthreads();
  const int row = xcd_bucket(blockIdx.x, gridDim.x);
  const size_t tile = (size_t)row * kTrTile;
  const unsigned left = (unsigned)(n - (long long)tile);  // of the list from this tile on
  const ILCell* cells = FIRST ? src.cells + tile : nullptr;
  const uint2* packed = FIRST ? nullptr : src.packed + tile;
  unsigned key[kTrRounds];
#pragma unroll
  for (int r = 0; r < kTrRounds; ++r) {
    const unsigned e = threadIdx.x + r * kTrBlock;
    key[r] = 0;
    if (e < left) key[r] = FIRST ? (unsigned)cells[e].index : packed[e].x;
  }
  // neighbours often share their digit: one atomic per run of equal ones
  const int lane = threadIdx.x & (kWave - 1);
#pragma unroll
  for (int r = 0; r < kTrRounds; ++r) {
    const bool valid = threadIdx.x + r * kTrBlock < left;
    const int d = valid ? (int)((key[r] >> shift) & (unsigned)(nd - 1)) : -1;
    const int before = __shfl_up(d, 1, kWave);  // (every lane takes part)
    const bool head = lane == 0 || before != d;
    const unsigned long long later = __ballot(head) & ~((2ull << lane) - 1ull);
    if (head && valid) atomicAdd(&cnt[d], (later ? __ffsll((long long)later) - 1 : kWave) - lane);
  }
  __syncthreads();
  for (int d = threadIdx.x; d < nd; d += kTrBlock)
    counts[(size_t)row * nd + d] = cnt[d];
}

// Column sums of `per` rows of counts into row blockIdx.x of sums.
__global__ __launch_bounds__(kTrBlock) void tr_row_sums_kernel(const int* counts, int rows,
                                                               int per, int nd, int* sums) {
  const int r0 = blockIdx.x * per, r1 = min(rows, r0 + per);
  for (int d = threadIdx.x; d < nd; d += kTrBlock) {
    int s = 0;
#pragma unroll 8
    for (int r = r0; r < r1; ++r) s += counts[(size_t)r * nd + d];
    sums[(size_t)blockIdx.x * nd + d] = s;
  }
}

// Rows of counts (rows <= kTrRows) -> exclusive sums down the columns, in
// place, and the columns' totals. One thread per digit.
__global__ __launch_bounds__(kWave) void tr_columns_kernel(int* counts, int rows, int nd,
                                                           int* total) {
  const int d = blockIdx.x * kWave + threadIdx.x;
  if (d >= nd) return;
  int at = 0;
  int r = 0;
  constexpr int U = 32;  // rows in flight
  for (; r + U <= rows; r += U) {
    int v[U];
#pragma unroll
    for (int k = 0; k < U; ++k) v[k] = counts[(size_t)(r + k) * nd + d];
#pragma unroll
    for (int k = 0; k < U; ++k) {
      counts[(size_t)(r + k) * nd + d] = at;
      at += v[k];
    }
  }
  for (; r < rows; ++r) {
    const int v = counts[(size_t)r * nd + d];
    counts[(size_t)r * nd + d] = at;
    at += v;
  }
  total[d] = at;
}

// Digit totals -> the digits' first places, in place. One block.
__global__ __launch_bounds__(kTrBlock) void tr_digits_kernel(int* total, int nd) {
  __shared__ int wave_sum[kTrWaves];
  constexpr int D = kTrMaxDigits / kTrBlock;  // digits per thread, consecutive
  const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
  int v[D], sum = 0;
#pragma unroll
  for (int k = 0; k < D; ++k) {
    const int d = threadIdx.x * D + k;
    v[k] = d < nd ? total[d] : 0;
    sum += v[k];
  }
  int incl = sum;
#pragma unroll
  for (int m = 1; m < kWave; m <<= 1) {
    const int y = __shfl_up(incl, m, kWave);
    if (lane >= m) incl += y;
  }
  if (lane == kWave - 1) wave_sum[wv] = incl;
  __syncthreads();
  int run = incl - sum;
  for (int w = 0; w < wv; ++w) run += wave_sum[w];
#pragma unroll
  for (int k = 0; k < D; ++k) {
    const int d = threadIdx.x * D + k;
    if (d < nd) total[d] = run;
    run += v[k];
  }
}

// Offsets of the rows blockIdx.x stands for, from its row of sums (offsets).
__global__ __launch_bounds__(kTrBlock) void tr_offsets_kernel(int* counts, int rows, int per,
                                                              int nd, const int* sums) {
  const int r0 = blockIdx.x * per, r1 = min(rows, r0 + per);
  for (int d = threadIdx.x; d < nd; d += kTrBlock) {
    int at = sums[(size_t)blockIdx.x * nd + d];
#pragma unroll 8
    for (int r = r0; r < r1; ++r) {
      int* c = counts + (size_t)r * nd + d;
      const int v = *c;
      *c = at;
      at += v;
    }
  }
}

// Entries of a tile to their places: its row of counts holds its offset
// within each digit's entries, digit_base the digits' first places. LAST: keys and values to arrays of their own, else packed.
template <bool FIRST, bool LAST>
__global__ __launch_bounds__(kTrBlock) __attribute__((amdgpu_waves_per_eu(8))) void tr_scatter_kernel(TrSource src, int n, int shift,
                                                              int bits, const int* counts,
                                                              const int* digit_base, uint2* out, unsigned* key_out,
                                                              unsigned* val_out) {
  // the wavefronts' digit counters, then the tile's entries in digit order
  __shared__ uint2 lds[kTrTile];
  unsigned short(*cnt)[kTrMaxDigits] = reinterpret_cast<unsigned short(*)[kTrMaxDigits]>(lds);
  static_assert(sizeof(lds) >= sizeof(unsigned short) * kTrWaves * kTrMaxDigits, "counters");
  __shared__ int offset[kTrMaxDigits];
  __shared__ int wave_sum[kTrWaves];
  const int nd = 1 << bits;
  const unsigned dmask = (unsigned)(nd - 1);
  const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
  const int row = xcd_bucket(blockIdx.x, gridDim.x);
  for (int d = threadIdx.x; d < nd; d += kTrBlock) {
    offset[d] = counts[(size_t)row * nd + d] + digit_base[d];
#pragma unroll
    for (int w = 0; w < kTrWaves; ++w) cnt[w][d] = 0;
  }
  const size_t tile = (size_t)row * kTrTile;
  const unsigned left = (unsigned)(n - (long long)tile);  // of the list from this tile on
  const unsigned e0 = wv * kTrWaveTile + lane;            // this lane's first entry in the tile
  uint2 kv[kTrRounds];
  if constexpr (FIRST) {
    const ILCell* cells = src.cells + tile;
#pragma unroll
    for (int r = 0; r < kTrRounds; ++r) {
      ILCell c = {0, 0};
      if (e0 + r * kWave < left) c = cells[e0 + r * kWave];
      kv[r] = make_uint2((unsigned)c.index, (unsigned)c.offsetID);
    }
    // the bucket of the wavefront's first entry (the last one that begins at
    // or before it), then each lane steps on from its entry to its next one
    const int first = (int)min((long long)tile + wv * kTrWaveTile, (long long)n - 1);
    int lo = 0, hi = src.nb;  // marks[lo] <= first < marks[hi]; 64 probes a step
    while (hi - lo > 1) {
      const int step = (hi - lo + kWave - 1) / kWave;
      const int at = lo + lane * step;
      const int k = __popcll(__ballot(at < hi && src.marks[min(at, hi)] <= first)) - 1;
      lo += max(k, 0) * step;
      hi = min(hi, lo + step);
    }
    int b = lo, next = src.marks[lo + 1];
#pragma unroll
    for (int r = 0; r < kTrRounds; ++r) {
      if (e0 + r * kWave < left) {
        const long long e = (long long)tile + e0 + r * kWave;
        while (e >= next && b + 1 < src.nb) next = src.marks[++b + 1];
      }
      kv[r].y = ((unsigned)b << kBucketShift) | (kv[r].y >> 22);
    }
  } else {
    const uint2* packed = src.packed + tile;
#pragma unroll
    for (int r = 0; r < kTrRounds; ++r) {
      kv[r] = make_uint2(0, 0);
      if (e0 + r * kWave < left) kv[r] = packed[e0 + r * kWave];
    }
  }
  __syncthreads();
  // rank within the wavefront's entries of the same digit, 64 at a time
  const unsigned long long below = (1ull << lane) - 1ull;
  unsigned rank[kTrRounds / 2] = {};  // two of 16 bits in each
#pragma unroll
  for (int r = 0; r < kTrRounds; ++r) {
    const bool valid = e0 + r * kWave < left;
    const unsigned d = (kv[r].x >> shift) & dmask;
    unsigned long long same = __ballot(valid);
    for (int k = 0; k < bits; ++k) {
      const bool bit = (d >> k) & 1u;
      const unsigned long long m = __ballot(bit);
      same &= bit ? m : ~m;
    }
    const int before = __popcll(same & below);
    int at = 0;
    if (valid) {
      at = cnt[wv][d];
      if (before == 0) cnt[wv][d] = (unsigned short)(at + __popcll(same));
    }
    rank[r / 2] |= (unsigned)(at + before) << (16 * (r & 1));
    __builtin_amdgcn_sched_barrier(0);  // one round's ballots in registers at a time
  }
  __syncthreads();
  // chain the wavefronts per digit, and the digits: a counter becomes the
  // place of its wavefront's first entry of the digit within the tile, an
  // offset the distance from there to the place in the output
  constexpr int D = kTrMaxDigits / kTrBlock;  // digits per thread, consecutive
  int count[D], sum = 0;
#pragma unroll
  for (int k = 0; k < D; ++k) {
    const int d = threadIdx.x * D + k;
    count[k] = 0;
    if (d < nd)
#pragma unroll
      for (int w = 0; w < kTrWaves; ++w) count[k] += cnt[w][d];
    sum += count[k];
  }
  int incl = sum;
#pragma unroll
  for (int m = 1; m < kWave; m <<= 1) {
    const int y = __shfl_up(incl, m, kWave);
    if (lane >= m) incl += y;
  }
  if (lane == kWave - 1) wave_sum[wv] = incl;
  __syncthreads();
  int run = incl - sum;
  for (int w = 0; w < wv; ++w) run += wave_sum[w];
#pragma unroll
  for (int k = 0; k < D; ++k) {
    const int d = threadIdx.x * D + k;
    if (d < nd) {
      offset[d] -= run;
      int at = run;
#pragma unroll
      for (int w = 0; w < kTrWaves; ++w) {
        const int v = cnt[w][d];
        cnt[w][d] = (unsigned short)at;
        at += v;
      }
    }
    run += count[k];
  }
  __syncthreads();
  // entries into digit order (their places first: the counters share the
  // memory), then out, neighbours of a digit side by side
#pragma unroll
  for (int r = 0; r < kTrRounds; r += 2) {
    unsigned p = rank[r / 2];
    if (e0 + r * kWave < left) p += cnt[wv][(kv[r].x >> shift) & dmask];
    if (e0 + (r + 1) * kWave < left)
      p += (unsigned)cnt[wv][(kv[r + 1].x >> shift) & dmask] << 16;
    rank[r / 2] = p;
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kTrRounds; ++r)
    if (e0 + r * kWave < left) lds[(rank[r / 2] >> (16 * (r & 1))) & 0xffffu] = kv[r];
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kTrRounds; ++r) {
    const unsigned i = threadIdx.x + r * kTrBlock;
    if (i >= left) continue;
    const uint2 v = lds[i];
    const size_t at = (size_t)(offset[(v.x >> shift) & dmask] + (int)i);
    if constexpr (LAST) {
      key_out[at] = v.x;
      val_out[at] = v.y;
    } else {
      out[at] = v;
    }
  }
}

// Passes and digit bits of the sort of keys below 2^end_bit.
struct TrPlan {
  int passes, bits, tiles, per, rows;  // rows > 0: tiles summed `per` at a time into `rows` rows
};

static inline TrPlan tr_plan(long long n, int end_bit) {
  TrPlan p;
  p.passes = (end_bit + kTrMaxBits - 1) / kTrMaxBits;
  if (p.passes < 1) p.passes = 1;
  p.bits = (end_bit + p.passes - 1) / p.passes;
  if (p.bits < 1) p.bits = 1;
  p.tiles = (int)((n + kTrTile - 1) / kTrTile);
  p.per = (p.tiles + kTrRows - 1) / kTrRows;
  p.rows = p.tiles > kTrRows ? (p.tiles + p.per - 1) / p.per : 0;
  return p;
}

// ints of the counter scratch
static inline size_t tr_count_ints(const TrPlan& p) {
  return (size_t)(p.tiles + p.rows + 1) << p.bits;
}

// Groups the n entries of the list by cell, each cell's in list order: buf0 and buf1 hold 2 n ints each;
// *key and *value return the grouped arrays (in one of them). counts:
// tr_count_ints. The highest digit goes first (the groups then follow one
// another in the order of their lowest digit): neighbouring buckets list
// mostly the same cells, so that either pass finds runs of equal digits (1%
// faster in all than the lowest first).
static int tr_sort(const ChangaGravityLaunch& pc, int n, int end_bit, int* buf0, int* buf1,
                   int* counts, const unsigned** key, const unsigned** value, hipStream_t s) {
  const TrPlan p = tr_plan(n, end_bit);
  const int nd = 1 << p.bits;
  int* sums = counts + ((size_t)p.tiles << p.bits);
  int* digits = sums + ((size_t)p.rows << p.bits);
  TrSource src = {static_cast<const ILCell*>(pc.list), pc.marks, pc.numBuckets, nullptr};
  const dim3 tiles(p.tiles), block(kTrBlock);
  for (int k = 0; k < p.passes; ++k) {
    const int shift = (p.passes - 1 - k) * p.bits;
    const bool first = k == 0, last = k == p.passes - 1;
    int* to = (k & 1) ? buf1 : buf0;
    uint2* out = reinterpret_cast<uint2*>(to);
    unsigned* ko = reinterpret_cast<unsigned*>(to);
    unsigned* vo = ko + n;
    hipLaunchKernelGGL(first ? tr_count_kernel<true> : tr_count_kernel<false>, tiles, block, 0, s,
                       src, n, shift, p.bits, counts);
    CGPU_CHECK(hipGetLastError());
    if (p.rows) {
      hipLaunchKernelGGL(tr_row_sums_kernel, dim3(p.rows), block, 0, s, counts, p.tiles, p.per, nd,
                         sums);
      CGPU_CHECK(hipGetLastError());
    }
    hipLaunchKernelGGL(tr_columns_kernel, dim3((nd + kWave - 1) / kWave), dim3(kWave), 0, s,
                       p.rows ? sums : counts, p.rows ? p.rows : p.tiles, nd, digits);
    CGPU_CHECK(hipGetLastError());
    hipLaunchKernelGGL(tr_digits_kernel, dim3(1), block, 0, s, digits, nd);
    CGPU_CHECK(hipGetLastError());
    if (p.rows) {
      hipLaunchKernelGGL(tr_offsets_kernel, dim3(p.rows), block, 0, s, counts, p.tiles, p.per, nd,
                         sums);
      CGPU_CHECK(hipGetLastError());
    }
    const auto scatter = first ? (last ? tr_scatter_kernel<true, true>
                                       : tr_scatter_kernel<true, false>)
                               : (last ? tr_scatter_kernel<false, true>
                                       : tr_scatter_kernel<false, false>);
    hipLaunchKernelGGL(scatter, tiles, block, 0, s, src, n, shift, p.bits, counts, digits, out,
                       ko, vo);
    CGPU_CHECK(hipGetLastError());
    src.packed = out;
    *key = ko;
    *value = vo;
  }
  return 0;
}

}  // namespace cgpu
