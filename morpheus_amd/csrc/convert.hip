// convert.hip -- on-GPU format conversion, bit-exact with the reference
// Serial converters (core/src/impl/<Fmt>/Serial/Morpheus_Convert_Impl.hpp),
// which the reference HIP backend does not provide (it throws
// NotImplementedException, core/src/impl/Csr/HIP/Morpheus_Convert_Impl.hpp:39-76).
//
// Conversion is pure indexing, so every step is a histogram, a prefix sum,
// a compaction or a scatter:
//  * the sequential "walks" of the Serial code become prefix sums over flag
//    arrays (entry positions) and over run heads (position of an entry inside
//    its run of equal row indices, the row_id/n walk of the ELL and HYB
//    converters);
//  * where the Serial code can write one slot twice (repeated (row, col)
//    entries, rows split into several runs) the later entry in input order
//    wins, reproduced with an atomicMax on the entry index per slot;
//  * the stable (row, col) sort of core/src/impl/Coo/Serial/
//    Morpheus_Sort_Impl.hpp:111-166 is a stable LSD radix sort (8-bit
//    digits, per-tile counts, ranks from wave ballots), skipped when the
//    entries are already sorted, as in the reference;
//  * values are moved as raw bits; the zero test of DIA -> COO (which drops
//    +0.0 and -0.0) is a test of the bits without the sign.
#include <algorithm>
#include <vector>

#include "mph_internal.hpp"

namespace mph {

namespace {

constexpr int kT = 256;

inline unsigned blocks_for(int64_t n, int per = kT) {
  return (unsigned)std::max<int64_t>(1, ceil_div(n, per));
}

// ------------------------------------------------------------- raw values
template <int B>
struct RawT;
template <>
struct RawT<2> {
  using T = uint16_t;
  static constexpr T mag = 0x7fffu;
};
template <>
struct RawT<4> {
  using T = uint32_t;
  static constexpr T mag = 0x7fffffffu;
};
template <>
struct RawT<8> {
  using T = uint64_t;
  static constexpr T mag = 0x7fffffffffffffffull;
};

// ------------------------------------------------------------- small kernels
__global__ void fill_i32_kernel(int32_t* p, int64_t n, int32_t v) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// Histogram of non-negative int32 keys: a workgroup counts kHItems entries
// per thread into an LDS hash table (linear probing, kHProbe steps) and
// adds the table to cnt once; keys that find no slot go to cnt directly.
// Sorted COO entries hit few distinct rows / diagonals per workgroup (a
// 27-point stencil: 27 diagonals), which a global atomic per entry
// serialised (109M adds on 27 counters took 49 ms).
constexpr int kHSlots = 1024;
constexpr int kHItems = 16;
constexpr int kHProbe = 8;

template <typename KeyFn>
__device__ __forceinline__ void lds_histogram(int64_t n, int32_t* __restrict__ cnt, KeyFn key) {
  __shared__ int32_t hk[kHSlots];
  __shared__ int32_t hc[kHSlots];
  for (int q = threadIdx.x; q < kHSlots; q += blockDim.x) {
    hk[q] = -1;
    hc[q] = 0;
  }
  __syncthreads();
  const int64_t base = (int64_t)blockIdx.x * blockDim.x * kHItems + threadIdx.x;
  for (int k = 0; k < kHItems; k++) {
    const int64_t i = base + (int64_t)k * blockDim.x;
    if (i >= n) break;
    const int32_t kk = key(i);
    const uint32_t h = ((uint32_t)kk * 2654435761u) >> 22;  // 10 bits
    bool done = false;
    for (int p = 0; p < kHProbe && !done; p++) {
      const uint32_t q = (h + p) & (kHSlots - 1);
      int32_t cur = hk[q];
      if (cur == -1) cur = atomicCAS(&hk[q], -1, kk);
      if (cur == -1 || cur == kk) {
        atomicAdd(&hc[q], 1);
        done = true;
      }
    }
    if (!done) atomicAdd(&cnt[kk], 1);
  }
  __syncthreads();
  for (int q = threadIdx.x; q < kHSlots; q += blockDim.x)
    if (hc[q] > 0) atomicAdd(&cnt[hk[q]], hc[q]);
}

inline unsigned hist_blocks(int64_t n) { return (unsigned)ceil_div(n, (int64_t)kT * kHItems); }

__global__ __launch_bounds__(kT) void row_hist_kernel(const int32_t* __restrict__ ri, int64_t nnz,
                                                      int32_t* __restrict__ cnt) {
  lds_histogram(nnz, cnt, [&](int64_t i) { return ri[i]; });
}

// Reductions to one word: a workgroup strides over the array, reduces in
// registers and LDS, and adds its result with one atomic.  An atomic per
// element on one address was served one at a time: the maxima of 14.6M COO
// indices took 2.6 ms, now about 15 us (the 58 MB read at the stream rate).
constexpr int64_t kReduceBlocks = 256;  // (2048 spent 20 us on the atomics, 512 10)
inline unsigned reduce_blocks(int64_t n) {
  return (unsigned)std::min<int64_t>(blocks_for(n, 4 * kT), kReduceBlocks);
}

template <typename T, typename Op>
__device__ __forceinline__ T block_reduce(T v, Op op) {
  __shared__ T part[kT / kWave];
  for (int d = kWave / 2; d > 0; d >>= 1) v = op(v, shfl_xor(v, d));
  __syncthreads();  // (the previous reduction's partials are read)
  if (threadIdx.x % kWave == 0) part[threadIdx.x / kWave] = v;
  __syncthreads();
  v = part[0];
  for (int w = 1; w < kT / kWave; w++) v = op(v, part[w]);
  return v;
}

// the largest of a[0, n) and 0
__global__ __launch_bounds__(kT) void max_kernel(const int32_t* __restrict__ a, int64_t n,
                                                 int32_t* __restrict__ out) {
  const int64_t step = (int64_t)gridDim.x * kT;
  int32_t m = 0;
  for (int64_t i = (int64_t)blockIdx.x * kT + threadIdx.x; i < n; i += step) m = max(m, a[i]);
  m = block_reduce(m, [](int32_t u, int32_t v) { return max(u, v); });
  if (threadIdx.x == 0 && m > 0) atomicMax(out, m);
}

// sum over rows of min(cnt[r], K)
__global__ __launch_bounds__(kT) void clipped_sum_kernel(const int32_t* __restrict__ cnt,
                                                         int64_t n, int32_t K,
                                                         unsigned long long* out) {
  const int64_t step = (int64_t)gridDim.x * kT;
  unsigned long long t = 0;
  for (int64_t i = (int64_t)blockIdx.x * kT + threadIdx.x; i < n; i += step)
    t += (unsigned long long)min(cnt[i], K);
  t = block_reduce(t, [](unsigned long long u, unsigned long long v) { return u + v; });
  if (threadIdx.x == 0 && t > 0) atomicAdd(out, t);
}

// first index p > 0 with ri[p] < ri[p-1] (rows decrease), else n
__global__ void first_descent_kernel(const int32_t* __restrict__ ri, int64_t n,
                                     int32_t* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= 1 && i < n && ri[i] < ri[i - 1]) atomicMin(out, (int32_t)i);
}

// One pass over the entries of a COO list: index ranges, the order of the
// entries, and (rows not decreasing) the row offsets, whose slots ro[prev + 1
// .. r] entry i fills when its row r differs from the entry before it.  Reads
// 8 B an entry once, where the range checks, the sortedness test and a row
// histogram (an LDS hash table: 6 ps an entry) each were a pass.  With
// indices out of range, or rows that decrease, ro is incomplete; every write
// stays inside it.  More than kFarGap rows without an entry are left out and
// raise kGaps, for gap_offsets_kernel: filled here, each by the lane or wave
// that met it, the gaps of rows in no order came to a third of the rows an
// entry (2M shuffled entries on 1M rows 127 ms), and one gap of 4M rows took
// 1.8 ms.  (The COO part of a power-law HYB has gaps of more than 32 rows, none
// that far: left out too, they cost the other kernel 40 us on 1M rows.)
constexpr int32_t kBadRow = 1, kBadCol = 2, kRowsDown = 4, kUnsorted = 8, kRepeated = 16,
                  kGaps = 32;
constexpr int kScanPer = 8;  // entries per thread
constexpr int kScanTile = kT * kScanPer;
constexpr uint32_t kLongGap = 32, kFarGap = 1024;

// The `gap` rows up to `row` start at entry i: by the lane, long gaps by the
// whole wave, unless one of its lanes saw rows decrease (ro is not used then).
__device__ __forceinline__ void fill_offsets(int32_t* __restrict__ ro, int32_t row, uint32_t gap,
                                             int32_t i, bool down, int32_t& bad) {
  const bool lng = gap > kLongGap;
  if (!lng) {
    int32_t* p = ro + row - gap;
    for (uint32_t k = 1; k <= gap; k++) p[k] = i;
  }
  uint64_t m = __ballot(lng && gap <= kFarGap);
  if (lng && gap > kFarGap) bad |= kGaps;
  if (m == 0 || __ballot(down) != 0) return;
  const int lane = threadIdx.x % kWave;
  while (m) {
    const int src = __ffsll((unsigned long long)m) - 1;
    m &= m - 1;
    int32_t* p = ro + (int64_t)shfl(row, src) - shfl(gap, src);
    const uint32_t n = shfl(gap, src);
    const int32_t at = shfl(i, src);
    for (uint32_t k = 1 + lane; k <= n; k += kWave) p[k] = at;
  }
}

// Sets the bits of `bad` that any thread of the workgroup has; a word that
// already holds them is not written again (unsorted entries would all hit one
// address; even reading it once a wave took 15 us for 9.2M of them).
__device__ __forceinline__ void raise_flags(int32_t* __restrict__ flags, int32_t bad) {
  __shared__ int32_t all;
  __syncthreads();
  if (threadIdx.x == 0) all = 0;
  __syncthreads();
  for (int d = kWave / 2; d > 0; d >>= 1) bad |= shfl_xor(bad, d);
  if (bad && threadIdx.x % kWave == 0) atomicOr(&all, bad);
  __syncthreads();
  if (threadIdx.x == 0 && all &&
      (__hip_atomic_load(flags, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & all) != all)
    atomicOr(flags, all);
}

// Marks the bits of keys in a bitmap (lanes with `need` set; every lane of
// the wave calls it).  A workgroup gathers its keys in an LDS table (linear
// probing, kSeenProbe steps), equal keys of a wave entered once for its first
// kMatchRounds distinct ones; keys that find no slot mark their bit at once.  mark_bits_flush then sets the
// table's bits that are not yet set: a stencil's few diagonals would
// otherwise queue up on a few words (about 11 ns for each wave's atomic on
// one address; 117 us for 14.6M entries when each wave read and set its bits
// itself, 52 us so).
constexpr int kSeen = 2 * kT;
constexpr int kSeenProbe = 4;
constexpr int kMatchRounds = 8;
__device__ __forceinline__ uint32_t seen_slot(int32_t key) {
  return ((uint32_t)key * 2654435761u) >> 23;  // 9 bits
}

__device__ __forceinline__ void set_bit(uint32_t* __restrict__ bits, int32_t key) {
  const uint32_t bit = 1u << (key & 31);
  if (!(__hip_atomic_load(&bits[key >> 5], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & bit))
    atomicOr(&bits[key >> 5], bit);
}

__device__ __forceinline__ void enter_key(uint32_t* __restrict__ bits, int32_t* seen, int32_t key) {
  const uint32_t slot = seen_slot(key);
  for (int p = 0; p < kSeenProbe; p++) {
    const uint32_t q = (slot + p) & (kSeen - 1);
    int32_t cur = seen[q];
    if (cur == -1) {
      const int32_t old = atomicCAS(&seen[q], -1, key);
      cur = old == -1 ? key : old;
    }
    if (cur == key) return;
  }
  set_bit(bits, key);
}

__device__ __forceinline__ void mark_bits(uint32_t* __restrict__ bits, int32_t* seen, int32_t key,
                                          bool need) {
  const int lane = threadIdx.x % kWave;
  const uint32_t slot = seen_slot(key);
#pragma unroll
  for (int p = 0; p < kSeenProbe; p++) need = need && seen[(slot + p) & (kSeen - 1)] != key;
  uint64_t m = __ballot(need);
  for (int round = 0; m && round < kMatchRounds; round++) {
    const int src = __ffsll((unsigned long long)m) - 1;
    const int32_t k = shfl(key, src);
    if (lane == src) enter_key(bits, seen, k);
    if (key == k) need = false;
    m = __ballot(need);
  }
  if (need) enter_key(bits, seen, key);
}

__device__ __forceinline__ void mark_bits_flush(uint32_t* __restrict__ bits, const int32_t* seen) {
  __syncthreads();
  for (int q = threadIdx.x; q < kSeen; q += kT)
    if (seen[q] >= 0) set_bit(bits, seen[q]);
}

// Adds keys to counters cnt, the same way: counts gather in the workgroup's
// table and reach memory once; equal keys of a wave are added together for
// the first kMatchRounds distinct ones, the other lanes add themselves.  Few
// workgroups take many tiles each (kCountBlocks), since every workgroup's
// atomic on a stencil's counters waits its turn.
constexpr int64_t kCountBlocks = 1024;
__device__ __forceinline__ void add_key(int32_t* __restrict__ cnt, int32_t* hk, int32_t* hc,
                                        int32_t key, int32_t n) {
  const uint32_t slot = seen_slot(key);
  for (int p = 0; p < kSeenProbe; p++) {
    const uint32_t q = (slot + p) & (kSeen - 1);
    int32_t cur = hk[q];
    if (cur == -1) {
      const int32_t old = atomicCAS(&hk[q], -1, key);
      cur = old == -1 ? key : old;
    }
    if (cur == key) {
      atomicAdd(&hc[q], n);
      return;
    }
  }
  atomicAdd(&cnt[key], n);
}

__device__ __forceinline__ void count_keys(int32_t* __restrict__ cnt, int32_t* hk, int32_t* hc,
                                           int32_t key, bool need) {
  const int lane = threadIdx.x % kWave;
  uint64_t m = __ballot(need);
  for (int round = 0; m && round < kMatchRounds; round++) {
    const int src = __ffsll((unsigned long long)m) - 1;
    const int32_t k = shfl(key, src);
    const uint64_t same = __ballot(need && key == k);
    if (lane == src) add_key(cnt, hk, hc, k, __popcll(same));
    if (key == k) need = false;
    m &= ~same;
  }
  if (need) add_key(cnt, hk, hc, key, 1);
}

// What coo_scan_kernel also gathers: the bitmap of the diagonals used, a
// count per diagonal, or the bits that any row / any column from 0 has
// (flags[1] / flags[2]: as wide as the largest index, without a maximum pass).
enum DiagMode { kNoDiags, kDiagBits, kDiagCounts, kWidths };

template <bool COLS, bool OFFSETS, DiagMode DIAGS>
__global__ __launch_bounds__(kT) void coo_scan_kernel(
    const int32_t* __restrict__ ri, const int32_t* __restrict__ ci, int64_t nnz, int64_t nrows,
    int64_t ncols, int32_t* __restrict__ ro, uint32_t* __restrict__ diags,
    int32_t* __restrict__ flags) {
  __shared__ int32_t seen[kSeen];
  __shared__ int32_t seen_n[DIAGS == kDiagCounts ? kSeen : 1];
  if (DIAGS == kDiagBits || DIAGS == kDiagCounts) {
    for (int q = threadIdx.x; q < kSeen; q += kT) {
      seen[q] = -1;
      if (DIAGS == kDiagCounts) seen_n[q] = 0;
    }
    __syncthreads();
  }
  const int lane = threadIdx.x % kWave;
  int32_t bad = 0, wide_r = 0, wide_c = 0;
  int64_t last = -2;  // the last entry's row, in the lane that holds it
  for (int64_t tile = (int64_t)blockIdx.x * kScanTile; tile < nnz;
       tile += (int64_t)gridDim.x * kScanTile) {
    const int64_t base = tile + threadIdx.x;
    int32_t r[kScanPer], c[kScanPer];
#pragma unroll
    for (int k = 0; k < kScanPer; k++) {
      const int64_t i = base + (int64_t)k * kT;
      r[k] = i < nnz ? ri[i] : 0;
      c[k] = COLS && i < nnz ? ci[i] : 0;
    }
#pragma unroll
    for (int k = 0; k < kScanPer; k++) {
      const int64_t i = base + (int64_t)k * kT;
      int32_t pr = shfl_up(r[k], 1), pc = COLS ? shfl_up(c[k], 1) : 0;
      if (lane == 0 && i > 0 && i < nnz) {
        pr = ri[i - 1];
        if (COLS) pc = ci[i - 1];
      }
      const bool in = i < nnz;
      const bool row_ok = r[k] >= 0 && r[k] < nrows;
      const bool col_ok = !COLS || (c[k] >= 0 && c[k] < ncols);
      if (in) {
        wide_r |= r[k];
        wide_c |= max(c[k], 0);
        if (!row_ok) bad |= kBadRow;
        if (!col_ok) bad |= kBadCol;
        if (i > 0) {
          if (pr > r[k]) bad |= kRowsDown | kUnsorted | kRepeated;
          if (COLS && pr == r[k] && pc > c[k]) bad |= kUnsorted | kRepeated;
          if (COLS && pr == r[k] && pc == c[k]) bad |= kRepeated;
        }
      }
      if (OFFSETS) {
        const int32_t before = i == 0 ? -1 : max(pr, -1);
        const bool up = in && row_ok && before < r[k];
        fill_offsets(ro, r[k], up ? (uint32_t)r[k] - (uint32_t)before : 0u, (int32_t)i,
                     in && i > 0 && pr > r[k], bad);
        if (in && i == nnz - 1 && row_ok) last = r[k];
      }
      const int32_t key = (int32_t)((int64_t)c[k] - r[k] + nrows - 1);
      if (DIAGS == kDiagBits) mark_bits(diags, seen, key, in && row_ok && col_ok);
      if (DIAGS == kDiagCounts)
        count_keys(reinterpret_cast<int32_t*>(diags), seen, seen_n, key, in && row_ok && col_ok);
    }
  }
  if (OFFSETS && last >= -1) {  // the rows after the last entry's, by its lane
    if (nrows - last > kFarGap)
      bad |= kGaps;
    else
      for (int64_t q = last + 1; q <= nrows; q++) ro[q] = (int32_t)nnz;
  }
  raise_flags(flags, bad);
  if (DIAGS == kWidths) {
    raise_flags(flags + 1, wide_r);
    raise_flags(flags + 2, wide_c);
  }
  if (DIAGS == kDiagBits) mark_bits_flush(diags, seen);
  if (DIAGS == kDiagCounts) {
    __syncthreads();
    for (int q = threadIdx.x; q < kSeen; q += kT)
      if (seen_n[q] > 0) atomicAdd(reinterpret_cast<int32_t*>(diags) + seen[q], seen_n[q]);
  }
}

// The first entry from row r on of n entries in row order, by one wave, 64
// probes a round.
__device__ __forceinline__ int64_t wave_first_entry(const int32_t* __restrict__ ri, int64_t n,
                                                    int64_t r) {
  const int lane = threadIdx.x % kWave;
  int64_t lo = -1, hi = n;  // ri[lo] < r <= ri[hi]
  while (hi - lo > 1) {
    const int64_t step = (hi - lo - 1 + kWave - 1) / kWave;
    const int64_t at = lo + 1 + step * lane;
    const uint64_t lt = __ballot(at < hi && ri[at] < r);
    const int below = __popcll(lt);  // probes 0 .. below - 1
    const int64_t next = below < kWave ? min(hi, lo + 1 + step * below) : hi;
    if (below > 0) lo = lo + 1 + step * (below - 1);
    hi = next;
  }
  return hi;
}

// The row offsets of entries in row order that coo_scan_kernel left out rows
// of (flags, if given: its word; without kGaps, or with decreasing rows, there
// is nothing to do).  A workgroup takes kScanTile rows: the entries of all of
// them by two wave searches, and each row's first by a search among those.
__global__ __launch_bounds__(kT) void gap_offsets_kernel(const int32_t* __restrict__ ri, int64_t nnz,
                                                         int64_t nrows, int32_t* __restrict__ ro,
                                                         const int32_t* __restrict__ flags) {
  if (flags && (*flags & (kGaps | kRowsDown | kBadRow)) != kGaps) return;
  __shared__ int64_t ends[2];
  const int64_t base = (int64_t)blockIdx.x * kScanTile;
  const int64_t top = min(base + kScanTile, nrows + 1);  // rows [base, top)
  if (threadIdx.x < 2 * kWave) {
    const int64_t e = wave_first_entry(ri, nnz, threadIdx.x < kWave ? base : top - 1);
    if (threadIdx.x % kWave == 0) ends[threadIdx.x / kWave] = e;
  }
  __syncthreads();
  for (int64_t r = base + threadIdx.x; r < top; r += kT) {
    int64_t lo = ends[0], hi = ends[1];
    while (lo < hi) {
      const int64_t mid = (lo + hi) >> 1;
      if (ri[mid] < r) lo = mid + 1; else hi = mid;
    }
    ro[r] = (int32_t)lo;
  }
}

// rows of a CSR's entries, a workgroup per kScanTile of them: each row that
// starts in the tile marks its first entry in LDS (of rows without entries
// the last mark stays), a maximum scan spreads the marks, and the rows are
// written in order.  A binary search of the offsets per entry took 205 us for
// 14.6M entries (0.28 TB/s).  A tile that spans more rows than the marks are
// worth (long runs of empty rows) searches the offsets instead.
__global__ __launch_bounds__(kT) void expand_rows_kernel(const int32_t* __restrict__ ro,
                                                         int64_t nrows, int64_t nnz, int64_t shift,
                                                         int32_t* __restrict__ ri_out) {
  __shared__ int32_t mark[kScanTile];
  __shared__ int32_t wtop[kT / kWave];
  __shared__ int32_t ends[2];
  const int64_t base = (int64_t)blockIdx.x * kScanTile;
  const int n = (int)min((int64_t)kScanTile, nnz - base);
  if (threadIdx.x < 2 * kWave) {
    // the row of the tile's first / last entry, the last r with ro[r] <= j:
    // one wave each, 64 probes a round
    const int lane = threadIdx.x % kWave;
    const int64_t j = threadIdx.x < kWave ? base : base + n - 1;
    int64_t lo = 0, hi = nrows;  // ro[lo] <= j < ro[hi]
    while (hi - lo > 1) {
      const int64_t step = (hi - lo + kWave - 1) / kWave;
      const int64_t at = lo + step * lane;
      const uint64_t le = __ballot(at < hi && ro[at] <= j);
      const int top = 63 - __clzll((unsigned long long)le);
      lo += step * top;
      hi = min(hi, lo + step);
    }
    if (lane == 0) ends[threadIdx.x / kWave] = (int32_t)lo;
  }
  for (int q = threadIdx.x; q < kScanTile; q += kT) mark[q] = 0;
  __syncthreads();
  const int64_t r0 = ends[0], r1 = ends[1];
  if (r1 - r0 > 16 * kScanTile) {
    for (int q = threadIdx.x; q < n; q += kT) {
      const int64_t j = base + q;
      int64_t lo = r0, hi = r1 + 1;
      while (hi - lo > 1) {
        const int64_t mid = (lo + hi) >> 1;
        if (ro[mid] <= j) lo = mid; else hi = mid;
      }
      ri_out[j + shift] = (int32_t)lo;
    }
    return;
  }
  for (int64_t r = r0 + 1 + threadIdx.x; r <= r1; r += kT) {
    const int64_t at = ro[r] - base;
    if (at >= 0 && at < kScanTile) atomicMax(&mark[at], (int32_t)(r - r0));
  }
  __syncthreads();
  // thread t scans entries [8 t, 8 t + 8)
  int32_t m[kScanPer], top = 0;
#pragma unroll
  for (int k = 0; k < kScanPer; k++) {
    top = max(top, mark[threadIdx.x * kScanPer + k]);
    m[k] = top;
  }
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  int32_t inc = top;
  for (int d = 1; d < kWave; d <<= 1) {
    const int32_t o = shfl_up(inc, d);
    if (lane >= d) inc = max(inc, o);
  }
  if (lane == kWave - 1) wtop[wave] = inc;
  int32_t before = shfl_up(inc, 1);
  if (lane == 0) before = 0;
  __syncthreads();
  for (int w = 0; w < wave; w++) before = max(before, wtop[w]);
#pragma unroll
  for (int k = 0; k < kScanPer; k++) mark[threadIdx.x * kScanPer + k] = max(before, m[k]);
  __syncthreads();
  for (int q = threadIdx.x; q < n; q += kT) ri_out[base + q + shift] = (int32_t)(r0 + mark[q]);
}

inline unsigned scan_blocks(int64_t n) { return blocks_for(n, kScanTile); }

// ------------------------------------------------------------- radix sort
// Stable LSD radix sort of COO entries by (row << cb | col), 8 bits a pass.
// A workgroup takes a tile of 4096 entries: equal digits of a wave are found
// with ballots, the tile is put in digit order in LDS (keys, then values,
// through the same memory, so that three workgroups fit a CU), and written in
// runs (a tile's entries of one digit are consecutive in the output).  The
// first pass builds the keys from the indices, the last writes rows, columns
// and values to their places.  Each pass moves 2 (8 + W) bytes an entry and
// reads the keys once more to count.  9.2M shuffled FP64 entries, 40 key
// bits: 5 passes of 73-80 us and 17 us of counting (4.3 TB/s); 4-bit digits with
// positions instead of values took 10 of 73 us and a 182 us value gather.
constexpr int kSortBits = 8;
constexpr int kSortBins = 1 << kSortBits;
constexpr int kSortThreads = 512;
constexpr int kSortPer = 8;
constexpr int kSortTile = kSortThreads * kSortPer;
constexpr int kSortWaves = kSortThreads / kWave;

struct SortKeys {
  const int32_t *ri, *ci;    // first pass: the key is (ri << cb) | ci
  const uint64_t* key;       // later passes
  int cb, shift, mask;       // the pass's digit: mask of the key shifted
  template <bool FIRST>
  __device__ __forceinline__ uint64_t get(int64_t i) const {
    if (!FIRST) return key[i];
    return ((uint64_t)(uint32_t)ri[i] << cb) | (uint32_t)ci[i];
  }
  __device__ __forceinline__ int digit(uint64_t k) const {
    return (int)(k >> shift) & mask;
  }
};

template <bool FIRST>
__global__ __launch_bounds__(kSortThreads) void sort_count_kernel(SortKeys K, int64_t n,
                                                                  int32_t* __restrict__ hist,
                                                                  int64_t nb) {
  __shared__ int32_t h[kSortBins];
  if (threadIdx.x < kSortBins) h[threadIdx.x] = 0;
  __syncthreads();
  const int64_t base = (int64_t)blockIdx.x * kSortTile + threadIdx.x;
  uint64_t k[kSortPer];
#pragma unroll
  for (int q = 0; q < kSortPer; q++)
    k[q] = K.get<FIRST>(min(base + (int64_t)q * kSortThreads, n - 1));
#pragma unroll
  for (int q = 0; q < kSortPer; q++)
    if (base + (int64_t)q * kSortThreads < n) atomicAdd(&h[K.digit(k[q])], 1);
  __syncthreads();
  if (threadIdx.x < kSortBins) hist[threadIdx.x * nb + blockIdx.x] = h[threadIdx.x];
}

// keys and values between the passes; the arrays the last one writes
template <typename W>
struct SortOut {
  uint64_t* key;
  W* v;
  int32_t *ri, *ci;
};

template <bool FIRST, bool LAST, typename W>
__global__ __launch_bounds__(kSortThreads) void sort_scatter_kernel(
    SortKeys K, const W* v, int64_t n, const int32_t* __restrict__ offs, int64_t nb,
    SortOut<W> out) {
  __shared__ uint64_t sk[kSortTile];
  __shared__ int32_t wc_[kSortWaves][kSortBins];
  __shared__ int32_t start[kSortBins], dst[kSortBins], wsum[kSortBins / kWave];
  W* sv = reinterpret_cast<W*>(sk);
  volatile int32_t(*wc)[kSortBins] = wc_;  // written by one lane, read by others of its wave
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const uint64_t lt = (lane == 0) ? 0ull : ((~0ull) >> (64 - lane));
  const int64_t tile = (int64_t)blockIdx.x * kSortTile;
  const int count = (int)min((int64_t)kSortTile, n - tile);
  for (int q = threadIdx.x; q < kSortWaves * kSortBins; q += kSortThreads)
    wc[q / kSortBins][q % kSortBins] = 0;
  // wave w holds entries [512 w, 512 (w + 1)) of the tile, 64 a round, so
  // rounds and waves keep the input order
  const int at = wave * kWave * kSortPer + lane;
  uint64_t k[kSortPer];
  W x[kSortPer];
  int32_t rank[kSortPer];
#pragma unroll
  for (int q = 0; q < kSortPer; q++) {
    const int64_t i = min(tile + at + q * kWave, n - 1);
    k[q] = K.get<FIRST>(i);
    x[q] = v[i];
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < kSortPer; q++) {
    const bool in = at + q * kWave < count;
    const int d = K.digit(k[q]);
    uint64_t m = __ballot(in);
#pragma unroll
    for (int b = 0; b < kSortBits; b++) {
      const uint64_t one = __ballot((d >> b) & 1);
      m &= (d >> b) & 1 ? one : ~one;
    }
    const int before = __popcll(m & lt);
    const int32_t old = wc[wave][d];
    __builtin_amdgcn_wave_barrier();
    if (in && before == 0) wc[wave][d] = old + __popcll(m);
    __builtin_amdgcn_wave_barrier();
    rank[q] = old + before;
  }
  __syncthreads();
  // per digit: its entries of the waves before, and its place in the tile
  int32_t total = 0, inc = 0;
  if (threadIdx.x < kSortBins) {
    for (int w = 0; w < kSortWaves; w++) {
      const int32_t c = wc[w][threadIdx.x];
      wc[w][threadIdx.x] = total;
      total += c;
    }
    inc = total;
    for (int d = 1; d < kWave; d <<= 1) {
      const int32_t o = shfl_up(inc, d);
      if (lane >= d) inc += o;
    }
    if (lane == kWave - 1) wsum[wave] = inc;
  }
  __syncthreads();
  if (threadIdx.x < kSortBins) {
    for (int w = 0; w < wave; w++) inc += wsum[w];
    start[threadIdx.x] = inc - total;
    dst[threadIdx.x] = offs[threadIdx.x * nb + blockIdx.x] - (inc - total);
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < kSortPer; q++) {
    if (at + q * kWave >= count) break;
    const int d = K.digit(k[q]);
    rank[q] += start[d] + wc[wave][d];
    sk[rank[q]] = k[q];
  }
  __syncthreads();
  int64_t o[kSortPer];
#pragma unroll
  for (int q = 0; q < kSortPer; q++) {
    const int j = threadIdx.x + q * kSortThreads;
    if (j >= count) break;
    const uint64_t key = sk[j];
    o[q] = (int64_t)dst[K.digit(key)] + j;
    if (LAST) {
      out.ri[o[q]] = (int32_t)(key >> K.cb);
      out.ci[o[q]] = (int32_t)(key & ((1ull << K.cb) - 1));
    } else {
      out.key[o[q]] = key;
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < kSortPer; q++) {
    if (at + q * kWave >= count) break;
    sv[rank[q]] = x[q];
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < kSortPer; q++) {
    const int j = threadIdx.x + q * kSortThreads;
    if (j >= count) break;
    out.v[o[q]] = sv[j];
  }
}

int bits_for(int64_t maxv) {
  int b = 0;
  while (b < 31 && (int64_t(1) << b) <= maxv) b++;
  return b;
}

int fill_i32(int32_t* p, int64_t n, int32_t v, hipStream_t s) {
  if (n <= 0) return MPH_OK;
  hipLaunchKernelGGL(fill_i32_kernel, dim3(blocks_for(n)), dim3(kT), 0, s, p, n, v);
  MPH_HIP_CHECK(hipGetLastError());
  return MPH_OK;
}

int copy_dev(void* dst, const void* src, size_t bytes, hipStream_t s) {
  if (bytes == 0) return MPH_OK;
  MPH_HIP_CHECK(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, s));
  return MPH_OK;
}

// Stable sort of COO entries by (row, col), rows below 2^rb and columns below
// 2^cb; kByRow: by row only, the columns carried along.  kLowBits: the columns
// carried whole too, and sorted by their low cb bits, rounded up to a multiple
// of 4 (a column below 0 has no other order).  The outputs may be the inputs.
enum SortBy { kByRowCol, kByRow, kLowBits };

template <typename W>
int radix_sort(int64_t n, int rb, int cb, SortBy by, const int32_t* ri, const int32_t* ci,
               const void* v, int32_t* ri_out, int32_t* ci_out, void* v_out, hipStream_t s) {
  if (n <= 0) return MPH_OK;
  Tmp t(s);
  const int64_t nb = ceil_div(n, kSortTile);
  // the digits: shift and mask of each pass
  constexpr int kMaxPasses = 8;
  int shift[kMaxPasses], mask[kMaxPasses], passes = 0;
  auto digits = [&](int from, int to) {
    for (int b = from; b < to; b += kSortBits) {
      shift[passes] = b;
      mask[passes++] = (1 << std::min(kSortBits, to - b)) - 1;
    }
  };
  if (by == kByRowCol) {
    digits(0, rb + cb);
  } else {
    if (by == kLowBits) digits(0, (int)ceil_div(cb, 4) * 4);
    cb = 32;
    digits(cb, cb + rb);
  }
  // at least two passes: the last one's input is never the arrays it writes
  // (a pass that sees digits 0 only moves)
  while (passes < 2) {
    shift[passes] = 0;
    mask[passes++] = 0;
  }
  uint64_t* key[2];
  W* val[2];
  int32_t *hist, *offs;
  int64_t* tmp;
  for (int q = 0; q < (passes > 2 ? 2 : 1); q++) {
    MPH_CHECK_STATUS(t.alloc(&key[q], n));
    MPH_CHECK_STATUS(t.alloc(&val[q], n));
  }
  MPH_CHECK_STATUS(t.alloc(&hist, kSortBins * nb));
  MPH_CHECK_STATUS(t.alloc(&offs, kSortBins * nb + 1));
  MPH_CHECK_STATUS(t.alloc(&tmp, scan_tmp_elems(kSortBins * nb)));
  const dim3 g((unsigned)nb), b(kSortThreads);
  for (int q = 0; q < passes; q++) {
    const SortKeys K{ri, ci, q > 0 ? key[(q - 1) & 1] : nullptr, cb, shift[q], mask[q]};
    const W* vin = q > 0 ? val[(q - 1) & 1] : static_cast<const W*>(v);
    if (q == 0)
      hipLaunchKernelGGL(sort_count_kernel<true>, g, b, 0, s, K, n, hist, nb);
    else
      hipLaunchKernelGGL(sort_count_kernel<false>, g, b, 0, s, K, n, hist, nb);
    MPH_CHECK_STATUS(exclusive_scan_i32(hist, offs, kSortBins * nb, tmp, s));
    const bool last = q + 1 == passes;
    const SortOut<W> out{last ? nullptr : key[q & 1], last ? static_cast<W*>(v_out) : val[q & 1],
                         ri_out, ci_out};
    if (q == 0)
      hipLaunchKernelGGL((sort_scatter_kernel<true, false, W>), g, b, 0, s, K, vin, n, offs, nb,
                         out);
    else if (!last)
      hipLaunchKernelGGL((sort_scatter_kernel<false, false, W>), g, b, 0, s, K, vin, n, offs, nb,
                         out);
    else
      hipLaunchKernelGGL((sort_scatter_kernel<false, true, W>), g, b, 0, s, K, vin, n, offs, nb,
                         out);
    MPH_HIP_CHECK(hipGetLastError());
  }
  return MPH_OK;  // (t waits for the stream)
}

int radix_sort(int64_t n, int rb, int cb, SortBy by, const int32_t* ri, const int32_t* ci,
               const void* v, int vsize, int32_t* ri_out, int32_t* ci_out, void* v_out,
               hipStream_t s) {
  if (vsize == 8)
    return radix_sort<uint64_t>(n, rb, cb, by, ri, ci, v, ri_out, ci_out, v_out, s);
  if (vsize == 4)
    return radix_sort<uint32_t>(n, rb, cb, by, ri, ci, v, ri_out, ci_out, v_out, s);
  return radix_sort<uint16_t>(n, rb, cb, by, ri, ci, v, ri_out, ci_out, v_out, s);
}

// What coo_scan_kernel finds, as an error.
int scan_status(int32_t flags) {
  if (flags & kBadRow) return invalid("COO row_indices: index out of range");
  if (flags & kBadCol) return invalid("COO column_indices: index out of range");
  return MPH_OK;
}

// the three flags of coo_scan_kernel<kWidths> (indices up to INT32_MAX - 1 in range)
int scan_order(const int32_t* ri, const int32_t* ci, int64_t nnz, hipStream_t s, int32_t* flags) {
  std::fill(flags, flags + 3, 0);
  if (nnz <= 0) return MPH_OK;
  Tmp t(s);
  int32_t* d;
  MPH_CHECK_STATUS(t.alloc(&d, 3));
  MPH_CHECK_STATUS(fill_zero(d, 3 * sizeof(int32_t), s));
  hipLaunchKernelGGL((coo_scan_kernel<true, false, kWidths>), dim3(scan_blocks(nnz)), dim3(kT), 0, s,
                     ri, ci, nnz, (int64_t)INT32_MAX, (int64_t)INT32_MAX, (int32_t*)nullptr,
                     (uint32_t*)nullptr, d);
  MPH_HIP_CHECK(hipGetLastError());
  MPH_CHECK_STATUS(t.read(d, flags, 3));
  t.idle = true;
  return MPH_OK;
}

int is_sorted_dev(const int32_t* ri, const int32_t* ci, int64_t nnz, hipStream_t s,
                  int* sorted) {
  *sorted = 1;
  if (nnz <= 1) return MPH_OK;  // (the arrays are not looked at)
  int32_t flags[3];
  MPH_CHECK_STATUS(scan_order(ri, ci, nnz, s, flags));
  *sorted = !(flags[0] & kUnsorted);
  return MPH_OK;
}

// in-place stable (row, col) sort of COO arrays, if they are not in order;
// check: with indices below 0 refused (the conversions carry such columns)
int sort_coo(int64_t nnz, int32_t* ri, int32_t* ci, void* v, int vsize, bool check,
             hipStream_t s) {
  if (nnz <= 1) return MPH_OK;
  int32_t flags[3];
  MPH_CHECK_STATUS(scan_order(ri, ci, nnz, s, flags));
  if (check) MPH_CHECK_STATUS(scan_status(flags[0]));
  if (!(flags[0] & kUnsorted)) return MPH_OK;
  return radix_sort(nnz, bits_for(flags[1]), bits_for(flags[2]),
                    (flags[0] & kBadCol) ? kLowBits : kByRowCol, ri, ci, v, vsize, ri, ci, v, s);
}

// ------------------------------------------------------------- emitters
// Entries of a DIA part in (row, column) order.  The Serial converter walks
// the diagonals and sorts the entries afterwards; walking the rows, with the
// diagonals in ascending order of their offsets (equal offsets in storage
// order, as the stable sort leaves them), gives that order at once: a count
// per row, a scan over the rows, and the entries written to their places.
// (row r, diagonal d) is stored iff its column is inside [0, ncols) (rows
// i_start + n, n < N of :97-101) and its value is not a zero (full_mask:
// integer values, where every bit counts; floating-point values drop the sign
// bit, so that -0.0 is a zero too).
template <typename W>
struct DiaSlots {
  const W* val;
  const int32_t* off;  // by slot
  const int32_t* ord;  // slot -> stored diagonal (null: the same)
  int64_t pitch, ncols;
  W mask;
  __device__ __forceinline__ void load(int64_t r, int s, int32_t& c, W& v, bool& ok) const {
    const int64_t col = r + off[s];
    v = val[r + pitch * (ord ? ord[s] : s)];
    ok = col >= 0 && col < ncols;
    c = (int32_t)col;
  }
  __device__ __forceinline__ void finish(int64_t, int, int32_t, W& v, bool& ok) const {
    ok = ok && (v & mask) != 0;
  }
};

// Entries of an ELL part, slots that hold a column, in slot order.
template <typename W>
struct EllSlots {
  const int32_t* eci;
  const W* ev;
  int64_t pitch;
  __device__ __forceinline__ void load(int64_t r, int s, int32_t& c, W&, bool& ok) const {
    c = eci[r + pitch * s];
    ok = c != -1;
  }
  __device__ __forceinline__ void finish(int64_t r, int s, int32_t, W& v, bool& ok) const {
    if (ok) v = ev[r + pitch * s];
  }
};

// The slots of a row in segments of `len`, counted and emitted as if they were
// rows of their own, in the order (row, segment): one where rows are short,
// more where a few rows hold many slots (a thread or lane per row took 500 ms
// for one row of 2M diagonals, 254 ms for as many ELL slots).
struct Segs {
  int32_t len, n;
};
constexpr int kSegSlots = 256;

Segs segments(int64_t nrows, int64_t slots) {
  if (slots <= kSegSlots) return {kSegSlots, 1};
  int64_t len = kSegSlots;
  // shorter, down to a batch of the emission, where they would not fill the
  // device (one row of 2M diagonals 376 -> 144 us)
  while (len > 32 && nrows * ceil_div(slots, len) < 65536) len /= 2;
  while (ceil_div(slots, len) > 32768 && nrows >= kWave) len *= 2;  // (a grid's second dimension)
  return {(int32_t)len, (int32_t)ceil_div(slots, len)};
}

// The row and segment of thread t: rows next to each other.  (The kernels over
// rows of one segment are instances of their own, SEGS false: the segments
// took them registers and 3 to 5% of their time.)
template <bool SEGS>
__device__ __forceinline__ void row_segment(int64_t t, int64_t nrows, int64_t& r, int32_t& y) {
  y = SEGS ? (int32_t)(t / nrows) : 0;
  r = t - (int64_t)y * nrows;
}

template <bool SEGS, typename W>
__global__ __launch_bounds__(kT) void dia_row_count_kernel(DiaSlots<W> src, int64_t nrows,
                                                           int32_t ns, Segs g,
                                                           int32_t* __restrict__ cnt) {
  using I = std::conditional_t<SEGS, int64_t, int32_t>;
  const int64_t t = (int64_t)blockIdx.x * kT + threadIdx.x;
  if (t >= (SEGS ? nrows * g.n : nrows)) return;
  int64_t r;
  int32_t y;
  row_segment<SEGS>(t, nrows, r, y);
  int32_t n = 0;
  const I end = SEGS ? (I)min((int64_t)ns, ((int64_t)y + 1) * g.len) : (I)ns;
  for (I s0 = SEGS ? (I)y * g.len : 0; s0 < end; s0 += kScanPer) {
    W v[kScanPer];
    bool ok[kScanPer];
    int32_t c;
#pragma unroll
    for (int k = 0; k < kScanPer; k++) {
      ok[k] = false;
      if (s0 + k < end) src.load(r, (int)(s0 + k), c, v[k], ok[k]);
    }
#pragma unroll
    for (int k = 0; k < kScanPer; k++) {
      if (ok[k]) src.finish(r, (int)(s0 + k), c, v[k], ok[k]);
      n += ok[k] ? 1 : 0;
    }
  }
  cnt[SEGS ? r * g.n + y : r] = n;
}

// The entries of 64 rows' segments a workgroup: lane = row (kWhole: of one
// segment), of the segment blockIdx.y (kSegment), or, with fewer rows than
// lanes, lane = one of 64 consecutive (row, segment) (kNarrow); each wave a quarter of the slots, batches of 32
// slots.  The entries are staged in LDS in output order and written coalesced
// (written from the row walk, each store of a wave spreads over 64 rows'
// entries); those of segment q = (row, segment) go to rowpos[q], rowpos[q] + 1,
// ... (a row's range may be longer: HYB's COO entries follow).  Reads the
// slots once, coalesced, writes 8 + W bytes an entry once.
constexpr int kEmitRows = kWave;
constexpr int kEmitWaves = kT / kWave;
constexpr int kEmitPer = 8;  // slots per lane and batch
constexpr int kEmitBatch = kEmitWaves * kEmitPer;

enum EmitBy { kWhole, kSegment, kNarrow };

template <EmitBy BY, typename W, typename Src>
__global__ __launch_bounds__(kT) void emit_rows_kernel(Src src, int64_t nrows, int32_t ns, Segs g,
                                                       const int32_t* __restrict__ rowpos,
                                                       int32_t* __restrict__ ri,
                                                       int32_t* __restrict__ ci,
                                                       W* __restrict__ vo) {
  __shared__ W sv[kEmitRows * kEmitBatch];
  __shared__ int32_t sc[kEmitRows * kEmitBatch];
  __shared__ uint8_t sr[kEmitRows * kEmitBatch];
  __shared__ int32_t cnt[kEmitWaves][kEmitRows];
  __shared__ int32_t dst[kEmitRows];  // output position of the row's first entry, less its LDS place
  __shared__ int32_t total;
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  constexpr bool NARROW = BY == kNarrow;
  using I = std::conditional_t<NARROW, int64_t, int32_t>;  // (a segment may end past the slots)
  __shared__ int32_t srow[NARROW ? kEmitRows : 1];
  const int64_t r0 = (int64_t)blockIdx.x * kEmitRows;
  int64_t r = r0 + lane;
  int32_t seg = BY == kSegment ? (int32_t)blockIdx.y : 0;
  if (NARROW) {
    const int64_t q = r;
    r = q / g.n;
    seg = (int32_t)(q - r * g.n);
    if (wave == 0) srow[lane] = (int32_t)r;  // (read after the barriers below)
  }
  const int32_t first_slot = BY == kWhole ? 0 : seg * g.len;
  const int32_t len = NARROW ? g.len : BY == kSegment ? min(g.len, ns - first_slot) : ns;
  int32_t pos = r < nrows ? rowpos[BY == kWhole ? r : r * g.n + seg] : 0;
  for (int s0 = 0; s0 < len; s0 += kEmitBatch) {
    // the batch's slots in order over the waves
    const int per = (min(kEmitBatch, len - s0) + kEmitWaves - 1) / kEmitWaves;
    const I sl = (I)first_slot + s0, sb = sl + wave * per;
    const I se = min(min((I)(sb + per), (I)(sl + kEmitBatch)), min((I)ns, (I)((I)first_slot + len)));
    W v[kEmitPer];
    int32_t c[kEmitPer];
    bool ok[kEmitPer];
#pragma unroll
    for (int k = 0; k < kEmitPer; k++) {
      ok[k] = false;
      if (sb + k < se && r < nrows) src.load(r, (int)(sb + k), c[k], v[k], ok[k]);
    }
    int32_t n = 0;
#pragma unroll
    for (int k = 0; k < kEmitPer; k++) {
      if (ok[k]) src.finish(r, (int)(sb + k), c[k], v[k], ok[k]);
      n += ok[k] ? 1 : 0;
    }
    cnt[wave][lane] = n;
    __syncthreads();
    int32_t before = 0, row_n = 0;
    for (int w = 0; w < kEmitWaves; w++) {
      const int32_t q = cnt[w][lane];
      before += w < wave ? q : 0;
      row_n += q;
    }
    int32_t inc = row_n;  // (the same in every wave)
    for (int d = 1; d < kWave; d <<= 1) {
      const int32_t o = shfl_up(inc, d);
      if (lane >= d) inc += o;
    }
    const int32_t first = inc - row_n;
    if (wave == 0) {
      dst[lane] = pos - first;
      if (lane == kWave - 1) total = inc;
    }
    int32_t at = first + before;
#pragma unroll
    for (int k = 0; k < kEmitPer; k++)
      if (ok[k]) {
        sv[at] = v[k];
        sc[at] = c[k];
        sr[at] = (uint8_t)lane;
        at++;
      }
    __syncthreads();
    for (int j = threadIdx.x; j < total; j += kT) {
      const int q = sr[j];
      const int64_t o = (int64_t)dst[q] + j;
      ri[o] = NARROW ? srow[q] : (int32_t)(r0 + q);
      ci[o] = sc[j];
      vo[o] = sv[j];
    }
    pos += row_n;
    __syncthreads();
  }
}

template <typename W, typename Src>
void emit_rows(const Src& src, int64_t nrows, int32_t ns, const Segs& g, const int32_t* rowpos,
               int32_t* ri, int32_t* ci, void* v_, hipStream_t s) {
  W* v = static_cast<W*>(v_);
  const unsigned gx = blocks_for(nrows, kEmitRows);
  if (g.n == 1)
    hipLaunchKernelGGL((emit_rows_kernel<kWhole, W, Src>), dim3(gx), dim3(kT), 0, s, src, nrows, ns,
                       g, rowpos, ri, ci, v);
  else if (nrows < kEmitRows)
    hipLaunchKernelGGL((emit_rows_kernel<kNarrow, W, Src>),
                       dim3(blocks_for(nrows * g.n, kEmitRows)), dim3(kT), 0, s, src, nrows, ns, g,
                       rowpos, ri, ci, v);
  else
    hipLaunchKernelGGL((emit_rows_kernel<kSegment, W, Src>),
                       dim3(gx, (unsigned)ceil_div(ns, g.len)), dim3(kT), 0, s, src, nrows, ns, g,
                       rowpos, ri, ci, v);
}

// zero the COO slots [from, nnz) left unfilled
template <typename W>
__global__ void zero_tail_kernel(int64_t from, int64_t nnz, int32_t* ri, int32_t* ci, void* v_) {
  W* v = static_cast<W*>(v_);
  const int64_t i = from + (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < nnz) {
    ri[i] = 0;
    ci[i] = 0;
    v[i] = 0;
  }
}

// Per row and segment, the ELL slots that hold a column, plus with the row's
// last segment its entries of the row-sorted COO part (tro null: none); stats:
// [0] raised when some row's columns are not in ascending order (its COO
// entries after its slots; the order among the COO entries is checked by
// coo_scan_kernel), [1] 1 + the last slot any row uses.  A segment looks up to
// kSegBack slots back for the column before its first; not finding one counts
// as out of order (the list is then sorted, whatever its order).
constexpr int kSegBack = 64;
template <bool SEGS>
__global__ __launch_bounds__(kT) void ell_row_count_kernel(
    const int32_t* __restrict__ eci, int64_t nrows, int64_t width, int64_t pitch, Segs g,
    const int32_t* __restrict__ tro, const int32_t* __restrict__ tci, int32_t* __restrict__ cnt,
    int32_t* __restrict__ stats) {
  int32_t bad = 0, top = 0;
  for (int64_t t = (int64_t)blockIdx.x * kT + threadIdx.x; t < (SEGS ? nrows * g.n : nrows);
       t += (int64_t)gridDim.x * kT) {
    int64_t r;
    int32_t y;
    row_segment<SEGS>(t, nrows, r, y);
    int32_t n = 0, prev = INT32_MIN;
    const int64_t begin = SEGS ? (int64_t)y * g.len : 0;
    const int64_t end = SEGS ? min(width, begin + g.len) : width;
    bool known = !SEGS || y == 0;
    for (int64_t b = begin - 1; !known && b >= max(begin - kSegBack, (int64_t)0); b--) {
      const int32_t c = eci[r + pitch * b];
      known = c != -1;
      if (known) prev = c;
    }
    for (int64_t s0 = begin; s0 < end; s0 += kScanPer) {
      int32_t c[kScanPer];
#pragma unroll
      for (int k = 0; k < kScanPer; k++) c[k] = s0 + k < end ? eci[r + pitch * (s0 + k)] : -1;
#pragma unroll
      for (int k = 0; k < kScanPer; k++)
        if (c[k] != -1) {
          bad |= c[k] < prev || !known ? 1 : 0;
          if (SEGS) known = true;
          prev = c[k];
          n++;
          top = max(top, (int32_t)(s0 + k) + 1);
        }
    }
    if (tro && (!SEGS || y == g.n - 1)) {
      const int32_t ts = tro[r], te = tro[r + 1];
      if (te > ts && (!known || (prev != INT32_MIN && tci[ts] < prev))) bad = 1;
      n += te - ts;
    }
    cnt[SEGS ? r * g.n + y : r] = n;
  }
  raise_flags(&stats[0], bad);
  top = block_reduce(top, [](int32_t u, int32_t v) { return max(u, v); });
  if (threadIdx.x == 0 && top > 0 &&
      __hip_atomic_load(&stats[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < top)
    atomicMax(&stats[1], top);
}

// HYB -> COO, the COO part: entry j of row r ends r's range
template <typename W>
__global__ void hyb_tail_emit_kernel(const int32_t* __restrict__ tri,
                                     const int32_t* __restrict__ tci,
                                     const void* __restrict__ tv_, int64_t n,
                                     const int32_t* __restrict__ tro,
                                     const int32_t* __restrict__ rowpos, int32_t segs,
                                     int32_t* __restrict__ ri, int32_t* __restrict__ ci,
                                     void* __restrict__ vo_) {
  const W* tv = static_cast<const W*>(tv_);
  W* vo = static_cast<W*>(vo_);
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n) return;
  const int32_t r = tri[j];
  const int64_t o = (int64_t)rowpos[((int64_t)r + 1) * segs] - tro[r + 1] + j;
  ri[o] = r;
  ci[o] = tci[j];
  vo[o] = tv[j];
}

// ------------------------------------------------------------- COO -> X
// run heads: head[i] = 1 when entry i starts a run of equal rows
__global__ void run_head_kernel(const int32_t* __restrict__ ri, int64_t nnz,
                                int32_t* __restrict__ head) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < nnz) head[i] = (i == 0 || ri[i] != ri[i - 1]) ? 1 : 0;
}

// runpos[k] = index of the k-th run head (hscan = exclusive scan of heads)
__global__ void run_pos_kernel(const int32_t* __restrict__ head,
                               const int32_t* __restrict__ hscan, int64_t nnz,
                               int32_t* __restrict__ runpos) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < nnz && head[i]) runpos[hscan[i]] = (int32_t)i;
}

__device__ __forceinline__ int64_t pos_in_run(const int32_t* head, const int32_t* hscan,
                                              const int32_t* runpos, int64_t i) {
  const int64_t run = hscan[i] + head[i] - 1;  // inclusive count - 1
  return i - runpos[run];
}

// ELL / HYB placement: slot (row, n) claimed by the latest entry
__global__ void ell_claim_kernel(const int32_t* __restrict__ ri, int64_t nnz, int64_t K,
                                 int64_t pitch, const int32_t* __restrict__ head,
                                 const int32_t* __restrict__ hscan,
                                 const int32_t* __restrict__ runpos,
                                 int32_t* __restrict__ winner, int32_t* __restrict__ over) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nnz) return;
  const int64_t n = pos_in_run(head, hscan, runpos, i);
  if (n < K) atomicMax(&winner[ri[i] + pitch * n], (int32_t)i);
  else if (over) over[i] = 1;
}

template <typename W>
__global__ void ell_place_kernel(const int32_t* __restrict__ ri, const int32_t* __restrict__ ci,
                                 const void* __restrict__ v_, int64_t nnz, int64_t K, int64_t pitch,
                                 const int32_t* __restrict__ head,
                                 const int32_t* __restrict__ hscan,
                                 const int32_t* __restrict__ runpos,
                                 const int32_t* __restrict__ winner, int32_t* __restrict__ eci,
                                 void* __restrict__ ev_) {
  const W* v = static_cast<const W*>(v_);
  W* ev = static_cast<W*>(ev_);
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nnz) return;
  const int64_t n = pos_in_run(head, hscan, runpos, i);
  if (n >= K) return;
  const int64_t slot = ri[i] + pitch * n;
  if (winner[slot] == (int32_t)i) {
    eci[slot] = ci[i];
    ev[slot] = v[i];
  }
}

template <typename W>
__global__ void tail_place_kernel(const int32_t* __restrict__ ri, const int32_t* __restrict__ ci,
                                  const void* __restrict__ v_, int64_t nnz,
                                  const int32_t* __restrict__ over,
                                  const int32_t* __restrict__ opos, int32_t* __restrict__ tri,
                                  int32_t* __restrict__ tci, void* __restrict__ tv_) {
  const W* v = static_cast<const W*>(v_);
  W* tv = static_cast<W*>(tv_);
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nnz || !over[i]) return;
  const int64_t p = opos[i];
  tri[p] = ri[i];
  tci[p] = ci[i];
  tv[p] = v[i];
}

// COO -> ELL / HYB when the rows do not decrease: row r's entries are
// [ro[r], ro[r + 1]), its n-th in slot n, so every slot is written once, in
// row order per slot (coalesced), padding (-1, 0) included.  64 rows and `per`
// slots a workgroup, each wave every fourth slot; the rows' entries are read
// coalesced into LDS when they fit, or directly.  (With rows that decrease,
// a row may have several runs, and the latest entry claims each slot first,
// above.)
constexpr int kEllStage = 2048;
constexpr int64_t kFillBlocks = 2048;  // workgroups enough to fill the device
template <typename W>
__global__ __launch_bounds__(kT) void ell_fill_rows_kernel(
    const int32_t* __restrict__ ro, const int32_t* __restrict__ ci, const void* __restrict__ v_,
    int64_t nrows, int64_t K, int64_t width, int64_t per, int64_t pitch, int32_t* __restrict__ eci,
    void* __restrict__ ev_) {
  __shared__ int32_t sc[kEllStage];
  __shared__ W sv[kEllStage];
  const W* v = static_cast<const W*>(v_);
  W* ev = static_cast<W*>(ev_);
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int64_t r0 = (int64_t)blockIdx.x * kWave, r = r0 + lane;
  const int64_t e0 = ro[min(r0, nrows)], e1 = ro[min(r0 + kWave, nrows)];
  const bool staged = e1 - e0 <= kEllStage;
  if (staged) {
    for (int64_t q = threadIdx.x; q < e1 - e0; q += kT) {
      sc[q] = ci[e0 + q];
      sv[q] = v[e0 + q];
    }
    __syncthreads();
  }
  if (r >= pitch) return;
  const int64_t b = r < nrows ? ro[r] : 0, len = r < nrows ? min((int64_t)ro[r + 1] - b, K) : 0;
  const int64_t n0 = per * blockIdx.y, n1 = min(width, n0 + per);
  for (int64_t n = n0 + wave; n < n1; n += kT / kWave) {
    int32_t c = -1;
    W x = 0;
    if (n < len) {
      c = staged ? sc[b - e0 + n] : ci[b + n];
      x = staged ? sv[b - e0 + n] : v[b + n];
    }
    eci[r + pitch * n] = c;
    ev[r + pitch * n] = x;
  }
}

// The same for fewer rows than a wave has lanes: a thread per slot, the rows
// of one slot next to each other.
template <typename W>
__global__ __launch_bounds__(kT) void ell_fill_slots_kernel(
    const int32_t* __restrict__ ro, const int32_t* __restrict__ ci, const void* __restrict__ v_,
    int64_t nrows, int64_t K, int64_t slots, int64_t pitch, int32_t* __restrict__ eci,
    void* __restrict__ ev_) {
  const int64_t i = (int64_t)blockIdx.x * kT + threadIdx.x;
  if (i >= slots) return;
  const int64_t n = i / pitch, r = i - n * pitch;
  const int64_t b = r < nrows ? ro[r] : 0;
  const bool in = r < nrows && n < min((int64_t)ro[r + 1] - b, K);
  eci[i] = in ? ci[b + n] : -1;
  static_cast<W*>(ev_)[i] = in ? static_cast<const W*>(v_)[b + n] : 0;
}

// entries past a row's first K, per row
__global__ void over_count_kernel(const int32_t* __restrict__ ro, int64_t nrows, int32_t K,
                                  int32_t* __restrict__ cnt) {
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r < nrows) cnt[r] = max(0, ro[r + 1] - ro[r] - K);
}

// HYB's COO part: those entries, row r's at opos[r], opos[r] + 1, ...  A
// thread's entries are loaded together, so the row lookups of all are in
// flight at once: 101 us for 16M power-law FP32 entries, 13.4M of them past
// their row's K (106 us with one entry a thread).
template <typename W>
__global__ __launch_bounds__(kT) void over_place_kernel(
    const int32_t* __restrict__ ri, const int32_t* __restrict__ ci, const void* __restrict__ v_,
    int64_t nnz, int64_t K, const int32_t* __restrict__ ro, const int32_t* __restrict__ opos,
    int32_t* __restrict__ tri, int32_t* __restrict__ tci, void* __restrict__ tv_) {
  const W* v = static_cast<const W*>(v_);
  W* tv = static_cast<W*>(tv_);
  const int64_t base = (int64_t)blockIdx.x * kScanTile + threadIdx.x;
  int32_t r[kScanPer], c[kScanPer], b[kScanPer], o[kScanPer];
  W x[kScanPer];
#pragma unroll
  for (int k = 0; k < kScanPer; k++) {
    const int64_t i = min(base + (int64_t)k * kT, nnz - 1);
    r[k] = ri[i];
    c[k] = ci[i];
    x[k] = v[i];
  }
#pragma unroll
  for (int k = 0; k < kScanPer; k++) {
    b[k] = ro[r[k]];
    o[k] = opos[r[k]];
  }
#pragma unroll
  for (int k = 0; k < kScanPer; k++) {
    const int64_t i = base + (int64_t)k * kT, n = i - b[k] - K;
    if (i >= nnz || n < 0) continue;
    const int64_t at = o[k] + n;
    tri[at] = r[k];
    tci[at] = c[k];
    tv[at] = x[k];
  }
}

// of row offsets: the longest row, and the sum of min(length, K)
__global__ __launch_bounds__(kT) void row_lengths_kernel(const int32_t* __restrict__ ro,
                                                         int64_t nrows, int32_t K,
                                                         unsigned long long* __restrict__ out) {
  const int64_t step = (int64_t)gridDim.x * kT;
  int32_t m = 0;
  unsigned long long t = 0;
  for (int64_t r = (int64_t)blockIdx.x * kT + threadIdx.x; r < nrows; r += step) {
    const int32_t len = ro[r + 1] - ro[r];
    m = max(m, len);
    t += (unsigned long long)max(0, min(len, K));
  }
  m = block_reduce(m, [](int32_t u, int32_t v) { return max(u, v); });
  t = block_reduce(t, [](unsigned long long u, unsigned long long v) { return u + v; });
  if (threadIdx.x == 0) {
    if (__hip_atomic_load(&out[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) <
        (unsigned long long)m)
      atomicMax(&out[0], (unsigned long long)m);
    if (t > 0) atomicAdd(&out[1], t);
  }
}

// DIA / HDC placement: the first offset equal to col - row (binary search of
// the ascending offsets) -- the first match of the reference's linear scan
__device__ __forceinline__ int64_t find_first(const int32_t* off, int64_t n, int32_t key) {
  int64_t lo = 0, hi = n;
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if (off[mid] < key) lo = mid + 1; else hi = mid;
  }
  return (lo < n && off[lo] == key) ? lo : -1;
}

__global__ void dia_claim_kernel(const int32_t* __restrict__ ri, const int32_t* __restrict__ ci,
                                 int64_t nnz, const int32_t* __restrict__ off, int64_t ndiag,
                                 int64_t pitch, int32_t* __restrict__ winner,
                                 int32_t* __restrict__ rest) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nnz) return;
  const int64_t d = find_first(off, ndiag, ci[i] - ri[i]);
  if (d >= 0) atomicMax(&winner[ri[i] + pitch * d], (int32_t)i);
  else if (rest) rest[i] = 1;
}

template <typename W>
__global__ void dia_place_kernel(const int32_t* __restrict__ ri, const int32_t* __restrict__ ci,
                                 const void* __restrict__ v_, int64_t nnz,
                                 const int32_t* __restrict__ off, int64_t ndiag, int64_t pitch,
                                 const int32_t* __restrict__ winner, void* __restrict__ dv_) {
  const W* v = static_cast<const W*>(v_);
  W* dv = static_cast<W*>(dv_);
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nnz) return;
  const int64_t d = find_first(off, ndiag, ci[i] - ri[i]);
  if (d < 0) return;
  const int64_t slot = ri[i] + pitch * d;
  if (winner[slot] == (int32_t)i) dv[slot] = v[i];
}

// DIA / HDC placement of entries in strictly ascending (row, column) order:
// no slot is written twice, so the values go straight to their slots.
// Consecutive entries of a diagonal are consecutive in memory; a workgroup's
// kScanTile entries write runs of hundreds of rows.  (With repeated or
// unsorted entries, the latest entry claims each slot first, below.)
constexpr int kPlaceOffsets = 1024;  // offsets kept in LDS
template <typename W>
__global__ __launch_bounds__(kT) void dia_place_once_kernel(
    const int32_t* __restrict__ ri, const int32_t* __restrict__ ci, const void* __restrict__ v_,
    int64_t nnz, const int32_t* __restrict__ off, int64_t ndiag, int64_t pitch,
    void* __restrict__ dv_) {
  __shared__ int32_t soff[kPlaceOffsets];
  const W* v = static_cast<const W*>(v_);
  W* dv = static_cast<W*>(dv_);
  const bool lds = ndiag <= kPlaceOffsets;
  if (lds) {
    for (int q = threadIdx.x; q < ndiag; q += kT) soff[q] = off[q];
    __syncthreads();
  }
  const int64_t base = (int64_t)blockIdx.x * kScanTile + threadIdx.x;
  int32_t r[kScanPer], c[kScanPer];
  W x[kScanPer];
#pragma unroll
  for (int k = 0; k < kScanPer; k++) {
    const int64_t i = base + (int64_t)k * kT;
    if (i < nnz) {
      r[k] = ri[i];
      c[k] = ci[i];
      x[k] = v[i];
    }
  }
#pragma unroll
  for (int k = 0; k < kScanPer; k++) {
    if (base + (int64_t)k * kT >= nnz) break;
    const int64_t d = find_first(lds ? soff : off, ndiag, c[k] - r[k]);
    if (d >= 0) dv[r[k] + pitch * d] = x[k];
  }
}

// HDC from entries in strictly ascending order: entries whose diagonal is
// not among the offsets are counted per tile; then, with the tiles' positions
// known, the values go to their diagonals and the others, in order, to the
// CSR part's arrays.
template <bool PLACE, typename W>
__global__ __launch_bounds__(kT) void hdc_split_kernel(
    const int32_t* __restrict__ ri, const int32_t* __restrict__ ci, const void* __restrict__ v_,
    int64_t nnz, const int32_t* __restrict__ off, int64_t ndiag, int64_t pitch,
    void* __restrict__ dv_, int32_t* __restrict__ tile_n, const int32_t* __restrict__ tile_pos,
    int32_t* __restrict__ rri, int32_t* __restrict__ rci, void* __restrict__ rv_) {
  __shared__ int32_t soff[kPlaceOffsets];
  __shared__ int32_t wn[kScanPer][kT / kWave];
  const W* v = static_cast<const W*>(v_);
  const bool lds = ndiag <= kPlaceOffsets;
  if (lds)
    for (int q = threadIdx.x; q < ndiag; q += kT) soff[q] = off[q];
  __syncthreads();
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const uint64_t lt = (lane == 0) ? 0ull : ((~0ull) >> (64 - lane));
  const int64_t base = (int64_t)blockIdx.x * kScanTile + threadIdx.x;
  int32_t r[kScanPer], c[kScanPer], rank[kScanPer];
  W x[kScanPer];
#pragma unroll
  for (int k = 0; k < kScanPer; k++) {
    const int64_t i = base + (int64_t)k * kT;
    r[k] = c[k] = 0;
    if (i < nnz) {
      r[k] = ri[i];
      c[k] = ci[i];
      if (PLACE) x[k] = v[i];
    }
  }
#pragma unroll
  for (int k = 0; k < kScanPer; k++) {
    const bool in = base + (int64_t)k * kT < nnz;
    const int64_t d = in ? find_first(lds ? soff : off, ndiag, c[k] - r[k]) : 0;
    const uint64_t m = __ballot(in && d < 0);
    rank[k] = in && d < 0 ? __popcll(m & lt) : -1;
    if (lane == 0) wn[k][wave] = __popcll(m);
    if (PLACE && in && d >= 0) static_cast<W*>(dv_)[r[k] + pitch * d] = x[k];
  }
  __syncthreads();
  if (!PLACE) {
    if (threadIdx.x == 0) {
      int32_t n = 0;
      for (int q = 0; q < kScanPer * (kT / kWave); q++) n += wn[q / (kT / kWave)][q % (kT / kWave)];
      tile_n[blockIdx.x] = n;
    }
    return;
  }
  int32_t before = tile_pos[blockIdx.x];
#pragma unroll
  for (int k = 0; k < kScanPer; k++) {
    for (int w = 0; w < kT / kWave; w++) {
      if (w == wave && rank[k] >= 0) {
        const int64_t o = before + rank[k];
        rri[o] = r[k];
        rci[o] = c[k];
        static_cast<W*>(rv_)[o] = x[k];
      }
      before += wn[k][w];
    }
  }
}

// Two lists in (row, column) order merged: entry e of list A lands after the
// B entries before it (row r's from bro[r * step] on).  LATER: A's entries
// follow equal ones of B.
template <bool LATER, typename W>
__global__ __launch_bounds__(kT) void merge_rows_kernel(
    const int32_t* __restrict__ ri, const int32_t* __restrict__ ci, const void* __restrict__ v_,
    int64_t n, const int32_t* __restrict__ bro, int32_t step, const int32_t* __restrict__ bci,
    int32_t* __restrict__ ri_out, int32_t* __restrict__ ci_out, void* __restrict__ vo_) {
  const int64_t e = (int64_t)blockIdx.x * kT + threadIdx.x;
  if (e >= n) return;
  const int32_t r = ri[e], c = ci[e];
  const W x = static_cast<const W*>(v_)[e];
  int64_t lo = bro[(int64_t)r * step], hi = bro[((int64_t)r + 1) * step];  // B entries of the row before (r, c)
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if (LATER ? bci[mid] <= c : bci[mid] < c) lo = mid + 1; else hi = mid;
  }
  const int64_t o = e + lo;
  ri_out[o] = r;
  ci_out[o] = c;
  static_cast<W*>(vo_)[o] = x;
}

// The bitmap of used diagonals (bit col - row + nrows - 1) to ascending offsets.
__global__ void bit_count_kernel(const uint32_t* __restrict__ bits, int64_t words,
                                 int32_t* __restrict__ cnt) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < words) cnt[i] = __popc(bits[i]);
}

__global__ void bit_offsets_kernel(const uint32_t* __restrict__ bits,
                                   const int32_t* __restrict__ pos, int64_t words, int64_t nrows,
                                   int32_t* __restrict__ off) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= words) return;
  int64_t p = pos[i];
  for (uint32_t w = bits[i]; w; w &= w - 1)
    off[p++] = (int32_t)(i * 32 + __ffs(w) - 1 - nrows + 1);
}

__global__ __launch_bounds__(kT) void diag_hist_kernel(const int32_t* __restrict__ ri,
                                                       const int32_t* __restrict__ ci, int64_t nnz,
                                                       int64_t nrows, int32_t* __restrict__ cnt) {
  lds_histogram(nnz, cnt, [&](int64_t i) { return (int32_t)((int64_t)ci[i] - ri[i] + nrows - 1); });
}

__global__ void nonzero_flag_kernel(const int32_t* __restrict__ cnt, int64_t n, int32_t thr,
                                    int32_t* __restrict__ flag) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) flag[i] = cnt[i] >= thr ? 1 : 0;
}

__global__ void compact_offsets_kernel(const int32_t* __restrict__ flag,
                                       const int32_t* __restrict__ pos, int64_t n,
                                       int64_t nrows, int32_t* __restrict__ off) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n && flag[i]) off[pos[i]] = (int32_t)(i - nrows + 1);
}

// HDC sizes: selected diagonals (cnt >= thr), their entries, the rest
__global__ __launch_bounds__(kT) void hdc_sizes_kernel(
    const int32_t* __restrict__ cnt, int64_t n, int32_t thr,
    unsigned long long* out /* ndiag, dia_nnz, csr_nnz */) {
  const int64_t step = (int64_t)gridDim.x * kT;
  unsigned long long nd = 0, in = 0, rest = 0;
  for (int64_t i = (int64_t)blockIdx.x * kT + threadIdx.x; i < n; i += step) {
    const int32_t c = cnt[i];
    if (c >= thr) {
      nd++;
      in += c;
    } else {
      rest += c;
    }
  }
  auto add = [](unsigned long long u, unsigned long long v) { return u + v; };
  nd = block_reduce(nd, add);
  in = block_reduce(in, add);
  rest = block_reduce(rest, add);
  if (threadIdx.x == 0) {
    if (nd) atomicAdd(&out[0], nd);
    if (in) atomicAdd(&out[1], in);
    if (rest) atomicAdd(&out[2], rest);
  }
}

// ------------------------------------------------------------- dispatch by size
#define MPH_LAUNCH_W(kernel, vsize, grid, s, ...)                                  \
  do {                                                                              \
    if ((vsize) == 8)                                                               \
      hipLaunchKernelGGL(kernel<uint64_t>, grid, dim3(kT), 0, s, __VA_ARGS__);      \
    else if ((vsize) == 4)                                                          \
      hipLaunchKernelGGL(kernel<uint32_t>, grid, dim3(kT), 0, s, __VA_ARGS__);      \
    else                                                                            \
      hipLaunchKernelGGL(kernel<uint16_t>, grid, dim3(kT), 0, s, __VA_ARGS__);      \
  } while (0)

// kernels of (bool, word)
#define MPH_LAUNCH_BW(kernel, flag, vsize, grid, s, ...)                                \
  do {                                                                                  \
    if ((vsize) == 8)                                                                   \
      hipLaunchKernelGGL((kernel<flag, uint64_t>), grid, dim3(kT), 0, s, __VA_ARGS__);  \
    else if ((vsize) == 4)                                                              \
      hipLaunchKernelGGL((kernel<flag, uint32_t>), grid, dim3(kT), 0, s, __VA_ARGS__);  \
    else                                                                                \
      hipLaunchKernelGGL((kernel<flag, uint16_t>), grid, dim3(kT), 0, s, __VA_ARGS__);  \
  } while (0)

// (conversion moves values as raw words: 32-bit integer values too)
int check_vt(int vt) {
  if (vt != MPH_F64 && vt != MPH_F32 && vt != MPH_BF16 && vt != MPH_I32)
    return invalid("unknown value type");
  return MPH_OK;
}

int check_coo_in(int64_t nrows, int64_t ncols, int64_t nnz, const int32_t* ri,
                 const int32_t* ci, hipStream_t s) {
  if (nrows < 0 || ncols < 0 || nnz < 0) return invalid("negative size");
  if (nnz > 0 && !ri) return invalid("null COO row indices");
  MPH_CHECK_STATUS(check_index_range(ri, nnz, nrows, false, s, "COO row_indices"));
  if (ci) MPH_CHECK_STATUS(check_index_range(ci, nnz, ncols, false, s, "COO column_indices"));
  else if (nnz > 0 && ncols != INT32_MAX) return invalid("null COO column indices");
  return MPH_OK;
}

// run heads / scans shared by COO -> ELL and COO -> HYB
struct Runs {
  int32_t *head = nullptr, *hscan = nullptr, *runpos = nullptr;
};

int build_runs(const int32_t* ri, int64_t nnz, Tmp& t, Runs& R, hipStream_t s) {
  int64_t* tmp;
  MPH_CHECK_STATUS(t.alloc(&R.head, nnz));
  MPH_CHECK_STATUS(t.alloc(&R.hscan, nnz + 1));
  MPH_CHECK_STATUS(t.alloc(&R.runpos, nnz));
  MPH_CHECK_STATUS(t.alloc(&tmp, scan_tmp_elems(nnz)));
  hipLaunchKernelGGL(run_head_kernel, dim3(blocks_for(nnz)), dim3(kT), 0, s, ri, nnz, R.head);
  MPH_CHECK_STATUS(exclusive_scan_i32(R.head, R.hscan, nnz, tmp, s));
  hipLaunchKernelGGL(run_pos_kernel, dim3(blocks_for(nnz)), dim3(kT), 0, s, R.head, R.hscan, nnz,
                     R.runpos);
  MPH_HIP_CHECK(hipGetLastError());
  return MPH_OK;
}

// row histogram of COO rows (nrows counters)
int row_counts(const int32_t* ri, int64_t nnz, int64_t nrows, Tmp& t, int32_t** cnt,
               hipStream_t s) {
  MPH_CHECK_STATUS(t.alloc(cnt, nrows + 1));
  MPH_CHECK_STATUS(fill_i32(*cnt, nrows + 1, 0, s));
  if (nnz > 0)
    hipLaunchKernelGGL(row_hist_kernel, dim3(hist_blocks(nnz)), dim3(kT), 0, s, ri, nnz, *cnt);
  MPH_HIP_CHECK(hipGetLastError());
  return MPH_OK;
}

int check_coo_args(int64_t nrows, int64_t ncols, int64_t nnz, const int32_t* ri,
                   const int32_t* ci, bool cols) {
  if (nrows < 0 || ncols < 0 || nnz < 0) return invalid("negative size");
  if (nnz > 0 && !ri) return invalid("null COO row indices");
  if (nnz > 0 && cols && !ci) return invalid("null COO column indices");
  return MPH_OK;
}

// (diagonals are numbered in 32 bits)
int check_diagonals(int64_t nrows, int64_t ncols) {
  if (nrows + ncols - 1 > INT32_MAX) return invalid("more diagonals than the int32 range");
  return MPH_OK;
}

// The diagonals a COO list uses, and how its entries are ordered.
struct DiaScan {
  uint32_t* bits = nullptr;
  int32_t* pos = nullptr;
  int64_t words = 0, ndiag = 0;
  int32_t flags = 0;
};

int dia_scan(int64_t nrows, int64_t ncols, int64_t nnz, const int32_t* ri, const int32_t* ci,
             Tmp& t, DiaScan& D, hipStream_t s) {
  MPH_CHECK_STATUS(check_diagonals(nrows, ncols));
  D.words = ceil_div(nrows + ncols - 1, 32);
  int32_t *flags, *cnt, *hf, *hn;
  int64_t* tmp;
  MPH_CHECK_STATUS(t.alloc(&D.bits, D.words + 1));
  MPH_CHECK_STATUS(t.alloc(&cnt, D.words));
  MPH_CHECK_STATUS(t.alloc(&D.pos, D.words + 1));
  MPH_CHECK_STATUS(t.alloc(&tmp, scan_tmp_elems(D.words)));
  MPH_CHECK_STATUS(fill_zero(D.bits, sizeof(uint32_t) * (size_t)(D.words + 1), s));
  flags = reinterpret_cast<int32_t*>(D.bits + D.words);
  hipLaunchKernelGGL((coo_scan_kernel<true, false, kDiagBits>), dim3(scan_blocks(nnz)), dim3(kT), 0, s,
                     ri, ci, nnz, nrows, ncols, (int32_t*)nullptr, D.bits, flags);
  hipLaunchKernelGGL(bit_count_kernel, dim3(blocks_for(D.words)), dim3(kT), 0, s, D.bits, D.words,
                     cnt);
  MPH_HIP_CHECK(hipGetLastError());
  MPH_CHECK_STATUS(exclusive_scan_i32(cnt, D.pos, D.words, tmp, s));
  MPH_CHECK_STATUS(t.fetch(flags, &hf));
  MPH_CHECK_STATUS(t.fetch(D.pos + D.words, &hn));
  MPH_CHECK_STATUS(t.wait());
  D.flags = *hf;
  D.ndiag = *hn;
  return scan_status(D.flags);
}

// what coo_scan_kernel left of the row offsets (flags as it raised them; null:
// known to be kGaps)
int fill_gaps(const int32_t* ri, int64_t nnz, int64_t nrows, int32_t* ro, const int32_t* flags,
              hipStream_t s) {
  hipLaunchKernelGGL(gap_offsets_kernel, dim3(scan_blocks(nrows + 1)), dim3(kT), 0, s, ri, nnz, nrows,
                     ro, flags);
  MPH_HIP_CHECK(hipGetLastError());
  return MPH_OK;
}

// The rows of a COO list: the longest, the sum of min(length, K), the order
// of the entries and, rows not decreasing, their offsets.
struct RowScan {
  int32_t* ro = nullptr;
  int32_t flags = 0;
  int64_t longest = 0, clipped = 0;
};

int row_scan(int64_t nrows, int64_t nnz, const int32_t* ri, int64_t K, Tmp& t, RowScan& R,
             hipStream_t s) {
  unsigned long long *acc, *h;  // longest, clipped, flags
  const int32_t k = (int32_t)std::min<int64_t>(K, INT32_MAX);
  MPH_CHECK_STATUS(t.alloc(&R.ro, nrows + 1));
  MPH_CHECK_STATUS(t.alloc(&acc, 3));
  MPH_CHECK_STATUS(fill_zero(acc, 3 * sizeof(unsigned long long), s));
  int32_t* flags = reinterpret_cast<int32_t*>(acc + 2);
  if (nnz > 0)
    hipLaunchKernelGGL((coo_scan_kernel<false, true, kNoDiags>), dim3(scan_blocks(nnz)), dim3(kT), 0,
                       s, ri, (const int32_t*)nullptr, nnz, nrows, (int64_t)INT32_MAX, R.ro,
                       (uint32_t*)nullptr, flags);
  else
    MPH_CHECK_STATUS(fill_zero(R.ro, sizeof(int32_t) * (size_t)(nrows + 1), s));
  // (incomplete offsets give numbers not used)
  auto lengths = [&]() -> int {
    hipLaunchKernelGGL(row_lengths_kernel, dim3(reduce_blocks(nrows)), dim3(kT), 0, s, R.ro, nrows, k,
                       acc);
    MPH_HIP_CHECK(hipGetLastError());
    MPH_CHECK_STATUS(t.fetch(acc, &h, 3));
    return t.wait();
  };
  MPH_CHECK_STATUS(lengths());
  R.flags = (int32_t)h[2];
  MPH_CHECK_STATUS(scan_status(R.flags));
  if ((R.flags & (kGaps | kRowsDown)) == kGaps) {
    MPH_CHECK_STATUS(fill_gaps(ri, nnz, nrows, R.ro, nullptr, s));
    MPH_CHECK_STATUS(fill_zero(acc, 2 * sizeof(unsigned long long), s));
    MPH_CHECK_STATUS(lengths());
  }
  R.longest = (int64_t)h[0];
  R.clipped = (int64_t)h[1];
  if (R.flags & kRowsDown) {  // count the entries of each row
    int32_t *cnt, *mx, *hm;
    MPH_CHECK_STATUS(row_counts(ri, nnz, nrows, t, &cnt, s));
    MPH_CHECK_STATUS(t.alloc(&mx, 1));
    MPH_CHECK_STATUS(fill_zero(mx, sizeof(int32_t), s));
    MPH_CHECK_STATUS(fill_zero(acc, sizeof(unsigned long long), s));
    hipLaunchKernelGGL(max_kernel, dim3(reduce_blocks(nrows)), dim3(kT), 0, s, cnt, nrows, mx);
    hipLaunchKernelGGL(clipped_sum_kernel, dim3(reduce_blocks(nrows)), dim3(kT), 0, s, cnt, nrows,
                       k, acc);
    MPH_HIP_CHECK(hipGetLastError());
    MPH_CHECK_STATUS(t.fetch(mx, &hm));
    MPH_CHECK_STATUS(t.fetch(acc, &h));
    MPH_CHECK_STATUS(t.wait());
    R.longest = *hm;
    R.clipped = (int64_t)*h;
  }
  return MPH_OK;
}

// HDC keeps the diagonals with at least a fifth of the rows' entries.
int32_t hdc_threshold(int64_t nrows) { return (int32_t)((double)nrows * 0.2); }

struct HdcScan {
  int32_t* cnt = nullptr;  // entries per diagonal
  int32_t flags = 0;
  int64_t ndiag = 0, dia_nnz = 0, csr_nnz = 0;
};

int hdc_scan(int64_t nrows, int64_t ncols, int64_t nnz, const int32_t* ri, const int32_t* ci,
             Tmp& t, HdcScan& H, hipStream_t s) {
  MPH_CHECK_STATUS(check_diagonals(nrows, ncols));
  const int64_t nb = nrows + ncols - 1;
  unsigned long long *acc, *h;  // ndiag, dia_nnz, csr_nnz, flags
  MPH_CHECK_STATUS(t.alloc(&H.cnt, nb));
  MPH_CHECK_STATUS(t.alloc(&acc, 4));
  MPH_CHECK_STATUS(fill_zero(H.cnt, sizeof(int32_t) * (size_t)nb, s));
  MPH_CHECK_STATUS(fill_zero(acc, 4 * sizeof(unsigned long long), s));
  if (nnz > 0)
    hipLaunchKernelGGL((coo_scan_kernel<true, false, kDiagCounts>),
                       dim3((unsigned)std::min<int64_t>(scan_blocks(nnz), kCountBlocks)), dim3(kT),
                       0, s, ri, ci, nnz, nrows, ncols, (int32_t*)nullptr,
                       reinterpret_cast<uint32_t*>(H.cnt), reinterpret_cast<int32_t*>(acc + 3));
  hipLaunchKernelGGL(hdc_sizes_kernel, dim3(reduce_blocks(nb)), dim3(kT), 0, s, H.cnt, nb,
                     hdc_threshold(nrows), acc);
  MPH_HIP_CHECK(hipGetLastError());
  MPH_CHECK_STATUS(t.fetch(acc, &h, 4));
  MPH_CHECK_STATUS(t.wait());
  H.flags = (int32_t)h[3];
  MPH_CHECK_STATUS(scan_status(H.flags));
  H.ndiag = (int64_t)h[0];
  H.dia_nnz = (int64_t)h[1];
  H.csr_nnz = (int64_t)h[2];
  return MPH_OK;
}

// The values of a COO list on the diagonals of `off` (ascending); values of
// slots without an entry are 0.  `flags` as coo_scan_kernel leaves them.
// rest, if given, is set where an entry's diagonal is not among them.
int dia_place(int64_t nnz, const int32_t* ri, const int32_t* ci, const void* v, int vs,
              const int32_t* off, int64_t ndiag, int64_t pitch, int32_t flags, void* dv,
              int32_t* rest, Tmp& t, hipStream_t s) {
  MPH_CHECK_STATUS(fill_zero(dv, (size_t)vs * pitch * ndiag, s));
  if (nnz == 0) return MPH_OK;
  if (!(flags & kRepeated) && !rest) {
    MPH_LAUNCH_W(dia_place_once_kernel, vs, dim3(scan_blocks(nnz)), s, ri, ci, v, nnz, off, ndiag,
                 pitch, dv);
  } else {
    int32_t* win;
    MPH_CHECK_STATUS(t.alloc(&win, std::max<int64_t>(pitch * ndiag, 1)));
    MPH_CHECK_STATUS(fill_i32(win, pitch * ndiag, -1, s));
    hipLaunchKernelGGL(dia_claim_kernel, dim3(blocks_for(nnz)), dim3(kT), 0, s, ri, ci, nnz, off,
                       ndiag, pitch, win, rest);
    MPH_LAUNCH_W(dia_place_kernel, vs, dim3(blocks_for(nnz)), s, ri, ci, v, nnz, off, ndiag, pitch,
                 win, dv);
  }
  MPH_HIP_CHECK(hipGetLastError());
  return MPH_OK;
}

// The ELL part of a COO list: each row's first K entries, slots without one
// padded.  over, if given (nnz words, cleared), is set for the entries past
// the K-th; it needs rows that decrease.
int ell_place(int64_t nrows, int64_t nnz, const int32_t* ri, const int32_t* ci, const void* v,
              int vs, int64_t K, int64_t width, int64_t pitch, const RowScan& S, int32_t* eci,
              void* ev, int32_t* over, Tmp& t, hipStream_t s) {
  if (width * pitch == 0) return MPH_OK;
  if (!(S.flags & kRowsDown)) {
    if (pitch < kWave) {
      MPH_LAUNCH_W(ell_fill_slots_kernel, vs, dim3(blocks_for(width * pitch)), s, S.ro, ci, v, nrows,
                   K, width * pitch, pitch, eci, ev);
    } else {
      // few rows and many slots: the slots shared out too, 32 or more a
      // workgroup (one workgroup per 64 rows took 1.2 ms for 100 rows of 20k
      // entries, 24 ms for 4 of 500k)
      const int64_t gx = ceil_div(pitch, kWave);
      const int64_t gy = std::max<int64_t>(1, std::min(ceil_div(width, 32), kFillBlocks / gx));
      const int64_t per = ceil_div(width, gy);
      MPH_LAUNCH_W(ell_fill_rows_kernel, vs, dim3((unsigned)gx, (unsigned)ceil_div(width, per)), s,
                   S.ro, ci, v, nrows, K, width, per, pitch, eci, ev);
    }
    MPH_HIP_CHECK(hipGetLastError());
    return MPH_OK;
  }
  Runs R;
  int32_t* win;
  MPH_CHECK_STATUS(fill_i32(eci, width * pitch, -1, s));
  MPH_CHECK_STATUS(fill_zero(ev, (size_t)vs * width * pitch, s));
  MPH_CHECK_STATUS(build_runs(ri, nnz, t, R, s));
  MPH_CHECK_STATUS(t.alloc(&win, width * pitch));
  MPH_CHECK_STATUS(fill_i32(win, width * pitch, -1, s));
  hipLaunchKernelGGL(ell_claim_kernel, dim3(blocks_for(nnz)), dim3(kT), 0, s, ri, nnz, K, pitch,
                     R.head, R.hscan, R.runpos, win, over);
  MPH_LAUNCH_W(ell_place_kernel, vs, dim3(blocks_for(nnz)), s, ri, ci, v, nnz, K, pitch, R.head,
               R.hscan, R.runpos, win, eci, ev);
  MPH_HIP_CHECK(hipGetLastError());
  return MPH_OK;
}

// The entries of a DIA part in (row, column) order, shared by DIA -> COO and
// HDC -> COO; returns their count (and the first entry of each row and segment
// (segments(nrows, ndiag)) in rowpos, if given and the part is not empty).
template <typename W>
int emit_dia_part_w(int64_t nrows, int64_t ncols, int64_t ndiag, int64_t pitch,
                    const int32_t* off, const void* val, int vt, int64_t cap, int32_t* ri,
                    int32_t* ci, void* v, int32_t* rowpos, int64_t* count, hipStream_t s) {
  *count = 0;
  if (nrows == 0 || ndiag == 0) return MPH_OK;
  Tmp t(s);
  int32_t *cnt, *htot, *hoff;
  int64_t* tmp;
  const Segs g = segments(nrows, ndiag);
  const int64_t parts = nrows * g.n;
  MPH_CHECK_STATUS(t.alloc(&cnt, parts));
  if (!rowpos) MPH_CHECK_STATUS(t.alloc(&rowpos, parts + 1));
  MPH_CHECK_STATUS(t.alloc(&tmp, scan_tmp_elems(parts)));
  DiaSlots<W> src{static_cast<const W*>(val), off, nullptr, pitch, ncols,
                  vt == MPH_I32 ? (W)~(W)0 : RawT<sizeof(W)>::mag};
  auto row_count = g.n > 1 ? dia_row_count_kernel<true, W> : dia_row_count_kernel<false, W>;
  hipLaunchKernelGGL(row_count, dim3(blocks_for(parts)), dim3(kT), 0, s, src, nrows, (int32_t)ndiag, g,
                     cnt);
  MPH_HIP_CHECK(hipGetLastError());
  MPH_CHECK_STATUS(exclusive_scan_i32(cnt, rowpos, parts, tmp, s));
  MPH_CHECK_STATUS(t.fetch(rowpos + parts, &htot));
  // whether the offsets ascend: on the host, which then orders the slots, or,
  // where rows have several segments (counted in storage order) and the copy
  // may take long, on the device, the order left to the sort
  const bool few = g.n == 1;
  if (few) {
    MPH_CHECK_STATUS(t.fetch(off, &hoff, ndiag));
  } else {
    int32_t* d;
    MPH_CHECK_STATUS(t.alloc(&d, 1));
    MPH_CHECK_STATUS(fill_zero(d, sizeof(int32_t), s));
    hipLaunchKernelGGL((coo_scan_kernel<false, false, kNoDiags>), dim3(scan_blocks(ndiag)), dim3(kT),
                       0, s, off, (const int32_t*)nullptr, ndiag, (int64_t)INT32_MAX,
                       (int64_t)INT32_MAX, (int32_t*)nullptr, (uint32_t*)nullptr, d);
    MPH_HIP_CHECK(hipGetLastError());
    MPH_CHECK_STATUS(t.fetch(d, &hoff));
  }
  MPH_CHECK_STATUS(t.wait());
  const int64_t tot = *htot;
  if (tot > cap) return invalid("DIA holds more non-zeros than its nnz");
  const bool ascend = few ? std::is_sorted(hoff, hoff + ndiag) : !(*hoff & kRowsDown);
  if (few && !ascend) {
    // slots in ascending order of the offsets, equal ones in storage order
    std::vector<int32_t> ord(ndiag);
    for (int64_t d = 0; d < ndiag; d++) ord[d] = (int32_t)d;
    std::stable_sort(ord.begin(), ord.end(), [&](int32_t a, int32_t b) { return hoff[a] < hoff[b]; });
    int32_t *d_ord, *d_off, *h;
    MPH_CHECK_STATUS(t.alloc(&h, 2 * ndiag, true));
    MPH_CHECK_STATUS(t.alloc(&d_ord, 2 * ndiag));
    d_off = d_ord + ndiag;
    for (int64_t d = 0; d < ndiag; d++) {
      h[d] = ord[d];
      h[ndiag + d] = hoff[ord[d]];
    }
    MPH_HIP_CHECK(hipMemcpyAsync(d_ord, h, sizeof(int32_t) * 2 * (size_t)ndiag,
                                 hipMemcpyHostToDevice, s));
    src.ord = d_ord;
    src.off = d_off;
  }
  if (tot > 0) {
    emit_rows<W>(src, nrows, (int32_t)ndiag, g, rowpos, ri, ci, v, s);
    MPH_HIP_CHECK(hipGetLastError());
    if (!few && !ascend) MPH_CHECK_STATUS(sort_coo(tot, ri, ci, v, sizeof(W), false, s));
  }
  *count = tot;
  return MPH_OK;  // (t waits for the stream)
}

int emit_dia_part(int64_t nrows, int64_t ncols, int64_t ndiag, int64_t pitch,
                  const int32_t* off, const void* val, int vt, int64_t cap, int32_t* ri,
                  int32_t* ci, void* v, int32_t* rowpos, int64_t* count, hipStream_t s) {
  auto go = [&](auto tag) {
    return emit_dia_part_w<decltype(tag)>(nrows, ncols, ndiag, pitch, off, val, vt, cap, ri, ci, v,
                                          rowpos, count, s);
  };
  switch (value_size(vt)) {
    case 8: return go(uint64_t{});
    case 4: return go(uint32_t{});
    default: return go(uint16_t{});
  }
}

int zero_tail(int64_t from, int64_t nnz, int32_t* ri, int32_t* ci, void* v, int vsize,
              hipStream_t s) {
  if (from >= nnz) return MPH_OK;
  MPH_LAUNCH_W(zero_tail_kernel, vsize, dim3(blocks_for(nnz - from)), s, from, nnz, ri, ci,
               v);
  MPH_HIP_CHECK(hipGetLastError());
  return MPH_OK;
}

// ELL (+ a COO part of tnnz entries with row offsets tro, tail_sorted when
// each row's columns ascend) -> COO, rows in order: counts, a scan, the
// slots, the COO part.  Sorted only if the stored order is not already.
int ell_part_to_coo(int64_t nrows, int64_t nnz, int64_t width, int64_t pitch, const int32_t* eci,
                    const void* ev, const int32_t* tro, int64_t tnnz, const int32_t* tri,
                    const int32_t* tci, const void* tv, bool tail_unsorted, const char* too_many,
                    int vt, int32_t* ri_out, int32_t* ci_out, void* v_out, hipStream_t s) {
  const int vs = (int)value_size(vt);
  int64_t tot = 0;
  bool sorted = true;
  if (nrows > 0) {
    Tmp t(s);
    int32_t *cnt, *rowpos, *stats, *ht, *hs;
    int64_t* tmp;
    const Segs g = segments(nrows, width);
    const int64_t parts = nrows * g.n;
    MPH_CHECK_STATUS(t.alloc(&cnt, parts));
    MPH_CHECK_STATUS(t.alloc(&rowpos, parts + 1));
    MPH_CHECK_STATUS(t.alloc(&tmp, scan_tmp_elems(parts)));
    MPH_CHECK_STATUS(t.alloc(&stats, 2));
    MPH_CHECK_STATUS(fill_zero(stats, 2 * sizeof(int32_t), s));
    auto count = g.n > 1 ? ell_row_count_kernel<true> : ell_row_count_kernel<false>;
    hipLaunchKernelGGL(count, dim3(std::min(blocks_for(parts), 2048u)), dim3(kT), 0, s, eci, nrows,
                       width, pitch, g, tro, tci, cnt, stats);
    MPH_HIP_CHECK(hipGetLastError());
    MPH_CHECK_STATUS(exclusive_scan_i32(cnt, rowpos, parts, tmp, s));
    MPH_CHECK_STATUS(t.fetch(rowpos + parts, &ht));
    MPH_CHECK_STATUS(t.fetch(stats, &hs, 2));
    MPH_CHECK_STATUS(t.wait());
    tot = *ht;
    sorted = hs[0] == 0 && !tail_unsorted;
    const int32_t slots = hs[1];
    if (tot > nnz) return invalid(too_many);
    if (slots > 0) {
      auto emit = [&](auto tag) {
        using W = decltype(tag);
        emit_rows<W>(EllSlots<W>{eci, static_cast<const W*>(ev), pitch}, nrows, slots, g, rowpos,
                     ri_out, ci_out, v_out, s);
      };
      if (vs == 8) emit(uint64_t{});
      else if (vs == 4) emit(uint32_t{});
      else emit(uint16_t{});
    }
    if (tnnz > 0)
      MPH_LAUNCH_W(hyb_tail_emit_kernel, vs, dim3(blocks_for(tnnz)), s, tri, tci, tv, tnnz, tro,
                   rowpos, g.n, ri_out, ci_out, v_out);
    MPH_HIP_CHECK(hipGetLastError());
  }
  if (tot == nnz && sorted) return MPH_OK;
  MPH_CHECK_STATUS(zero_tail(tot, nnz, ri_out, ci_out, v_out, vs, s));
  return sort_coo(nnz, ri_out, ci_out, v_out, vs, false, s);
}

}  // namespace

}  // namespace mph

using namespace mph;

extern "C" {

int mph_convert_csr_to_coo(int64_t nrows, int64_t nnz, const int32_t* ro, const int32_t* ci,
                           const void* v, int vt, int32_t* ri_out, int32_t* ci_out,
                           void* v_out, mph_stream_t stream) {
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  MPH_CHECK_STATUS(check_vt(vt));
  if (nrows < 0 || nnz < 0) return invalid("negative size");
  MPH_CHECK_STATUS(check_row_offsets(ro, nrows, nnz, s, "CSR row_offsets"));
  if (nnz == 0) return MPH_OK;
  hipLaunchKernelGGL(expand_rows_kernel, dim3(scan_blocks(nnz)), dim3(kT), 0, s, ro, nrows, nnz,
                     (int64_t)0, ri_out);
  MPH_HIP_CHECK(hipGetLastError());
  if (ci_out != ci) MPH_CHECK_STATUS(copy_dev(ci_out, ci, sizeof(int32_t) * nnz, s));
  if (v_out != v) MPH_CHECK_STATUS(copy_dev(v_out, v, value_size(vt) * nnz, s));
  return MPH_OK;
}

int mph_convert_coo_to_csr(int64_t nrows, int64_t nnz, const int32_t* ri, const int32_t* ci,
                           const void* v, int vt, int32_t* ro_out, int32_t* ci_out,
                           void* v_out, mph_stream_t stream) {
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  MPH_CHECK_STATUS(check_vt(vt));
  MPH_CHECK_STATUS(check_coo_args(nrows, INT32_MAX, nnz, ri, nullptr, false));
  if (nnz == 0) return fill_zero(ro_out, sizeof(int32_t) * (size_t)(nrows + 1), s);
  const int vs = (int)value_size(vt);
  Tmp t(s);
  int32_t* flags;
  int32_t h = 0;
  MPH_CHECK_STATUS(t.alloc(&flags, 1));
  MPH_CHECK_STATUS(fill_zero(flags, sizeof(int32_t), s));
  hipLaunchKernelGGL((coo_scan_kernel<false, true, kNoDiags>), dim3(scan_blocks(nnz)), dim3(kT), 0, s,
                     ri, ci, nnz, nrows, (int64_t)INT32_MAX, ro_out, (uint32_t*)nullptr, flags);
  MPH_HIP_CHECK(hipGetLastError());
  MPH_CHECK_STATUS(t.read(flags, &h));
  MPH_CHECK_STATUS(scan_status(h));
  if (!(h & kRowsDown)) {
    t.idle = true;
    if (h & kGaps) MPH_CHECK_STATUS(fill_gaps(ri, nnz, nrows, ro_out, nullptr, s));
    if (ci_out != ci) MPH_CHECK_STATUS(copy_dev(ci_out, ci, sizeof(int32_t) * nnz, s));
    if (v_out != v) MPH_CHECK_STATUS(copy_dev(v_out, v, (size_t)vs * nnz, s));
    return MPH_OK;
  }
  // stable scatter by row in input order == stable sort by row
  int32_t* rows;
  MPH_CHECK_STATUS(t.alloc(&rows, nnz));
  MPH_CHECK_STATUS(radix_sort(nnz, bits_for(nrows - 1), 0, kByRow, ri, ci, v, vs, rows, ci_out,
                              v_out, s));
  MPH_CHECK_STATUS(fill_zero(flags, sizeof(int32_t), s));
  hipLaunchKernelGGL((coo_scan_kernel<false, true, kNoDiags>), dim3(scan_blocks(nnz)), dim3(kT), 0,
                     s, rows, (const int32_t*)nullptr, nnz, nrows, (int64_t)INT32_MAX, ro_out,
                     (uint32_t*)nullptr, flags);
  MPH_HIP_CHECK(hipGetLastError());
  return fill_gaps(rows, nnz, nrows, ro_out, flags, s);
}

int mph_convert_coo_to_dia_size(int64_t nrows, int64_t ncols, int64_t nnz, const int32_t* ri,
                                const int32_t* ci, int64_t* ndiag, mph_stream_t stream) {
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  if (!ndiag) return invalid("null ndiag");
  *ndiag = 0;
  MPH_CHECK_STATUS(check_coo_args(nrows, ncols, nnz, ri, ci, true));
  if (nnz == 0) return MPH_OK;
  Tmp t(s);
  DiaScan D;
  MPH_CHECK_STATUS(dia_scan(nrows, ncols, nnz, ri, ci, t, D, s));
  t.idle = true;
  *ndiag = D.ndiag;
  if (mph_exceeds_tolerance(nrows, nnz, D.ndiag)) {
    set_error("DiaMatrix fill-in would exceed maximum tolerance");
    return MPH_ERR_FORMAT_CONVERSION;
  }
  return MPH_OK;
}

int mph_convert_coo_to_dia(int64_t nrows, int64_t ncols, int64_t nnz, const int32_t* ri,
                           const int32_t* ci, const void* v, int vt, int64_t ndiag,
                           int64_t pitch, int32_t* off_out, void* val_out,
                           mph_stream_t stream) {
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  MPH_CHECK_STATUS(check_vt(vt));
  if (nnz == 0) return MPH_OK;
  MPH_CHECK_STATUS(check_coo_args(nrows, ncols, nnz, ri, ci, true));
  Tmp t(s);
  DiaScan D;
  MPH_CHECK_STATUS(dia_scan(nrows, ncols, nnz, ri, ci, t, D, s));
  if (mph_exceeds_tolerance(nrows, nnz, D.ndiag)) {
    set_error("DiaMatrix fill-in would exceed maximum tolerance");
    return MPH_ERR_FORMAT_CONVERSION;
  }
  if (D.ndiag != ndiag) return invalid("ndiag does not match the COO entries");
  if (pitch < nrows) return invalid("pitch must be >= nrows");
  hipLaunchKernelGGL(bit_offsets_kernel, dim3(blocks_for(D.words)), dim3(kT), 0, s, D.bits, D.pos,
                     D.words, nrows, off_out);
  MPH_HIP_CHECK(hipGetLastError());
  return dia_place(nnz, ri, ci, v, (int)value_size(vt), off_out, ndiag, pitch, D.flags, val_out,
                   nullptr, t, s);
}

int mph_convert_dia_to_coo(int64_t nrows, int64_t ncols, int64_t nnz, int64_t ndiag,
                           int64_t pitch, const int32_t* off, const void* val, int vt,
                           int32_t* ri_out, int32_t* ci_out, void* v_out,
                           mph_stream_t stream) {
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  MPH_CHECK_STATUS(check_vt(vt));
  if (nnz == 0) return MPH_OK;
  if (ndiag > 0 && pitch < nrows) return invalid("pitch must be >= nrows");
  const int vs = (int)value_size(vt);
  int64_t cnt = 0;
  MPH_CHECK_STATUS(emit_dia_part(nrows, ncols, ndiag, pitch, off, val, vt, nnz, ri_out, ci_out,
                                 v_out, nullptr, &cnt, s));
  if (cnt == nnz) return MPH_OK;  // in order
  MPH_CHECK_STATUS(zero_tail(cnt, nnz, ri_out, ci_out, v_out, vs, s));
  return sort_coo(nnz, ri_out, ci_out, v_out, vs, false, s);
}

int mph_convert_coo_to_ell_size(int64_t nrows, int64_t nnz, const int32_t* ri, int64_t* K,
                                mph_stream_t stream) {
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  if (!K) return invalid("null entries_per_row");
  *K = 0;
  MPH_CHECK_STATUS(check_coo_args(nrows, INT32_MAX, nnz, ri, nullptr, false));
  Tmp t(s);
  RowScan R;
  MPH_CHECK_STATUS(row_scan(nrows, nnz, ri, 0, t, R, s));
  t.idle = true;
  *K = R.longest;
  if (mph_exceeds_tolerance(nrows, nnz, R.longest)) {
    set_error("EllMatrix fill-in would exceed maximum tolerance");
    return MPH_ERR_FORMAT_CONVERSION;
  }
  return MPH_OK;
}

int mph_convert_coo_to_ell(int64_t nrows, int64_t nnz, const int32_t* ri, const int32_t* ci,
                           const void* v, int vt, int64_t K, int64_t width, int64_t pitch,
                           int32_t* ci_out, void* v_out, mph_stream_t stream) {
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  MPH_CHECK_STATUS(check_vt(vt));
  MPH_CHECK_STATUS(check_coo_args(nrows, INT32_MAX, nnz, ri, nullptr, false));
  Tmp t(s);
  RowScan R;
  MPH_CHECK_STATUS(row_scan(nrows, nnz, ri, 0, t, R, s));
  if (mph_exceeds_tolerance(nrows, nnz, R.longest)) {
    set_error("EllMatrix fill-in would exceed maximum tolerance");
    return MPH_ERR_FORMAT_CONVERSION;
  }
  if (R.longest != K) return invalid("entries_per_row does not match the COO entries");
  if (width < K || pitch < nrows) return invalid("ELL width / pitch too small");
  return ell_place(nrows, nnz, ri, ci, v, (int)value_size(vt), width, width, pitch, R, ci_out,
                   v_out, nullptr, t, s);
}

int mph_convert_ell_to_coo(int64_t nrows, int64_t nnz, int64_t width, int64_t pitch,
                           const int32_t* eci, const void* ev, int vt, int32_t* ri_out,
                           int32_t* ci_out, void* v_out, mph_stream_t stream) {
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  MPH_CHECK_STATUS(check_vt(vt));
  if (nnz == 0) return MPH_OK;
  if (width > 0 && pitch < nrows) return invalid("pitch must be >= nrows");
  return ell_part_to_coo(nrows, nnz, width, pitch, eci, ev, nullptr, 0, nullptr, nullptr, nullptr,
                         false, "ELL holds more entries than its nnz", vt, ri_out, ci_out, v_out,
                         s);
}

int mph_convert_coo_to_hyb_size(int64_t nrows, int64_t nnz, const int32_t* ri, int64_t* K,
                                int64_t* ell_nnz, int64_t* coo_nnz, mph_stream_t stream) {
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  if (!K || !ell_nnz || !coo_nnz) return invalid("null size outputs");
  if (nrows <= 0) return invalid("HYB needs at least one row");
  MPH_CHECK_STATUS(check_coo_args(nrows, INT32_MAX, nnz, ri, nullptr, false));
  Tmp t(s);
  RowScan R;
  *K = std::max<int64_t>(1, nnz / nrows);
  MPH_CHECK_STATUS(row_scan(nrows, nnz, ri, *K, t, R, s));
  t.idle = true;
  *ell_nnz = R.clipped;
  *coo_nnz = nnz - R.clipped;
  if (mph_exceeds_tolerance(nrows, R.clipped, *K)) {
    set_error("EllMatrix fill-in would exceed maximum tolerance");
    return MPH_ERR_FORMAT_CONVERSION;
  }
  return MPH_OK;
}

int mph_convert_coo_to_hyb(int64_t nrows, int64_t nnz, const int32_t* ri, const int32_t* ci,
                           const void* v, int vt, int64_t K, int64_t width, int64_t pitch,
                           int32_t* eci, void* ev, int32_t* cri, int32_t* cci, void* cv,
                           mph_stream_t stream) {
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  MPH_CHECK_STATUS(check_vt(vt));
  if (nrows <= 0) return invalid("HYB needs at least one row");
  MPH_CHECK_STATUS(check_coo_args(nrows, INT32_MAX, nnz, ri, nullptr, false));
  Tmp t(s);
  RowScan R;
  const int64_t k = std::max<int64_t>(1, nnz / nrows);
  MPH_CHECK_STATUS(row_scan(nrows, nnz, ri, k, t, R, s));
  if (mph_exceeds_tolerance(nrows, R.clipped, k)) {
    set_error("EllMatrix fill-in would exceed maximum tolerance");
    return MPH_ERR_FORMAT_CONVERSION;
  }
  if (k != K) return invalid("entries_per_row does not match the COO entries");
  if (width < K || pitch < nrows) return invalid("ELL width / pitch too small");
  const int vs = (int)value_size(vt);
  const int64_t cn = nnz - R.clipped;
  if (!(R.flags & kRowsDown)) {
    // row r's entries past the K-th follow those of the rows before it
    MPH_CHECK_STATUS(ell_place(nrows, nnz, ri, ci, v, vs, K, width, pitch, R, eci, ev, nullptr, t, s));
    if (cn == 0) return MPH_OK;
    int32_t *cnt, *opos;
    int64_t* tmp;
    MPH_CHECK_STATUS(t.alloc(&cnt, nrows));
    MPH_CHECK_STATUS(t.alloc(&opos, nrows + 1));
    MPH_CHECK_STATUS(t.alloc(&tmp, scan_tmp_elems(nrows)));
    hipLaunchKernelGGL(over_count_kernel, dim3(blocks_for(nrows)), dim3(kT), 0, s, R.ro, nrows,
                       (int32_t)K, cnt);
    MPH_CHECK_STATUS(exclusive_scan_i32(cnt, opos, nrows, tmp, s));
    MPH_LAUNCH_W(over_place_kernel, vs, dim3(scan_blocks(nnz)), s, ri, ci, v, nnz, K, R.ro, opos, cri,
                 cci, cv);
    MPH_HIP_CHECK(hipGetLastError());
    return MPH_OK;
  }
  int32_t *over, *opos;
  int64_t* tmp;
  MPH_CHECK_STATUS(t.alloc(&over, nnz));
  MPH_CHECK_STATUS(t.alloc(&opos, nnz + 1));
  MPH_CHECK_STATUS(t.alloc(&tmp, scan_tmp_elems(nnz)));
  MPH_CHECK_STATUS(fill_i32(over, nnz, 0, s));
  MPH_CHECK_STATUS(ell_place(nrows, nnz, ri, ci, v, vs, K, width, pitch, R, eci, ev, over, t, s));
  MPH_CHECK_STATUS(exclusive_scan_i32(over, opos, nnz, tmp, s));
  int32_t tail = 0;
  MPH_CHECK_STATUS(t.read(opos + nnz, &tail));
  if (tail > cn) return invalid("COO entries are not grouped by row (HYB tail overflow)");
  if (tail < cn) MPH_CHECK_STATUS(zero_tail(tail, cn, cri, cci, cv, vs, s));
  if (tail > 0)
    MPH_LAUNCH_W(tail_place_kernel, vs, dim3(blocks_for(nnz)), s, ri, ci, v, nnz, over, opos, cri,
                 cci, cv);
  MPH_HIP_CHECK(hipGetLastError());
  return MPH_OK;
}

int mph_convert_hyb_to_coo(int64_t nrows, int64_t nnz, int64_t width, int64_t pitch,
                           const int32_t* eci, const void* ev, int64_t coo_nnz,
                           const int32_t* cri, const int32_t* cci, const void* cv, int vt,
                           int32_t* ri_out, int32_t* ci_out, void* v_out,
                           mph_stream_t stream) {
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  MPH_CHECK_STATUS(check_vt(vt));
  if (nnz == 0) return MPH_OK;
  if (width > 0 && pitch < nrows) return invalid("pitch must be >= nrows");
  Tmp t(s);
  int32_t *tro, *flags, h = 0;
  int64_t P = std::max<int64_t>(coo_nnz, 0);
  MPH_CHECK_STATUS(t.alloc(&tro, std::max<int64_t>(nrows, 0) + 1));
  if (P > 0) {
    MPH_CHECK_STATUS(t.alloc(&flags, 1));
    MPH_CHECK_STATUS(fill_zero(flags, sizeof(int32_t), s));
    hipLaunchKernelGGL((coo_scan_kernel<true, true, kNoDiags>), dim3(scan_blocks(P)), dim3(kT), 0, s,
                       cri, cci, P, nrows, (int64_t)INT32_MAX, tro, (uint32_t*)nullptr, flags);
    MPH_HIP_CHECK(hipGetLastError());
    MPH_CHECK_STATUS(t.read(flags, &h));
    if (h & kBadRow) return invalid("HYB COO row_indices: index out of range");
    if (h & kRowsDown) {
      // the reference's forward walk consumes the longest row-sorted prefix
      int32_t *d, first = 0;
      MPH_CHECK_STATUS(t.alloc(&d, 1));
      MPH_CHECK_STATUS(fill_i32(d, 1, (int32_t)P, s));
      hipLaunchKernelGGL(first_descent_kernel, dim3(blocks_for(P)), dim3(kT), 0, s, cri, P, d);
      MPH_HIP_CHECK(hipGetLastError());
      MPH_CHECK_STATUS(t.read(d, &first));
      P = first;
      MPH_CHECK_STATUS(fill_zero(flags, sizeof(int32_t), s));
      hipLaunchKernelGGL((coo_scan_kernel<true, true, kNoDiags>), dim3(scan_blocks(P)), dim3(kT), 0, s,
                         cri, cci, P, nrows, (int64_t)INT32_MAX, tro, (uint32_t*)nullptr, flags);
      MPH_HIP_CHECK(hipGetLastError());
      MPH_CHECK_STATUS(t.read(flags, &h));
    }
    if (h & kGaps) MPH_CHECK_STATUS(fill_gaps(cri, P, nrows, tro, nullptr, s));
  } else {
    MPH_CHECK_STATUS(fill_zero(tro, sizeof(int32_t) * (size_t)(std::max<int64_t>(nrows, 0) + 1), s));
  }
  return ell_part_to_coo(nrows, nnz, width, pitch, eci, ev, tro, P, cri, cci, cv,
                         (h & kUnsorted) != 0, "HYB holds more entries than its nnz", vt, ri_out,
                         ci_out, v_out, s);
}

int mph_convert_coo_to_hdc_size(int64_t nrows, int64_t ncols, int64_t nnz, const int32_t* ri,
                                const int32_t* ci, int64_t* ndiag, int64_t* dia_nnz,
                                int64_t* csr_nnz, mph_stream_t stream) {
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  if (!ndiag || !dia_nnz || !csr_nnz) return invalid("null size outputs");
  if (nrows <= 0 || ncols <= 0) return invalid("HDC needs a non-empty shape");
  MPH_CHECK_STATUS(check_coo_args(nrows, ncols, nnz, ri, ci, true));
  Tmp t(s);
  HdcScan H;
  MPH_CHECK_STATUS(hdc_scan(nrows, ncols, nnz, ri, ci, t, H, s));
  t.idle = true;
  *ndiag = H.ndiag;
  *dia_nnz = H.dia_nnz;
  *csr_nnz = H.csr_nnz;
  if (mph_exceeds_tolerance(nrows, *dia_nnz, *ndiag)) {
    set_error("DiaMatrix fill-in would exceed maximum tolerance");
    return MPH_ERR_FORMAT_CONVERSION;
  }
  return MPH_OK;
}

int mph_convert_coo_to_hdc(int64_t nrows, int64_t ncols, int64_t nnz, const int32_t* ri,
                           const int32_t* ci, const void* v, int vt, int64_t ndiag,
                           int64_t pitch, int32_t* off_out, void* dv, int32_t* csr_ro,
                           int32_t* csr_ci, void* csr_v, mph_stream_t stream) {
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  MPH_CHECK_STATUS(check_vt(vt));
  if (nrows <= 0 || ncols <= 0) return invalid("HDC needs a non-empty shape");
  MPH_CHECK_STATUS(check_coo_args(nrows, ncols, nnz, ri, ci, true));
  Tmp t(s);
  HdcScan H;
  MPH_CHECK_STATUS(hdc_scan(nrows, ncols, nnz, ri, ci, t, H, s));
  if (mph_exceeds_tolerance(nrows, H.dia_nnz, H.ndiag)) {
    set_error("DiaMatrix fill-in would exceed maximum tolerance");
    return MPH_ERR_FORMAT_CONVERSION;
  }
  if (H.ndiag != ndiag) return invalid("ndiag does not match the COO entries");
  if (ndiag > 0 && pitch < nrows) return invalid("pitch must be >= nrows");
  const int64_t cn = H.csr_nnz, nb = nrows + ncols - 1;
  const int vs = (int)value_size(vt);
  const int32_t thr = hdc_threshold(nrows);
  int32_t *flag, *pos;
  int64_t* tmp;
  MPH_CHECK_STATUS(t.alloc(&tmp, scan_tmp_elems(std::max(nb, std::max(nnz, nrows)))));
  if (ndiag > 0) {
    MPH_CHECK_STATUS(t.alloc(&flag, nb));
    MPH_CHECK_STATUS(t.alloc(&pos, nb + 1));
    hipLaunchKernelGGL(nonzero_flag_kernel, dim3(blocks_for(nb)), dim3(kT), 0, s, H.cnt, nb, thr,
                       flag);
    MPH_CHECK_STATUS(exclusive_scan_i32(flag, pos, nb, tmp, s));
    hipLaunchKernelGGL(compact_offsets_kernel, dim3(blocks_for(nb)), dim3(kT), 0, s, flag, pos, nb,
                       nrows, off_out);
    MPH_HIP_CHECK(hipGetLastError());
  }
  // core/src/impl/Hdc/Serial/Morpheus_Convert_Impl.hpp:169-195 records the
  // midpoint bin as offset 0 (its true offset only for square matrices) and
  // then sorts the offsets
  const int64_t mid = nb / 2;
  if (nrows != ncols && ndiag > 0) {
    int32_t sel = 0;
    MPH_CHECK_STATUS(t.read(flag + mid, &sel));
    if (sel) {
      std::vector<int32_t> h(ndiag);
      MPH_CHECK_STATUS(t.read(off_out, h.data(), ndiag));
      const int32_t dmid = (int32_t)(mid - nrows + 1);
      for (auto& o : h)
        if (o == dmid) { o = 0; break; }
      std::sort(h.begin(), h.end());
      MPH_HIP_CHECK(hipMemcpyAsync(off_out, h.data(), sizeof(int32_t) * ndiag,
                                   hipMemcpyHostToDevice, s));
      MPH_HIP_CHECK(hipStreamSynchronize(s));
    }
  }
  // DIA part (later entry wins), the rest in input order to the CSR part
  int32_t *rows_rest, nrest = 0;
  MPH_CHECK_STATUS(t.alloc(&rows_rest, std::max<int64_t>(cn, 1)));
  if (nnz > 0 && !(H.flags & kRepeated)) {
    const unsigned tiles = scan_blocks(nnz);
    int32_t *tile_n, *tile_pos;
    MPH_CHECK_STATUS(t.alloc(&tile_n, tiles));
    MPH_CHECK_STATUS(t.alloc(&tile_pos, (int64_t)tiles + 1));
    MPH_CHECK_STATUS(fill_zero(dv, (size_t)vs * pitch * ndiag, s));
    hipLaunchKernelGGL((hdc_split_kernel<false, uint16_t>), dim3(tiles), dim3(kT), 0, s, ri, ci, v,
                       nnz, off_out, ndiag, pitch, dv, tile_n, (const int32_t*)nullptr,
                       (int32_t*)nullptr, (int32_t*)nullptr, (void*)nullptr);
    MPH_CHECK_STATUS(exclusive_scan_i32(tile_n, tile_pos, tiles, tmp, s));
    MPH_CHECK_STATUS(t.read(tile_pos + tiles, &nrest));
    if (nrest > cn) return invalid("HDC CSR part overflow (non-square midpoint diagonal)");
    MPH_LAUNCH_BW(hdc_split_kernel, true, vs, dim3(tiles), s, ri, ci, v, nnz, off_out, ndiag, pitch,
                  dv, (int32_t*)nullptr, tile_pos, rows_rest, csr_ci, csr_v);
  } else {
    int32_t *rest, *rpos;
    MPH_CHECK_STATUS(t.alloc(&rest, nnz));
    MPH_CHECK_STATUS(t.alloc(&rpos, nnz + 1));
    MPH_CHECK_STATUS(fill_i32(rest, nnz, 0, s));
    MPH_CHECK_STATUS(
        dia_place(nnz, ri, ci, v, vs, off_out, ndiag, pitch, H.flags, dv, rest, t, s));
    MPH_CHECK_STATUS(exclusive_scan_i32(rest, rpos, nnz, tmp, s));
    MPH_CHECK_STATUS(t.read(rpos + nnz, &nrest));
    if (nrest > cn) return invalid("HDC CSR part overflow (non-square midpoint diagonal)");
    if (nrest > 0)
      MPH_LAUNCH_W(tail_place_kernel, vs, dim3(blocks_for(nnz)), s, ri, ci, v, nnz, rest, rpos,
                   rows_rest, csr_ci, csr_v);
  }
  MPH_HIP_CHECK(hipGetLastError());
  // CSR part: per-row counts of the rest, exclusive scan, row_offsets[n] = cn
  if (nrest == 0) {
    MPH_CHECK_STATUS(fill_zero(csr_ro, sizeof(int32_t) * (size_t)(nrows + 1), s));
  } else if (!(H.flags & kRowsDown)) {
    int32_t* flags;
    MPH_CHECK_STATUS(t.alloc(&flags, 1));
    MPH_CHECK_STATUS(fill_zero(flags, sizeof(int32_t), s));
    hipLaunchKernelGGL((coo_scan_kernel<false, true, kNoDiags>), dim3(scan_blocks(nrest)), dim3(kT),
                       0, s, rows_rest, (const int32_t*)nullptr, (int64_t)nrest, nrows,
                       (int64_t)INT32_MAX, csr_ro, (uint32_t*)nullptr, flags);
    MPH_HIP_CHECK(hipGetLastError());
    MPH_CHECK_STATUS(fill_gaps(rows_rest, nrest, nrows, csr_ro, flags, s));
  } else {
    int32_t* rcnt;
    MPH_CHECK_STATUS(row_counts(rows_rest, nrest, nrows, t, &rcnt, s));
    MPH_CHECK_STATUS(exclusive_scan_i32(rcnt, csr_ro, nrows, tmp, s));
  }
  // the reference writes row_offsets[nrows] = csr_nnz (:225)
  hipLaunchKernelGGL(fill_i32_kernel, dim3(1), dim3(1), 0, s, csr_ro + nrows, (int64_t)1,
                     (int32_t)cn);
  if (nrest < cn) {
    MPH_CHECK_STATUS(fill_i32(csr_ci + nrest, cn - nrest, 0, s));
    MPH_CHECK_STATUS(fill_zero(static_cast<uint8_t*>(csr_v) + (size_t)vs * nrest,
                               (size_t)vs * (cn - nrest), s));
  }
  MPH_HIP_CHECK(hipGetLastError());
  return MPH_OK;
}

int mph_convert_hdc_to_coo(int64_t nrows, int64_t ncols, int64_t nnz, int64_t ndiag,
                           int64_t pitch, const int32_t* doff, const void* dval,
                           int64_t csr_nnz, const int32_t* csr_ro, const int32_t* csr_ci,
                           const void* csr_v, int vt, int32_t* ri_out, int32_t* ci_out,
                           void* v_out, mph_stream_t stream) {
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  MPH_CHECK_STATUS(check_vt(vt));
  if (nnz == 0) return MPH_OK;
  if (ndiag > 0 && pitch < nrows) return invalid("pitch must be >= nrows");
  MPH_CHECK_STATUS(check_row_offsets(csr_ro, nrows, csr_nnz, s, "HDC CSR row_offsets"));
  const int vs = (int)value_size(vt);
  int64_t nd = 0;
  if (csr_nnz == 0) {
    MPH_CHECK_STATUS(emit_dia_part(nrows, ncols, ndiag, pitch, doff, dval, vt, nnz, ri_out, ci_out,
                                   v_out, nullptr, &nd, s));
    if (nd == nnz) return MPH_OK;  // in order
    MPH_CHECK_STATUS(zero_tail(nd, nnz, ri_out, ci_out, v_out, vs, s));
    return sort_coo(nnz, ri_out, ci_out, v_out, vs, false, s);
  }
  // the CSR part's rows, and whether each row's columns ascend
  Tmp t(s);
  int32_t *crow, *rowpos, *flags, h = 0;
  MPH_CHECK_STATUS(t.alloc(&crow, csr_nnz));
  MPH_CHECK_STATUS(t.alloc(&flags, 1));
  MPH_CHECK_STATUS(fill_zero(flags, sizeof(int32_t), s));
  hipLaunchKernelGGL(expand_rows_kernel, dim3(scan_blocks(csr_nnz)), dim3(kT), 0, s, csr_ro, nrows,
                     csr_nnz, (int64_t)0, crow);
  hipLaunchKernelGGL((coo_scan_kernel<true, false, kNoDiags>), dim3(scan_blocks(csr_nnz)), dim3(kT),
                     0, s, crow, csr_ci, csr_nnz, nrows, ncols, (int32_t*)nullptr,
                     (uint32_t*)nullptr, flags);
  MPH_HIP_CHECK(hipGetLastError());
  MPH_CHECK_STATUS(t.read(flags, &h));
  const bool sorted = !(h & kUnsorted);
  bool in_order;
  if (sorted && !(h & kBadCol) && ndiag > 0 && nrows > 0) {
    // both parts in order: the DIA part's entries, then both lists merged (a
    // DIA entry before the CSR entries of its row and column, as the stable
    // sort of the DIA entries followed by the CSR entries leaves them)
    int32_t *dri, *dci;
    uint8_t* dv;
    const int64_t cap = std::min(nnz, nrows * ndiag);
    const Segs dia_segs = segments(nrows, ndiag);
    MPH_CHECK_STATUS(t.alloc(&rowpos, nrows * dia_segs.n + 1));
    MPH_CHECK_STATUS(t.alloc(&dri, cap));
    MPH_CHECK_STATUS(t.alloc(&dci, cap));
    MPH_CHECK_STATUS(t.alloc(&dv, cap * vs));
    MPH_CHECK_STATUS(emit_dia_part(nrows, ncols, ndiag, pitch, doff, dval, vt, cap, dri, dci, dv,
                                   rowpos, &nd, s));
    if (nd + csr_nnz > nnz) return invalid("HDC holds more entries than its nnz");
    if (nd > 0)
      MPH_LAUNCH_BW(merge_rows_kernel, false, vs, dim3(blocks_for(nd)), s, dri, dci, dv, nd, csr_ro, 1,
                    csr_ci, ri_out, ci_out, v_out);
    MPH_LAUNCH_BW(merge_rows_kernel, true, vs, dim3(blocks_for(csr_nnz)), s, crow, csr_ci, csr_v,
                  csr_nnz, rowpos, dia_segs.n, dci, ri_out, ci_out, v_out);
    MPH_HIP_CHECK(hipGetLastError());
    in_order = true;
  } else {
    // the DIA part's entries, then the CSR part's
    MPH_CHECK_STATUS(emit_dia_part(nrows, ncols, ndiag, pitch, doff, dval, vt, nnz, ri_out, ci_out,
                                   v_out, nullptr, &nd, s));
    if (nd + csr_nnz > nnz) return invalid("HDC holds more entries than its nnz");
    MPH_CHECK_STATUS(copy_dev(ri_out + nd, crow, sizeof(int32_t) * csr_nnz, s));
    MPH_CHECK_STATUS(copy_dev(ci_out + nd, csr_ci, sizeof(int32_t) * csr_nnz, s));
    MPH_CHECK_STATUS(copy_dev(static_cast<uint8_t*>(v_out) + (size_t)vs * nd, csr_v,
                              (size_t)vs * csr_nnz, s));
    in_order = sorted && nd == 0;
  }
  if (nd + csr_nnz == nnz && in_order) return MPH_OK;
  MPH_CHECK_STATUS(zero_tail(nd + csr_nnz, nnz, ri_out, ci_out, v_out, vs, s));
  return sort_coo(nnz, ri_out, ci_out, v_out, vs, false, s);
}

int mph_coo_sort_by_row_and_column(int64_t nnz, int32_t* ri, int32_t* ci, void* v, int vt,
                                   mph_stream_t stream) {
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  MPH_CHECK_STATUS(check_vt(vt));
  if (nnz <= 1) return MPH_OK;
  return sort_coo(nnz, ri, ci, v, (int)value_size(vt), true, s);
}

int mph_coo_is_sorted(int64_t nnz, const int32_t* ri, const int32_t* ci, int* sorted,
                      mph_stream_t stream) {
  if (!sorted) return invalid("null output");
  return is_sorted_dev(ri, ci, nnz, reinterpret_cast<hipStream_t>(stream), sorted);
}

int mph_coo_count_nnz_per_diagonal(int64_t nrows, int64_t ncols, int64_t nnz, const int32_t* ri,
                                   const int32_t* ci, int32_t* out, int init,
                                   mph_stream_t stream) {
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  MPH_CHECK_STATUS(check_coo_in(nrows, ncols, nnz, ri, ci, s));
  const int64_t nb = nrows + ncols - 1;
  if (init) MPH_CHECK_STATUS(fill_i32(out, nb, 0, s));
  if (nnz > 0)
    hipLaunchKernelGGL(diag_hist_kernel, dim3(hist_blocks(nnz)), dim3(kT), 0, s, ri, ci, nnz,
                       nrows, out);
  MPH_HIP_CHECK(hipGetLastError());
  return MPH_OK;
}

}  // extern "C"
