// spmv_dia_ell.hip -- DIA and ELL SpMV / SpMM.
//
// Replaces core/src/impl/Dia/HIP/Morpheus_Multiply_Impl.hpp:41-85 (kernel
// core/src/impl/Dia/Kernels/Morpheus_Multiply_Impl.hpp:37-84) and
// core/src/impl/Ell/HIP/Morpheus_Multiply_Impl.hpp:41-80 (kernel
// core/src/impl/Ell/Kernels/Morpheus_Multiply_Impl.hpp:37-65).
//
// Both are one thread per row over column-major (LayoutLeft) storage, so
// every diagonal / slot is one fully coalesced, non-temporal stream across a
// wavefront.  DIA offsets are wave-uniform and come through scalar loads;
// the x entries of clusters of nearby diagonals are staged in LDS per
// workgroup (dia_staged_kernel), and y is written once (the reference zeroes
// y in a separate launch and then read-modify-writes it per 256-diagonal
// chunk, and skips the zeroing when ndiag == 0).  ELL visits entries_per_row slots,
// not the 32-padded width, when the analysis has confirmed that the slots
// beyond entries_per_row hold only the -1 padding.  FP32 / BF16 SpMV of DIA, and
// of ELL with few slots and many rows, takes two adjacent rows per thread
// (row-pair kernels below); FP32 / BF16 rows of
// more than kCompensateLen diagonals / slots take a Dot2-compensated kernel.
// SpMM gives each row a lane group (16 bytes of its columns per lane); DIA may
// give each group 4 consecutive rows, which share the X rows of each run of
// consecutive diagonals (dia_spmm_form).  A split FP64 HDC
// whose CSR rows are short adds them in the staged DIA pass.
#include <algorithm>
#include <cstdlib>

#include "mph_internal.hpp"

namespace mph {

template <typename V>
struct DiaArgs {
  int64_t nrows, ncols;
  int32_t ndiag;
  int64_t pitch;
  const int32_t* __restrict__ off;
  const V* __restrict__ val;
  const typename vtraits<V>::vec* __restrict__ x;
  typename vtraits<V>::vec* __restrict__ y;
  int32_t ld;
  int init;
  // dia_staged_kernel<V, true>: HDC's CSR part, added per row after the
  // diagonals
  const int32_t* __restrict__ tro;
  const int32_t* __restrict__ tci;
  const V* __restrict__ tval;
  // dia_spmm_runs_kernel: workgroups of a plane, and an XCD's share of them
  // (0: rows in order), see dia_plane_block
  int32_t plane, plane_xcd;
};

// The row block of a workgroup, -1 for none.  In order, each XCD walks one
// contiguous range of rows, and an X row that the outermost diagonals reach
// comes back a reach of rows later, when its L2 line is gone.  A grid's
// outermost diagonals lie a plane of nodes away: each XCD then takes an
// eighth of every plane, plane after plane, so that the rows its neighbours
// read are still in its L2 (27-point 160^3, 16 FP64 columns: 2.47 GB fetched
// -> 1.47).
template <typename V>
__device__ __forceinline__ int64_t dia_plane_block(const DiaArgs<V>& a, int64_t rows_per_block) {
  if (a.plane == 0) return xcd_remap(blockIdx.x, gridDim.x);
  const uint32_t i = blockIdx.x / kNumXcd;
  const int64_t c = (int64_t)(blockIdx.x % kNumXcd) * a.plane_xcd + i % a.plane_xcd;
  const int64_t b = (int64_t)(i / a.plane_xcd) * a.plane + c;
  return c < a.plane && b * rows_per_block < a.nrows ? b : -1;
}

// t[u][q] += v[u][w] * x[c[u][w]][q] over a batch of B diagonals / slots,
// skipping c < 0.  The x loads are unconditional (c < 0 reads x[0]) and the
// sums are selected rather than branched, so the batch's gathers are all in
// flight before the first product: under a branch each gather was waited on
// before the next was issued.  Same fused multiply-adds in the same order
// as t += v * x.  With many right-hand sides (KR * RPT > 2) the gathers of
// one diagonal / slot are issued together instead, to bound registers.
template <typename V, int KR, int RPT, int B>
__device__ __forceinline__ void batch_fma(typename vtraits<V>::acc (&t)[RPT][KR],
                                          const V (&v)[RPT][B], const int64_t (&c)[RPT][B],
                                          const typename vtraits<V>::vec* __restrict__ x,
                                          int32_t ld) {
  using Acc = typename vtraits<V>::acc;
  if constexpr (KR * RPT <= 2) {
    Acc xq[RPT][B][KR];
#pragma unroll
    for (int w = 0; w < B; w++)
#pragma unroll
      for (int u = 0; u < RPT; u++)
#pragma unroll
        for (int q = 0; q < KR; q++) xq[u][w][q] = (Acc)x[(c[u][w] >= 0 ? c[u][w] : 0) * ld + q];
#pragma unroll
    for (int w = 0; w < B; w++)
#pragma unroll
      for (int u = 0; u < RPT; u++)
#pragma unroll
        for (int q = 0; q < KR; q++) {
          const Acc f = __builtin_fma(vtraits<V>::widen(v[u][w]), xq[u][w][q], t[u][q]);
          t[u][q] = c[u][w] >= 0 ? f : t[u][q];
        }
  } else {
#pragma unroll
    for (int w = 0; w < B; w++)
#pragma unroll
      for (int u = 0; u < RPT; u++) {
        const int64_t xc = c[u][w] >= 0 ? c[u][w] : 0;
#pragma unroll
        for (int q = 0; q < KR; q++) {
          const Acc xq = (Acc)x[xc * ld + q];
          if (c[u][w] >= 0) t[u][q] += vtraits<V>::widen(v[u][w]) * xq;
        }
      }
  }
}

template <typename V, int KR, int RPT>
__global__ __launch_bounds__(256) void dia_kernel(DiaArgs<V> a) {
  using Acc = typename vtraits<V>::acc;
  using Vec = typename vtraits<V>::vec;
  const uint32_t b = xcd_remap(blockIdx.x, gridDim.x);
  const int64_t row0 = ((int64_t)b * 256 * RPT) + threadIdx.x;
  Acc t[RPT][KR];
#pragma unroll
  for (int u = 0; u < RPT; u++)
#pragma unroll
    for (int q = 0; q < KR; q++) t[u][q] = 0;
  // batches of 8 diagonals: offsets, values and x entries of the batch are
  // all requested before any of them is consumed
  // (The branch-free loads of ell_kernel made this kernel slower: S7
  // 31.6 -> 34.0 us, S27 210 -> 223 us in FP64; its value loads already
  // stream at the read rate of the device.)
  for (int d0 = 0; d0 < a.ndiag; d0 += 8) {
    V v[RPT][8];
    int64_t c[RPT][8];
#pragma unroll
    for (int w = 0; w < 8; w++) {
      const int d = d0 + w;
      const int64_t o = d < a.ndiag ? (int64_t)a.off[d] : 0;
#pragma unroll
      for (int u = 0; u < RPT; u++) {
        const int64_t row = row0 + u * 256;
        const int64_t col = row + o;
        const bool ok = d < a.ndiag && row < a.nrows && col >= 0 && col < a.ncols;
        c[u][w] = ok ? col : -1;
        v[u][w] = ok ? ld_stream(a.val + a.pitch * d + row) : V{};
      }
    }
#pragma unroll
    for (int u = 0; u < RPT; u++) hold_raw(v[u]);
#pragma unroll
    for (int w = 0; w < 8; w++)
#pragma unroll
      for (int u = 0; u < RPT; u++)
        if (c[u][w] >= 0)
#pragma unroll
          for (int q = 0; q < KR; q++)
            t[u][q] += vtraits<V>::widen(v[u][w]) * (Acc)a.x[c[u][w] * a.ld + q];
  }
#pragma unroll
  for (int u = 0; u < RPT; u++) {
    const int64_t row = row0 + u * 256;
    if (row < a.nrows) {
#pragma unroll
      for (int q = 0; q < KR; q++) {
        Vec* yp = a.y + row * a.ld + q;
        *yp = a.init ? (Vec)t[u][q] : (Vec)((Acc)*yp + t[u][q]);
      }
    }
  }
}

// The x entries a workgroup stages, in two halves: the loads into registers
// (N a thread, LDS entries first + 256 k), and their stores to LDS, so that a
// kernel's first values are requested between the two and one round trip to
// memory serves both (FP64: 27-point 160^3 186 -> 181 us, 7-point 128^3 29.2
// -> 28.1 us, 4M rows of 9 diagonals 69 -> 64.6 us).  WIN: rows beyond 256 (each cluster's
// window is that much longer, and starts that much later per cluster).
template <typename Vec, int N, int WIN>
__device__ __forceinline__ void stage_load(const DiaStage& cl, const Vec* __restrict__ x,
                                           int64_t ncols, int64_t r0, int first, Vec (&xr)[N]) {
  const int total = cl.base[cl.n - 1] + cl.len[cl.n - 1] + WIN * cl.n;
#pragma unroll
  for (int k = 0; k < N; k++) {
    const int e = first + (int)threadIdx.x + 256 * k;
    int32_t shift = cl.omin[0] - cl.base[0];
    for (int c = 1; c < cl.n; c++)
      if (e >= cl.base[c] + WIN * c) shift = cl.omin[c] - cl.base[c] - WIN * c;
    const int64_t col = r0 + shift + e;
    xr[k] = (e < total && col >= 0 && col < ncols) ? x[col] : (Vec)0;
  }
}

template <typename Vec, int N, int WIN>
__device__ __forceinline__ void stage_store(const DiaStage& cl, Vec* xs, int first,
                                            const Vec (&xr)[N]) {
  const int total = cl.base[cl.n - 1] + cl.len[cl.n - 1] + WIN * cl.n;
#pragma unroll
  for (int k = 0; k < N; k++) {
    const int e = first + (int)threadIdx.x + 256 * k;
    if (e < total) xs[e] = xr[k];
  }
}

// LDS entries a thread requests before the first values; those of a wide
// stage beyond them follow after (requesting all of the 27-point stencil's
// windows ahead, 8 a thread, cost its FP64 kernel more in registers than it
// saved: 180 -> 184 us, and the 7-point stencil's 28.1 -> 31.0 us)
constexpr int kStageAhead = 4;

// DIA SpMV with x staged in LDS per cluster of nearby diagonals (the
// clusters come from dia_analyse).  For each cluster of two or more
// diagonals the workgroup's 256 rows read x[r0 + omin .. r0 + 255 + omax]
// once, coalesced, into LDS; every diagonal of the cluster then takes its x
// entries from there instead of a global load (on the 27-point stencil the
// x loads per row drop from 27 to about 7).  Diagonals are summed in storage
// order, as dia_kernel sums them: the two kernels give identical results.
template <typename V, bool TAIL = false>
__global__ __launch_bounds__(256) void dia_staged_kernel(DiaArgs<V> a, DiaStage cl) {
  using Acc = typename vtraits<V>::acc;
  using Vec = typename vtraits<V>::vec;
  __shared__ Vec xs[kDiaStageMax];
  const int64_t r0 = (int64_t)xcd_remap(blockIdx.x, gridDim.x) * 256;
  const int64_t row = r0 + threadIdx.x;
  Vec xr[kStageAhead];
  stage_load<Vec, kStageAhead, 0>(cl, a.x, a.ncols, r0, 0, xr);
  Acc t = 0;
  for (int d0 = 0; d0 < a.ndiag; d0 += 8) {
    V v[8];
    int64_t col[8];
    bool ok[8];
#pragma unroll
    for (int w = 0; w < 8; w++) {
      const int d = d0 + w;
      const int64_t o = d < a.ndiag ? (int64_t)a.off[d] : 0;
      col[w] = row + o;
      ok[w] = d < a.ndiag && row < a.nrows && col[w] >= 0 && col[w] < a.ncols;
      v[w] = ok[w] ? ld_stream(a.val + a.pitch * d + row) : V{};
    }
    if (d0 == 0) {
      stage_store<Vec, kStageAhead, 0>(cl, xs, 0, xr);
      const int total = cl.base[cl.n - 1] + cl.len[cl.n - 1];
      for (int first = 256 * kStageAhead; first < total; first += 256 * kStageAhead) {
        stage_load<Vec, kStageAhead, 0>(cl, a.x, a.ncols, r0, first, xr);
        stage_store<Vec, kStageAhead, 0>(cl, xs, first, xr);
      }
      __syncthreads();
    }
    hold_raw(v);
#pragma unroll
    for (int w = 0; w < 8; w++) {
      const int d = d0 + w;
      const int32_t lb = d < a.ndiag ? cl.lb[d] : kDiaDirect;  // uniform
      if (lb != kDiaDirect) {
        // (inside the cluster's window whenever ok)
        if (ok[w]) t += vtraits<V>::widen(v[w]) * (Acc)xs[lb + (int32_t)(col[w] - r0)];
      } else {
        if (ok[w]) t += vtraits<V>::widen(v[w]) * (Acc)a.x[col[w]];
      }
    }
  }
  if constexpr (TAIL) {
    // HDC: the row's CSR entries (a few at most), in order after the
    // diagonals -- the reference's DIA product followed by its CSR product
    // accumulating onto it
    if (row < a.nrows) {
      const int32_t s0 = a.tro[row], s1 = a.tro[row + 1];
      for (int32_t j = s0; j < s1; j++) t += vtraits<V>::widen(a.tval[j]) * (Acc)a.x[a.tci[j]];
    }
  }
  if (row < a.nrows) a.y[row] = a.init ? (Vec)t : (Vec)((Acc)a.y[row] + t);
}

template <typename V>
struct EllArgs {
  int64_t nrows;
  int64_t ncols;  // set for ell_kernel (its x loads read x[0] for empty slots)
  int32_t loop;  // slots visited per row
  int64_t pitch;
  const int32_t* __restrict__ ci;
  const V* __restrict__ val;
  const typename vtraits<V>::vec* __restrict__ x;
  typename vtraits<V>::vec* __restrict__ y;
  int32_t ld;
  int init;
  // ell_kernel only: per row, 1 + its last slot holding a column (nullptr:
  // every row visits `loop` slots)
  const uint8_t* __restrict__ cnt;
};

template <typename V, int KR, int RPT>
__global__ __launch_bounds__(256) void ell_kernel(EllArgs<V> a) {
  using Acc = typename vtraits<V>::acc;
  using Vec = typename vtraits<V>::vec;
  const uint32_t b = xcd_remap(blockIdx.x, gridDim.x);
  const int64_t row0 = ((int64_t)b * 256 * RPT) + threadIdx.x;
  Acc t[RPT][KR];
#pragma unroll
  for (int u = 0; u < RPT; u++)
#pragma unroll
    for (int q = 0; q < KR; q++) t[u][q] = 0;
  // slots each row visits, and the wave's loop bound (uniform)
  int32_t lim[RPT];
  int32_t wl = a.loop;
  if (a.cnt) {
    int32_t m = 0;
#pragma unroll
    for (int u = 0; u < RPT; u++) {
      const int64_t row = row0 + u * 256;
      lim[u] = row < a.nrows ? (int32_t)a.cnt[row] : 0;
      m = max(m, lim[u]);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = max(m, __shfl_xor(m, o));
    wl = __builtin_amdgcn_readfirstlane(m);
  } else {
#pragma unroll
    for (int u = 0; u < RPT; u++) lim[u] = a.loop;
  }
  // batches of slots: indices first, then values and x entries
  auto batch = [&](auto size, int n0) {
    constexpr int B = decltype(size)::value;
    // index and value loads are unconditional (slots outside the matrix, or
    // beyond the row's count, read slot 0 and are discarded): a load under a
    // branch is waited on where the branch joins, which left one index load
    // in flight at a time
    int32_t ci[RPT][B];
    int64_t slot[RPT][B];
#pragma unroll
    for (int w = 0; w < B; w++)
#pragma unroll
      for (int u = 0; u < RPT; u++) {
        const int64_t row = row0 + u * 256;
        const bool in = n0 + w < lim[u] && row < a.nrows;
        slot[u][w] = in ? row + a.pitch * (n0 + w) : 0;
        ci[u][w] = ld_stream(a.ci + slot[u][w]);
      }
    V v[RPT][B];
#pragma unroll
    for (int w = 0; w < B; w++)
#pragma unroll
      for (int u = 0; u < RPT; u++) v[u][w] = ld_stream(a.val + slot[u][w]);
    // the indices are looked at only now: scheduled among the value loads,
    // their first use held the loads after it back by a round trip (8 slots,
    // 64k rows, FP64 3.39 -> 3.09 us)
    __builtin_amdgcn_sched_barrier(0);
    int64_t c[RPT][B];
#pragma unroll
    for (int w = 0; w < B; w++)
#pragma unroll
      for (int u = 0; u < RPT; u++) {
        const bool in = n0 + w < lim[u] && row0 + u * 256 < a.nrows;
        c[u][w] = in ? (int64_t)ci[u][w] : -1;
      }
#pragma unroll
    for (int u = 0; u < RPT; u++) hold_raw(v[u]);
    // x loads unconditional as well (padding slots read x[0], unused)
    batch_fma<V, KR, RPT>(t, v, c, a.x, a.ld);
  };
  // 8 slots a batch and the rest in one batch of its own size: a batch's loads
  // past the last slot are issued all the same.  Batches of 8 only, then 8
  // and a 4, then 8 / 6 / 4 / 2, then this one, FP64: 5-point 1001^2 18.0,
  // -, 15.8, 14.5 us; band of 9, 4M rows, 117, 104, 98, 95.6 us; 27-point
  // 127^3 158.5, 148.6, 148.8, 147.7 us; 7-point 127^3 42.1, 42.0, 42.0, 40.0 us
  if (a.ncols <= 0) wl = 0;  // (no x entry to read)
  int n0 = 0;
  for (; wl - n0 >= 8; n0 += 8) batch(std::integral_constant<int, 8>{}, n0);
  switch (wl - n0) {
    case 7: batch(std::integral_constant<int, 7>{}, n0); break;
    case 6: batch(std::integral_constant<int, 6>{}, n0); break;
    case 5: batch(std::integral_constant<int, 5>{}, n0); break;
    case 4: batch(std::integral_constant<int, 4>{}, n0); break;
    case 3: batch(std::integral_constant<int, 3>{}, n0); break;
    case 2: batch(std::integral_constant<int, 2>{}, n0); break;
    case 1: batch(std::integral_constant<int, 1>{}, n0); break;
    default: break;
  }
#pragma unroll
  for (int u = 0; u < RPT; u++) {
    const int64_t row = row0 + u * 256;
    if (row < a.nrows) {
#pragma unroll
      for (int q = 0; q < KR; q++) {
        Vec* yp = a.y + row * a.ld + q;
        *yp = a.init ? (Vec)t[u][q] : (Vec)((Acc)*yp + t[u][q]);
      }
    }
  }
}

// ----------------------------------------------------------- SpMM lane groups
// k right-hand sides (row-major X[ncols][ld], Y[nrows][ld]): KL lanes per
// row, each owning 16 bytes of the row's columns (2 FP64 / 4 FP32), so a
// row of x or y moves as KL adjacent 16-byte pieces, and a wave moves 64 / KL
// rows.  DIA's x rows of adjacent rows are adjacent, so a wave's x load
// reads one contiguous 1 KiB span; the y stores are contiguous the same way.
// (One thread per row with k scalar loads instead puts 64 rows 8k bytes
// apart into every load instruction: 64 cache lines per instruction.)  The
// KL lanes of a row load the same value / index (one broadcast line).  Sums
// run over diagonals / slots in the same order as the one-thread kernels.
template <typename Vec>
struct Piece;
template <>
struct Piece<double> {
  using T = double __attribute__((ext_vector_type(2)));
  static constexpr int Q = 2;
};
template <>
struct Piece<float> {
  using T = float __attribute__((ext_vector_type(4)));
  static constexpr int Q = 4;
};

template <typename V, int KL>
__global__ __launch_bounds__(256) void dia_spmm_kernel(DiaArgs<V> a) {
  using Acc = typename vtraits<V>::acc;
  using Vec = typename vtraits<V>::vec;
  using P = Piece<Vec>;
  constexpr int Q = P::Q;
  const uint32_t b = xcd_remap(blockIdx.x, gridDim.x);
  const int64_t row = (int64_t)b * (256 / KL) + threadIdx.x / KL;
  const int l = threadIdx.x % KL;
  // rows past the end stay in the wave (their lanes may hold the batch's
  // offsets read back below) and do no work
  const bool live = row < a.nrows;
  Acc t[Q];
#pragma unroll
  for (int q = 0; q < Q; q++) t[q] = 0;
  for (int d0 = 0; d0 < a.ndiag; d0 += 8) {
    // the batch's eight offsets in one round trip: lane w loads offset
    // d0 + w and the wave reads them back lane by lane (left to the
    // compiler, the BF16 kernel loaded them one at a time, each waited on
    // before the next)
    const int lane = threadIdx.x % kWave;
    const int32_t mo = lane < 8 && d0 + lane < a.ndiag ? a.off[d0 + lane] : 0;
    int32_t o8[8];
#pragma unroll
    for (int w = 0; w < 8; w++) o8[w] = __builtin_amdgcn_readlane(mo, w);
    V v[8];
    int64_t c[8];
#pragma unroll
    for (int w = 0; w < 8; w++) {
      const int d = d0 + w;
      const int64_t o = o8[w];
      const int64_t col = row + o;
      const bool ok = live && d < a.ndiag && col >= 0 && col < a.ncols;
      c[w] = ok ? col : -1;
      v[w] = ok ? ld_stream(a.val + a.pitch * d + row) : V{};
    }
    typename P::T xv[8];
#pragma unroll
    for (int w = 0; w < 8; w++)
      xv[w] = c[w] >= 0 ? *reinterpret_cast<const typename P::T*>(a.x + c[w] * a.ld + l * Q)
                        : (typename P::T)0;
    hold_raw(v);
#pragma unroll
    for (int w = 0; w < 8; w++)
      if (c[w] >= 0) {
        const Acc vw = vtraits<V>::widen(v[w]);
#pragma unroll
        for (int q = 0; q < Q; q++) t[q] += vw * (Acc)xv[w][q];
      }
  }
  if (!live) return;
  typename P::T* yp = reinterpret_cast<typename P::T*>(a.y + row * a.ld + l * Q);
  typename P::T out;
  if (a.init) {
#pragma unroll
    for (int q = 0; q < Q; q++) out[q] = (Vec)t[q];
  } else {
    const typename P::T old = *yp;
#pragma unroll
    for (int q = 0; q < Q; q++) out[q] = (Vec)((Acc)old[q] + t[q]);
  }
  *yp = out;
}

// DIA SpMM with R consecutive rows per lane group (R = 4), in two forms.  For
// each run of diagonals whose offsets step by one (o, o + 1, ..., at most
// kDiaRunMax), a group loads the R + m - 1 X pieces that the run covers once
// and slides over them, instead of one X piece per row and diagonal (the
// 27-point stencil: 6 X loads for 4 rows x 3 diagonals instead of 12).  Each
// row still sums its diagonals in storage order, as dia_spmm_kernel does, with
// the same skips, so all give identical results.  Loads are unconditional
// (columns outside x read a column inside, a row past the matrix its last
// row).  Which form runs where: dia_spmm_form.
constexpr int kDiaRunMax = 3;
constexpr int kDiaSpmmRows = 4;  // R

// The slide form: each lane loads its X pieces itself, the run's values come
// through LDS (loaded by the whole workgroup, so no lane group leaves before
// the end).  Nothing is requested ahead: a run costs two round trips, but many
// workgroups fit a CU, so it wins where the staged form's few would not fill
// the device.
template <typename V, int KL, int R>
__global__ __launch_bounds__(256) void dia_spmm_slide_kernel(DiaArgs<V> a) {
  using Acc = typename vtraits<V>::acc;
  using Vec = typename vtraits<V>::vec;
  using P = Piece<Vec>;
  constexpr int Q = P::Q;
  constexpr int W = R + kDiaRunMax - 1;
  constexpr int kRows = 256 / KL * R;  // rows of the workgroup
  // the run's values for the workgroup's rows, loaded by all its threads in
  // one coalesced pass per diagonal (each lane then reads its R rows'
  // values from here instead of R loads of its own)
  __shared__ V s_val[kDiaRunMax][kRows];
  const uint32_t b = xcd_remap(blockIdx.x, gridDim.x);
  const int64_t wr0 = (int64_t)b * kRows;
  const int gl = threadIdx.x / KL;
  const int64_t row0 = wr0 + (int64_t)gl * R;
  const int l = threadIdx.x % KL;
  const int64_t last = a.nrows - 1;
  Acc t[R][Q];
#pragma unroll
  for (int i = 0; i < R; i++)
#pragma unroll
    for (int q = 0; q < Q; q++) t[i][q] = 0;
  for (int d = 0; d < a.ndiag;) {
    const int64_t o = a.off[d];
    int m = 1;
    while (m < kDiaRunMax && d + m < a.ndiag && (int64_t)a.off[d + m] == o + m) m++;
    // the X rows first: the value stores below wait for every older load
    typename P::T xw[W];
#pragma unroll
    for (int i = 0; i < W; i++) {
      const int64_t col = row0 + o + i;
      const bool in = i < R + m - 1 && col >= 0 && col < a.ncols;
      xw[i] = *reinterpret_cast<const typename P::T*>(a.x + (in ? col : 0) * a.ld + l * Q);
    }
    __syncthreads();  // the previous run's values are read
    for (int j = 0; j < m; j++)
      for (int e = threadIdx.x; e < kRows; e += 256)
        s_val[j][e] = ld_stream(a.val + a.pitch * (d + j) + min(wr0 + e, last));
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kDiaRunMax; j++) {
      if (j < m) {
#pragma unroll
        for (int i = 0; i < R; i++) {
          const int64_t col = row0 + i + o + j;
          const bool ok = row0 + i < a.nrows && col >= 0 && col < a.ncols;
          const Acc vw = vtraits<V>::widen(s_val[j][gl * R + i]);
#pragma unroll
          for (int q = 0; q < Q; q++) {
            const Acc f = t[i][q] + vw * (Acc)xw[i + j][q];
            t[i][q] = ok ? f : t[i][q];
          }
        }
      }
    }
    d += m;
  }
#pragma unroll
  for (int i = 0; i < R; i++) {
    const int64_t row = row0 + i;
    if (row < a.nrows) {
      typename P::T* yp = reinterpret_cast<typename P::T*>(a.y + row * a.ld + l * Q);
      typename P::T out;
      if (a.init) {
#pragma unroll
        for (int q = 0; q < Q; q++) out[q] = (Vec)t[i][q];
      } else {
        const typename P::T old = *yp;
#pragma unroll
        for (int q = 0; q < Q; q++) out[q] = (Vec)((Acc)old[q] + t[i][q]);
      }
      *yp = out;
    }
  }
}

// The staged form: the workgroup loads the X rows of the run too, once and
// coalesced, and hands them over through LDS; each lane reads its R + m - 1 X
// pieces from there.  Products are selected only where a workgroup's columns
// leave x.
//
// What bounds it: the L1.  With every lane loading its own X pieces the L1
// served each X row three times a run and stood still half of the time on
// rows another lane had requested already (TCP_PENDING_STALL_CYCLES); the
// fetched bytes, 2.5 or 1.5 GB depending on the order of the workgroups, made
// no difference.  A workgroup's runs follow one another, so the next run is
// requested before the current one is summed, and the offsets come 64 at a
// time into a register, the runs cut from it with scalar code (read from
// memory, a run's offsets were a chain of round trips).  27-point 160^3,
// FP64: 16 columns 632 -> 531 us (3.6 TB/s of X, Y and values once each; the
// L1's return path is still busy 92% of the time), 8 columns 412 -> 324 us;
// FP32, 16 columns 365 -> 293 us.  VGPRs hold four waves to a SIMD; compiled
// for five it spills (927 us).
template <typename V, int KL, int R>
__global__ __launch_bounds__(256) void dia_spmm_runs_kernel(DiaArgs<V> a) {
  using Acc = typename vtraits<V>::acc;
  using Vec = typename vtraits<V>::vec;
  using P = Piece<Vec>;
  constexpr int Q = P::Q;
  constexpr int W = R + kDiaRunMax - 1;
  constexpr int kRows = 256 / KL * R;  // rows of the workgroup
  constexpr int kXRows = kRows + kDiaRunMax - 1;
  constexpr int kX = (kXRows * KL + 255) / 256;            // X pieces a thread loads
  constexpr int kVals = (kDiaRunMax * kRows + 255) / 256;  // values a thread loads
  // X rows in LDS, one row left free after every R, so that the lane groups
  // of a read lie on different banks
  __shared__ typename P::T s_x[(kXRows + (kXRows - 1) / R) * KL];
  __shared__ V s_val[kDiaRunMax * kRows];
  const int64_t wb = dia_plane_block(a, kRows);
  if (wb < 0) return;  // the whole workgroup
  const int64_t wr0 = wb * kRows;
  const int gl = threadIdx.x / KL;
  const int64_t row0 = wr0 + (int64_t)gl * R;
  const int l = threadIdx.x % KL;
  const int64_t last = a.nrows - 1;
  Acc t[R][Q];
#pragma unroll
  for (int i = 0; i < R; i++)
#pragma unroll
    for (int q = 0; q < Q; q++) t[i][q] = 0;

  // the runs: 64 offsets in a register, bit w of `step` set when offset w
  // continues the one before it
  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const uint32_t x_lane = (uint32_t)((gl * a.ld + l * Q) * (int)sizeof(Vec));
  int32_t offs = 0;
  uint64_t step = 0;
  int d = 0, d0 = -kWave;  // next diagonal, first offset held
  int64_t o = 0;           // the run requested last: first offset, diagonals,
  int m = 0;
  bool inner = false;      // and all its columns inside x, all rows inside
  typename P::T xn[kX];
  V vn[kVals];
  auto request = [&]() {
    if (d - d0 >= kWave) {
      d0 = d;
      offs = a.off[min(d + lane, a.ndiag - 1)];
      const int32_t prev = shfl_up(offs, 1);
      step = __ballot(lane > 0 && d + lane < a.ndiag && (int64_t)prev + 1 == offs);
    }
    const int w = d - d0;
    o = __builtin_amdgcn_readlane(offs, w);
    m = 1;
    while (m < kDiaRunMax && w + m < kWave && ((step >> (w + m)) & 1)) m++;
    inner = wr0 + kRows <= a.nrows && wr0 + o >= 0 && wr0 + kXRows + o <= a.ncols;
    if (inner) {
      // uniform addresses, each lane at a fixed distance
      const char* xb = reinterpret_cast<const char*>(a.x + (wr0 + o) * a.ld);
      const int64_t xstep = (int64_t)(256 / KL) * a.ld * sizeof(Vec);
#pragma unroll
      for (int k = 0; k < kX; k++)
        if (k + 1 < kX || gl + k * (256 / KL) < kXRows)
          xn[k] = *reinterpret_cast<const typename P::T*>(xb + k * xstep + x_lane);
#pragma unroll
      for (int k = 0; k < kVals; k++) {
        const int e = wave * kWave + 256 * k;  // uniform
        const int j = min(e / kRows, m - 1);
        vn[k] = ld_stream(a.val + (a.pitch * (d + j) + wr0 + e % kRows) + lane);
      }
    } else {
#pragma unroll
      for (int k = 0; k < kX; k++) {
        const int64_t col = min(max(wr0 + gl + k * (256 / KL) + o, (int64_t)0), a.ncols - 1);
        xn[k] = *reinterpret_cast<const typename P::T*>(a.x + col * a.ld + l * Q);
      }
#pragma unroll
      for (int k = 0; k < kVals; k++) {
        const int e = threadIdx.x + 256 * k;
        const int j = min(e / kRows, m - 1);
        vn[k] = ld_stream(a.val + a.pitch * (d + j) + min(wr0 + e % kRows, last));
      }
    }
    d += m;
  };

  if (a.ndiag > 0) request();
  while (m > 0) {
    __syncthreads();  // the run before is read
#pragma unroll
    for (int k = 0; k < kX; k++) {
      const int r = gl + k * (256 / KL);
      if (k + 1 < kX || r < kXRows) s_x[(r + r / R) * KL + l] = xn[k];
    }
#pragma unroll
    for (int k = 0; k < kVals; k++) {
      const int e = threadIdx.x + 256 * k;
      if (kVals * 256 == kDiaRunMax * kRows || e < kDiaRunMax * kRows) s_val[e] = vn[k];
    }
    __syncthreads();
    const int64_t co = o;
    const int cm = m;
    const bool cin = inner;
    m = 0;
    if (d < a.ndiag) request();
    typename P::T xw[W];
#pragma unroll
    for (int i = 0; i < W; i++) xw[i] = s_x[(gl * (R + 1) + i + i / R) * KL + l];
#pragma unroll
    for (int j = 0; j < kDiaRunMax; j++) {
      if (j < cm) {
#pragma unroll
        for (int i = 0; i < R; i++) {
          const Acc vw = vtraits<V>::widen(s_val[j * kRows + gl * R + i]);
          if (cin) {
#pragma unroll
            for (int q = 0; q < Q; q++) t[i][q] += vw * (Acc)xw[i + j][q];
          } else {
            const int64_t col = row0 + i + co + j;
            const bool ok = row0 + i < a.nrows && col >= 0 && col < a.ncols;
#pragma unroll
            for (int q = 0; q < Q; q++) {
              const Acc f = t[i][q] + vw * (Acc)xw[i + j][q];
              t[i][q] = ok ? f : t[i][q];
            }
          }
        }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < R; i++) {
    const int64_t row = row0 + i;
    if (row < a.nrows) {
      typename P::T* yp = reinterpret_cast<typename P::T*>(a.y + row * a.ld + l * Q);
      typename P::T out;
      if (a.init) {
#pragma unroll
        for (int q = 0; q < Q; q++) out[q] = (Vec)t[i][q];
      } else {
        const typename P::T old = *yp;
#pragma unroll
        for (int q = 0; q < Q; q++) out[q] = (Vec)((Acc)old[q] + t[i][q]);
      }
      *yp = out;
    }
  }
}

template <typename V, int KL>
__global__ __launch_bounds__(256) void ell_spmm_kernel(EllArgs<V> a) {
  using Acc = typename vtraits<V>::acc;
  using Vec = typename vtraits<V>::vec;
  using P = Piece<Vec>;
  constexpr int Q = P::Q;
  const uint32_t b = xcd_remap(blockIdx.x, gridDim.x);
  const int64_t row = (int64_t)b * (256 / KL) + threadIdx.x / KL;
  const int l = threadIdx.x % KL;
  if (row >= a.nrows) return;
  Acc t[Q];
#pragma unroll
  for (int q = 0; q < Q; q++) t[q] = 0;
  for (int n0 = 0; n0 < a.loop; n0 += 8) {
    int64_t c[8];
#pragma unroll
    for (int w = 0; w < 8; w++)
      c[w] = n0 + w < a.loop ? (int64_t)ld_stream(a.ci + row + a.pitch * (n0 + w)) : -1;
    V v[8];
#pragma unroll
    for (int w = 0; w < 8; w++)
      v[w] = c[w] >= 0 ? ld_stream(a.val + row + a.pitch * (n0 + w)) : V{};
    typename P::T xv[8];
#pragma unroll
    for (int w = 0; w < 8; w++)
      xv[w] = c[w] >= 0 ? *reinterpret_cast<const typename P::T*>(a.x + c[w] * a.ld + l * Q)
                        : (typename P::T)0;
    hold_raw(v);
#pragma unroll
    for (int w = 0; w < 8; w++)
      if (c[w] >= 0) {
        const Acc vw = vtraits<V>::widen(v[w]);
#pragma unroll
        for (int q = 0; q < Q; q++) t[q] += vw * (Acc)xv[w][q];
      }
  }
  typename P::T* yp = reinterpret_cast<typename P::T*>(a.y + row * a.ld + l * Q);
  typename P::T out;
  if (a.init) {
#pragma unroll
    for (int q = 0; q < Q; q++) out[q] = (Vec)t[q];
  } else {
    const typename P::T old = *yp;
#pragma unroll
    for (int q = 0; q < Q; q++) out[q] = (Vec)((Acc)old[q] + t[q]);
  }
  *yp = out;
}

// ----------------------------------------------------------- row pairs
// FP32 / BF16 DIA SpMV: a thread takes the adjacent rows 2t and 2t + 1, so
// that one load moves the two rows' values of a diagonal (8 B in FP32, 4 B in
// BF16).  With one row per thread a 16-bit value stream moved 128 B per wave
// load, and BF16 ran slower than FP32.  Used when the pitch is even (a pair
// never straddles two diagonals; an odd row count then leaves the pair's
// second element inside the pitch) and the values are aligned to the pair.
template <typename V>
__global__ __launch_bounds__(256) void dia_pair_kernel(DiaArgs<V> a) {
  using P = Pair<V>;
  const uint32_t b = xcd_remap(blockIdx.x, gridDim.x);
  const int64_t row = ((int64_t)b * 256 + threadIdx.x) * 2;
  const typename P::T* pv = reinterpret_cast<const typename P::T*>(a.val);
  float t0 = 0, t1 = 0;
  for (int d0 = 0; d0 < a.ndiag; d0 += 8) {
    float v0[8], v1[8];
    int64_t c0[8], c1[8];
#pragma unroll
    for (int w = 0; w < 8; w++) {
      const int d = d0 + w;
      const bool in = d < a.ndiag && row < a.nrows;
      const int64_t o = d < a.ndiag ? (int64_t)a.off[d] : 0;
      const typename P::T pw = in ? ld_stream(pv + (a.pitch * d + row) / 2) : (typename P::T)0;
      P::split(pw, v0[w], v1[w]);
      const int64_t col0 = row + o, col1 = row + 1 + o;
      c0[w] = in && col0 >= 0 && col0 < a.ncols ? col0 : -1;
      c1[w] = in && row + 1 < a.nrows && col1 >= 0 && col1 < a.ncols ? col1 : -1;
    }
#pragma unroll
    for (int w = 0; w < 8; w++) {
      if (c0[w] >= 0) t0 += v0[w] * a.x[c0[w]];
      if (c1[w] >= 0) t1 += v1[w] * a.x[c1[w]];
    }
  }
  if (row < a.nrows) a.y[row] = a.init ? t0 : a.y[row] + t0;
  if (row + 1 < a.nrows) a.y[row + 1] = a.init ? t1 : a.y[row + 1] + t1;
}

// dia_pair_kernel with x staged in LDS per cluster of nearby diagonals (as
// dia_staged_kernel, over the workgroup's 512 rows); same sums in the same
// order as dia_pair_kernel.
template <typename V>
__global__ __launch_bounds__(256) void dia_pair_staged_kernel(DiaArgs<V> a, DiaStage cl) {
  using P = Pair<V>;
  __shared__ float xs[2 * kDiaStageMax];
  const int64_t r0 = (int64_t)xcd_remap(blockIdx.x, gridDim.x) * 512;
  const int64_t row = r0 + 2 * threadIdx.x;
  for (int c = 0; c < cl.n; c++) {
    const int32_t base = cl.base[c] + 256 * c, len = cl.len[c] + 256;
    for (int j = threadIdx.x; j < len; j += 256) {
      const int64_t col = r0 + cl.omin[c] + j;
      xs[base + j] = (col >= 0 && col < a.ncols) ? a.x[col] : 0.0f;
    }
  }
  __syncthreads();
  const typename P::T* pv = reinterpret_cast<const typename P::T*>(a.val);
  float t0 = 0, t1 = 0;
  for (int d0 = 0; d0 < a.ndiag; d0 += 8) {
    float v0[8], v1[8];
    int64_t c0[8], c1[8];
#pragma unroll
    for (int w = 0; w < 8; w++) {
      const int d = d0 + w;
      const bool in = d < a.ndiag && row < a.nrows;
      const int64_t o = d < a.ndiag ? (int64_t)a.off[d] : 0;
      const typename P::T pw = in ? ld_stream(pv + (a.pitch * d + row) / 2) : (typename P::T)0;
      P::split(pw, v0[w], v1[w]);
      const int64_t col0 = row + o, col1 = row + 1 + o;
      c0[w] = in && col0 >= 0 && col0 < a.ncols ? col0 : -1;
      c1[w] = in && row + 1 < a.nrows && col1 >= 0 && col1 < a.ncols ? col1 : -1;
    }
#pragma unroll
    for (int w = 0; w < 8; w++) {
      const int d = d0 + w;
      const int32_t lb = d < a.ndiag ? cl.lb2[d] : kDiaDirect;  // uniform
      if (lb != kDiaDirect) {
        // (inside the cluster's window whenever the column is)
        if (c0[w] >= 0) t0 += v0[w] * xs[lb + (int32_t)(c0[w] - r0)];
        if (c1[w] >= 0) t1 += v1[w] * xs[lb + (int32_t)(c1[w] - r0)];
      } else {
        if (c0[w] >= 0) t0 += v0[w] * a.x[c0[w]];
        if (c1[w] >= 0) t1 += v1[w] * a.x[c1[w]];
      }
    }
  }
  if (row < a.nrows) a.y[row] = a.init ? t0 : a.y[row] + t0;
  if (row + 1 < a.nrows) a.y[row + 1] = a.init ? t1 : a.y[row + 1] + t1;
}

// ELL: the pair's two column indices are one load too (8 B).  Which sizes it
// takes: ell_pair_ok.
template <typename V>
__global__ __launch_bounds__(256) void ell_pair_kernel(EllArgs<V> a) {
  using P = Pair<V>;
  const uint32_t b = xcd_remap(blockIdx.x, gridDim.x);
  const int64_t row = ((int64_t)b * 256 + threadIdx.x) * 2;
  const typename P::T* pv = reinterpret_cast<const typename P::T*>(a.val);
  const uint64_t* pc = reinterpret_cast<const uint64_t*>(a.ci);
  float t0 = 0, t1 = 0;
  const bool in = row < a.nrows;
  for (int n0 = 0; n0 < a.loop; n0 += 8) {
    int32_t c0[8], c1[8];
#pragma unroll
    for (int w = 0; w < 8; w++) {
      const int n = n0 + w;
      const uint64_t cw = in && n < a.loop ? ld_stream(pc + (a.pitch * n + row) / 2) : ~0ull;
      c0[w] = (int32_t)(uint32_t)cw;
      // the pair's second row may lie past nrows, inside the pitch
      c1[w] = row + 1 < a.nrows ? (int32_t)(uint32_t)(cw >> 32) : -1;
    }
    float v0[8], v1[8];
#pragma unroll
    for (int w = 0; w < 8; w++) {
      const int n = n0 + w;
      const typename P::T pw =
          (c0[w] >= 0 || c1[w] >= 0) ? ld_stream(pv + (a.pitch * n + row) / 2) : (typename P::T)0;
      P::split(pw, v0[w], v1[w]);
    }
#pragma unroll
    for (int w = 0; w < 8; w++) {
      if (c0[w] >= 0) t0 += v0[w] * a.x[c0[w]];
      if (c1[w] >= 0) t1 += v1[w] * a.x[c1[w]];
    }
  }
  if (row < a.nrows) a.y[row] = a.init ? t0 : a.y[row] + t0;
  if (row + 1 < a.nrows) a.y[row + 1] = a.init ? t1 : a.y[row + 1] + t1;
}

// The same for a stage of at most kStageAhead entries a thread (a band, two
// planes of a small grid): the first batch's value pairs are requested before
// the stage is stored, raw until their products, 12 diagonals a batch.  A
// workgroup's rows were three round trips one after another (x, eight
// diagonals, the rest); 4M rows, 9 diagonals: FP32 40.9 -> 34.3 us, BF16 37.8
// -> 30.8 us (3.4 TB/s); a wide stage gains nothing (27-point 160^3 FP32 103
// -> 108 us, BF16 88 -> 99 us) and keeps the kernel above.
template <typename V>
__global__ __launch_bounds__(256) void dia_pair_ahead_kernel(DiaArgs<V> a, DiaStage cl) {
  using P = Pair<V>;
  constexpr int U = 12;  // diagonals a batch, their pairs raw until the products
  __shared__ float xs[256 * kStageAhead];
  const int64_t r0 = (int64_t)xcd_remap(blockIdx.x, gridDim.x) * 512;
  const int64_t row = r0 + 2 * threadIdx.x;
  float xr[kStageAhead];
  stage_load<float, kStageAhead, 256>(cl, a.x, a.ncols, r0, 0, xr);
  const typename P::T* pv = reinterpret_cast<const typename P::T*>(a.val);
  float t0 = 0, t1 = 0;
  for (int d0 = 0; d0 < a.ndiag; d0 += U) {
    typename P::T pw[U];
#pragma unroll
    for (int w = 0; w < U; w++) {
      const int d = min(d0 + w, a.ndiag - 1);
      pw[w] = ld_stream(pv + (a.pitch * d + min(row, a.pitch - 2)) / 2);
    }
    if (d0 == 0) {
      stage_store<float, kStageAhead, 256>(cl, xs, 0, xr);
      __syncthreads();
    }
#pragma unroll
    for (int w = 0; w < U; w++) {
      const int d = d0 + w;
      if (d >= a.ndiag) break;
      const int64_t o = a.off[d];
      const int32_t lb = cl.lb2[d];  // uniform
      float v0, v1;
      P::split(pw[w], v0, v1);
      const int64_t c0 = row + o, c1 = row + 1 + o;
      const bool in0 = row < a.nrows && c0 >= 0 && c0 < a.ncols;
      const bool in1 = row + 1 < a.nrows && c1 >= 0 && c1 < a.ncols;
      if (lb != kDiaDirect) {
        // (inside the cluster's window whenever the column is)
        if (in0) t0 += v0 * xs[lb + (int32_t)(c0 - r0)];
        if (in1) t1 += v1 * xs[lb + (int32_t)(c1 - r0)];
      } else {
        if (in0) t0 += v0 * a.x[c0];
        if (in1) t1 += v1 * a.x[c1];
      }
    }
  }
  if (row < a.nrows) a.y[row] = a.init ? t0 : a.y[row] + t0;
  if (row + 1 < a.nrows) a.y[row + 1] = a.init ? t1 : a.y[row + 1] + t1;
}

// FP32 / BF16 rows of more than kCompensateLen diagonals / slots: thread
// (row, column q) sums its row as Dot2 pairs (TwoSum on the additions, the
// FMA TwoProduct on the products) and adds the old y through TwoSum when
// accumulating.  Diagonals / slots in storage order, as the other kernels.
template <typename V, bool DIA>
__global__ __launch_bounds__(256) void dia_ell_comp_kernel(DiaArgs<V> d, EllArgs<V> e, int32_t k) {
  using Acc = typename vtraits<V>::acc;
  using Vec = typename vtraits<V>::vec;
  const int64_t nrows = DIA ? d.nrows : e.nrows;
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nrows * k) return;
  const int64_t row = t / k, q = t % k;
  csum<Acc> cs{0, 0};
  if constexpr (DIA) {
    for (int32_t n = 0; n < d.ndiag; n++) {
      const int64_t col = row + d.off[n];
      if (col >= 0 && col < d.ncols)
        cs.add_prod(vtraits<V>::widen(ld_stream(d.val + d.pitch * n + row)),
                    (Acc)d.x[col * d.ld + q]);
    }
  } else {
    for (int32_t n = 0; n < e.loop; n++) {
      const int64_t slot = row + e.pitch * n;
      const int32_t c = ld_stream(e.ci + slot);
      if (c >= 0) cs.add_prod(vtraits<V>::widen(ld_stream(e.val + slot)), (Acc)e.x[(int64_t)c * e.ld + q]);
    }
  }
  Vec* yp = (DIA ? d.y : e.y) + row * (DIA ? d.ld : e.ld) + q;
  if (!(DIA ? d.init : e.init)) cs.combine((Acc)*yp, (Acc)0);
  *yp = (Vec)cs.value();
}

namespace {

template <typename V, bool DIA>
int launch_comp(mph_matrix_impl* A, int k, const void* x, void* y, int init, hipStream_t s) {
  DiaArgs<V> d{};
  EllArgs<V> e{};
  if constexpr (DIA) {
    d.nrows = A->nrows;
    d.ncols = A->ncols;
    d.ndiag = (int32_t)A->ndiag;
    d.pitch = A->dia_pitch;
    d.off = A->dia_off;
    d.val = static_cast<const V*>(A->dia_v);
    d.x = static_cast<const typename vtraits<V>::vec*>(x);
    d.y = static_cast<typename vtraits<V>::vec*>(y);
    d.ld = k;
    d.init = init;
  } else {
    e.nrows = A->nrows;
    e.ncols = A->ncols;
    e.loop = (int32_t)A->ell_loop;
    e.pitch = A->ell_pitch;
    e.ci = A->ell_ci;
    e.val = static_cast<const V*>(A->ell_v);
    e.x = static_cast<const typename vtraits<V>::vec*>(x);
    e.y = static_cast<typename vtraits<V>::vec*>(y);
    e.ld = k;
    e.init = init;
  }
  const int64_t n = A->nrows * (int64_t)k;
  if (n == 0) return MPH_OK;
  hipLaunchKernelGGL((dia_ell_comp_kernel<V, DIA>), dim3((unsigned)ceil_div(n, 256)), dim3(256), 0,
                     s, d, e, (int32_t)k);
  MPH_HIP_CHECK(hipGetLastError());
  return MPH_OK;
}

template <typename V, int KR, int RPT>
int launch_dia_k(mph_matrix_impl* A, const void* x, void* y, int ld, int init,
                 hipStream_t s) {
  DiaArgs<V> a{};
  a.nrows = A->nrows;
  a.ncols = A->ncols;
  a.ndiag = (int32_t)A->ndiag;
  a.pitch = A->dia_pitch;
  a.off = A->dia_off;
  a.val = static_cast<const V*>(A->dia_v);
  a.x = static_cast<const typename vtraits<V>::vec*>(x);
  a.y = static_cast<typename vtraits<V>::vec*>(y);
  a.ld = ld;
  a.init = init;
  const int64_t nb = ceil_div(A->nrows, 256 * RPT);
  if (nb == 0) return MPH_OK;
  hipLaunchKernelGGL((dia_kernel<V, KR, RPT>), dim3((unsigned)nb), dim3(256), 0,
                     s, a);
  MPH_HIP_CHECK(hipGetLastError());
  return MPH_OK;
}

template <typename V>
int launch_dia_staged(mph_matrix_impl* A, const void* x, void* y, int init, hipStream_t s) {
  DiaArgs<V> a{};
  a.nrows = A->nrows;
  a.ncols = A->ncols;
  a.ndiag = (int32_t)A->ndiag;
  a.pitch = A->dia_pitch;
  a.off = A->dia_off;
  a.val = static_cast<const V*>(A->dia_v);
  a.x = static_cast<const typename vtraits<V>::vec*>(x);
  a.y = static_cast<typename vtraits<V>::vec*>(y);
  a.ld = 1;
  a.init = init;
  const int64_t nb = ceil_div(A->nrows, 256);
  if (nb == 0) return MPH_OK;
  hipLaunchKernelGGL(dia_staged_kernel<V>, dim3((unsigned)nb), dim3(256), 0, s, a, A->dia_stage);
  MPH_HIP_CHECK(hipGetLastError());
  return MPH_OK;
}

template <typename V, int KR, int RPT>
int launch_ell_k(mph_matrix_impl* A, const void* x, void* y, int ld, int init,
                 hipStream_t s) {
  EllArgs<V> a{};
  a.nrows = A->nrows;
  a.ncols = A->ncols;
  a.loop = (int32_t)A->ell_loop;
  a.pitch = A->ell_pitch;
  a.ci = A->ell_ci;
  a.val = static_cast<const V*>(A->ell_v);
  a.x = static_cast<const typename vtraits<V>::vec*>(x);
  a.y = static_cast<typename vtraits<V>::vec*>(y);
  a.ld = ld;
  a.init = init;
  a.cnt = A->rb.ell_cnt;
  const int64_t nb = ceil_div(A->nrows, 256 * RPT);
  if (nb == 0) return MPH_OK;
  hipLaunchKernelGGL((ell_kernel<V, KR, RPT>), dim3((unsigned)nb), dim3(256), 0,
                     s, a);
  MPH_HIP_CHECK(hipGetLastError());
  return MPH_OK;
}

// Which kernel takes a DIA SpMM pass of `lanes` lanes a row: one row per lane
// group (dia_spmm_kernel), or kDiaSpmmRows in the slide or the staged form.
// The lines lie where the three were measured: FP64 k = 4, 8, 16, FP32 / BF16
// k = 8, 16, 32, bands of 3 to 25 diagonals of 10k to 2M rows, 5-, 7- and
// 27-point grids of 30 to 1000 a side; no point is more than 3% slower than
// the slide form from 4 lanes and the one-row kernel below, which ran there
// before the staged form.  `full`: workgroups of the forms (1024 / lanes
// rows) a CU.
//  * 2 lanes: the staged form on runs of nearly three diagonals once it fills
//    the device (27-point 128^3 FP64 157 -> 117 us, FP32 107 -> 86; below,
//    9-diagonal band of 131k rows FP64 6.4 -> 7.1), BF16 four times as late
//    (27-point 100^3 43.1 -> 45.0, 128^3 85.5 -> 79.2); shorter runs lose
//    (5-point 1000^2 FP64 21.0 -> 24.8).
//  * The staged form requests a run ahead, and four of its workgroups fit a
//    CU: it wins from 3 a CU in FP64 (slide against staged: 27-point 160^3
//    k = 16 632 -> 531 us; 500k rows, 9 diagonals, k = 8 28.0 -> 21.3) or 2
//    with 9 diagonals or more (131k rows, k = 8 9.8 -> 8.0), and in FP32 where
//    its last round is full (9 diagonals, k = 32, 1024 workgroups 12.2 -> 10.4;
//    1563: 17.2 -> 17.8; 3907: 37.6 -> 34.8), with 16 lanes later (27-point
//    64^3 k = 64 71.6 -> 75.6).  One or two runs and a second round barely
//    begun lose in FP64 too (1563, 3 diagonals, k = 16 10.7 -> 12.2).  BF16
//    moves half the values for the same X: the staged form gains once X leaves
//    the last cache (27-point 128^3 k = 16 186 -> 158 us; 100^3 67.2 -> 73.3),
//    or, where the diagonals reach no farther than a workgroup's rows, from
//    10.5 a CU (420k rows, 9 diagonals, k = 32 28.1 -> 26.0) and in one full
//    round (131k rows, 17 diagonals, k = 32 16.1 -> 15.2).
//  * The slide form beats the one-row kernel where its workgroups fill the
//    device (300k rows, 9 diagonals, BF16 k = 16 15.4 -> 12.3), with fewer
//    only where the one-row kernel's batches of 8 diagonals run part empty
//    (131k rows FP32 k = 16: 3 diagonals 5.7 -> 4.7 us, 9 8.4 -> 7.2, 7 6.0 ->
//    6.6), and loses on runs of mostly one diagonal (7-point 64^3 BF16 k = 16
//    9.5 -> 11.3).
// MPH_DIA_SPMM_RUNS=0 / 1 / 2 forces the one-row kernel / the staged form /
// the slide form.
enum class DiaSpmm { kRow, kSlide, kStage };

DiaSpmm dia_spmm_form(const mph_matrix_impl* A, int lanes) {
  if (A->ncols == 0) return DiaSpmm::kRow;
  if (const char* env = std::getenv("MPH_DIA_SPMM_RUNS")) {
    const int mode = std::atoi(env);
    return mode <= 0 ? DiaSpmm::kRow : mode == 1 ? DiaSpmm::kStage : DiaSpmm::kSlide;
  }
  const int64_t nd = A->ndiag, runs = A->dia_runs, rows = 256 / lanes * kDiaSpmmRows;
  if (lanes < 2) return DiaSpmm::kRow;
  const double full = (double)ceil_div(A->nrows, rows) / device_cu_count();
  const bool f64 = A->vt == MPH_F64, f32 = A->vt == MPH_F32;
  // one diagonal, or more than kDiaStageMaxDiags: the analysis does not look
  // at the runs (its copy of the offsets would cost it 19 us)
  if (runs == 0)
    return lanes < 4 || full < 3 ? DiaSpmm::kRow : f64 ? DiaSpmm::kStage : DiaSpmm::kSlide;
  // one or two runs, and a second round of workgroups barely begun
  const bool brief = runs <= 2 && full > 5 && full < 6.4;
  if (lanes == 2)
    return 10 * nd >= 27 * runs && full >= (f64 ? 2 : f32 ? 3.5 : 15) && !brief ? DiaSpmm::kStage
                                                                               : DiaSpmm::kRow;
  const bool singles = 2 * nd < 3 * runs;  // runs of mostly one diagonal
  const bool near = A->dia_reach <= rows;
  const bool one_round = full >= 3.5 && full <= 4;
  bool stage;
  if (f64)
    stage = (full >= 3 || (full >= 1.9 && nd >= 9 && !singles)) && !brief;
  else if (f32)
    stage = one_round || (full >= 3 && full <= 4 && nd >= 9) ||
            full >= (lanes < 16 ? 6.4 : near ? 10 : 24);
  else
    stage = !singles && (near ? one_round || full >= 10.5 : full >= 24);
  if (stage) return DiaSpmm::kStage;
  if (singles && full < 24) return DiaSpmm::kRow;
  const double used = (double)nd / (double)(8 * ceil_div(nd, 8));  // of the one-row kernel's batches
  const bool slide = full >= 3 || (full >= 1.9 && used <= 0.71) || (full >= 1 && used <= (f64 ? 0.6 : 0.4));
  return slide ? DiaSpmm::kSlide : DiaSpmm::kRow;
}

template <typename V, bool DIA, int KL>
int launch_spmm_lanes(mph_matrix_impl* A, const void* x, void* y, int ld, int init,
                      hipStream_t s) {
  const int64_t nb = ceil_div(A->nrows, 256 / KL);
  if (nb == 0) return MPH_OK;
  if constexpr (DIA) {
    DiaArgs<V> a{};
    a.nrows = A->nrows;
    a.ncols = A->ncols;
    a.ndiag = (int32_t)A->ndiag;
    a.pitch = A->dia_pitch;
    a.off = A->dia_off;
    a.val = static_cast<const V*>(A->dia_v);
    a.x = static_cast<const typename vtraits<V>::vec*>(x);
    a.y = static_cast<typename vtraits<V>::vec*>(y);
    a.ld = ld;
    a.init = init;
    const DiaSpmm form = dia_spmm_form(A, KL);
    constexpr int R = kDiaSpmmRows;
    if (form == DiaSpmm::kStage) {
      // plane order where two reaches of X exceed half an XCD's L2 and a
      // plane has workgroups to share out (27-point 160^3 FP64 k = 16 551 ->
      // 537 us, k = 32 1000 -> 950 us, FP32 k = 16 even)
      constexpr int64_t rows = 256 / KL * R;
      const int64_t nbr = ceil_div(A->nrows, rows), plane = (A->dia_reach + rows / 2) / rows;
      int64_t grid = nbr;
      if (2 * A->dia_reach * ld * (int64_t)sizeof(*a.x) > (2 << 20) && plane >= 4 * kNumXcd &&
          plane < nbr) {
        a.plane = (int32_t)plane;
        a.plane_xcd = (int32_t)ceil_div(plane, kNumXcd);
        grid = kNumXcd * a.plane_xcd * ceil_div(nbr, plane);
      }
      hipLaunchKernelGGL((dia_spmm_runs_kernel<V, KL, R>), dim3((unsigned)grid), dim3(256), 0, s, a);
    } else if (form == DiaSpmm::kSlide) {
      hipLaunchKernelGGL((dia_spmm_slide_kernel<V, KL, R>),
                         dim3((unsigned)ceil_div(A->nrows, (int64_t)(256 / KL) * R)), dim3(256), 0, s,
                         a);
    } else {
      hipLaunchKernelGGL((dia_spmm_kernel<V, KL>), dim3((unsigned)nb), dim3(256), 0, s, a);
    }
  } else {
    EllArgs<V> a{};
    a.nrows = A->nrows;
    a.loop = (int32_t)A->ell_loop;
    a.pitch = A->ell_pitch;
    a.ci = A->ell_ci;
    a.val = static_cast<const V*>(A->ell_v);
    a.x = static_cast<const typename vtraits<V>::vec*>(x);
    a.y = static_cast<typename vtraits<V>::vec*>(y);
    a.ld = ld;
    a.init = init;
    hipLaunchKernelGGL((ell_spmm_kernel<V, KL>), dim3((unsigned)nb), dim3(256), 0, s, a);
  }
  MPH_HIP_CHECK(hipGetLastError());
  return MPH_OK;
}

template <typename V, bool DIA, int RPT>
int launch_fmt(mph_matrix_impl* A, int k, const void* x, void* y, int init,
               hipStream_t s) {
  using Vec = typename vtraits<V>::vec;
  constexpr int Q = Piece<Vec>::Q;
  // lane groups when every row of X / Y starts on 16 bytes
  const bool pieces = k > 1 && (k * sizeof(Vec)) % 16 == 0 &&
                      reinterpret_cast<uintptr_t>(x) % 16 == 0 &&
                      reinterpret_cast<uintptr_t>(y) % 16 == 0;
  int done = 0;
  while (done < k) {
    const int rem = k - done;
    const Vec* xs = static_cast<const Vec*>(x) + done;
    Vec* ys = static_cast<Vec*>(y) + done;
    if (pieces && rem >= Q) {
      const int kl = rem >= 16 * Q ? 16 : rem >= 8 * Q ? 8 : rem >= 4 * Q ? 4 : rem >= 2 * Q ? 2 : 1;
      // (5 to 7 columns that lane groups would split into passes take one)
      if (RPT > 1 || rem >= 8 || kl * Q == rem) {
        int st;
        switch (kl) {
          case 16: st = launch_spmm_lanes<V, DIA, 16>(A, xs, ys, k, init, s); break;
          case 8: st = launch_spmm_lanes<V, DIA, 8>(A, xs, ys, k, init, s); break;
          case 4: st = launch_spmm_lanes<V, DIA, 4>(A, xs, ys, k, init, s); break;
          case 2: st = launch_spmm_lanes<V, DIA, 2>(A, xs, ys, k, init, s); break;
          default: st = launch_spmm_lanes<V, DIA, 1>(A, xs, ys, k, init, s); break;
        }
        if (st != MPH_OK) return st;
        done += kl * Q;
        continue;
      }
    }
    // what is left below 8 columns in one pass over the matrix
    int kr = rem >= 16 ? 16 : rem >= 8 ? 8 : rem;
    if (RPT > 1 && kr < 8) kr = rem >= 4 ? 4 : rem >= 2 ? 2 : 1;
    int st;
#define MPH_LAUNCH(KRV)                                             \
  st = DIA ? launch_dia_k<V, KRV, RPT>(A, xs, ys, k, init, s)       \
           : launch_ell_k<V, KRV, RPT>(A, xs, ys, k, init, s)
    switch (kr) {
      case 16: MPH_LAUNCH(16); break;
      case 8: MPH_LAUNCH(8); break;
      case 4: MPH_LAUNCH(4); break;
      case 2: MPH_LAUNCH(2); break;
      case 1: MPH_LAUNCH(1); break;
      default:
        st = MPH_OK;
        if constexpr (RPT == 1) {
          switch (kr) {
            case 7: MPH_LAUNCH(7); break;
            case 6: MPH_LAUNCH(6); break;
            case 5: MPH_LAUNCH(5); break;
            default: MPH_LAUNCH(3); break;
          }
        }
    }
#undef MPH_LAUNCH
    if (st != MPH_OK) return st;
    done += kr;
  }
  return MPH_OK;
}

// the DIA row-pair kernels: FP32 / BF16 SpMV with the default launch shape, an
// even pitch and values aligned to the pair loads
template <typename V>
int launch_dia_pair(mph_matrix_impl* A, const void* x, void* y, int init, hipStream_t s) {
  const int64_t nb = ceil_div(A->nrows, 512);
  if (nb == 0) return MPH_OK;
  DiaArgs<V> a{};
  a.nrows = A->nrows;
  a.ncols = A->ncols;
  a.ndiag = (int32_t)A->ndiag;
  a.pitch = A->dia_pitch;
  a.off = A->dia_off;
  a.val = static_cast<const V*>(A->dia_v);
  a.x = static_cast<const float*>(x);
  a.y = static_cast<float*>(y);
  a.ld = 1;
  a.init = init;
  const DiaStage& cl = A->dia_stage;
  // the kernel that requests ahead takes 12 diagonals a batch, the other 8,
  // and both load a batch past its last diagonal all the same: the first where
  // it pads no more, up to 20 diagonals (4M rows FP32: 9 diagonals 39.1 ->
  // 32.8 us, 17 61.2 -> 59.1; 13 46.0 -> 49.8, 15 51.0 -> 54.5, BF16 23
  // 57.5 -> 59.7, 31 73.2 -> 79.1)
  const int64_t nd = A->ndiag;
  const bool ahead = nd <= 20 && 12 * ceil_div(nd, 12) <= 8 * ceil_div(nd, 8) && cl.n > 0 &&
                     cl.base[cl.n - 1] + cl.len[cl.n - 1] + 256 * cl.n <= 256 * kStageAhead;
  if (cl.n > 0 && cl.pair && ahead)
    hipLaunchKernelGGL(dia_pair_ahead_kernel<V>, dim3((unsigned)nb), dim3(256), 0, s, a, cl);
  else if (cl.n > 0 && cl.pair)
    hipLaunchKernelGGL(dia_pair_staged_kernel<V>, dim3((unsigned)nb), dim3(256), 0, s, a, cl);
  else
    hipLaunchKernelGGL(dia_pair_kernel<V>, dim3((unsigned)nb), dim3(256), 0, s, a);
  MPH_HIP_CHECK(hipGetLastError());
  return MPH_OK;
}

template <typename V>
int launch_ell_pair(mph_matrix_impl* A, const void* x, void* y, int init, hipStream_t s) {
  EllArgs<V> a{};
  a.nrows = A->nrows;
  a.loop = (int32_t)A->ell_loop;
  a.pitch = A->ell_pitch;
  a.ci = A->ell_ci;
  a.val = static_cast<const V*>(A->ell_v);
  a.x = static_cast<const float*>(x);
  a.y = static_cast<float*>(y);
  a.ld = 1;
  a.init = init;
  hipLaunchKernelGGL(ell_pair_kernel<V>, dim3((unsigned)ceil_div(A->nrows, 512)), dim3(256), 0, s,
                     a);
  MPH_HIP_CHECK(hipGetLastError());
  return MPH_OK;
}

bool pair_ok(const mph_matrix_impl* A, int k, int64_t pitch, const void* v) {
  return k == 1 && A->tuning.rows_per_thread == 0 && (A->vt == MPH_F32 || A->vt == MPH_BF16) &&
         pitch % 2 == 0 && reinterpret_cast<uintptr_t>(v) % (2 * value_size(A->vt)) == 0;
}

bool dia_pair_ok(const mph_matrix_impl* A, int k) { return pair_ok(A, k, A->dia_pitch, A->dia_v); }

// ELL takes row pairs where the one-row kernel's workgroups, 8 a CU at once,
// do not fit and have little to do: up to 3 slots (FP32, 1M rows: 2 slots one
// row 5.5 us, pairs 4.7; 3 slots 6.8, 6.0; 3M 19.0, 18.6; even at 500k), up to
// 5 while the second round of them is short (850k rows: 4 slots 7.2, 6.4; 1.5M
// 10.9, 12.9).  Elsewhere one row per thread wins: its loads are not under
// branches (27-point 128^3 FP32 pairs 96-98 us, one row 76.7; pairs without
// branches 102).
bool ell_pair_ok(const mph_matrix_impl* A, int k) {
  const int64_t wgs = ceil_div(A->nrows, 256), cus = device_cu_count();
  return pair_ok(A, k, A->ell_pitch, A->ell_v) && !A->rb.ell_cnt &&
         reinterpret_cast<uintptr_t>(A->ell_ci) % 8 == 0 && wgs > 8 * cus &&
         (A->ell_loop <= 3 || (A->ell_loop <= 5 && wgs <= 14 * cus));
}

template <bool DIA>
int dispatch(mph_matrix_impl* A, int k, const void* x, void* y, int init,
             hipStream_t s) {
  if (A->vt != MPH_F64 && (DIA ? A->ndiag : A->ell_loop) > kCompensateLen)
    return A->vt == MPH_F32 ? launch_comp<float, DIA>(A, k, x, y, init, s)
                            : launch_comp<bf16, DIA>(A, k, x, y, init, s);
  if (DIA && dia_pair_ok(A, k))
    return A->vt == MPH_F32 ? launch_dia_pair<float>(A, x, y, init, s)
                            : launch_dia_pair<bf16>(A, x, y, init, s);
  if (!DIA && ell_pair_ok(A, k))
    return A->vt == MPH_F32 ? launch_ell_pair<float>(A, x, y, init, s)
                            : launch_ell_pair<bf16>(A, x, y, init, s);
  if (DIA && k == 1 && A->dia_stage.n > 0 && A->tuning.rows_per_thread == 0)
    return A->vt == MPH_F64   ? launch_dia_staged<double>(A, x, y, init, s)
           : A->vt == MPH_F32 ? launch_dia_staged<float>(A, x, y, init, s)
                              : launch_dia_staged<bf16>(A, x, y, init, s);
  const bool two = A->tuning.rows_per_thread == 2;
  switch (A->vt) {
    case MPH_F64:
      return two ? launch_fmt<double, DIA, 2>(A, k, x, y, init, s)
                 : launch_fmt<double, DIA, 1>(A, k, x, y, init, s);
    case MPH_F32:
      return two ? launch_fmt<float, DIA, 2>(A, k, x, y, init, s)
                 : launch_fmt<float, DIA, 1>(A, k, x, y, init, s);
    case MPH_BF16:
      return two ? launch_fmt<bf16, DIA, 2>(A, k, x, y, init, s)
                 : launch_fmt<bf16, DIA, 1>(A, k, x, y, init, s);
  }
  return invalid("unknown value type");
}

}  // namespace

// Clusters of consecutive diagonals (storage order) whose offsets span at
// most kDiaClusterSpan; a cluster of two or more diagonals is staged.  More
// than kDiaStageMaxDiags diagonals, more than kDiaMaxClusters staged
// clusters, windows beyond kDiaStageMax entries or nothing worth staging:
// the plain kernel (n = 0).
int dia_analyse(mph_matrix_impl* A, hipStream_t s) {
  A->dia_stage = DiaStage{};
  A->dia_reach = A->dia_runs = 0;
  const int64_t nd = A->ndiag;
  if (nd < 2 || nd > kDiaStageMaxDiags || A->nrows == 0 || A->ncols == 0) return MPH_OK;
  int mode = 2;  // MPH_DIA_STAGE: 0 off, 1 the one-row kernels only, 2 also the row pairs
  if (const char* env = std::getenv("MPH_DIA_STAGE")) mode = std::atoi(env);
  std::vector<int32_t> off((size_t)nd);
  MPH_HIP_CHECK(hipMemcpyAsync(off.data(), A->dia_off, sizeof(int32_t) * nd,
                               hipMemcpyDeviceToHost, s));
  MPH_HIP_CHECK(hipStreamSynchronize(s));
  // for the SpMM's run forms: the farthest diagonal, and the runs
  for (int64_t i = 0, len = 0; i < nd; i++) {
    A->dia_reach = std::max<int64_t>(A->dia_reach, std::abs((int64_t)off[i]));
    len = i > 0 && len < kDiaRunMax && (int64_t)off[i - 1] + 1 == off[i] ? len + 1 : 1;
    A->dia_runs += len == 1 ? 1 : 0;
  }
  if (mode <= 0) return MPH_OK;
  DiaStage st{};
  int32_t used = 0;
  int64_t staged_diags = 0;
  for (int64_t i = 0; i < nd;) {
    int64_t lo = off[i], hi = off[i], j = i + 1;
    while (j < nd && std::max<int64_t>(hi, off[j]) - std::min<int64_t>(lo, off[j]) <= kDiaClusterSpan) {
      lo = std::min<int64_t>(lo, off[j]);
      hi = std::max<int64_t>(hi, off[j]);
      j++;
    }
    int32_t lb = kDiaDirect, lb2 = kDiaDirect;
    if (j - i >= 2) {
      const int32_t len = (int32_t)(256 + hi - lo);
      if (st.n == kDiaMaxClusters || used + len > kDiaStageMax ||
          lo < -(int64_t)(INT32_MAX - 4 * kDiaStageMax))
        return MPH_OK;
      const int c = st.n++;
      st.omin[c] = (int32_t)lo;
      st.base[c] = used;
      st.len[c] = len;
      lb = used - (int32_t)lo;
      lb2 = used + 256 * c - (int32_t)lo;
      used += len;
      staged_diags += j - i;
    }
    for (int64_t d = i; d < j; d++) {
      st.lb[d] = lb;
      st.lb2[d] = lb2;
    }
    i = j;
  }
  if (st.n == 0) return MPH_OK;
  // the row-pair layout: windows 256 entries longer
  // the row pairs move half the bytes per x entry and finish a workgroup's
  // rows sooner: staging pays there only when the staged clusters average
  // kDiaPairMinDiags diagonals or more (27-point stencil: 9 per cluster, FP32
  // 125 -> 108 us; 7-point: one cluster of 5, BF16 21.5 -> 23.7 us)
  st.pair = mode >= 2 && used + 256 * st.n <= 2 * kDiaStageMax &&
            staged_diags >= (int64_t)kDiaPairMinDiags * st.n;
  A->dia_stage = st;
  return MPH_OK;
}

int dia_multiply(mph_matrix_impl* A, int k, const void* x, void* y, int init,
                 hipStream_t s) {
  return dispatch<true>(A, k, x, y, init, s);
}

int hdc_tail_multiply(mph_matrix_impl* A, const void* x, void* y, int init, hipStream_t s) {
  if (A->format != MPH_HDC || A->vt != MPH_F64 || A->dia_stage.n == 0)
    return runtime_error("HDC tail pass: unsupported plan");
  DiaArgs<double> a{};
  a.nrows = A->nrows;
  a.ncols = A->ncols;
  a.ndiag = (int32_t)A->ndiag;
  a.pitch = A->dia_pitch;
  a.off = A->dia_off;
  a.val = static_cast<const double*>(A->dia_v);
  a.x = static_cast<const double*>(x);
  a.y = static_cast<double*>(y);
  a.ld = 1;
  a.init = init;
  a.tro = A->csr_ro;
  a.tci = A->csr_ci;
  a.tval = static_cast<const double*>(A->csr_v);
  const int64_t nb = ceil_div(A->nrows, 256);
  if (nb == 0) return MPH_OK;
  hipLaunchKernelGGL((dia_staged_kernel<double, true>), dim3((unsigned)nb), dim3(256), 0, s, a,
                     A->dia_stage);
  MPH_HIP_CHECK(hipGetLastError());
  return MPH_OK;
}

int ell_multiply(mph_matrix_impl* A, int k, const void* x, void* y, int init,
                 hipStream_t s) {
  return dispatch<false>(A, k, x, y, init, s);
}

}  // namespace mph
