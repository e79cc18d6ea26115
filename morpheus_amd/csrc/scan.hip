// scan.hip -- device prefix sums and fills used by the analysis and the
// on-GPU converters.  Per-tile sums, then the per-tile exclusive scan, each
// workgroup adding up the sums of the tiles before its own; past kDirectTiles
// tiles a single-workgroup scan of the sums runs between the two.
#include "mph_internal.hpp"

namespace mph {

namespace {

constexpr int kScanThreads = 256;
constexpr int kScanItems = 8;
constexpr int kScanTile = kScanThreads * kScanItems;
// up to this many tiles (8.4M counts) every workgroup reads the sums before
// it (at most 32 KiB, from L2): the scan of 575K digit counts in the COO sort
// takes 11 us in two launches, 15 us in three.
constexpr int64_t kDirectTiles = 4096;

// Inclusive scan of one value per thread over a 256-thread block.
template <typename T>
__device__ T block_inclusive_scan(T v, T* s_wave, T& total) {
  const int lane = threadIdx.x % kWave;
  const int wave = threadIdx.x / kWave;
  for (int d = 1; d < kWave; d <<= 1) {
    T o = shfl_up(v, d);
    if (lane >= d) v += o;
  }
  if (lane == kWave - 1) s_wave[wave] = v;
  __syncthreads();
  T base = 0;
  total = 0;
  for (int w = 0; w < kScanThreads / kWave; w++) {
    if (w < wave) base += s_wave[w];
    total += s_wave[w];
  }
  __syncthreads();
  return v + base;
}

__global__ __launch_bounds__(kScanThreads) void tile_sums_kernel(
    const int32_t* __restrict__ in, int64_t n, int64_t* __restrict__ sums) {
  __shared__ int64_t s_wave[kScanThreads / kWave];
  const int64_t base = (int64_t)blockIdx.x * kScanTile;
  int64_t v = 0;
  for (int k = 0; k < kScanItems; k++) {
    const int64_t i = base + threadIdx.x + (int64_t)k * kScanThreads;
    if (i < n) v += in[i];
  }
  int64_t total;
  block_inclusive_scan<int64_t>(v, s_wave, total);
  if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

__global__ __launch_bounds__(kScanThreads) void scan_sums_kernel(
    int64_t* __restrict__ sums, int64_t nt) {
  __shared__ int64_t s_wave[kScanThreads / kWave];
  int64_t carry = 0;
  for (int64_t base = 0; base < nt; base += kScanThreads) {
    const int64_t i = base + threadIdx.x;
    const int64_t v = i < nt ? sums[i] : 0;
    int64_t total;
    const int64_t inc = block_inclusive_scan<int64_t>(v, s_wave, total);
    if (i < nt) sums[i] = carry + inc - v;
    carry += total;
  }
  if (threadIdx.x == 0) sums[nt] = carry;
}

__global__ __launch_bounds__(kScanThreads) void tile_scan_kernel(
    const int32_t* __restrict__ in, int32_t* __restrict__ out, int64_t n,
    const int64_t* __restrict__ sums, int64_t nt, int direct) {
  __shared__ int64_t s_wave[kScanThreads / kWave];
  const int64_t base = (int64_t)blockIdx.x * kScanTile;
  // each thread owns kScanItems consecutive elements
  const int64_t mine = base + (int64_t)threadIdx.x * kScanItems;
  int32_t vals[kScanItems];
  for (int k = 0; k < kScanItems; k++) vals[k] = mine + k < n ? in[mine + k] : 0;
  int64_t before = 0, local = 0;
  if (direct) {
    int64_t v = 0;
    for (int64_t q = threadIdx.x; q < blockIdx.x; q += kScanThreads) v += sums[q];
    block_inclusive_scan<int64_t>(v, s_wave, before);
  } else {
    before = sums[blockIdx.x];
  }
  for (int k = 0; k < kScanItems; k++) local += vals[k];
  int64_t total;
  const int64_t inc = block_inclusive_scan<int64_t>(local, s_wave, total);
  int64_t run = before + inc - local;
  for (int k = 0; k < kScanItems; k++) {
    const int64_t i = mine + k;
    if (i < n) out[i] = (int32_t)run;
    run += vals[k];
  }
  if (blockIdx.x == nt - 1 && threadIdx.x == kScanThreads - 1) out[n] = (int32_t)run;
}

template <typename W>
__global__ __launch_bounds__(256) void fill_zero_kernel(W* __restrict__ p, int64_t nwords) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nwords; i += stride)
    p[i] = W{};
}

}  // namespace

int64_t scan_tmp_elems(int64_t n) { return ceil_div(n, kScanTile) + 2; }

int exclusive_scan_i32(const int32_t* in, int32_t* out, int64_t n,
                       int64_t* tmp, hipStream_t s) {
  if (n < 0) return invalid("scan: negative length");
  const int64_t nt = ceil_div(n, kScanTile);
  if (nt == 0) {
    // out[0] = 0
    hipLaunchKernelGGL(fill_zero_kernel<int32_t>, dim3(1), dim3(64), 0, s, out, (int64_t)1);
    MPH_HIP_CHECK(hipGetLastError());
    return MPH_OK;
  }
  hipLaunchKernelGGL(tile_sums_kernel, dim3((unsigned)nt), dim3(kScanThreads),
                     0, s, in, n, tmp);
  const bool direct = nt <= kDirectTiles;
  if (!direct)
    hipLaunchKernelGGL(scan_sums_kernel, dim3(1), dim3(kScanThreads), 0, s, tmp, nt);
  hipLaunchKernelGGL(tile_scan_kernel, dim3((unsigned)nt), dim3(kScanThreads), 0, s, in, out, n, tmp,
                     nt, direct ? 1 : 0);
  MPH_HIP_CHECK(hipGetLastError());
  return MPH_OK;
}

// Clears device memory with a kernel rather than hipMemsetAsync so that the
// call stays safe inside captured hipGraphs.  16-byte stores over the aligned
// part, then the bytes left.
int fill_zero(void* p, size_t bytes, hipStream_t s) {
  if (bytes == 0) return MPH_OK;
  const size_t wide = reinterpret_cast<uintptr_t>(p) % 16 == 0 ? bytes / 16
                                                                : 0;
  const size_t word = reinterpret_cast<uintptr_t>(p) % 4 == 0 ? (bytes - wide * 16) / 4 : 0;
  auto launch = [&](auto tag, size_t at, size_t n) {
    using W = decltype(tag);
    if (n == 0) return;
    const unsigned g = (unsigned)std::min<int64_t>(ceil_div((int64_t)n, 256), 16384);
    hipLaunchKernelGGL(fill_zero_kernel<W>, dim3(g), dim3(256), 0, s,
                       reinterpret_cast<W*>(static_cast<uint8_t*>(p) + at), (int64_t)n);
  };
  launch(uint4{}, 0, wide);
  launch(uint32_t{}, wide * 16, word);
  launch(uint8_t{}, wide * 16 + word * 4, bytes - wide * 16 - word * 4);
  MPH_HIP_CHECK(hipGetLastError());
  return MPH_OK;
}

}  // namespace mph
