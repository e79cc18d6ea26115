// validate.hip -- one-time checks run by the analysis, so that malformed
// input or a malformed analysis is reported as MPH_ERR_INVALID_INPUT /
// MPH_ERR_RUNTIME instead of reaching a kernel as an out-of-range access.
//
//  * index arrays: every row / column index inside its dimension (ELL: or
//    the -1 padding marker); CSR row offsets start at 0, never decrease and
//    end at nnz;
//  * (row-block plans are checked by the kernel that writes their records,
//    spmv_rowblock.hip.)
#include <functional>
#include <vector>

#include "mph_internal.hpp"

namespace mph {

namespace {

// Bad entries raise `bit` in flag[0]: eight indices a thread, loaded
// together (one a thread took 22 us for 16M indices, 2.9 TB/s).  Nothing is
// read when a launch before this one raised a bit of `unless`: n is then not
// known to be the array's length.
constexpr int kCheckPer = 8;
__global__ __launch_bounds__(256) void index_range_kernel(const int32_t* __restrict__ idx,
                                                          int64_t n, int64_t hi, int allow_m1,
                                                          int32_t bit, int32_t unless,
                                                          int32_t* __restrict__ flag) {
  if (__hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & unless) return;
  const int64_t base = (int64_t)blockIdx.x * 256 * kCheckPer + threadIdx.x;
  int32_t v[kCheckPer];
  bool ok = true;
#pragma unroll
  for (int k = 0; k < kCheckPer; k++) v[k] = idx[min(base + k * 256, n - 1)];
#pragma unroll
  for (int k = 0; k < kCheckPer; k++)
    ok = ok && ((v[k] >= 0 && v[k] < hi) || (allow_m1 && v[k] == -1));
  if (!ok) atomicOr(flag, bit);
}

__global__ __launch_bounds__(256) void row_offsets_kernel(const int32_t* __restrict__ ro,
                                                          int64_t nrows, int64_t nnz, int32_t bit,
                                                          int32_t* __restrict__ flag) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i > nrows) return;
  bool ok = true;
  if (i == 0) ok = ro[0] == 0;
  if (i == nrows) ok = ok && (int64_t)ro[nrows] == nnz;
  if (i < nrows) ok = ok && ro[i] <= ro[i + 1];
  if (!ok) atomicOr(flag, bit);
}

void launch_index_range(const int32_t* idx, int64_t n, int64_t hi, bool allow_m1, int32_t bit,
                        int32_t unless, int32_t* flag, hipStream_t s) {
  hipLaunchKernelGGL(index_range_kernel, dim3((unsigned)ceil_div(n, 256 * kCheckPer)), dim3(256), 0,
                     s, idx, n, hi, allow_m1 ? 1 : 0, bit, unless, flag);
}

void launch_row_offsets(const int32_t* ro, int64_t nrows, int64_t nnz, int32_t bit, int32_t* flag,
                        hipStream_t s) {
  hipLaunchKernelGGL(row_offsets_kernel, dim3((unsigned)ceil_div(nrows + 1, 256)), dim3(256), 0, s,
                     ro, nrows, nnz, bit, flag);
}

int run_flag_check(hipStream_t s, int* bad,
                   const std::function<void(int32_t*)>& launch) {
  Tmp t(s);
  int32_t* flag = nullptr;
  MPH_CHECK_STATUS(t.alloc(&flag, 1));
  MPH_CHECK_STATUS(fill_zero(flag, sizeof(int32_t), s));
  launch(flag);
  MPH_HIP_CHECK(hipGetLastError());
  MPH_CHECK_STATUS(t.read(flag, bad));
  t.idle = true;
  return MPH_OK;
}

}  // namespace

int check_index_range(const int32_t* idx, int64_t n, int64_t hi, bool allow_m1,
                      hipStream_t s, const char* what) {
  if (n <= 0) return MPH_OK;
  int bad = 0;
  MPH_CHECK_STATUS(run_flag_check(s, &bad, [&](int32_t* flag) {
    launch_index_range(idx, n, hi, allow_m1, 1, 0, flag, s);
  }));
  if (bad) return invalid(std::string(what) + ": index out of range");
  return MPH_OK;
}

int check_row_offsets(const int32_t* ro, int64_t nrows, int64_t nnz,
                      hipStream_t s, const char* what) {
  int bad = 0;
  MPH_CHECK_STATUS(run_flag_check(s, &bad, [&](int32_t* flag) {
    launch_row_offsets(ro, nrows, nnz, 1, flag, s);
  }));
  if (bad)
    return invalid(std::string(what) +
                   ": row offsets must start at 0, not decrease and end at nnz");
  return MPH_OK;
}

int check_csr(const int32_t* ro, int64_t nrows, int64_t nnz, const int32_t* ci, int64_t ncols,
              hipStream_t s) {
  int bad = 0;
  MPH_CHECK_STATUS(run_flag_check(s, &bad, [&](int32_t* flag) {
    launch_row_offsets(ro, nrows, nnz, 1, flag, s);
    // (nnz columns only if the offsets end there)
    if (nnz > 0) launch_index_range(ci, nnz, ncols, false, 2, 1, flag, s);
  }));
  if (bad & 1)
    return invalid("CSR row_offsets: row offsets must start at 0, not decrease and end at nnz");
  if (bad & 2) return invalid("CSR column_indices: index out of range");
  return MPH_OK;
}

}  // namespace mph
