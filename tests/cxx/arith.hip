// Test caller of the kernels' division and square root (csrc/physics.hpp): elementwise over host
// arrays of n values.  op 0: quot in FP64, 1: quot in FP32, 2: sqrt_ in FP64.  Returns 0 when all
// HIP calls succeeded.
#include "../../idefix_amd/csrc/physics.hpp"

namespace {
template <typename T, int OP>
__global__ void k_arith(const T *a, const T *b, T *out, int n) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= n) return;
  if constexpr (OP == 2) out[q] = idfx::sqrt_(a[q]);
  else out[q] = idfx::quot(a[q], idfx::recip(b[q]));
}
template <typename T, int OP>
int run(const void *a, const void *b, void *out, int n) {
  const size_t bytes = sizeof(T) * (size_t)n;
  T *d = nullptr;
  if (hipMalloc(&d, 3 * bytes) != hipSuccess) return 1;
  int st = hipMemcpy(d, a, bytes, hipMemcpyHostToDevice) != hipSuccess ||
           hipMemcpy(d + n, b, bytes, hipMemcpyHostToDevice) != hipSuccess;
  if (!st) {
    hipLaunchKernelGGL((k_arith<T, OP>), dim3((n + 255) / 256), dim3(256), 0, nullptr, d, d + n, d + 2 * n, n);
    st = hipGetLastError() != hipSuccess || hipMemcpy(out, d + 2 * n, bytes, hipMemcpyDeviceToHost) != hipSuccess;
  }
  return (hipFree(d) != hipSuccess) | st;
}
}  // namespace

extern "C" int arith(int op, const void *a, const void *b, void *out, int n) {
  if (n < 1 || n > (1 << 28)) return 1;
  return op == 0 ? run<double, 0>(a, b, out, n) : op == 1 ? run<float, 1>(a, b, out, n)
                                                : op == 2 ? run<double, 2>(a, b, out, n) : 1;
}
