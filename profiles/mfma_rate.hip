// Rate of bare f16 MFMAs on all CUs, operands in registers, constant and random data.
//   hipcc --offload-arch=gfx950 -O3 -Xclang -target-feature -Xclang -packed-fp32-ops \
//       profiles/mfma_rate.hip -o <out>/mfma_rate
#include <hip/hip_runtime.h>
#include <cstdio>
#include <cstdlib>
#include <vector>
typedef float f16v __attribute__((ext_vector_type(16)));
typedef float f4v __attribute__((ext_vector_type(4)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
// Eight waves a workgroup, one workgroup a CU; four operand pairs and four accumulators a wave.
template <bool kBig>
__global__ __launch_bounds__(512) void rate(const h8* in, float* out, int steps) {
  h8 a[4], b[4];
  for (int i = 0; i < 4; ++i) { a[i] = in[(threadIdx.x + 512 * i) & 4095]; b[i] = in[(threadIdx.x + 512 * (i + 4)) & 4095]; }
  float s = 0;
  if constexpr (kBig) {
    f16v c[4] = {};
    for (int t = 0; t < steps; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) c[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[i], b[i], c[i], 0, 0, 0);
    for (int i = 0; i < 4; ++i) for (int r = 0; r < 16; ++r) s += c[i][r];
  } else {
    f4v c[4] = {};
    for (int t = 0; t < 2 * steps; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) c[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[i], b[i], c[i], 0, 0, 0);
    for (int i = 0; i < 4; ++i) for (int r = 0; r < 4; ++r) s += c[i][r];
  }
  out[blockIdx.x * 512 + threadIdx.x] = s;
}
int main() {
  const int steps = 20000, blocks = 256;
  std::vector<_Float16> h(4096 * 8);
  h8* in; float* out;
  if (hipMalloc(&in, 4096 * 16) != hipSuccess || hipMalloc(&out, blocks * 512 * 4) != hipSuccess) return 1;
  for (int random = 0; random < 2; ++random) {
    srand(1);
    for (auto& v : h) v = random ? (_Float16)((rand() % 2001 - 1000) / 500.0f) : (_Float16)1.0f;
    if (hipMemcpy(in, h.data(), h.size() * 2, hipMemcpyHostToDevice) != hipSuccess) return 1;
    for (int big = 0; big < 2; ++big) {
      hipEvent_t e0, e1; (void)hipEventCreate(&e0); (void)hipEventCreate(&e1);
      float best = 1e9f;
      for (int i = 0; i < 6; ++i) {
        (void)hipEventRecord(e0);
        if (big) rate<true><<<blocks, 512>>>(in, out, steps); else rate<false><<<blocks, 512>>>(in, out, steps);
        (void)hipEventRecord(e1);
        if (hipEventSynchronize(e1) != hipSuccess) return 1;
        float ms; (void)hipEventElapsedTime(&ms, e0, e1); if (ms < best) best = ms;
      }
      // 32x32x16: steps * 4 MFMAs of 32768 operations a wave; 16x16x32: twice as many of 16384
      const double flop = (double)steps * 4 * 32768 * 8 * blocks;
      // a SIMD issues for its two waves: 32 (16) cycles each
      const double cycles = (double)steps * 4 * 32 * 2;
      printf("%s data, %s: %.3f ms, %.2f PFLOP/s, %.2f GHz if the cores never idle\n", random ? "random" : "constant",
             big ? "32x32x16" : "16x16x32", best, flop / best * 1e-12, cycles / best * 1e-6);
    }
  }
  return 0;
}
