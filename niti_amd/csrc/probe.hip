// Measurement aid: a register-resident int8 MFMA loop (no LDS, no memory traffic inside the loop) over operands
// the caller supplies.  The rate this loop sustains is the matrix-unit ceiling for those operand VALUES: on MI355X
// the shader clock follows the power the multipliers draw, so uniform random int8 operands run at a markedly lower
// clock (and rate) than constant ones.  bench.py reports both next to the datasheet peak.
#include <type_traits>

#include "common.h"

namespace niti {
namespace {

// 8 wavefronts per workgroup; `iters` rounds of 12 x 65536 operations each on operand fragments loaded once, in the register shape
// of the convolution kernel that uses the instruction: 12 products of 32 x 32 x 32 on 2 x 2 accumulator tiles (2 filter fragments of each
// of 3 taps x 2 pixel fragments), or 24 of 16 x 16 x 64 on 2 x 4 (x 4 pixel fragments).
template <bool k16x16x64>
__global__ __launch_bounds__(512, 2) void mfma_probe_kernel(const int8_t* __restrict__ operands, long long bytes, int iters,
                                                            int32_t* __restrict__ out, long long* __restrict__ clocks) {
  using Sum = std::conditional_t<k16x16x64, v4i, v16i>;
  constexpr int P = k16x16x64 ? 4 : 2, E = k16x16x64 ? 4 : 16;
  const int tid = threadIdx.x;
  v4i pc[P], wf[3][2];
  const long long frag = (static_cast<long long>(blockIdx.x) * 512 + tid) * (6 + P);   // this lane's first 16-byte fragment
  const long long nfrag = bytes / 16;
  auto load = [&](int i) { return reinterpret_cast<const v4i*>(operands)[(frag + i) % nfrag]; };
#pragma unroll
  for (int j = 0; j < P; ++j) pc[j] = load(j);
#pragma unroll
  for (int s = 0; s < 3; ++s)
#pragma unroll
    for (int i = 0; i < 2; ++i) wf[s][i] = load(P + s * 2 + i);
  Sum acc[2][P];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < P; ++j)
#pragma unroll
      for (int e = 0; e < E; ++e) acc[i][j][e] = 0;
  const long long c0 = __builtin_readcyclecounter();
  const long long w0 = wall_clock64();
  for (int it = 0; it < iters; ++it) {
#pragma unroll
    for (int s = 0; s < 3; ++s)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < P; ++j) {
          if constexpr (k16x16x64) acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf[s][i], pc[j], acc[i][j], 0, 0, 0);
          else acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(wf[s][i], pc[j], acc[i][j], 0, 0, 0);
        }
    // the accumulators wrap; keep the operands opaque so that the loop is not folded
#pragma unroll
    for (int j = 0; j < P; ++j) asm volatile("" : "+v"(pc[j]));
  }
  int sum = 0;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < P; ++j)
#pragma unroll
      for (int e = 0; e < E; ++e) sum += acc[i][j][e];
  out[static_cast<long long>(blockIdx.x) * 512 + tid] = sum;
  if (blockIdx.x == 0 && tid == 0 && clocks != nullptr) {
    clocks[0] = __builtin_readcyclecounter() - c0;   // shader clocks
    clocks[1] = wall_clock64() - w0;                 // 100 MHz ticks
  }
}

template <bool k16x16x64>
int probe(const char* who, const int8_t* operands, size_t operand_bytes, int workgroups, int iters, int32_t* out, int64_t* clocks, void* stream) {
  clear_error();
  if (operands == nullptr || out == nullptr || !aligned16(operands)) return fail(NITI_ERR_INVALID_ARG, "%s: null or misaligned pointer", who);
  if (operand_bytes < 128 || workgroups <= 0 || workgroups > 65535 || iters <= 0)
    return fail(NITI_ERR_INVALID_ARG, "%s: operand_bytes=%zu workgroups=%d iters=%d", who, operand_bytes, workgroups, iters);
  hipLaunchKernelGGL(mfma_probe_kernel<k16x16x64>, dim3(workgroups), dim3(512), 0, static_cast<hipStream_t>(stream), operands,
                     static_cast<long long>(operand_bytes), iters, out, reinterpret_cast<long long*>(clocks));
  return check_launch(who);
}

}  // namespace
}  // namespace niti

using namespace niti;

extern "C" int niti_mfma_probe_i8(const int8_t* operands, size_t operand_bytes, int workgroups, int iters, int32_t* out,
                                  int64_t* clocks, void* stream) {
  return probe<false>("mfma_probe", operands, operand_bytes, workgroups, iters, out, clocks, stream);
}

extern "C" int niti_mfma_probe_i8_16x16x64(const int8_t* operands, size_t operand_bytes, int workgroups, int iters, int32_t* out,
                                           int64_t* clocks, void* stream) {
  return probe<true>("mfma_probe_16x16x64", operands, operand_bytes, workgroups, iters, out, clocks, stream);
}
