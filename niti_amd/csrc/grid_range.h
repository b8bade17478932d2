// Tensor-wide range of a launch whose workgroups are all resident: every workgroup publishes its largest magnitude in a
// slot of its own, reads all slots and rounds with the shift that follows.  `Args` is the kernel's argument structure; it
// has sync, spin_limit, sticky, bw_mode, target_bits, shift_out, exp_a, exp_b, exp_out.
#pragma once
#include "common.h"
#include "requant_math.h"

namespace niti {

constexpr int kSlot0 = 16;   // sync words: 0 range out, 1 wait gave up, 16.. one slot per workgroup
constexpr int kMaxSlots = 4096;

// Four sums -> four rounded values, the branches on the method taken once for all of them and everything in 32 bits (a
// tile's 32 values per thread rounded one by one in 64-bit arithmetic took as long as the tensor-wide exchange)
__device__ inline v4i round4_any(v4i x, int shift, int method, bool trunc, v4i u) {
  v4i r;
  if (shift < 1) {
#pragma unroll
    for (int e = 0; e < 4; ++e) r[e] = wrap_to_i8(x[e]);
  } else if (method == NITI_ROUND_STOCHASTIC) {
#pragma unroll
    for (int e = 0; e < 4; ++e) r[e] = round_sto32(x[e], shift, trunc, u[e]);
  } else if (method == NITI_ROUND_PSEUDO_STOCHASTIC) {
#pragma unroll
    for (int e = 0; e < 4; ++e) r[e] = round_one32<NITI_ROUND_PSEUDO_STOCHASTIC>(x[e], shift, trunc);
  } else if (!trunc) {
#pragma unroll
    for (int e = 0; e < 4; ++e) r[e] = round_nearest_floor_fast(x[e], shift - 1, -127);
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) r[e] = round_one32<NITI_ROUND_NEAREST>(x[e], shift, trunc);
  }
  return r;
}

template <class Args>
__device__ inline void write_scalars(const Args& a, uint32_t gmax, int shift) {
  const int sh = shift > 0 ? shift : 0;
  a.sync[0] = gmax;
  if (a.shift_out != nullptr) *a.shift_out = sh;
  if (a.exp_out != nullptr) *a.exp_out = sh + (a.exp_a != nullptr ? *a.exp_a : 0) + (a.exp_b != nullptr ? *a.exp_b : 0);
}

// Called by wavefront 0 of every workgroup with the workgroup's largest magnitude: the largest over the grid.
template <class Args>
__device__ inline uint32_t exchange_range(const Args& a, uint32_t bmax) {
  const int lane = threadIdx.x & 63;
  const int nb = gridDim.x * gridDim.y;
  const int b = blockIdx.y * gridDim.x + blockIdx.x;
  uint32_t* const slots = a.sync + kSlot0;
  if (lane == 0) __hip_atomic_store(slot_word(slots, b), bmax + 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const uint32_t g = wait_slots(slots, nb, a.spin_limit, &a.sync[1], a.sticky);
  return g != 0u ? g - 1u : 0u;
}

// the workgroup's shift from every wavefront's largest magnitude: wmax[] holds one word per wavefront, gshare the result
template <int NWAVES, class Args>
__device__ inline int grid_shift(const Args& a, uint32_t lmax, uint32_t* wmax, uint32_t* gshare) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  lmax = wave_max_u32(lmax);
  if (lane == 0) wmax[wave] = lmax;
  __syncthreads();
  if (wave == 0) {
    uint32_t b = lane < NWAVES ? wmax[lane] : 0u;
    b = wave_max_u32(b);
    const uint32_t g = exchange_range(a, b);
    if (lane == 0) *gshare = g;
  }
  __syncthreads();
  const uint32_t gmax = *gshare;
  const int shift = bitwidth_of(gmax, a.bw_mode) - a.target_bits;
  if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) write_scalars(a, gmax, shift);
  return shift;
}

}  // namespace niti
