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

struct Nothing {
  __device__ void operator()() const {}
};

// The workgroup's shift from every wavefront's largest magnitude: wmax[] holds one word per wavefront, gshare the result.
// `block` of `blocks` workgroups take part.  meanwhile(): called by every wavefront behind the workgroup's own slot and in front of
// the looks at the others', for requests whose trip to memory may run beside the exchange.
template <int NWAVES, class Args, class Meanwhile = Nothing>
__device__ inline int grid_shift(const Args& a, uint32_t lmax, uint32_t* wmax, uint32_t* gshare, int block, int blocks, Meanwhile meanwhile = {}) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  lmax = wave_max_u32(lmax);
  if (lane == 0) wmax[wave] = lmax;
  __syncthreads();
  if (wave == 0) {
    const uint32_t b = wave_max_u32(lane < NWAVES ? wmax[lane] : 0u);
    if (lane == 0) __hip_atomic_store(slot_word(a.sync + kSlot0, block), b + 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  meanwhile();
  if (wave == 0) {
    const uint32_t g = wait_slots(a.sync + kSlot0, blocks, a.spin_limit, &a.sync[1], a.sticky);
    if (lane == 0) *gshare = g != 0u ? g - 1u : 0u;
  }
  __syncthreads();
  const uint32_t gmax = *gshare;
  const int shift = bitwidth_of(gmax, a.bw_mode) - a.target_bits;
  if (block == 0 && threadIdx.x == 0) write_scalars(a, gmax, shift);
  return shift;
}
template <int NWAVES, class Args, class Meanwhile = Nothing>
__device__ inline int grid_shift(const Args& a, uint32_t lmax, uint32_t* wmax, uint32_t* gshare, Meanwhile meanwhile = {}) {
  return grid_shift<NWAVES>(a, lmax, wmax, gshare, blockIdx.y * gridDim.x + blockIdx.x, gridDim.x * gridDim.y, meanwhile);
}

// A weight update next to the data gradient `first` that reads the old weights, in one launch: the update's workgroups wait for
// both ranges - a workgroup of the data gradient fills its slot when it has read its weights - and the gradient's exponent
// builds on the error's that comes out of this launch.  Waits that give up say so in the data gradient's words, the first of the
// call's.  share: two words.  meanwhile(): see grid_shift.
template <int NWAVES, class Args, class Meanwhile>
__device__ inline int grid_shift_behind(const Args& a, const Args& first, int first_blocks, uint32_t lmax, uint32_t* wmax, uint32_t* share, int block,
                                        int blocks, Meanwhile meanwhile) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  lmax = wave_max_u32(lmax);
  if (lane == 0) wmax[wave] = lmax;
  __syncthreads();
  if (wave == 0) {
    const uint32_t b = wave_max_u32(lane < NWAVES ? wmax[lane] : 0u);
    if (lane == 0) __hip_atomic_store(slot_word(a.sync + kSlot0, block), b + 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  meanwhile();
  if (wave == 0) {
    const uint32_t f = wait_slots(first.sync + kSlot0, first_blocks, a.spin_limit, &first.sync[1], a.sticky, kWaitUpdate);
    const uint32_t g = wait_slots(a.sync + kSlot0, blocks, a.spin_limit, &first.sync[1], a.sticky, kWaitUpdate);
    if (lane == 0) {
      share[0] = g != 0u ? g - 1u : 0u;
      share[1] = f != 0u ? f - 1u : 0u;
    }
  }
  __syncthreads();
  const uint32_t gmax = share[0];
  const int shift = bitwidth_of(gmax, a.bw_mode) - a.target_bits;
  if (block == 0 && threadIdx.x == 0) {
    const int sh = max(shift, 0), before = max(bitwidth_of(share[1], first.bw_mode) - first.target_bits, 0);
    a.sync[0] = gmax;
    if (a.shift_out != nullptr) *a.shift_out = sh;
    if (a.exp_out != nullptr)
      *a.exp_out = sh + before + (first.exp_a != nullptr ? *first.exp_a : 0) + (first.exp_b != nullptr ? *first.exp_b : 0) + (a.exp_b != nullptr ? *a.exp_b : 0);
  }
  return shift;
}

}  // namespace niti
