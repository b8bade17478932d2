// Both gradients of a 3x3 layer whose weight gradient is the nine-tap kernel's, in two launches (ti_torch.py:404-437): the weight
// gradient's main loop, which leaves its partial sums in memory, then the data gradient, along with which they are added and the weights
// updated.
//
// Added by its own launch, the partial sums (24 to 28 MB whatever the layer) cost it an arrival wait, their way back from memory and a
// range exchange of its own, with the matrix units idle.  Here the next launch's start is the arrival, the sums come in while others
// multiply, and the two ranges are exchanged at the same time.  The copy of the filter that the data gradient reads is written behind the
// last of its slots.
//
// Both launches in replayed graphs against the data gradient's and the one-launch weight gradient's (us): 128 images of 32 x 32, 128 -> 128
// 59.6 -> 54.3, of 16 x 16, 128 -> 256 40.0 -> 34.5, 256 -> 256 55.8 -> 48.3, of 8 x 8, 256 -> 512 41.7 -> 36.2, 512 -> 512 53.9 -> 50.2;
// 80 of 16 x 16, 128 -> 256 41.3 -> 29.2.  Of the weight gradient's launch its main loop and the way out are left (25.5 -> 16.5 us at
// 16 x 16, 128 -> 256); the data gradient's grows by 3 to 7 us.  Timestamps of that layer: the slices are in at 9.5 us, their range known
// at 13.3, the error's at 14.4, the copy written at 15.6; the products end at 11.0.  What bounds it: the slices' way from memory beside the
// stages' loads, then one exchange.
#include <stdlib.h>

#include <algorithm>

#include "conv3x3_k64.h"
#include "conv_any.h"
#include "wgrad_finish.h"

namespace niti {
namespace {

constexpr int kBesideItems = 5, kWithinItems = 1;   // (two workgroups on a unit that multiply leave registers for one)
constexpr int per_cu_geometry(int ktile) { return ktile == 32 ? 1 : 2; }   // the 32-channel tile fits twice as it is

struct SumsWithin : SumsAlong<kWithinItems, false>, OneTile {
  using SumsAlong::SumsAlong;
};

// The first nx x ny workgroups are the data gradient's.  kOthers: the others finish the weight gradient; otherwise the last work.nblocks
// of them do so as well.
template <int Q, int BR, int NI, int KT, bool kOthers>
__global__ __launch_bounds__(512, 4) void conv3x3_k64_backward_kernel(const HaloArgs a, const FinishArgs f, const AlongWork work, const int nx, const int ny) {
  extern __shared__ __attribute__((aligned(16))) int8_t smem[];
  constexpr int kPer = per_cu_geometry(KT);
  const int id = blockIdx.x, first = nx * ny;
  const HaloPlace at{id % nx, id / nx, nx, ny};
  if constexpr (kOthers) {
    if (id < first) {
      NothingAlong along;
      k64_tile<Q, BR, NI, KT, kPer, true, true, false>(a, at, smem, along);
    } else {
      finish_beside(SumsAlong<kBesideItems, (KT < 128)>(f, work, id - first, smem), a, a.sync + kSyncSlot0, first);
    }
  } else {
    SumsWithin along(f, work, id - (first - work.nblocks), smem + KGeom<Q, BR, NI, KT, kPer>::LDS_BYTES);
    k64_tile<Q, BR, NI, KT, kPer, true, true, false>(a, at, smem, along);
  }
}

// More tiles of the data gradient than the device holds workgroups: several in turn, and the sums in front of the first of them.  Both
// launches against the data gradient's and the one-launch weight gradient's (us): 32 x 32, 128 -> 128 at 136 / 160 / 192 / 256 images
// 76.6 -> 69.9, 75.4 -> 70.0, 81.7 -> 75.5, 98.6 -> 91.6; 256 images of 16 x 16, 384 -> 256 153.1 -> 146.7, 512 -> 128 87.6 -> 87.6.  What bounds it: the
// tiles; the wait in front of the copy of the filter costs the 2 us of an exchange.  (15 or 16 registers spill, outside the loop.)
struct PairArgs {
  HaloArgs a;   // (first: tiles_in_turns)
  FinishArgs f;
  AlongWork work;
};
struct SumsInTurns : Turns {
  int8_t* const lds;
  bool summed = false;
  int guessed = 0;
  uint32_t wnew[kWithinItems];
  __device__ explicit SumsInTurns(int8_t* l) : lds(l) {}
  // made where it is used, from arguments the compiler has not seen: what follows from them is not kept in registers between the tiles
  __device__ __forceinline__ const PairArgs& arguments() const {
    using Args = const __attribute__((address_space(4))) PairArgs;
    Args* p = (Args*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *(const PairArgs*)p;
  }
  __device__ __forceinline__ SumsWithin sums() const {
    const PairArgs& args = arguments();
    return SumsWithin(args.f, args.work, static_cast<int>(blockIdx.x) - (static_cast<int>(gridDim.x) - args.work.nblocks), lds, thread());
  }
  __device__ __forceinline__ void begin() {
    if (!summed) sums().begin();
  }
  __device__ __forceinline__ void publish() {
    if (!summed) sums().publish();
    summed = true;
  }
  __device__ __forceinline__ void guess() {
    SumsWithin s = sums();
    s.guess();
    guessed = s.guessed;
#pragma unroll
    for (int i = 0; i < kWithinItems; ++i) wnew[i] = s.wnew[i];
  }
  __device__ __forceinline__ void wait(const HaloArgs& a) { sums().wait(a); }
  __device__ __forceinline__ void update(int shift, const int32_t* exp_a, const int32_t* exp_b) {
    Turns::update(shift, exp_a, exp_b);
    SumsWithin s = sums();
    if (s.block < 0) return;
    s.guessed = guessed;
#pragma unroll
    for (int i = 0; i < kWithinItems; ++i) s.wnew[i] = wnew[i];
    s.settle();
#pragma unroll
    for (int i = 0; i < kWithinItems; ++i) wnew[i] = s.wnew[i];
  }
  // Behind the last tile.  Tiles that are computed again read the copy of the filter again, so it changes when every workgroup has said that it has
  // none left (the third word of its slot).
  __device__ __forceinline__ void copy() {
    __syncthreads();
    const PairArgs& args = arguments();
    uint32_t* const done = args.a.sync + kSyncSlot0 + 2;
    if (threadIdx.x == 0) __hip_atomic_store(slot_word(done, blockIdx.x), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    SumsWithin s = sums();
    if (s.block < 0) return;
    if (s.wave == 0) wait_slots(done, gridDim.x, args.a.spin_limit, &args.a.sync[1], args.a.sticky, kWaitUpdate);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kWithinItems; ++i) s.wnew[i] = wnew[i];
    s.store_copy(final_shift, args.a.exp_a, args.a.exp_b);
  }
};
static_assert(kSlotStride >= 3, "a third word");
template <int Q, int BR, int NI, int KT>
__global__ __launch_bounds__(512, 4) void conv3x3_k64_backward_turns_kernel(const PairArgs, const int nx, const int ny) {
  extern __shared__ __attribute__((aligned(16))) int8_t smem[];
  SumsInTurns along(smem + KGeom<Q, BR, NI, KT, 2>::LDS_BYTES);
  tiles_in_turns(nx, ny, along, [&](const HaloArgs& a, const HaloPlace at) { k64_tile<Q, BR, NI, KT, 2, true, true, false>(a, at, smem, along); });
  along.copy();
}

enum PairWay { kBeside, kWithin, kInTurns };   // the sums: by workgroups of their own, by some of those with one tile each, with several
template <int Q, int BR, int NI, int KT, PairWay kWay>
constexpr auto pair_kernel() {
  if constexpr (kWay == kInTurns) return conv3x3_k64_backward_turns_kernel<Q, BR, NI, KT>;
  else return conv3x3_k64_backward_kernel<Q, BR, NI, KT, kWay == kBeside>;
}

struct PairPlan {
  int ktile;    // channel tile of the data gradient
  int nx, ny;   // its tiles, 0: not this way
  PairWay way;
  int blocks;   // workgroups of the launch
  AlongWork work;
};

// calls f(width, rows, images, channel tile, way) with the plan's numbers as types
template <class F>
auto with_geometry(int H, const PairPlan& p, F f) {
  using std::integral_constant;
  const auto tiles = [&](auto q, auto br, auto ni) {
    constexpr integral_constant<PairWay, kBeside> beside{};
    constexpr integral_constant<PairWay, kWithin> within{};
    if constexpr (decltype(q)::value <= 16) {
      if (p.ktile == 32) return f(q, br, ni, integral_constant<int, 32>{}, beside);
    }
    if (p.ktile == 64) return p.way == kBeside ? f(q, br, ni, integral_constant<int, 64>{}, beside) : f(q, br, ni, integral_constant<int, 64>{}, within);
    constexpr integral_constant<int, 128> wide{};
    return p.way == kBeside ? f(q, br, ni, wide, beside) : p.way == kWithin ? f(q, br, ni, wide, within) : f(q, br, ni, wide, integral_constant<PairWay, kInTurns>{});
  };
  if (H == 32) return tiles(integral_constant<int, 32>{}, integral_constant<int, 8>{}, integral_constant<int, 1>{});
  if (H == 16) return tiles(integral_constant<int, 16>{}, integral_constant<int, 16>{}, integral_constant<int, 1>{});
  return tiles(integral_constant<int, 8>{}, integral_constant<int, 8>{}, integral_constant<int, 4>{});
}

constexpr size_t kHalfLds = 80 * 1024;   // two workgroups on a unit

// Whether two of the plan's workgroups fit on a compute unit, in LDS for its chunks and in registers
bool fits_twice(int H, const PairPlan& p) {
  return with_geometry(H, p, [&](auto q, auto br, auto ni, auto kt, auto way) {
    constexpr int Q = decltype(q)::value, BR = decltype(br)::value, NI = decltype(ni)::value, KT = decltype(kt)::value;
    constexpr bool beside = decltype(way)::value == kBeside;
    using G = KGeom<Q, BR, NI, KT, per_cu_geometry(KT)>;
    static_assert(G::LDS_BYTES <= kHalfLds, "two workgroups on a unit");
    static_assert(8 * 32 * G::PT * (G::NWF * 32 + 16) <= G::TILE_BYTES, "int8 patches must stay clear of the reduction words");
    if (p.work.own > 8 * (beside ? kBesideItems : kWithinItems) || along_lds(p.work.own) + (beside ? 0 : G::LDS_BYTES) > kHalfLds) return false;
    static bool of[kDeviceSlots] = {};
    bool& twice = of[device_slot()];
    if (!twice) {
      auto k = pair_kernel<Q, BR, NI, KT, decltype(way)::value>();
      int per_cu = 0;
      if (hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, kHalfLds) != hipSuccess ||
          hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(k), 512, kHalfLds) != hipSuccess)
        return false;
      twice = per_cu >= 2;
    }
    return twice;
  });
}

PairPlan plan_for(int N, int H, int C, int K, int slices) {
  PairPlan p{};
  if (C % 64 != 0 || K <= 64 || (K + 31) / 32 % 2 != 0 || !conv3x3_halo_supported(N, H, H, K, C, 3, 3, 1, 1)) return p;   // the data gradient: K -> C
  const int cus = compute_units();
  const long long ptiles = (static_cast<long long>(N) * H * H + 255) / 256, units = static_cast<long long>(K) * 9 * C / 4;
  const auto blocks = [&](int ktile) { return ptiles * ((C + ktile - 1) / ktile); };
  p.ktile = H <= 16 && blocks(32) <= cus ? 32 : C == 64 || blocks(64) <= cus ? 64 : 128;
  const long long nb = blocks(p.ktile);
  if (nb < 2 || nb > kMaxSlots || (nb > 2LL * cus && p.ktile != 128)) return PairPlan{};
  p.nx = static_cast<int>(ptiles);
  p.ny = (C + p.ktile - 1) / p.ktile;
  const int room = static_cast<int>(std::max(2LL * cus - nb, 0LL)), held = static_cast<int>(std::min(nb, 2LL * cus));
  p.way = room >= cus / 4 ? kBeside : nb <= held ? kWithin : kInTurns;
  // Where those that multiply fill the device, the later ones of the two on each unit add the slices before their first stage: their
  // neighbours have the matrix units to themselves meanwhile (128 images of 32 x 32, 128 -> 128: 8.5 us, of which 4 show).
  // More than one of them per unit take part where that leaves none with more chunks than it has room for (both launches against the
  // data gradient's and the one-launch weight gradient's: 16 x 16, 256 -> 256 at 160 / 192 / 256 images 68.8 -> 60.3, 73.4 -> 65.3, 83.3 -> 80.4 us;
  // 200 images 256 -> 320 119.3 -> 109.7; five eighths or all of the workgroups instead of half 0 to 2 us slower).
  const long long least = ((units + 63) / 64 + 8 * kWithinItems - 1) / (8 * kWithinItems);
  p.work = along_work(units, slices, p.way == kBeside ? std::min(room, cus) : static_cast<int>(std::min<long long>(std::max<long long>(least, cus), held)));
  p.blocks = held + (p.way == kBeside ? p.work.nblocks : 0);
  return fits_twice(H, p) ? p : PairPlan{};
}

PairPlan pair_plan(int N, int H, int C, int K) {
  if ((H != 8 && H != 16 && H != 32) || C % 64 != 0 || K <= 0) return PairPlan{};
  const int slices = wgrad3x3_planes_blocks(N, H, C, K) / (((K + 127) / 128) * (C / 32));
  if (slices == 0) return PairPlan{};
  static thread_local KeptPerShape<PairPlan> kept;
  return kept.get({N, H, H, C, K, 3, 3, 1, 1}, slices, [&] { return plan_for(N, H, C, K, slices); });
}

size_t finish_words(const PairPlan& p) { return static_cast<size_t>(kFinishSlot0) + slot_words(p.work.nblocks); }

}  // namespace

size_t conv_pair_words(int N, int H, int C, int K) {
  const PairPlan p = pair_plan(N, H, C, K);
  if (p.nx == 0) return 0;
  return conv3x3_halo_sync_words(p.nx * p.ny) + finish_words(p) + static_cast<size_t>(wgrad3x3_planes_blocks(N, H, C, K)) + 1;
}
// Least squares over 420 layers of 64 to 512 channels, 2 to 300 images of 8 x 8 to 32 x 32, in replayed graphs: 7% rms.
double conv_pair_us(int N, int H, int C, int K, double dgrad_us) {
  int bands = 0;
  if (wgrad3x3_planes_blocks(N, H, C, K, &bands) == 0) return 0.0;
  return 9.5 + 1.85 * bands + 0.2e-6 * static_cast<double>(wgrad3x3_workspace(N, H, C, K)) + 0.85 * dgrad_us;
}
size_t conv_pair_workspace(int N, int H, int C, int K) { return pair_plan(N, H, C, K).nx == 0 ? 0 : wgrad3x3_workspace(N, H, C, K); }

int launch_conv_pair(const int8_t* err, const int8_t* act, int8_t* w, int8_t* dx, int N, int H, int C, int K, bool roundtrip, uint32_t* sync,
                     const RequantSpec& rq, const RequantSpec& grad, int8_t* g8, int8_t* wprep, void* workspace, hipStream_t stream) {
  const PairPlan p = pair_plan(N, H, C, K);
  if (p.nx == 0) return fail(NITI_ERR_UNSUPPORTED, "conv_backward_pair: shape not covered");
  HaloArgs a;
  int st = halo_requant_args(a, err, wprep, dx, N, H, K, C, (roundtrip ? NITI_EPI_F32_ROUNDTRIP : 0u) | NITI_CONV_FILTER_FORWARD_COPY, sync, rq);
  if (st != NITI_OK) return st;
  uint32_t* const sync_w = sync + conv3x3_halo_sync_words(p.nx * p.ny);
  FinishArgs f;
  st = launch_wgrad3x3_planes(act, err, w, N, H, C, K, roundtrip, sync_w, sync_w + finish_words(p), grad, g8, wprep, workspace, &f, stream);
  if (st != NITI_OK) return st;
  return with_geometry(H, p, [&](auto q, auto br, auto ni, auto kt, auto way) {
    constexpr int Q = decltype(q)::value, BR = decltype(br)::value, NI = decltype(ni)::value, KT = decltype(kt)::value;
    constexpr PairWay kWay = decltype(way)::value;
    constexpr size_t own = KGeom<Q, BR, NI, KT, per_cu_geometry(KT)>::LDS_BYTES;
    const size_t sums = along_lds(p.work.own), lds = kWay == kBeside ? std::max(own, sums) : own + sums;
    if constexpr (kWay == kInTurns) hipLaunchKernelGGL((pair_kernel<Q, BR, NI, KT, kWay>()), dim3(p.blocks), dim3(512), lds, stream, PairArgs{a, f, p.work}, p.nx, p.ny);
    else hipLaunchKernelGGL((pair_kernel<Q, BR, NI, KT, kWay>()), dim3(p.blocks), dim3(512), lds, stream, a, f, p.work, p.nx, p.ny);
    return check_launch("conv3x3_k64_backward");
  });
}

}  // namespace niti
