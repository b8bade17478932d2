// int8 products of matrices with any extents and alignment, in any of the four operand layouts, as one launch: int32
// results (the drop-in int8_mm, niti_gemm_i8), results rounded to int8 across the tensor-wide range, or rounded and
// subtracted from the weights (TiLinear's passes, ti_torch.py:241-266).
//
// What it replaces: products outside the whole-tile kernels went through copies of both operands (transposed, rows padded to
// 16 bytes), a fill of the result, a reduction split over workgroups by atomics, a pass for the range and one for the
// rounding - up to eight launches of which none had work for the chip.  These products are small (a hidden layer on a
// batch), so a launch costs what its latency chain costs: fill the pipe, walk the reduction, exchange the range, store.
#include "gemm_any.h"

#include <stdlib.h>

#include "any_tile.h"

namespace niti {
namespace {

// kAligned: both operands' rows start on 16-byte boundaries
template <class T, bool TA, bool kAligned> using OperandA = DenseOperand<Pieces<!TA, T::BM, T::BK>, kAligned>;
template <class T, bool TB, bool kAligned> using OperandB = DenseOperand<Pieces<TB, T::BN, T::BK>, kAligned>;
template <class T, bool TA, bool TB>
constexpr int lds_bytes() { return any_lds_bytes<T, OperandA<T, TA, true>, OperandB<T, TB, true>>(); }

// tile `id` of nt x mt
template <class T, bool TA, bool TB, int MODE, bool kAligned, class ShiftOf>
__device__ __forceinline__ void gemm_any_tile(const AnyArgs& g, int id, int nt, int mt, int8_t* smem, ShiftOf shift_of) {
  // Workgroups go to the eight dies in turn, and each die has its own L2: a die takes a run of neighbouring tiles, along the
  // side on which neighbours share the lines of an operand with the reduction index slow.
  const int nb = nt * mt;
  const int tile = T::BM >= 128 ? id : (id & 7) * (nb >> 3) + min(id & 7, nb & 7) + (id >> 3);
  const int n0 = (TA ? tile / mt : tile % nt) * T::BN, m0 = (TA ? tile % mt : tile / nt) * T::BM;
  const OperandA<T, TA, kAligned> oa(g.a, TA ? g.k : g.m, TA ? g.m : g.k, m0);
  const OperandB<T, TB, kAligned> ob(g.b, TB ? g.n : g.k, TB ? g.k : g.n, n0);
  any_tile<T, OperandA<T, TA, kAligned>, OperandB<T, TB, kAligned>, MODE>(g, g.c, oa, ob, m0, n0, 0, (g.k + T::BK - 1) / T::BK, smem, shift_of);
}

template <class T, bool TA, bool TB, int MODE, bool kAligned>
__global__ __launch_bounds__(512) void gemm_any_kernel(const AnyArgs g) {
  extern __shared__ __attribute__((aligned(16))) int8_t smem[];
  gemm_any_tile<T, TA, TB, MODE, kAligned>(g, blockIdx.y * gridDim.x + blockIdx.x, gridDim.x, gridDim.y, smem,
                                           [&](uint32_t lmax, uint32_t* words, auto meanwhile) { return grid_shift<8>(g, lmax, words, words + 8, meanwhile); });
}

// TiLinear's backward pass as one launch: the first `nd` workgroups take the data gradient, the others the weight gradient and
// its update, which waits until the old weights have been read.  The two have nothing else to do with each other and each
// alone is the length of its latency chain on part of the chip: together they take little more than the longer one (100 x
// 1000 -> 300: 12.9 -> 8.5 us).
template <class TD, class TW, bool kAligned>
__global__ __launch_bounds__(512, kAligned || TW::BM < 128 ? 4 : 2) void gemm_backward_kernel(const AnyArgs d, const AnyArgs w, const int nd) {
  extern __shared__ __attribute__((aligned(16))) int8_t smem[];
  const int id = blockIdx.x;
  if (id < nd) {
    gemm_any_tile<TD, false, false, kRequant, kAligned>(d, id, (d.n + TD::BN - 1) / TD::BN, (d.m + TD::BM - 1) / TD::BM, smem,
                                                        [&](uint32_t lmax, uint32_t* words, auto meanwhile) { return grid_shift<8>(d, lmax, words, words + 8, id, nd, meanwhile); });
  } else {
    const int nw = static_cast<int>(gridDim.x) - nd;
    gemm_any_tile<TW, true, false, kUpdate, kAligned>(w, id - nd, (w.n + TW::BN - 1) / TW::BN, (w.m + TW::BM - 1) / TW::BM, smem,
                                                      [&](uint32_t lmax, uint32_t* words, auto meanwhile) { return grid_shift_behind<8>(w, d, nd, lmax, words, words + 8, id - nd, nw, meanwhile); });
  }
}

template <class T>
long long tiles_of(int m, int n) { return static_cast<long long>((m + T::BM - 1) / T::BM) * ((n + T::BN - 1) / T::BN); }

// workgroups of this kernel the device holds at once; 0: cannot be launched
template <class T, bool TA, bool TB, int MODE, bool kAligned>
int resident() {
  static int of[kDeviceSlots] = {};
  int& r = of[device_slot()];
  if (r == 0) {
    auto k = gemm_any_kernel<T, TA, TB, MODE, kAligned>;
    constexpr int lds = lds_bytes<T, TA, TB>();
    int dev = 0, cus = 0, per_cu = 0;
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess ||
        hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(k), 512, lds) != hipSuccess)
      return 0;
    r = cus * per_cu;
  }
  return r;
}

template <class T, bool TA, bool TB, int MODE, bool kAligned>
int launch_as(const AnyArgs& a, hipStream_t s) {
  if (resident<T, TA, TB, MODE, kAligned>() == 0) return fail(NITI_ERR_LAUNCH, "gemm_any: cannot reserve %d bytes of LDS", lds_bytes<T, TA, TB>());
  const dim3 grid((a.n + T::BN - 1) / T::BN, (a.m + T::BM - 1) / T::BM);
  hipLaunchKernelGGL((gemm_any_kernel<T, TA, TB, MODE, kAligned>), grid, dim3(512), static_cast<size_t>(lds_bytes<T, TA, TB>()), s, a);
  return check_launch("gemm_any");
}

int pinned_tile() {   // NITI_ANY_TILE = 0 .. 2 pins the tile (tests, measurements)
  const char* e = getenv("NITI_ANY_TILE");
  return e != nullptr && e[0] >= '0' && e[0] <= '2' ? e[0] - '0' : -1;
}

// The largest tile that still leaves the chip busy.  A tile twice as wide reads its operands half as often from L2 and in
// longer pieces where the reduction index is slow; below these counts of workgroups the launch's length is one workgroup's
// walk along the reduction, which the small tile's eight wavefronts share.  Measured (us, 32 / 64 / 128 tile): 777 x 333 x 1000
// 6.5 / 6.5 / 12.3, 256 x 2048 x 512 4.4 / 4.1 / 6.9, 1024^3 10.1 / 6.0 / 9.6, 2048^3 54 / 26 / 19; both operands slow
// (weight gradients: a short reduction, many results) 300 x 1000 x 100 7.8 / 7.1 / 10.5.
template <bool TA, bool TB>
int pick_tile(int m, int n) {
  const int pin = pinned_tile();
  if (pin >= 0) return pin;
  if (tiles_of<TileL>(m, n) >= 160) return 2;
  if (tiles_of<TileM>(m, n) >= (TA && !TB ? 64 : 100)) return 1;
  return 0;
}

template <bool TA, bool TB>
bool aligned_rows(const AnyArgs& a) {
  return aligned16(a.a) && aligned16(a.b) && (TA ? a.m : a.k) % 16 == 0 && (TB ? a.k : a.n) % 16 == 0;
}

template <class T, bool TA, bool TB, int MODE>
int launch(const AnyArgs& a, hipStream_t s) {
  return aligned_rows<TA, TB>(a) ? launch_as<T, TA, TB, MODE, true>(a, s) : launch_as<T, TA, TB, MODE, false>(a, s);
}

template <bool TA, bool TB>
int launch_i32(const AnyArgs& a, hipStream_t s) {
  switch (pick_tile<TA, TB>(a.m, a.n)) {
    case 0: return launch<TileS, TA, TB, kInt32>(a, s);
    case 1: return launch<TileM, TA, TB, kInt32>(a, s);
    default: return launch<TileL, TA, TB, kInt32>(a, s);
  }
}

// whether a launch that rounds can use the tile: all its workgroups must be resident, whatever the alignment
template <class T, bool TA, bool TB, int MODE>
bool fits(int m, int n) {
  const long long nb = tiles_of<T>(m, n);
  return nb <= kMaxSlots && nb <= resident<T, TA, TB, MODE, true>() && nb <= resident<T, TA, TB, MODE, false>();
}
template <bool TA, bool TB, int MODE>
int pick_resident(int m, int n) {   // -1: none
  const int pin = pinned_tile();
  for (int t = pin >= 0 ? pin : pick_tile<TA, TB>(m, n); t <= 2; ++t) {
    if (t == 0 ? fits<TileS, TA, TB, MODE>(m, n) : t == 1 ? fits<TileM, TA, TB, MODE>(m, n) : fits<TileL, TA, TB, MODE>(m, n)) return t;
    if (pin >= 0) break;
  }
  return -1;
}

template <bool TA, bool TB, int MODE>
int launch_round(const AnyArgs& a, hipStream_t s) {
  switch (pick_resident<TA, TB, MODE>(a.m, a.n)) {
    case 0: return launch<TileS, TA, TB, MODE>(a, s);
    case 1: return launch<TileM, TA, TB, MODE>(a, s);
    case 2: return launch<TileL, TA, TB, MODE>(a, s);
    default: return fail(NITI_ERR_UNSUPPORTED, "gemm_any: the workgroups of a %d x %d result do not fit on the device at once", a.m, a.n);
  }
}

// ---- data gradient and weight update together
template <class TD, class TW>
constexpr int backward_lds() { return lds_bytes<TD, false, false>() > lds_bytes<TW, true, false>() ? lds_bytes<TD, false, false>() : lds_bytes<TW, true, false>(); }

// workgroups of the variant the device holds at once
template <class TD, class TW, bool kAligned>
int backward_resident() {
  static int of[kDeviceSlots] = {};
  int& r = of[device_slot()];
  if (r == 0) {
    auto k = gemm_backward_kernel<TD, TW, kAligned>;
    int dev = 0, cus = 0, per_cu = 0;
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, backward_lds<TD, TW>()) != hipSuccess ||
        hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(k), 512, backward_lds<TD, TW>()) != hipSuccess)
      return 0;
    r = cus * per_cu;
  }
  return r;
}

// calls f(data gradient's tile, weight gradient's tile) with the pair of tiles
template <class F>
auto with_tiles(int td, int tw, F f) {
  if (td == 0) return tw == 0 ? f(TileS{}, TileS{}) : tw == 1 ? f(TileS{}, TileM{}) : f(TileS{}, TileL{});
  return tw == 0 ? f(TileM{}, TileS{}) : tw == 1 ? f(TileM{}, TileM{}) : f(TileM{}, TileL{});
}

struct BackwardPlan {
  int td, tw;         // tiles
  long long nd, nw;   // workgroups, nd 0: not together
};
BackwardPlan plan_backward(int m, int o, int f) {
  BackwardPlan p{pick_tile<false, false>(m, f), pick_tile<true, false>(o, f), 0, 0};
  if (p.td > 1) return p;    // a data gradient that fills the chip on its own
  with_tiles(p.td, p.tw, [&](auto d, auto w) {
    using TD = decltype(d);
    using TW = decltype(w);
    const long long nd = tiles_of<TD>(m, f), nw = tiles_of<TW>(o, f);
    const int fit = o % 16 == 0 && f % 16 == 0 ? backward_resident<TD, TW, true>() : backward_resident<TD, TW, false>();
    if (nd > kMaxSlots || nw > kMaxSlots || nd + nw > fit) return 0;
    p.nd = nd;
    p.nw = nw;
    return 0;
  });
  return p;
}

}  // namespace

bool gemm_any_backward_blocks(int m, int o, int f, int* nd, int* nw) {
  if (!gemm_any_shape(m, f, o) || !gemm_any_shape(o, f, m)) return false;
  const BackwardPlan p = plan_backward(m, o, f);
  *nd = static_cast<int>(p.nd);
  *nw = static_cast<int>(p.nw);
  return p.nd != 0;
}

int launch_gemm_any_backward(const AnyArgs& d, const AnyArgs& w, hipStream_t stream) {
  const BackwardPlan p = plan_backward(d.m, d.k, d.n);
  if (p.nd == 0) return fail(NITI_ERR_UNSUPPORTED, "gemm_any: the workgroups of both gradients do not fit on the device at once");
  const bool aligned = aligned_rows<false, false>(d) && aligned_rows<true, false>(w);
  const int nd = static_cast<int>(p.nd);
  if (!aligned && d.k % 16 == 0 && d.n % 16 == 0) {   // planned with the rows' extents alone: pointers off 16 bytes
    const long long fit = with_tiles(p.td, p.tw, [](auto dt, auto wt) { return static_cast<long long>(backward_resident<decltype(dt), decltype(wt), false>()); });
    if (p.nd + p.nw > fit) return fail(NITI_ERR_UNSUPPORTED, "gemm_any: the workgroups of both gradients do not fit on the device at once");
  }
  return with_tiles(p.td, p.tw, [&](auto dt, auto wt) {
    using TD = decltype(dt);
    using TW = decltype(wt);
    const dim3 grid(static_cast<unsigned>(p.nd + p.nw));
    constexpr size_t lds = backward_lds<TD, TW>();
    if (aligned) hipLaunchKernelGGL((gemm_backward_kernel<TD, TW, true>), grid, dim3(512), lds, stream, d, w, nd);
    else hipLaunchKernelGGL((gemm_backward_kernel<TD, TW, false>), grid, dim3(512), lds, stream, d, w, nd);
    return check_launch("gemm_backward");
  });
}

bool gemm_any_large(int m, int n) { return tiles_of<TileL>(m, n) >= 160; }

bool gemm_any_shape(int m, int n, int k) {
  if (m <= 0 || n <= 0 || k <= 0) return false;
  const long long mk = static_cast<long long>(m) * (k + 512LL), nk = static_cast<long long>(n) * (k + 512LL);   // the last chunk's rows counted whole
  return mk < kOutside && nk < kOutside && (m + 31) / 32 <= 65535;
}

int launch_gemm_any(int trans_a, int trans_b, const AnyArgs& a, hipStream_t stream) {
  if (trans_a != 0) return trans_b != 0 ? launch_i32<true, true>(a, stream) : launch_i32<true, false>(a, stream);
  return trans_b != 0 ? launch_i32<false, true>(a, stream) : launch_i32<false, false>(a, stream);
}

long long gemm_any_round_blocks(AnyRound what, int m, int n, int k) {
  if (!gemm_any_shape(m, n, k)) return 0;
  const int t = what == kAnyForward ? pick_resident<false, true, kRequant>(m, n)
                : what == kAnyDgrad ? pick_resident<false, false, kRequant>(m, n)
                                    : pick_resident<true, false, kUpdate>(m, n);
  switch (t) {
    case 0: return tiles_of<TileS>(m, n);
    case 1: return tiles_of<TileM>(m, n);
    case 2: return tiles_of<TileL>(m, n);
    default: return 0;
  }
}

int launch_gemm_any_round(AnyRound what, const AnyArgs& a, hipStream_t stream) {
  switch (what) {
    case kAnyForward: return launch_round<false, true, kRequant>(a, stream);
    case kAnyDgrad: return launch_round<false, false, kRequant>(a, stream);
    default: return launch_round<true, false, kUpdate>(a, stream);
  }
}

}  // namespace niti
