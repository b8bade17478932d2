// Data gradient and weight gradient of a convolution as one launch (ti_torch.py:404-437).
//
// Both read the error map and nothing of each other; on small layers each alone is one latency chain (prologue, walk along the
// reduction, exchange of the range, store) on part of the chip.  The first workgroups of this launch take the data gradient's
// tiles (with rounding, mask and where asked the max-pool's backward pass), the others the weight gradient's.  Where the
// reduction over the pixels is not cut the weights are updated in the same launch, behind the last read of the old ones; where
// it is cut the partial sums go to memory and the finishing launch of wgrad3x3.hip follows.
#include <stdlib.h>

#include "conv_operands.h"

namespace niti {
namespace {

template <class TD, class TW, int MODE>
__global__ __launch_bounds__(512, 4) void conv_backward_kernel(const ConvAnyArgs d, const ConvAnyArgs w, const int nd, const int slices) {
  extern __shared__ __attribute__((aligned(16))) int8_t smem[];
  const int id = blockIdx.x;
  if (id < nd) {
    conv_any_tile<TD, kConvDgrad, kRequant>(d, id, (d.g.n + TD::BN - 1) / TD::BN, (d.g.m + TD::BM - 1) / TD::BM, 1, smem,
                                            [&](uint32_t lmax, uint32_t* words, auto meanwhile) { return grid_shift<8>(d.g, lmax, words, words + 8, id, nd, meanwhile); });
  } else {
    const int nw = static_cast<int>(gridDim.x) - nd;
    conv_any_tile<TW, kConvWgrad, MODE>(w, id - nd, (w.g.n + TW::BN - 1) / TW::BN, (w.g.m + TW::BM - 1) / TW::BM, slices, smem,
                                        [&](uint32_t lmax, uint32_t* words, auto meanwhile) { return grid_shift_behind<8>(w.g, d.g, nd, lmax, words, words + 8, id - nd, nw, meanwhile); });
  }
}

template <class TD, class TW>
constexpr int pair_lds() { return lds_bytes<TD, kConvDgrad>() > lds_bytes<TW, kConvWgrad>() ? lds_bytes<TD, kConvDgrad>() : lds_bytes<TW, kConvWgrad>(); }

template <class TD, class TW, int MODE>
int resident() {
  static int of[kDeviceSlots] = {};
  int& r = of[device_slot()];
  if (r == 0) {
    auto k = conv_backward_kernel<TD, TW, MODE>;
    int dev = 0, cus = 0, per_cu = 0;
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, pair_lds<TD, TW>()) != hipSuccess ||
        hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(k), 512, pair_lds<TD, TW>()) != hipSuccess)
      return 0;
    r = cus * per_cu;
  }
  return r;
}

template <class F>
auto with_tile(int t, F f) {
  return t == 0 ? f(TileS{}) : t == 1 ? f(TileM{}) : t == 2 ? f(TileH{}) : f(TileL{});
}
// calls f(data gradient's tile, weight gradient's tile)
template <class F>
auto with_tiles(int td, int tw, F f) {
  return with_tile(tw, [&](auto w) { return td == 0 ? f(TileS{}, w) : td == 1 ? f(TileM{}, w) : f(TileH{}, w); });
}

struct Plan {
  int td, tw;           // tiles
  long long nd, nw;     // workgroups, nd 0: not together
  int slices, per;      // of the reduction over the pixels; chunks of a slice
  double us;            // estimated time, the finishing launch included
};

// The tiles and slices with the least estimated time among those whose workgroups are resident together.  A chunk's time as in
// conv_any.hip; the launch is as long as its longest chain or as the chip needs for all chunks, whichever is more.
Plan estimate(const ConvShape& s) {
  constexpr double kBase = 7.0, kChunkD[3] = {0.58, 0.58, 0.47}, kChunkW[4] = {0.68, 0.61, 0.47, 0.68}, kFinish = 3.5, kMillionSums = 1.6;   // us
  constexpr int kBlock[4] = {TileS::BK, TileM::BK, TileH::BK, TileL::BK};
  const char* te = getenv("NITI_ANY_TILE");
  const char* se = getenv("NITI_ANY_SLICES");
  const int pin = te != nullptr && te[0] >= '0' && te[0] <= '3' ? te[0] - '0' : -1, pin_slices = se != nullptr ? atoi(se) : 0;
  const int cus = compute_units();
  int dm, dn, dk, wm, wn, wk;
  product_of(kConvDgrad, s, &dm, &dn, &dk);
  product_of(kConvWgrad, s, &wm, &wn, &wk);
  Plan best{};
  for (int td = 0; td < 3; ++td) {
    if (pin >= 0 && td != (pin < 3 ? pin : 2)) continue;
    const long long nd = with_tile(td, [&](auto t) { return tiles_of<decltype(t)>(dm, dn); });
    const int cd = (dk + kBlock[td] - 1) / kBlock[td];
    if (nd > 2 * cus) continue;
    for (int tw = 0; tw < 4; ++tw) {
      if (pin >= 0 && tw != pin) continue;
      const long long tiles = with_tile(tw, [&](auto t) { return tiles_of<decltype(t)>(wm, wn); });
      const int cw = (wk + kBlock[tw] - 1) / kBlock[tw];
      for (int round = 0; round < 4; ++round) {   // whole; as many workgroups as the data gradient leaves of 1, 1.5, 2 per compute unit
        long long want = pin_slices > 0 ? pin_slices : round == 0 ? 1 : (cus / 2 * (round + 1) - nd) / tiles;
        if (want < 1 || (want == 1 && round > 0 && pin_slices == 0)) continue;
        if (want > cw) want = cw;
        const int per = static_cast<int>((cw + want - 1) / want), slices = (cw + per - 1) / per;
        const long long nw = tiles * slices;
        if (nd + nw > 2 * cus || (slices > 1 && wgrad_finish_blocks(static_cast<long long>(wm) * wn) == 0)) continue;
        const double chain_d = cd * kChunkD[td], chain_w = per * kChunkW[tw], all = (nd * chain_d + nw * chain_w) / cus;
        double us = kBase + (chain_d > chain_w ? (chain_d > all ? chain_d : all) : (chain_w > all ? chain_w : all));
        if (slices > 1) us += kFinish + kMillionSums * 1e-6 * slices * static_cast<double>(wm) * wn;
        if (best.nd != 0 && us >= best.us) continue;
        const int fit = with_tiles(td, tw, [&](auto d, auto w) {
          return slices > 1 ? resident<decltype(d), decltype(w), kInt32>() : resident<decltype(d), decltype(w), kUpdate>();
        });
        if (nd + nw <= fit) best = Plan{td, tw, nd, nw, slices, per, us};
      }
    }
  }
  return best;
}

Plan plan_of(const ConvShape& s) {
  if (!conv_any_shape(kConvDgrad, s) || !conv_any_shape(kConvWgrad, s)) return Plan{};
  if (getenv("NITI_ANY_TILE") != nullptr || getenv("NITI_ANY_SLICES") != nullptr) return estimate(s);
  static thread_local KeptPerShape<Plan> kept;
  return kept.get(s, 0, [&] { return estimate(s); });
}

size_t words_of(const ConvShape& s, const Plan& p) {
  const long long second = p.slices > 1 ? wgrad_finish_blocks(static_cast<long long>(s.K) * s.R * s.S * s.C) : p.nw;
  return 2 * static_cast<size_t>(kSlot0) + slot_words(static_cast<int>(p.nd)) + slot_words(static_cast<int>(second));
}
long long slice_of(const ConvShape& s) { return slice_stride(static_cast<long long>(s.K) * s.R * s.S * s.C); }

}  // namespace

double conv_backward_us(const ConvShape& s) { return plan_of(s).us; }

size_t conv_backward_words(const ConvShape& s) {
  const Plan p = plan_of(s);
  return p.nd == 0 ? 0 : words_of(s, p);
}

size_t conv_backward_workspace(const ConvShape& s) {
  const Plan p = plan_of(s);
  return p.slices > 1 ? static_cast<size_t>(p.slices) * slice_of(s) * sizeof(int32_t) : 0;
}

int launch_conv_backward(const ConvShape& s, const int8_t* err, const int8_t* act, int8_t* w, int8_t* dx, bool roundtrip, uint32_t* sync, const RequantSpec& rq,
                         const RequantSpec& grad, int8_t* g8, int8_t* wprep, void* workspace, hipStream_t stream) {
  const Plan p = plan_of(s);
  if (p.nd == 0) return fail(NITI_ERR_UNSUPPORTED, "conv_backward: the workgroups of both gradients do not fit on the device at once");
  ConvAnyArgs d = args_of(kConvDgrad, s, err, w, roundtrip);
  set_rounding(d.g, rq, sync);
  d.g.out8 = dx;
  if (rq.unpool != nullptr) {
    d.g.pool_x = rq.pool_x;
    d.g.unpool = rq.unpool;
    d.g.ties_all = rq.ties_all;
    d.g.map_h = s.H;
    d.g.map_w = s.W;
    d.g.by_map = Reciprocal(s.H * s.W);
    d.g.by_map_w = Reciprocal(s.W);
  }
  uint32_t* const sync_w = sync + kSlot0 + slot_words(static_cast<int>(p.nd));
  ConvAnyArgs g = args_of(kConvWgrad, s, err, act, p.slices == 1 && roundtrip);
  g.chunks_per_slice = p.per;
  if (p.slices > 1) {
    g.g.c = static_cast<int32_t*>(workspace);
    g.slice = slice_of(s);
  } else {
    set_rounding(g.g, grad, sync_w);
    g.g.w = w;
    g.g.out8 = g8;
    g.g.wprep = wprep;
    g.g.channels = s.C;
    g.g.by_channels = Reciprocal(s.C);
  }
  const int st = with_tiles(p.td, p.tw, [&](auto dt, auto wt) {
    using TD = decltype(dt);
    using TW = decltype(wt);
    const dim3 grid(static_cast<unsigned>(p.nd + p.nw));
    constexpr size_t lds = pair_lds<TD, TW>();
    const int nd = static_cast<int>(p.nd);
    if (p.slices > 1) hipLaunchKernelGGL((conv_backward_kernel<TD, TW, kInt32>), grid, dim3(512), lds, stream, d, g, nd, p.slices);
    else hipLaunchKernelGGL((conv_backward_kernel<TD, TW, kUpdate>), grid, dim3(512), lds, stream, d, g, nd, 1);
    return check_launch("conv_backward");
  });
  if (st != NITI_OK || p.slices == 1) return st;
  RequantSpec behind = grad;
  behind.exp_a = rq.exp_out;
  return launch_wgrad_finish(static_cast<const int32_t*>(workspace), slice_of(s), p.slices, static_cast<long long>(s.K) * s.R * s.S * s.C, s.C, w, s.C, roundtrip,
                             sync_w, behind, g8, nullptr, wprep, stream, sync);
}

}  // namespace niti
