// int8 convolutions outside the 3x3 kernels' square maps (any map, filter, stride and padding; channels a multiple of 16), and
// their data and weight gradients, as products whose operands are read in place (ti_torch.py:374-440).
//
// What it replaces: the filter was flipped and transposed for the data gradient, activations and errors were transposed to
// put the batch next to each other for the weight gradient, whose reduction was then split over workgroups by atomics into a
// cleared buffer, and rounding was a pass of its own - 14 launches and 130 us for the three passes of a layer with 2 GOP
// each.  Here a pass is one product on the tile of any_tile.h, whose operands find their pieces as follows:
//   forward        pixels x filters, over (r, s, c): the pixels' pieces come from the map at (p stride - pad + r, q stride - pad + s),
//                  zero outside it (a piece of 16 channels lies in one tap); the filters are rows as stored
//   data gradient  pixels x channels, over (r, s, k): the same with the error map; step (r, s, k) of the filters is row
//                  [k][R-1-r][S-1-s] of w, in which the channels are side by side: reduction index slow
//   weight gradient filters x (r, s, c), over the pixels: both operands have the reduction index slow; the activations' piece
//                  is fixed in (r, s, c) and moves over the map
// Divisions by the extents are multiplications by reciprocals that the host prepares.
#include "conv_any.h"

#include <stdlib.h>
#include <string.h>

#include "conv_operands.h"

namespace niti {
namespace {

template <class T, ConvPass PASS, int MODE>
__global__ __launch_bounds__(512) void conv_any_kernel(const ConvAnyArgs a) {
  extern __shared__ __attribute__((aligned(16))) int8_t smem[];
  conv_any_tile<T, PASS, MODE>(a, (blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x, gridDim.x, gridDim.y, gridDim.z, smem,
                               [&](uint32_t lmax, uint32_t* words, auto meanwhile) { return grid_shift<8>(a.g, lmax, words, words + 8, meanwhile); });
}

// workgroups of this kernel the device holds at once; 0: cannot be launched
template <class T, ConvPass PASS, int MODE>
int resident() {
  static int of[kDeviceSlots] = {};
  int& r = of[device_slot()];
  if (r == 0) {
    auto k = conv_any_kernel<T, PASS, MODE>;
    constexpr int lds = lds_bytes<T, PASS>();
    int dev = 0, cus = 0, per_cu = 0;
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess ||
        hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(k), 512, lds) != hipSuccess)
      return 0;
    r = cus * per_cu;
  }
  return r;
}

template <class T, ConvPass PASS, int MODE>
int launch(const ConvAnyArgs& a, int slices, hipStream_t s) {
  if (resident<T, PASS, MODE>() == 0) return fail(NITI_ERR_LAUNCH, "conv_any: cannot reserve %d bytes of LDS", lds_bytes<T, PASS>());
  const dim3 grid((a.g.n + T::BN - 1) / T::BN, (a.g.m + T::BM - 1) / T::BM, slices);
  hipLaunchKernelGGL((conv_any_kernel<T, PASS, MODE>), grid, dim3(512), static_cast<size_t>(lds_bytes<T, PASS>()), s, a);
  return check_launch("conv_any");
}

int pinned_tile() {   // NITI_ANY_TILE = 0 .. 3 pins the tile (tests, measurements)
  const char* e = getenv("NITI_ANY_TILE");
  return e != nullptr && e[0] >= '0' && e[0] <= '3' ? e[0] - '0' : -1;
}

// Forward and data gradient: the widest tile that still gives the chip enough workgroups - a tile twice as wide reads less
// from LDS per product, and few workgroups walk the reduction one after the other.  Measured (us, 32 x 32 / 64 x 64 / 128 x 64 /
// 128 x 128; 64 x 64 tiles in brackets): [66] 5.1 / 5.9 / 8.0 / 11.4, [175] 5.8 / 4.1 / 4.8 / 6.4, [636] 20.7 / 13.3 / 13.6 / 19.5,
// [1014] 18.0 / 9.9 / 8.8 / 11.5, [3050] 64 / 28 / 25 / 35 (64 filters: half of a 128-wide tile idle), [6272] 202 / 119 / 103 / 90.
int pick_tile(int m, int n) {
  const int pin = pinned_tile();
  if (pin >= 0) return pin;
  const long long large = tiles_of<TileL>(m, n), high = tiles_of<TileH>(m, n);
  if (large >= 1024 && 20 * large <= 11 * high) return 3;
  if (high >= 450) return 2;
  return tiles_of<TileM>(m, n) >= 100 ? 1 : 0;
}

template <ConvPass PASS, int MODE>
int launch_tile(int tile, const ConvAnyArgs& a, int slices, hipStream_t s) {
  switch (tile) {
    case 0: return launch<TileS, PASS, MODE>(a, slices, s);
    case 1: return launch<TileM, PASS, MODE>(a, slices, s);
    case 2: return launch<TileH, PASS, MODE>(a, slices, s);
    default: return launch<TileL, PASS, MODE>(a, slices, s);
  }
}
long long tiles_with(int tile, int m, int n) {
  return tile == 0 ? tiles_of<TileS>(m, n) : tile == 1 ? tiles_of<TileM>(m, n) : tile == 2 ? tiles_of<TileH>(m, n) : tiles_of<TileL>(m, n);
}
template <ConvPass PASS, int MODE>
int resident_with(int tile) {
  return tile == 0 ? resident<TileS, PASS, MODE>() : tile == 1 ? resident<TileM, PASS, MODE>() : tile == 2 ? resident<TileH, PASS, MODE>() : resident<TileL, PASS, MODE>();
}
// the tile of a launch that rounds (all workgroups resident), -1: none
template <ConvPass PASS, int MODE>
int pick_resident(int m, int n) {
  const int pin = pinned_tile();
  for (int t = pick_tile(m, n); t <= 3; ++t) {
    const long long nb = tiles_with(t, m, n);
    if (nb <= kMaxSlots && nb <= resident_with<PASS, MODE>(t)) return t;
    if (pin >= 0) break;
  }
  return -1;
}

size_t words_for(long long blocks) { return static_cast<size_t>(kSlot0) + slot_words(static_cast<int>(blocks)); }

// ---- weight gradient: tile and slices of the reduction
struct Split {
  int tile, slices, per;   // chunks of a slice
  double us;               // estimated time
};
int chunk_of(int tile) { return tile == 0 ? TileS::BK : tile == 1 ? TileM::BK : TileL::BK; }
long long slice_of(const ConvShape& s) { return slice_stride(static_cast<long long>(s.K) * s.R * s.S * s.C); }
// The tile and the number of slices with the least estimated time.  A compute unit's time is its rounds of workgroups times
// their chunks; a tile costs its prologue and epilogue, and cutting the reduction costs the finishing launch and the partial
// sums' way through memory.  The constants are a least-squares fit (13% rms) to 46 layers, 0.1 to 23 GOP, each with every tile
// and 1 to 48 slices; the pick is within 2% of the best of them on the geometric mean.
Split estimate_split(const ConvShape& s) {
  constexpr double kTile[4] = {6.4, 7.9, 8.7, 10.3}, kChunk[4] = {0.68, 0.61, 0.47, 0.68}, kRound[4] = {0.8, 2.0, 0.0, 0.0};   // us
  constexpr double kFinish = 2.0, kMillionSums = 1.6;
  int m, n, k;
  product_of(kConvWgrad, s, &m, &n, &k);
  const int pin = pinned_tile(), cus = compute_units();
  const char* e = getenv("NITI_ANY_SLICES");   // pins the number of slices (tests, measurements)
  Split best{0, 0, 0, 0};
  for (int t = 0; t < 4; ++t) {
    if (pin >= 0 && t != pin) continue;
    const long long tiles = tiles_with(t, m, n);
    const int chunks = (k + chunk_of(t) - 1) / chunk_of(t);
    for (int round = 0; round <= 4; ++round) {   // one workgroup per tile; as many as 3/4, 1, 2, 3 times the compute units
      long long want = e != nullptr ? atoi(e) : round == 0 ? 1 : (round == 1 ? cus * 3 / 4 : cus * (round - 1)) / tiles;
      if (want < 1 || (want == 1 && round > 0 && e == nullptr)) continue;
      if (want > chunks) want = chunks;
      const int per = static_cast<int>((chunks + want - 1) / want), slices = (chunks + per - 1) / per;
      const double blocks = static_cast<double>(tiles) * slices;
      const double rounds = blocks > 2 * cus ? blocks / cus : blocks > cus ? 2 : 1;
      double us = kTile[t] + rounds * per * kChunk[t] + (rounds - 1) * kRound[t];
      if (slices > 1 || blocks > 2 * cus) us += kFinish + kMillionSums * 1e-6 * slices * static_cast<double>(m) * n;
      if (best.slices == 0 || us < best.us) best = Split{t, slices, per, us};
    }
  }
  return best;
}

// the pick for a shape is asked for several times per call: each thread keeps the last few
Split pick_split(const ConvShape& s) {
  if (getenv("NITI_ANY_TILE") != nullptr || getenv("NITI_ANY_SLICES") != nullptr) return estimate_split(s);
  struct Entry {
    int key[7];
    Split split;
  };
  static thread_local Entry kept[16] = {};
  const int key[7] = {s.N, s.H * 65536 + s.W, s.C, s.K, s.R * 65536 + s.S, s.pad, device_slot()};
  unsigned h = 0;
  for (int v : key) h = h * 31u + static_cast<unsigned>(v);
  Entry& e = kept[(h ^ (h >> 8)) & 15u];
  if (memcmp(e.key, key, sizeof(key)) != 0) {
    memcpy(e.key, key, sizeof(key));
    e.split = estimate_split(s);
  }
  return e.split;
}

}  // namespace

bool conv_any_shape(ConvPass pass, const ConvShape& s) {
  if (s.N <= 0 || s.H <= 0 || s.W <= 0 || s.C <= 0 || s.K <= 0 || s.R <= 0 || s.S <= 0 || s.stride <= 0 || s.pad < 0) return false;
  if (s.H + 2 * s.pad < s.R || s.W + 2 * s.pad < s.S || s.C % 16 != 0) return false;
  if (pass != kConvForward && (s.stride != 1 || s.K % 16 != 0)) return false;
  if (pass == kConvDgrad && (s.R != s.S || s.pad > s.R - 1)) return false;
  const long long limit = kOutside - (1LL << 26);
  const long long in = static_cast<long long>(s.N) * s.H * s.W, out = static_cast<long long>(s.N) * s.P() * s.Q();
  const long long taps = static_cast<long long>(s.R) * s.S;
  if (s.H > 32768 || s.W > 32768 || s.R > 32768 || s.S > 32768 || s.pad > 32768 || s.stride > 32768) return false;
  if (in + 1024 > limit / s.C || out + 1024 > limit / s.K || taps > (1 << 24) / (s.C > s.K ? s.C : s.K)) return false;
  if (static_cast<long long>(s.K) * taps * s.C > limit) return false;
  return (out + 31) / 32 <= 65535 && (in + 31) / 32 <= 65535;
}

int launch_conv_any(ConvPass pass, const ConvShape& s, const int8_t* x, const int8_t* w, int32_t* y, bool roundtrip, uint32_t* absmax, hipStream_t stream) {
  ConvAnyArgs a = args_of(pass, s, x, w, roundtrip);
  a.g.c = y;
  a.g.absmax = absmax;
  const int t = pick_tile(a.g.m, a.g.n);
  return pass == kConvForward ? launch_tile<kConvForward, kInt32>(t, a, 1, stream) : launch_tile<kConvDgrad, kInt32>(t, a, 1, stream);
}

static int requant_tile(ConvPass pass, const ConvShape& s) {
  int m, n, k;
  product_of(pass, s, &m, &n, &k);
  return pass == kConvForward ? pick_resident<kConvForward, kRequant>(m, n) : pick_resident<kConvDgrad, kRequant>(m, n);
}

size_t conv_any_requant_words(ConvPass pass, const ConvShape& s) {
  if (!conv_any_shape(pass, s)) return 0;
  const int t = requant_tile(pass, s);
  if (t < 0) return 0;
  int m, n, k;
  product_of(pass, s, &m, &n, &k);
  return words_for(tiles_with(t, m, n));
}

// The walk of a workgroup, longer the more of them there are; from one per compute unit on, units have two.  Least squares over 642
// launches of the 3 x 3 maps that requant_us (conv3x3_halo.hip) is fitted to: 5% rms, from 0.84 to 1.21 of the measured time.
double conv_any_forward_us(const ConvShape& s, size_t* words) {
  *words = 0;
  if (!conv_any_shape(kConvForward, s)) return 0.0;
  const int t = requant_tile(kConvForward, s);
  if (t < 0) return 0.0;
  int m, n, k;
  product_of(kConvForward, s, &m, &n, &k);
  *words = words_for(tiles_with(t, m, n));
  if (t > 1) return 1e9;   // the wide tiles: not for the few workgroups this is asked for
  const double chunks = t == 0 ? (k + TileS::BK - 1) / TileS::BK : (k + TileM::BK - 1) / TileM::BK;
  const double fill = static_cast<double>(tiles_with(t, m, n)) / compute_units();
  if (t == 0) return fill <= 1.0 ? 5.1 + 0.55 * chunks + 0.8 * fill : 4.9 + (0.64 + 0.35 * fill) * chunks + 0.6 * fill;
  return fill <= 1.0 ? 5.4 + 0.69 * chunks + 0.5 * fill : 6.0 + (0.44 + 0.40 * fill) * chunks + 1.2 * fill;
}

double conv_any_dgrad_us(const ConvShape& s) {
  if (conv_any_requant_words(kConvDgrad, s) == 0) return 0.0;
  constexpr double kChunk[4] = {0.58, 0.58, 0.47, 0.68};
  int m, n, k;
  product_of(kConvDgrad, s, &m, &n, &k);
  const int t = requant_tile(kConvDgrad, s), block = t == 0 ? TileS::BK : t == 1 ? TileM::BK : TileL::BK;
  return 5.5 + (tiles_with(t, m, n) > compute_units() ? 1.5 : 1.0) * kChunk[t] * ((k + block - 1) / block);
}

int launch_conv_any_requant(ConvPass pass, const ConvShape& s, const int8_t* x, const int8_t* w, int8_t* y, bool roundtrip, uint32_t* sync,
                            const RequantSpec& rq, hipStream_t stream) {
  ConvAnyArgs a = args_of(pass, s, x, w, roundtrip);
  set_rounding(a.g, rq, sync);
  a.g.out8 = y;
  if (rq.pool != nullptr) {
    a.g.pool = rq.pool;
    a.g.map_h = a.P;
    a.g.map_w = a.Q;
    a.g.by_map = a.by_pq;
    a.g.by_map_w = Reciprocal(a.Q / 2);
  }
  const int t = requant_tile(pass, s);
  if (rq.pool != nullptr && (t == 3 || pass != kConvForward || a.P % 2 != 0 || a.Q % 2 != 0 || s.K % 4 != 0))
    return fail(NITI_ERR_UNSUPPORTED, "conv_any: this launch's tiles do not fit whole pooling windows");
  if (t < 0) return fail(NITI_ERR_UNSUPPORTED, "conv_any: the workgroups of a %d x %d result do not fit on the device at once", a.g.m, a.g.n);
  return pass == kConvForward ? launch_tile<kConvForward, kRequant>(t, a, 1, stream) : launch_tile<kConvDgrad, kRequant>(t, a, 1, stream);
}

size_t conv_any_wgrad_workspace(const ConvShape& s) {
  if (!conv_any_shape(kConvWgrad, s)) return 0;
  return static_cast<size_t>(pick_split(s).slices) * slice_of(s) * sizeof(int32_t);
}

double conv_any_wgrad_us(const ConvShape& s) { return conv_any_shape(kConvWgrad, s) ? pick_split(s).us : 0.0; }

static int launch_slices(const ConvShape& s, const Split& p, const int8_t* act, const int8_t* err, void* workspace, hipStream_t stream) {
  ConvAnyArgs a = args_of(kConvWgrad, s, err, act, false);
  a.g.c = static_cast<int32_t*>(workspace);
  a.chunks_per_slice = p.per;
  a.slice = slice_of(s);
  return launch_tile<kConvWgrad, kInt32>(p.tile, a, p.slices, stream);
}

int launch_conv_any_wgrad(const ConvShape& s, const int8_t* act, const int8_t* err, int32_t* dw, bool roundtrip, uint32_t* absmax, void* workspace,
                          hipStream_t stream) {
  const Split p = pick_split(s);
  if (p.slices == 1) {
    ConvAnyArgs a = args_of(kConvWgrad, s, err, act, roundtrip);
    a.g.c = dw;
    a.g.absmax = absmax;
    a.chunks_per_slice = p.per;
    return launch_tile<kConvWgrad, kInt32>(p.tile, a, 1, stream);
  }
  const int st = launch_slices(s, p, act, err, workspace, stream);
  if (st != NITI_OK) return st;
  return launch_wgrad_reduce(static_cast<const int32_t*>(workspace), slice_of(s), p.slices, dw, static_cast<int64_t>(s.K) * s.R * s.S * s.C, roundtrip, absmax,
                             stream);
}

size_t conv_any_wgrad_update_words(const ConvShape& s) {
  if (!conv_any_shape(kConvWgrad, s)) return 0;
  const Split p = pick_split(s);
  int m, n, k;
  product_of(kConvWgrad, s, &m, &n, &k);
  const long long nb = tiles_with(p.tile, m, n);
  const long long finish = wgrad_finish_blocks(static_cast<long long>(m) * n);
  if (finish == 0) return 0;   // also where nothing is split: padded channels or a wanted int32 gradient take the finishing launch
  return words_for(nb > finish && nb <= kMaxSlots ? nb : finish);
}

int launch_conv_any_wgrad_update(const ConvShape& s, const int8_t* act, const int8_t* err, int8_t* w, int w_channels, bool roundtrip, uint32_t* sync,
                                 const RequantSpec& rq, int8_t* g8, int32_t* dw, int8_t* wprep, void* workspace, hipStream_t stream) {
  const Split p = pick_split(s);
  int m, n, k;
  product_of(kConvWgrad, s, &m, &n, &k);
  const long long nb = tiles_with(p.tile, m, n);
  if (p.slices == 1 && w_channels == s.C && dw == nullptr && nb <= kMaxSlots && nb <= resident_with<kConvWgrad, kUpdate>(p.tile)) {
    ConvAnyArgs a = args_of(kConvWgrad, s, err, act, roundtrip);
    set_rounding(a.g, rq, sync);
    a.g.w = w;
    a.g.wprep = wprep;
    a.g.channels = s.C;
    a.g.by_channels = Reciprocal(s.C);
    a.g.out8 = g8;
    a.chunks_per_slice = p.per;
    return launch_tile<kConvWgrad, kUpdate>(p.tile, a, 1, stream);
  }
  const int st = launch_slices(s, p, act, err, workspace, stream);
  if (st != NITI_OK) return st;
  return launch_wgrad_finish(static_cast<const int32_t*>(workspace), slice_of(s), p.slices, static_cast<long long>(m) * n, s.C, w, w_channels, roundtrip, sync,
                             rq, g8, dw, wprep, stream);
}

}  // namespace niti
