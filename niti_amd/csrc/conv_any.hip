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

#include "any_tile.h"

namespace niti {
namespace {

struct ConvAnyArgs {
  AnyArgs g;
  int N, H, W, C;          // the map whose taps are taken
  int R, S, stride, pad, P, Q;
  int pixels, filters;     // N P Q; data gradient: rows of w
  long long map_bytes, w_bytes;
  Reciprocal by_pq, by_q, by_c, by_s;
  int chunks_per_slice;    // weight gradient: the reduction is cut into gridDim.z slices ...
  long long slice;         // ... whose int32 sums lie this far apart
};

__device__ inline v4i load_piece(__amdgpu_buffer_rsrc_t rsrc, int off) {
  return __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc, off, 0, 0));
}
struct Piece {
  v4i v;
};

// Positions move on by a chunk at a time: steps with carries, no divisions (with the divisions, 7 quarter-rate multiplications
// per piece, the address arithmetic of a weight gradient took longer than its products: 64 x 64 tiles 0.65 us per 256 pixels).

// rows: output pixels; reduction: (r, s, c), c fastest
template <class G_>
struct PixelRows {
  using G = G_;
  using Raw = Piece;
  const ConvAnyArgs& a;
  __amdgpu_buffer_rsrc_t rsrc;
  int h[G::N], w[G::N], at[G::N];   // tap (0, 0) of the pixel
  int r, s, ch;                     // this thread's tap and channel in the next chunk ...
  int delta;                        // ... and their distance from tap (0, 0)
  int dr, ds, dch;                  // a chunk's length in the same terms
  __device__ PixelRows(const ConvAnyArgs& args, int first) : a(args) {
    rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(a.g.a), 0, static_cast<int>(a.map_bytes), 0x00020000);
#pragma unroll
    for (int i = 0; i < G::N; ++i) {
      const int m = first + G::row(i);
      const int n = a.by_pq.of(m), pq = m - n * (a.P * a.Q);
      const int p = a.by_q.of(pq), q = pq - p * a.Q;
      h[i] = m < a.pixels ? p * a.stride - a.pad : -0x20000000;   // no tap of it is inside
      w[i] = q * a.stride - a.pad;
      at[i] = ((n * a.H + p * a.stride - a.pad) * a.W + w[i]) * a.C;
    }
    const int tap = a.by_c.of(G::col());
    r = a.by_s.of(tap);
    s = tap - r * a.S;
    ch = G::col() - tap * a.C;
    delta = (r * a.W + s) * a.C + ch;
    const int taps = a.by_c.of(G::BK);
    dr = a.by_s.of(taps);
    ds = taps - dr * a.S;
    dch = G::BK - taps * a.C;
  }
  __device__ void load(int, Raw (&raw)[G::N]) {
    const int rr = r < a.R ? r : 0x40000000;                      // behind the reduction's end: outside for every pixel
#pragma unroll
    for (int i = 0; i < G::N; ++i) {
      const bool in = static_cast<unsigned>(h[i] + rr) < static_cast<unsigned>(a.H) && static_cast<unsigned>(w[i] + s) < static_cast<unsigned>(a.W);
      raw[i].v = load_piece(rsrc, in ? at[i] + delta : kOutside);
    }
    ch += dch;
    s += ds;
    r += dr;
    delta += (dr * a.W + ds) * a.C + dch;
    if (ch >= a.C) {       // the next tap is the next pixel: delta points there
      ch -= a.C;
      ++s;
    }
    if (s >= a.S) {        // the next row of taps
      s -= a.S;
      ++r;
      delta += (a.W - a.S) * a.C;
    }
  }
  __device__ v4i piece(const Raw& r, int, int, bool) const { return r.v; }
};

// reduction: (r, s, k) of the data gradient, k fastest; columns: channels
template <class G_>
struct FlippedFilter {
  using G = G_;
  using Raw = Piece;
  const ConvAnyArgs& a;
  __amdgpu_buffer_rsrc_t rsrc;
  int k[G::N], at[G::N];   // filter and byte offset of the pieces in the next chunk
  int left[G::N];          // steps of the reduction from there on
  int dk, step, carry;
  __device__ FlippedFilter(const ConvAnyArgs& args, int first) : a(args) {
    rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(a.g.b), 0, static_cast<int>(a.w_bytes), 0x00020000);
    const int line = a.R * a.S * a.g.n;                           // bytes of a filter
#pragma unroll
    for (int i = 0; i < G::N; ++i) {
      const int tap = a.by_c.of(G::row(i));
      k[i] = G::row(i) - tap * a.C;
      at[i] = k[i] * line + (a.R * a.S - 1 - tap) * a.g.n + first + G::col();
      left[i] = a.g.k - G::row(i);
    }
    const int taps = a.by_c.of(G::BK);
    dk = G::BK - taps * a.C;
    step = dk * line - taps * a.g.n;
    carry = -a.C * line - a.g.n;
  }
  __device__ void load(int, Raw (&raw)[G::N]) {
#pragma unroll
    for (int i = 0; i < G::N; ++i) {
      raw[i].v = load_piece(rsrc, left[i] > 0 ? at[i] : kOutside);
      left[i] -= G::BK;
      k[i] += dk;
      const bool over = k[i] >= a.C;
      k[i] -= over ? a.C : 0;
      at[i] += step + (over ? carry : 0);
    }
  }
  __device__ v4i piece(const Raw& r, int, int, bool) const { return r.v; }
};

// reduction: output pixels; columns: (r, s, c)
template <class G_>
struct TapColumns {
  using G = G_;
  using Raw = Piece;
  const ConvAnyArgs& a;
  __amdgpu_buffer_rsrc_t rsrc;
  int r, s;                              // this thread's tap relative to the pixel
  int p[G::N], q[G::N], at[G::N];        // pixel of the pieces in the next chunk, offset of the tap there (pixels behind the last
                                         // image: behind the map)
  int dp, dq, step, next_row, next_image;
  __device__ TapColumns(const ConvAnyArgs& args, int first, int chunk) : a(args) {
    rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(a.g.b), 0, static_cast<int>(a.map_bytes), 0x00020000);
    const int col = first + G::col();
    const int tap = a.by_c.of(col);
    r = a.by_s.of(tap) - a.pad;
    s = tap - a.by_s.of(tap) * a.S - a.pad;
    const int c = col - tap * a.C;
#pragma unroll
    for (int i = 0; i < G::N; ++i) {
      const int m = chunk * G::BK + G::row(i);
      const int n = a.by_pq.of(m), pq = m - n * (a.P * a.Q);
      p[i] = a.by_q.of(pq);
      q[i] = pq - p[i] * a.Q;
      at[i] = ((n * a.H + p[i] + r) * a.W + q[i] + s) * a.C + c;
    }
    const int dn = a.by_pq.of(G::BK), rest = G::BK - dn * (a.P * a.Q);
    dp = a.by_q.of(rest);
    dq = rest - dp * a.Q;
    step = ((dn * a.H + dp) * a.W + dq) * a.C;
    next_row = (a.W - a.Q) * a.C;
    next_image = (a.H - a.P) * a.W * a.C;
  }
  __device__ void load(int, Raw (&raw)[G::N]) {
#pragma unroll
    for (int i = 0; i < G::N; ++i) {
      const bool in = static_cast<unsigned>(p[i] + r) < static_cast<unsigned>(a.H) && static_cast<unsigned>(q[i] + s) < static_cast<unsigned>(a.W);
      raw[i].v = load_piece(rsrc, in ? at[i] : kOutside);
      q[i] += dq;
      const bool row = q[i] >= a.Q;
      q[i] -= row ? a.Q : 0;
      p[i] += dp + (row ? 1 : 0);
      const bool image = p[i] >= a.P;
      p[i] -= image ? a.P : 0;
      at[i] += step + (row ? next_row : 0) + (image ? next_image : 0);
    }
  }
  __device__ v4i piece(const Raw& r, int, int, bool) const { return r.v; }
};

template <class T, ConvPass PASS>
struct Operands;
template <class T>
struct Operands<T, kConvForward> {
  using A = PixelRows<Pieces<true, T::BM, T::BK>>;
  using B = DenseOperand<Pieces<true, T::BN, T::BK>, true, false>;
};
template <class T>
struct Operands<T, kConvDgrad> {
  using A = PixelRows<Pieces<true, T::BM, T::BK>>;
  using B = FlippedFilter<Pieces<false, T::BN, T::BK>>;
};
template <class T>
struct Operands<T, kConvWgrad> {
  using A = DenseOperand<Pieces<false, T::BM, T::BK>, true, false>;
  using B = TapColumns<Pieces<false, T::BN, T::BK>>;
};

template <class T, ConvPass PASS, int MODE>
__global__ __launch_bounds__(512) void conv_any_kernel(const ConvAnyArgs a) {
  extern __shared__ __attribute__((aligned(16))) int8_t smem[];
  using A = typename Operands<T, PASS>::A;
  using B = typename Operands<T, PASS>::B;
  // Workgroups go to the eight dies in turn, and each die has its own L2: a die takes a run of neighbouring tiles (they share
  // pixels), of the same slice of the reduction where it is cut.
  const int nt = gridDim.x, per = nt * gridDim.y, nb = per * gridDim.z;
  const int id = (blockIdx.z * gridDim.y + blockIdx.y) * nt + blockIdx.x;
  const int place = (id & 7) * (nb >> 3) + min(id & 7, nb & 7) + (id >> 3);
  const int slice = place / per, tile = place - slice * per;
  const int n0 = tile % nt * T::BN, m0 = tile / nt * T::BM;
  auto shift_of = [&](uint32_t lmax, uint32_t* words) { return grid_shift<8>(a.g, lmax, words, words + 8); };
  if constexpr (PASS == kConvWgrad) {
    const int first = slice * a.chunks_per_slice;
    const int chunks = min((a.g.k + T::BK - 1) / T::BK, first + a.chunks_per_slice);
    any_tile<T, A, B, MODE>(a.g, a.g.c + slice * a.slice, A(a.g.a, a.g.k, a.g.m, m0), B(a, n0, first), m0, n0, first, chunks, smem, shift_of);
  } else {
    const int chunks = (a.g.k + T::BK - 1) / T::BK;
    if constexpr (PASS == kConvForward)
      any_tile<T, A, B, MODE>(a.g, a.g.c, A(a, m0), B(a.g.b, a.g.n, a.g.k, n0), m0, n0, 0, chunks, smem, shift_of);
    else
      any_tile<T, A, B, MODE>(a.g, a.g.c, A(a, m0), B(a, n0), m0, n0, 0, chunks, smem, shift_of);
  }
}

template <class T>
long long tiles_of(int m, int n) { return static_cast<long long>((m + T::BM - 1) / T::BM) * ((n + T::BN - 1) / T::BN); }

template <class T, ConvPass PASS>
constexpr int lds_bytes() { return any_lds_bytes<T, typename Operands<T, PASS>::A, typename Operands<T, PASS>::B>(); }

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

ConvAnyArgs map_args(ConvPass pass, const ConvShape& s) {
  ConvAnyArgs a;
  const bool dg = pass == kConvDgrad;
  a.N = s.N;
  a.H = dg ? s.P() : s.H;
  a.W = dg ? s.Q() : s.W;
  a.C = dg ? s.K : s.C;
  a.R = s.R;
  a.S = s.S;
  a.stride = s.stride;
  a.pad = dg ? s.R - 1 - s.pad : s.pad;
  a.P = dg ? s.H : s.P();
  a.Q = dg ? s.W : s.Q();
  a.pixels = s.N * a.P * a.Q;
  a.filters = s.K;
  a.map_bytes = static_cast<long long>(s.N) * a.H * a.W * a.C;
  a.w_bytes = static_cast<long long>(s.K) * s.R * s.S * s.C;
  a.by_pq = Reciprocal(a.P * a.Q);
  a.by_q = Reciprocal(a.Q);
  a.by_c = Reciprocal(a.C);
  a.by_s = Reciprocal(a.S);
  a.chunks_per_slice = 0;
  a.slice = 0;
  return a;
}
// m, n, k of the pass's product
void product_of(ConvPass pass, const ConvShape& s, int* m, int* n, int* k) {
  const int pixels = s.N * s.P() * s.Q();
  *m = pass == kConvForward ? pixels : pass == kConvDgrad ? s.N * s.H * s.W : s.K;
  *n = pass == kConvForward ? s.K : pass == kConvDgrad ? s.C : s.R * s.S * s.C;
  *k = pass == kConvForward ? s.R * s.S * s.C : pass == kConvDgrad ? s.R * s.S * s.K : pixels;
}
ConvAnyArgs args_of(ConvPass pass, const ConvShape& s, const int8_t* x, const int8_t* y, bool roundtrip) {
  ConvAnyArgs a = map_args(pass, s);
  product_of(pass, s, &a.g.m, &a.g.n, &a.g.k);
  a.g.a = x;
  a.g.b = y;
  a.g.roundtrip = roundtrip ? 1 : 0;
  return a;
}
void set_rounding(AnyArgs& g, const RequantSpec& rq, uint32_t* sync) {
  g.sync = sync;
  g.target_bits = rq.target_bits;
  g.method = rq.method;
  g.trunc = rq.trunc;
  g.bw_mode = rq.bw_mode;
  g.rq_flags = rq.flags;
  g.spin_limit = rq.spin_limit;
  g.sticky = rq.sticky;
  g.shift_out = rq.shift_out;
  g.exp_a = rq.exp_a;
  g.exp_b = rq.exp_b;
  g.exp_out = rq.exp_out;
  g.mask = rq.mask;
  g.rand = rq.rand;
}
size_t words_for(long long blocks) { return static_cast<size_t>(kSlot0) + slot_words(static_cast<int>(blocks)); }

// ---- weight gradient: tile and slices of the reduction
struct Split {
  int tile, slices, per;   // chunks of a slice
  double us;               // estimated time
};
int chunk_of(int tile) { return tile == 0 ? TileS::BK : tile == 1 ? TileM::BK : TileL::BK; }
long long slice_of(const ConvShape& s) {
  const long long n = static_cast<long long>(s.K) * s.R * s.S * s.C;
  return (n + 1023) / 1024 * 1024 + 1088;   // the same element of consecutive slices in different memory channels
}
// The tile and the number of slices with the least estimated time.  A compute unit's time is its rounds of workgroups times
// their chunks; a tile costs its prologue and epilogue, and cutting the reduction costs the finishing launch and the partial
// sums' way through memory.  The constants are a least-squares fit (13% rms) to 46 layers, 0.1 to 23 GOP, each with every tile
// and 1 to 48 slices; the pick is within 2% of the best of them on the geometric mean.
Split estimate_split(const ConvShape& s) {
  constexpr double kTile[4] = {6.4, 7.9, 8.7, 10.3}, kChunk[4] = {0.68, 0.61, 0.47, 0.68}, kRound[4] = {0.8, 2.0, 0.0, 0.0};   // us
  constexpr double kFinish = 2.0, kMillionSums = 1.6;
  int m, n, k;
  product_of(kConvWgrad, s, &m, &n, &k);
  const int pin = pinned_tile();
  const char* e = getenv("NITI_ANY_SLICES");   // pins the number of slices (tests, measurements)
  Split best{0, 0, 0, 0};
  for (int t = 0; t < 4; ++t) {
    if (pin >= 0 && t != pin) continue;
    const long long tiles = tiles_with(t, m, n);
    const int chunks = (k + chunk_of(t) - 1) / chunk_of(t);
    for (int round = 0; round <= 4; ++round) {   // one workgroup per tile; 192, 256, 512, 768 workgroups
      long long want = e != nullptr ? atoi(e) : round == 0 ? 1 : (round == 1 ? 192 : 256 * (round - 1)) / tiles;
      if (want < 1 || (want == 1 && round > 0 && e == nullptr)) continue;
      if (want > chunks) want = chunks;
      const int per = static_cast<int>((chunks + want - 1) / want), slices = (chunks + per - 1) / per;
      const double blocks = static_cast<double>(tiles) * slices;
      const double rounds = blocks > 512 ? blocks / 256 : blocks > 256 ? 2 : 1;
      double us = kTile[t] + rounds * per * kChunk[t] + (rounds - 1) * kRound[t];
      if (slices > 1 || blocks > 512) us += kFinish + kMillionSums * 1e-6 * slices * static_cast<double>(m) * n;
      if (best.slices == 0 || us < best.us) best = Split{t, slices, per, us};
    }
  }
  return best;
}

// the pick for a shape is asked for several times per call: each thread keeps the last few
Split pick_split(const ConvShape& s) {
  if (getenv("NITI_ANY_TILE") != nullptr || getenv("NITI_ANY_SLICES") != nullptr) return estimate_split(s);
  struct Entry {
    int key[6];
    Split split;
  };
  static thread_local Entry kept[16] = {};
  const int key[6] = {s.N, s.H * 65536 + s.W, s.C, s.K, s.R * 65536 + s.S, s.pad};
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

int launch_conv_any_requant(ConvPass pass, const ConvShape& s, const int8_t* x, const int8_t* w, int8_t* y, bool roundtrip, uint32_t* sync,
                            const RequantSpec& rq, hipStream_t stream) {
  ConvAnyArgs a = args_of(pass, s, x, w, roundtrip);
  set_rounding(a.g, rq, sync);
  a.g.out8 = y;
  const int t = requant_tile(pass, s);
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
