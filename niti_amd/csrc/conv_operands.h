// How the passes of a convolution find their operands' pieces on the tile of any_tile.h (conv_any.hip, conv_backward.hip).
#pragma once
#include "any_tile.h"
#include "conv_any.h"

namespace niti {

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
  static constexpr bool kPairs = false;
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
      int p, q;
      if (a.g.pool == nullptr) {
        p = a.by_q.of(pq);
        q = pq - p * a.Q;
      } else {               // window by window
        const int window = pq >> 2, wp = a.g.by_map_w.of(window);
        p = 2 * wp + ((pq >> 1) & 1);
        q = 2 * (window - wp * (a.Q >> 1)) + (pq & 1);
      }
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
  static constexpr bool kPairs = false;
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
  static constexpr bool kPairs = false;
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

// tile and slice `id` of nt x mt x slices
template <class T, ConvPass PASS, int MODE, class ShiftOf>
__device__ __forceinline__ void conv_any_tile(const ConvAnyArgs& a, int id, int nt, int mt, int slices, int8_t* smem, ShiftOf shift_of) {
  using A = typename Operands<T, PASS>::A;
  using B = typename Operands<T, PASS>::B;
  // Workgroups go to the eight dies in turn, and each die has its own L2: a die takes a run of neighbouring tiles (they share
  // pixels), of the same slice of the reduction where it is cut.
  const int per = nt * mt, nb = per * slices;
  const int place = (id & 7) * (nb >> 3) + min(id & 7, nb & 7) + (id >> 3);
  const int slice = place / per, tile = place - slice * per;
  const int n0 = tile % nt * T::BN, m0 = tile / nt * T::BM;
  const int total = (a.g.k + T::BK - 1) / T::BK;
  if constexpr (PASS == kConvWgrad) {
    const int first = slice * a.chunks_per_slice;
    any_tile<T, A, B, MODE>(a.g, a.g.c + slice * a.slice, A(a.g.a, a.g.k, a.g.m, m0), B(a, n0, first), m0, n0, first,
                            min(total, first + a.chunks_per_slice), smem, shift_of);
  } else if constexpr (PASS == kConvForward) {
    any_tile<T, A, B, MODE>(a.g, a.g.c, A(a, m0), B(a.g.b, a.g.n, a.g.k, n0), m0, n0, 0, total, smem, shift_of);
  } else {
    any_tile<T, A, B, MODE>(a.g, a.g.c, A(a, m0), B(a, n0), m0, n0, 0, total, smem, shift_of);
  }
}

template <class T>
long long tiles_of(int m, int n) { return static_cast<long long>((m + T::BM - 1) / T::BM) * ((n + T::BN - 1) / T::BN); }

template <class T, ConvPass PASS>
constexpr int lds_bytes() { return any_lds_bytes<T, typename Operands<T, PASS>::A, typename Operands<T, PASS>::B>(); }

inline ConvAnyArgs map_args(ConvPass pass, const ConvShape& s) {
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
inline void product_of(ConvPass pass, const ConvShape& s, int* m, int* n, int* k) {
  const int pixels = s.N * s.P() * s.Q();
  *m = pass == kConvForward ? pixels : pass == kConvDgrad ? s.N * s.H * s.W : s.K;
  *n = pass == kConvForward ? s.K : pass == kConvDgrad ? s.C : s.R * s.S * s.C;
  *k = pass == kConvForward ? s.R * s.S * s.C : pass == kConvDgrad ? s.R * s.S * s.K : pixels;
}
inline ConvAnyArgs args_of(ConvPass pass, const ConvShape& s, const int8_t* x, const int8_t* y, bool roundtrip) {
  ConvAnyArgs a = map_args(pass, s);
  product_of(pass, s, &a.g.m, &a.g.n, &a.g.k);
  a.g.a = x;
  a.g.b = y;
  a.g.roundtrip = roundtrip ? 1 : 0;
  return a;
}
inline void set_rounding(AnyArgs& g, const RequantSpec& rq, uint32_t* sync) {
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

}  // namespace niti
