// The tile of the products and convolutions of any extents (gemm_any.hip, conv_any.hip): a workgroup of 512 threads, 8
// wavefronts, owns BM x BN of a result and walks the reduction in chunks of BK.
//
// A chunk travels memory -> registers -> LDS in 16-byte pieces, two LDS buffers, DEPTH chunks in flight while one multiplies.
// What differs from one kernel to the next is where a piece comes from - an operand class says so.  An operand whose
// reduction index is the fast one lies in LDS row by row (pitch BK + 16: sixteen rows fall into different banks) and is read
// by ds_read_b128; one whose reduction index is slow lies as stored (pitch BM + 16) and is read by ds_read_b64_tr_b8, which
// hands a lane eight consecutive reduction steps of one column.  Nothing is re-laid in memory.
// The wavefronts are WM x WN places x WK parts of every chunk's steps; the parts are added through LDS on the way into a
// row-major arrangement, in which a thread takes four consecutive results and neighbours take neighbouring columns.
#pragma once
#include "gemm_any.h"
#include "grid_range.h"
#include "lds_asm.h"

namespace niti {

enum AnyMode { kInt32 = 0, kRequant = 1, kUpdate = 2 };

// WM x WN x WK wavefronts, each TM x TN products of 32 x 32; DEPTH chunks on their way to the registers, LOOK steps' fragments
// on their way from LDS
template <int WM_, int WN_, int WK_, int TM_, int TN_, int BK_, int DEPTH_, int LOOK_>
struct Tile {
  static constexpr int WM = WM_, WN = WN_, WK = WK_, TM = TM_, TN = TN_, BK = BK_, DEPTH = DEPTH_, LOOK = LOOK_;
  static constexpr int BM = 32 * WM * TM, BN = 32 * WN * TN;
  static constexpr int SPW = BK / 32 / WK;              // 32-step products of a wavefront per chunk
  static_assert(WM * WN * WK == 8 && BK % (32 * WK) == 0, "eight wavefronts");
};
using TileS = Tile<1, 1, 8, 1, 1, 512, 2, 2>;    //  32 x  32
using TileM = Tile<2, 2, 2, 1, 1, 256, 2, 4>;    //  64 x  64
using TileH = Tile<4, 2, 1, 1, 1, 128, 2, 4>;    // 128 x  64
using TileL = Tile<2, 4, 1, 2, 1, 128, 2, 2>;    // 128 x 128

// An operand's chunk: ROWS rows x BK reduction steps.  kFast: the reduction index is the fast one - LDS holds the rows one
// after the other, otherwise the steps.  Piece i of a thread lies at (row, col) of what LDS holds.
template <bool kFast_, int ROWS_, int BK_>
struct Pieces {
  static constexpr bool kFast = kFast_;
  static constexpr int ROWS = ROWS_, BK = BK_;
  static constexpr int PITCH = kFast ? BK + 16 : ROWS + (ROWS > 32 ? 16 : 0);
  static constexpr int BYTES = (kFast ? ROWS : BK) * PITCH;
  static constexpr int PER = (kFast ? BK : ROWS) / 16;        // pieces side by side
  static constexpr int N = ROWS * BK / 16 / 512;              // pieces of a thread
  static_assert(ROWS * BK % 8192 == 0 && 512 % PER == 0, "whole pieces, a thread's all in one column");
  __device__ static int row(int i) { return (static_cast<int>(threadIdx.x) + i * 512) / PER; }
  __device__ static int col() { return static_cast<int>(threadIdx.x) % PER * 16; }
};

constexpr int kPatchPitch = 36;                         // words per row of a 32 x 32 patch of sums
constexpr int kPatchBytes = 32 * kPatchPitch * 4;

template <class T, class OpA, class OpB>
constexpr int any_lds_bytes() {
  const int stage = 2 * (OpA::G::BYTES + OpB::G::BYTES);
  const int park = 8 * T::TM * T::TN * kPatchBytes;
  return (stage > park ? stage : park) + 32 * 4;
}

__device__ inline void fence_sync() {   // barrier that the compiler also treats as a fence for the hand-written LDS reads
  asm volatile("" ::: "memory");
  __syncthreads();
  asm volatile("" ::: "memory");
}

// One operand: its pieces of 16 bytes, of a [rows][len] matrix of total bytes.  A piece of a matrix whose rows do not start on
// 16-byte boundaries is put together from the two aligned granules it lies in: an unaligned 16-byte load occupies the address
// unit for every lane on its own (a launch of 14 chunks took 15 us).  Loads go through a buffer descriptor that ends with the
// matrix's last granule, so none fetches a granule without a byte of the operand in it, and are straight-line code (a
// branch in front of one makes the compiler wait for all loads in flight behind it).  Rows and columns outside the result give results
// nobody looks at; only the reduction's tail has to be zero, in the last chunk.
constexpr int kOutside = 0x70000000;   // byte offset behind any matrix these kernels take, any chunk added
// kCut: what lies behind the reduction's end has to be made zero (the other operand's is not zero there).
template <class G_, bool kAligned, bool kCut = true>   // G::kFast: a chunk advances along the row, otherwise along the rows
struct DenseOperand {
  using G = G_;
  static constexpr bool kFast = G::kFast, kPairs = !kAligned;
  struct Raw {
    v4i lo, hi;   // hi: unused when the rows are aligned
  };
  __amdgpu_buffer_rsrc_t rsrc;   // the granules of the matrix: what lies outside reads as zeros and is not fetched
  int rows, len, first, skip;    // first: row or column the tile starts at; skip: bytes of the first granule in front of the matrix
  int off[G::N];                 // this thread's pieces at chunk 0
  __device__ DenseOperand(const int8_t* base, int rows_, int len_, int first_)
      : rows(rows_), len(len_), first(first_), skip(kAligned ? 0 : static_cast<int>(reinterpret_cast<uintptr_t>(base) & 15)) {
    rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(base) - skip, 0, (rows * len + skip + 15) & ~15, 0x00020000);
#pragma unroll
    for (int i = 0; i < G::N; ++i) off[i] = kFast && row(i) >= rows ? kOutside : row(i) * len + col() + skip;
  }
  __device__ int row(int i) const { return kFast ? first + G::row(i) : G::row(i); }
  __device__ int col() const { return kFast ? G::col() : first + G::col(); }
  __device__ void load(int c, Raw (&r)[G::N]) const {
    const int step = c * G::BK * (kFast ? 1 : len);
#pragma unroll
    for (int i = 0; i < G::N; ++i) {
      const int at = off[i] + step;
      r[i].lo = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc, kAligned ? at : at & ~15, 0, 0));
      if (!kAligned) r[i].hi = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc, (at & ~15) + 16, 0, 0));
    }
  }
  __device__ v4i piece(const Raw& r, int i, int c, bool last) const {
    const v4i v = join(r, off[i]);
    if (!kCut || !last) return v;
    return cut(v, row(i) + (kFast ? 0 : c * G::BK), col() + (kFast ? c * G::BK : 0));
  }
  __device__ v4i join(const Raw& r, int off) const {   // chunks start a multiple of 16 bytes apart: off decides
    if (kAligned) return r.lo;
    // dwords 0 .. 7 of the two granules, from dword off / 4 % 4 on (values, not array elements: a select between elements
    // of a local array becomes a select of addresses and the array stays in memory)
    const bool two = (off & 8) != 0, one = (off & 4) != 0;
    auto pick = [](bool c, int x, int y) { return c ? x : y; };
    const int t0 = pick(two, r.lo[2], r.lo[0]), t1 = pick(two, r.lo[3], r.lo[1]), t2 = pick(two, r.hi[0], r.lo[2]),
              t3 = pick(two, r.hi[1], r.lo[3]), t4 = pick(two, r.hi[2], r.hi[0]), t5 = pick(two, r.hi[3], r.hi[1]);
    const int u0 = pick(one, t1, t0), u1 = pick(one, t2, t1), u2 = pick(one, t3, t2), u3 = pick(one, t4, t3), u4 = pick(one, t5, t4);
    const uint32_t b = static_cast<uint32_t>(off) & 3u;
    auto cat = [b](int hi, int lo) {
      return static_cast<int>(__builtin_amdgcn_alignbyte(static_cast<uint32_t>(hi), static_cast<uint32_t>(lo), b));
    };
    const v4i v = {cat(u1, u0), cat(u2, u1), cat(u3, u2), cat(u4, u3)};
    return v;
  }
  // the piece at (row, col) of the last chunk without what lies behind the reduction's end
  __device__ v4i cut(v4i v, int row, int col) const {
    const int keep = kFast ? len - col : (row < rows ? 16 : 0);
    if (keep >= 16) return v;
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const int n = keep - 4 * d;
      v[d] = n >= 4 ? v[d] : (n <= 0 ? 0 : v[d] & static_cast<int>((1u << (8 * n)) - 1u));
    }
    return v;
  }
};

// An operand's load(c, raw) is called for c = first, first + 1, ... in turn, piece(raw, i, c, last) once for each of its pieces.
// Chunks first .. chunks - 1 of the tile at (m0, n0) of the [g.m][g.n] result; int32 sums go to `out`.  shift_of(largest
// magnitude of the lane, 32 words of LDS, requests to send while it waits): the shift, for the modes that round.
template <class T, class OpA, class OpB, int MODE, class ShiftOf>
__device__ __forceinline__ void any_tile(const AnyArgs& g, int32_t* const out, OpA oa, OpB ob, const int m0, const int n0, const int first,
                                         const int chunks, int8_t* const smem, ShiftOf shift_of) {
  constexpr bool TA = !OpA::G::kFast, TB = OpB::G::kFast;
  constexpr int PA = OpA::G::PITCH, PB = OpB::G::PITCH;
  constexpr int BYTES_A = OpA::G::BYTES, BYTES_B = OpB::G::BYTES;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  typename OpA::Raw ra[T::DEPTH][OpA::G::N];
  typename OpB::Raw rb[T::DEPTH][OpB::G::N];
  auto stage = [&](int c, const typename OpA::Raw (&ra)[OpA::G::N], const typename OpB::Raw (&rb)[OpB::G::N]) {
    int8_t* const as = smem + ((c - first) & 1) * (BYTES_A + BYTES_B);
    int8_t* const bs = as + BYTES_A;
    const bool last = c == chunks - 1;
#pragma unroll
    for (int i = 0; i < OpA::G::N; ++i) *reinterpret_cast<v4i*>(as + OpA::G::row(i) * PA + OpA::G::col()) = oa.piece(ra[i], i, c, last);
#pragma unroll
    for (int i = 0; i < OpB::G::N; ++i) *reinterpret_cast<v4i*>(bs + OpB::G::row(i) * PB + OpB::G::col()) = ob.piece(rb[i], i, c, last);
  };

  const int kh = wave % T::WK, wn = wave / T::WK % T::WN, wm = wave / T::WK / T::WN;
  const int lr = lane & 31, lk = lane >> 5;
  const int j = lane & 15, gg = (lane >> 4) & 1;
  unsigned fa[T::TM], fb[T::TN];                        // where this lane's fragments lie in a buffer
#pragma unroll
  for (int t = 0; t < T::TM; ++t) {
    const int row = (wm * T::TM + t) * 32;
    fa[t] = !TA ? (row + lr) * PA + kh * (T::SPW * 32) + lk * 16
                : (kh * (T::SPW * 32) + lk * 16 + (j >> 1)) * PA + row + gg * 16 + 8 * (j & 1);
  }
#pragma unroll
  for (int t = 0; t < T::TN; ++t) {
    const int col = (wn * T::TN + t) * 32;
    fb[t] = BYTES_A + (TB ? (col + lr) * PB + kh * (T::SPW * 32) + lk * 16
                          : (kh * (T::SPW * 32) + lk * 16 + (j >> 1)) * PB + col + gg * 16 + 8 * (j & 1));
  }
  v16i acc[T::TM][T::TN];
#pragma unroll
  for (int i = 0; i < T::TM; ++i)
#pragma unroll
    for (int q = 0; q < T::TN; ++q)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][q][e] = 0;

  const unsigned lds0 = lds_addr(smem);
  // Fragments are read LOOK steps ahead of their products; `meanwhile` (the loads of a later chunk and their addresses) runs
  // behind the first reads.  One step at a time, a chunk took an LDS round trip per step: 64 x 64 tiles walked a long
  // reduction in 0.75 us per 256 steps.
  constexpr int LOOK = OpA::kPairs && T::LOOK > 2 ? 2 : T::LOOK;   // registers: granule pairs take twice as many
  constexpr int READS = (TA ? 2 : 1) * T::TM + (TB ? 1 : 2) * T::TN;   // of one step
  v2i alo[LOOK][T::TM], ahi[LOOK][T::TM], blo[LOOK][T::TN], bhi[LOOK][T::TN];
  v4i av[LOOK][T::TM], bv[LOOK][T::TN];
  auto multiply = [&](int c, auto meanwhile) {
    const unsigned base = lds0 + ((c - first) & 1) * (BYTES_A + BYTES_B);
    auto read = [&](auto step) {
      constexpr int s = decltype(step)::value, u = s % LOOK;
#pragma unroll
      for (int t = 0; t < T::TM; ++t) {
        if (!TA) {
          av[u][t] = lds_read_b128_at<s * 32>(base + fa[t]);
        } else {
          alo[u][t] = lds_read_tr8<s * 32 * PA>(base + fa[t]);
          ahi[u][t] = lds_read_tr8<s * 32 * PA + 8 * PA>(base + fa[t]);
        }
      }
#pragma unroll
      for (int t = 0; t < T::TN; ++t) {
        if (TB) {
          bv[u][t] = lds_read_b128_at<s * 32>(base + fb[t]);
        } else {
          blo[u][t] = lds_read_tr8<s * 32 * PB>(base + fb[t]);
          bhi[u][t] = lds_read_tr8<s * 32 * PB + 8 * PB>(base + fb[t]);
        }
      }
    };
    static_for<(LOOK < T::SPW ? LOOK : T::SPW)>([&](auto s) { read(s); });
    meanwhile();
    static_for<T::SPW>([&](auto step) {
      constexpr int s = decltype(step)::value, u = s % LOOK;
      constexpr int ahead = (s + LOOK < T::SPW ? s + LOOK : T::SPW) - s - 1;   // steps read and not yet wanted
      lds_settle<(ahead * READS < 15 ? ahead * READS : 15)>();
#pragma unroll
      for (int t = 0; t < T::TM; ++t) {
        if (!TA) asm volatile("" : "+v"(av[u][t]));
        else av[u][t] = lds_landed(alo[u][t], ahi[u][t]);
      }
#pragma unroll
      for (int t = 0; t < T::TN; ++t) {
        if (TB) asm volatile("" : "+v"(bv[u][t]));
        else bv[u][t] = lds_landed(blo[u][t], bhi[u][t]);
      }
      // MFMA A = 32 columns of the result, B = 32 rows: element 4 q + e of a lane is column 8 q + 4 (lane / 32) + e of row
      // lane % 32
#pragma unroll
      for (int i = 0; i < T::TM; ++i)
#pragma unroll
        for (int q = 0; q < T::TN; ++q) acc[i][q] = __builtin_amdgcn_mfma_i32_32x32x32_i8(bv[u][q], av[u][i], acc[i][q], 0, 0, 0);
      if constexpr (s + LOOK < T::SPW) read(std::integral_constant<int, s + LOOK>{});
    });
  };
  static_for<T::DEPTH>([&](auto d) {
    if (first + d < chunks) {
      oa.load(first + d, ra[d]);
      ob.load(first + d, rb[d]);
    }
  });
  for (int c0 = first; c0 < chunks; c0 += T::DEPTH) {
    static_for<T::DEPTH>([&](auto d) {
      const int c = c0 + d;
      if (c >= chunks) return;
      stage(c, ra[d], rb[d]);                           // the barrier in front of the last product: this buffer has been read
      fence_sync();
      multiply(c, [&] {
        if (c + T::DEPTH < chunks) {
          oa.load(c + T::DEPTH, ra[d]);
          ob.load(c + T::DEPTH, rb[d]);
        }
      });
    });
  }
  fence_sync();                                         // the staging area now takes the sums

  // sums, one 32 x 32 patch per wavefront and product, patches of one place (its WK parts) next to each other
  int* const patches = reinterpret_cast<int*>(smem);
#pragma unroll
  for (int i = 0; i < T::TM; ++i)
#pragma unroll
    for (int q = 0; q < T::TN; ++q) {
      const int place = (wm * T::TM + i) * (T::WN * T::TN) + wn * T::TN + q;
      int* const patch = patches + (place * T::WK + kh) * (32 * kPatchPitch) + lr * kPatchPitch + 4 * lk;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        *reinterpret_cast<v4i*>(patch + 8 * e) = v4i{acc[i][q][4 * e], acc[i][q][4 * e + 1], acc[i][q][4 * e + 2], acc[i][q][4 * e + 3]};
    }
  __syncthreads();
  constexpr int GROUPS = T::BM * T::BN / 4;             // of four consecutive results
  constexpr int G = (GROUPS + 511) / 512;
  v4i fin[G];
  uint32_t lmax = 0;
#pragma unroll
  for (int i = 0; i < G; ++i) {
    const int t = tid + i * 512;
    fin[i] = v4i{0, 0, 0, 0};
    if (GROUPS < 512 && t >= GROUPS) continue;
    const int row = t / (T::BN / 4), col = t % (T::BN / 4) * 4;
    const int place = (row >> 5) * (T::WN * T::TN) + (col >> 5);
    const int* const src = patches + place * T::WK * (32 * kPatchPitch) + (row & 31) * kPatchPitch + (col & 31);
#pragma unroll
    for (int h = 0; h < T::WK; ++h) fin[i] += *reinterpret_cast<const v4i*>(src + h * (32 * kPatchPitch));
    if (m0 + row < g.m) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (g.roundtrip != 0) fin[i][e] = f32_roundtrip(fin[i][e]);
        if (n0 + col + e < g.n) {
          const uint32_t u = uabs(fin[i][e]);
          lmax = u > lmax ? u : lmax;
        }
      }
    }
  }
  // What the rounding reads besides the sums - random integers, old weights, mask, windows - is requested for all of the thread's
  // results behind the workgroup's own slot and in front of the looks at the others': the trip to memory runs while the launch waits
  // for its range, and neither the requests nor the work on their addresses keep the other workgroups waiting for this slot.  Device
  // times, us, operands that are in no cache / in the caches, requests behind the exchange -> in front of the slot -> here:
  //   100 x 1000 -> 300, forward + backward      18.56 / 17.36 -> 17.72 / 16.84 -> 17.76 / 16.84
  //   the same, StoShift                         19.32 / 17.36 -> 17.60 / 16.72 -> 17.60 / 16.40
  //   300 x 2000 -> 1000                         41.88 / 38.16 -> 42.23 / 38.39 -> 40.47 / 36.76
  //   one image through 7 layers (nothing to request)  71.3 / 56.2 -> 72.3 / 57.1 -> 71.0 / 55.6
  v4i rnd[G];
  uint32_t wold[G];
  constexpr bool kUnpool = MODE == kRequant && G <= 4;   // the launches that use it have these tiles
  uint32_t window[kUnpool ? G : 1][4];
  constexpr bool kPool = MODE == kRequant && T::BN <= 64;      // a window's four rows lie in one wavefront
  auto place = [&](int row, int col) {                         // of a result
    if constexpr (kPool) {
      if (g.pool != nullptr) {
        const int image = g.by_map.of(row), rest = row - image * (g.map_h * g.map_w), window = rest >> 2, wh = g.by_map_w.of(window);
        row = image * (g.map_h * g.map_w) + (2 * wh + ((rest >> 1) & 1)) * g.map_w + 2 * (window - wh * (g.map_w >> 1)) + (rest & 1);
      }
    }
    return static_cast<long long>(row) * g.n + col;
  };
  auto window_at = [&](int row, int col) {
    const int image = g.by_map.of(row), rest = row - image * (g.map_h * g.map_w), h = g.by_map_w.of(rest), w = rest - h * g.map_w;
    return (static_cast<long long>(image * 2 * g.map_h + 2 * h) * (2 * g.map_w) + 2 * w) * g.n + col;
  };
  auto request = [&] {
#pragma unroll
    for (int i = 0; i < G; ++i) {
      const int t = tid + i * 512;
      const int row = m0 + t / (T::BN / 4), col = n0 + t % (T::BN / 4) * 4;
      rnd[i] = v4i{0, 0, 0, 0};
      wold[i] = 0;
      if ((GROUPS < 512 && t >= GROUPS) || row >= g.m || col + 4 > g.n) continue;
      const long long at = place(row, col);
      if (g.method == NITI_ROUND_STOCHASTIC) __builtin_memcpy(&rnd[i], g.rand + at, 16);
      if (MODE == kUpdate) __builtin_memcpy(&wold[i], g.w + at, 4);
      if (MODE == kRequant && g.mask != nullptr) __builtin_memcpy(&wold[i], g.mask + at, 4);
      if constexpr (kUnpool) {
        if (g.unpool != nullptr) {
          const int8_t* const from = g.pool_x + window_at(row, col);
#pragma unroll
          for (int q = 0; q < 4; ++q) __builtin_memcpy(&window[i][q], from + ((q >> 1) * 2 * g.map_w + (q & 1)) * static_cast<long long>(g.n), 4);
        }
      }
    }
  };
  uint32_t* const words = reinterpret_cast<uint32_t*>(smem + any_lds_bytes<T, OpA, OpB>() - 32 * 4);
  int shift = 0;
  if (MODE == kInt32) {
    if (g.absmax != nullptr) {
      lmax = wave_max_u32(lmax);
      if (lane == 0) words[wave] = lmax;
      __syncthreads();
      if (wave == 0) fold_absmax(g.absmax, lane < 8 ? words[lane] : 0u);
    }
  } else {
    shift = shift_of(lmax, words, request);
  }
  const bool trunc = g.trunc != 0, relu = (g.rq_flags & NITI_RQ_RELU) != 0;
#pragma unroll
  for (int i = 0; i < G; ++i) {
    const int t = tid + i * 512;
    if (GROUPS < 512 && t >= GROUPS) continue;
    const int row = m0 + t / (T::BN / 4), col = n0 + t % (T::BN / 4) * 4;
    if (row >= g.m || col >= g.n) continue;
    const long long at = place(row, col);
    const int here = min(4, g.n - col);
    if (MODE == kInt32) {
      if (here == 4) {
        __builtin_memcpy(out + at, &fin[i], 16);        // rows of any length: 4-byte aligned
      } else {
        for (int e = 0; e < here; ++e) out[at + e] = fin[i][e];
      }
      continue;
    }
    v4i u = rnd[i];
    if (g.method == NITI_ROUND_STOCHASTIC && here < 4)
      for (int e = 0; e < here; ++e) u[e] = g.rand[at + e];
    v4i r = round4_any(fin[i], shift, g.method, trunc, u);
    if (MODE == kRequant && relu) {
#pragma unroll
      for (int e = 0; e < 4; ++e) r[e] = max(r[e], 0);
    }
    if (MODE == kRequant && g.mask != nullptr) {          // zero where the mask is not positive
      uint32_t mk = wold[i];
      if (here < 4)
        for (int e = 0; e < here; ++e) mk |= static_cast<uint32_t>(static_cast<uint8_t>(g.mask[at + e])) << (8 * e);
#pragma unroll
      for (int e = 0; e < 4; ++e) r[e] = static_cast<int8_t>((mk >> (8 * e)) & 0xFFu) > 0 ? r[e] : 0;
    }
    if constexpr (kUnpool) {
      if (g.unpool != nullptr) {   // channels are a multiple of 16 here
        const uint32_t v = pack4_i8(r[0], r[1], r[2], r[3]);
        int8_t* const to = g.unpool + window_at(row, col);
        uint32_t taken = 0;        // bytes that an earlier position of the window (scan order) already received
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const uint32_t eq = equal_bytes(window[i][q], wold[i]);
          const uint32_t put = v & (g.ties_all != 0 ? eq : eq & ~taken);
          taken |= eq;
          __builtin_memcpy(to + ((q >> 1) * 2 * g.map_w + (q & 1)) * static_cast<long long>(g.n), &put, 4);
        }
        continue;
      }
    }
    if (here == 4) {
      const uint32_t packed = pack4_i8(r[0], r[1], r[2], r[3]);
      if constexpr (kPool) {
        if (g.pool != nullptr) {     // whole windows are inside the result or outside, columns a multiple of 4
          uint32_t mx = max_i8x4(packed, static_cast<uint32_t>(__shfl_xor(static_cast<int>(packed), T::BN / 4)));
          mx = max_i8x4(mx, static_cast<uint32_t>(__shfl_xor(static_cast<int>(mx), T::BN / 2)));
          if ((row & 3) == 0) __builtin_memcpy(g.pool + static_cast<long long>(row >> 2) * g.n + col, &mx, 4);
        }
      }
      if (MODE == kUpdate) {
        const uint32_t old = wold[i];
        int wn4[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) wn4[e] = clip127(static_cast<int>(static_cast<int8_t>((old >> (8 * e)) & 0xFFu)) - r[e]);
        const uint32_t fresh = pack4_i8(wn4[0], wn4[1], wn4[2], wn4[3]);
        __builtin_memcpy(g.w + at, &fresh, 4);
        if (g.wprep != nullptr) {
          const int tap = g.by_channels.of(col), ch = col - tap * g.channels;
          const int block = ((row >> 6) * ((g.channels + 31) >> 5) + (ch >> 5)) * 9 + tap;
          *reinterpret_cast<uint32_t*>(g.wprep + filter_copy_at(static_cast<uint32_t>(block), static_cast<uint32_t>(row) & 63u, static_cast<uint32_t>(ch))) = fresh;
        }
      }
      if (MODE == kRequant || g.out8 != nullptr) __builtin_memcpy(g.out8 + at, &packed, 4);
    } else {
      for (int e = 0; e < here; ++e) {
        if (MODE == kUpdate) g.w[at + e] = static_cast<int8_t>(clip127(static_cast<int>(g.w[at + e]) - r[e]));
        if (MODE == kRequant || g.out8 != nullptr) g.out8[at + e] = static_cast<int8_t>(r[e]);
      }
    }
  }
}

}  // namespace niti
