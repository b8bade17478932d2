// int8 products of matrices with any extents and alignment, in any of the four operand layouts, as one launch: int32
// results (the drop-in int8_mm, niti_gemm_i8), results rounded to int8 across the tensor-wide range, or rounded and
// subtracted from the weights (TiLinear's passes, ti_torch.py:241-266).
//
// What it replaces: products outside the whole-tile kernels went through copies of both operands (transposed, rows padded to
// 16 bytes), a fill of the result, a reduction split over workgroups by atomics, a pass for the range and one for the
// rounding - up to eight launches of which none had work for the chip.  These products are small (a hidden layer on a
// batch), so a launch costs what its latency chain costs: fill the pipe, walk the reduction, exchange the range, store.
//
// A workgroup (512 threads, 8 wavefronts) owns BM x BN of the result and walks the reduction in chunks of BK.  A chunk
// travels memory -> registers -> LDS in 16-byte pieces, two LDS buffers, DEPTH chunks in flight while one multiplies.  An operand
// whose reduction index is the fast one lies in LDS row by row (pitch BK + 16: sixteen rows fall into different banks) and
// is read by ds_read_b128; one whose reduction index is slow lies as stored (pitch BM + 16) and is read by
// ds_read_b64_tr_b8, which hands a lane eight consecutive reduction steps of one column.  Nothing is re-laid in memory.
// The wavefronts are WM x WN places x WK parts of every chunk's steps; the parts are added through LDS on the way into a
// row-major arrangement, in which a thread takes four consecutive results and neighbours take neighbouring columns.
#include "gemm_any.h"

#include <stdlib.h>

#include "grid_range.h"
#include "lds_asm.h"

namespace niti {
namespace {

enum Mode { kInt32 = 0, kRequant = 1, kUpdate = 2 };

// WM x WN x WK wavefronts, each TM x TN products of 32 x 32; DEPTH chunks on their way to the registers
template <int WM_, int WN_, int WK_, int TM_, int TN_, int BK_, int DEPTH_>
struct Tile {
  static constexpr int WM = WM_, WN = WN_, WK = WK_, TM = TM_, TN = TN_, BK = BK_, DEPTH = DEPTH_;
  static constexpr int BM = 32 * WM * TM, BN = 32 * WN * TN;
  static constexpr int SPW = BK / 32 / WK;              // 32-step products of a wavefront per chunk
  static_assert(WM * WN * WK == 8 && BK % (32 * WK) == 0, "eight wavefronts");
};
using TileS = Tile<1, 1, 8, 1, 1, 512, 2>;    //  32 x  32
using TileM = Tile<2, 2, 2, 1, 1, 256, 2>;    //  64 x  64
using TileL = Tile<2, 4, 1, 2, 1, 128, 2>;    // 128 x 128

// LDS bytes of an operand's chunk: rows x BK with the reduction index fast, BK x rows otherwise
template <bool kFast, int ROWS, int BK>
constexpr int chunk_pitch() { return kFast ? BK + 16 : ROWS + (ROWS > 32 ? 16 : 0); }
template <bool kFast, int ROWS, int BK>
constexpr int chunk_bytes() { return (kFast ? ROWS : BK) * chunk_pitch<kFast, ROWS, BK>(); }

constexpr int kPatchPitch = 36;                         // words per row of a 32 x 32 patch of sums
constexpr int kPatchBytes = 32 * kPatchPitch * 4;

template <class T, bool TA, bool TB>
constexpr int lds_bytes() {
  const int stage = 2 * (chunk_bytes<!TA, T::BM, T::BK>() + chunk_bytes<TB, T::BN, T::BK>());
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
template <bool kFast, bool kAligned>   // kFast: the reduction index is the fast one - a chunk advances along the row, otherwise along the rows
struct Operand {
  struct Raw {
    v4i lo, hi;   // hi: unused when the rows are aligned
  };
  __amdgpu_buffer_rsrc_t rsrc;   // the granules of the matrix: what lies outside reads as zeros and is not fetched
  int rows, len, skip;           // skip: bytes of the first granule in front of the matrix
  __device__ Operand(const int8_t* base, int rows_, int len_)
      : rows(rows_), len(len_), skip(kAligned ? 0 : static_cast<int>(reinterpret_cast<uintptr_t>(base) & 15)) {
    rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(base) - skip, 0, (rows * len + skip + 15) & ~15, 0x00020000);
  }
  // byte offset of a piece at chunk 0; rows outside the matrix lie behind every chunk's end
  __device__ int offset(int row, int col) const { return kFast && row >= rows ? kOutside : row * len + col + skip; }
  __device__ Raw load(int off, int k0) const {
    const int at = off + (kFast ? k0 : k0 * len);
    Raw r;
    r.lo = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc, kAligned ? at : at & ~15, 0, 0));
    if (!kAligned) r.hi = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc, (at & ~15) + 16, 0, 0));
    return r;
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

// kAligned: both operands' rows start on 16-byte boundaries
template <class T, bool TA, bool TB, int MODE, bool kAligned>
__global__ __launch_bounds__(512) void gemm_any_kernel(const AnyArgs g) {
  extern __shared__ __attribute__((aligned(16))) int8_t smem[];
  constexpr int PA = chunk_pitch<!TA, T::BM, T::BK>(), PB = chunk_pitch<TB, T::BN, T::BK>();
  constexpr int BYTES_A = chunk_bytes<!TA, T::BM, T::BK>(), BYTES_B = chunk_bytes<TB, T::BN, T::BK>();
  constexpr int NA = T::BM * T::BK / 16 / 512, NB = T::BN * T::BK / 16 / 512;     // pieces per thread and chunk
  static_assert(T::BM * T::BK % 8192 == 0 && T::BN * T::BK % 8192 == 0, "whole pieces");
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // Workgroups go to the eight dies in turn, and each die has its own L2: a die takes a run of neighbouring tiles, along the
  // side on which neighbours share the lines of an operand with the reduction index slow.
  const int nt = gridDim.x, mt = gridDim.y, nb = nt * mt;
  const int id = blockIdx.y * nt + blockIdx.x;
  const int tile = T::BM >= 128 ? id : (id & 7) * (nb >> 3) + min(id & 7, nb & 7) + (id >> 3);
  const int n0 = (TA ? tile / mt : tile % nt) * T::BN, m0 = (TA ? tile % mt : tile / nt) * T::BM;
  const int chunks = (g.k + T::BK - 1) / T::BK;
  using OpA = Operand<!TA, kAligned>;
  using OpB = Operand<TB, kAligned>;
  const OpA oa(g.a, TA ? g.k : g.m, TA ? g.m : g.k);
  const OpB ob(g.b, TB ? g.n : g.k, TB ? g.k : g.n);
  // piece i of this thread: (row, column) of the operand at chunk 0, and where it goes in LDS
  auto row_a = [&](int i) { return TA ? (tid + i * 512) / (T::BM / 16) : m0 + (tid + i * 512) / (T::BK / 16); };
  auto col_a = [&](int i) { return TA ? m0 + (tid + i * 512) % (T::BM / 16) * 16 : (tid + i * 512) % (T::BK / 16) * 16; };
  auto row_b = [&](int i) { return TB ? n0 + (tid + i * 512) / (T::BK / 16) : (tid + i * 512) / (T::BN / 16); };
  auto col_b = [&](int i) { return TB ? (tid + i * 512) % (T::BK / 16) * 16 : n0 + (tid + i * 512) % (T::BN / 16) * 16; };
  int off_a[NA], off_b[NB];
#pragma unroll
  for (int i = 0; i < NA; ++i) off_a[i] = oa.offset(row_a(i), col_a(i));
#pragma unroll
  for (int i = 0; i < NB; ++i) off_b[i] = ob.offset(row_b(i), col_b(i));

  typename OpA::Raw ra[T::DEPTH][NA];
  typename OpB::Raw rb[T::DEPTH][NB];
  auto load = [&](int c, typename OpA::Raw (&ra)[NA], typename OpB::Raw (&rb)[NB]) {
#pragma unroll
    for (int i = 0; i < NA; ++i) ra[i] = oa.load(off_a[i], c * T::BK);
#pragma unroll
    for (int i = 0; i < NB; ++i) rb[i] = ob.load(off_b[i], c * T::BK);
  };
  auto stage = [&](int c, const typename OpA::Raw (&ra)[NA], const typename OpB::Raw (&rb)[NB]) {
    int8_t* const as = smem + (c & 1) * (BYTES_A + BYTES_B);
    int8_t* const bs = as + BYTES_A;
    const int k0 = c * T::BK;
    const bool last = c == chunks - 1;
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      const int p = tid + i * 512;
      const int per = TA ? T::BM / 16 : T::BK / 16;
      v4i v = oa.join(ra[i], off_a[i]);
      if (last) v = oa.cut(v, row_a(i) + (TA ? k0 : 0), col_a(i) + (TA ? 0 : k0));
      *reinterpret_cast<v4i*>(as + p / per * PA + p % per * 16) = v;
    }
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int p = tid + i * 512;
      const int per = TB ? T::BK / 16 : T::BN / 16;
      v4i v = ob.join(rb[i], off_b[i]);
      if (last) v = ob.cut(v, row_b(i) + (TB ? 0 : k0), col_b(i) + (TB ? k0 : 0));
      *reinterpret_cast<v4i*>(bs + p / per * PB + p % per * 16) = v;
    }
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
  auto multiply = [&](int c) {
    const unsigned base = lds0 + (c & 1) * (BYTES_A + BYTES_B);
    static_for<T::SPW>([&](auto step) {
      constexpr int s = decltype(step)::value;
      v2i alo[T::TM], ahi[T::TM], blo[T::TN], bhi[T::TN];
      v4i av[T::TM], bv[T::TN];
#pragma unroll
      for (int t = 0; t < T::TM; ++t) {
        if (!TA) {
          av[t] = lds_read_b128_at<s * 32>(base + fa[t]);
        } else {
          alo[t] = lds_read_tr8<s * 32 * PA>(base + fa[t]);
          ahi[t] = lds_read_tr8<s * 32 * PA + 8 * PA>(base + fa[t]);
        }
      }
#pragma unroll
      for (int t = 0; t < T::TN; ++t) {
        if (TB) {
          bv[t] = lds_read_b128_at<s * 32>(base + fb[t]);
        } else {
          blo[t] = lds_read_tr8<s * 32 * PB>(base + fb[t]);
          bhi[t] = lds_read_tr8<s * 32 * PB + 8 * PB>(base + fb[t]);
        }
      }
      lds_settle<0>();
#pragma unroll
      for (int t = 0; t < T::TM; ++t) {
        if (!TA) asm volatile("" : "+v"(av[t]));
        else av[t] = lds_landed(alo[t], ahi[t]);
      }
#pragma unroll
      for (int t = 0; t < T::TN; ++t) {
        if (TB) asm volatile("" : "+v"(bv[t]));
        else bv[t] = lds_landed(blo[t], bhi[t]);
      }
      // MFMA A = 32 columns of the result, B = 32 rows: element 4 q + e of a lane is column 8 q + 4 (lane / 32) + e of row
      // lane % 32
#pragma unroll
      for (int i = 0; i < T::TM; ++i)
#pragma unroll
        for (int q = 0; q < T::TN; ++q) acc[i][q] = __builtin_amdgcn_mfma_i32_32x32x32_i8(bv[q], av[i], acc[i][q], 0, 0, 0);
    });
  };
  static_for<T::DEPTH>([&](auto d) {
    if (d < chunks) load(d, ra[d], rb[d]);
  });
  for (int c0 = 0; c0 < chunks; c0 += T::DEPTH) {
    static_for<T::DEPTH>([&](auto d) {
      const int c = c0 + d;
      if (c >= chunks) return;
      stage(c, ra[d], rb[d]);                           // the barrier in front of the last product: this buffer has been read
      if (c + T::DEPTH < chunks) load(c + T::DEPTH, ra[d], rb[d]);
      fence_sync();
      multiply(c);
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
        if (MODE == kInt32 && g.roundtrip != 0) fin[i][e] = f32_roundtrip(fin[i][e]);
        if (n0 + col + e < g.n) {
          const uint32_t u = uabs(fin[i][e]);
          lmax = u > lmax ? u : lmax;
        }
      }
    }
  }
  uint32_t* const words = reinterpret_cast<uint32_t*>(smem + lds_bytes<T, TA, TB>() - 32 * 4);
  int shift = 0;
  if (MODE == kInt32) {
    if (g.absmax != nullptr) {
      lmax = wave_max_u32(lmax);
      if (lane == 0) words[wave] = lmax;
      __syncthreads();
      if (wave == 0) fold_absmax(g.absmax, lane < 8 ? words[lane] : 0u);
    }
  } else {
    shift = grid_shift<8>(g, lmax, words, words + 8);
  }
  const bool trunc = g.trunc != 0, relu = (g.rq_flags & NITI_RQ_RELU) != 0;
  // what the rounding reads is requested for all of the thread's results in front of the first store (the compiler keeps
  // loads of an array behind stores to it: one trip to memory per group otherwise)
  v4i rnd[G];
  uint32_t wold[G];
  if (MODE != kInt32) {
#pragma unroll
    for (int i = 0; i < G; ++i) {
      const int t = tid + i * 512;
      const int row = m0 + t / (T::BN / 4), col = n0 + t % (T::BN / 4) * 4;
      rnd[i] = v4i{0, 0, 0, 0};
      wold[i] = 0;
      if ((GROUPS < 512 && t >= GROUPS) || row >= g.m || col + 4 > g.n) continue;
      const long long at = static_cast<long long>(row) * g.n + col;
      if (g.method == NITI_ROUND_STOCHASTIC) __builtin_memcpy(&rnd[i], g.rand + at, 16);
      if (MODE == kUpdate) __builtin_memcpy(&wold[i], g.w + at, 4);
    }
  }
#pragma unroll
  for (int i = 0; i < G; ++i) {
    const int t = tid + i * 512;
    if (GROUPS < 512 && t >= GROUPS) continue;
    const int row = m0 + t / (T::BN / 4), col = n0 + t % (T::BN / 4) * 4;
    if (row >= g.m || col >= g.n) continue;
    const long long at = static_cast<long long>(row) * g.n + col;
    const int here = min(4, g.n - col);
    if (MODE == kInt32) {
      if (here == 4) {
        __builtin_memcpy(g.c + at, &fin[i], 16);        // rows of any length: 4-byte aligned
      } else {
        for (int e = 0; e < here; ++e) g.c[at + e] = fin[i][e];
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
    if (here == 4) {
      const uint32_t packed = pack4_i8(r[0], r[1], r[2], r[3]);
      if (MODE == kUpdate) {
        const uint32_t old = wold[i];
        int wn4[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) wn4[e] = clip127(static_cast<int>(static_cast<int8_t>((old >> (8 * e)) & 0xFFu)) - r[e]);
        const uint32_t fresh = pack4_i8(wn4[0], wn4[1], wn4[2], wn4[3]);
        __builtin_memcpy(g.w + at, &fresh, 4);
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

}  // namespace

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
