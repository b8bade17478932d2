// What the 3x3 convolution kernels on 4 ... 32 pixel wide maps share: their arguments, the grid-wide range exchange around
// their main loops and the epilogue that turns a workgroup's int32 sums into int32 or rounded int8 results.
#pragma once
#include <type_traits>

#include "common.h"
#include "lds_asm.h"
#include "requant_math.h"

namespace niti {

struct HaloArgs {
  const int8_t* x;    // [N,Q,Q,C]
  const int8_t* wp;   // prepared filter: [ceil(K/64)][cslices][9][64][32], rows XOR-swizzled
  int32_t* y;         // [N,Q,Q,K]
  uint32_t* absmax;
  int N, C, K;
  int cslices;        // ceil(C / 32)
  int src_cslices;    // kWT only: 32-channel slices of the forward filter copy read as the data gradient's filter
  long long x_bytes, wp_bytes, y_bytes;
  unsigned flags;
  // requantising variant only
  int8_t* y8;         // [N,Q,Q,K] int8
  const int8_t* mask; // optional [N,Q,Q,K] int8: outputs whose mask byte is not positive are stored as zero
  uint32_t* sync;     // word 0: max |sum| of the launch (output), word 1: set when the wait gave up,
                      // words kSyncSlot0..: one slot per workgroup, max + 1; all zero on entry
  long long y8_bytes;
  int8_t* pool;       // optional [N,Q/2,Q/2,K] int8: 2x2 / stride-2 maximum of y8 (the max-pool that follows the layer)
  long long pool_bytes;
  // data gradient through a 2x2 / stride-2 max-pool in front of the layer: `mask` is the pooled map (this launch's
  // result is the gradient with respect to it), pool_x the pooling's input [N,2Q,2Q,K]; the rounded, masked result
  // goes to the position(s) of each window that equal the pooled value, into unpool [N,2Q,2Q,K], and y8 is not written
  const int8_t* pool_x;
  int8_t* unpool;
  long long unpool_bytes;
  int ties_all;
  int target_bits, method, trunc, bw_mode;
  const int32_t* rand;   // NITI_ROUND_STOCHASTIC: one random integer per output element [N,Q,Q,K], low `shift` bits used
  unsigned rq_flags;
  long long spin_limit;  // wall-clock ticks (100 MHz) the wait may last
  uint32_t* sticky;      // device-wide word set when the wait gives up, may be null
  int32_t* shift_out;
  const int32_t* exp_a;
  const int32_t* exp_b;
  int32_t* exp_out;
};
constexpr int kSyncSlot0 = 16;
static_assert(kSlotStride >= 2, "workgroups with several tiles keep the shift a tile was stored with in the word behind its slot");
constexpr int kMaxSlots = 4096;

// The same convolution on products of 64 channels (conv3x3_k64.h); the filter copy must hold a whole number of 64-channel
// slices (an even cslices).
int launch_conv3x3_k64_int32(const HaloArgs& a, int H, int ktile, hipStream_t stream);
int launch_conv3x3_k64_requant(const HaloArgs& a, int H, int ktile, hipStream_t stream);
int launch_conv3x3_k64_sto(const HaloArgs& a, int H, int ktile, hipStream_t stream);

// the arguments of a launch of the requantising variant (conv3x3_halo.hip)
int halo_requant_args(HaloArgs& a, const int8_t* x, const int8_t* wp, int8_t* y8, int N, int H, int C, int K, unsigned flags, uint32_t* sync,
                      const RequantSpec& rq);

namespace {

// Which of the convolution's tiles this is: x along the pixels, y along the channel tiles, of nx * ny.
struct HaloPlace {
  int x, y, nx, ny;
  __device__ int block() const { return y * nx + x; }
  __device__ int blocks() const { return nx * ny; }
};
__device__ inline HaloPlace halo_grid_place() { return {static_cast<int>(blockIdx.x), static_cast<int>(blockIdx.y), static_cast<int>(gridDim.x), static_cast<int>(gridDim.y)}; }

constexpr int kOob = -1;
constexpr int kOobFar = static_cast<int>(0x80000000u);   // out of range whatever scalar offset below 2^31 is added

// s_waitcnt vmcnt(N) with the other counters left alone
template <int N>
__device__ inline void hc_wait_vmcnt() {
  static_assert(N >= 0 && N <= 15);
  __builtin_amdgcn_s_waitcnt(0x0F70 | N);
}
__device__ inline void hc_sync() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// NITI_RQ_SHIFT_HINT: *shift_out holds the caller's prediction (the previous training step's shift of this tensor).
// Read at a tile's start, a whole main loop before it is needed; tile 0 overwrites the word only after all slots are filled, i.e. after
// this line has been passed for every tile.
// The load is unconditional (from the range word when there is no prediction), its address looks lane-dependent to
// the compiler and its result is not looked at before the epilogue: a load inside a branch, or one whose result the
// compiler knows to be the same in all lanes (and moves to a scalar register at once), would be waited for on the
// spot - a trip to memory in front of the first stage's loads.
struct ShiftHint {
  bool hinted;
  int predicted_raw;
};
__device__ inline ShiftHint halo_shift_hint(const HaloArgs& a, int settle_shift) {
  ShiftHint h;
  h.hinted = (a.rq_flags & NITI_RQ_SHIFT_HINT) != 0 && a.shift_out != nullptr && settle_shift < 0;
  const int32_t* const src = h.hinted ? a.shift_out : reinterpret_cast<const int32_t*>(a.sync);
  h.predicted_raw = __hip_atomic_load(src + opaque_zero(), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return h;
}

// The 16-byte pieces in which a wavefront stores its rounded results, and what they need from memory besides the sums: the mask
// bytes (ReLU backward of the layer below / the pooled map) and, with the max-pool's backward pass folded in, the windows of the
// pooling's input.  Neither depends on the rounding.  kRegs256 (one workgroup per compute unit): the main loop's last slice
// requests them, in the place of the loads that have nothing left to fetch, and all stay in registers (without a mask or a
// pooling the requests are out of range: zeros, no memory traffic).  Otherwise the first two
// mask pieces and the first window are requested in front of the range reduction and later ones two (one) pieces ahead of
// their use; the wavefronts with four accumulator tiles in 128 registers request two mask pieces behind the rounding, later ones two
// pieces ahead, and windows where they are used (256 images of 16 x 16, 256 -> 256, data gradient with every mask piece where it is used
// 36.2 us, so 35.7; of 32 x 32, 128 -> 128 44.9 / 43.8; through the pooling 57.9 / 55.5).
template <int Q, int KT, bool kTwo, int NWF, int PT, bool kRegs256>
struct HaloPieces {
  static constexpr int LPP = NWF * 2;       // lanes (16-byte pieces) per pixel
  static constexpr int PPI = 64 / LPP;      // pixels per store instruction
  static constexpr int NPIECE = 32 * PT / PPI;
  static constexpr bool kMaskAhead = kRegs256 || NWF * PT <= 2;
  static constexpr int MKD = kRegs256 ? NPIECE : (!kMaskAhead ? 1 : (NPIECE < 2 ? NPIECE : 2));
  static constexpr int XWD = kRegs256 ? NPIECE : 1;
  // With the max-pool's backward pass folded in, the two wavefronts that share pixels exchange halves of their patches: each
  // then writes the windows of half its pixels at the tile's full width.  At its own width a wavefront wrote every line of the
  // four times larger result in pieces of 32 (64) bytes, and the lines left the cache half written (16 x 16 -> 32 x 32, 128
  // channels, 256 images: 46.9 us, 24.7 of them without the folded pass).
  static constexpr bool kPairs = !kTwo && KT != 32;
  static constexpr int LPU = KT / 16, PPU = 64 / LPU;
  bool pairs;
  int mfirst, mstep, ch;
  __device__ HaloPieces(const HaloArgs& a, int pixbase, int kt, int wp_, int wc, int lane) {
    pairs = kPairs && a.unpool != nullptr;
    mfirst = pixbase + (kTwo ? wc * 256 : 0) + wp_ * (32 * PT) + (pairs ? wc * (16 * PT) + lane / LPU : lane / LPP);
    mstep = pairs ? PPU : PPI;
    ch = pairs ? kt * KT + lane % LPU * 16 : (kTwo ? kt * KT : kt * KT + wc * (KT / 2)) + lane % LPP * 16;
  }
  __device__ bool inside(const HaloArgs& a, int t) const { return mfirst + t * mstep < static_cast<long long>(a.N) * Q * Q && ch < a.K; }
  __device__ int offset(const HaloArgs& a, int t) const { return inside(a, t) ? (mfirst + t * mstep) * a.K + ch : kOob; }
  __device__ v4i mask(const HaloArgs& a, int t) const {
    const __amdgpu_buffer_rsrc_t rm = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(a.mask), 0, a.mask != nullptr ? a.y8_bytes : 0, 0x00020000);
    return __builtin_amdgcn_raw_buffer_load_b128(rm, offset(a, t), 0, 0);
  }
  // the window of pooled pixel m in the pooling's input
  __device__ int window_offset(const HaloArgs& a, int t, int k) const {
    const int m = mfirst + t * mstep;
    const int n = m / (Q * Q), rem = m - n * (Q * Q);
    const int pp = rem / Q, pq = rem - pp * Q;
    return inside(a, t) ? ((n * 2 * Q + 2 * pp + (k >> 1)) * 2 * Q + 2 * pq + (k & 1)) * a.K + ch : kOob;
  }
  __device__ void window_offsets(const HaloArgs& a, int t, int (&wo)[4]) const {
#pragma unroll
    for (int k = 0; k < 4; ++k) wo[k] = window_offset(a, t, k);
  }
  __device__ v4i window(const HaloArgs& a, int t, int k) const {
    const __amdgpu_buffer_rsrc_t rxp = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(a.pool_x), 0, a.unpool != nullptr ? a.unpool_bytes : 0, 0x00020000);
    return __builtin_amdgcn_raw_buffer_load_b128(rxp, window_offset(a, t, k), 0, 0);
  }
  __device__ void windows(const HaloArgs& a, int t, v4i (&xw)[4]) const {
#pragma unroll
    for (int k = 0; k < 4; ++k) xw[k] = window(a, t, k);
  }
};
template <int Q, int KT, bool kTwo, int NWF, int PT, bool kRegs256>
struct HaloAhead {
  using P = HaloPieces<Q, KT, kTwo, NWF, PT, kRegs256>;
  v4i mk[P::MKD];
  v4i xw[P::XWD][4];
};

// A workgroup's only tile; see Turns
struct OneTile {
  __device__ int thread() const { return threadIdx.x; }
  __device__ int again() const { return -1; }       // the final shift, when the tile is stored again with it
  __device__ bool early() const { return false; }   // stored by the shift as it looks from here; nobody waits
};
// What a workgroup does besides: see SumsAlong (wgrad_finish.h).
struct NothingAlong : OneTile {
  __device__ void begin() {}
  __device__ void publish() {}
  __device__ void guess() {}
  __device__ void wait(const HaloArgs&) const {}
  __device__ void update(int, const int32_t*, const int32_t*) const {}
};

// Results of a workgroup: 8 wavefronts of PT x 32 pixels x NWF x 32 channels (wp_: pixel group, wc: channel group; kTwo: wc is
// the 256-pixel half, all wavefronts have the same 64 channels).  q[(i * PT + j) * 4 + g]: four consecutive channels of one pixel
// of the 32-channel tile i and 32-pixel tile j; L says which: channel L::channel(g, lane) .. + 3 of the tile, pixel
// L::pixel(g, lane).  smem: the main loop's tiles, dead once every wavefront is here; red: 16 words
// that no load of the main loop writes.
template <int Q, int KT, bool kTwo, int NWF, int PT, bool kFused, bool kSto, bool kRegs256, class L, class Along>
__device__ __forceinline__ void halo_epilogue(const HaloArgs& a, const HaloPlace at, v4i (&q)[NWF * PT * 4], int8_t* const smem, uint32_t* const red, const int pixbase,
                                              const int kt, const int wp_, const int wc, const int settle_shift, const ShiftHint hint,
                                              const HaloPieces<Q, KT, kTwo, NWF, PT, kRegs256>& pc, HaloAhead<Q, KT, kTwo, NWF, PT, kRegs256>& ahead, Along& along) {
  const int tid = along.thread();
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool hinted = hint.hinted;
  const int predicted_raw = hint.predicted_raw;
  const bool roundtrip = (a.flags & NITI_EPI_F32_ROUNDTRIP) != 0;
  int vmax = 0, vmin = 0;
#pragma unroll
  for (int t = 0; t < NWF * PT * 4; ++t)
#pragma unroll
    for (int e = 0; e < 4; e += 2) {
      vmax = max(vmax, max(q[t][e], q[t][e + 1]));
      vmin = min(vmin, min(q[t][e], q[t][e + 1]));
    }
  // The fp32 round trip is the identity up to 2^24, so it is applied (wavefront-uniformly) only beyond; it is
  // monotonic and odd, so the range after it follows from the extreme values alone, and the sums themselves
  // are converted where they are consumed below instead of in a second copy of the accumulators.
  bool rt = false;
  if (roundtrip) rt = wave_max_u32(max(static_cast<uint32_t>(vmax), 0u - static_cast<uint32_t>(vmin))) > (1u << 24);
  if (rt) {
    vmax = f32_roundtrip(vmax);
    vmin = f32_roundtrip(vmin);
  }
  const uint32_t lmax = max(static_cast<uint32_t>(vmax), 0u - static_cast<uint32_t>(vmin));
  const long long total_pix = static_cast<long long>(a.N) * Q * Q;
  const int chbase = kTwo ? kt * KT : kt * KT + wc * (KT / 2);
  const int pixwave = pixbase + (kTwo ? wc * 256 : 0) + wp_ * (32 * PT);   // first pixel of this wavefront
  if constexpr (!kFused) {
    hc_sync();  // all wavefronts are done with the tiles: reuse LDS as per-wavefront transposition patches
    constexpr int ROWB = 32 * 4 + 16;  // one 32-channel tile row of int32, padded
    int8_t* patch = smem + wave * (32 * ROWB);
    const int rrow = lane >> 3, rcol = lane & 7;  // 8 lanes x 16 bytes = one 32-channel row
    const __amdgpu_buffer_rsrc_t ry = __builtin_amdgcn_make_buffer_rsrc(a.y, 0, a.y_bytes, 0x00020000);
#pragma unroll
    for (int j = 0; j < PT; ++j) {
      const int mrow = pixwave + j * 32 + rrow;
#pragma unroll
      for (int i = 0; i < NWF; ++i) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          v4i v = q[(i * PT + j) * 4 + g];
          if (rt) {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = f32_roundtrip(v[e]);
          }
          *reinterpret_cast<v4i*>(patch + L::pixel(g, lane) * ROWB + L::channel(g, lane) * 4) = v;
        }
        // same wavefront reads back what it wrote: LDS operations of one wavefront complete in order
        const int ch = chbase + i * 32 + rcol * 4;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const v4i v = *reinterpret_cast<const v4i*>(patch + (t * 8 + rrow) * ROWB + rcol * 16);
          const int m = mrow + t * 8;
          const int off = (m < total_pix && ch < a.K) ? (m * a.K + ch) * 4 : kOob;
          __builtin_amdgcn_raw_buffer_store_b128(v, ry, off, 0, 2);
        }
      }
    }
    // one atomic per workgroup at most: same-address atomics serialise in the memory system
    if (a.absmax != nullptr) {
      const uint32_t wmax = wave_max_u32(lmax);
      if (lane == 0) red[wave] = wmax;
      __syncthreads();
      if (wave == 0) fold_absmax(a.absmax, lane < 8 ? red[lane] : 0u);
    }
  } else {
    // ---- tensor-wide range: workgroup maximum -> own slot -> maximum over the slots of all workgroups.
    // Results are stored before the range is final: the slots filled so far (read before this workgroup's own
    // maximum is known, so the latency hides behind that reduction) and the own maximum give a shift that is the
    // final one unless another workgroup raises the bit width; the int8 stores of all workgroups then overlap the
    // wait for the last slots instead of following it in one burst.  When the final shift differs, the sums (still
    // in registers) are rounded and stored once more.
    const int nb = at.blocks();
    uint32_t* const slots = a.sync + kSyncSlot0;
    constexpr int kLook = 8;   // slots a lane reads with its loads in flight together
    const bool nowait = along.early();
    const bool settled = settle_shift >= 0;
    constexpr int PROW = NWF * 32 + 16;  // the wavefront's channels of one pixel, padded
    int8_t* patch = smem + wave * (32 * PT * PROW);
    const __amdgpu_buffer_rsrc_t ry = __builtin_amdgcn_make_buffer_rsrc(a.y8, 0, a.y8_bytes, 0x00020000);
    using P = HaloPieces<Q, KT, kTwo, NWF, PT, kRegs256>;
    constexpr int LPP = P::LPP, PPI = P::PPI, NPIECE = P::NPIECE, MKD = P::MKD;
    constexpr bool kMaskAhead = P::kMaskAhead;
    const int piece = lane % LPP;
    const int mstep = pc.mstep, ch = pc.ch;
    const int8_t* const from = pc.pairs ? smem + (wp_ + 4 * (lane % P::LPU / (KT / 32))) * (32 * PT * PROW) + (wc * (16 * PT) + lane / P::LPU) * PROW + lane % P::LPU % (KT / 32) * 16
                                        : patch + lane / LPP * PROW + piece * 16;
    // mask bytes and pooling windows: see HaloPieces
    auto request_first = [&] {
      if (kMaskAhead && !kRegs256 && a.mask != nullptr) {
#pragma unroll
        for (int t = 0; t < MKD; ++t) ahead.mk[t] = pc.mask(a, t);
        if (a.unpool != nullptr) pc.windows(a, 0, ahead.xw[0]);
      }
    };
    request_first();
    // Without a prediction, a hint: the first 64 * kLook slots as they are now.  With one the look would only put a
    // trip to memory between the last product and the first store.
    uint32_t early[kLook];
#pragma unroll
    for (int u = 0; u < kLook; ++u) {
      const int i = u * 64 + lane;
      early[u] = (wave == 0 && i < nb && !nowait && !settled && !hinted) ? __hip_atomic_load(slot_word(slots, i), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0u;
    }
    const uint32_t wmax = wave_max_u32(lmax);
    if (lane == 0) red[wave] = wmax;
    __syncthreads();  // the tiles are dead from here on
    // every wavefront forms the workgroup's maximum itself: with a prediction nothing else stands between it and its stores
    uint32_t gmax = red[0];
#pragma unroll
    for (int w = 1; w < 8; ++w) gmax = max(gmax, red[w]);
    if (tid == 0 && !settled) __hip_atomic_store(slot_word(slots, at.block()), gmax + 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    along.publish();
    if (nb > 1 && !nowait && !settled && !hinted) {
      if (wave == 0) {
        uint32_t g = gmax + 1u;
#pragma unroll
        for (int u = 0; u < kLook; ++u) g = early[u] > g ? early[u] : g;
        g = wave_max_u32(g);
        if (lane == 0) red[8] = g - 1u;
      }
      __syncthreads();
      gmax = red[8];
    }
    // a shift below 1 means "no shift" whatever its value; the prediction counts unless this workgroup's own sums or
    // the slots seen so far already need more (or the range is final already)
    int shift = max(bitwidth_of(gmax, a.bw_mode) - a.target_bits, 0);
    bool final_range = nb == 1;
    if (!final_range && hinted) shift = max(shift, predicted_raw);
    if (settled) shift = settle_shift;
    if (nowait) {   // the shift this tile is stored with: see tiles_in_turns
      if (tid == 0) __hip_atomic_store(slot_word(slots, at.block()) + 1, static_cast<uint32_t>(shift), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    final_range = final_range || nowait || settled;
    const bool trunc = a.trunc != 0;
    const bool relu = (a.rq_flags & NITI_RQ_RELU) != 0;
    const bool psto = a.method == NITI_ROUND_PSEUDO_STOCHASTIC;
    // StoShift: the caller's random integer of each output element decides its rounding step; a tile that is rounded
    // twice (final shift unlike the first) takes the low bits of the same integers for the other shift
    constexpr bool sto = kSto;
    const __amdgpu_buffer_rsrc_t rrand = __builtin_amdgcn_make_buffer_rsrc(const_cast<int32_t*>(a.rand), 0, sto ? a.y8_bytes * 4 : 0, 0x00020000);
    if (rt) {   // once, in place: the values are rounded up to twice below
#pragma unroll
      for (int t = 0; t < NWF * PT * 4; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) q[t][e] = f32_roundtrip(q[t][e]);
    }
#pragma nounroll
    for (int pass = 0; pass < 2; ++pass) {
      // addresses are worked out in every pass rather than kept in registers that the wavefronts with four accumulator tiles do not have
      P pieces = pc;
      if constexpr (!kMaskAhead) asm volatile("" : "+v"(pieces.mfirst));
      // the sums look modified to the compiler in every pass: nothing derived from them (magnitudes, signs) is
      // computed ahead of the loop and kept in 64 more registers
#pragma unroll
      for (int t = 0; t < NWF * PT * 4; ++t) asm volatile("" : "+v"(q[t]));
      // round, pack four channels per dword, transpose through a per-wavefront patch, store 16-byte pieces; the
      // common rounding mode gets a short form
      // The shift is the same in every lane but has come through LDS, which the compiler cannot know: made a scalar
      // here, the choice between the two forms below is ONE scalar branch.  (Left inside the loops as a per-lane
      // condition it cost every value both forms' set-up under execution masks and a taken branch.)
      const int ushift = __builtin_amdgcn_readfirstlane(shift);
      const bool fast = ushift >= 1 && !trunc && !psto && !sto;
      const int sm1 = ushift - 1, lo = relu ? 0 : -127;
      auto round_tiles = [&](auto fastc) {
        constexpr bool kFast = decltype(fastc)::value;
#pragma unroll
        for (int j = 0; j < PT; ++j)
#pragma unroll
          for (int i = 0; i < NWF; ++i)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
              uint32_t packed;
              const v4i s4 = q[(i * PT + j) * 4 + g];
              if constexpr (kFast) {
                packed = round4_nearest_floor_fast(s4[0], s4[1], s4[2], s4[3], sm1, lo);
              } else {
                int r[4];
                v4i u = {0, 0, 0, 0};
                if (sto) {   // the four values are consecutive channels of one pixel
                  const int m = pixwave + j * 32 + L::pixel(g, lane), c0 = chbase + i * 32 + L::channel(g, lane);
                  u = __builtin_amdgcn_raw_buffer_load_b128(rrand, (m < total_pix && c0 < a.K) ? (m * a.K + c0) * 4 : kOob, 0, 0);
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                  const int x = s4[e];
                  if (ushift >= 1)
                    r[e] = sto    ? round_sto32(x, ushift, trunc, u[e])
                           : psto ? round_one32<NITI_ROUND_PSEUDO_STOCHASTIC>(x, ushift, trunc)
                                  : round_one32<NITI_ROUND_NEAREST>(x, ushift, trunc);
                  else r[e] = wrap_to_i8(x);
                  if (relu && r[e] < 0) r[e] = 0;
                }
                packed = pack4_i8(r[0], r[1], r[2], r[3]);
              }
              *reinterpret_cast<uint32_t*>(patch + (j * 32 + L::pixel(g, lane)) * PROW + i * 32 + L::channel(g, lane)) = packed;
            }
      };
      if (fast) round_tiles(std::true_type{});
      else round_tiles(std::false_type{});
      // same wavefront reads back what it wrote: LDS operations of one wavefront complete in order
      // without room for them earlier: two mask pieces at a time from here on (all four: 1 to 3 us more a launch for what they spill)
      v4i mask_of[2];
      if (!kMaskAhead && a.mask != nullptr) {
#pragma unroll
        for (int t = 0; t < 2; ++t) mask_of[t] = pieces.mask(a, t);
      }
      if (pc.pairs) __syncthreads();
#pragma unroll
      for (int t = 0; t < 32 * PT / PPI; ++t) {
        v4i v = *reinterpret_cast<const v4i*>(from + t * mstep * PROW);
        const int off = pieces.offset(a, t);
        v4i mk;
        if (a.mask != nullptr) {  // ReLU backward of the layer below, folded in: its output is this layer's input
          if constexpr (kMaskAhead) {
            mk = ahead.mk[t % MKD];
            if (t + MKD < NPIECE) ahead.mk[t % MKD] = pieces.mask(a, t + MKD);
          } else {
            mk = mask_of[t % 2];
            if (t + 2 < NPIECE) mask_of[t % 2] = pieces.mask(a, t + 2);
          }
#pragma unroll
          for (int d = 0; d < 4; ++d) v[d] &= static_cast<int>(positive_bytes(static_cast<uint32_t>(mk[d])));
        }
        if (a.unpool != nullptr) {
          // max-pool backward folded in (mk holds the pooled values): the window of pooled pixel m in the pooling's input
          const __amdgpu_buffer_rsrc_t ru = __builtin_amdgcn_make_buffer_rsrc(a.unpool, 0, a.unpool_bytes, 0x00020000);
          int wo[4];
          pieces.window_offsets(a, t, wo);
          v4i xw[4], ow[4];
          if constexpr (kMaskAhead) {
#pragma unroll
            for (int k = 0; k < 4; ++k) xw[k] = ahead.xw[t % P::XWD][k];
            if (t + P::XWD < NPIECE) pieces.windows(a, t + P::XWD, ahead.xw[t % P::XWD]);
          } else {
            pieces.windows(a, t, xw);
          }
#pragma unroll
          for (int d = 0; d < 4; ++d) {
            uint32_t taken = 0;   // bytes whose gradient an earlier position of the window (scan order) already received
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              const uint32_t eq = equal_bytes(static_cast<uint32_t>(xw[k][d]), static_cast<uint32_t>(mk[d]));
              const uint32_t keep = a.ties_all != 0 ? eq : eq & ~taken;
              ow[k][d] = static_cast<int>(static_cast<uint32_t>(v[d]) & keep);
              taken |= eq;
            }
          }
#pragma unroll
          for (int k = 0; k < 4; ++k) __builtin_amdgcn_raw_buffer_store_b128(ow[k], ru, wo[k], 0, 0);
        } else {
          // the 128-channel tile writes 64 bytes per pixel and wavefront: streaming stores start the write-back of the
          // 16 MiB result while the kernel still runs (measured 2 us per launch); the 32-byte pieces of the 64-channel
          // tile are slower that way
          __builtin_amdgcn_raw_buffer_store_b128(v, ry, off, 0, NWF == 2 ? 2 : 0);
        }
      }
      if (a.pool != nullptr) {
        // The max-pool behind this layer, from the rounded values still in the patch: the wavefront's 32 PT pixels are a
        // strip of whole image rows (or whole images), i.e. 8 PT whole 2 x 2 windows; a lane takes 16 channels of one.
        constexpr int PC = Q / 2;   // pooled pixels per row
        for (int pq = lane / LPP; pq < 8 * PT; pq += PPI) {
          const int l0 = 2 * (pq / PC) * Q + 2 * (pq % PC);   // upper left pixel of the window inside the strip
          const int8_t* src = patch + l0 * PROW + piece * 16;
          const v4i p00 = *reinterpret_cast<const v4i*>(src), p01 = *reinterpret_cast<const v4i*>(src + PROW);
          const v4i p10 = *reinterpret_cast<const v4i*>(src + Q * PROW), p11 = *reinterpret_cast<const v4i*>(src + (Q + 1) * PROW);
          v4i mx;
#pragma unroll
          for (int d = 0; d < 4; ++d)
            mx[d] = static_cast<int>(max_i8x4(max_i8x4(static_cast<uint32_t>(p00[d]), static_cast<uint32_t>(p01[d])),
                                              max_i8x4(static_cast<uint32_t>(p10[d]), static_cast<uint32_t>(p11[d]))));
          const int m0 = pixwave + l0;
          const int n = m0 / (Q * Q), rem = m0 - n * (Q * Q);
          const int pr = rem / Q, pcol = rem - pr * Q;
          const int pix2 = (n * PC + (pr >> 1)) * PC + (pcol >> 1);
          const int off = (m0 < total_pix && ch < a.K) ? pix2 * a.K + ch : kOob;
          const __amdgpu_buffer_rsrc_t rp = __builtin_amdgcn_make_buffer_rsrc(a.pool, 0, a.pool_bytes, 0x00020000);
          __builtin_amdgcn_raw_buffer_store_b128(mx, rp, off, 0, 0);
        }
      }
      if (final_range) break;
      along.guess();
      // ---- wait for the slots of all workgroups; the maximum over them is the tensor's range
      if (wave == 0) {
        const uint32_t g = wait_slots(slots, nb, a.spin_limit, &a.sync[1], a.sticky);
        if (lane == 0) red[9] = g != 0u ? g - 1u : 0u;   // (not red[8]: no barrier has passed since the others read that)
      }
      along.wait(a);
      __syncthreads();
      final_range = true;
      gmax = red[9];
      const int fshift = max(bitwidth_of(gmax, a.bw_mode) - a.target_bits, 0);
      along.update(fshift, a.exp_a, a.exp_b);
      if (fshift == shift) break;
      shift = fshift;
      __builtin_amdgcn_s_waitcnt(0);   // the stores of the first pass leave before those that replace them
      request_first();
    }
    if (at.block() == 0 && tid == 0 && !nowait && !settled) {
      const int sh = shift > 0 ? shift : 0;
      a.sync[0] = gmax;
      if (a.shift_out != nullptr) *a.shift_out = sh;
      if (a.exp_out != nullptr)
        *a.exp_out = sh + (a.exp_a != nullptr ? *a.exp_a : 0) + (a.exp_b != nullptr ? *a.exp_b : 0);
    }
  }
}

// ---- more tiles than the device holds workgroups at once: every workgroup takes several in turn, the last of them (number blockIdx.x) as
// always.  The earlier ones are stored by the predicted shift, or what their own sums need, and leave a slot each; behind the wait of the
// last one, when the final shift is known, those that were stored with another are computed again and stored with it.
// One launch for all tiles without waiting and a second one that computed every tile again unless its shift was right took, with
// predictions that fail (as about half of those inside a training step do) and with good ones (us): 256 images of 32 x 32, 128 -> 128
// 67.4 / 44.1, so 57.5 / 42.1; data gradient 73.1 / 48.2, 62.6 / 46.6; 192 images 55.6 / 36.4, 47.6 / 35.2; 136 images 50.1 / 33.1, 43.2 / 33.5;
// 256 of 16 x 16, 256 -> 512 121.1 / 64.4, 96.1 / 63.6; 256 of 32 x 32, 256 -> 256 (four tiles each) 242 / 125, 223 / 129.  So with
// four tiles each and predictions that hold it is the slower way by about 2% (through the layer 123.4 / 125.5), with two it is not (136 to 256 images,
// 128 -> 128, 32.1 ... 41.7 / 31.0 ... 40.8).  It waits for its whole grid, which the two launches did not: it wants the device to itself, as
// the launches that fit at once do.  What bounds it: the first stage of each tile waits for its loads behind the stores of the one before.
struct Turns : NothingAlong {
  int final_shift = 0, settle_shift = -1;
  bool is_early = false;
  // (a new value to the compiler in every turn, like the arguments: what follows from them is worked out again rather than kept in registers)
  __device__ int thread() const {
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
  }
  __device__ int again() const { return settle_shift; }
  __device__ bool early() const { return is_early; }
  __device__ void update(int shift, const int32_t*, const int32_t*) { final_shift = shift; }
};
// tile(args, at), with `along` (Turns), in a kernel whose first argument is its HaloArgs and whose grid has at most as many workgroups as there are tiles (nx * ny)
template <class Along, class F>
__device__ __forceinline__ void tiles_in_turns(const int nx, const int ny, Along& along, F tile) {
  using Args = const __attribute__((address_space(4))) HaloArgs;
  const int step = gridDim.x, own = blockIdx.x;
  const auto take = [&](int id) {
    const HaloPlace at{id % nx, id / nx, nx, ny};
    Args* args = (Args*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(args));
    tile(*(const HaloArgs*)args, at);
  };
  // ids: own + n * step, .., own + step, own, then own + step, .. again
  const int last = own + (nx * ny - 1 - own) / step * step;
  bool back = false;
  for (int id = last;;) {
    along.is_early = !back && id != own;
    bool stored = false;
    if (back) {
      Args* args = (Args*)__builtin_amdgcn_kernarg_segment_ptr();
      // (written in front of the own tile's loads, which have been waited for since)
      stored = static_cast<int>(__hip_atomic_load(slot_word(args->sync + kSyncSlot0, id) + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) == along.settle_shift;
    }
    if (!stored) take(id);
    back = back || id == own;
    if (back) {
      id += step;
      if (id > last) return;
      along.settle_shift = __builtin_amdgcn_readfirstlane(along.final_shift);
    } else {
      id -= step;
    }
    __syncthreads();   // the tile before has left LDS
  }
}

// what a kernel's launches remember per device
struct HaloLaunch {
  bool attr_set[kDeviceSlots] = {};   // function attributes are per device
  int resident[kDeviceSlots] = {};    // workgroups the device holds at once
};
template <class Kernel>
int halo_attributes(Kernel k, HaloLaunch& state, size_t lds, bool count) {
  const int slot = device_slot();
  if (state.attr_set[slot]) return NITI_OK;
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)
    return fail(NITI_ERR_LAUNCH, "conv3x3_halo: cannot reserve %zu bytes of LDS", lds);
  if (count) {
    int dev = 0, cus = 0, per_cu = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(k), 512, lds) != hipSuccess)
      return fail(NITI_ERR_LAUNCH, "conv3x3_halo: cannot query occupancy");
    state.resident[slot] = cus * per_cu;
  }
  state.attr_set[slot] = true;
  return NITI_OK;
}

// A launch of ceil(pixels / px) x ceil(K / ktile) tiles by kernel `one`, or by kernel `several` where they are more than the device holds of
// its workgroups (the same kernel twice: a tile that is not chosen for such launches).
template <class Kernel>
struct HaloKernel {
  Kernel k;
  size_t lds;
};
template <class Kernel>
HaloKernel(Kernel, size_t) -> HaloKernel<Kernel>;
template <bool kFused, class One, class Several>
int launch_halo_kernel(HaloKernel<One> one, HaloKernel<Several> several, HaloLaunch (&state)[2], int px, int ktile, int Q, const HaloArgs& a, hipStream_t stream) {
  int st = halo_attributes(one.k, state[0], one.lds, kFused);
  if (st != NITI_OK) return st;
  const long long pix = static_cast<long long>(a.N) * Q * Q;
  const dim3 grid(static_cast<unsigned>((pix + px - 1) / px), (a.K + ktile - 1) / ktile);
  const long long tiles = static_cast<long long>(grid.x) * grid.y;
  if (kFused && tiles > state[0].resident[device_slot()]) {
    if constexpr (std::is_same_v<One, Several>) {
      return fail(NITI_ERR_UNSUPPORTED, "conv3x3_halo: %lld workgroups of this tile do not fit on the device at once", tiles);
    } else {
      if (tiles > kMaxSlots) return fail(NITI_ERR_UNSUPPORTED, "conv3x3_halo: %lld tiles exceed the %d range slots", tiles, kMaxSlots);
      st = halo_attributes(several.k, state[1], several.lds, true);
      if (st != NITI_OK) return st;
      const long long fit = state[1].resident[device_slot()];
      hipLaunchKernelGGL(several.k, dim3(static_cast<unsigned>(tiles < fit ? tiles : fit)), dim3(512), several.lds, stream, a, static_cast<int>(grid.x), static_cast<int>(grid.y));
      return check_launch("conv3x3_halo");
    }
  }
  hipLaunchKernelGGL(one.k, grid, dim3(512), one.lds, stream, a);
  return check_launch("conv3x3_halo");
}

}  // namespace
}  // namespace niti
