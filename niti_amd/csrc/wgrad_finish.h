// What follows the main loop of the 3x3 weight gradient (wgrad3x3.hip): the partial sums of all slices -> rounded gradient -> updated
// weights, in a launch of its own, at the end of the main loop's launch, or along with the data gradient (conv3x3_k64_backward.hip).
#pragma once
#include <type_traits>

#include "common.h"
#include "requant_math.h"

namespace niti {

// Partial sums -> rounded gradient -> updated weights in one launch (the int32 gradient is not stored unless
// asked for).  A workgroup owns kFinishV x 64 int4 columns at a grid-wide stride; its NW wavefronts each add every
// NW-th slice of every column (no barrier in between, so all those loads are in flight together), column v is
// then completed through LDS by wavefront v % NW, which keeps the sums in registers.  The workgroup publishes its
// largest magnitude in its slot and waits for the slots of all workgroups (all resident: the host sizes the grid
// for that; the wait is bounded by a wall-clock limit), derives the shift from the maximum over the slots, and
// every wavefront applies w = clip(w - round(sum >> shift)) to its columns.  NW = 16 serves the launches with
// many slices and few columns, NW = 4 the others.
constexpr int kFinishV = 16;
constexpr int kFusedV = 48;         // columns per lane in the one-launch form (8 wavefronts: six each)
constexpr int kArriveSlots = 256;   // workgroups of the one-launch form at most
constexpr uint32_t kPartialBias = 1u << 23;   // added to the partial sums of the one-launch form before they are cut to 24 bits
constexpr int kFinishSlot0 = 16;
struct FinishArgs {
  const int32_t* partial;
  long long slice_stride;
  int splits;
  long long nv;        // int4 columns of the gradient: K*9*C / 4
  int C, Cw;           // channels per gradient row / per weight row (Cw <= C; the rest is channel padding)
  int8_t* w;           // [K][9][Cw], updated in place
  int8_t* g8;          // optional rounded gradient, laid out like w
  int32_t* dw;         // optional int32 gradient [K][9][C]
  int8_t* wprep;       // optional: the halo convolution kernel's forward copy of the [K][9][C] filter, kept in step with w
  uint32_t* sync;      // word 0: max |sum| (output); words kFinishSlot0..: slots, zero on entry
  // a finishing launch's wait gave up: word 1 of the call's sync words, into which flag_code is or-ed (elsewhere: word 1 of `sync`, or of the
  // data gradient's where the sums are added along with it - words that those kernels have at hand, unlike registers for one more pointer)
  uint32_t* flag;
  uint32_t flag_code;
  int roundtrip, target_bits, method, trunc, bw_mode;
  int predict;         // *shift_out holds a predicted shift on entry
  long long spin_limit;
  uint32_t* sticky;    // device-wide word set when the wait gives up, may be null
  int32_t* shift_out;
  const int32_t* exp_a;
  const int32_t* exp_b;
  int32_t* exp_out;
  uint32_t* arrive;    // one-launch form only: a slot per workgroup, zero on entry, filled when its partial sums are in memory
  // Slices of planes (one-launch form, and update along with the data gradient).  A slice then holds, per group of four consecutive
  // output channels kg, tap t and input channel c (unit u = (kg * 9 + t) * C + c), three planes: bits 0..15 of the four sums (8 bytes at 8u), bits 16..23 (4 bytes at
  // units * 8 + 4u) and bits 24..31 (4 bytes at units * 12 + 4u).  The third plane is written only by a workgroup whose
  // sums do not fit 24 bits; it says so in wide[tile + tiles * slice] (zero on entry) and in the value of its arrival slot or, along
  // with the data gradient, in the word behind all of these.
  uint32_t* wide;
  int tiles_k, tiles_c;
};

// The nine-tap kernel's launch that leaves its sums in planes (wgrad3x3.hip), and the arguments of what adds them; `wide` are that
// many zeroed words and one more: wgrad3x3_planes_blocks, 0 where that kernel does not take the shape; bands: of 256 pixels that a
// workgroup walks.
int wgrad3x3_planes_blocks(int N, int H, int C, int K, int* bands = nullptr);
int launch_wgrad3x3_planes(const int8_t* act, const int8_t* err, int8_t* w, int N, int H, int C, int K, bool roundtrip, uint32_t* sync, uint32_t* wide,
                           const RequantSpec& rq, int8_t* g8, int8_t* wprep, void* workspace, FinishArgs* finish, hipStream_t stream);

namespace {

typedef unsigned int v2u __attribute__((ext_vector_type(2)));

// Four sums of a gradient -> the rounded gradient; shift: a scalar
__device__ __forceinline__ v4i rounded4(const v4i s, const int shift, const bool psto, const bool trunc) {
  v4i r;
  if (shift < 1) {
#pragma unroll
    for (int e = 0; e < 4; ++e) r[e] = wrap_to_i8(s[e]);
  } else if (psto) {
#pragma unroll
    for (int e = 0; e < 4; ++e) r[e] = round_one32<NITI_ROUND_PSEUDO_STOCHASTIC>(s[e], shift, trunc);
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) r[e] = round_one32<NITI_ROUND_NEAREST>(s[e], shift, trunc);
  }
  return r;
}
// Four weights and their rounded gradient, as words: the updated weights; gp: the gradient's word
__device__ __forceinline__ uint32_t updated4(const uint32_t wold, const v4i r, uint32_t& gp) {
  uint32_t wnew = 0;
  gp = 0;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int wo = static_cast<int>(static_cast<int8_t>((wold >> (8 * e)) & 0xFFu));
    wnew |= (static_cast<uint32_t>(clip127(wo - r[e])) & 0xFFu) << (8 * e);
    gp |= (static_cast<uint32_t>(r[e]) & 0xFFu) << (8 * e);
  }
  return wnew;
}

template <int NW>
struct FinishShared {
  v4i part[2][NW][64];
  uint32_t wmax[NW];
  uint32_t gshare;
};


// The columns of workgroup `block` out of `nblocks` (V = int4 columns per lane it may own, NW its wavefronts).
// kPlanes: the sums were written by this same launch (by other dies' workgroups, with write-through stores): they
// are read with loads that do not hit a line another die may have changed (byte offsets then fit 31 bits: host check).  A column
// is then a unit (four output channels) while it is added and an int4 of weights from then on.
template <int NW, int V, bool kPlanes>
struct FinishColumns {
  static constexpr int OWN = V / NW > 0 ? V / NW : 1;   // columns a wavefront completes
  static constexpr int VS = V < NW ? V : NW;            // columns a workgroup has when the slices are shared (fewer rounds than wavefronts)

  const FinishArgs& a;
  const int block, nblocks, lane, wave;
  const uint32_t C, Cw;
  // division by the channel count: a shift for the usual powers of two (a 32-bit division is some forty instructions,
  // and this part of the launch runs few wavefronts)
  const int c_log2;
  const bool same_layout;
  uint32_t wold[OWN];
  v4i fin[OWN];

  __device__ FinishColumns(const FinishArgs& args, int block_, int nblocks_)
      : a(args), block(block_), nblocks(nblocks_), lane(threadIdx.x & 63), wave(__builtin_amdgcn_readfirstlane(threadIdx.x >> 6)),
        C(static_cast<uint32_t>(args.C)), Cw(static_cast<uint32_t>(args.Cw)), c_log2((C & (C - 1u)) == 0u ? 31 - __builtin_clz(C) : -1),
        same_layout(args.Cw == args.C) {}

  __device__ uint32_t div_c(uint32_t x) const { return c_log2 >= 0 ? x >> c_log2 : x / C; }
  __device__ long long column(int v) const { return (static_cast<long long>(v) * nblocks + block) * 64 + lane; }
  __device__ long long out_col(long long col) const {
    if constexpr (kPlanes) {
      const uint32_t rt = div_c(static_cast<uint32_t>(col)), c = static_cast<uint32_t>(col) - rt * C, kg = rt / 9u, tap = rt - kg * 9u;
      return static_cast<long long>(((kg * 4u + (c & 3u)) * 9u + tap) * (C >> 2) + (c >> 2));
    } else {
      return col;
    }
  }

  // Adds the slices: `fin` are the sums of this wavefront's columns (after the fp32 round trip where asked), wold their old weights.
  // any_wide (uniform): some workgroup wrote the third plane (top bytes) of its part of its slice.  Returns the wavefront's largest magnitude.
  __device__ __forceinline__ uint32_t gather(FinishShared<NW>& sh, const bool any_wide) {
    const __amdgpu_buffer_rsrc_t rpart =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<int32_t*>(a.partial), 0, kPlanes ? static_cast<int>(a.slice_stride * a.splits * 4) : 0, 0x00020000);
    constexpr int kSc1 = 16;   // cache policy bit: coherent across the dies' L2 caches
    const int units = static_cast<int>(a.nv);
    // kMixed = false: no workgroup wrote a third plane, every sum is the sign-extended 24-bit value
    auto slice_col = [&](auto mixed, int z, long long col) -> v4i {
      if constexpr (kPlanes) {
        const int zoff = __builtin_amdgcn_readfirstlane(static_cast<int>(z * a.slice_stride * 4));   // z is the same in all lanes
        const v2u lo = __builtin_amdgcn_raw_buffer_load_b64(rpart, static_cast<int>(col) * 8, zoff, kSc1);
        const uint32_t mid = __builtin_amdgcn_raw_buffer_load_b32(rpart, units * 8 + static_cast<int>(col) * 4, zoff, kSc1);
        v4i r;   // biased sums, 24 bits each
        r[0] = static_cast<int>(__builtin_amdgcn_perm(mid, lo[0], 0x0C040100u));   // 0, mid.b0, lo.b1, lo.b0
        r[1] = static_cast<int>(__builtin_amdgcn_perm(mid, lo[0], 0x0C050302u));
        r[2] = static_cast<int>(__builtin_amdgcn_perm(mid, lo[1], 0x0C060100u));
        r[3] = static_cast<int>(__builtin_amdgcn_perm(mid, lo[1], 0x0C070302u));
        if constexpr (decltype(mixed)::value) {   // rare: the writer of this column's tile in slice z tells whether it wrote top bytes
          const uint32_t rt = static_cast<uint32_t>(col) / C;   // kg * 9 + t
          const uint32_t tile = (rt / 9u >> 5) + static_cast<uint32_t>(a.tiles_k) * ((static_cast<uint32_t>(col) - rt * C) >> 5);
          const bool wide = __hip_atomic_load(a.wide + tile + static_cast<uint32_t>(a.tiles_k * a.tiles_c) * static_cast<uint32_t>(z), __ATOMIC_RELAXED,
                                              __HIP_MEMORY_SCOPE_AGENT) != 0u;
          uint32_t hi = 0;
          if (wide) hi = __builtin_amdgcn_raw_buffer_load_b32(rpart, units * 12 + static_cast<int>(col) * 4, zoff, kSc1);
#pragma unroll
          for (int e = 0; e < 4; ++e) r[e] = static_cast<int>(static_cast<uint32_t>(r[e]) | ((hi >> (8 * e)) << 24));
        }
        return r;
      } else {
        return reinterpret_cast<const v4i*>(a.partial + z * a.slice_stride)[col];
      }
    };
    // the old weights are requested first: they depend on nothing and are wanted right after the sums
#pragma unroll
    for (int j = 0; j < OWN; ++j) {
      const int v = j * NW + wave;
      const long long col = column(v);
      wold[j] = (same_layout && v < V && col < a.nv) ? reinterpret_cast<const uint32_t*>(a.w)[out_col(col)] : 0u;
    }
    uint32_t lmax = 0;
    auto complete = [&](v4i s) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (a.roundtrip) s[e] = f32_roundtrip(s[e]);
        const uint32_t u = uabs(s[e]);
        lmax = u > lmax ? u : lmax;
      }
      return s;
    };
    // Every wavefront has columns of its own at least in the first round (uniform over the grid): then each adds all
    // slices of its own columns and nothing goes through LDS.  With fewer columns than wavefronts the slices are
    // shared instead (phases 1 and 2 below), so that no wavefront idles while another walks over all slices.
    const bool direct = a.nv >= static_cast<long long>(NW) * nblocks * 64;
    // the whole gathering phase exists twice, so that the usual case (no third plane anywhere) has no branch between
    // its loads and keeps them all in flight
    const int bias_total = kPlanes ? static_cast<int>(static_cast<uint32_t>(a.splits) * kPartialBias) : 0;   // modulo 2^32, as the sums
    auto add_slices = [&](auto mixed) {
      if (direct) {
#pragma unroll
        for (int j = 0; j < OWN; ++j) {
          const int v = j * NW + wave;
          const long long col = column(v);
          v4i s = {0, 0, 0, 0};
          if (v < V && col < a.nv) {
            int z = 0;
            for (; z + 3 < a.splits; z += 4) {
              const v4i v0 = slice_col(mixed, z + 0, col);
              const v4i v1 = slice_col(mixed, z + 1, col);
              const v4i v2 = slice_col(mixed, z + 2, col);
              const v4i v3 = slice_col(mixed, z + 3, col);
              s += (v0 + v1) + (v2 + v3);
            }
            for (; z < a.splits; ++z) s += slice_col(mixed, z, col);
            s -= bias_total;
          }
          fin[j] = complete(s);
        }
      } else {
        v4i sum[VS];
        // phase 1: every wavefront adds its share of the slices for all of the workgroup's columns
#pragma unroll
        for (int v = 0; v < VS; ++v) {
          const long long col = column(v);
          v4i s = {0, 0, 0, 0};
          if (col < a.nv) {
            int z = wave;
            for (; z + 3 * NW < a.splits; z += 4 * NW) {
              const v4i v0 = slice_col(mixed, z + 0 * NW, col);
              const v4i v1 = slice_col(mixed, z + 1 * NW, col);
              const v4i v2 = slice_col(mixed, z + 2 * NW, col);
              const v4i v3 = slice_col(mixed, z + 3 * NW, col);
              s += (v0 + v1) + (v2 + v3);
            }
            for (; z < a.splits; z += NW) s += slice_col(mixed, z, col);
          }
          sum[v] = s;
        }
        // phase 2: column v is completed by wavefront v % NW (two LDS buffers in turn: one barrier per column)
#pragma unroll
        for (int v = 0; v < VS; ++v) {
          if (static_cast<long long>(v) * nblocks * 64 >= a.nv) continue;  // uniform over the grid: nothing at this stride
          sh.part[v & 1][wave][lane] = sum[v];
          __syncthreads();
          if (wave == v % NW) {
            v4i s = sh.part[v & 1][0][lane];
#pragma unroll
            for (int w = 1; w < NW; ++w) s += sh.part[v & 1][w][lane];
            if (column(v) < a.nv) s -= bias_total;
            fin[v / NW] = complete(s);
          }
        }
      }
    };
    if (kPlanes && any_wide) add_slices(std::true_type{});
    else add_slices(std::false_type{});
    // kPlanes: a lane holds four output channels of one input channel, its quad four consecutive input channels: a
    // 4 x 4 transposition inside the quad (two rounds of swaps) gives every lane four input channels of one output
    // channel, the form of the weights in memory, and out_col the column that is (quads lie inside one row: C % 4 == 0)
    if constexpr (kPlanes) {
      const bool odd1 = (lane & 1) != 0, odd2 = (lane & 2) != 0;
#pragma unroll
      for (int j = 0; j < OWN; ++j) {
        v4i s = fin[j], x;
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = __builtin_amdgcn_mov_dpp(s[e ^ 1], 0xB1, 0xf, 0xf, true);   // quad_perm:[1,0,3,2]
#pragma unroll
        for (int e = 0; e < 4; ++e) s[e] = (((e & 1) != 0) == odd1) ? s[e] : x[e];
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = __builtin_amdgcn_mov_dpp(s[e ^ 2], 0x4E, 0xf, 0xf, true);   // quad_perm:[2,3,0,1]
#pragma unroll
        for (int e = 0; e < 4; ++e) s[e] = (((e & 2) != 0) == odd2) ? s[e] : x[e];
        fin[j] = s;
      }
    }
    return wave_max_u32(lmax);
  }

  // the workgroup's largest magnitude (in every wavefront), published in its slot
  __device__ uint32_t publish(FinishShared<NW>& sh, uint32_t wave_max) const {
    if (lane == 0) sh.wmax[wave] = wave_max;
    __syncthreads();
    uint32_t bmax = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) bmax = max(bmax, sh.wmax[w]);
    if (wave == 0 && lane == 0)
      __hip_atomic_store(slot_word(a.sync + kFinishSlot0, block), bmax + 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return bmax;
  }

  // where the four weights of column `col` lie in the forward copy
  __device__ uint32_t* copy_word(long long col) const {
    const uint32_t e0 = static_cast<uint32_t>(col) * 4u, rt = div_c(e0), c0 = e0 - rt * C;
    const uint32_t k = rt / 9u, tap = rt - k * 9u;
    return reinterpret_cast<uint32_t*>(a.wprep + filter_copy_at(((k >> 6) * ((C + 31u) >> 5) + (c0 >> 5)) * 9u + tap, k & 63u, c0));
  }

  // Every wavefront rounds its columns and updates their weights (element counts fit 31 bits: host check).  dw is stored the first time only.
  // shift: the same in every lane, but it has come through LDS or memory, which the compiler cannot know - as a scalar
  // the choices below are scalar branches instead of both sides under execution masks
  __device__ __forceinline__ void update(int shift_any, bool first) const {
    const int shift = __builtin_amdgcn_readfirstlane(shift_any);
    const bool trunc = a.trunc != 0;
    const bool psto = a.method == NITI_ROUND_PSEUDO_STOCHASTIC;
#pragma unroll
    for (int j = 0; j < OWN; ++j) {
      const int v = j * NW + wave;
      if (v >= V) continue;
      const long long gcol = column(v);
      if (gcol >= a.nv) continue;
      const long long col = out_col(gcol);
      const v4i s = fin[j];
      if (first && a.dw != nullptr) reinterpret_cast<v4i*>(a.dw)[col] = s;
      uint32_t wnew = 0;   // the four updated weights (zero where the gradient column is channel padding)
      const v4i r = rounded4(s, shift, psto, trunc);
      if (same_layout) {
        uint32_t gp;
        wnew = updated4(wold[j], r, gp);
        reinterpret_cast<uint32_t*>(a.w)[col] = wnew;
        if (a.g8 != nullptr) reinterpret_cast<uint32_t*>(a.g8)[col] = gp;
      } else {   // applied once only (the old weights are read here)
        const uint32_t e0 = static_cast<uint32_t>(col) * 4u, rt = div_c(e0), c0 = e0 - rt * C;   // rt = k * 9 + tap
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (c0 + e < Cw) {
            const uint32_t wi = rt * Cw + c0 + e;
            const int wn = clip127(static_cast<int>(a.w[wi]) - r[e]);
            a.w[wi] = static_cast<int8_t>(wn);
            wnew |= (static_cast<uint32_t>(wn) & 0xFFu) << (8 * e);
            if (a.g8 != nullptr) a.g8[wi] = static_cast<int8_t>(r[e]);
          }
        }
      }
      if (a.wprep != nullptr) *copy_word(col) = wnew;
    }
  }
};

// The finishing pass of workgroup `block` out of `nblocks`.
// predicted_raw: the word read from a.shift_out (or anything when there is no prediction) at kernel start.
// With a predicted shift (a.predict) the update is applied before the range is final, so that its stores overlap
// the wait for the other workgroups, and applied once more from the same old weights if the final shift differs.
template <int NW, int V, bool kPlanes = false>
__device__ __forceinline__ void finish_columns(const FinishArgs& a, const int block, const int nblocks, FinishShared<NW>& sh,
                                               const int predicted_raw, const bool any_wide = false) {
  FinishColumns<NW, V, kPlanes> cols(a, block, nblocks);
  const uint32_t bmax = cols.publish(sh, cols.gather(sh, any_wide));
  const bool has_prediction = a.predict != 0 && a.shift_out != nullptr;
  const bool speculate = a.predict != 0 && cols.same_layout && nblocks > 1;
  int applied = -1;
  if (speculate) {
    applied = max(max(bitwidth_of(bmax, a.bw_mode) - a.target_bits, 0), has_prediction ? predicted_raw : 0);
    cols.update(applied, true);
  }
  if (cols.wave == 0) {
    const uint32_t g = wait_slots(a.sync + kFinishSlot0, nblocks, a.spin_limit, kPlanes ? &a.sync[1] : a.flag, a.sticky, kPlanes ? kWaitRange : a.flag_code);
    if (cols.lane == 0) sh.gshare = g != 0u ? g - 1u : 0u;
  }
  __syncthreads();
  const uint32_t gmax = sh.gshare;
  const int shift = max(bitwidth_of(gmax, a.bw_mode) - a.target_bits, 0);
  if (block == 0 && threadIdx.x == 0) {
    a.sync[0] = gmax;
    if (a.shift_out != nullptr) *a.shift_out = shift;
    if (a.exp_out != nullptr)
      *a.exp_out = shift + (a.exp_a != nullptr ? *a.exp_a : 0) + (a.exp_b != nullptr ? *a.exp_b : 0);
  }
  if (shift != applied) {
    if (applied >= 0) __builtin_amdgcn_s_waitcnt(0);   // the first update's stores leave before those that replace them
    cols.update(shift, applied < 0);
  }
}

// ---- the same along with the data gradient ---------------------------------------------------------------------
// (conv3x3_k64_backward.hip) `nblocks` workgroups of the data gradient's launch add the slices and update the weights: workgroups of
// their own that share the units with those that multiply, or where these fill the device the later ones of them (pair_plan), before their first stage.
// Loads on a unit that multiplies wait behind its stages' (36 loads a wavefront in batches of eight took 10 to 15 us, where a trip to
// memory is 2): a lane takes two units of a slice at a time (16 + 8 bytes) and has its loads - 9 to 12 at the usual 9216 unit slices
// per workgroup - in flight together.  The sums are added up in LDS.  A half-wave works on a chunk of 64 units, the sixteen of them on
// 16 / groups chunks x `groups` shares of the slices.  The input channels are a multiple of 64, so that a chunk is 64 of them
// for four output channels and one tap.
constexpr int kAlongBatch = 12;   // loads in flight together
inline constexpr size_t along_lds(int own) { return 64 + static_cast<size_t>(own) * 1280; }

struct AlongWork {
  int nblocks;       // workgroups that take part
  int own;           // chunks of a workgroup at most; its chunk l is chunk l * nblocks + block
  int groups_log2;   // shares the slices of a chunk are cut into
  int loads;         // of a lane
};
inline AlongWork along_work(long long units, int splits, int nblocks) {
  AlongWork best{nblocks, static_cast<int>(((units + 63) / 64 + nblocks - 1) / nblocks), 0, 0};
  for (int g = 0; g <= 4; ++g) {
    const int sets = 16 >> g;
    const int loads = (best.own + sets - 1) / sets * ((splits + (1 << g) - 1) >> g);
    if (best.loads == 0 || loads < best.loads) {
      best.groups_log2 = g;
      best.loads = loads;
    }
  }
  return best;
}

// Layouts alike, C a multiple of 64, no int32 gradient, planes from an earlier launch, nblocks > 1: host check.
// kItems: words of weights a thread has at most (own <= 8 kItems).  kStream: the slices' loads leave nothing in the caches.  That is the
// faster way where the sums take as long as the products beside them: 128 images of 8 x 8, 256 -> 512 38.9 -> 36.2 us for both launches,
// 80 of 16 x 16, 128 -> 256 31.5 -> 29.2; where the products take longer they lose by it: 256 -> 256 48.3 -> 49.1, of 32 x 32, 128 -> 128 54.4 -> 55.2.
template <int kItems, bool kStream>
struct SumsAlong {
  const FinishArgs& a;
  const AlongWork& work;
  const int block;              // < 0: this workgroup takes no part
  int8_t* const lds;            // along_lds(own) bytes: words, sums, old weights
  const int lane, wave;
  int guessed;
  uint32_t wnew[kItems];

  __device__ SumsAlong(const FinishArgs& args, const AlongWork& w, int block_, int8_t* lds_, int thread = threadIdx.x)
      : a(args), work(w), block(block_), lds(lds_), lane(thread & 63), wave(__builtin_amdgcn_readfirstlane(thread >> 6)) {}

  __device__ int* sums(int l, int e, int unit) const { return reinterpret_cast<int*>(lds + 64) + (l * 4 + e) * 64 + unit; }   // [chunk][output channel of the unit][unit]
  // 0 largest magnitude, 1 wavefronts that have folded theirs in, 2 range, 3 the data gradient's range, 4 predicted shift
  __device__ uint32_t* words() const { return reinterpret_cast<uint32_t*>(lds); }

  __device__ uint32_t* old_word(int j) const { return reinterpret_cast<uint32_t*>(lds + 64 + work.own * 1024) + item_own(j) * 64 + lane; }   // of item j

  // A chunk's four output channels, tap and first input channel; the same in all lanes
  struct Place {
    uint32_t k, tap, c;
  };
  __device__ Place place(int chunk) const {
    const uint32_t per_row = static_cast<uint32_t>(a.C) >> 6, ch = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(chunk));
    const uint32_t rt = (per_row & (per_row - 1u)) == 0u ? ch >> (31 - __builtin_clz(per_row)) : ch / per_row, kg = rt / 9u;
    return {kg * 4u, rt - kg * 9u, (ch - rt * per_row) * 64u};
  }
  // Item j of a thread is four input channels of one output channel of this chunk (the first wavefronts, which wait for the ranges, have the
  // last ones).
  __device__ int item_own(int j) const { return j * 8 + 7 - wave; }
  __device__ int item_chunk(int j) const { return item_own(j) * work.nblocks + block; }
  __device__ bool has_item(int j) const { return item_own(j) < work.own && item_chunk(j) * 64 < static_cast<int>(a.nv); }
  __device__ uint32_t item_word(int j) const {   // of the weights
    const Place p = place(item_chunk(j));
    return (((p.k + (static_cast<uint32_t>(lane) >> 4)) * 9u + p.tap) * static_cast<uint32_t>(a.C) + p.c >> 2) + (static_cast<uint32_t>(lane) & 15u);
  }
  __device__ uint32_t* item_copy(int j) const {   // in the forward copy
    const Place p = place(item_chunk(j));
    const uint32_t q = static_cast<uint32_t>(lane) & 15u, row = (p.k & 63u) + (static_cast<uint32_t>(lane) >> 4);
    const uint32_t block64 = ((p.k >> 6) * (static_cast<uint32_t>(a.C) >> 5) + (p.c >> 5) + (q >> 3)) * 9u + p.tap;
    return reinterpret_cast<uint32_t*>(a.wprep + filter_copy_at(block64, row, q * 4u));
  }
  __device__ v4i item(int j) const {
    v4i s = *reinterpret_cast<const v4i*>(sums(item_own(j), lane >> 4, 4 * (lane & 15))) - static_cast<int>(static_cast<uint32_t>(a.splits) * kPartialBias);   // modulo 2^32
    if (a.roundtrip) {
#pragma unroll
      for (int e = 0; e < 4; ++e) s[e] = f32_roundtrip(s[e]);
    }
    return s;
  }

  // Adds the slices in LDS.  Every wavefront's additions are done, and what it wrote to LDS is there, behind the next barrier.
  __device__ __forceinline__ void begin() {
    if (block < 0) return;
    const int G = 1 << work.groups_log2, sets = 16 >> work.groups_log2, steps = (a.splits + G - 1) >> work.groups_log2;
    const int half = wave * 2 + (lane >> 5), group = half & (G - 1), set = half >> work.groups_log2;
    const int pair = 2 * (lane & 31), units = static_cast<int>(a.nv), stride = static_cast<int>(a.slice_stride * 4);
    const __amdgpu_buffer_rsrc_t planes = __builtin_amdgcn_make_buffer_rsrc(const_cast<int32_t*>(a.partial), 0, stride * a.splits, 0x00020000);
    // Load i of a lane is step i % steps of the slices in round i / steps of the chunks.  Past the last slice it is out of range (zeros).
    const int unit = (set * work.nblocks + block) * 64 + pair;
    int ask_step = 0, ask_round = 0;
    v4i low[kAlongBatch];
    v2u mid[kAlongBatch];
    auto request = [&] {
#pragma unroll
      for (int i = 0; i < kAlongBatch; ++i) {
        const int z = group + ask_step * G, u = unit + ask_round * sets * work.nblocks * 64;
        const bool real = z < a.splits && u < units;
        low[i] = __builtin_amdgcn_raw_buffer_load_b128(planes, real ? z * stride + u * 8 : -1, 0, kStream ? 2 : 0);
        mid[i] = __builtin_amdgcn_raw_buffer_load_b64(planes, real ? z * stride + units * 8 + u * 4 : -1, 0, kStream ? 2 : 0);
        if (++ask_step == steps) {
          ask_step = 0;
          ++ask_round;
        }
      }
    };
    request();
    const uint32_t any_wide = a.wide[a.tiles_k * a.tiles_c * a.splits + opaque_zero()];
    const bool has_prediction = a.predict != 0 && a.shift_out != nullptr;
    const int predicted_raw = __hip_atomic_load((has_prediction ? a.shift_out : reinterpret_cast<const int32_t*>(a.sync)) + opaque_zero(), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __builtin_amdgcn_sched_barrier(0);
    uint32_t wold[kItems];
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
      wold[j] = 0;   // (the load is not under a lane's condition: it would be waited for on the spot)
      if (j * 8 < work.own) wold[j] = reinterpret_cast<const uint32_t*>(a.w)[has_item(j) ? item_word(j) : 0u];
    }
    for (int i = threadIdx.x; i < work.own * 64; i += 512) *reinterpret_cast<v4i*>(sums(0, 0, 4 * i)) = v4i{0, 0, 0, 0};
    if (threadIdx.x < 2) words()[threadIdx.x] = 0u;
    __syncthreads();
    auto fold = [&](int l, v4i x0, v4i x1) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        __hip_atomic_fetch_add(sums(l, e, pair), x0[e], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        __hip_atomic_fetch_add(sums(l, e, pair + 1), x1[e], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      }
    };
    int got_step = 0, got = set;
    v4i s0 = {0, 0, 0, 0}, s1 = {0, 0, 0, 0};
    for (int left = work.loads;;) {
#pragma unroll
      for (int i = 0; i < kAlongBatch; ++i) {
        const uint32_t m0 = mid[i][0], m1 = mid[i][1];
        const uint32_t l0 = static_cast<uint32_t>(low[i][0]), l1 = static_cast<uint32_t>(low[i][1]), l2 = static_cast<uint32_t>(low[i][2]), l3 = static_cast<uint32_t>(low[i][3]);
        // biased sums, 24 bits each: 0, mid byte, two low bytes
        s0 += v4i{static_cast<int>(__builtin_amdgcn_perm(m0, l0, 0x0C040100u)), static_cast<int>(__builtin_amdgcn_perm(m0, l0, 0x0C050302u)),
                  static_cast<int>(__builtin_amdgcn_perm(m0, l1, 0x0C060100u)), static_cast<int>(__builtin_amdgcn_perm(m0, l1, 0x0C070302u))};
        s1 += v4i{static_cast<int>(__builtin_amdgcn_perm(m1, l2, 0x0C040100u)), static_cast<int>(__builtin_amdgcn_perm(m1, l2, 0x0C050302u)),
                  static_cast<int>(__builtin_amdgcn_perm(m1, l3, 0x0C060100u)), static_cast<int>(__builtin_amdgcn_perm(m1, l3, 0x0C070302u))};
        if (++got_step == steps) {
          if (got < work.own) fold(got, s0, s1);
          s0 = s1 = v4i{0, 0, 0, 0};
          got_step = 0;
          got += sets;
        }
      }
      if ((left -= kAlongBatch) <= 0) break;
      request();
    }
#pragma unroll
    for (int j = 0; j < kItems; ++j)
      if (item_own(j) < work.own) *old_word(j) = wold[j];
    if (threadIdx.x == 0) words()[4] = static_cast<uint32_t>(predicted_raw);
    if (__any(any_wide != 0u)) {   // rare: top bytes, from the workgroups that wrote some
      for (int l = set; l < work.own; l += sets) {
        const int u = (l * work.nblocks + block) * 64 + pair;
        if (u >= units) break;
        const uint32_t C = static_cast<uint32_t>(a.C), rt = static_cast<uint32_t>(u) / C;   // kg * 9 + t
        const uint32_t tile = (rt / 9u >> 5) + static_cast<uint32_t>(a.tiles_k) * ((static_cast<uint32_t>(u) - rt * C) >> 5);
        for (int z = group; z < a.splits; z += G) {
          if (a.wide[tile + static_cast<uint32_t>(a.tiles_k * a.tiles_c * z)] == 0u) continue;
          const v2u hi = __builtin_amdgcn_raw_buffer_load_b64(planes, z * stride + units * 12 + u * 4, 0, 0);
          fold(l, v4i{static_cast<int>(hi[0] << 24), static_cast<int>(hi[0] >> 8 << 24), static_cast<int>(hi[0] >> 16 << 24), static_cast<int>(hi[0] >> 24 << 24)},
               v4i{static_cast<int>(hi[1] << 24), static_cast<int>(hi[1] >> 8 << 24), static_cast<int>(hi[1] >> 16 << 24), static_cast<int>(hi[1] >> 24 << 24)});
        }
      }
    }
  }

  // All sums in LDS: the gradient's slot, filled by the wavefront that comes last.
  __device__ __forceinline__ void publish() {
    if (block < 0) return;
    uint32_t lmax = 0;
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
      if (j * 8 >= work.own || !has_item(j)) continue;   // uniform
      const v4i s = item(j);
#pragma unroll
      for (int e = 0; e < 4; ++e) lmax = max(lmax, uabs(s[e]));
    }
    lmax = wave_max_u32(lmax);
    if (lane == 0) {
      __hip_atomic_fetch_max(&words()[0], lmax, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      // (LDS operations of one wavefront are carried out in order)
      if (__hip_atomic_fetch_add(&words()[1], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) == 7u)
        __hip_atomic_store(slot_word(a.sync + kFinishSlot0, block), __hip_atomic_load(&words()[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) + 1u, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    }
  }

  // New weights with this shift; the copy is left for later.
  __device__ __forceinline__ void round_items(int shift) {
    const bool trunc = a.trunc != 0, psto = a.method == NITI_ROUND_PSEUDO_STOCHASTIC;
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
      wnew[j] = 0;
      if (j * 8 >= work.own || !has_item(j)) continue;   // uniform
      const v4i s = item(j);
      const v4i r = rounded4(s, shift, psto, trunc);
      uint32_t gp;
      wnew[j] = updated4(*old_word(j), r, gp);
      const uint32_t word = item_word(j);
      reinterpret_cast<uint32_t*>(a.w)[word] = wnew[j];
      if (a.g8 != nullptr) reinterpret_cast<uint32_t*>(a.g8)[word] = gp;
    }
  }
  __device__ int shift_of(uint32_t gmax) const { return __builtin_amdgcn_readfirstlane(max(bitwidth_of(gmax, a.bw_mode) - a.target_bits, 0)); }

  // While the slots fill: the weights with the predicted shift, or what the sums seen so far need (put right in settle)
  __device__ __forceinline__ void guess() {
    if (block < 0) return;
    guessed = a.predict != 0 && a.shift_out != nullptr ? max(__builtin_amdgcn_readfirstlane(static_cast<int>(words()[4])), 0)
                                                       : shift_of(__hip_atomic_load(&words()[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
    round_items(guessed);
  }
  // A wavefront's wait for the gradient's range; a barrier follows.  One that gives up says so in the words of the data gradient `first`, the
  // first of the call's (and its limit is the one that counts: kernel arguments of which fewer stay in registers.  With a pointer for
  // the flag among FinishArgs 128 images of 32 x 32, 128 -> 128 took 52.1 us backward, 51.2 this way).
  template <class First>
  __device__ __forceinline__ void wait(int waiter, const First& first) const {
    if (block < 0 || wave != waiter) return;
    const uint32_t g = wait_slots(a.sync + kFinishSlot0, work.nblocks, first.spin_limit, &first.sync[1], first.sticky, kWaitUpdate);
    if (lane == 0) words()[2] = g != 0u ? g - 1u : 0u;
  }
  // Behind it: the weights are right.
  __device__ __forceinline__ void settle() {
    const int shift = shift_of(words()[2]);
    if (shift == guessed) return;
    __builtin_amdgcn_s_waitcnt(0);   // the first stores leave before those that replace them
    round_items(shift);
  }
  // Every workgroup of the data gradient has read the copy of the filter (its slot is filled): it changes.  The gradient's exponent
  // builds on the error's, whose shift and exponents these are.
  __device__ __forceinline__ void store_copy(int error_shift, const int32_t* exp_a, const int32_t* exp_b) const {
#pragma unroll
    for (int j = 0; j < kItems; ++j)
      if (j * 8 < work.own && has_item(j)) *item_copy(j) = wnew[j];
    if (block == 0 && threadIdx.x == 0) {
      const uint32_t gmax = words()[2];
      const int shift = shift_of(gmax);
      a.sync[0] = gmax;
      if (a.shift_out != nullptr) *a.shift_out = shift;
      if (a.exp_out != nullptr)
        *a.exp_out = shift + max(error_shift, 0) + (exp_a != nullptr ? *exp_a : 0) + (exp_b != nullptr ? *exp_b : 0) + (a.exp_b != nullptr ? *a.exp_b : 0);
    }
  }

  // In a workgroup that multiplies as well, behind the error's range
  template <class First>
  __device__ __forceinline__ void wait(const First& first) const { wait(1, first); }
  __device__ __forceinline__ void update(int error_shift, const int32_t* exp_a, const int32_t* exp_b) {
    if (block < 0) return;
    settle();
    store_copy(error_shift, exp_a, exp_b);
  }
};

// A workgroup that does nothing else, beside the `first_blocks` ones of the data gradient `first`
template <int kItems, bool kStream, class First>
__device__ __forceinline__ void finish_beside(SumsAlong<kItems, kStream> along, const First& first, uint32_t* first_slots, const int first_blocks) {
  along.begin();
  __syncthreads();
  // from here on few instructions, all of them on the way to the range (the loads in front would hold up the other workgroup's)
  __builtin_amdgcn_s_setprio(3);
  along.publish();
  along.guess();
  along.wait(0, first);
  __syncthreads();
  along.settle();
  if (along.wave == 0) {
    // one slot at first: the others are looked at when the data gradient is about to end
    wait_slots(slot_word(first_slots, along.block % first_blocks), 1, first.spin_limit, &first.sync[1], first.sticky, kWaitUpdate);
    const uint32_t f = wait_slots(first_slots, first_blocks, first.spin_limit, &first.sync[1], first.sticky, kWaitUpdate);
    if (along.lane == 0) along.words()[3] = f != 0u ? f - 1u : 0u;
  }
  __syncthreads();
  along.store_copy(bitwidth_of(along.words()[3], first.bw_mode) - first.target_bits, first.exp_a, first.exp_b);
}

}  // namespace
}  // namespace niti
