// int8 3x3 / stride 1 / pad 1 convolution with the activation halo tile in LDS (see conv3x3_halo.hip), on
// v_mfma_i32_16x16x64_i8: 64 input channels per product instead of 32.
//
// Why this instruction: the matrix units are power-limited on random operands, and a 16 x 16 x 64 product moves half
// the accumulator bytes of a 32 x 32 x 32 one per operation.  A register-resident loop (probe.hip) sustains 3.9 to 4.1 POP/s at 2.0 GHz on
// uniform random int8 where the 32 x 32 x 32 form sustains 3.5 at 1.75, and with two workgroups on a compute unit (four wavefronts per
// matrix unit taking turns) 3.9 to 4.1 against 2.5 to 3.0.
//
// A workgroup owns 256 consecutive output pixels x KT output channels (128, 64 or 32) and walks over the input channels in
// slices of 64.  8 wavefronts: 4 pixel groups of 64 x 2 channel groups of KT/2 (KT = 32: 8 pixel groups of 32).  Of 32
// consecutive pixels a lane of 16 holds an even and an odd one in two fragments: the right-hand neighbours of the even pixels
// are then the odd fragment as it stands and the left-hand ones of the odd pixels the even fragment, so that a filter row needs
// two shifted fragments per 32 pixels (one DPP AND per register) instead of four.
//
// LDS: activation slices in two buffers, [even columns][odd columns][64 bytes], 16-byte pieces XOR-swizzled by the slot so that
// the 16 slots of a fragment read fall into all banks; the filter through a ring of stages - one tap of 128 channels (8 KB),
// or a filter row (24 / 12 / 6 KB).
// Launch time against the kernel of 32-channel slices (128 images, forward / data gradient, rounded, us, replayed graphs of launches
// on operands in turn): 128 -> 128 at 32 x 32 23.1 / 22.1 -> 21.3 / 20.6; 128 -> 256 at 16 x 16 14.8 / 12.7 -> 12.2 / 12.1;
// 256 -> 256 21.6 / 22.1 -> 18.0 / 18.2; 256 -> 512 at 8 x 8 12.0 / 14.6 -> 11.4 / 12.5; 512 -> 512 19.9 / 20.0 -> 17.6 / 17.7.  What
// bounds it now: of 18 us at 256 -> 256, 12.5 are the loop (products alone 8.8 at 2.1 GHz), 1.2 the way to the first stage, 4 the
// range exchange, rounding and stores behind the last product.
//
// The number of loads a wavefront has in flight at any point is a compile-time constant: loads behind the last slice go to
// out-of-range offsets (zeros, no memory traffic), surplus activation loads to a dump slot.
#pragma once
#include <utility>

#include "conv3x3_epilogue.h"

namespace niti {
namespace {

// PER_CU: workgroups per compute unit the kernel is made for.  One (launches of at most as many workgroups as units): a stage is
// a filter row, the ring four or five deep.  Two: <= 80 KB and <= 128 registers, so that stages are single taps at 128 channels.
template <int Q, int BR, int NI, int KT, int PER_CU>
struct KGeom {
  static constexpr int PX = BR * NI * Q;                  // output pixels per workgroup
  static constexpr int HR = BR + 2;
  static constexpr int HALF = NI * HR * (Q / 2);          // slots of one column parity
  static constexpr int ACT_INSTR = 2 * HALF / 16;         // one instruction fills 16 slots
  static constexpr int ACT_BYTES = ACT_INSTR * 1024;
  static constexpr int ACT_LOADS = (ACT_INSTR + 7) / 8;   // per wavefront per slice
  static constexpr int PT = KT == 32 ? 1 : 2;             // 32-pixel tiles per wavefront
  static constexpr int NWF = KT == 128 ? 2 : 1;           // 32-channel tiles per wavefront
  static constexpr int TPS = (PER_CU == 2 && (KT == 128 || Q == 4)) ? 1 : 3;   // taps per filter stage
  static constexpr int S = 9 / TPS;                       // stages per slice
  static constexpr int W_INSTR = TPS * KT / 16;
  static constexpr int WL = (W_INSTR + 7) / 8;            // filter loads per wavefront per stage
  static constexpr int W_BYTES = W_INSTR * 1024;
  // stages in the ring
  static constexpr int R = PER_CU == 1 ? (KT == 128 ? 4 : 5) : (KT == 128 ? (Q == 4 ? 3 : 4) : (Q == 4 ? 6 : 3));
  static constexpr bool AHEAD = PER_CU == 1 || (KT == 128 && R >= 4);   // fragments of the next stage are read in front of its barrier
  static constexpr int NBUF = KT == 128 ? 2 : 3;          // filter fragment buffers: the units of a slice (18 or 9) are a multiple
  static constexpr int TILE_BYTES = 2 * ACT_BYTES + R * W_BYTES;
  static constexpr int LDS_BYTES = TILE_BYTES + 1024 + 64;   // + dump slot, reduction words
  static_assert(PX == 256, "a workgroup owns 256 output pixels");
  static_assert(PER_CU == 1 || KT >= 64, "the narrowest tile is for launches that leave units idle");
  static_assert(2 * HALF % 16 == 0, "whole load instructions");
  static_assert(KT != 32 || Q <= 16, "the 32-channel tile's wavefronts own 32 pixels: whole 2 x 2 windows only up to 16-pixel rows");
  static_assert(NI == 1 || BR == Q, "several images per workgroup only as whole images");
  static_assert(PER_CU * LDS_BYTES <= 160 * 1024, "workgroups per compute unit");
  // activation loads of the next slice that stage u of a slice issues, in front of its filter loads
  static constexpr int act_in_stage(int u) { return S == 3 ? (u == 0 ? ACT_LOADS : 0) : (u < ACT_LOADS ? 1 : 0); }
  static constexpr int act_before(int u) {
    int n = 0;
    for (int i = 0; i < u; ++i) n += act_in_stage(i);
    return n;
  }
  // Loads that may still be in flight when stage u of a slice starts: those younger than everything the stage (or, with
  // AHEAD, also the first reads of the next one) needs.  Order: activations of slice 0, filter stages 0 .. R-2; stage t: its
  // activation loads, then filter stage t + R - 1.
  static constexpr int in_flight(int u, bool first_slice) {
    const int t = S * 4 + u;                        // some stage far from the start
    const int start = first_slice ? S * 4 : 0;      // stages before it do not exist
    const int need_w = t + (AHEAD ? 1 : 0);
    const bool need_act = u == 0 || (AHEAD && u == S - 1);   // the loads of that slice: issued in the S stages before its first
    const int act_slice = u == 0 ? t / S : t / S + 1;
    int n = 0;
    for (int s = t - 1; s >= 0; --s) {
      if (s < start) break;
      if (s + R - 1 <= need_w) return n;
      n += WL;
      if (act_in_stage(s % S) > 0 && need_act && s / S + 1 == act_slice) return n;
      n += act_in_stage(s % S);
    }
    // the loads in front of the first stage: filter stages R-2 .. 0
    for (int s = start + R - 2; s >= start; --s) {
      if (s <= need_w) return n;
      n += WL;
    }
    return n;
  }
};

// the register quad g of a 32 x 32 tile: 16-channel half g / 2, column parity g % 2
struct Layout16 {
  static __device__ int channel(int g, int lane) { return 16 * (g >> 1) + 4 * (lane >> 4); }
  static __device__ int pixel(int g, int lane) { return 2 * (lane & 15) + (g & 1); }
};

// A fragment's four dwords from the neighbouring lane of the row of 16 (kLeft: the lane below, else the lane above; zero where
// there is none), and-ed with keep where kKeep.  Wait states as the compiler would place them are written out (it does not see
// inside): two in front (a vector instruction that wrote a source just before), two behind (a product that reads the result).
template <bool kLeft, bool kKeep>
__device__ inline v4i neighbour4(v4i x, int keep) {
  int r0, r1, r2, r3;
#define NITI_NEIGHBOUR(OP, ARG, DIR)                                                                  \
  asm("s_nop 1\n\t" OP " %0, %4" ARG " " DIR ":1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"       \
      OP " %1, %5" ARG " " DIR ":1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"                       \
      OP " %2, %6" ARG " " DIR ":1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"                       \
      OP " %3, %7" ARG " " DIR ":1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\ts_nop 1"                \
      : "=&v"(r0), "=&v"(r1), "=&v"(r2), "=&v"(r3)                                                    \
      : "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]), "v"(keep))
  if constexpr (kKeep) {
    if constexpr (kLeft) NITI_NEIGHBOUR("v_and_b32_dpp", ", %8", "row_shr");
    else NITI_NEIGHBOUR("v_and_b32_dpp", ", %8", "row_shl");
  } else {
    if constexpr (kLeft) NITI_NEIGHBOUR("v_mov_b32_dpp", "", "row_shr");
    else NITI_NEIGHBOUR("v_mov_b32_dpp", "", "row_shl");
  }
#undef NITI_NEIGHBOUR
  return v4i{r0, r1, r2, r3};
}

// d += a b, as inline assembly: with the builtin the compiler moves the accumulators between registers (destination unlike the
// third operand), and at the 128 registers of two workgroups per compute unit that ends in spills inside the loop.  The wait
// states it would add are the caller's: a vector instruction's result needs two before a product reads it (neighbour4 ends in
// them), and mfma_settle() stands between the last product and the first other use of a sum.
__device__ inline void mfma64(v4i& d, v4i a, v4i b) { asm volatile("v_mfma_i32_16x16x64_i8 %0, %1, %2, %0" : "+v"(d) : "v"(a), "v"(b)); }
__device__ inline void mfma_settle() { asm volatile("s_nop 15\n\ts_nop 15"); }

// (What is left: the StoShift instances for two workgroups per unit spill 6 registers at 64 channels and 17 or 18 at 128, and those that take
// several tiles in turn 2 to 11 (StoShift 7 to 25), none of them inside the loop; no other instance spills.)
// kWT: the filter operand is the forward copy of the filter of the convolution whose data gradient this launch computes; its
// blocks of 64 reduction channels x 32 outputs are transposed by ds_read_b64_tr_b8 when the fragments are read.
// kSto: StoShift on random integers read in the epilogue.
template <int Q, int BR, int NI, int KT, int PER_CU, bool kFused, bool kWT, bool kSto, class Along>
__device__ __forceinline__ void k64_tile(const HaloArgs& a, const HaloPlace at, int8_t* const smem, Along& along) {
  static_assert(kFused || !kSto);
  using G = KGeom<Q, BR, NI, KT, PER_CU>;
  constexpr int PT = G::PT, NWF = G::NWF, TPS = G::TPS, S = G::S, R = G::R, WL = G::WL;
  int8_t* const dump = smem + G::TILE_BYTES;

  const int tid = along.thread();
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int pixbase = at.x * G::PX;  // first output pixel of this workgroup in [N*Q*Q]
  const int kt = at.y;
  const int n0 = pixbase / (Q * Q);
  const int p0 = (pixbase - n0 * (Q * Q)) / Q;

  const int settle_shift = along.again();   // the final shift, when this workgroup has to store its tile again
  along.begin();

  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(a.x), 0, a.x_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(a.wp), 0, a.wp_bytes, 0x00020000);

  ShiftHint hint{false, 0};
  if constexpr (kFused) hint = halo_shift_hint(a, settle_shift);

  const int nsl = (a.C + 63) >> 6;   // 64-channel slices
  const unsigned act_lds = lds_addr(smem), w_lds = lds_addr(smem + 2 * G::ACT_BYTES), dump_lds = lds_addr(dump);

  // ---- activation staging: an instruction fills 16 slots of 64 bytes; lane -> (slot lane/4, piece lane%4)
  int act_off[G::ACT_LOADS];   // byte offset of this lane's 16 bytes for channel slice 0, or kOobFar
#pragma unroll
  for (int i = 0; i < G::ACT_LOADS; ++i) {
    const int slot = (wave + 8 * i) * 16 + (lane >> 2);
    const int par = slot >= G::HALF ? 1 : 0;
    const int t = slot - par * G::HALF;
    const int row = t / (Q / 2), col = 2 * (t - row * (Q / 2)) + par;
    const int ni = row / G::HR, h = row - ni * G::HR;
    const int ih = p0 + h - 1;
    act_off[i] = (slot < 2 * G::HALF && n0 + ni < a.N && ih >= 0 && ih < Q) ? (((n0 + ni) * Q + ih) * Q + col) * a.C + ((lane & 3) ^ ((t >> 1) & 3)) * 16 : kOobFar;
  }
  auto issue_act = [&](int cs, int buf, auto ic) {
    constexpr int i = decltype(ic)::value;
    const unsigned dst = wave + 8 * i < G::ACT_INSTR ? act_lds + buf * G::ACT_BYTES + (wave + 8 * i) * 1024 : dump_lds;
    // Channels behind the last one (the next pixel's first ones, or zeros behind the map) meet zeros of the filter copy; a slice
    // behind the last one is not fetched.
    const int off = cs < nsl ? act_off[i] : kOobFar;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, NITI_LDS_AT(dst), 16, off, cs * 64, 0, 0);
  };

  // ---- filter staging.  The copy is [64-channel group][32-channel slice][tap][64 rows][32 bytes].  Instruction q of a stage
  // holds 1 KB of tap q / (KT/16) of the stage; within the tap
  //   forward: [64-row group (KT = 128)][slice parity][64 rows, as 2 x 32 (KT = 32: this tile's 32)][32 bytes]
  //   kWT:     [32-channel output slice][64 reduction rows, as 2 x 32][32 bytes]
  // A group or slice beyond the last one re-reads the last (its sums are never stored).
  // The copy swaps a row's 16-byte halves by row bit 3.  On the way to LDS (a lane may fetch any 16 bytes) that becomes no swap
  // for the forward pass and a swap by row bits 3 and 4 for kWT: with these all lanes of a fragment's read fall into
  // different banks (4 clocks a ds_read_b128 where the copy's own order takes 6).
  const int lane_src = (lane ^ ((kWT ? lane >> 5 : lane >> 4) & 1)) * 16;
  const int ngroups = (a.K + 63) / 64;
  int wsrc[WL];
#pragma unroll
  for (int i = 0; i < WL; ++i) {
    const int q = wave + 8 * i;
    const int x = q / (KT / 16), qq = q % (KT / 16);
    const int s = TPS == 3 ? (x == 0 ? 1 : (x == 1 ? 2 : 0)) : 0;   // taps of a row in the order they are multiplied: centre, right, left
    int off;
    if (kWT) {
      const int os = min(kt * (KT / 32) + (qq >> 1), a.src_cslices - 1);
      off = (os * 9 + (TPS == 3 ? 2 - s : 0)) * 2048 + (qq & 1) * 1024 + lane_src;
    } else if (KT == 32) {
      off = (min(kt >> 1, ngroups - 1) * a.cslices + qq) * (9 * 2048) + s * 2048 + (kt & 1) * 1024 + lane_src;
    } else {
      const int g = min(KT == 128 ? kt * 2 + (qq >> 2) : kt, ngroups - 1);
      off = (g * a.cslices + ((qq >> 1) & 1)) * (9 * 2048) + s * 2048 + (qq & 1) * 1024 + lane_src;
    }
    wsrc[i] = off;
  }
  // stage u of slice cs into ring slot st
  auto issue_w = [&](int cs, auto uc, unsigned st, auto ic) {
    constexpr int u = decltype(uc)::value, i = decltype(ic)::value;
    constexpr int r = TPS == 3 ? u : u / 3;
    constexpr int s = TPS == 3 ? 0 : (u % 3 == 0 ? 1 : (u % 3 == 1 ? 2 : 0));
    const int rel = kWT ? cs * a.src_cslices * (9 * 2048) + (TPS == 3 ? 6 - 3 * r : 8 - 3 * r - s) * 2048
                        : (cs * 2 * 9 + 3 * r + s) * 2048;
    const bool real = G::W_INSTR % 8 == 0 || wave + 8 * i < G::W_INSTR;
    const unsigned dst = real ? st + (wave + 8 * i) * 1024 : dump_lds;
    const int off = real && cs < nsl ? wsrc[i] : kOobFar;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, NITI_LDS_AT(dst), 16, off, cs < nsl ? rel : 0, 0, 0);
  };

  // The first loads leave before the fragment addresses below are worked out
  static_for<G::ACT_LOADS>([&](auto ic) { issue_act(0, 0, ic); });
  static_for<R - 1>([&](auto tc) {
    constexpr int t = decltype(tc)::value;
    static_for<WL>([&](auto ic) { issue_w(t / S, std::integral_constant<int, t % S>{}, w_lds + t * G::W_BYTES, ic); });
  });
  __builtin_amdgcn_sched_barrier(0);

  // ---- fragment addressing
  const int wp_ = KT == 32 ? wave : (wave & 3);   // group of 32 PT pixels
  const int wc = KT == 32 ? 0 : (wave >> 2);      // channel group of KT/2
  const int li = lane & 15, lk = lane >> 4;
  // kWT: x = 16-channel half of the output slice xor 8-row half of the reduction rows
  unsigned w_addr[kWT ? 2 : 1];
  if constexpr (kWT) {
#pragma unroll
    for (int x = 0; x < 2; ++x) w_addr[x] = w_lds + (KT == 128 ? wc * 4096 : (KT == 64 ? wc * 2048 : 0)) + lk * 512 + (li >> 1) * 32 + ((x ^ (lk & 1)) << 4) + 8 * (li & 1);
  } else {
    w_addr[0] = w_lds + (KT == 128 ? wc * 4096 : (KT == 64 ? wc * 1024 : 0)) + (lk >> 1) * (KT == 32 ? 1024 : 2048) + li * 32 + ((lk & 1) << 4);
  }
  constexpr int TAPB = KT * 64;                   // bytes of a tap inside a stage
  // activation fragment of filter row r, column parity 0.  The swizzle repeats every 8 slots: filter rows of maps of at least 16
  // pixels, the wavefront's further 32-pixel tiles (16 slots on) and images (Q = 8: 40 slots on) are constant offsets
  constexpr int PA = Q == 4 ? PT : 1, PR = Q >= 16 ? 1 : (Q == 8 ? 2 : 3);
  unsigned p_addr[PA][PR];
#pragma unroll
  for (int j = 0; j < PA; ++j) {
    const int pix = wp_ * (32 * PT) + j * 32 + 2 * li;
    const int prow = pix / Q;
    const int t0 = ((prow / BR) * G::HR + prow % BR) * (Q / 2) + (pix % Q) / 2;
#pragma unroll
    for (int r = 0; r < PR; ++r) {
      const int t = t0 + r * (Q / 2);
      p_addr[j][r] = act_lds + t * 64 + ((lk ^ ((t >> 1) & 3)) << 4);
    }
  }
  // is there a pixel to the left of the even one, to the right of the odd one (rows of 32: the shift itself brings in zeros)
  const int keep_l = Q < 32 && (2 * li) % Q == 0 ? 0 : -1;
  const int keep_r = Q < 32 && (2 * li + 1) % Q == Q - 1 ? 0 : -1;

  // results' mask bytes and pooling windows: requested in the last slice (PER_CU == 1), see HaloPieces
  constexpr bool kAhead = kFused && PER_CU == 1;
  using Pieces = HaloPieces<Q, KT, false, NWF, PT, PER_CU == 1>;
  const Pieces pieces(a, pixbase, kt, wp_, wc, lane);
  HaloAhead<Q, KT, false, NWF, PT, PER_CU == 1> ahead;
  constexpr int kSpare = G::ACT_LOADS + S * WL;   // loads of the last slice, none of which has anything to fetch (R > S)
  static_assert(!kAhead || (R > S && kSpare >= Pieces::NPIECE));

  v4i acc[NWF * PT * 4];   // [(i * PT + j) * 4 + g], see Layout16
#pragma unroll
  for (int t = 0; t < NWF * PT * 4; ++t) acc[t] = v4i{0, 0, 0, 0};
#pragma unroll
  for (int t = 0; t < NWF * PT * 4; ++t) asm volatile("" : "+v"(acc[t]));   // written here, not in front of the first products

  // The reads are inline assembly, counted by hand, and run one unit - 32 channels of a tap: 2 filter fragments, 4 PT
  // products, the row's 2 PT activation fragments in front of its first - ahead of the products; with AHEAD across the barrier.
  v4i pc[2 * PT];                     // this row's activation fragments
  v4i wb[G::NBUF][2];                       // forward: filter fragments [unit % NBUF]
  v2i wlo[G::NBUF][2], whi[G::NBUF][2];           // kWT: their halves
  constexpr int U = NWF;              // units per tap
  constexpr int kFilterReads = kWT ? 4 : 2;
  auto request_filter = [&](auto bc, auto xc, auto vc, unsigned stage_off) {   // unit v of tap x of the stage
    constexpr int b = decltype(bc)::value, x = decltype(xc)::value, v = decltype(vc)::value;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if constexpr (kWT) {
        constexpr int off = x * TAPB + v * 2048;
        wlo[b][h] = h == 0 ? lds_read_tr8<off>(w_addr[0] + stage_off) : lds_read_tr8<off>(w_addr[kWT ? 1 : 0] + stage_off);
        whi[b][h] = h == 0 ? lds_read_tr8<off + 256>(w_addr[kWT ? 1 : 0] + stage_off) : lds_read_tr8<off + 256>(w_addr[0] + stage_off);
      } else {
        constexpr int off = x * TAPB + v * 1024;
        wb[b][h] = h == 0 ? lds_read_b128_at<off>(w_addr[0] + stage_off) : lds_read_b128_at<off + 512>(w_addr[0] + stage_off);
      }
    }
  };
  auto request_act = [&](auto rc, unsigned buf_off) {
    constexpr int r = decltype(rc)::value;
    static_for<PT>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      const unsigned at = p_addr[PA == 1 ? 0 : j][r % PR] + buf_off;
      constexpr int tile_slots = PA > 1 ? 0 : (Q == 8 ? j / 2 * 40 + j % 2 * 16 : j * 16);
      constexpr int off = (tile_slots + r / PR * PR * (Q / 2)) * 64;
      pc[2 * j] = lds_read_b128_at<off>(at);
      pc[2 * j + 1] = lds_read_b128_at<off + G::HALF * 64>(at);
    });
  };

  __builtin_amdgcn_s_setprio(3);   // the main loop's instructions go ahead of a co-resident workgroup's epilogue
  unsigned st_cur = 0, st_load = (R - 1) * G::W_BYTES;   // ring slot of this stage, of the stage to load
  v4i ps[2 * PT];
  if constexpr (G::AHEAD) {
    hc_wait_vmcnt<G::in_flight(0, true)>();
    hc_sync();
    request_act(std::integral_constant<int, 0>{}, 0u);
    request_filter(std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{}, 0u);
  }
  auto slice = [&](int ci, auto lastc) {
    constexpr bool kLast = decltype(lastc)::value;   // the last slice, with the requests for the results' masks and windows
    const unsigned act_cur = (ci & 1) * G::ACT_BYTES, act_next = G::ACT_BYTES - act_cur;
    static_for<S>([&](auto uc) {
      constexpr int u = decltype(uc)::value;
      if (ci == 0) hc_wait_vmcnt<G::in_flight(u, true)>();
      else hc_wait_vmcnt<G::in_flight(u, false)>();
      hc_sync();
      const unsigned st_next = st_cur + G::W_BYTES == R * G::W_BYTES ? 0 : st_cur + G::W_BYTES;
      if constexpr (!G::AHEAD) {
        if constexpr (TPS == 3 || u % 3 == 0) request_act(std::integral_constant<int, TPS == 3 ? u : u / 3>{}, act_cur);
        request_filter(std::integral_constant<int, (u * TPS * U) % G::NBUF>{}, std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{}, st_cur);
      }
      static_for<TPS * U>([&](auto nc) {
        constexpr int n = decltype(nc)::value;              // unit inside the stage
        constexpr int flat = u * TPS * U + n;               // unit inside the slice (of 9 U)
        constexpr int x = n / U, v = n % U;
        constexpr int tap = (u * TPS + x) % 3;              // 0 centre, 1 right, 2 left
        constexpr int b = flat % G::NBUF;
        constexpr bool last_in_stage = n == TPS * U - 1;
        // request the next unit
        constexpr int next_b = (flat + 1) % G::NBUF;
        static_assert(9 * U % G::NBUF == 0);
        constexpr bool next_act = last_in_stage && G::AHEAD && !(kLast && u + 1 == S) && (TPS == 3 || (u + 1) % 3 == 0);
        if constexpr (!last_in_stage) {
          request_filter(std::integral_constant<int, next_b>{}, std::integral_constant<int, (n + 1) / U>{}, std::integral_constant<int, (n + 1) % U>{}, st_cur);
          lds_settle<kFilterReads>();
        } else if constexpr (G::AHEAD && !(kLast && u + 1 == S)) {
          request_filter(std::integral_constant<int, next_b>{}, std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{}, st_next);
          lds_settle<kFilterReads>();
        } else {
          lds_settle<0>();
        }
        if constexpr (tap == 0 && v == 0) {
#pragma unroll
          for (int p = 0; p < 2 * PT; ++p) {
            asm volatile("" : "+v"(pc[p]));   // landed: nothing that reads it moves in front of the wait above
          }
        }
        v4i w[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          if constexpr (kWT) {
            w[h] = lds_landed(wlo[b][h], whi[b][h]);
          } else {
            asm volatile("" : "+v"(wb[b][h]));
            w[h] = wb[b][h];
          }
        }
        // the pixels under this tap: even ones, odd ones
        if constexpr (v == 0) {
#pragma unroll
          for (int j = 0; j < PT; ++j) {
            if constexpr (tap == 0) {
              ps[2 * j] = pc[2 * j];
              ps[2 * j + 1] = pc[2 * j + 1];
            } else if constexpr (tap == 1) {
              ps[2 * j] = pc[2 * j + 1];
              ps[2 * j + 1] = neighbour4<false, Q != 32>(pc[2 * j], keep_r);
            } else {
              ps[2 * j] = neighbour4<true, Q != 32>(pc[2 * j + 1], keep_l);
              ps[2 * j + 1] = pc[2 * j];
            }
          }
        }
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int j = 0; j < PT; ++j)
#pragma unroll
            for (int par = 0; par < 2; ++par) {
              v4i& d = acc[(v * PT + j) * 4 + h * 2 + par];
              mfma64(d, w[h], ps[2 * j + par]);
            }
        __builtin_amdgcn_sched_barrier(0);   // the next unit's requests and wait stay behind these products
        // the next row's activation fragments come into the registers that these products were the last to read
        if constexpr (next_act) request_act(std::integral_constant<int, TPS == 3 ? (u + 1) % 3 : ((u + 1) % 9) / 3>{}, u + 1 == S ? act_next : act_cur);
        // The next loads go out behind the stage's products, one behind each unit's: a wavefront issues in order, and the memory
        // pipeline takes a few hundred clocks to accept a load of 64-byte pieces.
        constexpr int ACTS = G::act_in_stage(u), LOADS = ACTS + WL, UNITS = TPS * U;
        static_for<LOADS>([&](auto kc) {
          constexpr int k = decltype(kc)::value;
          if constexpr (n == (k < UNITS - 1 ? k : UNITS - 1)) {
            constexpr int tl = u + R - 1;
            constexpr int e = (u > 0 ? G::ACT_LOADS : 0) + u * WL + k;   // number of this load inside a slice (S == 3)
            if constexpr (kLast) {
              constexpr int w = e - Pieces::NPIECE;
              if constexpr (w < 0) ahead.mk[e] = pieces.mask(a, e);
              else if constexpr (w < 4 * Pieces::NPIECE) ahead.xw[w / 4][w % 4] = pieces.window(a, w / 4, w % 4);
            } else if constexpr (k < ACTS) issue_act(ci + 1, (ci + 1) & 1, std::integral_constant<int, G::act_before(u) + k>{});
            else issue_w(ci + tl / S, std::integral_constant<int, tl % S>{}, w_lds + st_load, std::integral_constant<int, k - ACTS>{});
            __builtin_amdgcn_sched_barrier(0);
          }
        });
      });
      st_load = st_cur;
      st_cur = st_next;
    });
  };
  for (int ci = 0; ci < nsl - (kAhead ? 1 : 0); ++ci) slice(ci, std::false_type{});
  if constexpr (kAhead) slice(nsl - 1, std::true_type{});
  // the loads and reads issued past the end are done before the tiles are reused
  hc_wait_vmcnt<0>();
  if constexpr (G::AHEAD && !kAhead) {
    lds_settle<0>();
    // the registers of the fragments requested for a next slice stay theirs until they have landed
#pragma unroll
    for (int p = 0; p < 2 * PT; ++p) asm volatile("" ::"v"(pc[p]));
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if constexpr (kWT) asm volatile("" ::"v"(wlo[0][h]), "v"(whi[0][h]));
      else asm volatile("" ::"v"(wb[0][h]));
    }
  }
  if constexpr (kAhead) {
    // the windows that found no place in the last slice
#pragma unroll
    for (int w = kSpare - Pieces::NPIECE; w < 4 * Pieces::NPIECE; ++w) ahead.xw[w / 4][w % 4] = pieces.window(a, w / 4, w % 4);
  }
  mfma_settle();
#pragma unroll
  for (int t = 0; t < NWF * PT * 4; ++t) asm volatile("" : "+v"(acc[t]));   // not read in front of that wait
  __builtin_amdgcn_s_setprio(0);
  halo_epilogue<Q, KT, false, NWF, PT, kFused, kSto, PER_CU == 1, Layout16>(a, at, acc, smem, reinterpret_cast<uint32_t*>(dump + 1024), pixbase, kt, wp_, wc, settle_shift, hint, pieces, ahead, along);
}
template <int Q, int BR, int NI, int KT, int PER_CU, bool kFused, bool kWT, bool kSto>
__global__ __launch_bounds__(512, 2 * PER_CU) void conv3x3_k64_kernel(const HaloArgs a) {
  extern __shared__ __attribute__((aligned(16))) int8_t smem[];
  NothingAlong along;
  k64_tile<Q, BR, NI, KT, PER_CU, kFused, kWT, kSto>(a, halo_grid_place(), smem, along);
}

// the same for launches with more tiles than the device holds workgroups
template <int Q, int BR, int NI, int KT, bool kWT, bool kSto>
__global__ __launch_bounds__(512, 4) void conv3x3_k64_turns_kernel(const HaloArgs, const int nx, const int ny) {
  extern __shared__ __attribute__((aligned(16))) int8_t smem[];
  Turns along;
  tiles_in_turns(nx, ny, along, [&](const HaloArgs& a, const HaloPlace at) { k64_tile<Q, BR, NI, KT, 2, true, kWT, kSto>(a, at, smem, along); });
}

template <int Q, int BR, int NI, int KT, int PER_CU, bool kFused, bool kWT, bool kSto>
int launch_k64(const HaloArgs& a, hipStream_t stream) {
  using G = KGeom<Q, BR, NI, KT, PER_CU>;
  static_assert(8 * 32 * (32 * 4 + 16) <= G::TILE_BYTES, "int32 patches must stay clear of the reduction words");
  static_assert(8 * 32 * G::PT * (G::NWF * 32 + 16) <= G::TILE_BYTES, "int8 patches must stay clear of the reduction words");
  static_assert(KT != 32 || 2 * G::LDS_BYTES <= 160 * 1024, "two 32-channel workgroups on a unit where a launch is pinned to them");
  static HaloLaunch state[2];
  const HaloKernel one{conv3x3_k64_kernel<Q, BR, NI, KT, PER_CU, kFused, kWT, kSto>, G::LDS_BYTES};
  if constexpr (kFused && KT != 32) {
    const HaloKernel several{conv3x3_k64_turns_kernel<Q, BR, NI, KT, kWT, kSto>, KGeom<Q, BR, NI, KT, 2>::LDS_BYTES};
    return launch_halo_kernel<true>(one, several, state, G::PX, KT, Q, a, stream);
  } else {
    return launch_halo_kernel<kFused>(one, one, state, G::PX, KT, Q, a, stream);   // (32 channels: see halo_narrow_fits)
  }
}

// One workgroup per compute unit as long as the launch has no more of them; NITI_HALO_PER_CU pins the choice (tests).
template <bool kFused, bool kWT, bool kSto>
int launch_k64_tiles(const HaloArgs& a, int H, int ktile, hipStream_t stream) {
  const long long nb = (static_cast<long long>(a.N) * H * H + 255) / 256 * ((a.K + ktile - 1) / ktile);
  const char* e = getenv("NITI_HALO_PER_CU");
  const bool one = e != nullptr ? e[0] == '1' : nb <= compute_units();
  if (ktile == 32) {
    if (H == 16) return launch_k64<16, 16, 1, 32, 1, kFused, kWT, kSto>(a, stream);
    if (H == 8) return launch_k64<8, 8, 4, 32, 1, kFused, kWT, kSto>(a, stream);
    return launch_k64<4, 4, 16, 32, 1, kFused, kWT, kSto>(a, stream);
  }
  if (ktile == 64) {
    if (H == 32) return one ? launch_k64<32, 8, 1, 64, 1, kFused, kWT, kSto>(a, stream) : launch_k64<32, 8, 1, 64, 2, kFused, kWT, kSto>(a, stream);
    if (H == 16) return one ? launch_k64<16, 16, 1, 64, 1, kFused, kWT, kSto>(a, stream) : launch_k64<16, 16, 1, 64, 2, kFused, kWT, kSto>(a, stream);
    if (H == 8) return one ? launch_k64<8, 8, 4, 64, 1, kFused, kWT, kSto>(a, stream) : launch_k64<8, 8, 4, 64, 2, kFused, kWT, kSto>(a, stream);
    return one ? launch_k64<4, 4, 16, 64, 1, kFused, kWT, kSto>(a, stream) : launch_k64<4, 4, 16, 64, 2, kFused, kWT, kSto>(a, stream);
  }
  if (H == 32) return one ? launch_k64<32, 8, 1, 128, 1, kFused, kWT, kSto>(a, stream) : launch_k64<32, 8, 1, 128, 2, kFused, kWT, kSto>(a, stream);
  if (H == 16) return one ? launch_k64<16, 16, 1, 128, 1, kFused, kWT, kSto>(a, stream) : launch_k64<16, 16, 1, 128, 2, kFused, kWT, kSto>(a, stream);
  if (H == 8) return one ? launch_k64<8, 8, 4, 128, 1, kFused, kWT, kSto>(a, stream) : launch_k64<8, 8, 4, 128, 2, kFused, kWT, kSto>(a, stream);
  return one ? launch_k64<4, 4, 16, 128, 1, kFused, kWT, kSto>(a, stream) : launch_k64<4, 4, 16, 128, 2, kFused, kWT, kSto>(a, stream);
}

}  // namespace
}  // namespace niti
