// int8 products of matrices with any extents, in any of the four operand layouts, read as stored (gemm_any.hip).
#pragma once
#include "common.h"

namespace niti {

// x / d for 0 <= x < 2^31: with 2^(s-1) < d <= 2^s and mul = floor(2^(31+s) / d) + 1, mul d exceeds 2^(31+s) by at most d <= 2^s,
// hence x mul / 2^(31+s) exceeds x / d by less than 1 / d
struct Reciprocal {
  uint32_t mul, shift;   // mul 0: d = 1
  explicit Reciprocal(int d = 1) : mul(0), shift(0) {
    if (d < 2) return;
    int s = 1;
    while ((1LL << s) < d) ++s;
    mul = static_cast<uint32_t>((1ULL << (31 + s)) / static_cast<unsigned>(d) + 1);
    shift = static_cast<uint32_t>(s - 1);
  }
  __device__ int of(int x) const { return mul != 0u ? static_cast<int>(__umulhi(static_cast<uint32_t>(x), mul) >> shift) : x; }
};

struct AnyArgs {
  const int8_t* a;       // [m][k], or [k][m] when transposed
  const int8_t* b;       // [n][k] when transposed, or [k][n]
  int m, n, k;
  // int32 result
  int32_t* c = nullptr;  // [m][n]
  uint32_t* absmax = nullptr;
  int roundtrip = 0;
  // result rounded to int8, or rounded and subtracted from the weights
  int8_t* out8 = nullptr;   // [m][n]; weight update: the rounded gradient, may be null
  int8_t* w = nullptr;      // [m][n], weight update only
  int8_t* wprep = nullptr;  // weight update of a [m][9][channels] filter: the 3x3 forward kernel's copy of it, kept in step
  int channels = 0;
  Reciprocal by_channels{};
  const int8_t* mask = nullptr;   // laid out like out8: results are zero where it is not positive (not for the weight update)
  // with a mask: the result is the gradient of a 2x2 / stride-2 max-pool's output (= mask, [rows][map_h][map_w][n]) and goes to
  // the position(s) of each window of the pool's input pool_x that hold the maximum, in unpool; out8 is not written
  // pool: rows come window by window (2 x 2 pixels of the [map_h][map_w] result, by_map_w divides by map_w / 2) and the maximum of
  // each window goes there as well
  int8_t* pool = nullptr;
  const int8_t* pool_x = nullptr;
  int8_t* unpool = nullptr;
  int ties_all = 0, map_h = 0, map_w = 0;
  Reciprocal by_map{}, by_map_w{};
  const int32_t* rand = nullptr;
  uint32_t* sync = nullptr;
  int target_bits = 7, method = 0, trunc = 0, bw_mode = 0;
  unsigned rq_flags = 0;
  long long spin_limit = 0;
  uint32_t* sticky = nullptr;
  int32_t* shift_out = nullptr;
  const int32_t* exp_a = nullptr;
  const int32_t* exp_b = nullptr;
  int32_t* exp_out = nullptr;
};

bool gemm_any_shape(int m, int n, int k);                       // extents within the kernels' index arithmetic
bool gemm_any_large(int m, int n);                              // the result fills the chip with 128 x 128 tiles
int launch_gemm_any(int trans_a, int trans_b, const AnyArgs& a, hipStream_t stream);
// workgroups of the launch that rounds (= sync slots), 0 when no variant's grid fits on the current device at once
enum AnyRound { kAnyForward = 0, kAnyDgrad = 1, kAnyUpdate = 2 };   // layouts NT, NN, TN
long long gemm_any_round_blocks(AnyRound what, int m, int n, int k);
int launch_gemm_any_round(AnyRound what, const AnyArgs& a, hipStream_t stream);
// Both gradients of a [m][f] -> [m][o] layer as one launch: d = data gradient (NN: error, w), w = update (TN: error, act) whose
// exponent builds on d's (w.exp_a is not read); workgroups of each = slots of each.  false: not resident together
bool gemm_any_backward_blocks(int m, int o, int f, int* nd, int* nw);
int launch_gemm_any_backward(const AnyArgs& d, const AnyArgs& w, hipStream_t stream);

}  // namespace niti
