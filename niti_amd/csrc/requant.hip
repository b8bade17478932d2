// Integer requantisation kernels: per-tensor max |x|, shift-round-clip back to int8 (nearest,
// stochastic with supplied random integers, pseudo-stochastic), the fused gradient rounding +
// weight update, ReLU forward/backward.  All are single-pass HBM-bandwidth kernels that move
// 16 int32 (64 bytes in, 16 bytes out) per thread per step; the shift is derived on the
// device from the max the producer kernel left in memory.
#include "common.h"
#include "requant_math.h"

namespace niti {
namespace {

__global__ __launch_bounds__(256) void absmax_i32_kernel(const int32_t* __restrict__ x, int64_t n, uint32_t* absmax) {
  const int64_t nv = n >> 2;
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  const int64_t t0 = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  uint32_t lmax = 0;
  const v4i* xv = reinterpret_cast<const v4i*>(x);
  for (int64_t i = t0; i < nv; i += stride) {
    const v4i v = xv[i];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t u = uabs(v[e]);
      lmax = u > lmax ? u : lmax;
    }
  }
  for (int64_t i = (nv << 2) + t0; i < n; i += stride) {
    const uint32_t u = uabs(x[i]);
    lmax = u > lmax ? u : lmax;
  }
  fold_absmax(absmax, lmax);
}

struct RequantArgs {
  const int32_t* x;
  int8_t* y;        // requant: output.  grad update: optional rounded gradient
  int8_t* w;        // grad update only
  const int32_t* rand;
  const uint32_t* absmax;
  int32_t* shift_out;
  const int32_t* exp_a;
  const int32_t* exp_b;
  int32_t* exp_out;
  int64_t n;
  int target_bits, trunc, bw_mode;
  unsigned flags;
};

// kUpdate == false: y = requant(x).  kUpdate == true: g = requant(x); w = clip(w - g); y (optional) = g
template <int kMethod, bool kUpdate>
__global__ __launch_bounds__(256) void requant_kernel(const RequantArgs a) {
  const int shift = bitwidth_of(*a.absmax, a.bw_mode) - a.target_bits;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    const int sh = shift > 0 ? shift : 0;
    if (a.shift_out != nullptr) *a.shift_out = sh;
    if (a.exp_out != nullptr)
      *a.exp_out = sh + (a.exp_a != nullptr ? *a.exp_a : 0) + (a.exp_b != nullptr ? *a.exp_b : 0);
  }
  // random integers are reduced to their low `shift` bits: values already in [0, 2^shift) pass
  // unchanged, wider uniform bits become uniform in [0, 2^shift) without the host knowing shift
  const int rm = shift >= 1 ? static_cast<int>((1u << (shift > 31 ? 31 : shift)) - 1u) : 0;
  const v4i rmask = {rm, rm, rm, rm};
  const bool trunc = a.trunc != 0;
  const bool relu = (a.flags & NITI_RQ_RELU) != 0;
  auto one = [&](int x, int u) -> int {
    int r;
    if (shift >= 1) r = round_one<kMethod>(x, shift, trunc, u);
    else r = wrap_to_i8(x);
    if (relu && r < 0) r = 0;
    return r;
  };
  const int64_t nv = a.n >> 4;  // groups of 16 elements
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  const int64_t t0 = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const v4i* xv = reinterpret_cast<const v4i*>(a.x);
  const v4i* uv = reinterpret_cast<const v4i*>(a.rand);
  for (int64_t i = t0; i < nv; i += stride) {
    v4i out;
    v4i wv = {0, 0, 0, 0};
    if (kUpdate) wv = reinterpret_cast<const v4i*>(a.w)[i];
    v4i neww;
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const v4i v = xv[i * 4 + d];
      v4i u = {0, 0, 0, 0};
      if (kMethod == NITI_ROUND_STOCHASTIC && shift >= 1) u = uv[i * 4 + d] & rmask;
      uint32_t packed = 0, packedw = 0;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int r = one(v[e], u[e]);
        packed |= (static_cast<uint32_t>(r) & 0xFFu) << (8 * e);
        if (kUpdate) {
          const int wold = static_cast<int>(static_cast<int8_t>((static_cast<uint32_t>(wv[d]) >> (8 * e)) & 0xFFu));
          packedw |= (static_cast<uint32_t>(clip127(wold - r)) & 0xFFu) << (8 * e);
        }
      }
      out[d] = static_cast<int>(packed);
      neww[d] = static_cast<int>(packedw);
    }
    if (kUpdate) {
      reinterpret_cast<v4i*>(a.w)[i] = neww;
      if (a.y != nullptr) reinterpret_cast<v4i*>(a.y)[i] = out;
    } else {
      reinterpret_cast<v4i*>(a.y)[i] = out;
    }
  }
  for (int64_t i = (nv << 4) + t0; i < a.n; i += stride) {
    int u = 0;
    if (kMethod == NITI_ROUND_STOCHASTIC && shift >= 1) u = a.rand[i] & rmask[0];
    const int r = one(a.x[i], u);
    if (kUpdate) {
      a.w[i] = static_cast<int8_t>(clip127(static_cast<int>(a.w[i]) - r));
      if (a.y != nullptr) a.y[i] = static_cast<int8_t>(r);
    } else {
      a.y[i] = static_cast<int8_t>(r);
    }
  }
}

__global__ __launch_bounds__(256) void weight_update_kernel(int8_t* w, const int8_t* __restrict__ g, int64_t n) {
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride)
    w[i] = static_cast<int8_t>(clip127(static_cast<int>(w[i]) - static_cast<int>(g[i])));
}

// ---- input quantiser (TiFloatToInt8, ti_torch.py:341-356) with the layout change that follows it (ti_net.py:19) ----
// r = max |x| over the batch (float bits of non-negative values order like unsigned integers)
__global__ __launch_bounds__(256) void absmax_f32_kernel(const float* __restrict__ x, int64_t n, uint32_t* __restrict__ out) {
  __shared__ uint32_t wmax[4];
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  uint32_t m = 0;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride) {
    const uint32_t b = __float_as_uint(x[i]) & 0x7FFFFFFFu;
    m = b > m ? b : m;
  }
  m = wave_max_u32(m);
  if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x < 64) fold_absmax(out, threadIdx.x < 4 ? wmax[threadIdx.x] : 0u);
}

// Largest |x| per workgroup, stored (not folded into a zeroed word: no fill in front, no atomics on one address - with a
// thousand workgroups folding into one word the pass took 9.5 us for 1.5 MB and 18.5 us for 3 MB, memory-bound it is
// about 2).  Also copies the batch's class indices where the caller keeps them in a buffer of its own.
constexpr int kQuantParts = 256;   // partial maxima: one per thread of the workgroups that read them
__global__ __launch_bounds__(256) void absmax_parts_f32_kernel(const float* __restrict__ x, int64_t n, uint32_t* __restrict__ parts,
                                                               const int64_t* __restrict__ t_in, int64_t* __restrict__ t_out, int nt) {
  __shared__ uint32_t wmax[4];
  const int64_t stride = static_cast<int64_t>(gridDim.x) * 256;
  const int64_t t0 = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  for (int64_t i = t0; i < nt; i += stride) t_out[i] = t_in[i];
  uint32_t m = 0;
  const int64_t nv = aligned16_dev(x) ? n >> 2 : 0;
  for (int64_t i = t0; i < nv; i += stride) {
    const v4i v = reinterpret_cast<const v4i*>(x)[i];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t b = static_cast<uint32_t>(v[e]) & 0x7FFFFFFFu;
      m = b > m ? b : m;
    }
  }
  for (int64_t i = (nv << 2) + t0; i < n; i += stride) {
    const uint32_t b = __float_as_uint(x[i]) & 0x7FFFFFFFu;
    m = b > m ? b : m;
  }
  m = wave_max_u32(m);
  if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t g = wmax[0];
    for (int i = 1; i < 4; ++i) g = wmax[i] > g ? wmax[i] : g;
    parts[blockIdx.x] = g;
  }
}

// bw = ceil(log2 r); y = int8(clamp(round_half_even(x * 2^(bits - bw)), -128, 127)), float NCHW -> int8 NHWC with the
// channels zero-padded to cpad; exp_out = bw - bits.  The product and the rounding are the reference's float32 operations.
// r = the largest of nparts partial maxima (one word: the caller's absmax_bits); nparts == 0 (a batch of a few images):
// every workgroup takes the maximum over the whole batch itself, which saves the launch in front of this one.
// The last kZeroBlocks workgroups clear `zero` where asked (the words that the launches behind this one exchange their ranges
// through: one launch less).
constexpr int kZeroBlocks = 16;
__global__ __launch_bounds__(256) void quantize_f32_i8_kernel(const float* __restrict__ x, int8_t* __restrict__ y, int64_t pixels,
                                                              int C, int HW, int cpad, const uint32_t* __restrict__ parts, int nparts,
                                                              int32_t* exp_out, int bits, const int64_t* __restrict__ t_in,
                                                              int64_t* __restrict__ t_out, int nt, v4i* __restrict__ zero, int zero_quads) {
  if (static_cast<int>(blockIdx.x) >= static_cast<int>(gridDim.x) - (zero_quads > 0 ? kZeroBlocks : 0)) {
    const v4i nothing = {0, 0, 0, 0};
    for (int i = (static_cast<int>(blockIdx.x) - static_cast<int>(gridDim.x) + kZeroBlocks) * 256 + static_cast<int>(threadIdx.x); i < zero_quads; i += kZeroBlocks * 256)
      zero[i] = nothing;
    return;
  }
  __shared__ uint32_t wmax[4];
  const int64_t stride = static_cast<int64_t>(gridDim.x - (zero_quads > 0 ? kZeroBlocks : 0)) * blockDim.x;
  const int64_t p0 = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  // Four channels of a pixel, their loads in flight together (channels behind the last one: that one again); the first pixel's leave
  // in front of the range.  What bounds the kernel for a few images are its trips to memory one after the other: one image of 3 channels 4.4 us
  // with twelve for the range and one for each channel, so 3.2.  (128 / 256 images 5.0 / 5.2 either way.)
  auto fetch = [&](int64_t p, int c0, float (&f)[4]) {
    const int64_t n = p / HW, hw = p - n * HW;
    const float* const src = x + n * C * HW + hw;
#pragma unroll
    for (int e = 0; e < 4; ++e) f[e] = src[static_cast<int64_t>(min(c0 + e, C - 1)) * HW];
  };
  float first[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  if (p0 < pixels) fetch(p0, 0, first);
  uint32_t m = 0;
  if (nparts > 0) {
    if (static_cast<int>(threadIdx.x) < nparts) m = parts[threadIdx.x];
  } else {
    const int n = static_cast<int>(pixels * C);   // (a few images)
    for (int i = threadIdx.x; i < n; i += 8 * 256) {
      float f[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) f[u] = x[min(i + u * 256, n - 1)];
#pragma unroll
      for (int u = 0; u < 8; ++u) m = max(m, __float_as_uint(f[u]) & 0x7FFFFFFFu);
    }
    if (blockIdx.x == 0)
      for (int i = threadIdx.x; i < nt; i += 256) t_out[i] = t_in[i];
  }
  m = wave_max_u32(m);
  if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = m;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 4; ++i) m = wmax[i] > m ? wmax[i] : m;
  const float r = __uint_as_float(m);
  // ceil(log2 r) from the exponent and mantissa of r = m 2^e, 0.5 <= m < 1 (exact; a library log2f rounds k + log2(1 + d)
  // back to k for the first float32 values above 2^k, k >= 4, and differs between platforms there)
  int fe = 0;
  const float fm = frexpf(r, &fe);
  const int bw = fm == 0.5f ? fe - 1 : fe;
  const float scale = ldexpf(1.0f, bits - bw);
  if (blockIdx.x == 0 && threadIdx.x == 0 && exp_out != nullptr) *exp_out = r > 0.0f ? bw - bits : 0;
  auto quad = [&](int64_t p, int c0) {   // four channels of a pixel as one word
    if (c0 >= C || !(r > 0.0f)) return 0u;
    float f[4];
    if (c0 == 0 && p == p0) {
#pragma unroll
      for (int e = 0; e < 4; ++e) f[e] = first[e];
    } else {
      fetch(p, c0, f);
    }
    uint32_t word = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int q = static_cast<int>(fminf(fmaxf(rintf(f[e] * scale), -128.0f), 127.0f));
      word |= c0 + e < C ? (static_cast<uint32_t>(q) & 0xFFu) << (8 * e) : 0u;
    }
    return word;
  };
  const bool wide = cpad % 16 == 0 && aligned16_dev(y);
  for (int64_t p = p0; p < pixels; p += stride) {
    int8_t* dst = y + p * cpad;
    if (wide) {
      for (int c0 = 0; c0 < cpad; c0 += 16) {
        v4i o;
#pragma unroll
        for (int d = 0; d < 4; ++d) o[d] = static_cast<int>(quad(p, c0 + 4 * d));
        *reinterpret_cast<v4i*>(dst + c0) = o;
      }
    } else {
      for (int c0 = 0; c0 < cpad; c0 += 4) *reinterpret_cast<uint32_t*>(dst + c0) = quad(p, c0);
    }
  }
}

// y[m][f] = x[m][f] * mask[f] with mask bytes 0 / 1 (a keep / drop decision per feature); optionally exp_out = exp_in + add
__global__ __launch_bounds__(256) void mask_features_kernel(const int8_t* __restrict__ x, const int8_t* __restrict__ mask,
                                                            int8_t* __restrict__ y, int64_t rows, int features,
                                                            const int32_t* exp_in, int32_t* exp_out, int exp_add) {
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  const int64_t t0 = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t0 == 0 && exp_out != nullptr) *exp_out = (exp_in != nullptr ? *exp_in : 0) + exp_add;
  const int fv = features >> 4;   // features % 16 == 0 (host check)
  const int64_t nv = rows * fv;
  for (int64_t i = t0; i < nv; i += stride) {
    const int f = static_cast<int>(i % fv);
    const v4i xv = reinterpret_cast<const v4i*>(x)[i];
    const v4i mv = reinterpret_cast<const v4i*>(mask)[f];
    v4i o;
#pragma unroll
    for (int d = 0; d < 4; ++d) o[d] = xv[d] & static_cast<int>((static_cast<uint32_t>(mv[d]) & 0x01010101u) * 0xFFu);
    reinterpret_cast<v4i*>(y)[i] = o;
  }
}

// kBwd == false: y = max(x, 0).  kBwd == true: y = x(act) > 0 ? dy : 0
template <bool kBwd>
__global__ __launch_bounds__(256) void relu_kernel(const int8_t* __restrict__ x, const int8_t* __restrict__ dy,
                                                   int8_t* __restrict__ y, int64_t n) {
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  const int64_t t0 = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const bool vec = aligned16_dev(x) && aligned16_dev(y) && (!kBwd || aligned16_dev(dy));
  const int64_t nv = vec ? (n >> 4) : 0;
  for (int64_t i = t0; i < nv; i += stride) {
    const v4i xv = reinterpret_cast<const v4i*>(x)[i];
    v4i dv = {0, 0, 0, 0};
    if (kBwd) dv = reinterpret_cast<const v4i*>(dy)[i];
    v4i o;
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      uint32_t p = 0;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int xe = static_cast<int8_t>((static_cast<uint32_t>(xv[d]) >> (8 * e)) & 0xFFu);
        const uint32_t src = kBwd ? ((static_cast<uint32_t>(dv[d]) >> (8 * e)) & 0xFFu) : (static_cast<uint32_t>(xe) & 0xFFu);
        p |= (xe > 0 ? src : 0u) << (8 * e);
      }
      o[d] = static_cast<int>(p);
    }
    reinterpret_cast<v4i*>(y)[i] = o;
  }
  for (int64_t i = (nv << 4) + t0; i < n; i += stride) y[i] = x[i] > 0 ? (kBwd ? dy[i] : x[i]) : static_cast<int8_t>(0);
}

inline int grid_for(int64_t work_items, int block, int cap = 4096) {
  int64_t g = (work_items + block - 1) / block;
  if (g < 1) g = 1;
  return static_cast<int>(g > cap ? cap : g);
}

template <bool kUpdate>
int launch_requant(const RequantArgs& a, int method, hipStream_t stream) {
  const dim3 grid(grid_for((a.n + 15) / 16, 256)), block(256);
  switch (method) {
    case NITI_ROUND_NEAREST:
      hipLaunchKernelGGL((requant_kernel<NITI_ROUND_NEAREST, kUpdate>), grid, block, 0, stream, a);
      break;
    case NITI_ROUND_STOCHASTIC:
      hipLaunchKernelGGL((requant_kernel<NITI_ROUND_STOCHASTIC, kUpdate>), grid, block, 0, stream, a);
      break;
    case NITI_ROUND_PSEUDO_STOCHASTIC:
      hipLaunchKernelGGL((requant_kernel<NITI_ROUND_PSEUDO_STOCHASTIC, kUpdate>), grid, block, 0, stream, a);
      break;
    default:
      return fail(NITI_ERR_INVALID_ARG, "requant: unknown rounding method %d", method);
  }
  return check_launch("requant");
}

int check_requant_common(const char* who, const void* x, int64_t n, const uint32_t* absmax, int target_bits, int method,
                         int div_mode, int bw_mode, const int32_t* rand) {
  if (n < 0) return fail(NITI_ERR_INVALID_ARG, "%s: n=%lld", who, static_cast<long long>(n));
  if (n == 0) return NITI_OK;
  if (x == nullptr || absmax == nullptr) return fail(NITI_ERR_INVALID_ARG, "%s: null pointer", who);
  if (!aligned16(x)) return fail(NITI_ERR_INVALID_ARG, "%s: input must be 16-byte aligned", who);
  if (target_bits < 1 || target_bits > 7) return fail(NITI_ERR_INVALID_ARG, "%s: target_bits=%d outside 1..7", who, target_bits);
  if (div_mode != NITI_DIV_FLOOR && div_mode != NITI_DIV_TRUNC) return fail(NITI_ERR_INVALID_ARG, "%s: div_mode=%d", who, div_mode);
  if (bw_mode != NITI_BW_INT && bw_mode != NITI_BW_F32) return fail(NITI_ERR_INVALID_ARG, "%s: bw_mode=%d", who, bw_mode);
  if (method == NITI_ROUND_STOCHASTIC && (rand == nullptr || !aligned16(rand)))
    return fail(NITI_ERR_INVALID_ARG, "%s: stochastic rounding needs a 16-byte aligned rand tensor", who);
  return NITI_OK;
}

}  // namespace
}  // namespace niti

using namespace niti;

extern "C" int niti_absmax_i32(const int32_t* x, int64_t n, uint32_t* absmax, void* stream) {
  clear_error();
  if (n < 0) return fail(NITI_ERR_INVALID_ARG, "absmax: n=%lld", static_cast<long long>(n));
  if (n == 0) return NITI_OK;
  if (x == nullptr || absmax == nullptr) return fail(NITI_ERR_INVALID_ARG, "absmax: null pointer");
  if (!aligned16(x)) return fail(NITI_ERR_INVALID_ARG, "absmax: input must be 16-byte aligned");
  hipLaunchKernelGGL(absmax_i32_kernel, dim3(grid_for((n + 3) / 4, 256, 2048)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), x, n, absmax);
  return check_launch("absmax_i32");
}

extern "C" int niti_requant_i32_i8(const int32_t* x, int8_t* y, int64_t n, const uint32_t* absmax, int target_bits,
                                   int method, int div_mode, int bw_mode, const int32_t* rand, unsigned flags,
                                   int32_t* shift_out, const int32_t* exp_a, const int32_t* exp_b, int32_t* exp_out,
                                   void* stream) {
  clear_error();
  int st = check_requant_common("requant", x, n, absmax, target_bits, method, div_mode, bw_mode, rand);
  if (st != NITI_OK || n == 0) return st;
  if (y == nullptr || !aligned16(y)) return fail(NITI_ERR_INVALID_ARG, "requant: output must be non-null and 16-byte aligned");
  RequantArgs a{x, y, nullptr, rand, absmax, shift_out, exp_a, exp_b, exp_out, n, target_bits, div_mode == NITI_DIV_TRUNC, bw_mode, flags};
  return launch_requant<false>(a, method, static_cast<hipStream_t>(stream));
}

extern "C" int niti_grad_update_i8(const int32_t* g, int8_t* w, int64_t n, const uint32_t* absmax, int mu, int method,
                                   int div_mode, int bw_mode, const int32_t* rand, int8_t* g8_out, int32_t* shift_out,
                                   const int32_t* exp_a, const int32_t* exp_b, int32_t* exp_out, void* stream) {
  clear_error();
  int st = check_requant_common("grad_update", g, n, absmax, mu, method, div_mode, bw_mode, rand);
  if (st != NITI_OK || n == 0) return st;
  if (w == nullptr || !aligned16(w)) return fail(NITI_ERR_INVALID_ARG, "grad_update: weights must be non-null and 16-byte aligned");
  if (g8_out != nullptr && !aligned16(g8_out)) return fail(NITI_ERR_INVALID_ARG, "grad_update: g8_out must be 16-byte aligned");
  RequantArgs a{g, g8_out, w, rand, absmax, shift_out, exp_a, exp_b, exp_out, n, mu, div_mode == NITI_DIV_TRUNC, bw_mode, 0u};
  return launch_requant<true>(a, method, static_cast<hipStream_t>(stream));
}

extern "C" int niti_weight_update_i8(int8_t* w, const int8_t* g, int64_t n, void* stream) {
  clear_error();
  if (n < 0) return fail(NITI_ERR_INVALID_ARG, "weight_update: n=%lld", static_cast<long long>(n));
  if (n == 0) return NITI_OK;
  if (w == nullptr || g == nullptr) return fail(NITI_ERR_INVALID_ARG, "weight_update: null pointer");
  hipLaunchKernelGGL(weight_update_kernel, dim3(grid_for(n, 256)), dim3(256), 0, static_cast<hipStream_t>(stream), w, g, n);
  return check_launch("weight_update");
}

extern "C" int niti_relu_i8_fwd(const int8_t* x, int8_t* y, int64_t n, void* stream) {
  clear_error();
  if (n < 0) return fail(NITI_ERR_INVALID_ARG, "relu: n=%lld", static_cast<long long>(n));
  if (n == 0) return NITI_OK;
  if (x == nullptr || y == nullptr) return fail(NITI_ERR_INVALID_ARG, "relu: null pointer");
  hipLaunchKernelGGL(relu_kernel<false>, dim3(grid_for((n + 15) / 16, 256)), dim3(256), 0, static_cast<hipStream_t>(stream),
                     x, static_cast<const int8_t*>(nullptr), y, n);
  return check_launch("relu_fwd");
}

extern "C" int niti_quantize_f32_i8(const float* x, int8_t* y, int N, int C, int H, int W, int cpad, int bits, uint32_t* absmax_bits,
                                    int32_t* exp_out, void* stream) {
  clear_error();
  if (N <= 0 || C <= 0 || H <= 0 || W <= 0 || cpad < C || cpad % 4 != 0 || bits < 1 || bits > 7)
    return fail(NITI_ERR_INVALID_ARG, "quantize: N=%d C=%d H=%d W=%d cpad=%d bits=%d", N, C, H, W, cpad, bits);
  if (x == nullptr || y == nullptr || absmax_bits == nullptr) return fail(NITI_ERR_INVALID_ARG, "quantize: null pointer");
  if (reinterpret_cast<uintptr_t>(y) % 4 != 0) return fail(NITI_ERR_INVALID_ARG, "quantize: output must be 4-byte aligned");
  const int64_t pixels = static_cast<int64_t>(N) * H * W, n = pixels * C;
  hipStream_t s = static_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(absmax_f32_kernel, dim3(grid_for(n, 256, 1024)), dim3(256), 0, s, x, n, absmax_bits);
  hipLaunchKernelGGL(quantize_f32_i8_kernel, dim3(grid_for(pixels, 256)), dim3(256), 0, s, x, y, pixels, C, H * W, cpad, absmax_bits, 1,
                     exp_out, bits, static_cast<const int64_t*>(nullptr), static_cast<int64_t*>(nullptr), 0, static_cast<v4i*>(nullptr), 0);
  return check_launch("quantize");
}

extern "C" int niti_quantize_batch_zero_f32_i8(const float* x, int8_t* y, int N, int C, int H, int W, int cpad, int bits, uint32_t* parts,
                                               int32_t* exp_out, const int64_t* target_in, int64_t* target_out, int targets, uint32_t* zero,
                                               int zero_words, void* stream) {
  clear_error();
  if (N <= 0 || C <= 0 || H <= 0 || W <= 0 || cpad < C || cpad % 4 != 0 || bits < 1 || bits > 7 || targets < 0)
    return fail(NITI_ERR_INVALID_ARG, "quantize_batch: N=%d C=%d H=%d W=%d cpad=%d bits=%d targets=%d", N, C, H, W, cpad, bits, targets);
  if (x == nullptr || y == nullptr || parts == nullptr || (targets > 0 && (target_in == nullptr || target_out == nullptr)))
    return fail(NITI_ERR_INVALID_ARG, "quantize_batch: null pointer");
  if (reinterpret_cast<uintptr_t>(y) % 4 != 0) return fail(NITI_ERR_INVALID_ARG, "quantize_batch: output must be 4-byte aligned");
  if (zero_words < 0 || zero_words % 4 != 0 || (zero_words > 0 && (zero == nullptr || !aligned16(zero))))
    return fail(NITI_ERR_INVALID_ARG, "quantize_batch: words to clear must be whole, aligned groups of four");
  const int64_t pixels = static_cast<int64_t>(N) * H * W, n = pixels * C;
  hipStream_t s = static_cast<hipStream_t>(stream);
  // up to 12 Ki values (four CIFAR images, 48 loads a thread) a workgroup reads the batch in less time than a launch takes
  const bool solo = n <= 12288;
  int nparts = 0;
  if (!solo) {
    nparts = grid_for((n + 3) / 4, 1024, kQuantParts);
    hipLaunchKernelGGL(absmax_parts_f32_kernel, dim3(nparts), dim3(256), 0, s, x, n, parts, target_in, target_out, targets);
  }
  hipLaunchKernelGGL(quantize_f32_i8_kernel, dim3(grid_for(pixels, 256) + (zero_words > 0 ? kZeroBlocks : 0)), dim3(256), 0, s, x, y, pixels, C, H * W, cpad,
                     parts, nparts, exp_out, bits, target_in, target_out, solo ? targets : 0, reinterpret_cast<v4i*>(zero), zero_words / 4);
  return check_launch("quantize_batch");
}

extern "C" int niti_quantize_batch_f32_i8(const float* x, int8_t* y, int N, int C, int H, int W, int cpad, int bits, uint32_t* parts,
                                          int32_t* exp_out, const int64_t* target_in, int64_t* target_out, int targets, void* stream) {
  return niti_quantize_batch_zero_f32_i8(x, y, N, C, H, W, cpad, bits, parts, exp_out, target_in, target_out, targets, nullptr, 0, stream);
}

extern "C" int niti_mask_features_i8(const int8_t* x, const int8_t* mask, int8_t* y, int64_t rows, int features,
                                     const int32_t* exp_in, int32_t* exp_out, int exp_add, void* stream) {
  clear_error();
  if (rows < 0 || features <= 0 || features % 16 != 0)
    return fail(NITI_ERR_INVALID_ARG, "mask_features: rows=%lld features=%d (a multiple of 16)", static_cast<long long>(rows), features);
  if (x == nullptr || mask == nullptr || y == nullptr) return fail(NITI_ERR_INVALID_ARG, "mask_features: null pointer");
  if (!aligned16(x) || !aligned16(mask) || !aligned16(y)) return fail(NITI_ERR_INVALID_ARG, "mask_features: pointers must be 16-byte aligned");
  const int64_t nv = rows * (features >> 4);
  hipLaunchKernelGGL(mask_features_kernel, dim3(grid_for(nv > 0 ? nv : 1, 256)), dim3(256), 0, static_cast<hipStream_t>(stream), x, mask, y,
                     rows, features, exp_in, exp_out, exp_add);
  return check_launch("mask_features");
}

extern "C" int niti_relu_i8_bwd(const int8_t* act, const int8_t* dy, int8_t* dx, int64_t n, void* stream) {
  clear_error();
  if (n < 0) return fail(NITI_ERR_INVALID_ARG, "relu_bwd: n=%lld", static_cast<long long>(n));
  if (n == 0) return NITI_OK;
  if (act == nullptr || dy == nullptr || dx == nullptr) return fail(NITI_ERR_INVALID_ARG, "relu_bwd: null pointer");
  hipLaunchKernelGGL(relu_kernel<true>, dim3(grid_for((n + 15) / 16, 256)), dim3(256), 0, static_cast<hipStream_t>(stream),
                     act, dy, dx, n);
  return check_launch("relu_bwd");
}
