// int8 GEMM with int32 results for operands whose reduction index is the slow one in b, both staged through LDS as whole
// 128-byte lines, read as they are stored:
//   NN  c[m][n] = sum_k a[m][k] b[k][n]   - the form the reference's extension receives (int8mm.cpp:9-14,
//       int8mm_kernel.cu:8-34; ti_torch.py:152-176 hands it row-major [m,k] and [k,n])
//   TT  c[m][n] = sum_k a[k][m] b[n][k]   - the NN product of (b, a) written transposed: how the drop-in int8_mm
//       fills the [n,m] buffer whose transposed view the reference returns (int8mm.cpp:9-14)
// (n and k multiples of 128) A workgroup owns 32 rows x 128 columns of c and a range of the reduction, and runs the
// whole-line product of nn_lines.h over it.  blockIdx.z splits the reduction when the tiles alone would leave most of the
// device idle: the parts then write int32 partial results and km_reduce_parts_kernel adds them.
// Other products: gemm_any.hip.
#include "common.h"
#include "gemm_any.h"
#include "nn_lines.h"

namespace niti {
namespace {

constexpr int kLnPatchPitch = 128 * 4 + 16;

struct LnArgs {
  const int8_t* a;
  const int8_t* b;
  int32_t* out;           // c, or the partial results [part][m * n]
  uint32_t* absmax;
  int m, n, k;
  int chunks_per_part;
  int parts;
  int roundtrip;
  int transposed_out;
};

__global__ __launch_bounds__(512) void gemm_nn_lines_kernel(const LnArgs g) {
  extern __shared__ __attribute__((aligned(16))) int8_t smem[];   // the stages; later 16 KB of parked sums, then the patch
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n0 = blockIdx.x * 128;
  const int m0 = blockIdx.y * 32;
  const int c0 = blockIdx.z * g.chunks_per_part;
  const int nchunks = min(g.chunks_per_part, (g.k >> 7) - c0);
  const int ft = wave & 3, kh = wave >> 2;
  const int lr = lane & 31, lk = lane >> 5;
  v16i acc = lines_product(g.a, g.b, g.m, g.n, g.k, m0, n0, c0, nchunks, smem);
  lines_add_halves(acc, smem);
  // element 4 q + e of a lane is column n0 + ft * 32 + 8 q + 4 (lane / 32) + e of row m0 + lane % 32
  const bool last = g.parts == 1;
  int32_t* const out = g.out + static_cast<long long>(blockIdx.z) * g.m * g.n;
  int8_t* const patch = smem + 16384;                            // [32 rows][128 columns] of int32, clear of the parked sums
  if (kh == 0) {
    uint32_t lmax = 0;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      int v = acc[e];
      if (last && g.roundtrip) v = f32_roundtrip(v);
      acc[e] = v;
      const uint32_t u = uabs(v);                         // rows beyond m are sums of zeros
      lmax = u > lmax ? u : lmax;
    }
    if (last && g.absmax != nullptr) fold_absmax(g.absmax, lmax);
    if (g.transposed_out) {   // 32 lanes write 32 consecutive rows of one column: a line
      if (m0 + lr < g.m) {
#pragma unroll
        for (int e = 0; e < 16; ++e)
          out[static_cast<long long>(n0 + ft * 32 + 8 * (e >> 2) + 4 * lk + (e & 3)) * g.m + m0 + lr] = acc[e];
      }
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<v4i*>(patch + lr * kLnPatchPitch + (ft * 32 + 8 * q + 4 * lk) * 4) =
            v4i{acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
    }
  }
  if (g.transposed_out) return;
  __syncthreads();
  const int row = tid >> 4, p16 = tid & 15;
  if (m0 + row >= g.m) return;
#pragma unroll
  for (int i = 0; i < 2; ++i)
    *reinterpret_cast<v4i*>(out + static_cast<long long>(m0 + row) * g.n + n0 + (p16 + 16 * i) * 4) =
        *reinterpret_cast<const v4i*>(patch + row * kLnPatchPitch + (p16 + 16 * i) * 16);
}

// c[i] = sum over the parts of the partial results: two elements per thread (the result is small - many short
// wavefronts cover the device better than few long ones), the loads of eight parts in flight together
__global__ __launch_bounds__(256) void km_reduce_parts_kernel(const int32_t* __restrict__ part, int32_t* __restrict__ c, long long pairs, int parts,
                                                              int roundtrip, uint32_t* absmax) {
  const long long i = static_cast<long long>(blockIdx.x) * 256 + threadIdx.x;
  uint32_t lmax = 0;
  if (i < pairs) {
    v2i s = {0, 0};
    for (int p0 = 0; p0 < parts; p0 += 8) {
      v2i v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int p = p0 + u < parts ? p0 + u : p0;          // a repeated part is not added below
        v[u] = *reinterpret_cast<const v2i*>(part + 2 * (static_cast<long long>(p) * pairs + i));
      }
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (p0 + u < parts) s += v[u];
    }
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      if (roundtrip) s[e] = f32_roundtrip(s[e]);
      const uint32_t u = uabs(s[e]);
      lmax = u > lmax ? u : lmax;
    }
    *reinterpret_cast<v2i*>(c + 2 * i) = s;
  }
  if (absmax != nullptr) fold_absmax(absmax, lmax);
}

// The whole-line kernel's plan for an NN product (after the TT form has been turned into one): 0 parts = not taken.
struct LnPlan {
  int parts, chunks_per_part;
};
LnPlan lines_plan(int m, int n, int k) {
  LnPlan p{0, 0};
  if (n % 128 != 0 || k % 128 != 0 || (m + 31) / 32 > 65535) return p;
  if (static_cast<long long>(m) * k >= 0x7fffffffLL || static_cast<long long>(k) * n >= 0x7fffffffLL) return p;
  static const bool off = [] {
    const char* e = getenv("NITI_GEMM_LINES");
    return e != nullptr && e[0] == '0';
  }();
  if (off) return p;
  const long long tiles = static_cast<long long>(n / 128) * ((m + 31) / 32);
  const int chunks = k / 128;
  int parts = 1;
  if (tiles < 192) {
    parts = static_cast<int>((256 + tiles - 1) / tiles);
    if (parts > chunks / 2) parts = chunks / 2;
    if (parts > 32) parts = 32;
    if (parts < 1) parts = 1;
  }
  p.chunks_per_part = (chunks + parts - 1) / parts;
  p.parts = (chunks + p.chunks_per_part - 1) / p.chunks_per_part;
  return p;
}

}  // namespace

// Extents that every kernel which may take the product reads as stored: niti_gemm_i8_workspace counts no copies of the operands.
// (gemm_any.hip reads all others as stored as well, but the workspace stays what callers have been told.)
bool gemm_in_place_shape(int trans_a, int trans_b, int m, int n, int k) {
  if (m <= 0 || n <= 0 || k <= 0 || k % 32 != 0) return false;
  if (trans_b != 0) return trans_a != 0 && m % 32 == 0 && (n + 127) / 128 <= 65535;   // TT = NN of (b, a), transposed
  if (n % 32 != 0) return false;
  if (trans_a != 0 && m % 16 != 0) return false;
  return (m + 127) / 128 <= 65535;
}

// Where this kernel is the faster one: this / gemm_any.hip, us, the same operands again and again (they lie in the caches) and new
// ones at every call (they do not), at 512 ... 8192 steps for eight results in each form.
//   Rows of tiles that fill the device without 128 x 128 tiles doing so: 512 x 2048 NN at 512 steps 4.8 / 5.0 and new 5.0 / 5.4, 1024
//   6.1 / 6.2 and 6.9 / 7.1, 3072 11.1 / 14.3 and 20.3 / 17.0, 5120 17.6 / 21.0 and 33.0 / 27.2, 6144 26.9 / 24.4 and 38.4 / 31.7:
//   taken up to 5120 while b stays in the caches (128 x 8192 at 3072 11.1 / 14.4, 4096 21.5 / 17.6).  TT, whose stores are columns:
//   384 x 2048 at 512 4.4 / 4.6 and 4.6 / 4.7, 1024 5.6 / 5.7 and 6.6 / 6.0, 2048 8.1 / 7.7 and 10.4 / 8.4, 4096 17.9 / 11.7.
//   The reduction split over workgroups (two launches): 128 x 1024 NN at 3072 8.0 / 6.4 and 8.3 / 9.1, 4096 8.4 / 7.5 and 8.8 / 11.1, 5120
//   8.6 / 8.3 and 9.5 / 13.1, 6144 8.9 / 9.4 and 10.7 / 17.2, 8192 9.5 / 17.5; TT of it 5120 8.4 / 7.9 and 9.2 / 11.8; 128 x 128 NN at
//   4096 6.7 / 6.6 and 6.7 / 9.3; 512 x 512 at 5120 10.2 / 10.2 and 11.8 / 11.9.
bool gemm_lines_shape(int trans_a, int trans_b, int m, int n, int k) {
  if ((trans_a != 0) != (trans_b != 0) || !gemm_in_place_shape(trans_a, trans_b, m, n, k)) return false;
  if (gemm_any_large(m, n)) return false;
  const LnPlan p = trans_b != 0 ? lines_plan(n, m, k) : lines_plan(m, n, k);
  if (p.parts > 1) return k > 5000;
  return p.parts == 1 && k >= 512 && (trans_b != 0 ? k < 1024 : k <= 5120 && static_cast<long long>(k) * n <= (24 << 20));
}

// bytes of partial results the whole-line kernel wants for this product (0: none)
size_t gemm_lines_workspace(int trans_a, int trans_b, int m, int n, int k) {
  if (trans_b != 0) {
    const int t = m;
    m = n;
    n = t;
    trans_a = 0;
  }
  if (trans_a != 0) return 0;
  const LnPlan p = lines_plan(m, n, k);
  return p.parts > 1 ? static_cast<size_t>(p.parts) * m * n * 4 : 0;
}

int launch_gemm_lines(int trans_b, const int8_t* a, const int8_t* b, int32_t* c, int m, int n, int k, bool roundtrip, uint32_t* absmax,
                      void* workspace, hipStream_t stream) {
  // TT: rows of the kernel's product = n (rows of b), columns = m (columns of a)
  LnArgs l{trans_b != 0 ? b : a, trans_b != 0 ? a : b, c, absmax, trans_b != 0 ? n : m, trans_b != 0 ? m : n, k, 0, 0, roundtrip ? 1 : 0, trans_b};
  const LnPlan p = lines_plan(l.m, l.n, k);
  l.chunks_per_part = p.chunks_per_part;
  l.parts = p.parts;
  if (p.parts > 1) l.out = static_cast<int32_t*>(workspace);
  static bool attr_set[kDeviceSlots] = {};
  bool& done = attr_set[device_slot()];
  if (!done) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_nn_lines_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kLinesLdsBytes) != hipSuccess)
      return fail(NITI_ERR_LAUNCH, "gemm: cannot reserve %d bytes of LDS", kLinesLdsBytes);
    done = true;
  }
  hipLaunchKernelGGL(gemm_nn_lines_kernel, dim3(l.n / 128, (l.m + 31) / 32, p.parts), dim3(512), static_cast<size_t>(kLinesLdsBytes), stream, l);
  if (p.parts > 1) {
    const long long pairs = static_cast<long long>(l.m) * l.n / 2;
    hipLaunchKernelGGL(km_reduce_parts_kernel, dim3(static_cast<unsigned>((pairs + 255) / 256)), dim3(256), 0, stream,
                       static_cast<const int32_t*>(workspace), c, pairs, p.parts, l.roundtrip, absmax);
  }
  return check_launch("gemm_nn_lines");
}

}  // namespace niti
