// Convolution entries of niti_amd._host (see host.h).
#include "host.h"

#include <ATen/ops/slice.h>

namespace niti_host {
namespace {

struct Dims {
  int N, H, W, C, K, R, S;   // the forward convolution's extents
};
int out_extent(int in, int r, int stride, int pad) {
  const int t = in + 2 * pad - r;
  return stride <= 0 || t < 0 ? 0 : t / stride + 1;
}
Dims forward_dims(const at::Tensor& x, const at::Tensor& w, const char* who) {
  if (x.dim() != 4 || w.dim() != 4) refuse(std::string(who) + ": [N,H,W,C] and [K,R,S,C] tensors expected");
  const Dims d{static_cast<int>(x.size(0)), static_cast<int>(x.size(1)), static_cast<int>(x.size(2)), static_cast<int>(x.size(3)),
               static_cast<int>(w.size(0)), static_cast<int>(w.size(1)), static_cast<int>(w.size(2))};
  if (w.size(3) != d.C)
    refuse(std::string(who) + ": channel mismatch " + std::to_string(d.C) + " vs " + std::to_string(w.size(3)));
  return d;
}
// extents of the convolution whose error map is `err`
Dims gradient_dims(const at::Tensor& err, const at::Tensor& w, int pad, const char* who) {
  if (err.dim() != 4 || w.dim() != 4) refuse(std::string(who) + ": [N,P,Q,K] and [K,R,S,C] tensors expected");
  const int R = static_cast<int>(w.size(1)), S = static_cast<int>(w.size(2));
  if (w.size(0) != err.size(3)) refuse(std::string(who) + ": channel mismatch");
  return Dims{static_cast<int>(err.size(0)), static_cast<int>(err.size(1)) - 2 * pad + R - 1, static_cast<int>(err.size(2)) - 2 * pad + S - 1,
              static_cast<int>(w.size(3)), static_cast<int>(w.size(0)), R, S};
}

// a kernel-ready filter copy that a launch reads (or, forward, keeps in step)
void want_copy(Opt prepared, const Dims& d, int stride, int pad, int dgrad, const char* who) {
  if (prepared == nullptr) return;
  want_bytes(*prepared, static_cast<int64_t>(niti_conv2d_i8_filter_workspace(d.N, d.H, d.W, d.C, d.K, d.R, d.S, stride, pad, dgrad)), who, "a prepared filter");
}

struct Rounding {
  int bits, method, div, bw;
};
Rounding rounding_of(Args& a) {
  Rounding r;
  r.bits = a.i();
  r.method = a.i();
  r.div = a.i();
  r.bw = a.i();
  return r;
}

bool is_i8(const at::Tensor& t) { return t.scalar_type() == at::kChar; }
bool aligned16(const at::Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; }

// ---- int32 results -----------------------------------------------------------------------------------------------
at::Tensor fprop_i32(const at::Tensor& x, const at::Tensor& w, int stride, int pad, unsigned flags, uint32_t* absmax, Opt prepared) {
  const char* who = "conv2d_fprop";
  if (!is_i8(x) || !is_i8(w)) refuse(std::string(who) + ": int8 tensors expected");
  const Dims d = forward_dims(x, w, who);
  at::Tensor y = empty32({d.N, out_extent(d.H, d.R, stride, pad), out_extent(d.W, d.S, stride, pad), d.K}, x);
  at::Tensor ws;
  size_t bytes = 0;
  const int8_t* wp = prepared != nullptr ? ptr<int8_t>(*prepared) : ptr<int8_t>(w);
  want_copy(prepared, d, stride, pad, 0, who);
  if (prepared != nullptr) {
    flags |= NITI_CONV_FILTER_PREPARED;
  } else {
    bytes = niti_conv2d_i8_filter_workspace(d.N, d.H, d.W, d.C, d.K, d.R, d.S, stride, pad, 0);
    if (bytes > 0) ws = empty8({static_cast<int64_t>(bytes)}, x);
  }
  check(niti_conv2d_i8_fprop(ptr<int8_t>(x), wp, ptr<int32_t>(y), d.N, d.H, d.W, d.C, d.K, d.R, d.S, stride, pad, flags, absmax,
                             bytes > 0 ? ws.data_ptr() : nullptr, bytes, stream_of(x)),
        "niti_conv2d_i8_fprop");
  return y;
}

// `prepared`: a kernel-ready filter copy; `forward_copy`: it is the forward pass's
at::Tensor dgrad_i32(const at::Tensor& err, const at::Tensor& w, int stride, int pad, unsigned flags, uint32_t* absmax, Opt prepared,
                     bool forward_copy) {
  const Dims d = gradient_dims(err, w, pad, "conv2d_dgrad");
  want_copy(prepared, d, stride, pad, forward_copy ? 0 : 1, "conv2d_dgrad");
  if (d.H < 0 || d.W < 0) refuse("conv2d_dgrad: filter larger than the padded input");
  at::Tensor dx = empty32({d.N, d.H, d.W, d.C}, err);
  at::Tensor ws;
  size_t bytes = 0;
  const int8_t* wp = ptr<int8_t>(w);
  if (prepared != nullptr) {
    flags |= NITI_CONV_FILTER_PREPARED | (forward_copy ? NITI_CONV_FILTER_FORWARD_COPY : 0u);
    wp = ptr<int8_t>(*prepared);
  } else {
    bytes = niti_conv2d_i8_filter_workspace(d.N, d.H, d.W, d.C, d.K, d.R, d.S, stride, pad, 1);
    ws = empty8({static_cast<int64_t>(bytes > 16 ? bytes : 16)}, err);
  }
  check(niti_conv2d_i8_dgrad(ptr<int8_t>(err), wp, ptr<int32_t>(dx), d.N, d.H, d.W, d.C, d.K, d.R, d.S, stride, pad, flags, absmax,
                             prepared != nullptr ? nullptr : ws.data_ptr(), bytes, stream_of(err)),
        "niti_conv2d_i8_dgrad");
  return dx;
}

at::Tensor wgrad_i32(const at::Tensor& act, const at::Tensor& err, int R, int S, int stride, int pad, unsigned flags, uint32_t* absmax, Opt workspace) {
  if (act.dim() != 4 || err.dim() != 4) refuse("conv2d_wgrad: [N,H,W,C] and [N,P,Q,K] tensors expected");
  const int N = static_cast<int>(act.size(0)), H = static_cast<int>(act.size(1)), W = static_cast<int>(act.size(2)),
            C = static_cast<int>(act.size(3)), K = static_cast<int>(err.size(3));
  want_bytes(err, static_cast<int64_t>(N) * out_extent(H, R, 1, pad) * out_extent(W, S, 1, pad) * K, "conv2d_wgrad", "an error map");
  const size_t bytes = niti_conv2d_i8_wgrad_workspace(N, H, W, C, K, R, S, pad);
  at::Tensor ws = workspace != nullptr ? *workspace : scratch(bytes, act);
  if (static_cast<size_t>(ws.numel()) < bytes)
    refuse("conv2d_wgrad: workspace of " + std::to_string(bytes) + " bytes needed, got " + std::to_string(ws.numel()));
  at::Tensor dw = empty32({K, R, S, C}, act);
  check(niti_conv2d_i8_wgrad(ptr<int8_t>(act), ptr<int8_t>(err), ptr<int32_t>(dw), N, H, W, C, K, R, S, stride, pad, flags, absmax, ws.data_ptr(),
                             bytes, stream_of(act)),
        "niti_conv2d_i8_wgrad");
  return dw;
}

// fprop(x, w, stride, pad, flags, absmax, prepared) -> y
PyObject* fprop(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    Args a(args, n, 7, "conv2d_fprop");
    const at::Tensor& x = a.tensor();
    const at::Tensor& w = a.tensor();
    const int stride = a.i(), pad = a.i();
    const unsigned flags = static_cast<unsigned>(a.integer());
    Opt am = a.opt();
    return wrap(fprop_i32(x, w, stride, pad, flags, ptr<uint32_t>(am), a.opt()));
  });
}

// sp_conv(x, w, stride, pad): the drop-in convolution, results through float32 (cutlassconv_kernel.cu:180-319)
PyObject* sp_conv(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    if (n != 4) refuse("sp_conv: 4 arguments expected");
    const char* names[2] = {"input", "weight"};
    for (int i = 0; i < 2; ++i) {
      if (!THPVariable_Check(args[i])) refuse(std::string(names[i]) + " must be a tensor");
      const at::Tensor& t = THPVariable_Unpack(args[i]);
      if (!t.is_cuda()) refuse(std::string(names[i]) + " must be a CUDA tensor");
      if (!t.is_contiguous()) refuse(std::string(names[i]) + " must be contiguous");
      if (!is_i8(t)) refuse(std::string("expected scalar type Char but found ") + c10::toString(t.scalar_type()));
    }
    Args a(args, n, 4, "sp_conv");
    const at::Tensor& x = a.tensor();
    const at::Tensor& w = a.tensor();
    const int stride = a.i(), pad = a.i();
    return wrap(fprop_i32(x, w, stride, pad, NITI_EPI_F32_ROUNDTRIP, nullptr, nullptr));
  });
}

// dgrad(err, w, stride, pad, flags, absmax, prepared, forward_copy) -> dx
PyObject* dgrad(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    Args a(args, n, 8, "conv2d_dgrad");
    const at::Tensor& err = a.tensor();
    const at::Tensor& w = a.tensor();
    const int stride = a.i(), pad = a.i();
    const unsigned flags = static_cast<unsigned>(a.integer());
    Opt am = a.opt(), prepared = a.opt();
    return wrap(dgrad_i32(err, w, stride, pad, flags, ptr<uint32_t>(am), prepared, a.flag()));
  });
}

// wgrad(act, err, R, S, stride, pad, flags, absmax, workspace) -> dw
PyObject* wgrad(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    Args a(args, n, 9, "conv2d_wgrad");
    const at::Tensor& act = a.tensor();
    const at::Tensor& err = a.tensor();
    const int R = a.i(), S = a.i(), stride = a.i(), pad = a.i();
    const unsigned flags = static_cast<unsigned>(a.integer());
    Opt am = a.opt();
    return wrap(wgrad_i32(act, err, R, S, stride, pad, flags, ptr<uint32_t>(am), a.opt()));
  });
}

// ---- results rounded to int8 in the launch -------------------------------------------------------------------------
struct Fused {
  bool current = false;   // forward: w holds the filter itself (next to `prepared`)
  bool dgrad = false, f32 = false, relu = false, hint = false, forward_copy = false, any_shape = false;
  int stride = 1, pad = 1, ties = 0;
  Rounding r{};
  Opt sync = nullptr, shift = nullptr, exp_a = nullptr, exp_b = nullptr, exp_out = nullptr, prepared = nullptr, mask = nullptr, pool_out = nullptr,
      pool_in = nullptr, rand = nullptr;
};

// Convolution + requantisation.  `soft` (a layer asking): returns false, with nothing launched, where the single-launch
// kernels do not cover the call or the device is too small for them.
bool conv_requant(const at::Tensor& x, const at::Tensor& w, const Dims& d, const Fused& f, bool soft, at::Tensor* y, at::Tensor* shift,
                  at::Tensor* sync_view, const char* who) {
  const int dg = f.dgrad ? 1 : 0;
  const bool sto = f.r.method == NITI_ROUND_STOCHASTIC;
  std::vector<int64_t> shape = f.dgrad ? std::vector<int64_t>{d.N, d.H, d.W, d.C}
                                       : std::vector<int64_t>{d.N, out_extent(d.H, d.R, f.stride, f.pad), out_extent(d.W, d.S, f.stride, f.pad), d.K};
  if (soft && sto && (f.pool_in != nullptr || d.H == 2)) return false;
  if (sto) {
    if (f.rand == nullptr || f.rand->scalar_type() != at::kInt || !has_shape(*f.rand, shape)) {
      if (soft) return false;
      refuse(std::string(who) + ": stochastic rounding needs `rand`, a contiguous int32 tensor shaped like the output");
    }
    if (f.pool_in != nullptr) refuse_niti(std::string(who) + ": stochastic rounding is not folded in together with the pooling's backward pass");
  } else if (f.rand != nullptr) {
    refuse(std::string(who) + ": `rand` is only used by method='sto'");
  }
  if (f.mask != nullptr && (!is_i8(*f.mask) || !has_shape(*f.mask, shape))) refuse(std::string(who) + ": relu_mask must be int8 and shaped like the output");
  if (f.pool_in != nullptr) {   // the result is written at the pooling input's size
    const std::vector<int64_t> big{shape[0], 2 * shape[1], 2 * shape[2], shape[3]};
    if (f.mask == nullptr || !is_i8(*f.pool_in) || !has_shape(*f.pool_in, big))
      refuse(std::string(who) + ": unpool needs relu_mask (the pooled map) and a contiguous int8 [N,2H,2W,C] pooling input");
    shape = big;
  }
  if (!is_i8(x) || !is_i8(w)) refuse(std::string(who) + ": int8 tensors expected");
  const bool any = soft || f.any_shape;
  // few images: the kernel for any shape, which reads the filter as stored
  const size_t small = soft && f.current ? niti_conv2d_i8_fprop_small_sync_words(d.N, d.H, d.W, d.C, d.K, d.R, d.S, f.stride, f.pad) : 0;
  const size_t words = small > 0 ? small : any ? niti_conv2d_i8_requant_sync_words_any(d.N, d.H, d.W, d.C, d.K, d.R, d.S, f.stride, f.pad, dg)
                           : niti_conv2d_i8_requant_sync_words(d.N, d.H, d.W, d.C, d.K, d.R, d.S, f.stride, f.pad, dg);
  if (words == 0) {
    if (soft) return false;
    refuse_niti(std::string(who) + ": shape not covered by the single-launch path");
  }
  size_t have = 0;
  uint32_t* sync = sync_words(f.sync, words, x, sync_view, &have, who);
  *y = empty8(shape, x);
  if (f.hint && f.shift == nullptr) refuse(std::string(who) + ": shift_hint needs shift_out, holding the predicted shift");
  *shift = f.shift != nullptr ? *f.shift : scalar32(x);
  unsigned flags = f.f32 ? NITI_EPI_F32_ROUNDTRIP : 0u;
  at::Tensor ws;
  size_t bytes = 0;
  const int8_t* wp = ptr<int8_t>(w);
  if (small > 0) {
    // nothing to prepare
  } else if (f.prepared != nullptr) {
    want_copy(f.prepared, d, f.stride, f.pad, f.dgrad && !f.forward_copy ? 1 : 0, who);
    flags |= NITI_CONV_FILTER_PREPARED | (f.forward_copy ? NITI_CONV_FILTER_FORWARD_COPY : 0u);
    wp = ptr<int8_t>(*f.prepared);
  } else {
    // only the 3x3 kernels, whose maps are squares of a power of two, read a copy of the filter
    if (!any || (d.R == 3 && d.S == 3 && d.H == d.W && (d.H & (d.H - 1)) == 0)) {
      bytes = niti_conv2d_i8_filter_workspace(d.N, d.H, d.W, d.C, d.K, d.R, d.S, f.stride, f.pad, dg);
      ws = empty8({static_cast<int64_t>(bytes > 16 ? bytes : 16)}, x);
    }
  }
  void* wsp = ws.defined() ? ws.data_ptr() : nullptr;
  const unsigned rq = (f.relu ? NITI_RQ_RELU : 0u) | (f.hint ? NITI_RQ_SHIFT_HINT : 0u) | (any ? NITI_RQ_ANY_SHAPE : 0u) | (small > 0 ? NITI_RQ_ANY_KERNEL : 0u);
  const int8_t* xp = ptr<int8_t>(x);
  int8_t* yp = ptr<int8_t>(*y);
  int32_t* sp = ptr<int32_t>(*shift);
  const int32_t *ea = ptr<int32_t>(f.exp_a), *eb = ptr<int32_t>(f.exp_b);
  int32_t* eo = ptr<int32_t>(f.exp_out);
  void* st = stream_of(x);
  int rc;
  if (sto && !f.dgrad)
    rc = niti_conv2d_i8_fprop_requant_sto(xp, wp, yp, ptr<int8_t>(f.pool_out), ptr<int32_t>(f.rand), d.N, d.H, d.W, d.C, d.K, d.R, d.S, f.stride,
                                          f.pad, flags, f.r.bits, f.r.div, f.r.bw, rq, sync, have, sp, ea, eb, eo, wsp, bytes, st);
  else if (sto)
    rc = niti_conv2d_i8_dgrad_requant_sto(xp, wp, yp, ptr<int32_t>(f.rand), d.N, d.H, d.W, d.C, d.K, d.R, d.S, f.stride, f.pad, flags, f.r.bits,
                                          f.r.div, f.r.bw, rq, ptr<int8_t>(f.mask), sync, have, sp, ea, eb, eo, wsp, bytes, st);
  else if (f.pool_in != nullptr)
    rc = niti_conv2d_i8_dgrad_requant_unpool(xp, wp, yp, ptr<int8_t>(f.mask), ptr<int8_t>(f.pool_in), f.ties, d.N, d.H, d.W, d.C, d.K, d.R, d.S,
                                             f.stride, f.pad, flags, f.r.bits, f.r.method, f.r.div, f.r.bw, rq, sync, have, sp, ea, eb, eo, wsp,
                                             bytes, st);
  else if (f.dgrad)
    rc = niti_conv2d_i8_dgrad_requant(xp, wp, yp, d.N, d.H, d.W, d.C, d.K, d.R, d.S, f.stride, f.pad, flags, f.r.bits, f.r.method, f.r.div, f.r.bw,
                                      rq, ptr<int8_t>(f.mask), sync, have, sp, ea, eb, eo, wsp, bytes, st);
  else if (f.pool_out != nullptr)
    rc = niti_conv2d_i8_fprop_requant_pool(xp, wp, yp, ptr<int8_t>(f.pool_out), d.N, d.H, d.W, d.C, d.K, d.R, d.S, f.stride, f.pad, flags, f.r.bits,
                                           f.r.method, f.r.div, f.r.bw, rq, sync, have, sp, ea, eb, eo, wsp, bytes, st);
  else
    rc = niti_conv2d_i8_fprop_requant(xp, wp, yp, d.N, d.H, d.W, d.C, d.K, d.R, d.S, f.stride, f.pad, flags, f.r.bits, f.r.method, f.r.div, f.r.bw,
                                      rq, sync, have, sp, ea, eb, eo, wsp, bytes, st);
  if (soft) return check_fits(rc, who);
  check(rc, who);
  return true;
}

// int32 sums -> int8, for the shapes outside the single-launch kernels
at::Tensor requant_i32(const at::Tensor& acc, const uint32_t* absmax, const Rounding& r, Opt rand, bool relu, int32_t* shift, Opt exp_a, Opt exp_b,
                       int32_t* exp_out) {
  if (rand != nullptr && (rand->scalar_type() != at::kInt || rand->numel() != acc.numel()))
    refuse("requant: rand must be int32 with one entry per element");
  at::Tensor y = empty8(acc.sizes(), acc);
  check(niti_requant_i32_i8(ptr<int32_t>(acc), ptr<int8_t>(y), acc.numel(), absmax, r.bits, r.method, r.div, r.bw, ptr<int32_t>(rand),
                            relu ? NITI_RQ_RELU : 0u, shift, ptr<int32_t>(exp_a), ptr<int32_t>(exp_b), exp_out, stream_of(acc)),
        "niti_requant_i32_i8");
  return y;
}

// requant_op(who, x, w, stride, pad, f32, bits, method, div, bw, relu, hint, sync, shift, exp_a, exp_b, exp_out, prepared,
//            forward_copy, mask, pool_out, pool_in, ties, rand, any_shape) -> (y, shift, sync): ops.conv2d_*_requant
PyObject* requant_op(PyObject* const* args, Py_ssize_t n, bool dg) {
  return guarded([&]() -> PyObject* {
    const char* who = dg ? "niti_conv2d_i8_dgrad_requant" : "niti_conv2d_i8_fprop_requant";
    Args a(args, n, 24, who);
    const at::Tensor& x = a.tensor();
    const at::Tensor& w = a.tensor();
    Fused f;
    f.dgrad = dg;
    f.stride = a.i();
    f.pad = a.i();
    f.f32 = a.flag();
    f.r = rounding_of(a);
    f.relu = a.flag();
    f.hint = a.flag();
    f.sync = a.opt();
    f.shift = a.opt();
    f.exp_a = a.opt();
    f.exp_b = a.opt();
    f.exp_out = a.opt();
    f.prepared = a.opt();
    f.forward_copy = a.flag();
    f.mask = a.opt();
    f.pool_out = a.opt();
    f.pool_in = a.opt();
    f.ties = a.i();
    f.rand = a.opt();
    f.any_shape = a.flag();
    const Dims d = dg ? gradient_dims(x, w, f.pad, who) : forward_dims(x, w, who);
    if (f.pool_out != nullptr &&
        (!is_i8(*f.pool_out) || !has_shape(*f.pool_out, {d.N, out_extent(d.H, d.R, f.stride, f.pad) / 2, out_extent(d.W, d.S, f.stride, f.pad) / 2, d.K})))
      refuse("conv2d_fprop_requant: pool_out must be a contiguous int8 [N,P/2,Q/2,K] tensor");
    at::Tensor y, shift, sync;
    conv_requant(x, w, d, f, false, &y, &shift, &sync, who);
    return tuple_of({y, shift, sync});
  });
}
PyObject* fprop_requant(PyObject*, PyObject* const* args, Py_ssize_t n) { return requant_op(args, n, false); }
PyObject* dgrad_requant(PyObject*, PyObject* const* args, Py_ssize_t n) { return requant_op(args, n, true); }

// layer_forward(fuse, x, w, stride, pad, f32, bits, method, div, bw, relu, shift state, exp_a, exp_b, prepared, pool, rand,
//               w current?)
//   -> (y, exponent, pooled map or None)
// TiConv2d.forward: convolution, act_calc and where asked the ReLU and the 2x2 max-pool behind it (`pool`), in one launch
// where the single-launch kernels cover the shape; otherwise convolution, then requantisation (nothing pooled).
PyObject* layer_forward(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    Args a(args, n, 18, "conv layer forward");
    const bool fuse = a.flag();
    const at::Tensor& x = a.tensor();
    const at::Tensor& w = a.tensor();
    Fused f;
    f.stride = a.i();
    f.pad = a.i();
    f.f32 = a.flag();
    f.r = rounding_of(a);
    f.relu = a.flag();
    f.shift = a.opt();
    f.hint = f.shift != nullptr;
    f.exp_a = a.exponent();
    f.exp_b = a.exponent();
    f.prepared = a.opt();
    const bool pool = a.flag();
    f.rand = a.opt();
    f.current = a.flag();
    const Dims d = forward_dims(x, w, "conv layer");
    at::Tensor y, shift, pooled, e = scalar32(x);
    f.exp_out = &e;
    if (fuse) {
      // the 3x3 kernels' maps
      if (pool && f.relu && f.stride == 1 && f.pad == 1 && d.R == 3 && d.S == 3 && d.H == d.W && d.H >= 2 && d.H <= 32 && (d.H & (d.H - 1)) == 0) {
        pooled = empty8({d.N, d.H / 2, d.W / 2, d.K}, x);
        f.pool_out = &pooled;
      }
      if (conv_requant(x, w, d, f, true, &y, &shift, nullptr, "niti_conv2d_i8_fprop_requant")) return tuple_of({y, e, pooled});
      if (f.pool_out != nullptr) {
        f.pool_out = nullptr;
        if (conv_requant(x, w, d, f, true, &y, &shift, nullptr, "niti_conv2d_i8_fprop_requant")) return tuple_of({y, e, at::Tensor()});
      }
    }
    uint32_t* am = arena_take(1, x, nullptr);
    at::Tensor acc = fprop_i32(x, w, f.stride, f.pad, f.f32 ? NITI_EPI_F32_ROUNDTRIP : 0u, am, f.prepared);
    y = requant_i32(acc, am, f.r, f.rand, f.relu, nullptr, f.exp_a, f.exp_b, ptr<int32_t>(e));
    return tuple_of({y, e, at::Tensor()});
  });
}

struct DataGradient {
  at::Tensor y, e;
  bool unpooled = false;
};
// TiConv2d.backward's data gradient: err_calc(conv_dgrad(err, w)), zeroed where `f.mask` (the layer's input) is not positive,
// and - `pool_in` given - routed through the 2x2 max-pool in front of the layer, one launch where the kernels cover it.
void data_gradient(bool fuse, const at::Tensor& err, const at::Tensor& w, Fused f, Opt pool_in, DataGradient* r) {
  const Dims d = gradient_dims(err, w, f.pad, "conv layer");
  // the forward pass's copy serves the data gradient only where both run the 3x3 kernel
  f.forward_copy = f.prepared != nullptr;
  if (f.forward_copy && niti_conv2d_i8_forward_copy_ok(d.N, d.H, d.W, d.C, d.K, d.R, d.S, f.stride, f.pad) == 0) {
    f.forward_copy = false;
    f.prepared = nullptr;
  }
  at::Tensor shift;
  f.exp_out = &r->e;
  bool done = false;
  if (fuse && pool_in != nullptr && d.H == d.W && d.H <= 32 && (d.H & (d.H - 1)) == 0) {
    f.pool_in = pool_in;
    done = conv_requant(err, w, d, f, true, &r->y, &shift, nullptr, "niti_conv2d_i8_dgrad_requant_unpool");
    r->unpooled = done;
    f.pool_in = nullptr;
  }
  if (fuse && !done) done = conv_requant(err, w, d, f, true, &r->y, &shift, nullptr, "niti_conv2d_i8_dgrad_requant");
  if (!done) {
    uint32_t* am = arena_take(1, err, nullptr);
    at::Tensor dx = dgrad_i32(err, w, f.stride, f.pad, f.f32 ? NITI_EPI_F32_ROUNDTRIP : 0u, am, f.prepared, f.forward_copy);
    r->y = requant_i32(dx, am, f.r, f.rand, false, nullptr, f.exp_a, f.exp_b, ptr<int32_t>(r->e));
    if (f.mask != nullptr)
      check(niti_relu_i8_bwd(ptr<int8_t>(*f.mask), ptr<int8_t>(r->y), ptr<int8_t>(r->y), r->y.numel(), stream_of(err)), "niti_relu_i8_bwd");
  }
}

struct Update {
  at::Tensor g8, dw, shift;
};
// weight gradient + grad_calc + update in one call; `soft` as in conv_requant
bool wgrad_update_fused(const at::Tensor& act, const at::Tensor& err, const at::Tensor& w, int stride, int pad, unsigned flags, const Rounding& r,
                        bool want_grad, bool want_dw, Opt sync, Opt shift, Opt exp_a, Opt exp_b, int32_t* exp_out, Opt workspace, Opt prepared,
                        bool soft, Update* u, at::Tensor* sync_view) {
  const char* who = "niti_conv2d_i8_wgrad_update";
  if (!is_i8(act) || !is_i8(err) || !is_i8(w)) refuse("conv2d_wgrad_update: int8 tensors expected");
  if (act.dim() != 4 || err.dim() != 4 || w.dim() != 4) refuse("conv2d_wgrad_update: four-dimensional tensors expected");
  const int N = static_cast<int>(act.size(0)), H = static_cast<int>(act.size(1)), W = static_cast<int>(act.size(2)), C = static_cast<int>(act.size(3));
  const int K = static_cast<int>(w.size(0)), R = static_cast<int>(w.size(1)), S = static_cast<int>(w.size(2)), Cw = static_cast<int>(w.size(3));
  if (err.size(3) != K) refuse("conv2d_wgrad_update: channel mismatch");
  const size_t words = niti_conv2d_i8_wgrad_update_sync_words(N, H, W, C, K, R, S, stride, pad);
  if (words == 0) {
    if (soft) return false;
    refuse_niti("conv2d_wgrad_update: shape not covered by the single-pass path");
  }
  if (!has_shape(err, {N, out_extent(H, R, 1, pad), out_extent(W, S, 1, pad), K})) refuse("conv2d_wgrad_update: error map does not match the activations");
  want_copy(prepared, Dims{N, H, W, C, K, R, S}, stride, pad, 0, "conv2d_wgrad_update");
  size_t have = 0;
  uint32_t* sp = sync_words(sync, words, act, sync_view, &have, "conv2d_wgrad_update");
  const size_t bytes = niti_conv2d_i8_wgrad_workspace(N, H, W, C, K, R, S, pad);
  at::Tensor ws = workspace != nullptr ? *workspace : scratch(bytes, act);
  if (static_cast<size_t>(ws.numel()) < bytes)
    refuse("conv2d_wgrad_update: workspace of " + std::to_string(bytes) + " bytes needed, got " + std::to_string(ws.numel()));
  if (want_grad) u->g8 = empty8(w.sizes(), w);
  if (want_dw) u->dw = empty32({K, R, S, C}, w);
  u->shift = shift != nullptr ? *shift : scalar32(w);
  const int rc = niti_conv2d_i8_wgrad_update(
      ptr<int8_t>(act), ptr<int8_t>(err), ptr<int8_t>(w), Cw, N, H, W, C, K, R, S, stride, pad, flags, r.bits, r.method, r.div, r.bw, sp, have,
      want_grad ? ptr<int8_t>(u->g8) : nullptr, want_dw ? ptr<int32_t>(u->dw) : nullptr, ptr<int8_t>(prepared), ptr<int32_t>(u->shift),
      ptr<int32_t>(exp_a), ptr<int32_t>(exp_b), exp_out, ws.data_ptr(), bytes, stream_of(act));
  if (soft) return check_fits(rc, who);
  check(rc, who);
  return true;
}

// wgrad_update(act, err, w, stride, pad, flags, mu, method, div, bw, sync, want_grad, want_dw, shift, exp_a, exp_b, exp_out,
//              workspace, prepared) -> (g8, dw, shift, sync)
PyObject* wgrad_update(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    Args a(args, n, 19, "conv2d_wgrad_update");
    const at::Tensor& act = a.tensor();
    const at::Tensor& err = a.tensor();
    const at::Tensor& w = a.tensor();
    const int stride = a.i(), pad = a.i();
    const unsigned flags = static_cast<unsigned>(a.integer());
    const Rounding r = rounding_of(a);
    Opt sync = a.opt();
    const bool want_grad = a.flag(), want_dw = a.flag();
    Opt shift = a.opt(), exp_a = a.opt(), exp_b = a.opt(), exp_out = a.opt(), workspace = a.opt(), prepared = a.opt();
    Update u;
    at::Tensor view;
    wgrad_update_fused(act, err, w, stride, pad, flags, r, want_grad, want_dw, sync, shift, exp_a, exp_b, ptr<int32_t>(exp_out), workspace, prepared,
                       false, &u, &view);
    return tuple_of({u.g8, u.dw, u.shift, view});
  });
}

struct WeightGradient {
  bool want_grad = false, want_dw = false;
  Rounding r{};
  unsigned flags = 0;
  Opt shift = nullptr, exp_a = nullptr, exp_b = nullptr, prepared = nullptr, rand = nullptr;
};
// TiConv2d.backward's weight gradient, grad_calc and update of w in place; returns whether one call did it all.  Without a
// one-call form the int32 gradient (its zero-padded channels dropped) is rounded and applied in a second step and returned.
bool weight_gradient(bool fuse, const at::Tensor& act, const at::Tensor& err, const at::Tensor& w, int stride, int pad, const WeightGradient& g, Update* u,
                     const at::Tensor& e) {
  // the one-call kernels load 16 bytes at a time; operands that start elsewhere are re-laid by the int32 gradient
  const bool one = fuse && aligned16(act) && aligned16(err) && wgrad_update_fused(act, err, w, stride, pad, g.flags | NITI_CONV_ANY_KERNEL | (g.shift != nullptr ? NITI_CONV_SHIFT_HINT : 0u), g.r,
                                              g.want_grad, g.want_dw, nullptr, g.shift, g.exp_a, g.exp_b, ptr<int32_t>(e), nullptr, g.prepared, true, u, nullptr);
  if (one) {
    if (g.want_dw && u->dw.size(3) != w.size(3)) u->dw = u->dw.slice(3, 0, w.size(3)).contiguous();
    return true;
  }
  uint32_t* am = arena_take(1, act, nullptr);
  u->dw = wgrad_i32(act, err, static_cast<int>(w.size(1)), static_cast<int>(w.size(2)), stride, pad, g.flags, am, nullptr);
  // zero-padded input channels give zero gradient columns (they cannot raise the range)
  if (u->dw.size(3) != w.size(3)) u->dw = u->dw.slice(3, 0, w.size(3)).contiguous();
  if (g.rand != nullptr && (g.rand->scalar_type() != at::kInt || g.rand->numel() != u->dw.numel()))
    refuse("grad_update: rand must be int32 with one entry per element");
  if (g.want_grad) u->g8 = empty8(w.sizes(), w);
  u->shift = scalar32(w);
  check(niti_grad_update_i8(ptr<int32_t>(u->dw), ptr<int8_t>(w), u->dw.numel(), am, g.r.bits, g.r.method, g.r.div, g.r.bw, ptr<int32_t>(g.rand),
                            g.want_grad ? ptr<int8_t>(u->g8) : nullptr, ptr<int32_t>(u->shift), ptr<int32_t>(g.exp_a), ptr<int32_t>(g.exp_b), ptr<int32_t>(e),
                            stream_of(act)),
        "niti_grad_update_i8");
  return false;
}

// both in one call where niti_conv2d_i8_backward or niti_conv2d_i8_backward_pair covers them
bool both_gradients(const at::Tensor& act, const at::Tensor& err, const at::Tensor& w, const Fused& f, Opt pool_in, const WeightGradient& g, DataGradient* r,
                    Update* u, const at::Tensor& e) {
  if (f.stride != 1 || g.want_dw || g.rand != nullptr || g.r.method == NITI_ROUND_STOCHASTIC || act.size(3) != w.size(3)) return false;
  if (!is_i8(act) || !is_i8(err) || !is_i8(w)) return false;
  for (Opt t : {&act, &err, &w, f.mask, f.rand, pool_in, g.prepared})
    if (t != nullptr && !aligned16(*t)) return false;
  const Dims d = gradient_dims(err, w, f.pad, "conv layer");
  if (!has_shape(act, {d.N, d.H, d.W, d.C}) || d.R != d.S) return false;
  const bool sto = f.r.method == NITI_ROUND_STOCHASTIC;
  std::vector<int64_t> shape{d.N, d.H, d.W, d.C};
  if (f.mask != nullptr && (!is_i8(*f.mask) || !has_shape(*f.mask, shape))) return false;
  if (sto && (f.rand == nullptr || f.rand->scalar_type() != at::kInt || !has_shape(*f.rand, shape))) return false;
  if (pool_in != nullptr) {
    shape = {d.N, 2LL * d.H, 2LL * d.W, d.C};
    if (sto || f.mask == nullptr || !is_i8(*pool_in) || !has_shape(*pool_in, shape)) pool_in = nullptr, shape = {d.N, d.H, d.W, d.C};
  }
  size_t words = 0;
  if (!sto && f.prepared != nullptr && g.prepared != nullptr && f.prepared->data_ptr() == g.prepared->data_ptr())
    words = niti_conv2d_i8_backward_pair_sync_words(d.N, d.H, d.W, d.C, d.K, d.R, d.S, f.pad);
  const bool pair = words != 0;
  if (!pair) words = niti_conv2d_i8_backward_sync_words(d.N, d.H, d.W, d.C, d.K, d.R, d.S, f.pad);
  if (words == 0) return false;
  want_copy(g.prepared, d, 1, f.pad, 0, "conv layer");
  const size_t bytes = (pair ? niti_conv2d_i8_backward_pair_workspace : niti_conv2d_i8_backward_workspace)(d.N, d.H, d.W, d.C, d.K, d.R, d.S, f.pad);
  at::Tensor ws;
  if (bytes > 0) ws = scratch(bytes, act);
  uint32_t* sync = arena_take(static_cast<long>(words), act, nullptr);
  r->y = empty8(shape, act);
  if (g.want_grad) u->g8 = empty8(w.sizes(), w);
  u->shift = g.shift != nullptr ? *g.shift : scalar32(w);
  // the pair's flag speaks of both words, one of which is fresh where only the other tensor has a prediction
  const bool hint = g.shift != nullptr && (!pair || f.shift != nullptr);
  const int rc = (pair ? niti_conv2d_i8_backward_pair : niti_conv2d_i8_backward)(
      ptr<int8_t>(err), ptr<int8_t>(act), ptr<int8_t>(w), ptr<int8_t>(r->y), d.N, d.H, d.W, d.C, d.K, d.R, d.S, f.pad,
      g.flags | (hint ? NITI_CONV_SHIFT_HINT : 0u), f.r.bits, f.r.method, sto ? ptr<int32_t>(f.rand) : nullptr, ptr<int8_t>(f.mask),
      ptr<int8_t>(pool_in), f.ties, g.r.bits, g.r.method, f.r.div, f.r.bw, sync, words, g.want_grad ? ptr<int8_t>(u->g8) : nullptr, ptr<int8_t>(g.prepared),
      ptr<int32_t>(f.shift), ptr<int32_t>(u->shift), ptr<int32_t>(f.exp_a), ptr<int32_t>(f.exp_b), ptr<int32_t>(g.exp_b), ptr<int32_t>(r->e), ptr<int32_t>(e),
      bytes > 0 ? ws.data_ptr() : nullptr, bytes, stream_of(act));
  if (!check_fits(rc, pair ? "niti_conv2d_i8_backward_pair" : "niti_conv2d_i8_backward")) return false;
  r->unpooled = pool_in != nullptr;
  return true;
}

PyObject* put_all(std::initializer_list<PyObject*> items) {   // takes the references over
  PyObject* out = PyTuple_New(static_cast<Py_ssize_t>(items.size()));
  if (out == nullptr) throw python_error();
  Py_ssize_t k = 0;
  for (PyObject* o : items) PyTuple_SET_ITEM(out, k++, o);
  return out;
}
PyObject* boolean(bool b) {
  PyObject* o = b ? Py_True : Py_False;
  Py_INCREF(o);
  return o;
}

void take_weight_gradient(Args& a, WeightGradient* g) {
  g->want_grad = a.flag();
  g->want_dw = a.flag();
  g->shift = a.opt();
}

// layer_wgrad_update(fuse, act, err, w, stride, pad, f32, mu, method, div, bw, want_grad, want_dw, shift state, exp_a, exp_b,
//                    prepared, rand) -> (g8, dw, shift, exponent, one call?): the first layer's backward pass
PyObject* layer_wgrad_update(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    Args a(args, n, 18, "conv layer weight gradient");
    const bool fuse = a.flag();
    const at::Tensor& act = a.tensor();
    const at::Tensor& err = a.tensor();
    const at::Tensor& w = a.tensor();
    const int stride = a.i(), pad = a.i();
    WeightGradient g;
    g.flags = a.flag() ? NITI_EPI_F32_ROUNDTRIP : 0u;
    g.r = rounding_of(a);
    take_weight_gradient(a, &g);
    g.exp_a = a.exponent();
    g.exp_b = a.exponent();
    g.prepared = a.opt();
    g.rand = a.opt();
    at::Tensor e = scalar32(act);
    Update u;
    const bool one = weight_gradient(fuse, act, err, w, stride, pad, g, &u, e);
    return put_all({wrap(u.g8), wrap(u.dw), wrap(u.shift), wrap(e), boolean(one)});
  });
}

// layer_backward(fuse, err, act, w, stride, pad, f32, error bits, method, div, bw, error shift state, exp_err, exp_w, forward copy, mask,
//                pool_in, ties, error rand, mu, gradient method, want_grad, want_dw, gradient shift state, exp_act, prepared, gradient rand)
//   -> (error, exponent, unpooled?, g8, dw, shift, exponent, one call?)
// TiConv2d.backward: both gradients in one launch where that is the faster way, one after the other otherwise.
PyObject* layer_backward(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    Args a(args, n, 27, "conv layer backward");
    const bool fuse = a.flag();
    const at::Tensor& err = a.tensor();
    const at::Tensor& act = a.tensor();
    const at::Tensor& w = a.tensor();
    Fused f;
    f.dgrad = true;
    f.stride = a.i();
    f.pad = a.i();
    f.f32 = a.flag();
    f.r = rounding_of(a);
    f.shift = a.opt();
    f.hint = f.shift != nullptr;
    f.exp_a = a.exponent();
    f.exp_b = a.exponent();
    f.prepared = a.opt();
    f.mask = a.opt();
    Opt pool_in = a.opt();
    f.ties = a.i();
    f.rand = a.opt();
    WeightGradient g;
    g.flags = f.f32 ? NITI_EPI_F32_ROUNDTRIP : 0u;
    g.r = f.r;
    g.r.bits = a.i();
    g.r.method = a.i();
    take_weight_gradient(a, &g);
    g.exp_b = a.exponent();
    g.prepared = a.opt();
    g.rand = a.opt();
    DataGradient r;
    r.e = scalar32(err);
    at::Tensor e = scalar32(act);
    Update u;
    bool one = fuse && both_gradients(act, err, w, f, pool_in, g, &r, &u, e);
    if (!one) {
      data_gradient(fuse, err, w, f, pool_in, &r);
      g.exp_a = &r.e;
      one = weight_gradient(fuse && g.rand == nullptr, act, err, w, f.stride, f.pad, g, &u, e);
    }
    return put_all({wrap(r.y), wrap(r.e), boolean(r.unpooled), wrap(u.g8), wrap(u.dw), wrap(u.shift), wrap(e), boolean(one)});
  });
}

#define FAST(name) reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(name)), METH_FASTCALL, nullptr
}  // namespace

PyMethodDef kConvMethods[] = {{"conv_fprop", FAST(fprop)},
                              {"sp_conv", FAST(sp_conv)},
                              {"conv_dgrad", FAST(dgrad)},
                              {"conv_wgrad", FAST(wgrad)},
                              {"conv_fprop_requant", FAST(fprop_requant)},
                              {"conv_dgrad_requant", FAST(dgrad_requant)},
                              {"conv_layer_forward", FAST(layer_forward)},
                              {"conv_layer_backward", FAST(layer_backward)},
                              {"conv_wgrad_update", FAST(wgrad_update)},
                              {"conv_layer_wgrad_update", FAST(layer_wgrad_update)},
                              {nullptr, nullptr, 0, nullptr}};

}  // namespace niti_host
