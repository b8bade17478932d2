// Fully connected entries of niti_amd._host (see host.h).
#include "host.h"

namespace niti_host {
namespace {

enum Pass { kForward = 0, kDgrad = 1, kWgrad = 2 };

struct Shape {
  int M, O, F;
};
Shape shape_of(const at::Tensor& rows, const at::Tensor& w, int inner, const char* who) {
  // rows: [M, F] (inner = 1) or [M, O] (inner = 0); w: [O, F]
  if (rows.dim() != 2 || w.dim() != 2 || rows.size(1) != w.size(inner) || rows.scalar_type() != at::kChar || w.scalar_type() != at::kChar)
    refuse(std::string(who) + ": int8 [M,features] tensor and int8 [O,F] weights expected");
  return {static_cast<int>(rows.size(0)), static_cast<int>(w.size(0)), static_cast<int>(w.size(1))};
}
void check_rand(Opt rand, int64_t n, const char* who) {
  if (rand != nullptr && (rand->scalar_type() != at::kInt || rand->numel() != n)) refuse(std::string(who) + ": rand must be int32 with one entry per element");
}

// Which kernels a pass runs on: those for few outputs (the classifier), those for any width, or the separate product and
// rounding.  The first two read the operands as stored and are one launch each.
enum Path { kFew, kWide, kSeparate };
Path path_of(Pass pass, bool fuse, const Shape& s, int method, Opt rand, size_t* words) {
  if (!fuse) return kSeparate;
  if (rand == nullptr && method != NITI_ROUND_STOCHASTIC && (*words = niti_fc_i8_sync_words(pass, s.M, s.O, s.F)) > 0) return kFew;
  if ((*words = niti_linear_i8_sync_words(pass, s.M, s.O, s.F)) > 0) return kWide;
  return kSeparate;
}

// linear_forward(fuse, act, w, bits, method, div, bw, exp_a, exp_b, rand) -> (out, exponent): act_calc(act @ w^T)
PyObject* forward(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    Args a(args, n, 10, "linear_forward");
    const bool fuse = a.flag();
    const at::Tensor& act = a.tensor();
    const at::Tensor& w = a.tensor();
    const int bits = a.i(), method = a.i(), div = a.i(), bw = a.i();
    Opt ea = a.exponent(), eb = a.exponent(), rand = a.opt();
    const Shape s = shape_of(act, w, 1, "linear_forward");
    check_rand(rand, static_cast<int64_t>(s.M) * s.O, "linear_forward");
    at::Tensor y, e = scalar32(act);
    size_t words = 0;
    void* st = stream_of(act);
    const Path p = path_of(kForward, fuse, s, method, rand, &words);
    if (p != kSeparate) {
      y = empty8({s.M, s.O}, act);
      uint32_t* sync = arena_take(static_cast<long>(words), act, nullptr);
      const int rc = p == kFew ? niti_fc_i8_fwd_requant(ptr<int8_t>(act), ptr<int8_t>(w), ptr<int8_t>(y), s.M, s.O, s.F, bits, method, div, bw, 0u, sync,
                                                        words, nullptr, ptr<int32_t>(ea), ptr<int32_t>(eb), ptr<int32_t>(e), st)
                               : niti_linear_i8_fwd_requant(ptr<int8_t>(act), ptr<int8_t>(w), ptr<int8_t>(y), s.M, s.O, s.F, bits, method, div, bw, 0u,
                                                            ptr<int32_t>(rand), sync, words, nullptr, ptr<int32_t>(ea), ptr<int32_t>(eb),
                                                            ptr<int32_t>(e), st);
      if (check_fits(rc, "niti_linear_i8_fwd_requant")) return tuple_of({y, e});
    }
    uint32_t* am = arena_take(1, act, nullptr);
    at::Tensor acc = gemm(act, w, false, true, am);   // act @ w^T, w read as stored
    y = empty8({s.M, s.O}, act);
    check(niti_requant_i32_i8(ptr<int32_t>(acc), ptr<int8_t>(y), acc.numel(), am, bits, method, div, bw, ptr<int32_t>(rand), 0u, nullptr,
                              ptr<int32_t>(ea), ptr<int32_t>(eb), ptr<int32_t>(e), st),
          "niti_requant_i32_i8");
    return tuple_of({y, e});
  });
}

struct Rounding {
  int bits, method, div, bw;
  Opt rand;
};

// err_calc(err @ w) -> y, its exponent in e
at::Tensor data_gradient(bool fuse, const at::Tensor& err, const at::Tensor& w, const Shape& s, const Rounding& r, Opt ea, Opt eb, const at::Tensor& e) {
  at::Tensor y = empty8({s.M, s.F}, err);
  size_t words = 0;
  void* st = stream_of(err);
  const Path p = path_of(kDgrad, fuse, s, r.method, r.rand, &words);
  if (p != kSeparate) {
    uint32_t* sync = arena_take(static_cast<long>(words), err, nullptr);
    const int rc = p == kFew ? niti_fc_i8_dgrad_requant(ptr<int8_t>(err), ptr<int8_t>(w), ptr<int8_t>(y), s.M, s.O, s.F, r.bits, r.method, r.div, r.bw, sync,
                                                        words, nullptr, ptr<int32_t>(ea), ptr<int32_t>(eb), ptr<int32_t>(e), st)
                             : niti_linear_i8_dgrad_requant(ptr<int8_t>(err), ptr<int8_t>(w), ptr<int8_t>(y), s.M, s.O, s.F, r.bits, r.method, r.div, r.bw,
                                                            ptr<int32_t>(r.rand), sync, words, nullptr, ptr<int32_t>(ea), ptr<int32_t>(eb),
                                                            ptr<int32_t>(e), st);
    if (check_fits(rc, "niti_linear_i8_dgrad_requant")) return y;
  }
  uint32_t* am = arena_take(1, err, nullptr);
  at::Tensor acc = gemm(err, w, false, false, am);
  check(niti_requant_i32_i8(ptr<int32_t>(acc), ptr<int8_t>(y), acc.numel(), am, r.bits, r.method, r.div, r.bw, ptr<int32_t>(r.rand), 0u, nullptr,
                            ptr<int32_t>(ea), ptr<int32_t>(eb), ptr<int32_t>(e), st),
        "niti_requant_i32_i8");
  return y;
}

// grad_calc(err^T @ act), w updated in place; returns the int32 gradient where there was one
at::Tensor weight_gradient(bool fuse, const at::Tensor& err, const at::Tensor& act, const at::Tensor& w, const Shape& s, const Rounding& r, int8_t* g8, Opt ea,
                           Opt eb, const at::Tensor& shift, const at::Tensor& e) {
  size_t words = 0;
  void* st = stream_of(err);
  const Path p = path_of(kWgrad, fuse, s, r.method, r.rand, &words);
  if (p != kSeparate) {
    uint32_t* sync = arena_take(static_cast<long>(words), err, nullptr);
    const int rc = p == kFew ? niti_fc_i8_wgrad_update(ptr<int8_t>(err), ptr<int8_t>(act), ptr<int8_t>(w), s.M, s.O, s.F, r.bits, r.method, r.div, r.bw, sync,
                                                       words, g8, ptr<int32_t>(shift), ptr<int32_t>(ea), ptr<int32_t>(eb), ptr<int32_t>(e), st)
                             : niti_linear_i8_wgrad_update(ptr<int8_t>(err), ptr<int8_t>(act), ptr<int8_t>(w), s.M, s.O, s.F, r.bits, r.method, r.div, r.bw,
                                                           ptr<int32_t>(r.rand), sync, words, g8, ptr<int32_t>(shift), ptr<int32_t>(ea),
                                                           ptr<int32_t>(eb), ptr<int32_t>(e), st);
    if (check_fits(rc, "niti_linear_i8_wgrad_update")) return at::Tensor();
  }
  uint32_t* am = arena_take(1, err, nullptr);
  at::Tensor acc = gemm(err, act, true, false, am);   // err^T @ act
  check(niti_grad_update_i8(ptr<int32_t>(acc), ptr<int8_t>(w), acc.numel(), am, r.bits, r.method, r.div, r.bw, ptr<int32_t>(r.rand), g8, ptr<int32_t>(shift),
                            ptr<int32_t>(ea), ptr<int32_t>(eb), ptr<int32_t>(e), st),
        "niti_grad_update_i8");
  return acc;
}

// linear_backward(fuse, err, act, w, error bits, error method, gradient bits, gradient method, div, bw, want_grad, keep_acc, exp_err,
//                 exp_w, exp_act, error rand, gradient rand) -> (error, error exponent, g8, int32 gradient, shift, exponent)
// TiLinear.backward: both gradients in one launch where they fit on the device together, one after the other otherwise.
PyObject* backward(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    Args a(args, n, 17, "linear_backward");
    const bool fuse = a.flag();
    const at::Tensor& err = a.tensor();
    const at::Tensor& act = a.tensor();
    const at::Tensor& w = a.tensor();
    Rounding re{}, rg{};
    re.bits = a.i();
    re.method = a.i();
    rg.bits = a.i();
    rg.method = a.i();
    re.div = rg.div = a.i();
    re.bw = rg.bw = a.i();
    const bool want_grad = a.flag(), keep = a.flag();
    Opt exp_err = a.exponent(), exp_w = a.exponent(), exp_act = a.exponent();
    re.rand = a.opt();
    rg.rand = a.opt();
    const Shape s = shape_of(err, w, 0, "linear_backward");
    if (act.dim() != 2 || act.size(0) != s.M || act.size(1) != s.F || act.scalar_type() != at::kChar) refuse("linear_backward: int8 act [M,F] expected");
    check_rand(re.rand, static_cast<int64_t>(s.M) * s.F, "linear_backward");
    check_rand(rg.rand, static_cast<int64_t>(s.O) * s.F, "linear_backward");
    at::Tensor g8, acc, y, ee = scalar32(err), shift = scalar32(w), ge = scalar32(w);
    if (want_grad) g8 = empty8({s.O, s.F}, w);
    int8_t* gp = want_grad ? ptr<int8_t>(g8) : nullptr;
    const size_t words = fuse && !keep ? niti_linear_i8_backward_sync_words(s.M, s.O, s.F) : 0;
    if (words > 0) {
      y = empty8({s.M, s.F}, err);
      uint32_t* sync = arena_take(static_cast<long>(words), err, nullptr);
      const int rc = niti_linear_i8_backward(ptr<int8_t>(err), ptr<int8_t>(act), ptr<int8_t>(w), ptr<int8_t>(y), s.M, s.O, s.F, re.bits, re.method, rg.bits,
                                             rg.method, re.div, re.bw, ptr<int32_t>(re.rand), ptr<int32_t>(rg.rand), sync, words, gp, nullptr,
                                             ptr<int32_t>(shift), ptr<int32_t>(exp_err), ptr<int32_t>(exp_w), ptr<int32_t>(exp_act), ptr<int32_t>(ee),
                                             ptr<int32_t>(ge), stream_of(err));
      if (check_fits(rc, "niti_linear_i8_backward")) return tuple_of({y, ee, g8, acc, shift, ge});
    }
    y = data_gradient(fuse, err, w, s, re, exp_err, exp_w, ee);
    acc = weight_gradient(fuse && !keep, err, act, w, s, rg, gp, &ee, exp_act, shift, ge);
    return tuple_of({y, ee, g8, acc, shift, ge});
  });
}

// head_forward(act, w, bits, method, div, bw, dropout (0 none, 1 mask given, 2 draw), mask, rng, exp_bias, target, loss_rand,
//              exp_a, exp_b) -> (logits, exponent, mask, loss gradient), or None where the kernel does not cover the call
PyObject* head_forward(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    Args a(args, n, 14, "head_forward");
    const at::Tensor& act = a.tensor();
    const at::Tensor& w = a.tensor();
    const int bits = a.i(), method = a.i(), div = a.i(), bw = a.i(), dropout = a.i();
    Opt mask_given = a.opt(), rng = a.opt();
    const int exp_bias = a.i();
    Opt target = a.opt(), loss_rand = a.opt(), ea = a.exponent(), eb = a.exponent();
    const Shape s = shape_of(act, w, 1, "head_forward");
    const size_t words = niti_head_i8_sync_words(0, s.M, s.O, s.F);
    if (words == 0) Py_RETURN_NONE;
    if (target != nullptr && (target->scalar_type() != at::kLong || target->numel() != s.M)) refuse("head_forward: int64 targets [M] expected");
    check_rand(loss_rand, static_cast<int64_t>(s.M) * s.O, "head_forward");
    if (mask_given != nullptr && (mask_given->scalar_type() != at::kChar || mask_given->numel() != s.F))
      refuse("head_forward: drop_mask must be a contiguous int8 tensor of F elements");
    if (rng != nullptr && (rng->scalar_type() != at::kInt || rng->numel() != 4)) refuse("head_forward: the generator state is an int32 tensor of 4 words");
    at::Tensor out = empty8({s.M, s.O}, act), e = scalar32(act), mask, loss;
    if (dropout != 0) mask = mask_given != nullptr ? *mask_given : empty8({s.F}, act);
    if (target != nullptr) loss = empty8({s.M, s.O}, act);
    uint32_t* sync = arena_take(static_cast<long>(words), act, nullptr);
    const int rc = niti_head_i8_forward(ptr<int8_t>(act), ptr<int8_t>(w), ptr<int8_t>(out), s.M, s.O, s.F, dropout,
                                        dropout != 0 ? ptr<int8_t>(mask) : nullptr, ptr<uint32_t>(rng), exp_bias, ptr<int64_t>(target),
                                        ptr<int32_t>(loss_rand), target != nullptr ? ptr<int8_t>(loss) : nullptr, bits, method, div, bw, 0u, sync, words,
                                        nullptr, ptr<int32_t>(ea), ptr<int32_t>(eb), ptr<int32_t>(e), stream_of(act));
    if (!check_fits(rc, "niti_head_i8_forward")) Py_RETURN_NONE;
    return tuple_of({out, e, mask, loss});
  });
}

// head_backward(err, act, w, err bits, err method, grad bits, grad method, div, bw, mask, want_grad, exp_err, exp_w, exp_act,
//               exp_act_bias, pool_in, pool_flags) -> (error, g8, grad shift, error exponent, gradient exponent, routed error),
// or None where the kernel does not cover the call.  pool_in: the input of the 2x2 max-pool whose flattened output act is.
PyObject* head_backward(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    Args a(args, n, 17, "head_backward");
    const at::Tensor& err = a.tensor();
    const at::Tensor& act = a.tensor();
    const at::Tensor& w = a.tensor();
    const int eb = a.i(), em = a.i(), gb = a.i(), gm = a.i(), div = a.i(), bw = a.i();
    Opt mask = a.opt();
    const bool want_grad = a.flag();
    Opt exp_err = a.exponent(), exp_w = a.exponent(), exp_act = a.exponent();
    const int bias = a.i();
    Opt pool_in = a.opt();
    const int pool_flags = a.i();
    const Shape s = shape_of(err, w, 0, "head_backward");
    if (act.dim() != 2 || act.size(0) != s.M || act.size(1) != s.F || act.scalar_type() != at::kChar) refuse("head_backward: int8 act [M,F] expected");
    if (mask != nullptr && (mask->scalar_type() != at::kChar || mask->numel() != s.F)) refuse("head_backward: drop_mask must be an int8 tensor of F elements");
    const size_t words = niti_head_i8_sync_words(1, s.M, s.O, s.F);
    if (words == 0) Py_RETURN_NONE;
    at::Tensor dx = empty8({s.M, s.F}, err), g8, routed, ee = scalar32(err), ge = scalar32(err), es = scalar32(err), gs = scalar32(err);
    if (want_grad) g8 = empty8({s.O, s.F}, w);
    int8_t* gp = want_grad ? ptr<int8_t>(g8) : nullptr;
    uint32_t* sync = arena_take(static_cast<long>(words), err, nullptr);
    int rc;
    if (pool_in != nullptr) {
      if (pool_in->dim() != 4 || pool_in->scalar_type() != at::kChar || pool_in->size(0) != s.M || pool_in->size(1) % 2 != 0 || pool_in->size(2) % 2 != 0 ||
          pool_in->size(1) / 2 * (pool_in->size(2) / 2) * pool_in->size(3) != s.F)
        refuse("head_backward: unpool wants the pool's contiguous int8 input [M,2P,2Q,C]");
      routed = empty8(pool_in->sizes(), err);
      rc = niti_head_i8_backward_unpool(ptr<int8_t>(err), ptr<int8_t>(act), ptr<int8_t>(mask), ptr<int8_t>(w), ptr<int8_t>(dx), s.M, s.O, s.F, eb, em, gb, gm,
                                        div, bw, sync, words, gp, ptr<int32_t>(es), ptr<int32_t>(gs), ptr<int32_t>(exp_err), ptr<int32_t>(exp_w),
                                        ptr<int32_t>(exp_act), bias, ptr<int32_t>(ee), ptr<int32_t>(ge), ptr<int8_t>(pool_in), ptr<int8_t>(routed),
                                        static_cast<int>(pool_in->size(1) / 2), static_cast<int>(pool_in->size(2) / 2), static_cast<int>(pool_in->size(3)),
                                        pool_flags, stream_of(err));
    } else {
      rc = niti_head_i8_backward(ptr<int8_t>(err), ptr<int8_t>(act), ptr<int8_t>(mask), ptr<int8_t>(w), ptr<int8_t>(dx), s.M, s.O, s.F, eb, em, gb, gm, div, bw,
                                 sync, words, gp, ptr<int32_t>(es), ptr<int32_t>(gs), ptr<int32_t>(exp_err), ptr<int32_t>(exp_w), ptr<int32_t>(exp_act), bias,
                                 ptr<int32_t>(ee), ptr<int32_t>(ge), stream_of(err));
    }
    if (!check_fits(rc, "niti_head_i8_backward")) Py_RETURN_NONE;
    return tuple_of({dx, g8, gs, ee, ge, routed});
  });
}

#define FAST(name) reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(name)), METH_FASTCALL, nullptr
}  // namespace

PyMethodDef kLinearMethods[] = {{"linear_forward", FAST(forward)},
                                {"linear_backward", FAST(backward)},
                                {"head_forward", FAST(head_forward)},
                                {"head_backward", FAST(head_backward)},
                                {nullptr, nullptr, 0, nullptr}};

}  // namespace niti_host
