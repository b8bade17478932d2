// Python module niti_amd._host: the tensor front end as native code (see host.h), and the entries that are not a layer's.
#include "host.h"

#include <ATen/ops/empty.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <hip/hip_runtime_api.h>

#include <map>
#include <tuple>
#include <vector>

namespace niti_host {
namespace {

PyObject* g_niti_error = nullptr;   // niti_amd._lib.NitiError

// ---- zeroed sync words -------------------------------------------------------------------------------------------
// The single-launch kernels want zeroed words.  An arena hands out slices of a chunk that is filled when its first slice
// since the reset is taken: one fill for the words of a whole step, contained in a graph that captures the step.  One
// arena per stream, so steps on different streams do not share words, and one per stream capture: its chunks come from
// the memory of the graph being captured.
constexpr long kChunkWords = 1L << 17;
constexpr size_t kMaxChunks = 8;    // a caller that never resets starts over behind this many
constexpr size_t kMaxArenas = 16;   // streams remembered; the least recently used one is given back
struct Arena {
  std::vector<at::Tensor> chunks;
  size_t chunk = 0;
  long pos = 0;
  std::vector<std::pair<size_t, long>> taken;   // slices since the reset
  at::Tensor scalars;                           // block that scalar32 cuts from, and what is left of it
  int scalars_left = 0;
  bool cleared = false;                         // the first chunk was cleared for the period that has just begun
  unsigned long long capture = 0, used = 0;
};
std::map<std::pair<int, void*>, Arena> g_arenas;
unsigned long long g_clock = 0;

unsigned long long capture_id(hipStream_t s) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  unsigned long long id = 0;
  if (hipStreamGetCaptureInfo(s, &status, &id) != hipSuccess || status == hipStreamCaptureStatusNone) return 0;
  return id + 1;
}

Arena& arena_of(int device, hipStream_t s) {
  const auto key = std::make_pair(device, static_cast<void*>(s));
  auto it = g_arenas.find(key);
  if (it == g_arenas.end()) {
    if (g_arenas.size() >= kMaxArenas) {
      auto old = g_arenas.begin();
      for (auto j = g_arenas.begin(); j != g_arenas.end(); ++j)
        if (j->second.used < old->second.used) old = j;
      g_arenas.erase(old);
    }
    it = g_arenas.emplace(key, Arena{}).first;
  }
  it->second.used = ++g_clock;
  return it->second;
}

void arena_restart(Arena& a) {
  a.chunk = 0;
  a.pos = 0;
  a.taken.clear();
}

// The arena of the tensor's device and current stream.  Where a capture has begun or ended since its last use it starts
// afresh: its memory has to be the graph's, and filled inside it.
Arena& arena_now(const at::Tensor& like) {
  hipStream_t s = static_cast<hipStream_t>(stream_of(like));
  Arena& a = arena_of(like.device().index(), s);
  const unsigned long long id = capture_id(s);
  if (id != a.capture) {
    a.chunks.clear();
    arena_restart(a);
    a.scalars = at::Tensor();
    a.scalars_left = 0;
    a.cleared = false;
    a.capture = id;
  }
  return a;
}

PyObject* arena_reset(PyObject*, PyObject* arg) {
  return guarded([&]() -> PyObject* {
    const long device = PyLong_AsLong(arg);
    if (device < 0) refuse("arena_reset: device index expected");
    arena_restart(arena_of(static_cast<int>(device), c10::hip::getCurrentHIPStream(static_cast<c10::DeviceIndex>(device)).stream()));
    Py_RETURN_NONE;
  });
}

PyObject* py_arena_take(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    Args a(args, n, 2, "arena_take");
    const long words = a.integer();
    const long device = a.integer();
    const at::Tensor like(at::detail::empty_cuda({0}, at::kInt, c10::Device(at::kCUDA, static_cast<c10::DeviceIndex>(device)), std::nullopt));
    at::Tensor view;
    arena_take(words, like, &view);
    return wrap(view);
  });
}

// flag words (word 1) of every slice handed out on the device since the resets, as a list of 1-element tensors
PyObject* arena_flags(PyObject*, PyObject* arg) {
  return guarded([&]() -> PyObject* {
    const long device = PyLong_AsLong(arg);
    PyObject* out = PyList_New(0);
    for (const auto& kv : g_arenas) {
      if (kv.first.first != device) continue;
      for (const auto& t : kv.second.taken) {
        PyObject* w = wrap(kv.second.chunks[t.first].narrow(0, t.second + 1, 1));
        PyList_Append(out, w);
        Py_DECREF(w);
      }
    }
    return out;
  });
}

// ---- scratch memory ----------------------------------------------------------------------------------------------
std::map<std::pair<int, void*>, std::pair<at::Tensor, unsigned long long>> g_scratch;

PyObject* py_scratch(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    Args a(args, n, 2, "scratch");
    const long bytes = a.integer();
    const long device = a.integer();
    const at::Tensor like(at::detail::empty_cuda({0}, at::kChar, c10::Device(at::kCUDA, static_cast<c10::DeviceIndex>(device)), std::nullopt));
    return wrap(scratch(static_cast<size_t>(bytes), like));
  });
}

// ---- products ----------------------------------------------------------------------------------------------------
at::Tensor gemm_out(const at::Tensor& a, const at::Tensor& b, bool ta, bool tb, uint32_t* absmax, Opt out, unsigned flags) {
  want_i8(a, "gemm");
  want_i8(b, "gemm");
  if (a.dim() != 2 || b.dim() != 2) refuse("gemm: matrices expected");
  const int64_t m = a.size(ta ? 1 : 0), k = a.size(ta ? 0 : 1), n = b.size(tb ? 0 : 1), k2 = b.size(tb ? 1 : 0);
  if (k != k2) refuse("gemm: inner extents differ (" + std::to_string(k) + " vs " + std::to_string(k2) + ")");
  if (out != nullptr) want_bytes(*out, 4 * m * n, "gemm", "an int32 result");
  at::Tensor c = out != nullptr ? *out : empty32({m, n}, a);
  const size_t bytes = niti_gemm_i8_workspace(ta, tb, static_cast<int>(m), static_cast<int>(n), static_cast<int>(k));
  at::Tensor ws;
  if (bytes > 0) ws = empty8({static_cast<int64_t>(bytes)}, a);
  check(niti_gemm_i8(ta, tb, ptr<int8_t>(a), ptr<int8_t>(b), ptr<int32_t>(c), static_cast<int>(m), static_cast<int>(n), static_cast<int>(k),
                     flags, absmax, bytes > 0 ? ws.data_ptr() : nullptr, bytes, stream_of(a)),
        "niti_gemm_i8");
  return c;
}

// gemm(a, b, trans_a, trans_b, absmax, out, flags) -> c
PyObject* py_gemm(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    Args g(args, n, 7, "gemm");
    const at::Tensor& a = g.tensor();
    const at::Tensor& b = g.tensor();
    const bool ta = g.flag(), tb = g.flag();
    Opt am = g.opt();
    Opt out = g.opt();
    return wrap(gemm_out(a, b, ta, tb, ptr<uint32_t>(am), out, static_cast<unsigned>(g.integer())));
  });
}

// The checks of the reference's extensions (CHECK_INPUT, .data<int8_t>()), in their words.
const at::Tensor& shim_input(PyObject* o, const char* name) {
  if (!THPVariable_Check(o)) refuse(std::string(name) + " must be a tensor");
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.is_cuda()) refuse(std::string(name) + " must be a CUDA tensor");
  if (!t.is_contiguous()) refuse(std::string(name) + " must be contiguous");
  return t;
}

// int8_mm(lhs [m,k], rhs [k,n]) -> int32 [m,n], the transposed view of an [n,m] buffer (int8mm_kernel.cu:8-34)
PyObject* int8_mm(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    if (n != 2) refuse("int8_mm: 2 arguments expected");
    const at::Tensor& lhs = shim_input(args[0], "lhs");
    const at::Tensor& rhs = shim_input(args[1], "rhs");
    if (lhs.scalar_type() != at::kChar || rhs.scalar_type() != at::kChar) refuse("expected scalar type Char");
    // [n,m] = rhs^T lhs^T: rhs is stored [k,n] ("a" transposed), lhs is stored [m,k] ("b" transposed)
    return wrap(gemm_out(rhs, lhs, true, true, nullptr, nullptr, 0u).t());
  });
}

// ---- range and requantisation ------------------------------------------------------------------------------------
// absmax_i32(x, absmax or None) -> absmax
PyObject* absmax_i32(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    Args a(args, n, 2, "absmax_i32");
    const at::Tensor& x = a.tensor();
    Opt given = a.opt();
    at::Tensor am;
    if (given != nullptr) {
      am = *given;
    } else {
      am = scalar32(x);
      am.zero_();
    }
    check(niti_absmax_i32(ptr<int32_t>(x), x.numel(), ptr<uint32_t>(am), stream_of(x)), "niti_absmax_i32");
    return wrap(am);
  });
}

// ---- pooling -----------------------------------------------------------------------------------------------------
int64_t pooled_side(int64_t v, int ks, int stride, int pad) {
  const int64_t t = v + 2 * pad - ks;   // rounded down like Python's //
  const int64_t q = stride > 0 ? (t >= 0 ? t / stride : -((-t + stride - 1) / stride)) + 1 : 0;
  return q > 0 ? q : 0;
}

// maxpool_fwd(x, kernel, stride, padding) -> y
PyObject* maxpool_fwd(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    Args a(args, n, 4, "maxpool_fwd");
    const at::Tensor& x = a.tensor();
    const int ks = a.i(), stride = a.i(), pad = a.i();
    want_i8(x, "maxpool_fwd");
    if (x.dim() != 4) refuse("maxpool_fwd: [N,H,W,C] tensor expected");
    const int64_t N = x.size(0), H = x.size(1), W = x.size(2), C = x.size(3);
    at::Tensor y = empty8({N, pooled_side(H, ks, stride, pad), pooled_side(W, ks, stride, pad), C}, x);
    check(niti_maxpool_i8_fwd(ptr<int8_t>(x), ptr<int8_t>(y), static_cast<int>(N), static_cast<int>(H), static_cast<int>(W),
                              static_cast<int>(C), ks, stride, pad, stream_of(x)),
          "niti_maxpool_i8_fwd");
    return wrap(y);
  });
}

// maxpool_bwd(y, dy, x, kernel, stride, padding, ties | flags) -> dx
PyObject* maxpool_bwd(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    Args a(args, n, 7, "maxpool_bwd");
    const at::Tensor& y = a.tensor();
    const at::Tensor& dy = a.tensor();
    const at::Tensor& x = a.tensor();
    const int ks = a.i(), stride = a.i(), pad = a.i(), ties = a.i();
    if (x.dim() != 4) refuse("maxpool_bwd: [N,H,W,C] tensor expected");
    const int64_t pooled = x.size(0) * pooled_side(x.size(1), ks, stride, pad) * pooled_side(x.size(2), ks, stride, pad) * x.size(3);
    want_bytes(y, pooled, "maxpool_bwd", "a pooled map");
    want_bytes(dy, pooled, "maxpool_bwd", "an error map");
    at::Tensor dx = empty(x.sizes(), x.scalar_type(), x);
    check(niti_maxpool_i8_bwd(ptr<int8_t>(y), ptr<int8_t>(dy), ptr<int8_t>(x), ptr<int8_t>(dx), static_cast<int>(x.size(0)),
                              static_cast<int>(x.size(1)), static_cast<int>(x.size(2)), static_cast<int>(x.size(3)), ks, stride, pad, ties,
                              stream_of(x)),
          "niti_maxpool_i8_bwd");
    return wrap(dx);
  });
}

// ---- input quantiser ---------------------------------------------------------------------------------------------
// quantize_input(x, bits, cpad, out, exp_out, target, target_out, step begins?) -> (y, exponent)
PyObject* quantize_input(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    Args a(args, n, 8, "quantize_input");
    const at::Tensor& x = a.tensor();
    const int bits = a.i();
    int64_t cpad = a.integer();
    Opt out = a.opt(), exp_given = a.opt(), target = a.opt(), target_out = a.opt();
    if (x.scalar_type() != at::kFloat || x.dim() != 4) refuse("quantize_input: contiguous float32 [N,C,H,W] tensor expected");
    const int64_t N = x.size(0), C = x.size(1), H = x.size(2), W = x.size(3);
    const int64_t c4 = (C + 3) / 4 * 4;
    if (c4 > cpad) cpad = c4;
    if (out != nullptr && (out->scalar_type() != at::kChar || !has_shape(*out, {N, H, W, cpad})))
      refuse("quantize_input: out must be a contiguous int8 [N,H,W," + std::to_string(cpad) + "] tensor");
    int64_t targets = 0;
    if (target != nullptr) {
      targets = target->numel();
      if (target->scalar_type() != at::kLong || target_out == nullptr || target_out->scalar_type() != at::kLong || target_out->numel() != targets)
        refuse("quantize_input: target and target_out must be int64 tensors of one size");
    }
    at::Tensor y = out != nullptr ? *out : empty8({N, H, W, cpad}, x);
    at::Tensor e = exp_given != nullptr ? *exp_given : scalar32(x);
    at::Tensor parts = scratch(256 * sizeof(int32_t), x);
    uint32_t* zero = nullptr;
    int zero_words = 0;
    Arena* const arena = a.flag() ? &arena_now(x) : nullptr;
    if (arena != nullptr) {   // a step begins: its first launch clears the sync words
      arena_restart(*arena);
      arena->cleared = false;
      if (arena->chunks.empty()) arena->chunks.push_back(empty32({kChunkWords}, x));
      zero = ptr<uint32_t>(arena->chunks[0]);
      zero_words = static_cast<int>(arena->chunks[0].numel());
      if (zero_words > kChunkWords) zero = nullptr, zero_words = 0;   // an unusually long one: left to its own fill
    }
    check(niti_quantize_batch_zero_f32_i8(ptr<float>(x), ptr<int8_t>(y), static_cast<int>(N), static_cast<int>(C), static_cast<int>(H),
                                     static_cast<int>(W), static_cast<int>(cpad), bits, ptr<uint32_t>(parts), ptr<int32_t>(e),
                                     ptr<int64_t>(target), ptr<int64_t>(target_out), static_cast<int>(targets), zero, zero_words, stream_of(x)),
          "niti_quantize_batch_f32_i8");
    if (arena != nullptr) arena->cleared = zero != nullptr;   // behind the check: a refused call has launched nothing
    return tuple_of({y, e});
  });
}

PyObject* set_error(PyObject*, PyObject* cls) {
  Py_XINCREF(cls);
  Py_XSETREF(g_niti_error, cls);
  Py_RETURN_NONE;
}

#define FAST(name) reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(name)), METH_FASTCALL, nullptr
PyMethodDef kMethods[] = {
    {"set_error", set_error, METH_O, nullptr},
    {"arena_reset", arena_reset, METH_O, nullptr},
    {"arena_take", FAST(py_arena_take)},
    {"arena_flags", arena_flags, METH_O, nullptr},
    {"scratch", FAST(py_scratch)},
    {"gemm", FAST(py_gemm)},
    {"int8_mm", FAST(int8_mm)},
    {"absmax_i32", FAST(absmax_i32)},
    {"maxpool_fwd", FAST(maxpool_fwd)},
    {"maxpool_bwd", FAST(maxpool_bwd)},
    {"quantize_input", FAST(quantize_input)},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_host", "Tensor front end of libniti_gfx950.", -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyObject* raise(const Refused& e) {
  PyErr_SetString(e.niti && g_niti_error != nullptr ? g_niti_error : PyExc_RuntimeError, e.what());
  return nullptr;
}

at::Tensor gemm(const at::Tensor& a, const at::Tensor& b, bool ta, bool tb, uint32_t* absmax) {
  return gemm_out(a, b, ta, tb, absmax, nullptr, 0u);
}

at::Tensor scalar32(const at::Tensor& like) {
  constexpr int kBlock = 128;
  Arena& a = arena_now(like);
  if (a.scalars_left == 0) {
    a.scalars = empty32({kBlock}, like);
    a.scalars_left = kBlock;
  }
  at::Tensor t = at::detail::make_tensor<c10::TensorImpl>(c10::Storage(a.scalars.storage()), a.scalars.key_set(), a.scalars.dtype());
  c10::TensorImpl* const impl = t.unsafeGetTensorImpl();
  impl->set_storage_offset(kBlock - a.scalars_left);
  impl->set_sizes_contiguous({1});
  if (--a.scalars_left == 0) a.scalars = at::Tensor();
  return t;
}

uint32_t* arena_take(long words, const at::Tensor& like, at::Tensor* view) {
  Arena& a = arena_now(like);
  hipStream_t s = static_cast<hipStream_t>(stream_of(like));
  if (a.chunks.empty()) a.chunks.push_back(empty32({words > kChunkWords ? words : kChunkWords}, like));
  while (a.pos + words > a.chunks[a.chunk].numel()) {
    a.chunk += 1;
    a.pos = 0;
    if (a.chunk == a.chunks.size()) {
      if (a.chunks.size() >= kMaxChunks && words <= kChunkWords && a.capture == 0) {
        // never reset: start over (the fill is ordered behind the launches that used the words; their flags are gone
        // from here but stay in the device-wide word)
        arena_restart(a);
        break;
      }
      a.chunks.push_back(empty32({words > kChunkWords ? words : kChunkWords}, like));
    }
  }
  at::Tensor& c = a.chunks[a.chunk];
  uint32_t* base = static_cast<uint32_t*>(c.data_ptr());
  if (a.pos == 0) {
    if (a.chunk != 0 || !a.cleared) check(niti_fill_u32(base, c.numel(), 0u, s), "niti_fill_u32");
    if (a.chunk == 0) a.cleared = false;
  }
  const long at = a.pos;
  a.pos += (words + 31) / 32 * 32;
  a.taken.emplace_back(a.chunk, at);
  if (view != nullptr) *view = c.narrow(0, at, words);
  return base + at;
}

// One grow-only buffer per stream for workspaces that live only inside a call: calls on one stream run in order, so they
// can all use the same memory, which keeps the partial sums of consecutive weight-gradient launches in one cache-resident
// region.  A captured call takes memory of its graph instead (the buffer may be replaced while the graph lives on).
at::Tensor scratch(size_t bytes, const at::Tensor& like) {
  hipStream_t s = static_cast<hipStream_t>(stream_of(like));
  if (capture_id(s) != 0) return empty8({static_cast<int64_t>(bytes > 16 ? bytes : 16)}, like);
  const auto key = std::make_pair(static_cast<int>(like.device().index()), static_cast<void*>(s));
  auto it = g_scratch.find(key);
  if (it == g_scratch.end()) {
    if (g_scratch.size() >= kMaxArenas) {
      auto old = g_scratch.begin();
      for (auto j = g_scratch.begin(); j != g_scratch.end(); ++j)
        if (j->second.second < old->second.second) old = j;
      g_scratch.erase(old);
    }
    it = g_scratch.emplace(key, std::make_pair(at::Tensor(), 0ULL)).first;
  }
  at::Tensor& buf = it->second.first;
  it->second.second = ++g_clock;
  if (!buf.defined() || buf.numel() < static_cast<int64_t>(bytes)) {
    buf = at::Tensor();   // given back before the larger one is asked for
    buf = empty8({static_cast<int64_t>(bytes > (1u << 20) ? bytes : (1u << 20))}, like);
  }
  return buf;
}

}  // namespace niti_host

PyMODINIT_FUNC PyInit__host() {
  PyObject* m = PyModule_Create(&niti_host::kModule);
  if (m == nullptr) return nullptr;
  if (PyModule_AddFunctions(m, niti_host::kConvMethods) != 0 || PyModule_AddFunctions(m, niti_host::kLinearMethods) != 0) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
