// int8 convolutions of any map, filter and channel count (multiples of 16 where stated), read as stored (conv_any.hip).
#pragma once
#include <string.h>

#include "common.h"

namespace niti {

// the forward convolution's extents
struct ConvShape {
  int N, H, W, C, K, R, S, stride, pad;
  int P() const { return (H + 2 * pad - R) / stride + 1; }
  int Q() const { return (W + 2 * pad - S) / stride + 1; }
};

enum ConvPass { kConvForward = 0, kConvDgrad = 1, kConvWgrad = 2 };

bool conv_any_shape(ConvPass pass, const ConvShape& s);   // extents and channel counts the kernels take (16-byte aligned pointers)
// forward: a = x, b = w; data gradient: a = error map, b = w (stride 1).  int32 sums, range folded into absmax.
int launch_conv_any(ConvPass pass, const ConvShape& s, const int8_t* a, const int8_t* b, int32_t* y, bool roundtrip, uint32_t* absmax, hipStream_t stream);
// the same rounded to int8 in the launch: sync words, 0 when no tile's grid is resident at once
size_t conv_any_requant_words(ConvPass pass, const ConvShape& s);
double conv_any_forward_us(const ConvShape& s, size_t* words);   // estimated time of the forward pass with rounding and its sync words, 0: does not run
double conv_any_dgrad_us(const ConvShape& s);   // estimated time of the data gradient with rounding, 0: does not run
int launch_conv_any_requant(ConvPass pass, const ConvShape& s, const int8_t* a, const int8_t* b, int8_t* y, bool roundtrip, uint32_t* sync,
                            const RequantSpec& rq, hipStream_t stream);
// weight gradient (stride 1)
size_t conv_any_wgrad_workspace(const ConvShape& s);
double conv_any_wgrad_us(const ConvShape& s);   // estimated time with update, 0: not a shape of these kernels
int launch_conv_any_wgrad(const ConvShape& s, const int8_t* act, const int8_t* err, int32_t* dw, bool roundtrip, uint32_t* absmax, void* workspace,
                          hipStream_t stream);
size_t conv_any_wgrad_update_words(const ConvShape& s);
int launch_conv_any_wgrad_update(const ConvShape& s, const int8_t* act, const int8_t* err, int8_t* w, int w_channels, bool roundtrip, uint32_t* sync,
                                 const RequantSpec& rq, int8_t* g8, int32_t* dw, int8_t* wprep, void* workspace, hipStream_t stream);

// Data gradient and weight gradient with update as one launch (conv_backward.hip; stride 1).  The gradient's exponent builds on
// the error's: grad.exp_a is not read.  words 0: not resident together.
double conv_backward_us(const ConvShape& s);   // estimated time
size_t conv_backward_words(const ConvShape& s);
size_t conv_backward_workspace(const ConvShape& s);
int launch_conv_backward(const ConvShape& s, const int8_t* err, const int8_t* act, int8_t* w, int8_t* dx, bool roundtrip, uint32_t* sync, const RequantSpec& rq,
                         const RequantSpec& grad, int8_t* g8, int8_t* wprep, void* workspace, hipStream_t stream);

// What a thread last worked out for a few layers, for answers that are asked for several times per call.  `extra`: whatever else the answer
// hangs on.
template <class T>
class KeptPerShape {
 public:
  template <class F>
  const T& get(const ConvShape& s, int extra, F make) {
    const int key[kKey] = {s.N, s.H, s.W, s.C, s.K, s.R, s.S, s.stride, s.pad, device_slot() + 1, extra};   // (never all zero)
    unsigned h = 0;
    for (int v : key) h = h * 31u + static_cast<unsigned>(v);
    Entry& e = kept_[(h ^ (h >> 8)) & 15u];
    if (memcmp(e.key, key, sizeof(key)) != 0) {
      e.value = make();
      memcpy(e.key, key, sizeof(key));
    }
    return e.value;
  }

 private:
  static constexpr int kKey = 11;
  struct Entry {
    int key[kKey];
    T value;
  };
  Entry kept_[16] = {};
};

// Both gradients of a 3x3 layer on H x H maps as the weight gradient's sums and the data gradient with the update beside it
// (conv3x3_k64_backward.hip); wprep is the filter copy that the data gradient reads.  words 0: not a shape of these kernels.
size_t conv_pair_words(int N, int H, int C, int K);
double conv_pair_us(int N, int H, int C, int K, double dgrad_us);   // estimated time, dgrad_us the data gradient's by itself
size_t conv_pair_workspace(int N, int H, int C, int K);
int launch_conv_pair(const int8_t* err, const int8_t* act, int8_t* w, int8_t* dx, int N, int H, int C, int K, bool roundtrip, uint32_t* sync,
                     const RequantSpec& rq, const RequantSpec& grad, int8_t* g8, int8_t* wprep, void* workspace, hipStream_t stream);

}  // namespace niti
