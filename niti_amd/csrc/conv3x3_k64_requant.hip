// Instances of the 64-channel-slice 3x3 convolution (conv3x3_k64.h): results rounded across the grid-wide range.
#include "conv3x3_k64.h"

namespace niti {

int launch_conv3x3_k64_requant(const HaloArgs& a, int H, int ktile, hipStream_t stream) {
  return a.src_cslices > 0 ? launch_k64_tiles<true, true, false>(a, H, ktile, stream) : launch_k64_tiles<true, false, false>(a, H, ktile, stream);
}

}  // namespace niti
