// Kernels of the sub-chunk DGDA prefill (dgda_sub.h) for d_k = 32.
#include "dgda_sub.h"

namespace maba {

int run_sub_k32(SubArgs& a, int dv, bool f32in, bool g16, bool gch, hipStream_t stream) {
  return dv == 32 ? run_sub_passes<false, 32, 32>(a, f32in, g16, gch, stream)
                  : run_sub_passes<false, 32, 64>(a, f32in, g16, gch, stream);
}

}  // namespace maba
