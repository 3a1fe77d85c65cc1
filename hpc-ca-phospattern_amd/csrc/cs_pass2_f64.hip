/* cs_pass2_f64.hip -- the FP64 two-step passes (k_pass2.h). */
#include "k_pass2.h"

bool cs_internal_pass2_f64(bool whole, uint32_t m1, uint32_t m2, const P2Args& a, hipStream_t stream)
{
  return whole ? launch_pass2<double, true>(m1, m2, a, stream) : launch_pass2<double, false>(m1, m2, a, stream);
}
