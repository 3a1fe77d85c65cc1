/* cs_pass2_f32.hip -- the FP32 two-step passes (k_pass2.h). */
#include "k_pass2.h"

bool cs_internal_pass2_f32(bool whole, uint32_t m1, uint32_t m2, const P2Args& a, hipStream_t stream)
{
  return whole ? launch_pass2<float, true>(m1, m2, a, stream) : launch_pass2<float, false>(m1, m2, a, stream);
}

bool cs_internal_pass2(size_t esize, bool whole, uint32_t m1, uint32_t m2, const P2Args& a, hipStream_t stream)
{
  return esize == 4 ? cs_internal_pass2_f32(whole, m1, m2, a, stream) : cs_internal_pass2_f64(whole, m1, m2, a, stream);
}
