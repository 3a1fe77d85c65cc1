/* cs_pass2_f32.hip -- the FP32 two-step passes (k_pass2.h). */
#include "k_pass2.h"

bool cs_internal_pass2_f32(bool whole, uint32_t m1, uint32_t m2, const P2Args& a, hipStream_t stream)
{
  return whole ? launch_pass2<float, true>(m1, m2, a, stream) : launch_pass2<float, false>(m1, m2, a, stream);
}

namespace {

__global__ void __launch_bounds__(256)
k_id_words(const uint8_t* __restrict__ ids, const P2Geo* __restrict__ geos, uint32_t* __restrict__ words)
{
  const P2Geo g = geos[blockIdx.y];
  const uint64_t v = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (v >= (uint64_t)g.plane * g.nz) return;
  const uint8_t* id = ids + g.id_off;
  const uint32_t z = (uint32_t)(v / g.plane), c = (uint32_t)(v - (uint64_t)z * g.plane);
  const uint32_t y = c / (uint32_t)g.nx, x = c - y * (uint32_t)g.nx;
  const uint64_t at[6] = {x > 0 ? v - 1 : v,
                          x + 1 < (uint32_t)g.nx ? v + 1 : v,
                          y > 0 ? v - g.nx : v,
                          y + 1 < (uint32_t)g.ny ? v + g.nx : v,
                          z > 0 ? v - g.plane : v,
                          z + 1 < (uint32_t)g.nz ? v + g.plane : v};
  uint32_t w = id[v];
#pragma unroll
  for (int k = 0; k < 6; k++) w |= (uint32_t)(id[at[k]] & 7) << (P2_NB + 3 * k);
  words[g.id_off + v] = w;
}

}  // namespace

void cs_internal_id_words(const uint8_t* ids, const P2Geo* geos, uint32_t count, uint64_t most_voxels,
                          uint32_t* words, hipStream_t stream)
{
  /* at most 65535 domains to a launch */
  for (uint32_t i = 0; i < count; i += 65535)
    hipLaunchKernelGGL(k_id_words, dim3((unsigned)((most_voxels + 255) / 256), std::min(count - i, 65535u)), dim3(256),
                       0, stream, ids, geos + i, words);
}

bool cs_internal_pass2(size_t esize, bool whole, uint32_t m1, uint32_t m2, const P2Args& a, hipStream_t stream)
{
  return esize == 4 ? cs_internal_pass2_f32(whole, m1, m2, a, stream) : cs_internal_pass2_f64(whole, m1, m2, a, stream);
}
