/*
 * cs_bridge.hip -- k_bridge's phases (csparks.hip) with one block per group
 * of connected boundary pairs, in one launch.
 */
#include "cs_bridge.h"

#include <cfloat>
#include <cmath>

#include "cs_physics.h"

namespace {

/* Tail and head as in k_bridge, in the same order and with the same code
 * (gate_one, flux_j).  A group's voxels, channels, rows and entries are
 * complete, so blocks are independent however many rows a problem has; the
 * level-1 values, the state and the channel states go to LDS first and the
 * phases read nothing else.  Bound by latency: three dependent rounds of
 * loads (group, records, values) and the gating arithmetic (one power per
 * channel and gating step; the draws are formed while the loads run), where
 * k_bridge loads anew in each of its four phases, in one block or in a
 * launch for each phase.  Per pass, before and now: 131x97x53 with a SERCA
 * sheet 19.2 and 8.8 us, 84^3 with one 19.7 and 9.4 us, 64x64x25 with 45
 * channels 7.7 and 6.6 us. */
template <typename T>
__global__ void __launch_bounds__(BG_THREADS)
k_bridge_groups(BgArgs a)
{
  struct Shared {
    double l1[BG_VOX], u[BG_VOX], rest[BG_VOX];
    uint64_t elem[BG_VOX];
    uint32_t slot[BG_VOX];
    BgChan chan[BG_CHAN];
    uint8_t state[BG_CHAN];
    double draw[2][BG_CHAN];   /* uniforms of the tail's and the head's gating */
    BgRow row[BG_ROW];
    BgEnt ent[BG_ENT];
    FluxParams flux[MAXF];
    double dt, h;
  };
  __shared__ Shared S;
  const BgGroup g = a.groups[blockIdx.x];
  const DevParams<T>* __restrict__ P = (const DevParams<T>*)a.params;
  T* __restrict__ u = (T*)a.u;
  const T* __restrict__ l1 = (const T*)a.l1;
  const uint32_t tid = threadIdx.x;

  for (uint32_t k = tid; k < g.nvox; k += BG_THREADS) {
    const BgVox v = a.vox[g.vox + k];
    S.rest[k] = v.rest;
    S.elem[k] = v.elem;
    S.slot[k] = v.slot;
    S.u[k] = (double)u[v.elem];
    S.l1[k] = a.do_tail ? (double)l1[v.slot] : 0.0;
  }
  for (uint32_t k = tid; k < g.nchan; k += BG_THREADS) {
    const BgChan c = a.chan[g.chan + k];
    S.chan[k] = c;
    S.state[k] = a.states[c.state];
    /* the draws depend on no value: they are formed while the loads run */
    const FluxParams& F = P->flux[c.flux];
    auto draw = [&](const F2Step& st) {
      if (!F.stochastic || !st.gate) return 0.0;
      return a.uniforms ? a.uniforms[st.uni_base + F.uniform_off + c.ch]
                        : cs_gate_uniform(a.seed, a.instance, st.ti, F.group, c.ch);
    };
    if (a.do_tail) S.draw[0][k] = draw(a.tail);
    if (a.do_head) S.draw[1][k] = draw(a.head);
  }
  for (uint32_t k = tid; k < g.nrow; k += BG_THREADS) S.row[k] = a.row[g.row + k];
  for (uint32_t k = tid; k < g.nent; k += BG_THREADS) S.ent[k] = a.ent[g.ent + k];
  {
    const uint32_t words = (uint32_t)(sizeof(FluxParams) * MAXF / sizeof(uint64_t));
    const uint64_t* src = reinterpret_cast<const uint64_t*>(P->flux);
    uint64_t* dst = reinterpret_cast<uint64_t*>(S.flux);
    for (uint32_t k = tid; k < words; k += BG_THREADS) dst[k] = src[k];
  }
  const double dt = P->dt, h = P->h, dts = dt * a.D;
  __syncthreads();

  auto gate = [&](const F2Step& st, const double* ca, const double* draw) {
    const double t = (double)st.ti * dt;
    for (uint32_t k = tid; k < g.nchan; k += BG_THREADS) {
      const BgChan c = S.chan[k];
      const FluxParams& F = S.flux[c.flux];
      const double c0 = F.stochastic ? ca[c.vox] + S.rest[c.vox] : 0.0;
      const uint8_t sv = gate_one(F, S.state[k], c0, st.ti, t, dts, a.seed, a.instance, draw + k, c.ch);
      S.state[k] = sv;
      a.states[c.state] = sv;
      if (sv) a.recruited[c.state] = 1;
    }
    __syncthreads();
  };
  auto row_flux = [&](const BgRow& w, uint32_t fluxmask, const double* val, double& sum) -> bool {
    sum = 0.0;
    bool any = false;
    if (w.skip) return false;
    for (uint32_t e = w.ent; e < (uint32_t)w.ent + w.nent; e++) {
      const BgEnt x = S.ent[e];
      const uint32_t f = x.flux_sign & 0xFFu;
      if (!((fluxmask >> f) & 1u)) continue;
      if (x.chan != BG_NONE && !S.state[x.chan]) continue;
      const double J = flux_j(S.flux[f], val[x.from], val[x.to], S.rest[x.from], S.rest[x.to], dt, h);
      sum += (x.flux_sign >> 8) ? J : -J;
      any = true;
    }
    return any;
  };

  if (a.do_tail) {
    if (a.tail.gate) gate(a.tail, S.l1, S.draw[0]);
    if (a.tail.fluxmask)
      for (uint32_t k = tid; k < g.nrow; k += BG_THREADS) {
        const BgRow w = S.row[k];
        double sum;
        if (row_flux(w, a.tail.fluxmask, S.l1, sum)) {
          const T v = (T)(S.u[w.vox] + sum);
          u[S.elem[w.vox]] = v;
          S.u[w.vox] = (double)v;
        }
      }
    __syncthreads();
  }
  if (a.do_head) {
    if (a.head.gate) gate(a.head, S.u, S.draw[1]);
    for (uint32_t k = tid; k < g.nrow; k += BG_THREADS) {
      const BgRow w = S.row[k];
      double sum;
      const bool any = row_flux(w, a.head.fluxmask, S.u, sum);
      a.fsum[S.slot[w.vox]] = any ? sum : 0.0;
    }
  }
}

}  // namespace

void cs_internal_bridge_groups(size_t esize, const BgArgs& a, hipStream_t stream)
{
  if (!a.ngroups) return;
  if (esize == 8) hipLaunchKernelGGL(k_bridge_groups<double>, dim3(a.ngroups), dim3(BG_THREADS), 0, stream, a);
  else hipLaunchKernelGGL(k_bridge_groups<float>, dim3(a.ngroups), dim3(BG_THREADS), 0, stream, a);
}
