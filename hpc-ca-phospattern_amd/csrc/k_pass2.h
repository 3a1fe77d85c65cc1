/*
 * k_pass2.h -- two time steps of five species in one pass over HBM.
 *
 * A block owns a tile of plane columns and marches z.  Its lanes cover the
 * tile and a ring of one column (P2Tile): every lane computes step 1
 * (level 1) at plane z, the owning lanes then step 2 (level 2) at plane
 * z-1 from level-1 values, so the intermediate state never leaves the
 * chip.  Lanes run over the tile's columns row by row whatever its width,
 * so a narrow or ragged domain wastes none, and a tile as wide as its
 * domain needs no ring in x.
 *
 * Level 0 comes from HBM once, by 16-byte chunks of the tile's rows with a
 * halo of one cell, into three LDS planes (z, z+1, z+2), asked for a plane
 * ahead of the store; step 1 reads its column and its neighbours there.
 * Level-1 planes of the species that step 2 diffuses are double-buffered in
 * LDS, one barrier per plane.  At the grid's faces a lane's neighbour cell
 * is its own (no flux through the face), so no lane selects anything.  z
 * neighbours sit in register rings that rotate by renaming.
 *
 * What bounds it: the phases of a plane one after the other, since a
 * block's waves move in step through loads, LDS, arithmetic (38% of cycles)
 * and stores, and row segments that start off a line or are shared by two
 * tiles load the L1; hence chunks instead of a load per value and neighbour,
 * tiles wide in x, and two blocks to a compute unit for smaller domains
 * (p2_whole).  On a domain beyond the last-level cache memory is next:
 * 400x400x200 FP32 moves 1.56 GB a pass at 4.6 TB/s, where k_stencil, whose
 * waves run apart, moves its bytes at 5.6 TB/s on the same grid.  On small
 * domains, the latency of a block's few planes.  A pass over two steps,
 * before (k_step2 in FP32, two k_stencil in FP64) and now: 400x400x200 FP32
 * 455 and 329 us, FP64 1076 and 669 us; 201x187x91 FP32 78 and 39 us; 84^3
 * FP64 43 and 23 us; 64x64x25 FP64 21 and 14 us.
 *
 * A lane reads one word per voxel, its id and its six neighbours' domains
 * (k_id_words), three planes ahead.  Bytes of ids, with six more loads where
 * a wave meets an interface, held a whole block up at each such plane: 512
 * dyads at 6 nm, 25 planes each, took 683 us a pass with them, 631 with the
 * words and 582 with no interface at all.
 *
 * Per voxel and level the arithmetic is stencil_columns' and
 * react_species_major's.  A lane keeps the rate and coefficient tables of
 * its current domain in registers and reads them again only when the
 * domain changes along z (a few times per column), where reading them per
 * voxel from LDS cost about as many LDS cycles as the neighbours do.
 *
 * Boundary fluxes: voxels of boundary pairs carry bit 6 of their id.  Step
 * 1's flux sums, formed before the pass, are added at level 1, and the
 * level-1 value of species 0 is kept per pair voxel: step 2's gating and
 * fluxes need only those and are added after the pass.
 * A lane keeps the index of its column's next pair voxel and the sum there;
 * looking both up at each pair voxel was a chain of loads per plane that
 * held the block up: on the 84^3 G1 geometry, a tenth of whose voxels are
 * in SERCA pairs, a pass takes 28 us (FP64), with the look-up 89.
 */
#ifndef K_PASS2_H
#define K_PASS2_H

#include "cs_device.h"
#include "cs_pass2.h"

namespace {

constexpr int P2_NS = 5;

template <typename T>
struct P2Tables {
  T coef[P2_NS][MAXD * MAXD];
  T dinit[P2_NS][MAXD * MAXD];
  RateTab<T> rt[MAXD][P2_NS];
  T rc0[MAXD];
  uint32_t fixed[MAXD];

  __device__ void load(const DevParams<T>* __restrict__ P, int tid, int nthr)
  {
    for (int i = tid; i < P2_NS * MAXD * MAXD; i += nthr) {
      coef[i / (MAXD * MAXD)][i % (MAXD * MAXD)] = P->coef[i / (MAXD * MAXD)][i % (MAXD * MAXD)];
      dinit[i / (MAXD * MAXD)][i % (MAXD * MAXD)] = P->dinit[i / (MAXD * MAXD)][i % (MAXD * MAXD)];
    }
    for (int i = tid; i < MAXD * P2_NS; i += nthr) rt[i / P2_NS][i % P2_NS] = P->rt[i / P2_NS][i % P2_NS];
    for (int i = tid; i < MAXD; i += nthr) {
      rc0[i] = P->rc0[i];
      fixed[i] = P->fixed_mask[i];
    }
  }
};

/* The tables of one domain, per lane. */
template <typename T>
struct P2Rates {
  T ka[P2_NS], j0[P2_NS], kon[P2_NS], koff[P2_NS], diag[P2_NS], c0;
};

/* LDS cell of the two species that diffuse on every step (Ca, ATP). */
template <typename T>
struct alignas(2 * sizeof(T)) P2Cell {
  T a, b;
};

template <uint32_t M>
constexpr int p2_slow() { return ((M >> 1) & 1) + ((M >> 2) & 1); }

/* LDS planes of level 1 (two buffers, a cell per lane): Ca and ATP
 * together, the slow species that diffuse on step 2 one after the other. */
template <typename T, uint32_t M, int CELLS>
struct P2Planes {
  P2Cell<T> q[2][CELLS];
  T slow[2][p2_slow<M>() ? p2_slow<M>() : 1][p2_slow<M>() ? CELLS : 1];

  __device__ __forceinline__ void put(int buf, int cell, const T (&v)[P2_NS])
  {
    q[buf][cell] = P2Cell<T>{v[0], v[3]};
    int k = 0;
    if ((M >> 1) & 1) slow[buf][k++][cell] = v[1];
    if ((M >> 2) & 1) slow[buf][k++][cell] = v[2];
  }
  __device__ __forceinline__ void get(int buf, int cell, T (&v)[P2_NS]) const
  {
    const P2Cell<T> c = q[buf][cell];
    v[0] = c.a;
    v[3] = c.b;
    int k = 0;
    if ((M >> 1) & 1) v[1] = slow[buf][k++][cell];
    if ((M >> 2) & 1) v[2] = slow[buf][k++][cell];
  }
};

typedef uint32_t u32x4v __attribute__((ext_vector_type(4)));

template <typename T, bool WHOLE, uint32_t M1, uint32_t M2>
__global__ void __launch_bounds__(p2_threads(sizeof(T), WHOLE), sizeof(T) == 4 ? 4 : 2)
k_pass2(P2Args a)
{
  constexpr int NS = P2_NS, BT = p2_threads(sizeof(T), WHOLE), SP = p2_stage(sizeof(T), WHOLE), CH = p2_chunk(sizeof(T));
  /* chunks a lane stages per plane, at most: of Ca and ATP, of the others */
  constexpr int NQD = (2 * SP / CH + BT - 1) / BT, NQO = (3 * SP / CH + BT - 1) / BT, NQ = NQD + NQO;
  /* Ca's and ATP's planes first: with their neighbours' offsets they are
   * the ones read most, and lie within the reach of an LDS instruction's
   * immediate offset from one address */
  struct Shared {
    alignas(16) T d[3][2 * SP + CH];   /* the last chunk takes what no cell needs */
    alignas(16) T o[3][3 * SP + CH];
    P2Planes<T, M2, BT> l1;
    P2Tables<T> tab;
  };
  __shared__ Shared sh;
  auto& S = sh.tab;
  auto& L1 = sh.l1;

  const int bid = xcd_tile(blockIdx.x, (int)a.ntiles, a.xcd);
  if (bid >= (int)a.ntiles) return;   /* whole padding blocks only: no barrier is skipped */
  const int tid = threadIdx.x;
  const P2Tile t = a.tiles[bid];
  const P2Geo g = a.geos[t.inst];
  const DevParams<T>* __restrict__ P = (const DevParams<T>*)a.params;
  S.load(P, tid, BT);

  /* lanes past the tile repeat its last column and store nothing */
  const int w = (int)t.w, n = w * (int)t.h, ln = min(tid, n - 1);
  const int ty = ln / w, tx = ln - ty * w;
  const int x = (int)t.x0 + tx, y = (int)t.y0 + ty;
  const bool owner = tid < n && x >= (int)t.ix0 && x < (int)t.ix1 && y >= (int)t.iy0 && y < (int)t.iy1;
  const int nx = g.nx, ny = g.ny, nz = g.nz;
  const int z0 = (int)t.z0, z1 = (int)t.z1;
  const uint32_t ES = (uint32_t)sizeof(T);
  const uint32_t col = (uint32_t)y * (uint32_t)nx + (uint32_t)x;
  const uint32_t bc = col * ES;
  const uint32_t NOACCESS = 0xFFFFFFF0u;   /* beyond any descriptor: reads 0, stores nothing */
  const uint32_t bs = owner ? bc : NOACCESS;

  /* the staged rectangle: the tile's columns and those around it, rows of
   * whole chunks from column sx (a row's last chunk may run into the next
   * row, or into the stack's padding) */
  const int sx = max((int)t.x0 - 1, 0) / CH * CH, sy = max((int)t.y0 - 1, 0);
  const int nch = (min((int)t.x0 + w + 1, nx) - sx + CH - 1) / CH, rows = min((int)t.y0 + (int)t.h + 1, ny) - sy;
  const int pitch = nch * CH;
  const size_t plane = g.plane;
  const uint32_t pbytes = (uint32_t)plane * ES, gbytes = (uint32_t)NS * pbytes;
  uint32_t qoff[NQ];   /* byte offset of a chunk within a z-group        */
  int qcell[NQ];       /* and its first element within a staged plane    */
#pragma unroll
  for (int k = 0; k < NQ; k++) {
    const bool dk = k < NQD;
    const int c = tid + (dk ? k : k - NQD) * BT, s = c / (rows * nch), rc = c - s * (rows * nch), r = rc / nch,
              q = rc - r * nch, sp = dk ? 3 * s : s + (s < 2 ? 1 : 2);   /* Ca, ATP; dye, CMDN, TRPN */
    const bool has = s < (dk ? 2 : 3);
    qoff[k] = has ? (uint32_t)sp * pbytes + ((uint32_t)(sy + r) * (uint32_t)nx + (uint32_t)(sx + q * CH)) * ES : NOACCESS;
    qcell[k] = has ? s * SP + r * pitch + q * CH : (dk ? 2 : 3) * SP;
  }
  /* this lane's cell and its neighbours' in a staged plane and in a level-1
   * plane; at the grid's faces the neighbour is the cell itself (no flux),
   * at the tile's edge level 1 has none that is needed */
  const int c0 = (y - sy) * pitch + x - sx;
  const int cxm = x > 0 ? c0 - 1 : c0, cxp = x + 1 < nx ? c0 + 1 : c0;
  const int cym = y > 0 ? c0 - pitch : c0, cyp = y + 1 < ny ? c0 + pitch : c0;
  const int lxm = tx > 0 ? ln - 1 : ln, lxp = tx + 1 < w ? ln + 1 : ln;
  const int lym = ty > 0 ? ln - w : ln, lyp = ty + 1 < (int)t.h ? ln + w : ln;

  /* level 0 spans planes [z0-2, z1+2) of u (the host keeps a block's groups
   * below 2^32 bytes) */
  const int zb = max(z0 - 2, 0), ze = min(nz, z1 + 2);
  const T* u = (const T*)a.u + g.u_off;
  T* un = (T*)a.un + g.u_off;
  const Rsrc rin = make_rsrc(u + (size_t)zb * NS * plane, (uint32_t)(ze - zb) * gbytes + 16);
  const Rsrc rout = make_rsrc(un + (size_t)z0 * NS * plane, (uint32_t)(z1 - z0) * gbytes);
  const Rsrc rid = make_rsrc(a.words + g.id_off + (size_t)zb * plane, (uint32_t)(ze - zb) * (uint32_t)plane * 4u);
  auto gofs = [&](int zz) { return (uint32_t)(min(max(zz, zb), ze - 1) - zb) * gbytes; };
  auto word = [&](int zz) {
    return (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(
        rid, (int)(col * 4u), (int)((uint32_t)(min(max(zz, zb), ze - 1) - zb) * (uint32_t)plane * 4u), 0);
  };

  const bool dirichlet = P->dirichlet != 0;
  const bool gface = x == 0 || y == 0 || x + 1 == nx || y + 1 == ny;

  P2Rates<T> R;
  int dcur = -1;
  auto rates = [&](int d) {
    if (__builtin_expect(__ballot(d != dcur) == 0, 1)) return;
    dcur = d;
    R.c0 = S.rc0[d];
#pragma unroll
    for (int s = 0; s < NS; s++) {
      if (((M1 | M2) >> s) & 1u) R.diag[s] = S.coef[s][d * MAXD + d];
      if (s == 0) continue;
      const RateTab<T> r = S.rt[d][s];
      R.ka[s] = r.dka;
      R.j0[s] = r.dj0;
      R.kon[s] = r.dkon;
      R.koff[s] = r.dkoff;
    }
  };

  /* One level at plane zz of this lane's column: vm, vc, vp its input at
   * zz-1, zz, zz+1, xm .. yp the in-plane neighbours of the species in M;
   * the result goes to nw. */
  auto level = [&](auto mask, uint32_t react, const int zz, const uint32_t id, const T (&vm)[NS], const T (&vc)[NS],
                   const T (&vp)[NS], const T (&xm)[NS], const T (&xp)[NS], const T (&ym)[NS], const T (&yp)[NS],
                   T (&nw)[NS]) __attribute__((always_inline)) {
    constexpr uint32_t M = decltype(mask)::value;
    const int d = id & 7;
    const bool uni = (id & 0x80) != 0;
    rates(d);
#pragma unroll
    for (int s = 0; s < NS; s++) nw[s] = vc[s];
    if (__builtin_expect(__ballot(!uni) == 0, 1)) {
#pragma unroll
      for (int s = 0; s < NS; s++)
        if ((M >> s) & 1u) {
          const T c = vc[s];
          const T exm = xm[s] - c, exp_ = xp[s] - c;
          const T eym = ym[s] - c, eyp = yp[s] - c;
          const T ezm = vm[s] - c, ezp = vp[s] - c;
          nw[s] = fma(R.diag[s], (ezm + ezp) + (eym + eyp) + (exm + exp_), c);
        }
    } else {
      auto nb = [&](int k) { return (int)(id >> (P2_NB + 3 * k)) & 7; };
      const int dxm = nb(0), dxp = nb(1), dym = nb(2), dyp = nb(3), dzm = nb(4), dzp = nb(5);
#pragma unroll
      for (int s = 0; s < NS; s++)
        if ((M >> s) & 1u) {
          const T c = vc[s];
          const T exm = xm[s] - c, exp_ = xp[s] - c;
          const T eym = ym[s] - c, eyp = yp[s] - c;
          const T ezm = vm[s] - c, ezp = vp[s] - c;
          const T* C = S.coef[s] + d * MAXD;
          if (uni) {
            nw[s] = fma(C[d], (ezm + ezp) + (eym + eyp) + (exm + exp_), c);
          } else {
            /* deviations of different domains differ by their resting values */
            const T* Dn = S.dinit[s] + d * MAXD;
            nw[s] = c + ((C[dzm] * (ezm + Dn[dzm]) + C[dzp] * (ezp + Dn[dzp])) +
                         (C[dym] * (eym + Dn[dym]) + C[dyp] * (eyp + Dn[dyp])) +
                         (C[dxm] * (exm + Dn[dxm]) + C[dxp] * (exp_ + Dn[dxp])));
          }
        }
    }
    if (__builtin_expect(react, 1)) {
      const T f0 = R.c0 + vc[0];
      T f = nw[0];
#pragma unroll
      for (int s = 1; s < NS; s++) {
        const T inc = (R.ka[s] * vc[0] + R.j0[s]) - vc[s] * (R.kon[s] * f0 + R.koff[s]);
        nw[s] += inc;
        f -= inc;
      }
      nw[0] = f;
    }
    const bool held = dirichlet && (gface || zz == 0 || zz == nz - 1);
    nw[0] = held ? T(0) : nw[0];   /* the resting value */
    if (__builtin_expect(a.any_fixed, 0)) {
      const uint32_t fm = S.fixed[d];
#pragma unroll
      for (int s = 0; s < NS; s++)
        if ((fm >> s) & 1u) nw[s] = T(0);
    }
  };

  auto fetch = [&](int zz, u32x4v (&q)[NQ]) __attribute__((always_inline)) {
    const uint32_t so = gofs(zz);
#pragma unroll
    for (int k = 0; k < NQ; k++)
      q[k] = __builtin_bit_cast(u32x4v, __builtin_amdgcn_raw_buffer_load_b128(rin, (int)qoff[k], (int)so, 0));
  };
  auto put = [&](int buf, const u32x4v (&q)[NQ]) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < NQ; k++) {
      T* to = k < NQD ? &sh.d[buf][qcell[k]] : &sh.o[buf][qcell[k]];
      *reinterpret_cast<u32x4v*>(to) = q[k];
    }
  };

  auto staged = [&](int buf, int s) -> const T* {
    return s == 0 ? sh.d[buf] : s == 3 ? sh.d[buf] + SP : s < 3 ? sh.o[buf] + (s - 1) * SP : sh.o[buf] + 2 * SP;
  };

  /* Registers.  A0..A2: this column at planes z-1, z, z+1 of the species
   * step 1 diffuses; B0..B2: level 1 at z-2, z-1, z; Q: chunks of plane z+2
   * (from the middle of a plane's work on, of z+3) on their way to LDS;
   * I0..I5: words.  The names rotate with period six, so nothing is copied. */
  T A0[NS], A1[NS], A2[NS], B0[NS], B1[NS], B2[NS];
  u32x4v Q[NQ];
  uint32_t I0, I1, I2, I3, I4 = 0, I5 = 0;
  const int zs = z0 - 1, zt = z1 == nz ? nz : z1;
  /* this column's next pair voxel and step 1's flux sum there: the lane
   * meets the column's pair voxels in order, so one search at the start
   * finds them all, and each sum is on its way since the one before */
  uint32_t kpair = a.col_start[g.col_off + col], kend = a.col_start[g.col_off + col + 1];
  double fnext;
  {
    u32x4v q[NQ], r[NQ];
    fetch(zs, q);
    fetch(zs + 1, r);
    fetch(zs + 2, Q);
#pragma unroll
    for (int s = 0; s < NS; s++) {
      A0[s] = A1[s] = A2[s] = T(0);
      if ((M1 >> s) & 1u) A0[s] = bload<T>(rin, bc, gofs(zs - 1) + s * pbytes);
    }
    I0 = word(zs - 1);
    I1 = word(zs);
    I2 = word(zs + 1);
    I3 = word(zs + 2);
    put(0, q);
    put(1, r);
    while (kpair < kend) {   /* the first at plane zs or above */
      const uint32_t mid = (kpair + kend) >> 1;
      if ((int)a.vz[mid] < zs) kpair = mid + 1;
      else kend = mid;
    }
    fnext = a.fsum[kpair];
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
#pragma unroll
    for (int s = 0; s < NS; s++) {
      if ((M1 >> s) & 1u) A1[s] = staged(0, s)[c0];
      B0[s] = B1[s] = B2[s] = T(0);
    }
  }

  /* One plane: level 1 at z (am, ac, ap = planes z-1, z, z+1 of this
   * column), then level 2 at z-1 (wm, wc, wn = level 1 at z-2, z-1, z).
   * Planes z and z+1 are staged; between the levels the chunks of plane
   * z+2, on their way since the plane before, are staged and those of plane
   * z+3 asked for.  The first two planes have no level 2 to compute.  Every
   * plane issues the same memory operations in the same order, with no path
   * around any of them, so each wait covers only what it needs. */
  auto iter = [&](auto l2c, auto s0c, auto bufc, const int z, T (&am)[NS], T (&ac)[NS], T (&ap)[NS], T (&wm)[NS],
                  T (&wc)[NS], T (&wn)[NS], uint32_t& idm, uint32_t& ic, uint32_t& iqn) __attribute__((always_inline)) {
    constexpr bool l2 = decltype(l2c)::value;
    constexpr int s0 = decltype(s0c)::value, s1 = (s0 + 1) % 3, s2 = (s0 + 2) % 3, buf = decltype(bufc)::value;
    __syncthreads();
    const bool below = z < nz;
    {
      T xm[NS], xp[NS], ym[NS], yp[NS], vc[NS];
#pragma unroll
      for (int s = 0; s < NS; s++) {
        const T* p0 = staged(s0, s);
        if ((M1 >> s) & 1u) {
          xm[s] = p0[cxm];
          xp[s] = p0[cxp];
          ym[s] = p0[cym];
          yp[s] = p0[cyp];
          ap[s] = staged(s1, s)[c0];
          vc[s] = ac[s];
        } else {
          vc[s] = p0[c0];
        }
      }
      level(std::integral_constant<uint32_t, M1>{}, a.react1, z, ic, am, vc, ap, xm, xp, ym, yp, wn);
    }
    /* a pair voxel: step 1's flux sum, then its level-1 value */
    if (__builtin_expect(__ballot((ic & ID_PAIR) && below && z >= 0) != 0, 0)) {
      if ((ic & ID_PAIR) && below && z >= 0) {
        wn[0] = (T)((double)wn[0] + fnext);
        if (owner && z >= z0 && z < z1) ((T*)a.l1)[kpair] = wn[0];
        fnext = a.fsum[++kpair];
      }
    }
    L1.put(buf, ln, wn);
    put(s2, Q);
    fetch(z + 3, Q);
    iqn = word(z + 3);
    if constexpr (l2) {
      const int zo = z - 1;
      T xm2[NS], xp2[NS], ym2[NS], yp2[NS], nw[NS];
      L1.get(1 - buf, lxm, xm2);
      L1.get(1 - buf, lxp, xp2);
      L1.get(1 - buf, lym, ym2);
      L1.get(1 - buf, lyp, yp2);
      /* the grid's z faces: plane -1 is plane 0, plane nz is plane nz-1 */
      T vm2[NS], vp2[NS];
#pragma unroll
      for (int s = 0; s < NS; s++) {
        vm2[s] = zo > 0 ? wm[s] : wc[s];
        vp2[s] = below ? wn[s] : wc[s];
      }
      level(std::integral_constant<uint32_t, M2>{}, a.react2, zo, idm, vm2, wc, vp2, xm2, xp2, ym2, yp2, nw);
      const uint32_t so = (uint32_t)(zo - z0) * gbytes;
#pragma unroll
      for (int s = 0; s < NS; s++) bstore<T>(rout, bs, so + s * pbytes, nw[s], false);
    }
  };

  constexpr std::integral_constant<int, 0> c_0{};
  constexpr std::integral_constant<int, 1> c_1{};
  constexpr std::integral_constant<int, 2> c_2{};
  constexpr std::bool_constant<false> no{};
  constexpr std::bool_constant<true> yes{};
  iter(no, c_0, c_0, zs, A0, A1, A2, B0, B1, B2, I0, I1, I4);
  iter(no, c_1, c_1, zs + 1, A1, A2, A0, B1, B2, B0, I1, I2, I5);
  /* each plane leaves the loop when the next one is past zt, so no path
   * runs a later plane after skipping one */
  for (int z = zs + 2;; z += 6) {
    iter(yes, c_2, c_0, z, A2, A0, A1, B2, B0, B1, I2, I3, I0);
    if (z + 1 > zt) break;
    iter(yes, c_0, c_1, z + 1, A0, A1, A2, B0, B1, B2, I3, I4, I1);
    if (z + 2 > zt) break;
    iter(yes, c_1, c_0, z + 2, A1, A2, A0, B1, B2, B0, I4, I5, I2);
    if (z + 3 > zt) break;
    iter(yes, c_2, c_1, z + 3, A2, A0, A1, B2, B0, B1, I5, I0, I3);
    if (z + 4 > zt) break;
    iter(yes, c_0, c_0, z + 4, A0, A1, A2, B0, B1, B2, I0, I1, I4);
    if (z + 5 > zt) break;
    iter(yes, c_1, c_1, z + 5, A1, A2, A0, B1, B2, B0, I1, I2, I5);
    if (z + 6 > zt) break;
  }
}

template <typename T, bool WHOLE>
bool launch_pass2(uint32_t m1, uint32_t m2, const P2Args& a, hipStream_t stream)
{
  const dim3 grid(xcd_launch((int)a.ntiles, a.xcd)), block(p2_threads(sizeof(T), WHOLE));
#define P2_LAUNCH(x, y)                                                          \
  if (m1 == x && m2 == y) {                                                      \
    hipLaunchKernelGGL((k_pass2<T, WHOLE, x, y>), grid, block, 0, stream, a);    \
    return true;                                                                 \
  }
  P2_PAIRS(P2_LAUNCH)
#undef P2_LAUNCH
  return false;
}

}  // namespace

#endif /* K_PASS2_H */
