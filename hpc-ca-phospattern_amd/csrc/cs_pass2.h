/*
 * cs_pass2.h -- the two-step pass over tiles of one or many domains:
 * records, tile planning (host) and the launch entry (cs_pass2_f32.hip,
 * cs_pass2_f64.hip hold the kernels, k_pass2.h the code).
 */
#ifndef CS_PASS2_H
#define CS_PASS2_H

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <vector>

/* A domain inside the field stack: element offset of its fields, byte
 * offset of its ids, first entry of its columns in the pair-voxel index
 * (plane + 1 entries), sizes. */
struct P2Geo {
  uint64_t u_off, id_off;
  uint32_t col_off, plane;
  int nx, ny, nz;
  uint32_t pad;
};

/* A voxel's word: its id byte (cs_device.h), then three bits each for the
 * domains of its neighbours at x-1, x+1, y-1, y+1, z-1, z+1 (its own domain
 * beyond the grid's faces). */
constexpr uint32_t P2_NB = 8;

/* A block's work: lanes cover the w x h columns from (x0, y0), a ring of
 * one column around the owned columns [ix0, ix1) x [iy0, iy1) wherever
 * those do not end at the grid's face; planes [z0, z1). */
struct P2Tile {
  uint32_t inst, x0, y0, w, h;
  uint32_t ix0, ix1, iy0, iy1;
  uint32_t z0, z1, pad;
};

/* One launch.  react: the step runs the buffer reactions (species-major).
 * The pair voxels of every domain, ordered by column and then z: vz[k] the
 * plane of pair voxel k, col_start[geo.col_off + column] its column's
 * first; fsum[k] the flux sum that step 1 adds to species 0 there (one entry
 * more than there are pair voxels), l1[k] receives species 0 after step 1.  any_fixed: some domain holds fixed
 * species. */
struct P2Args {
  const void* u;
  void* un;
  const uint32_t* words;   /* per voxel, at id_off + voxel */
  const void* params;
  const P2Geo* geos;
  const P2Tile* tiles;
  const uint32_t* col_start;
  const uint32_t* vz;
  const double* fsum;
  void* l1;
  uint32_t ntiles;
  int xcd;
  uint32_t react1, react2, any_fixed, pad;
};

/* Two block sizes: half a compute unit's lanes (two blocks share one, and
 * one's loads and stores run under the other's arithmetic), or all of them
 * for a tile twice as large (fewer bytes per owned column).  On the
 * 201x187x91 dyad, which the last-level cache holds, a pass takes 44 us with
 * the half blocks and 51 with the whole ones (FP32); on the 400x400x200 one,
 * 370 and 339 us.
 * Threads of a block, elements of a 16-byte chunk, and elements of one
 * species' staged plane (the tile with a halo of one cell, rows rounded up
 * to whole chunks), by field size. */
constexpr int p2_threads(size_t esize, bool whole) { return (esize == 4 ? 512 : 256) << (whole ? 1 : 0); }
constexpr int p2_chunk(size_t esize) { return (int)(16 / esize); }
constexpr int p2_stage(size_t esize, bool whole) { return (esize == 4 ? 680 : 340) << (whole ? 1 : 0); }
/* Whole blocks for a domain whose field stacks are beyond the last-level
 * cache (256 MB). */
inline bool p2_whole(uint64_t stack_bytes) { return 2 * stack_bytes > (256ull << 20); }
/* The field stacks end in this many bytes that a row's last chunk may read. */
constexpr size_t P2_PAD = 64;

/* Most planes of a block of a two-step pass: it spans four z-groups (every
 * species of a plane, `group` bytes) more than its planes, and `pad` bytes,
 * under 32-bit descriptor offsets.  0 when not even one plane fits. */
inline int p2_zlimit(uint64_t group, uint64_t nz, uint64_t pad)
{
  const uint64_t fit = ((1ull << 32) - 1 - pad) / group;
  return fit > 4 ? (int)std::min<uint64_t>(nz, fit - 4) : 0;
}

/* The words of `count` domains from their ids (blocks of 256 voxels of the
 * largest one, for each). */
void cs_internal_id_words(const uint8_t* ids, const P2Geo* geos, uint32_t count, uint64_t most_voxels,
                          uint32_t* words, hipStream_t stream);
/* Launch the pass compiled for the step masks m1, m2; false when there is
 * none. */
bool cs_internal_pass2(size_t esize, bool whole, uint32_t m1, uint32_t m2, const P2Args& a, hipStream_t stream);
bool cs_internal_pass2_f32(bool whole, uint32_t m1, uint32_t m2, const P2Args& a, hipStream_t stream);
bool cs_internal_pass2_f64(bool whole, uint32_t m1, uint32_t m2, const P2Args& a, hipStream_t stream);

/* Masks of the species that diffuse on a step: the reference's species
 * files (parameters/ *.h5: Ca, Fluo, CMDN-CSQN, ATP, TRPN) let Ca and ATP
 * diffuse on every step (0x9), the dye and CMDN on their own multiples of
 * dt (0x2, 0x4), TRPN never.  Each pair of two steps' masks is compiled
 * (P2_PAIRS(X): X(m1, m2) each). */
#define P2_FIRST(X, m2) X(0x9, m2) X(0xB, m2) X(0xD, m2) X(0xF, m2)
#define P2_PAIRS(X) P2_FIRST(X, 0x9) P2_FIRST(X, 0xB) P2_FIRST(X, 0xD) P2_FIRST(X, 0xF)

/* Substeps whose steps all have such masks. */
inline bool p2_substeps(const uint32_t* sub) { return sub[0] == 1 && sub[3] == 1 && sub[4] == 0; }

/* Columns of a plane split into kx x ky tiles. */
struct P2Split {
  uint32_t kx, ky;
};

/* Widest part of n cells in k parts, with the ring lanes it needs. */
inline uint32_t p2_part(uint32_t n, uint32_t k)
{
  uint32_t worst = 0;
  for (uint32_t i = 0; i < k; i++) {
    const uint32_t a = (uint32_t)((uint64_t)i * n / k), b = (uint32_t)((uint64_t)(i + 1) * n / k);
    worst = std::max(worst, b - a + (i > 0 ? 1u : 0u) + (i + 1 < k ? 1u : 0u));
  }
  return worst;
}

/* The split of the planes for blocks of the given size: with whole blocks
 * the one that moves the fewest 128-byte lines (a row of b bytes takes
 * b / 128 + 1 on average, read with its halo and written), with half blocks
 * the one with the fewest tiles; among equals the widest.  The time of a
 * pass over the 400x400x200 dyad follows the lines: widths of 31, 47, 60,
 * 69 and 135 columns (FP32, whole blocks) take 420, 395, 386, 363 and 339
 * us. */
inline P2Split p2_split(uint32_t nx, uint32_t ny, size_t esize, bool whole)
{
  const uint32_t threads = (uint32_t)p2_threads(esize, whole), stage = (uint32_t)p2_stage(esize, whole),
                 chunk = (uint32_t)p2_chunk(esize);
  auto lines = [esize](double n) { return n * (double)esize / 128.0 + 1.0; };
  P2Split best{0, 0};
  double least = 1e300;
  for (uint32_t kx = 1; kx <= nx; kx++) {
    const uint32_t w = p2_part(nx, kx);
    if (w > threads) continue;
    /* a staged row: the tile, two halo cells, and up to a chunk less one at
     * either end */
    const uint32_t row = (w + 2 + chunk - 1 + chunk - 1) / chunk * chunk, rows = stage / row;
    const uint32_t hcap = std::min(threads / w, rows > 2 ? rows - 2 : 0u);
    if (hcap >= 3 || hcap >= ny) {
      uint32_t ky = std::max(1u, (ny + hcap - 1) / hcap);
      while (p2_part(ny, ky) > hcap) ky++;
      const double ox = (double)nx / kx, oy = (double)ny / ky;   /* owned columns */
      const double cost = (double)kx * ky * (whole ? (oy + 4) * lines(ox + 4) + oy * lines(ox) : 1.0);
      if (cost < least) {
        least = cost;
        best = {kx, ky};
      }
    }
    if (w < 16) break;   /* narrower tiles only add ring lanes */
  }
  return best;
}

/* A tile's columns have a lane each and its staged rectangle a place (what
 * k_pass2 takes for granted). */
inline bool p2_fits(const P2Tile& t, uint32_t nx, uint32_t ny, size_t esize, bool whole)
{
  const uint32_t chunk = (uint32_t)p2_chunk(esize);
  const uint32_t sx = (t.x0 ? t.x0 - 1 : 0) / chunk * chunk, sy = t.y0 ? t.y0 - 1 : 0;
  const uint32_t pitch = (std::min(t.x0 + t.w + 1, nx) - sx + chunk - 1) / chunk * chunk;
  return t.w * t.h <= (uint32_t)p2_threads(esize, whole) &&
         pitch * (std::min(t.y0 + t.h + 1, ny) - sy) <= (uint32_t)p2_stage(esize, whole);
}

/* Tiles of one domain (planes in chunks whose sizes differ by at most one). */
inline void p2_tiles(uint32_t inst, uint32_t nx, uint32_t ny, uint32_t nz, const P2Split& sp, uint32_t zparts,
                     std::vector<P2Tile>& out)
{
  for (uint32_t q = 0; q < zparts; q++)
    for (uint32_t j = 0; j < sp.ky; j++)
      for (uint32_t i = 0; i < sp.kx; i++) {
        P2Tile t{};
        t.inst = inst;
        t.ix0 = (uint32_t)((uint64_t)i * nx / sp.kx);
        t.ix1 = (uint32_t)((uint64_t)(i + 1) * nx / sp.kx);
        t.iy0 = (uint32_t)((uint64_t)j * ny / sp.ky);
        t.iy1 = (uint32_t)((uint64_t)(j + 1) * ny / sp.ky);
        t.x0 = t.ix0 - (t.ix0 > 0 ? 1 : 0);
        t.y0 = t.iy0 - (t.iy0 > 0 ? 1 : 0);
        t.w = t.ix1 + (t.ix1 < nx ? 1 : 0) - t.x0;
        t.h = t.iy1 + (t.iy1 < ny ? 1 : 0) - t.y0;
        t.z0 = (uint32_t)((uint64_t)q * nz / zparts);
        t.z1 = (uint32_t)((uint64_t)(q + 1) * nz / zparts);
        out.push_back(t);
      }
}

/* Parts of the planes for `tiles` column tiles on `slots` places for a
 * block: the fewest rounds of blocks (whole ones while there are few; many
 * rounds overlap and only the last leaves places idle) times the planes of a
 * block with about four planes' time that a block takes beside them (it
 * computes two planes again, and fills its pipeline).  64x64x25 FP32: 11.2 us
 * with one plane to a block, 13.4 with two, 17.2 with four. */
inline uint32_t p2_zparts(uint64_t tiles, uint32_t nz, int slots, uint32_t zmax)
{
  uint32_t best = 1;
  double least = 1e300;
  for (uint32_t k = 1; k <= nz; k++) {
    const uint32_t zc = (nz + k - 1) / k;
    if (zc > zmax) continue;
    const double blocks = (double)(tiles * k) / slots;
    const double rounds = blocks >= 3 ? blocks + 0.5 : (double)((tiles * k + slots - 1) / slots);
    const double cost = rounds * (zc + 4);
    if (cost < least * 0.999) {
      least = cost;
      best = k;
    }
  }
  return best;
}

#endif /* CS_PASS2_H */
