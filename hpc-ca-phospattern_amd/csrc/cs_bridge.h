/*
 * cs_bridge.h -- channel gating and boundary fluxes around two-step passes
 * of a single domain, by groups of connected boundary pairs: records,
 * grouping (host) and the launch entry (cs_bridge.hip holds the kernel).
 */
#ifndef CS_BRIDGE_H
#define CS_BRIDGE_H

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <numeric>
#include <vector>

#include "cs_device.h"

/* What one of the two steps of a fused pass does. */
struct F2Step {
  uint32_t dmask, react, fluxmask, gate;
  uint64_t ti, uni_base;
};

/* Pair voxels, channels, rows and entries of one group.  Voxels are named
 * by their index within the group, entries of a row and the channel of an
 * entry too. */
struct BgGroup {
  uint32_t vox, nvox, chan, nchan, row, nrow, ent, nent;
};
struct BgVox {
  uint64_t elem;          /* species 0 of the voxel in the stack             */
  double rest;            /* its resting value                               */
  uint32_t slot, pad;     /* level-1 slot                                    */
};
struct BgChan {
  uint32_t vox, flux, ch, state;   /* cleft voxel, flux, index within it, state slot */
};
struct BgRow {
  uint16_t vox, skip, ent, nent;
};
constexpr uint16_t BG_NONE = 0xFFFF;
struct BgEnt {
  uint16_t from, to, chan;         /* BG_NONE: no channel gates the pair     */
  uint16_t flux_sign;              /* flux | (row at the to voxel) << 8      */
};

constexpr int BG_THREADS = 256;
/* Most of each that a block holds in LDS, and the rows that groups are
 * filled up to: one to a lane. */
constexpr uint32_t BG_VOX = 512, BG_CHAN = 512, BG_ROW = 512, BG_ENT = 1024, BG_FILL = 256;

struct BgArgs {
  void* u;
  const void* l1;
  double* fsum;
  const void* params;
  const BgGroup* groups;
  const BgVox* vox;
  const BgChan* chan;
  const BgRow* row;
  const BgEnt* ent;
  uint8_t* states;
  uint8_t* recruited;
  const double* uniforms;
  F2Step tail, head;
  uint32_t ngroups, do_tail, do_head, D, seed, instance;
};

void cs_internal_bridge_groups(size_t esize, const BgArgs& a, hipStream_t stream);

struct BgTables {
  std::vector<BgGroup> groups;
  std::vector<BgVox> vox;
  std::vector<BgChan> chan;
  std::vector<BgRow> row;
  std::vector<BgEnt> ent;
};

namespace {

/* Groups of the records of k_bridge (slots 0 .. nslots-1): pair voxels that
 * share a pair belong together, and whole components fill a group up to
 * BG_FILL rows, so no phase of the bridge needs another block's results.
 * False when a component is too large for a block (then k_bridge runs). */
[[maybe_unused]] bool bg_build(size_t nslots, const std::vector<BChan>& chans, const std::vector<BRow>& rows,
                     const std::vector<BEnt>& ents, BgTables& out)
{
  std::vector<uint32_t> root(nslots);
  std::iota(root.begin(), root.end(), 0u);
  auto find = [&](uint32_t v) {
    while (root[v] != v) v = root[v] = root[root[v]];
    return v;
  };
  std::vector<BgVox> all(nslots);
  for (const BEnt& e : ents) {
    all[e.slot_from] = BgVox{e.elem_from, e.rest_from, e.slot_from, 0};
    all[e.slot_to] = BgVox{e.elem_to, e.rest_to, e.slot_to, 0};
    const uint32_t a = find(e.slot_from), b = find(e.slot_to);
    root[std::max(a, b)] = std::min(a, b);
  }
  /* components in the order of their first slot, and the voxels, channels
   * and rows of each (a root is its component's first slot) */
  uint32_t ncomp = 0;
  std::vector<uint32_t> comp(nslots);
  for (uint32_t v = 0; v < nslots; v++) comp[v] = find(v) == v ? ncomp++ : comp[find(v)];
  struct Lists {
    std::vector<uint32_t> start, item;
    Lists(size_t n, uint32_t ncomp) : start(ncomp + 1, 0), item(n) {}
    uint32_t size(uint32_t c) const { return start[c + 1] - start[c]; }
    const uint32_t* begin(uint32_t c) const { return item.data() + start[c]; }
  };
  auto lists = [&](size_t n, auto slot) {
    Lists l(n, ncomp);
    for (size_t k = 0; k < n; k++) l.start[comp[slot(k)] + 1]++;
    for (uint32_t c = 0; c < ncomp; c++) l.start[c + 1] += l.start[c];
    std::vector<uint32_t> next(l.start.begin(), l.start.end() - 1);
    for (size_t k = 0; k < n; k++) l.item[next[comp[slot(k)]]++] = (uint32_t)k;
    return l;
  };
  const Lists pvox = lists(nslots, [](size_t k) { return (uint32_t)k; });
  const Lists pchan = lists(chans.size(), [&](size_t k) { return chans[k].slot_to; });
  const Lists prow = lists(rows.size(), [&](size_t k) { return rows[k].slot; });
  out = BgTables{};
  std::vector<uint16_t> local(nslots, 0);
  BgGroup g{};
  for (uint32_t p = 0; p < ncomp; p++) {
    const uint32_t nvox = pvox.size(p), nchan = pchan.size(p), nrow = prow.size(p);
    uint32_t nent = 0;
    for (uint32_t k = 0; k < nrow; k++) nent += rows[prow.begin(p)[k]].end - rows[prow.begin(p)[k]].start;
    if (nvox > BG_VOX || nchan > BG_CHAN || nrow > BG_ROW || nent > BG_ENT) return false;
    if (g.nvox && (g.nrow + nrow > BG_FILL || g.nvox + nvox > BG_VOX || g.nchan + nchan > BG_CHAN ||
                   g.nent + nent > BG_ENT)) {
      out.groups.push_back(g);
      g = BgGroup{(uint32_t)out.vox.size(), 0, (uint32_t)out.chan.size(), 0, (uint32_t)out.row.size(), 0,
                  (uint32_t)out.ent.size(), 0};
    }
    for (uint32_t k = 0; k < nvox; k++) {
      const uint32_t v = pvox.begin(p)[k];
      local[v] = (uint16_t)g.nvox++;
      out.vox.push_back(all[v]);
    }
    const uint32_t c0 = g.nchan;
    for (uint32_t k = 0; k < nchan; k++) {
      const uint32_t c = pchan.begin(p)[k];
      out.chan.push_back(BgChan{local[chans[c].slot_to], chans[c].flux, chans[c].ch, chans[c].state});
      g.nchan++;
    }
    for (uint32_t q = 0; q < nrow; q++) {
      const BRow& w = rows[prow.begin(p)[q]];
      out.row.push_back(BgRow{local[w.slot], (uint16_t)w.skip, (uint16_t)g.nent, (uint16_t)(w.end - w.start)});
      g.nrow++;
      for (uint32_t e = w.start; e < w.end; e++) {
        const BEnt& x = ents[e];
        uint16_t chan = BG_NONE;
        for (uint32_t k = 0; x.state != NO_ROW && k < nchan; k++)
          if (chans[pchan.begin(p)[k]].state == x.state) { chan = (uint16_t)(c0 + k); break; }
        if (x.state != NO_ROW && chan == BG_NONE) return false;
        out.ent.push_back(BgEnt{local[x.slot_from], local[x.slot_to], chan, (uint16_t)x.flux_sign});
        g.nent++;
      }
    }
  }
  if (g.nvox) out.groups.push_back(g);
  return true;
}

}  // namespace

#endif /* CS_BRIDGE_H */
