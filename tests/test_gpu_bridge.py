"""GPU: gating and boundary fluxes around two-step passes, by groups of
connected pairs (k_bridge_groups) or, where a component is larger than a
block holds, by phases over all rows (k_bridge), against one-step passes.

Both sum the same fluxes in the same order, so FP64 fields agree to 1e-13
per voxel over these runs and FP32 ones to 1e-5 of each species' largest
deviation from rest; channel states are equal.  Rows: fewer than a group
takes, thousands of them (a SERCA sheet), and chains of pairs that share
voxels, of exactly the voxels a block holds and of two more.
"""
import sys

import numpy as np
import pytest

import csparks as cs
import dyad
from helpers import deviation_close, rest_field, species_close, with_serca

pytestmark = pytest.mark.gpu


def _chain(length):
    """A SERCA sheet whose first row is one chain: pairs (x, x) and
    (x + 1, x), so `length` voxels on either side hang together."""
    d = with_serca(dyad.small_dyad(n=(length + 6, 12, 14), seed=9))
    nz = d.geometry.voxels.shape[2]
    pairs = [(3 + x + k, 3, nz - 3, 3 + x, 3, nz - 2) for x in range(length) for k in (0, 1) if x + k < length]
    pairs += [(3, y, nz - 3, 3, y, nz - 2) for y in range(5, 9)]
    bnds = [b for b in d.geometry.boundaries if b.name != "serca"]
    bnds.append(cs.Boundary("serca", "density", np.array(pairs, dtype=np.uint16)))
    g = d.geometry
    geom = cs.Geometry(voxels=g.voxels, h=g.h, domain_names=list(g.domain_names),
                       domain_connections=g.domain_connections, boundaries=bnds)
    return dyad.Dyad(geom, d.model, d.open_index, f"chain of {length}")


CASES = {"few rows": lambda: dyad.small_dyad(n=(20, 18, 14), seed=3),
         "sheet": lambda: with_serca(dyad.small_dyad(n=(131, 43, 14), seed=3)),
         "chain that fits": lambda: _chain(256),
         "chain too long": lambda: _chain(257)}


@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("rng", ["philox", "mt"])
def test_bridges_match_one_step_passes(name, precision, rng):
    print(f"case: {name} {precision} {rng}", flush=True)
    sys.stdout.flush()
    d = CASES[name]()
    opts = cs.Options(seed=6, open={"ryr": [d.open_index]}, t_close={"ryr": 1.0}, precision=precision, rng=rng)
    a, b = (cs.Simulation(d.geometry, d.model, opts) for _ in range(2))
    a.set_launch_config(fuse=1)
    b.set_launch_config(fuse=0)
    for n in (1, 20, 41):
        a.step(n)
        b.step(n)
    for f in range(2):
        np.testing.assert_array_equal(a.channel_states(f), b.channel_states(f))
        np.testing.assert_array_equal(a.recruited(f), b.recruited(f))
    for s in range(a.ns):
        if precision == "f32":
            ok, rel, err, dev = deviation_close(a.species(s), b.species(s), rest_field(d, s), 1e-5)
        else:
            ok, err = species_close(a.species(s), b.species(s), 1e-13)
        assert ok, f"species {s}: {err:.3e}"
    a.close()
    b.close()
