"""GPU: fields set and read back through the context's slab buffer.

The stack holds deviations from rest, so a value comes back within one
rounding of its deviation and one of the sum: 4 eps of the larger of value
and rest.  The reductions per domain, which read the stack with the ids,
tell a wrong place from a right one.  Sizes: smaller than a 32 x 32 tile,
tiles with remainders either way, one plane, and two slabs.
"""
import dataclasses
import sys

import numpy as np
import pytest

import csparks as cs
import dyad

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,precision", [((9, 9, 5), "f64"), ((31, 33, 32), "f32"), ((65, 9, 70), "f64"),
                                         ((33, 64, 1), "f32"), ((210, 203, 200), "f32")])
def test_fields_come_back_where_they_were_put(n, precision):
    print(f"case: {n} {precision}", flush=True)
    sys.stdout.flush()
    if n[2] == 1:
        d = dyad.small_dyad(n=(n[0], n[1], 8), seed=3)
        geom = dataclasses.replace(d.geometry, voxels=np.ascontiguousarray(d.geometry.voxels[:, :, 3:4]), boundaries=[])
        model = dataclasses.replace(d.model, ryr=None, p_ryr=None)
    else:
        d = dyad.small_dyad(n=n, seed=3)
        geom, model = d.geometry, d.model
    sim = cs.Simulation(geom, model, cs.Options(seed=1, precision=precision))
    rest = np.asarray(model.init)[geom.voxels]
    rng = np.random.default_rng(5)
    eps = np.finfo(np.float32 if precision == "f32" else np.float64).eps
    for s in (0, sim.ns - 1):
        x = rest[..., s] + rng.random(n) * (1.0 + np.arange(n[0])[:, None, None])
        sim.set_species(s, x)
        got = sim.species(s)
        assert np.all(np.abs(got - x) <= 4 * eps * np.maximum(np.abs(x), rest[..., s]))
        low, high, _ = sim.stats()
        for dom in np.unique(geom.voxels):
            at = geom.voxels == dom
            np.testing.assert_allclose([low[dom, s], high[dom, s]], [x[at].min(), x[at].max()], rtol=8 * eps)
    sim.close()
