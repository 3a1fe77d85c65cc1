"""GPU: fields set and read back by slabs through the context's spare stack.

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


@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("cut", [(1, 31, 14), (2, 31, 14), (1, 1, 14)])
def test_one_species_in_few_columns(cut, precision):
    """The doubles of one x plane of a single species may be larger than the
    field they come from.  The steps after a transfer start from the fields
    that were set: from rest plus a constant, which diffusion leaves alone
    (nothing reacts or flows), to the rounding of 8 sums."""
    print(f"case: {cut} {precision}", flush=True)
    sys.stdout.flush()
    d = dyad.small_dyad(n=(33, 31, 14), seed=3)
    g, m = d.geometry, d.model
    model = dataclasses.replace(m, species_names=m.species_names[:1], init=np.asarray(m.init)[:, :1],
                                diffusive=[[s for s in k if s == 0] for k in m.diffusive],
                                sigma=[[v for v, s in zip(sg, k) if s == 0] for sg, k in zip(m.sigma, m.diffusive)],
                                buffers=[[] for _ in m.buffers], ryr=None, p_ryr=None)
    geom = dataclasses.replace(g, voxels=np.zeros_like(g.voxels[:cut[0], :cut[1], :cut[2]]), boundaries=[])
    sim = cs.Simulation(geom, model, cs.Options(seed=1, precision=precision))
    eps = np.finfo(np.float32 if precision == "f32" else np.float64).eps
    rest = np.asarray(model.init)[geom.voxels][..., 0]
    x = rest + np.random.default_rng(5).random(cut)
    sim.set_species(0, x)
    assert np.all(np.abs(sim.species(0) - x) <= 4 * eps * np.maximum(x, rest))
    sim.set_species(0, rest + 1.0)
    sim.step(8)
    assert np.all(np.abs(sim.species(0) - (rest + 1.0)) <= 16 * eps * (rest + 1.0))
    sim.close()
