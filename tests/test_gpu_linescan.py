"""GPU: linescans of single domains and ensembles against sums of the
downloaded fields in NumPy.

Every term is positive (concentrations times Gaussian weights), so any
order of a sum of n terms errs by at most n eps relative: below 1e-10 for
the 4e5 terms of the largest grid here.  Sizes: one, a remainder of, and
several blocks of outputs; row chunks with a remainder; planes wider than
a block and so narrow that a block's lanes cover several rows at once.
"""
import sys

import numpy as np
import pytest

import csparks as cs
import dyad

pytestmark = pytest.mark.gpu

RTOL = 1e-10
CONV = (28853.9, 28853.9, 115416.0)
OFF = (3, -2, 1)


def _want(u, ids, h, axis, nd):
    w = []
    for ax in range(3):
        off = (u.shape[ax] // 2 + OFF[ax]) * h
        w.append(cs.gauss(off - np.arange(u.shape[ax]) * h, CONV[ax]))
    x = np.where(ids < nd, u, 0.0) if nd else u
    rest = [k for k in range(3) if k != axis]
    x = np.moveaxis(x, axis, 0)
    proj = np.einsum("kab,a,b->k", x, w[rest[0]], w[rest[1]])
    k = np.arange(u.shape[axis]) * h
    return cs.gauss(k[:, None] - k[None, :], CONV[axis]) @ proj


@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("n", [(9, 9, 5), (64, 63, 16), (65, 130, 17), (300, 67, 12)])
def test_linescans_match_numpy(n, precision):
    print(f"case: {n} {precision}", flush=True)
    sys.stdout.flush()
    ds = [dyad.small_dyad(n=m, seed=3) for m in (n, (20, 18, 14))]
    opts = [cs.Options(seed=2, open={"ryr": [d.open_index]}, precision=precision) for d in ds]
    ens = cs.Ensemble([(d.geometry, d.model, o) for d, o in zip(ds, opts)])
    sim = cs.Simulation(ds[0].geometry, ds[0].model, opts[0])
    sim.step(30)
    ens.step(30)
    for axis in range(3):
        for species, nd in ((0, 0), (1, 2)):
            got = sim.linescan(species, axis, OFF, CONV, nd)
            want = _want(sim.species(species), ds[0].geometry.voxels, ds[0].geometry.h, axis, nd)
            np.testing.assert_allclose(got, want, rtol=RTOL)
            for i, line in enumerate(ens.linescans(species, axis, OFF, CONV, nd)):
                want = _want(ens.species(i, species), ds[i].geometry.voxels, ds[i].geometry.h, axis, nd)
                np.testing.assert_allclose(line, want, rtol=RTOL)
    sim.close()
    ens.close()
