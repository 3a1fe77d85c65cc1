"""GPU: the general two-step pass (k_step2), which models outside the
five-slot layout take and that layout with fuse_fixed = 0, against one-step
passes and the CPU oracle.

Forms: the layout with step masks read at run time ("run time"), and a
model whose TRPN no buffer binds, whose FP32 passes have the masks compiled
in ("unbound").  FP64 fields agree with the oracle to 1e-10 and with
one-step passes to 1e-13 per voxel, FP32 ones to DEV_F32 and 1e-5 of each
species' largest deviation from rest; channel states are equal.  Cases:
tiles with remainders (62 inner columns, 14 rows in FP32 and 6 in FP64), the
grid's last column on a tile's last lane, one and two planes, held faces with
a SERCA sheet, gating and reactions on substeps, odd calls.
"""
import dataclasses
import sys

import numpy as np
import pytest

import csparks as cs
import dyad
import sparks
from helpers import DEV_F32, deviation_close, rest_field, species_close, with_serca
from oracle_py import Oracle

pytestmark = pytest.mark.gpu


def _model(d, form):
    if form == "run time":
        return d
    m = d.model
    m = dataclasses.replace(m, buffers=[[b for b in bs if b.bound != 4] for bs in m.buffers])
    return dyad.Dyad(d.geometry, m, d.open_index, d.description)


def _slab(nz):
    d = dyad.small_dyad(n=(61, 16, 8), seed=3)
    g = d.geometry
    geom = dataclasses.replace(g, voxels=np.ascontiguousarray(g.voxels[:, :, 3:3 + nz]), boundaries=[])
    return dyad.Dyad(geom, dataclasses.replace(d.model, ryr=None, p_ryr=None), 0, f"slab of {nz} planes")


CASES = {
    "several tiles": (lambda: dyad.small_dyad(n=(130, 30, 12), seed=6), {}, 5, 8),
    "last lane": (lambda: dyad.small_dyad(n=(63, 17, 8), seed=3), {}, 3, 0),
    "one plane": (lambda: _slab(1), {}, 1, 0),
    "two planes": (lambda: _slab(2), {}, 5, 0),
    "SERCA, held faces": (lambda: with_serca(dyad.small_dyad(n=(65, 14, 10), seed=9)), dict(force_dirichlet=True), 3, 0),
    "substeps": (lambda: dyad.small_dyad(seed=5),
                 dict(t_close={"ryr": 0.002, "p_ryr": 0.001}, dt_update_react=3.5e-5 * 3, dt_update_stoch=3.5e-5 * 2), 8, 1),
    "stochastic": (lambda: dyad.fast_spark_dyad(), {}, 6, 1),
}


@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("form", ["run time", "unbound"])
@pytest.mark.parametrize("name", list(CASES))
def test_matches_oracle_and_one_step_passes(name, form, precision):
    print(f"case: {name} {form} {precision}", flush=True)
    sys.stdout.flush()
    make, options, zchunk, xcd = CASES[name]
    d = _model(make(), form)
    channels = bool(d.geometry.boundaries)
    kw = dict(seed=7, rng="mt" if name == "stochastic" else "philox")
    if channels:
        kw["open"] = {"ryr": [d.open_index]}
        if name != "stochastic":
            kw["t_close"] = {"ryr": 1.0}
    opts = cs.Options(**{**kw, **options}, precision=precision)
    two, one = (cs.Simulation(d.geometry, d.model, opts) for _ in range(2))
    two.set_launch_config(fuse=1, fuse_fixed=0 if form == "run time" else 1, fuse_zchunk=zchunk, fuse_xcd=xcd)
    one.set_launch_config(fuse=0)
    # FP32 gating may draw apart from the oracle's FP64: there against one-step passes alone
    orc = Oracle(d.geometry, d.model, dataclasses.replace(opts, precision="f64")) \
        if precision == "f64" or name != "stochastic" else None
    runs = [r for r in (two, one, orc) if r]
    for s in range(two.ns):   # 20% off rest, so every face carries gradients from the first step
        x = rest_field(d, s) * (1 + 0.2 * np.random.default_rng(s).random(d.geometry.voxels.shape))
        for r in runs:
            r.set_species(s, x)
    for k in (30, 31, 40):
        for r in runs:
            r.step(k)
        for f in range(sparks.discrete_count(two)):
            np.testing.assert_array_equal(two.channel_states(f), one.channel_states(f))
            if orc:
                np.testing.assert_array_equal(two.channel_states(f), orc.states(f))
    for s in range(two.ns):
        others = [(one.species(s), 1e-13, 1e-5)] + ([(orc.species(s), 1e-10, DEV_F32)] if orc else [])
        for other, rtol, dev in others:
            if precision == "f64":
                ok, err = species_close(two.species(s), other, rtol)
            else:
                ok, _, err, _ = deviation_close(two.species(s), other, rest_field(d, s), dev)
            assert ok, f"species {s}: {err:.3e}"
    if opts.rng == "philox":   # the library times its own draws only
        assert two.time_passes(2)[2:] == (1, 1)
    for r in runs:
        r.close()
