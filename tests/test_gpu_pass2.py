"""GPU: the two-step pass over column tiles (k_pass2) against one-step
passes and against the general two-step pass (k_step2).

All three apply the same per-voxel updates.  FP64: two steps differ by the
order of a few additions, so a run of 41 steps stays within 1e-13 of each
species' magnitude (species_close); FP32 within 1e-5 of each species'
largest deviation from rest, the bounds the fused passes are held to.
Channel states are equal.

Grids: fewer columns than one block has lanes, one tile, and several tiles
in x and y with parts that differ by a column, for both field sizes; z
chunks of one plane, of the whole grid, and with a remainder; odd step
counts.  Masks: every pair of step masks (the dye and CMDN-CSQN diffusing
with substeps of 1 or more).  A domain wider than its tile, and the
default form (no launch shape set) against the same shape asked for.
"""
import dataclasses
import sys

import numpy as np
import pytest

import csparks as cs
import dyad
import sparks
from helpers import deviation_close, rest_field, species_close, with_serca

pytestmark = pytest.mark.gpu

RTOL_F64 = 1e-13
DEV_F32 = 1e-5


def _say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def _substeps(d, dye, cmdn):
    """The dyad with the dye's and CMDN's diffusion constants set so that
    they diffuse every `dye` and `cmdn` steps."""
    sigma = [list(s) for s in d.model.sigma]
    for i, diff in enumerate(d.model.diffusive):
        for k, s in enumerate(diff):
            if s == 1:
                sigma[i][k] = 220000.0 / (dye + 0.25)
            if s == 2:
                sigma[i][k] = 220000.0 / (cmdn + 0.25)
    return dyad.Dyad(d.geometry, dataclasses.replace(d.model, sigma=sigma), d.open_index, d.description)


def _compare(d, opts, steps, shapes):
    """Runs with the given launch settings; the first is the one compared."""
    sims = [cs.Simulation(d.geometry, d.model, opts) for _ in shapes]
    for sim, kw in zip(sims, shapes):
        if kw is not None:
            sim.set_launch_config(**kw)
        for k in steps:
            sim.step(k)
    tile, others = sims[0], sims[1:]
    _, _, passes, fused = tile.time_passes(2)
    assert fused == passes == 1
    for other in others:
        other.time_passes(2)
        for f in range(sparks.discrete_count(tile)):
            np.testing.assert_array_equal(tile.channel_states(f), other.channel_states(f))
        for s in range(tile.ns):
            if opts.precision == "f32":
                ok, rel, err, dev = deviation_close(tile.species(s), other.species(s), rest_field(d, s), DEV_F32)
                assert ok, f"species {s}: {err:.3e} > {DEV_F32} x {dev:.3e}"
            else:
                ok, err = species_close(tile.species(s), other.species(s), RTOL_F64)
                assert ok, f"species {s}: max rel err {err:.3e}"
    for sim in sims:
        sim.close()


@pytest.mark.parametrize("n,precision,zchunk", [
    ((9, 9, 5), "f64", 1), ((20, 18, 14), "f64", 14), ((43, 24, 9), "f64", 4), ((131, 40, 7), "f64", 3),
    ((9, 9, 5), "f32", 5), ((33, 31, 8), "f32", 3), ((64, 63, 6), "f32", 1), ((150, 97, 7), "f32", 4)])
def test_tiles_match_one_step_and_general_pass(n, precision, zchunk):
    d = dyad.small_dyad(n=n, seed=4)
    opts = cs.Options(seed=7, open={"ryr": [d.open_index, 2]}, t_close={"ryr": 1.0}, precision=precision)
    _say(f"case: {n} {precision} zchunk={zchunk}")
    fuse = dict(fuse=1, fuse_zchunk=zchunk)
    _compare(d, opts, [20, 19], [dict(fuse, fuse_xcd=4), dict(fuse=0), dict(fuse, fuse_fixed=0)])


@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("dye,cmdn", [(1, 1), (1, 3), (2, 1), (2, 3), (5, 8)])
def test_step_masks(dye, cmdn, precision):
    d = _substeps(dyad.small_dyad(n=(40, 23, 9), seed=5), dye, cmdn)
    opts = cs.Options(seed=3, open={"ryr": [d.open_index]}, precision=precision)
    setup = cs.Setup(d.geometry, d.model, opts)
    assert list(setup.problem.substeps)[:5] == [1, dye, cmdn, 1, 0]
    _say(f"case: substeps {dye}, {cmdn} {precision}")
    _compare(d, opts, [21, 20], [dict(fuse=1, fuse_zchunk=4), dict(fuse=0)])


@pytest.mark.parametrize("precision", ["f64", "f32"])
def test_options_in_the_default_form(precision):
    """SERCA, held faces, fixed domain species and reactions on every fifth
    step only; no launch shape set, against one-step passes."""
    d = with_serca(dyad.small_dyad(n=(65, 34, 12), h=12.0, seed=9))
    names = d.model.domain_names
    model = dataclasses.replace(d.model, fixed=[(names.index("cleft"), 1), (names.index("jsr"), 2)])
    d = dyad.Dyad(d.geometry, model, d.open_index, d.description)
    opts = cs.Options(h=12.0, seed=2, open={"ryr": [d.open_index]}, force_dirichlet=True, dt=1e-4,
                      dt_update_react=5e-4, precision=precision)
    assert cs.Setup(d.geometry, d.model, opts).problem.reaction_substep == 5
    _say(f"case: options {precision}")
    _compare(d, opts, [33, 20], [None, dict(fuse=0)])


@pytest.mark.parametrize("precision", ["f64", "f32"])
def test_blocks_of_the_whole_compute_unit(precision):
    """A field stack beyond the last-level cache takes blocks of twice the
    lanes: tiles and faces of a wide, thin domain."""
    n = (1203, 403, 15) if precision == "f64" else (1203, 803, 15)
    assert 2 * 5 * np.prod(n) * (8 if precision == "f64" else 4) > 256 << 20
    d = dyad.small_dyad(n=n, seed=4)
    opts = cs.Options(seed=7, open={"ryr": [d.open_index, 2]}, precision=precision)
    _say(f"case: {n} {precision}")
    _compare(d, opts, [10, 11], [dict(fuse=1, fuse_zchunk=4), dict(fuse=0)])
