"""GPU: an ensemble's two-step passes (k_pass2 over every realisation, with
k_batch_bridge2) against its one-step passes.

Steps run in pairs within a call and a single last step runs one by one,
so a run of single-step calls is the one-step path.  Both apply the same
per-voxel updates: FP64 fields agree to 1e-12 per voxel (species_close) and
FP32 fields to 1e-5 of each species' largest deviation from rest over these
runs, with equal channel states, latest open steps and recruitment.

Covered: realisations of different sizes with one and several tiles, step
counts of both parities, Philox and Mersenne-Twister draws, replayed
graphs whose period ends in the other buffer, realisations retired after
an odd number of passes, and both closure networks (their inputs at the
first step of a pair come from the voxels that the pass keeps).
"""
import dataclasses
import os
import sys

import numpy as np
import pytest

import closure
import csparks as cs
import dyad
from helpers import deviation_close, rest_field, species_close

pytestmark = pytest.mark.gpu

PARAMS = os.path.join(os.path.dirname(cs.__file__), "closure_params.npz")
RTOL_F64 = 1e-12
DEV_F32 = 1e-5
SHAPES = [(20, 18, 14), (9, 9, 12), (131, 40, 13), (43, 24, 12), (64, 63, 12)]


def _say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def _members(edit=lambda m: m):
    out = []
    for k, n in enumerate(SHAPES):
        d = dyad.small_dyad(n=n, seed=31 + k, num_ryr=9, num_pryr=3)
        kin = dict(Kd_open=5.0, k_max_open=200.0, k_min_close=50.0, k_max_close=50.0)
        m = dataclasses.replace(d.model, ryr=dataclasses.replace(d.model.ryr, **kin),
                                p_ryr=dataclasses.replace(d.model.p_ryr, **kin))
        out.append(dyad.Dyad(d.geometry, edit(m), d.open_index, d.description))
    return out


def _ensemble(ds, **kw):
    return cs.Ensemble([(d.geometry, d.model, cs.Options(seed=100 + k, open={"ryr": [d.open_index]}, **kw))
                        for k, d in enumerate(ds)], instances=list(range(len(ds))))


def _singly(ens, n):
    for _ in range(n):
        ens.step(1)


def _same(a, b, ds, precision="f64"):
    for x, y in zip(a.summary(), b.summary()):
        np.testing.assert_array_equal(x, y)
    np.testing.assert_array_equal(a.channel_open(), b.channel_open())
    for i, d in enumerate(ds):
        for s in range(a.ns):
            if precision == "f32":
                ok, rel, err, dev = deviation_close(a.species(i, s), b.species(i, s), rest_field(d, s), DEV_F32)
                assert ok, f"member {i} species {s}: {err:.3e} > {DEV_F32} x {dev:.3e}"
            else:
                ok, err = species_close(a.species(i, s), b.species(i, s), RTOL_F64)
                assert ok, f"member {i} species {s}: max rel err {err:.3e}"


@pytest.mark.parametrize("precision,rng", [("f64", "philox"), ("f32", "philox"), ("f64", "mt")])
def test_pairs_match_single_steps(precision, rng):
    ds = _members()
    a, b = (_ensemble(ds, precision=precision, rng=rng) for _ in range(2))
    _say(f"case: {precision} {rng}")
    for n in (2, 41, 30):
        a.step(n)
        _singly(b, n)
        _same(a, b, ds, precision)
    a.close()
    b.close()


def test_graph_period_that_ends_in_the_other_buffer():
    """Every species diffusing on every step gives a period of two steps,
    one pass."""
    def every_step(m):
        sigma = [[220000.0 / 1.25 if s in (1, 2) else v for v, s in zip(sg, df)] for sg, df in zip(m.sigma, m.diffusive)]
        return dataclasses.replace(m, sigma=sigma)
    ds = _members(every_step)
    a, b, c = (_ensemble(ds) for _ in range(3))
    assert a.period == 2
    a.set_graph(True)
    for n in (2, 6, 5, 2, 9):
        a.step(n)
        b.step(n)
        _singly(c, n)
        a.species(0, 0)   # eager work and a synchronisation between the replays
        for i in range(a.count):
            for s in range(a.ns):
                np.testing.assert_array_equal(a.species(i, s), b.species(i, s))
        _same(a, c, ds)
    for e in (a, b, c):
        e.close()


def test_retired_realisations_after_an_odd_number_of_passes():
    ds = _members()
    a, b = _ensemble(ds), _ensemble(ds)
    for e in (a, b):
        e.step(10)
    on = np.array([True, False, True, False, True])
    a.set_active(on)
    frozen = {i: [a.species(i, s) for s in range(a.ns)] for i in (1, 3)}
    frozen[3][0] = frozen[3][0] + 1.0
    a.set_species(3, 0, frozen[3][0])
    for n in (2, 3, 6, 1):
        a.step(n)
        b.step(n)
        for i in range(a.count):
            for s in range(a.ns):
                if on[i]:
                    np.testing.assert_array_equal(a.species(i, s), b.species(i, s))
                else:
                    np.testing.assert_allclose(a.species(i, s), frozen[i][s], rtol=1e-14)
    a.close()
    b.close()


@pytest.mark.parametrize("flux", [False, True], ids=["gating", "gating and flux"])
def test_closure_in_pairs_matches_single_steps(flux):
    ds = [dyad.ensemble_dyad(s, h=12.0, edge_nm=(192.0, 384.0), ryr=(9, 30)) for s in range(5)]
    net, _, _ = closure.load(PARAMS)
    fnet, _ = closure.load_flux(PARAMS)
    ens = []
    for _ in range(2):
        e = cs.Ensemble([(d.geometry, d.model, cs.Options(h=12.0, seed=20 + k, open={"ryr": [d.open_index]}))
                         for k, d in enumerate(ds)], instances=list(range(len(ds))))
        e.set_gating(cs.Ensemble.GATE_CLOSURE, net)
        if flux:
            e.set_flux_closure(fnet)
        ens.append(e)
    a, b = ens
    _say(f"case: closure flux={flux}")
    for n in (2, 21, 30):
        a.step(n)
        _singly(b, n)
        _same(a, b, ds)
        np.testing.assert_allclose(a.closure_predictions(), b.closure_predictions(), rtol=1e-9)
        if flux:
            np.testing.assert_allclose(a.flux_predictions(), b.flux_predictions(), rtol=1e-9)
        else:
            np.testing.assert_array_equal(a.monitor(), b.monitor())
    for e in ens:
        e.close()
