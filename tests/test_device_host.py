"""The library's host code on a stand-in for the HIP runtime
(device_stub.cpp): no GPU, kernels do nothing, allocations fail on demand,
and every launch is checked for pointers to memory that is not there.

Each case runs in a process of its own, where the stand-in is loaded before
the library.
"""
import ctypes as C
import dataclasses
import os
import subprocess
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
PKG = os.path.join(os.path.dirname(HERE), "hpc-ca-phospattern_amd")


class Stub:
    """The stand-in's own entry points."""

    def __init__(self, path):
        self.lib = C.CDLL(path, mode=C.RTLD_GLOBAL)
        self.lib.stub_fail_alloc_in.argtypes = [C.c_long]
        for name in ("stub_allocs", "stub_live_bytes", "stub_bad", "stub_launches"):
            getattr(self.lib, name).restype = C.c_long
        self.lib.stub_launches.argtypes = [C.c_char_p]
        self.lib.stub_bad_at.argtypes = [C.c_long]
        self.lib.stub_bad_at.restype = C.c_char_p

    def launches(self, part):
        return self.lib.stub_launches(part.encode())

    def sound(self):
        """No launch, copy or free touched memory that is not there, and no
        error waits for a later call to trip over."""
        bad = [self.lib.stub_bad_at(k).decode() for k in range(self.lib.stub_bad())]
        assert not bad, bad[:5]
        assert self.lib.stub_pending_error() == 0

    def failing(self, k, call):
        """`call` with its k-th allocation failing; whether it made that many."""
        before = self.lib.stub_allocs()
        self.lib.stub_fail_alloc_in(k)
        try:
            call()
        finally:
            self.lib.stub_fail_alloc_in(-1)
        return self.lib.stub_allocs() - before > k


def _ensemble(count=3, n=(20, 18, 14), **kw):
    import csparks as cs
    import dyad
    ds = [dyad.small_dyad(n=n, seed=3 + k) for k in range(count)]
    return cs.Ensemble([(d.geometry, d.model, cs.Options(seed=1 + k, open={"ryr": [0]}, **kw))
                        for k, d in enumerate(ds)], instances=list(range(count)))


def _net():
    import closure
    return closure.load(os.path.join(PKG, "closure_params.npz"))[0]


def ensemble_closure_without_memory(stub):
    """Closure gating needs a wider index of kept voxels than the ensemble
    was made with.  Without memory for it the call still succeeds, and steps
    (graphs among them) run on what there is; with it, they run in pairs."""
    net, k, more = _net(), 0, True
    while more:
        ens = _ensemble()
        ens.set_graph(True)
        ens.step(ens.period)
        more = stub.failing(k, lambda: ens.set_gating(ens.GATE_CLOSURE, net))
        stub.sound()
        pairs = stub.launches("k_pass2")
        ens.step(ens.period + 3)
        stub.sound()
        assert (stub.launches("k_pass2") > pairs) == (not more), f"allocation {k}"
        ens.set_gating(ens.GATE_OWN)
        pairs = stub.launches("k_pass2")
        ens.step(ens.period + 3)
        stub.sound()
        assert stub.launches("k_pass2") > pairs
        ens.close()
        k += 1
    assert k > 1


def ensemble_retiring_without_memory(stub):
    """Fewer active members may take more tiles than the list made for all
    of them holds: 260 members of one column tile each run 12 planes to a
    block, 250 of them 6 planes in twice as many blocks (at most 512 are
    resident).  Without memory for the longer list, steps run one by one,
    and in pairs again once a choice of members finds room."""
    def keep(ens, n):
        ens.set_active([k < n for k in range(ens.count)])

    ens = _ensemble(count=260, n=(9, 9, 12))
    ens.set_graph(True)
    ens.step(ens.period)
    assert stub.failing(0, lambda: keep(ens, 250)), "the case needs a longer list"
    stub.sound()
    pairs = stub.launches("k_pass2")
    ens.step(ens.period + 5)
    stub.sound()
    assert stub.launches("k_pass2") == pairs
    keep(ens, 249)
    ens.step(ens.period + 5)
    stub.sound()
    assert stub.launches("k_pass2") > pairs
    ens.close()


def ensemble_launch_without_memory(stub):
    """A launch shape whose tiles find no memory is refused; the one before
    stays, with its tiles (single steps run on them), also with members
    retired."""
    ens = _ensemble(n=(64, 63, 24))
    ens.set_active([True, False, True])
    shape = ens.launch()
    with pytest.raises(RuntimeError):
        stub.failing(0, lambda: ens.set_launch(rows=1, zchunk=2))
    assert ens.launch() == shape
    stub.sound()
    ens.step(1)
    stub.sound()
    ens.set_launch(rows=1, zchunk=2)
    ens.step(1)
    ens.close()


def flux_network_predicts_each_state_once(stub):
    """With the flux network a call of n steps predicts from the state it
    starts on and from the one after every step (n + 1 times; the range
    monitor counts each), in pairs and with a last single step alike."""
    import closure
    fnet = closure.load_flux(os.path.join(PKG, "closure_params.npz"))[0]
    net, ens = _net(), _ensemble()
    ens.set_gating(ens.GATE_CLOSURE, net)
    ens.set_flux_closure(fnet)
    for n in (1, 2, 3, 20, 21):
        before = stub.launches("k_closure_predict")
        ens.step(n)
        assert stub.launches("k_closure_predict") - before == n + 1, n
    ens.close()


def ensemble_launch_names_the_form(stub):
    """persistent says which passes run: 2 (the default of five-slot
    models) pairs of steps, 0 and 1 one-step passes of the given shape.
    What is read can be written back; the shape's other keys leave the form;
    autotune's answer, given to set_launch, keeps what it chose."""
    import csparks as cs
    import dyad
    forms = ("k_batch_tiles", "k_batch_stencil", "k_pass2")

    def passes(ens, n=4):
        before = [stub.launches(f) for f in forms]
        ens.step(n)
        return [stub.launches(f) - k for f, k in zip(forms, before)]

    ens = _ensemble()
    assert ens.launch()["persistent"] == 2 and passes(ens) == [0, 0, 2]
    ens.set_launch(**ens.launch())
    ens.set_launch(rows=8, zchunk=8)
    assert ens.launch()["persistent"] == 2 and passes(ens) == [0, 0, 2]
    for form in (0, 1):
        ens.set_launch(persistent=form)
        assert ens.launch()["persistent"] == form and passes(ens) == [4 * (form == k) for k in range(3)]
    ens.set_launch(persistent=2)
    assert passes(ens, 5) == [0, 1, 2]   # the odd step as it ran before
    with pytest.raises(RuntimeError):
        ens.set_launch(persistent=3)
    best, _ = ens.autotune(1)
    want = passes(ens)
    ens.set_launch(**best)
    assert passes(ens) == want and ens.launch() == best
    ens.close()

    d = dyad.small_dyad()   # a slab of one column in x cannot pair
    geom = cs.Geometry(voxels=np.ascontiguousarray(d.geometry.voxels[:1]), h=d.geometry.h,
                       domain_names=list(d.geometry.domain_names),
                       domain_connections=d.geometry.domain_connections, boundaries=[])
    one = cs.Ensemble([(geom, dataclasses.replace(d.model, ryr=None, p_ryr=None), cs.Options(seed=1))])
    assert one.launch()["persistent"] == 0
    with pytest.raises(RuntimeError):
        one.set_launch(persistent=2)
    assert sum(passes(one)) == 4
    one.close()


def launch_config_names_the_form(stub):
    """Five-slot models run pairs by default in both precisions and at every
    size; the launch config says so (fuse = 1, or fuse_fixed = 2), can be
    written back, and keeps the form when another key changes.  fuse = 0
    asks for one-step passes, and autotune's answer for what it chose."""
    import csparks as cs
    import dyad

    def pairs(sim, n=4):
        before = [stub.launches(k) for k in ("k_pass2", "k_stencil")]
        sim.step(n)
        two, one = (stub.launches(k) - b for k, b in zip(("k_pass2", "k_stencil"), before))
        assert 2 * two + one == n
        return two

    def says(cfg):
        return cfg["fuse"] == 1 or cfg["fuse_fixed"] == 2

    for n, precision in (((20, 18, 14), "f64"), ((20, 18, 14), "f32"), ((300, 300, 40), "f32")):
        d = dyad.small_dyad(n=n)
        sim = cs.Simulation(d.geometry, d.model, cs.Options(seed=1, open={"ryr": [0]}, precision=precision))
        assert pairs(sim) == 2 and says(sim.launch_config())
        sim.set_launch_config(**sim.launch_config())
        assert pairs(sim) == 2
        sim.set_launch_config(fuse_xcd=4)
        sim.set_launch_config(rows=8, zchunk=4)
        assert pairs(sim) == 2 and says(sim.launch_config())
        sim.set_launch_config(fuse=0)
        assert pairs(sim) == 0 and not says(sim.launch_config())
        sim.set_launch_config(rows=4)
        assert pairs(sim) == 0
        sim.set_launch_config(fuse=1)
        assert pairs(sim) == 2
        sim.set_launch_config(fuse=0, fuse_fixed=2)
        assert pairs(sim) == 2
        best, _ = sim.autotune(1)
        want = pairs(sim)
        assert (want == 2) == says(best)
        sim.set_launch_config(**best)
        assert pairs(sim) == want
        with pytest.raises(RuntimeError):
            sim.set_launch_config(fuse_fixed=3)
        sim.close()

    d = dyad.small_dyad()   # a slab of one column in x has no compiled pass
    geom = cs.Geometry(voxels=np.ascontiguousarray(d.geometry.voxels[:1]), h=d.geometry.h,
                       domain_names=list(d.geometry.domain_names),
                       domain_connections=d.geometry.domain_connections, boundaries=[])
    one = cs.Simulation(geom, dataclasses.replace(d.model, ryr=None, p_ryr=None), cs.Options(seed=1))
    assert not says(one.launch_config()) and pairs(one) == 0
    with pytest.raises(RuntimeError):
        one.set_launch_config(fuse_fixed=2)
    one.close()


def steps_allocate_nothing(stub):
    """The calls that choose a launch shape make its tile list: steps need
    no memory.  A shape whose list finds none is refused and the one before
    stays; a context that finds no room for what two-step passes need runs
    without them."""
    import csparks as cs
    import dyad
    d = dyad.small_dyad(n=(64, 63, 24))
    opts = cs.Options(seed=1, open={"ryr": [0]})

    def steps(sim):
        before = stub.lib.stub_allocs()
        two = stub.launches("k_pass2")
        sim.step(4)
        stub.sound()
        assert stub.lib.stub_allocs() == before
        return stub.launches("k_pass2") - two

    sim = cs.Simulation(d.geometry, d.model, opts)
    assert steps(sim) == 2
    shape = sim.launch_config()
    with pytest.raises(RuntimeError):
        stub.failing(0, lambda: sim.set_launch_config(fuse_zchunk=7))
    stub.sound()
    assert sim.launch_config() == shape and steps(sim) == 2
    sim.set_launch_config(fuse_zchunk=7)
    assert steps(sim) == 2
    sim.set_launch_config(fuse_zchunk=100)   # the grid's depth at most
    assert steps(sim) == 2
    sim.autotune(1)
    steps(sim)
    sim.close()

    # every allocation of cs_create in turn: refused, or without two-step passes
    made, k, more = [], 0, True
    while more:
        held = []
        try:
            more = stub.failing(k, lambda: held.append(cs.Simulation(d.geometry, d.model, opts)))
            made.append(steps(held[0]))
            stub.sound()
            held[0].close()
        except RuntimeError:
            pass
        k += 1
    assert made == [0, 0, 0, 2], made    # the domain's record, the words, the tiles; then none fails


def fields_move_without_memory(stub):
    """Setting and reading fields allocates nothing, and their staging stays
    inside the context's own memory, down to a plane of one species whose
    doubles are larger than the field."""
    import csparks as cs
    import dyad
    d = dyad.small_dyad(n=(33, 31, 14))
    g, m = d.geometry, d.model
    ca = dataclasses.replace(m, species_names=m.species_names[:1], init=np.asarray(m.init)[:, :1],
                             diffusive=[[s for s in k if s == 0] for k in m.diffusive],
                             sigma=[[v for v, s in zip(sg, k) if s == 0] for sg, k in zip(m.sigma, m.diffusive)],
                             buffers=[[] for _ in m.buffers], ryr=None, p_ryr=None)

    def cut(x, y, z):
        return cs.Geometry(voxels=np.ascontiguousarray(g.voxels[:x, :y, :z]), h=g.h,
                           domain_names=list(g.domain_names), domain_connections=g.domain_connections,
                           boundaries=[])

    for geom, model in ((g, m), (cut(1, 31, 14), ca), (cut(2, 31, 14), ca), (cut(1, 1, 14), ca), (cut(33, 1, 1), ca)):
        for precision in ("f32", "f64"):
            sim = cs.Simulation(geom, model, cs.Options(seed=1, precision=precision))
            before = stub.lib.stub_allocs()
            stub.lib.stub_fail_alloc_in(0)
            sim.set_species(0, sim.species(0))
            stub.lib.stub_fail_alloc_in(-1)
            assert stub.lib.stub_allocs() == before
            stub.sound()
            sim.close()


def five_species_outside_the_layout_run_compiled_masks(stub):
    """FP32 models of five species that the compiled pass of the five-slot
    layout does not take (a species without a buffer, TRPN diffusing on a
    substep) run two-step passes with their step masks compiled in, unless
    fuse_fixed = 0 asks for run-time masks."""
    import csparks as cs
    import dyad
    d = dyad.small_dyad(n=(40, 23, 9))
    m = d.model
    unbound = dataclasses.replace(m, buffers=[[b for b in bs if b.bound != 4] for bs in m.buffers])
    slow = dataclasses.replace(m, diffusive=[list(k) + [4] for k in m.diffusive],
                               sigma=[list(s) + [220000.0 / 100.25] for s in m.sigma])
    for model in (unbound, slow):
        sim = cs.Simulation(d.geometry, model, cs.Options(seed=1, open={"ryr": [0]}, precision="f32"))
        for fixed, masks in ((1, "9u, 9u, 2u>"), (0, "4294967295u, 4294967295u, 4294967295u>")):
            sim.set_launch_config(fuse=1, fuse_fixed=fixed)
            before = stub.launches("k_step2<float, 5, 16, false, " + masks)
            sim.step(40)
            assert stub.launches("k_step2<float, 5, 16, false, " + masks) > before, (fixed, masks)
        sim.close()
    assert stub.launches("k_pass2") == 0


def planes_under_32_bit_offsets(stub):
    """A block's z-groups end below 2^32 bytes, those of the five-slot pass
    with what a row's last chunk reads beyond them; the general pass reads
    nothing there, and its largest block is not smaller for it."""
    f = stub.lib.stub_zlimit
    f.argtypes = [C.c_uint64] * 3
    group = 20 * 17895697                  # 12 groups are 16 bytes short of 2^32
    assert (f(group, 100, 0), f(group, 100, 64)) == (8, 7)
    assert (f(group, 5, 0), f(group, 5, 64)) == (5, 5)
    assert (f(858993459, 9, 0), f(858993460, 9, 0), f(858993459, 9, 64)) == (1, 0, 0)
    for g in (4, 20, 40, 12345680, 858993440):
        for pad in (0, 64):
            k = f(g, 1 << 30, pad)
            assert (k + 4) * g + pad < 1 << 32 <= (k + 5) * g + pad or k == 1 << 30


def a_failed_call_leaves_no_error(stub):
    """A call that fails for want of memory reports it, once: steps of this
    and other contexts go on."""
    import csparks as cs
    import dyad
    d = dyad.small_dyad()
    opts = cs.Options(seed=1, open={"ryr": [0]})
    sim, ens, net = cs.Simulation(d.geometry, d.model, opts), _ensemble(), _net()
    line = (0, (0, 0, -3), d.model.conv)
    calls = [lambda: cs.Simulation(d.geometry, d.model, opts), lambda: sim.linescan(1, *line), _ensemble,
             lambda: ens.linescans(1, *line), ens.closure_features, ens.channel_ca, _net,
             lambda: net.forward(np.zeros((64, 30))), lambda: net.set_data(np.zeros((64, 30)), np.zeros(64))]
    for call in calls:
        with pytest.raises(RuntimeError):
            stub.failing(0, call)
        stub.sound()
        sim.step(2)
        ens.step(2)


def buffers_that_failed_to_grow(stub):
    """A call that finds no memory for more samples or draws fails; a
    smaller one after it allocates what it needs and runs."""
    import csparks as cs
    import dyad
    net = _net()
    for k in range(4):
        net.forward(np.zeros((100, 30)))
        with pytest.raises(RuntimeError):
            stub.failing(k, lambda: net.forward(np.zeros((500 + k, 30))))
        net.forward(np.zeros((80, 30)))
        net.grad(np.zeros((90, 30)), np.zeros(90))
        stub.sound()
    d = dyad.small_dyad()
    sim = cs.Simulation(d.geometry, d.model, cs.Options(seed=1, open={"ryr": [0]}, rng="mt"))
    for run in (sim, _ensemble(rng="mt")):
        run.step(4)
        with pytest.raises(RuntimeError):
            stub.failing(0, lambda: run.step(400))
        stub.sound()
        run.step(2)
        stub.sound()


def calls_use_their_own_device(stub):
    """Launch shapes, fields, outputs and steps of a context, an ensemble and
    a network stay on the device they were made on, whichever is current."""
    import csparks as cs
    import dyad
    d = dyad.small_dyad()
    sim = cs.Simulation(d.geometry, d.model, cs.Options(seed=1, open={"ryr": [0]}))
    ens, net = _ensemble(), _net()
    line = (0, (0, 0, -3), d.model.conv)
    for call in (lambda: sim.set_launch_config(fuse=1, fuse_zchunk=7), lambda: sim.step(4), lambda: sim.autotune(1),
                 lambda: sim.set_species(0, sim.species(0)), lambda: sim.linescan(1, *line), sim.stats,
                 lambda: ens.set_launch(zchunk=4), lambda: ens.set_active([True, False, True]),
                 lambda: ens.set_gating(ens.GATE_CLOSURE, net), lambda: ens.step(5), lambda: ens.autotune(1),
                 lambda: ens.linescans(1, *line), lambda: net.forward(np.zeros((64, 30)))):
        stub.lib.hipSetDevice(1)
        call()
        stub.sound()
    stub.lib.hipSetDevice(1)
    sim.step(4)
    ens.step(5)
    stub.sound()


def a_refused_training_set_is_given_back(stub):
    """cs_mlp_set_data without memory for all of the set keeps none of it;
    training asks for data, and a set that fits trains."""
    net = _net()
    x, t = np.zeros((400, 30)), np.zeros(400)
    empty = stub.lib.stub_live_bytes()
    k, more = 0, True
    while more:
        try:
            more = stub.failing(k, lambda: net.set_data(x, t))
        except RuntimeError:
            assert stub.lib.stub_live_bytes() == empty, k
            with pytest.raises(RuntimeError):
                net.train(1, 64, 1e-3)
        stub.sound()
        k += 1
    assert k == 5   # four allocations, then none fails
    net.train(3, 64, 1e-3)


CASES = (ensemble_closure_without_memory,
         ensemble_retiring_without_memory,
         ensemble_launch_without_memory,
         flux_network_predicts_each_state_once,
         ensemble_launch_names_the_form,
         launch_config_names_the_form,
         steps_allocate_nothing,
         fields_move_without_memory,
         five_species_outside_the_layout_run_compiled_masks,
         planes_under_32_bit_offsets,
         a_failed_call_leaves_no_error,
         buffers_that_failed_to_grow,
         calls_use_their_own_device,
         a_refused_training_set_is_given_back)


@pytest.fixture(scope="module")
def stand_in_library(tmp_path_factory):
    path = str(tmp_path_factory.mktemp("stub") / "device_stub.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-I", "/opt/rocm/include", "-I",
                    os.path.join(PKG, "csrc"), os.path.join(HERE, "device_stub.cpp"), "-o", path], check=True)
    return path


@pytest.mark.parametrize("case", CASES, ids=lambda c: c.__name__)
def test_host_code(case, stand_in_library):
    r = subprocess.run([sys.executable, os.path.abspath(__file__), stand_in_library, case.__name__],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr


if __name__ == "__main__":
    sys.path[:0] = [PKG]
    stand_in = Stub(sys.argv[1])
    globals()[sys.argv[2]](stand_in)
    stand_in.sound()
