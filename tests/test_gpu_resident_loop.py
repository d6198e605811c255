"""Resident time loops (one launch per loop, the state on chip) against the
same loops by steps (variant 27), bit for bit: seismograms, kernels, misfit
and snapshots at the edges of the loop kernels' tiles (60 columns; 4, 12, 20, 28
and 60 rows), with several shots side by side, and where the values leave the
range of the fast divisions."""
import ctypes as C
import threading

import numpy as np
import pytest

from conftest import small_config

pytestmark = pytest.mark.gpu


def _cfg(nx, nz, npb=6, nt=60, shots=1, nr=7, si=5, **over):
    nxi, nzi = nx - 2 * npb, nz - 2 * npb
    cfg = small_config(**{"domain.nt": nt, "domain.nx_inner": nxi, "domain.nz_inner": nzi,
                          "domain.nx_inner_boundary": 0, "domain.nz_inner_boundary": 0,
                          "boundary.np_boundary": npb, "inversion.snapshot_interval": si})
    # two coincident sources per shot, receivers over the whole width with
    # one on the grid's rim and two at one point
    ix = [(k + 1) * nxi // (shots + 1) for k in range(shots)]
    cfg["sources"].update(n_sources=2 * shots, n_shots=shots, ix_sources=[x for x in ix for _ in (0, 1)],
                          iz_sources=[nzi // 3] * (2 * shots),
                          moment_angles=[30.0 + 35.0 * k for k in range(2 * shots)],
                          which_source_to_fire_in_which_shot=[[2 * k, 2 * k + 1] for k in range(shots)])
    xr = [k * (nxi - 1) // max(nr - 1, 1) for k in range(nr)]
    zr = [nzi // 2] * nr
    if nr > 2:
        xr[0], zr[0] = -npb, nzi // 2
        xr[2], zr[2] = xr[1], zr[1]
    cfg["receivers"].update(nr=nr, ix_receivers=xr, iz_receivers=zr)
    for k, v in over.items():
        sec, key = k.split("__")
        cfg[sec][key] = v
    return cfg


def _fields(m, seed, scale=1.0):
    rng = np.random.default_rng(seed)
    vp, vs, rho = m.get_parameter_fields()
    vp = vp * scale * (1 + 0.2 * rng.random(vp.shape))
    return vp, vp * (0.4 + 0.1 * rng.random(vp.shape)), rho * (1 + 0.2 * rng.random(vp.shape))


def _gradient(cfg, variant=None, edit=None, before=None, scale=1.0):
    import psvwave_amd
    m = psvwave_amd.fdModel(cfg)
    if variant is not None:
        m.set_step_variant(variant)
    fields = _fields(m, 5, scale)
    if edit:
        fields = edit(*fields)
    m.set_parameter_fields(*fields)
    rng = np.random.default_rng(9)
    shape = (m.n_shots, m.nr, m.nt)
    m.set_observed_data(rng.standard_normal(shape), rng.standard_normal(shape))
    if before:
        before(m)
    for s in range(m.n_shots):
        m.forward_simulate(s)
    m.calculate_l2_misfit()
    m.calculate_l2_adjoint_sources()
    m.reset_kernels()
    for s in range(m.n_shots):
        m.adjoint_simulate(s)
    m.map_kernels_to_velocity()
    return [np.array(m.misfit), *m.get_synthetic_data(), *m.get_lame_kernels(), *m.get_kernels(),
            *m.get_snapshots()]


def _same(a, b, tag):
    for k, (x, y) in enumerate(zip(a, b)):
        assert np.array_equal(x, y, equal_nan=True), (tag, k)


# widths and heights around one, two and three tiles of every kernel, prime
# and square ones; the number of blocks decides which kernel runs
@pytest.mark.parametrize("nx,nz,shots", [
    (20, 20, 1), (60, 28, 1), (61, 29, 1), (59, 60, 2), (121, 61, 3), (180, 57, 2), (233, 113, 1),
    (541, 341, 1), (499, 359, 1), (800, 700, 1), (97, 401, 2), (641, 89, 4), (401, 307, 1), (887, 313, 2), (1201, 431, 1), (1789, 449, 1)])
def test_gradient_equals_steps(nx, nz, shots):
    print(f"[resident] {nx} x {nz}, {shots} shots", flush=True)
    cfg = _cfg(nx, nz, shots=shots, nt=40 if nx * nz > 100000 else 60)
    _same(_gradient(cfg), _gradient(cfg, 27), (nx, nz))


def test_gradient_equals_oracle(oracle_lib):
    from oracle.pyoracle import OracleModel
    cfg = _cfg(133, 71, nt=300, shots=2)
    got = _gradient(cfg)
    import psvwave_amd
    m = psvwave_amd.fdModel(cfg)
    o = OracleModel(cfg)
    o.set_parameter_fields(*_fields(m, 5))
    rng = np.random.default_rng(9)
    shape = (m.n_shots, m.nr, m.nt)
    o.set_observed_data(rng.standard_normal(shape), rng.standard_normal(shape))
    for s in range(2):
        o.forward_simulate(s)
    o.calculate_l2_misfit()
    o.calculate_l2_adjoint_sources()
    o.reset_kernels()
    for s in range(2):
        o.adjoint_simulate(s)
    o.map_kernels_to_velocity()
    _same(got[1:3], o.get_synthetic_data(), "traces")
    _same(got[6:9], o.get_kernels(), "kernels")


@pytest.mark.parametrize("name", ["subnormal", "overflow", "fluid", "no_lambda", "tiny_factors",
                                  "huge_factors"])
def test_values_outside_the_fast_range(name):
    """subnormal: source amplitudes that keep the field among 2^-1074 ..
    2^-900; overflow: an unstable step that runs into infinities; fluid and
    no_lambda: mu = 0, lambda = 0; material factors far from one."""
    print(f"[resident] {name}", flush=True)
    edit, over, scale = None, {}, 1.0
    if name == "subnormal":
        over = dict(sources__peak_frequency=900.0)  # a wavelet that starts at ~1e-300
    elif name == "overflow":
        over = dict(domain__dt=0.01)
    elif name == "fluid":
        def edit(vp, vs, rho):
            vs[:, :40] = 0.0
            return vp, vs, rho
    elif name == "no_lambda":
        def edit(vp, vs, rho):
            return vp * 0 + 2.0, vs * 0 + 2.0 ** 0.5, rho * 0 + 1.0
    elif name == "tiny_factors":
        def edit(vp, vs, rho):
            return vp * 1e-60, vs * 1e-60, rho
    else:
        def edit(vp, vs, rho):
            return vp * 1e20, vs * 1e20, rho
    cfg = _cfg(131, 97, nt=100, shots=2, **over)
    _same(_gradient(cfg, None, edit), _gradient(cfg, 27, edit), name)


def test_many_terms_and_receivers():
    """More than 64 injection targets in one strip (every column and both
    components of a row), and more receivers in a tile than threads (the
    loop then runs by steps)."""
    cfg = _cfg(140, 90, nt=60, nr=240, shots=2)
    _same(_gradient(cfg), _gradient(cfg, 27), "dense")
    cfg = _cfg(60, 40, nt=40, nr=1100)
    _same(_gradient(cfg), _gradient(cfg, 27), "crowded")


@pytest.mark.parametrize("every", [1, 3])
def test_refused_launch_runs_by_steps(every):
    from psvwave_amd import _lib
    lib = _lib.load()
    lib.psv_refuse_resident_loops.argtypes = [C.c_void_p]
    cfg = _cfg(131, 77, nt=60, shots=3)

    def refuse(m):
        m.set_checkpointing(every)
        _lib.check(lib.psv_refuse_resident_loops(m._h))

    n = 9 if every == 1 else 6
    try:
        got = _gradient(cfg, before=refuse)
    except ValueError:  # snapshots are not stored with checkpoints
        assert every > 1
        import psvwave_amd
        outs = []
        for variant, hook in ((None, refuse), (27, lambda m: m.set_checkpointing(every))):
            m = psvwave_amd.fdModel(cfg)
            if variant is not None:
                m.set_step_variant(variant)
            m.set_parameter_fields(*_fields(m, 5))
            hook(m)
            m.run_model(False, True)
            outs.append([*m.get_synthetic_data(), *m.get_lame_kernels()])
        _same(*outs, "refused, checkpoints")
        return
    _same(got[:n], _gradient(cfg, 27)[:n], "refused")


@pytest.mark.parametrize("nx, nz, nt, si, every, refused", [
    (131, 77, 60, 5, 5, False),     # 25 + 25 + 10 steps
    (131, 77, 61, 1, 2, False),     # a last segment of one step
    (90, 61, 60, 5, 12, False),     # one segment
    (90, 61, 40, 10, 2, True),
    (1200, 450, 24, 4, 3, False),   # too large for both directions at once
])
def test_checkpointed_segments(nx, nz, nt, si, every, refused):
    """Segments of a checkpointed adjoint as resident loops that take the
    state over, against full storage by steps."""
    import psvwave_amd
    from psvwave_amd import _lib
    lib = _lib.load()
    lib.psv_refuse_resident_loops.argtypes = [C.c_void_p]
    cfg = _cfg(nx, nz, nt=nt, si=si, shots=2)
    print(f"[resident] checkpoints {nx}x{nz} {nt} {si} {every}", flush=True)
    outs = []
    for variant in (None, 27):
        m = psvwave_amd.fdModel(cfg)
        if variant is not None:
            m.set_step_variant(variant)
        else:
            m.set_checkpointing(every)
        m.set_parameter_fields(*_fields(m, 5))
        for s in range(2):
            m.forward_simulate(s)
        m.calculate_l2_misfit()
        m.calculate_l2_adjoint_sources()
        m.reset_kernels()
        for s in range(2):
            if refused and variant is None:
                _lib.check(lib.psv_refuse_resident_loops(m._h))
            m.adjoint_simulate(s)
        outs.append([*m.get_synthetic_data(), *m.get_lame_kernels()])
    _same(*outs, "checkpoints")


def test_models_in_threads():
    """Loops of several models from several threads at once: the launches of
    all of them share the device."""
    cfgs = [_cfg(300, 200, nt=200, shots=2), _cfg(640, 300, nt=100, shots=1),
            _cfg(90, 61, nt=300, shots=3)]
    want = [_gradient(c, 27) for c in cfgs]
    got = [None] * len(cfgs)

    def work(i):
        for _ in range(3):
            got[i] = _gradient(cfgs[i])

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(cfgs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for i, (a, b) in enumerate(zip(got, want)):
        _same(a, b, i)


def _batch(cfgs, variant=None):
    import psvwave_amd
    b = psvwave_amd.Batch(cfgs)
    if variant is not None:
        b.set_variant(variant)
    rng = np.random.default_rng(4)
    for m, i in enumerate(b.infos):
        shape = (i["nx"], i["nz"])
        vp = 1800.0 + 600.0 * rng.random(shape)
        b.set_parameter_fields(m, vp, vp * (0.4 + 0.1 * rng.random(shape)),
                               1500.0 + 300.0 * rng.random(shape))
        shape = (i["n_shots"], i["nr"], i["nt"])
        b.set_observed_data(m, rng.standard_normal(shape), rng.standard_normal(shape))
    return b


# one launch of small tiles, one of 28-row tiles, and several launches
@pytest.mark.parametrize("sizes,shots", [
    ([(61, 47), (20, 33)], 2), ([(133, 71), (90, 61), (240, 117)], 3),
    ([(301 + 37 * k, 120 + 31 * (k % 5)) for k in range(12)], 2)])
def test_batch_equals_steps(sizes, shots):
    print(f"[resident] batch of {len(sizes)}", flush=True)
    cfgs = [_cfg(nx, nz, shots=shots, nt=40) for nx, nz in sizes]
    outs = []
    for variant in (None, 28):
        b = _batch(cfgs, variant)
        b.forward_all()
        traces = [b.get_synthetic_data(m) for m in range(len(b))]
        b.forward(shots - 1)
        again = [b.get_synthetic_data(m) for m in range(len(b))]
        grads = b.gradients()
        outs.append([x for t in traces + again for x in t] + [grads] +
                    [k for m in range(len(b)) for k in b.get_kernels(m)])
    _same(*outs, sizes[0])
