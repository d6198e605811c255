"""Calls that run out of device memory part of the way: the next call finds
nothing half-built, and its outputs are those of a model that never failed."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_resident_loop import _batch, _cfg, _fields, _gradient, _same

pytestmark = pytest.mark.gpu


def _fail(m, n):
    """The model's allocation after the next n fails."""
    from psvwave_amd import _lib
    lib = _lib.load()
    lib.psv_fail_allocation.argtypes = [C.c_void_p, C.c_int, C.c_int]
    _lib.check(lib.psv_fail_allocation(m._h, n, 1))


def _warm(m):
    """The tables of the resident loops, which count as allocations too."""
    for s in range(m.n_shots):
        m.forward_simulate(s, store_fields=False)
    m.synchronize()


def _run(m, cfg, seed, every=1):
    import psvwave_amd
    # (relative to the configuration's background, not to what m holds)
    m.set_parameter_fields(*_fields(psvwave_amd.fdModel(cfg), seed))
    rng = np.random.default_rng(9)
    shape = (m.n_shots, m.nr, m.nt)
    m.set_observed_data(rng.standard_normal(shape), rng.standard_normal(shape))
    for s in range(m.n_shots):
        m.forward_simulate(s)
    m.calculate_l2_misfit()
    m.calculate_l2_adjoint_sources()
    m.reset_kernels()
    for s in range(m.n_shots):
        m.adjoint_simulate(s)
    return [np.array(m.misfit), *m.get_synthetic_data(), *m.get_lame_kernels(),
            *(m.get_snapshots() if every == 1 else ())]


def _reference(cfg, seed):
    import psvwave_amd
    m = psvwave_amd.fdModel(cfg)
    m.set_step_variant(27)
    m.set_async(False)
    return _run(m, cfg, seed)


@pytest.mark.parametrize("variant", [None, 27])
@pytest.mark.parametrize("n", [0, 1, 4])
def test_snapshot_store(variant, n):
    """The n-th of the five arrays of the store; by steps, of the second
    lane's state first."""
    import psvwave_amd
    print(f"[allocation] store {variant} {n}", flush=True)
    cfg = _cfg(131, 77, nt=60, shots=3)
    m = psvwave_amd.fdModel(cfg)
    if variant is not None:
        m.set_step_variant(variant)
        _fail(m, n)
        with pytest.raises(RuntimeError, match="memory"):
            m.forward_simulate(0, store_fields=False)
        m.forward_simulate(0, store_fields=False)
        m.synchronize()
    else:
        _warm(m)
    _fail(m, n)
    with pytest.raises(RuntimeError, match="memory"):
        m.forward_simulate(0)
        m.synchronize()
    _same(_run(m, cfg, 6), _reference(cfg, 6), (variant, n))


@pytest.mark.parametrize("n", [0, 1])
def test_room_of_a_larger_launch(n):
    """Three loops after a launch of one: their arguments, then their exchange
    cells; a launch of one afterwards, then three again."""
    import psvwave_amd
    print(f"[allocation] room {n}", flush=True)
    cfg = _cfg(131, 77, nt=60, shots=3)
    m = psvwave_amd.fdModel(cfg)
    m.forward_simulate(0)
    m.synchronize()
    _fail(m, n)
    try:
        for s in range(m.n_shots):
            m.forward_simulate(s)
        m.synchronize()
    except RuntimeError as e:
        assert "memory" in str(e)
    for _ in range(70):  # past the forwards by steps that may follow
        m.forward_simulate(0)
        m.synchronize()
    _same(_run(m, cfg, 6), _reference(cfg, 6), n)


@pytest.mark.parametrize("variant, n", [(None, 0), (None, 3), (None, 4), (27, 0), (27, 9),
                                        (27, 10), (27, 13)])
def test_checkpoint_segments(variant, n):
    """Segment buffers that grow; by steps the recomputation's state first."""
    import psvwave_amd
    print(f"[allocation] segments {variant} {n}", flush=True)
    cfg = _cfg(131, 77, nt=60, shots=2)
    m = psvwave_amd.fdModel(cfg)
    if variant is not None:
        m.set_step_variant(variant)
    if variant is None:  # segments of two snapshots first
        m.set_checkpointing(2)
        _run(m, cfg, 7, 2)
    m.set_checkpointing(5)
    m.forward_simulate(0)
    m.synchronize()
    _fail(m, n)
    with pytest.raises(RuntimeError, match="memory"):
        m.adjoint_simulate(0)
    if variant is None:  # smaller segments, then the larger ones
        m.set_checkpointing(2)
        _same(_run(m, cfg, 7, 2), _reference(cfg, 7)[:6], "smaller")
        m.set_checkpointing(5)
    _same(_run(m, cfg, 6, 5), _reference(cfg, 6)[:6], (variant, n))


def test_nothing_changes_without_a_failure():
    cfg = _cfg(131, 77, nt=60, shots=3)
    _same(_gradient(cfg), _gradient(cfg, 27), "gradient")


@pytest.mark.parametrize("n", [0, 1])
def test_loops_without_room_run_by_steps(n):
    """No room for the arguments or the cells of three loops: the calls, which
    were all accepted, run by steps."""
    import psvwave_amd
    print(f"[allocation] forwards {n}", flush=True)
    cfg = _cfg(131, 77, nt=60, shots=3)
    m = psvwave_amd.fdModel(cfg)
    m.forward_simulate(0)
    m.synchronize()
    m.set_parameter_fields(*_fields(psvwave_amd.fdModel(cfg), 6))
    _fail(m, n)
    for s in range(m.n_shots):
        m.forward_simulate(s)
    want = _reference(cfg, 6)
    _same([*m.get_synthetic_data(), *m.get_snapshots()], want[1:3] + want[6:], n)


@pytest.mark.parametrize("n", [0, 1, 2, 3])
def test_adjoints_without_room(n):
    """Three adjoints after single forwards: no room for the first or second
    buffer of deferred kernel terms (fewer then share a launch), or for the
    arguments or cells of three loops (all by steps, terms in their order)."""
    import psvwave_amd
    print(f"[allocation] adjoints {n}", flush=True)
    cfg = _cfg(131, 77, nt=60, shots=3)
    m = psvwave_amd.fdModel(cfg)
    m.set_parameter_fields(*_fields(m, 6))
    rng = np.random.default_rng(9)
    shape = (m.n_shots, m.nr, m.nt)
    m.set_observed_data(rng.standard_normal(shape), rng.standard_normal(shape))
    for s in range(m.n_shots):
        m.forward_simulate(s)
        m.synchronize()
    m.calculate_l2_adjoint_sources()
    m.reset_kernels()
    _fail(m, n)
    for s in range(m.n_shots):
        m.adjoint_simulate(s)
    _same(m.get_lame_kernels(), _reference(cfg, 6)[3:6], n)
    _same(_run(m, cfg, 7), _reference(cfg, 7), "afterwards")


@pytest.mark.parametrize("n, times", [(0, 1), (3, 1), (0, 2), (0, 3), (3, 2)])
def test_batch_gradients(n, times):
    """The second member's snapshot store: after one failure the call runs by
    steps, after a second it is raised and leaves the kernels as they were,
    and the next one builds its launches anew."""
    from psvwave_amd import _lib
    print(f"[allocation] batch {n} {times}", flush=True)
    lib = _lib.load()
    lib.psv_batch_fail_allocation.argtypes = [C.c_void_p, C.c_int, C.c_int, C.c_int]
    cfgs = [_cfg(133, 71, shots=2, nt=40), _cfg(90, 61, shots=2, nt=40)]
    want = _batch(cfgs, 28)
    misfits = want.gradients()
    b = _batch(cfgs)
    b.forward_all()
    b.forward(0)  # (the members' tables are there)
    zero = [b.get_kernels(m) for m in range(2)]
    # (a store that failed is tried again from its first array)
    _lib.check(lib.psv_batch_fail_allocation(b._h, 1, n, times))
    if times > 1:
        with pytest.raises(RuntimeError, match="memory"):
            b.gradients()
        for m in range(2):
            _same(b.get_kernels(m), zero[m], "untouched")
    for k in range(3):
        _same([b.gradients()], [misfits], (n, times, k))
        for m in range(2):
            _same(b.get_kernels(m), want.get_kernels(m), (n, times, k, m))
    assert b.resident()


@pytest.mark.parametrize("n, times", [(0, 1), (4, 1), (10, 1), (11, 1), (12, 1), (13, 1), (14, 1),
                                      (0, 30)])
def test_tables_of_a_loop_kernel(n, times):
    """A kernel's 11 tables that find no room: another kernel or, where none has
    room, loops by steps; and the first kernel again the next time.  Then the
    words, the arguments and the cells of the first launch."""
    import psvwave_amd
    from psvwave_amd import _lib
    from test_gpu_loop_kernels import _rows
    print(f"[allocation] tables {n} {times}", flush=True)
    cfg = _cfg(131, 77, nt=60, shots=3)
    m = psvwave_amd.fdModel(cfg)
    lib = _lib.load()
    lib.psv_fail_allocation.argtypes = [C.c_void_p, C.c_int, C.c_int]
    _lib.check(lib.psv_fail_allocation(m._h, n, times))
    fields = _fields(psvwave_amd.fdModel(cfg), 6)
    m.set_parameter_fields(*fields)
    try:
        for s in range(m.n_shots):
            m.forward_simulate(s, store_fields=False)
        m.synchronize()
    except RuntimeError as e:  # the loops by steps found no room either
        assert times > 1 and "memory" in str(e)
    else:
        _same(m.get_synthetic_data(), _reference(cfg, 6)[1:3], (n, times))
    _lib.check(lib.psv_fail_allocation(m._h, 0, 0))
    for _ in range(64):  # the forwards by steps that may follow
        m.forward_simulate(0, store_fields=False)
    rows = C.c_int()
    lib.psv_resident_rows.argtypes = [C.c_void_p, C.c_int, C.POINTER(C.c_int)]
    for loops in (1, 3):
        _lib.check(lib.psv_resident_rows(m._h, loops, C.byref(rows)))
        assert rows.value == _rows(cfg, loops) > 0
    _same(_run(m, cfg, 7), _reference(cfg, 7), "afterwards")


def test_tables_of_a_batch():
    """No room for a member's tables: by steps, and resident the next time."""
    from psvwave_amd import _lib
    print("[allocation] batch tables", flush=True)
    lib = _lib.load()
    lib.psv_batch_fail_allocation.argtypes = [C.c_void_p, C.c_int, C.c_int, C.c_int]
    cfgs = [_cfg(133, 71, shots=2, nt=40), _cfg(90, 61, shots=2, nt=40)]
    b, want = _batch(cfgs), _batch(cfgs, 28)
    want.forward_all()
    # every kernel's tables, then the state of a lockstep by steps
    _lib.check(lib.psv_batch_fail_allocation(b._h, 1, 0, 30))
    b.forward_all()
    _lib.check(lib.psv_batch_fail_allocation(b._h, 1, 0, 0))
    for k in range(2):
        for m in range(2):
            _same(b.get_synthetic_data(m), want.get_synthetic_data(m), (k, m))
        assert b.resident()
        b.forward_all()
