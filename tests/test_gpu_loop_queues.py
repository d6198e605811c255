"""Asynchronous calls around a refused resident launch: the loops after it run
by steps on two lanes for a while, then as resident loops again, and every
output stays that of blocking calls by steps (variant 27), bit for bit."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_resident_loop import _cfg, _fields, _same

pytestmark = pytest.mark.gpu

STEPWISE = 64  # forwards by steps after a refused launch


def _model(cfg, by_steps):
    import psvwave_amd
    m = psvwave_amd.fdModel(cfg)
    if by_steps:
        m.set_step_variant(27)
        m.set_async(False)
    rng = np.random.default_rng(3)
    shape = (m.n_shots, m.nr, m.nt)
    m.set_observed_data(rng.standard_normal(shape), rng.standard_normal(shape))
    return m


def _refuse(m):
    from psvwave_amd import _lib
    lib = _lib.load()
    lib.psv_refuse_resident_loops.argtypes = [C.c_void_p]
    _lib.check(lib.psv_refuse_resident_loops(m._h))


@pytest.mark.parametrize("left", [1, 2, 3, 5])
def test_the_end_of_the_stepwise_forwards(left):
    """The last `left` forwards of the stepwise ones and the first resident
    one are pending when adjoints of all of them follow."""
    print(f"[queues] {left} stepwise forwards left", flush=True)
    cfg = _cfg(131, 77, nt=400, shots=3)
    outs = []
    for by_steps in (False, True):
        m = _model(cfg, by_steps)
        m.set_parameter_fields(*_fields(m, 5))
        if not by_steps:
            _refuse(m)
        for s in range(m.n_shots):
            m.forward_simulate(s)
        m.calculate_l2_misfit()
        m.calculate_l2_adjoint_sources()
        m.reset_kernels()
        if not by_steps:
            for _ in range(STEPWISE - left):
                m.forward_simulate(0, store_fields=False)
                m.synchronize()
        m.set_parameter_fields(*_fields(m, 6))  # other snapshots than before
        for s in (0, 1):
            m.forward_simulate(s)
        for s in (0, 1):
            m.adjoint_simulate(s)
        m.forward_simulate(2)
        m.adjoint_simulate(2)
        m.adjoint_simulate(0)
        m.forward_simulate(0)
        m.adjoint_simulate(1)
        outs.append([*m.get_lame_kernels(), *m.get_synthetic_data(), *m.get_snapshots()])
    _same(*outs, left)


def test_a_refusal_found_when_the_queue_is_full():
    """More calls than the queue keeps status words for, none of which waits:
    the refusal of the first is found in the midst of them."""
    print("[queues] full", flush=True)
    cfg = _cfg(90, 61, nt=20, shots=2)
    outs = []
    for by_steps in (False, True):
        m = _model(cfg, by_steps)
        m.set_parameter_fields(*_fields(m, 5))
        for s in range(m.n_shots):
            m.forward_simulate(s)
        m.calculate_l2_adjoint_sources()
        m.reset_kernels()
        m.set_parameter_fields(*_fields(m, 6))
        if not by_steps:
            _refuse(m)
        for k in range(300):
            m.forward_simulate(0)
            m.forward_simulate(1, store_fields=k % 3 == 0)
            m.adjoint_simulate(k & 1)
            m.adjoint_simulate(1)
        outs.append([*m.get_lame_kernels(), *m.get_synthetic_data(), *m.get_snapshots()])
    _same(*outs, "full")
