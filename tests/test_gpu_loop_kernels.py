"""Every kernel of the resident loops, named by the rows of its tiles, and the
one of 60 rows (16 wavefronts, a block per compute unit) at the edges of its
tiles, bit for bit against the loops by steps.  The largest grids run on it,
and so do those with 513 to 1024 receivers in a tile."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_resident_loop import _batch, _cfg, _fields, _gradient, _same

pytestmark = pytest.mark.gpu


def _rows(cfg, loops=1):
    import psvwave_amd
    from psvwave_amd import _lib
    lib = _lib.load()
    lib.psv_resident_rows.argtypes = [C.c_void_p, C.c_int, C.POINTER(C.c_int)]
    m, rows = psvwave_amd.fdModel(cfg), C.c_int()
    _lib.check(lib.psv_resident_rows(m._h, loops, C.byref(rows)))
    return rows.value


def _crowded(nx, nz, nr, **kw):
    """nr receivers, 513 of them at one point, the others over the grid."""
    cfg = _cfg(nx, nz, nr=1, **kw)
    npb = cfg["boundary"]["np_boundary"]
    x = [nx // 2 - npb] * 513 + [(7 * k) % nx - npb for k in range(nr - 513)]
    z = [nz // 2 - npb] * 513 + [(5 * k) % nz - npb for k in range(nr - 513)]
    cfg["receivers"].update(nr=nr, ix_receivers=x, iz_receivers=z)
    return cfg


# the sizes of test_gradient_equals_steps reach the kernels up to 28 rows
@pytest.mark.parametrize("nx, nz, shots, rows", [
    (121, 61, 1, 4), (401, 307, 1, 12), (800, 700, 1, 20), (1789, 449, 1, 28),
    (1860, 470, 1, 60), (1789, 479, 1, 60), (1801, 461, 1, 60), (1920, 480, 1, 60),
    (1921, 480, 1, 0), (2400, 1237, 1, 0)])
def test_the_kernel_of_a_grid(nx, nz, shots, rows):
    assert _rows(_cfg(nx, nz, nt=5, shots=shots)) == rows


@pytest.mark.parametrize("nx, nz", [(1860, 470), (1789, 479), (1920, 480)])
def test_largest_grids(nx, nz):
    print(f"[rows 60] {nx} x {nz}", flush=True)
    cfg = _cfg(nx, nz, nt=25)
    assert _rows(cfg) == 60
    _same(_gradient(cfg), _gradient(cfg, 27), (nx, nz))


@pytest.mark.parametrize("nx, nz, nr, shots", [
    (20, 20, 513, 1),      # one tile, smaller than its rims
    (60, 60, 1024, 1),     # one full tile, a receiver for each thread
    (61, 61, 700, 2), (121, 119, 600, 3), (180, 59, 1000, 1), (59, 240, 700, 2),
    (127, 64, 900, 2)])    # tiles of 42 and 43 columns, of 32 rows
def test_crowded_tiles(nx, nz, nr, shots):
    print(f"[rows 60] {nx} x {nz}, {nr} receivers, {shots} shots", flush=True)
    cfg = _crowded(nx, nz, nr, nt=60, shots=shots)
    assert _rows(cfg, shots) == 60
    _same(_gradient(cfg), _gradient(cfg, 27), (nx, nz, nr))


def test_checkpointed_segments():
    import psvwave_amd
    print("[rows 60] checkpoints", flush=True)
    cfg = _crowded(121, 119, 600, nt=60, shots=2)
    assert _rows(cfg, 2) == 60
    outs = []
    for variant in (None, 27):
        m = psvwave_amd.fdModel(cfg)
        if variant is not None:
            m.set_step_variant(variant)
        else:
            m.set_checkpointing(5)
        m.set_parameter_fields(*_fields(m, 5))
        m.run_model(False, True)
        outs.append([*m.get_synthetic_data(), *m.get_lame_kernels()])
    _same(*outs, "checkpoints")


@pytest.mark.parametrize("shots", [1, 2])
def test_batch(shots):
    """A member that no other kernel holds, beside small ones: one launch, and
    two."""
    print(f"[rows 60] batch, {shots} shots", flush=True)
    cfgs = [_cfg(nx, nz, shots=shots, nt=20) for nx, nz in [(1860, 470), (20, 33), (90, 131)]]
    assert _rows(cfgs[0]) == 60
    outs = []
    for variant in (None, 28):
        b = _batch(cfgs, variant)
        assert b.resident() == (variant is None)
        b.forward_all()
        traces = [x for m in range(len(b)) for x in b.get_synthetic_data(m)]
        grads = b.gradients()
        outs.append(traces + [grads] + [k for m in range(len(b)) for k in b.get_kernels(m)])
    _same(*outs, shots)


def test_beside_loops_of_other_kernels():
    """Blocks that need a whole compute unit and smaller ones, from two
    threads: the gate admits no launch that would wait for a unit."""
    import threading
    print("[rows 60] threads", flush=True)
    cfgs = [_cfg(1860, 470, nt=25), _cfg(640, 300, nt=100)]
    want = [_gradient(c, 27) for c in cfgs]
    got = [None] * 2

    def work(i):
        for _ in range(3):
            got[i] = _gradient(cfgs[i])

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for i in range(2):
        _same(got[i], want[i], i)
    assert all(np.isfinite(x).all() for g in got for x in g)
