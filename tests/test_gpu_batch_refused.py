"""A batch whose resident launches are refused: the loops of that call and of
the next 64 run by steps, on whatever step kernel the batch has."""
import ctypes as C

import pytest

from test_gpu_resident_loop import _batch, _cfg, _same

pytestmark = pytest.mark.gpu


def _refuse(b):
    from psvwave_amd import _lib
    lib = _lib.load()
    lib.psv_batch_refuse_resident_loops.argtypes = [C.c_void_p]
    _lib.check(lib.psv_batch_refuse_resident_loops(b._h))


def _configs(nt):
    return [_cfg(133, 71, shots=3, nt=nt), _cfg(90, 61, shots=3, nt=nt),
            _cfg(240, 117, shots=3, nt=nt)]


def _traces(b):
    return [x for m in range(len(b)) for x in b.get_synthetic_data(m)]


# two steps a launch, whose receivers record increments (6, 7; with an odd
# number of steps too), and one
@pytest.mark.parametrize("variant, nt", [(None, 40), (28, 41), (6, 40), (6, 41), (7, 60), (0, 41)])
def test_forwards(variant, nt):
    print(f"[refused] forwards {variant} {nt}", flush=True)
    cfgs = _configs(nt)
    want = _batch(cfgs, 28)
    want.forward_all()
    for call in ("all", "each"):
        b = _batch(cfgs, variant)
        _refuse(b)
        if call == "all":
            b.forward_all()
        else:
            for s in range(3):
                _refuse(b)
                b.forward(s)
        assert not b.resident()
        _same(_traces(b), _traces(want), (variant, nt, call))
        b.forward_all()
        _same(_traces(b), _traces(want), (variant, nt, call, "again"))


@pytest.mark.parametrize("variant", [None, 28, 9])
def test_gradients(variant):
    print(f"[refused] gradients {variant}", flush=True)
    cfgs = _configs(40)
    want = _batch(cfgs, 28)
    misfits = want.gradients()
    b = _batch(cfgs, variant)
    _refuse(b)
    for k in range(2):
        _same([b.gradients()], [misfits], (variant, k))
        for m in range(len(b)):
            _same(b.get_kernels(m), want.get_kernels(m), (variant, k, m))


def test_the_end_of_the_stepwise_calls():
    print("[refused] end", flush=True)
    cfgs = _configs(20)
    want = _batch(cfgs, 28)
    want.forward_all()
    b = _batch(cfgs)
    assert b.resident()
    _refuse(b)
    for k in range(70):
        b.forward_all()
        if k in (0, 1, 62, 63, 64, 65, 69):
            _same(_traces(b), _traces(want), k)
    assert b.resident()


def test_autotune_goes_on_by_steps():
    print("[refused] autotune", flush=True)
    cfgs = _configs(40)
    want = _batch(cfgs, 28)
    want.forward_all()
    b = _batch(cfgs)
    _refuse(b)
    b.autotune(steps=6)
    assert not b.resident()
    b.forward_all()
    _same(_traces(b), _traces(want), "autotune")
