"""Entry points that launch in a loop give up the interpreter's lock, whose
holder would stop every other Python thread while the GPU's queue is full."""
import ctypes

from rvgp_amd import _lib

KEEPS_LOCK = 4  # ctypes' FUNCFLAG_PYTHONAPI


def test_launch_loops_give_up_the_lock():
    L = _lib.load_symbols_only()
    assert ctypes.pythonapi.Py_IncRef._flags_ & KEEPS_LOCK
    for name in _lib.SIGNATURES:
        assert bool(getattr(L, name)._flags_ & KEEPS_LOCK) == (name not in _lib.LAUNCH_LOOPS), name
