"""A single-launch evaluation whose bounded waits gave up says nothing about the
matrix: the host optimiser's evaluation is then done launch by launch."""
import numpy as np
import pytest
import torch

from rvgp_amd import _lib
from rvgp_amd.dense import CholeskyError
from rvgp_amd.gp import GPREngine


def _engine(single, launches):
    """An engine on the host whose two evaluations report the given statuses."""
    e = GPREngine.__new__(GPREngine)
    e.u = torch.zeros(4, dtype=torch.float64)
    e._result = torch.zeros(10, dtype=torch.float64)
    e.out, e.status = e._result[:9], e._result[9:].view(torch.int32)[:1]

    def report(value, status):
        e.out.copy_(value + torch.arange(9.0))
        e.status.fill_(status)

    e.evaluate = lambda: report(100.0, single)
    e._evaluate_state = lambda: report(7.0, launches)
    return e


def test_an_evaluation_that_timed_out_is_done_launch_by_launch():
    v, g, out = _engine(_lib.ST_TIMEOUT, _lib.ST_OK).nlml_grad_u(np.zeros(4))
    assert v == 7.0 and np.array_equal(g, [12.0, 13.0, 14.0, 15.0]) and len(out) == 9


def test_only_a_matrix_that_is_not_positive_definite_raises():
    assert _engine(_lib.ST_OK, _lib.ST_NOT_SPD).nlml_grad_u(np.zeros(4))[0] == 100.0
    for single, launches in ((_lib.ST_NOT_SPD, _lib.ST_OK), (_lib.ST_TIMEOUT, _lib.ST_NOT_SPD)):
        with pytest.raises(CholeskyError):
            _engine(single, launches).nlml_grad_u(np.zeros(4))
