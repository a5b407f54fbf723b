"""Coefficient schedules on their way to the library (host only): any sequence of triples is taken, and read anew at
every call."""
import copy
import pickle

import numpy as np
import pytest
import torch

from dion_amd import newton_schulz as ns
from dion_amd import ops

ROWS = [[4.0, -6.5, 2.5], [3.0, -2.0, 1.0]]


def _values(coeffs):
    array, n_iters = ops._flat_coeffs(coeffs)
    return list(array), n_iters


@pytest.mark.parametrize("rows", [[list(r) for r in ROWS], [np.array(r) for r in ROWS], [torch.tensor(r) for r in ROWS],
                                  [tuple(r) for r in ROWS]], ids=["lists", "numpy", "tensors", "tuples"])
@pytest.mark.parametrize("outer", [tuple, list])
def test_rows_of_any_kind_are_read_at_every_call(outer, rows):
    rows = copy.deepcopy(rows)
    coeffs = outer(rows)
    assert _values(coeffs) == ([4.0, -6.5, 2.5, 3.0, -2.0, 1.0], 2)
    if isinstance(rows[0], tuple):
        return
    rows[0][0] = 8.0  # in place: the caller's row is another one now
    assert _values(coeffs)[0][0] == 8.0


def test_the_built_in_schedules_are_prepared_once():
    for s in (ns.NS5_COEFFS, ns.POLAR_EXPRESS_COEFFS):
        assert ops._flat_coeffs(s)[0] is ops._flat_coeffs(s)[0]
        assert _values(s) == _values([list(abc) for abc in s]) and isinstance(s, tuple)
        for other in (pickle.loads(pickle.dumps(s)), copy.deepcopy(s)):
            assert other == s and _values(other) == _values(s)
        assert _values(s[:2]) == (_values(s)[0][:6], 2)


def test_rows_that_are_no_triples_are_refused():
    with pytest.raises(ValueError):
        ops._flat_coeffs(((1.0, 2.0),))
