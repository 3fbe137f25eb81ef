"""The FEMM's checks whether geometry and dof numbers are those of its device
model, and the CSR matrix of a lumped mass, against the general forms."""
import numpy as np
import pytest
import scipy.sparse as sp

from flexshell import femm as FM


@pytest.mark.parametrize("a", [np.arange(12.0).reshape(4, 3), np.arange(12).reshape(2, 6),
                               np.asfortranarray(np.arange(12).reshape(2, 6)), np.arange(6, dtype=np.int32),
                               np.array([np.nan, 0.0, -0.0]), np.zeros((0, 3))])
def test_same_bits(a):
    assert FM._same_bits(a, a.copy())
    assert not FM._same_bits(a, a.reshape(-1, 1)) and not FM._same_bits(a, a.astype(np.float32))
    for i in range(a.size):
        b = a.copy(order="K")
        b.flat[i] = 99
        assert not FM._same_bits(a, b)
    if a.dtype == float and a.size == 3:
        assert not FM._same_bits(a, np.array([np.nan, -0.0, -0.0]))  # bits, not values


@pytest.mark.parametrize("d", [[1.0, 2.0, 3.0], [1.0, 0.0, 3.0], [np.nan, -0.0, np.inf], [0.0], [5.0]])
def test_diag(d):
    d = np.array(d)
    a, b = FM._diag(d.copy()), sp.diags(d, format="csr")
    assert type(a) is type(b) and a.shape == b.shape
    for x, y in ((a.data, b.data), (a.indices, b.indices), (a.indptr, b.indptr)):
        assert x.dtype == y.dtype and np.array_equal(x, y, equal_nan=x.dtype == float)
    assert not np.shares_memory(a.indices, a.indptr)
