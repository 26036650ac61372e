"""The int8 batch GEMV on fp16 matrix instructions (sdot_batch.hip): bit-identical to the oracle.

Every tile height (2 .. 12 rows; the next larger one with rows past the batch), groups of half a block of 64 positions,
one block and two, their largest sums, ragged rows and widths down to one block; larger batches and groups, which take
the other kernels, beside them.
"""
import numpy as np
import pytest

import oracle
from openneedle_amd.cq import CQMatrix
from tests.cases import activations, example

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def forced(monkeypatch):
    monkeypatch.setenv("NEEDLE2_GPU_INT8_KSPLIT", "never")
    monkeypatch.setenv("NEEDLE2_GPU_INT8_BATCH", "always")


def check(bits, group, rows, dim, batch):
    packed, norms, cb, dense = example(bits, rows=rows, dim=dim, group=group, seed=group + batch + rows)
    q = CQMatrix(packed, norms, dense.shape, bits, group, cb)
    x = activations((batch, dim), seed=batch)
    x[0] = 0
    x[1] = 0
    x[1, 5] = 1
    np.testing.assert_array_equal(q.matvec_int8(x), oracle.sdot_linear(packed, norms, dense.shape, bits, group, cb, x))


@pytest.mark.parametrize("group", [32, 64, 128, 1024])
@pytest.mark.parametrize("batch", [2, 3, 4, 5, 6, 8, 11, 12, 13, 33])
def test_tiles_and_groups(group, batch):
    check(4, group, 300, 1000, batch)


@pytest.mark.parametrize("group", [32, 64])
def test_one_block(group):
    check(4, group, 257, 33, 5)


@pytest.mark.parametrize("group", [64, 128, 1024])
def test_largest_sums(group):
    """Every activation and centroid of a group at the end of its range and of one sign: the largest sums."""
    rows, dim = 40, 1024
    packed, norms, cb, dense = example(4, rows=rows, dim=dim, group=group, seed=group)
    packed[:] = 0xFF  # the largest code everywhere
    x = np.zeros((4, dim), np.float32)
    x[:, 0::group] = 1.0  # a constant row after the transform: every quantised activation is 127
    x[1] *= -3
    x[2, 0::group] = np.linspace(1, 2, dim // group)
    q = CQMatrix(packed, norms, dense.shape, 4, group, cb)
    np.testing.assert_array_equal(q.matvec_int8(x), oracle.sdot_linear(packed, norms, dense.shape, 4, group, cb, x))
