"""The FP32 batch GEMV (cq_batch.h): several activation rows per pass over the codes, products on the matrix cores.

Bit-identical to the oracle at every tile height (2, 3, 4, 6, 8 rows, a last tile of fewer) with the K walk in one part
and in four (forced: test_every_tile_and_part), and in the launches that sizes pick, for groups below, equal to and
above one block of 64 positions, odd widths and rows, raw (up to 512 wide) and transformed inputs.
"""
import numpy as np
import pytest

import oracle
from openneedle_amd.cq import CQMatrix, Plan
from openneedle_amd.device import DeviceArray, Graph, Stream, synchronize
from tests.cases import activations, example

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits", [2, 4])
@pytest.mark.parametrize("group", [8, 16, 32, 64, 128, 256, 512])
@pytest.mark.parametrize("nb,parts", [(nb, ks) for nb in (2, 3, 4, 6, 8) for ks in (1, 4)])
def test_every_tile_and_part(bits, group, nb, parts, monkeypatch):
    """Every kernel, on batches of exactly one tile and of two with a last row alone, raw and transformed."""
    if group < 32 and (parts == 4 or nb in (3, 6)):
        pytest.skip("groups of 8 and 16 have tiles of 2, 4 and 8 rows in one part")
    monkeypatch.setenv("NEEDLE2_GPU_FP32_BATCH", f"{nb},{parts}")
    for dim in (2100, 500) if group <= 64 else (2100,):
        packed, norms, cb, dense = example(bits, rows=270, dim=dim, group=group, seed=group + nb + dim)
        q = CQMatrix(packed, norms, dense.shape, bits, group, cb)
        for batch in (nb, 2 * nb + 1):
            x = activations((batch, dim), seed=batch)
            expected = oracle.cq_linear(packed, norms, dense.shape, bits, group, cb, x, 4)
            np.testing.assert_array_equal(q.matvec(x), expected)


@pytest.mark.parametrize("group", [128, 256])
def test_two_rows_of_many_tiles(group):
    """Two 4-bit rows over 33 row tiles of 2100 columns, which take the batch kernel by themselves."""
    packed, norms, cb, dense = example(4, rows=8200, dim=2100, group=group, seed=group)
    x = activations((2, 2100), seed=3)
    q = CQMatrix(packed, norms, dense.shape, 4, group, cb)
    np.testing.assert_array_equal(q.matvec(x), oracle.cq_linear(packed, norms, dense.shape, 4, group, cb, x, 8))


@pytest.mark.parametrize("bits", [2, 3, 4])
@pytest.mark.parametrize("group", [8, 32, 64, 128, 512])
@pytest.mark.parametrize("rows,dim,batch", [
    (257, 1100, 2), (257, 1100, 3), (300, 2100, 7), (300, 513, 9),  # few tiles: four parts, low tiles
    (64, 100, 6),                                                  # a row of few groups: one part
    (1, 300, 2500), (520, 70, 1501),                               # many tiles: high ones, a short last one
])
def test_batch_tiles_and_parts(bits, group, rows, dim, batch):
    packed, norms, cb, dense = example(bits, rows=rows, dim=dim, group=group, seed=group + rows + batch)
    x = activations((batch, dim), seed=batch)
    expected = oracle.cq_linear(packed, norms, dense.shape, bits, group, cb, x, 4)
    q = CQMatrix(packed, norms, dense.shape, bits, group, cb)
    np.testing.assert_array_equal(q.matvec(x), expected)


def test_batch_plan_of_several_matrices():
    """A plan's matrices of different row counts in one launch, each with its own input."""
    made = [example(4, rows=r, dim=600, group=32, seed=r) for r in (33, 256, 700)]
    xs = [activations((5, 600), seed=k) for k in range(3)]
    d_x = [DeviceArray.from_host(x) for x in xs]
    d_y = [DeviceArray(4 * 5 * m[3].shape[0]) for m in made]
    mats = [CQMatrix(p, n, d.shape, 4, 32, cb) for p, n, cb, d in made]
    plan = Plan(mats, [d.ptr for d in d_x], [d.ptr for d in d_y], batch=5)
    plan.run()
    synchronize()
    for (p, n, cb, d), x, y in zip(made, xs, d_y):
        expected = oracle.cq_linear(p, n, d.shape, 4, 32, cb, x, 4)
        np.testing.assert_array_equal(y.download(np.empty(expected.shape, np.float32)), expected)


def test_batch_special_values():
    """Products that underflow to denormals or zero of either sign, infinities and NaN come out as the reference's
    separately rounded products and sums do."""
    packed, norms, cb, dense = example(4, rows=300, dim=512, group=64, seed=3)
    x = activations((6, 512), seed=4)
    x[0] *= 1e-38
    x[1] *= 1e-44
    x[2, ::2] = 0.0
    x[2, 1::2] *= -1e-40
    x[3] = -0.0
    x[4, 7] = np.inf
    x[5, 9] = np.nan
    expected = oracle.cq_linear(packed, norms, dense.shape, 4, 64, cb, x, 4)
    q = CQMatrix(packed, norms, dense.shape, 4, 64, cb)
    got = q.matvec(x)
    np.testing.assert_array_equal(got, expected)


@pytest.mark.parametrize("bits,group", [(4, 128), (2, 256)])
def test_one_handle_on_two_streams(bits, group):
    """Groups of 128 and 256 use no scratch of the handle on a caller's stream: products of different inputs enqueued on
    two streams, whose work may overlap, do not disturb each other, and neither does one on the handle's own."""
    packed, norms, cb, dense = example(bits, rows=3000, dim=4000, group=group, seed=group)
    q = CQMatrix(packed, norms, dense.shape, bits, group, cb)
    xs = [activations((4, 4000), seed=k) for k in range(3)]
    want = [oracle.cq_linear(packed, norms, dense.shape, bits, group, cb, x, 8) for x in xs]
    streams = [Stream(), Stream(), None]  # None: the handle's stream
    d_x = [DeviceArray.from_host(x) for x in xs]
    d_y = [[DeviceArray(want[0].nbytes) for _ in range(20)] for _ in streams]
    for n in range(20):
        for k, s in enumerate(streams):
            q.matvec_device(d_x[k].ptr, d_y[k][n].ptr, 4, s)
    synchronize()
    for k, w in enumerate(want):
        for y in d_y[k]:
            np.testing.assert_array_equal(y.to_host(np.float32, w.shape), w)


@pytest.mark.parametrize("group", [128, 256])
def test_first_call_in_a_capture(group):
    """A handle's first product may be captured: nothing is allocated for groups of 128 and 256."""
    packed, norms, cb, dense = example(4, rows=300, dim=1100, group=group, seed=group)
    warm, q = [CQMatrix(packed, norms, dense.shape, 4, group, cb) for _ in range(2)]
    x = activations((4, 1100), seed=8)
    want = oracle.cq_linear(packed, norms, dense.shape, 4, group, cb, x, 4)
    d_x, d_y, s = DeviceArray.from_host(np.zeros_like(x)), DeviceArray(want.nbytes), Stream()
    warm.matvec_device(d_x.ptr, d_y.ptr, 4, s)  # loads the kernel
    s.synchronize()
    with Graph.capture(s) as graph:
        q.matvec_device(d_x.ptr, d_y.ptr, 4, s)
    for scale in (1, 2, 4):
        d_x.upload(x * np.float32(scale))
        graph.launch(s)
        s.synchronize()
        np.testing.assert_array_equal(d_y.to_host(np.float32, want.shape), want * np.float32(scale))


@pytest.mark.parametrize("group", [32, 128])
def test_more_rows_than_a_grid_holds(group):
    """70001 rows: past the 65535 blocks of a grid's y, the one-row kernels in one launch (groups up to 64: rows in
    pairs, the last alone)."""
    packed, norms, cb, dense = example(4, rows=3, dim=128, group=group, seed=group)
    x = activations((70001, 128), seed=1)
    q = CQMatrix(packed, norms, dense.shape, 4, group, cb)
    np.testing.assert_array_equal(q.matvec(x), oracle.cq_linear(packed, norms, dense.shape, 4, group, cb, x, 8))
