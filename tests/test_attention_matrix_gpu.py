"""Decode attention on the int8 matrix instructions (attn_mfma_kernel): 1 (rows of 128), 2, 4 and 8 query heads per kv
head, at the edges of its 16- and 64-slot tiles, with slot lists, imported scales of either sign, uneven queries and
weights and non-finite input.

Tolerance: outputs are sums of at most `length` products of values of order 1, each operand held to fp32's relative
precision: atol=1e-6 + rtol=1e-5 against the fp64 closed form, as the vector kernel is held to.
"""
import numpy as np
import pytest

from openneedle_amd.kv import KVCache
from tests.test_attention_gpu import ATOL, RTOL, fp64_attention, make_cache, run_attention

pytestmark = pytest.mark.gpu

SHAPES = [(1, 128), (2, 32), (4, 32), (8, 32), (2, 64), (4, 64), (8, 64), (2, 128), (4, 128), (8, 128)]


def cache(group, hd, seqs=2, cap=700, kvh=2, seed=0, sign=False):
    rng = np.random.default_rng(group * 1000 + hd + seed)
    _, _, rows = make_cache(rng, seqs, cap, kvh, hd)
    kv = KVCache(1, cap, kvh, hd, seqs)
    out = []
    for s, ((k8, ks), (v8, vs)) in enumerate(rows):
        if sign:
            ks, vs = ks.copy(), vs.copy()
            ks[::3] *= -1
            vs[::2] *= -1
        kv.load(0, s, k8, v8, ks, vs)
        out.append((k8, v8, ks, vs))
    return rng, kv, out, rng.normal(size=(seqs, kvh * group, hd)).astype(np.float32)


@pytest.mark.parametrize("group,hd", SHAPES)
@pytest.mark.parametrize("length", [1, 15, 16, 17, 63, 64, 65, 256, 257, 600])
def test_tile_edges(group, hd, length):
    _, kv, rows, q = cache(group, hd)
    for splits in (0, 1, 2):
        got = run_attention(kv, q, length, splits=splits)
        for s, r in enumerate(rows):
            np.testing.assert_allclose(got[s], fp64_attention(q[s], *r, np.arange(length)), atol=ATOL, rtol=RTOL)


@pytest.mark.parametrize("group,hd", SHAPES)
def test_slot_list_and_signed_scales(group, hd):
    rng, kv, rows, q = cache(group, hd, sign=True)
    slots = rng.permutation(700)[:333].astype(np.int32)
    listed = slots.copy()
    listed[::7] = np.where(np.arange(len(listed[::7])) % 2, -1, 700)  # outside the cache: skipped
    live = listed[(listed >= 0) & (listed < 700)]
    got = run_attention(kv, q, len(listed), slots=np.tile(listed, (1, 1))[0])
    for s, r in enumerate(rows):
        np.testing.assert_allclose(got[s], fp64_attention(q[s], *r, live), atol=ATOL, rtol=RTOL)


@pytest.mark.parametrize("group,hd", [(4, 64), (8, 128), (2, 32)])
def test_non_finite_and_small_queries(group, hd):
    """A head with an infinity or NaN in its query has no softmax (its sum is NaN) and yields zeros; the other heads
    are untouched. Heads of any magnitude keep their precision."""
    _, kv, rows, q = cache(group, hd)
    q[0, 0, 3] = np.nan
    q[1, 1, 5] = np.inf
    q[0, 1] *= 1e-30
    q[1, 0] = 0
    got = run_attention(kv, q, 300)
    assert not got[0, 0].any() and not got[1, 1].any()
    for s, r in enumerate(rows):
        keep = [h for h in range(q.shape[1]) if np.isfinite(q[s, h]).all()]
        want = fp64_attention(np.where(np.isfinite(q[s]), q[s], 0), *r, np.arange(300))
        np.testing.assert_allclose(got[s, keep], want[keep], atol=ATOL, rtol=RTOL)


def test_tiny_and_non_finite_values():
    """V rows of tiny magnitude keep their relative precision; an infinite V scale reaches its kv head's outputs only."""
    _, kv, rows, q = cache(4, 64)
    k8, v8, ks, vs = rows[0]
    tiny = (vs * np.float32(1e-33)).astype(np.float32)
    kv.load(0, 0, k8, v8, ks, tiny)
    got = run_attention(kv, q, 500)
    want = fp64_attention(q[0], k8, v8, ks, tiny, np.arange(500))
    np.testing.assert_allclose(got[0], want, atol=1e-39, rtol=1e-4)
    bad = vs.copy()
    bad[7, 1] = np.inf
    kv.load(0, 0, k8, v8, ks, bad)
    got = run_attention(kv, q, 500)
    assert np.isfinite(got[0, :4]).all() and not np.isfinite(got[0, 4:]).any()


@pytest.mark.parametrize("group,hd", SHAPES)
@pytest.mark.parametrize("ratio", [1e4, 1e6, 1e8, 1e12, 1e30])
def test_uneven_queries(group, hd, ratio):
    """A query entry far above the rest (past the 2^36 that two digit groups cover from 1e12 on) over zero K codes:
    the other entries' products decide, at their own precision."""
    _, kv, rows, q = cache(group, hd)
    q[:, ::2, 5] = ratio
    out = []
    for s, (k8, v8, ks, vs) in enumerate(rows):
        k8 = k8.copy()
        k8[:, :, 5] = 0
        kv.load(0, s, k8, v8, ks, vs)
        out.append((k8, v8, ks, vs))
    for splits in (1, 2):
        got = run_attention(kv, q, 300, splits=splits)
        for s, r in enumerate(out):
            np.testing.assert_allclose(got[s], fp64_attention(q[s], *r, np.arange(300)), atol=ATOL, rtol=RTOL)
    listed = np.arange(299, -1, -1).astype(np.int32)
    got = run_attention(kv, q, 300, slots=listed)
    for s, r in enumerate(out):
        np.testing.assert_allclose(got[s], fp64_attention(q[s], *r, listed), atol=ATOL, rtol=RTOL)


@pytest.mark.parametrize("group,hd", SHAPES)
@pytest.mark.parametrize("margin", [10, 18, 30, 60])
def test_dominant_slot(group, hd, margin):
    """One slot whose score is `margin` above the rest, with zero V codes in half of the dimensions: there the outputs
    are the other slots' sums, all of one sign, each weight to fp32's relative precision (up to `margin` = 60 the
    weights lie 2^-87 below the largest). A score of size S carries three roundings, so a weight is good to
    3 S 2^-24: rtol 2e-5 at S = 66 + the sums'."""
    rng, kv, rows, q = cache(group, hd)
    sign = rng.choice([-1, 1], hd)
    q = (np.abs(q) * sign).astype(np.float32)
    out = []
    for s, (k8, v8, ks, vs) in enumerate(rows):
        k8, v8, ks = k8.copy(), v8.copy(), ks.copy()
        ks /= 4
        v8[:, :, ::2] = np.maximum(np.abs(v8[:, :, ::2]), 1)
        k8[77] = 127 * sign
        v8[77, :, ::2] = 0
        ks[77] = margin * np.sqrt(hd) / (127 * np.abs(q[s]).sum(axis=-1).mean())
        kv.load(0, s, k8, v8, ks, vs)
        out.append((k8, v8, ks, vs))
    for splits in (1, 2):
        got = run_attention(kv, q, 300, splits=splits)
        for s, r in enumerate(out):
            want = fp64_attention(q[s], *r, np.arange(300))
            np.testing.assert_allclose(got[s], want, atol=ATOL, rtol=RTOL)
            np.testing.assert_allclose(got[s][:, ::2], want[:, ::2], atol=1e-37, rtol=2e-5)


@pytest.mark.parametrize("group,hd", [(4, 64), (8, 128), (2, 32), (1, 128)])
def test_infinite_value_scale(group, hd):
    """An infinite V scale: infinities of the codes' signs, NaN for a zero code, as the products give."""
    _, kv, rows, q = cache(group, hd)
    k8, v8, ks, vs = rows[0]
    v8, vs = v8.copy(), vs.copy()
    v8[41, 1, 3] = 0
    vs[41, 1] = np.inf
    kv.load(0, 0, k8, v8, ks, vs)
    for splits in (1, 2):
        got = run_attention(kv, q, 400, splits=splits)[0]
        want = np.where(v8[41, 1] == 0, np.nan, np.where(v8[41, 1] > 0, np.inf, -np.inf))
        assert np.isfinite(got[:group]).all()
        for h in range(group, 2 * group):
            np.testing.assert_array_equal(got[h], want)


def test_tiny_value_scales():
    """Weights down to fp32's smallest normal numbers keep their precision (products of 127 are normal)."""
    _, kv, rows, q = cache(4, 64)
    k8, v8, ks, vs = rows[0]
    tiny = (vs * np.float32(2.0 ** -110)).astype(np.float32)
    kv.load(0, 0, k8, v8, ks, tiny)
    got = run_attention(kv, q, 1)
    np.testing.assert_allclose(got[0], fp64_attention(q[0], k8, v8, ks, tiny, np.arange(1)), atol=1e-44, rtol=1e-6)
