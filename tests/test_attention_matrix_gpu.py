"""Decode attention on the int8 matrix instructions (attn_mfma_kernel): 1 (rows of 128), 2, 4 and 8 query heads per kv
head, at the edges of its 16- and 64-slot tiles, with slot lists, imported scales of either sign and non-finite input.

Tolerance: outputs are sums of at most `length` products of values of order 1 in fp32 with splits that keep 26 bits
below the largest term: atol=1e-6 + rtol=1e-5 against the fp64 closed form, as the vector kernel is held to.
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
    are untouched. Queries of any magnitude split without loss."""
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
