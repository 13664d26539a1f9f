"""Neighbour-search parity: the device entry tree (Morton sort + implicit tree) against the
oracle's brute-force O(n^2) search under the (distance, index) rule, bit-exact indices and
distances.  Stands in for PrefixAccelStruct + __intersection__prefix_entry
(src/PrefixAccelStruct.cpp:66-221, shader/prefix_search_hit.cu:9-73)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def make_entries(n, seed):
    rng = np.random.default_rng(seed)
    centers = rng.random((16, 3)) * 10
    pos = centers[rng.integers(0, 16, n)] + rng.normal(scale=0.6, size=(n, 3))
    radius = rng.uniform(0.05, 0.5, n)
    valid = (rng.random(n) < 0.8).astype(np.uint8)
    q = pos[rng.integers(0, n, n // 2)] + rng.normal(scale=0.2, size=(n // 2, 3))
    return pos.astype(np.float32), radius.astype(np.float32), valid, q.astype(np.float32)


@pytest.mark.parametrize("k", [1, 8, 31])
def test_neighbor_sets_bit_exact(k, orc, cx_runtime, cx_ctx):
    pos, radius, valid, q = make_entries(6000, seed=k)
    io, do, co = orc.entries_query(pos, radius, valid, q, k, brute=True)
    E = cx_runtime.Entries(cx_ctx, pos.shape[0])
    E.build(pos, radius, valid, pos.min(0), pos.max(0))
    ig, dg, cg = E.query(q, k)
    print(f"k={k}: mean neighbours {co.mean():.2f}, full {np.mean(co == k):.2f}")
    assert np.array_equal(co, cg)
    for j in range(q.shape[0]):
        c = co[j]
        assert np.array_equal(io[j, :c], ig[j, :c]), j
        assert np.array_equal(do[j, :c].view(np.uint32), dg[j, :c].view(np.uint32)), j


def test_large_set_scan_spans_several_chunks(orc, cx_runtime, cx_ctx):
    """3 M entry slots, 80 % valid: every pass of the radix sort has more than 2048 tiles of 1024
    keys, so its per-digit scan carries across several block-wide chunks.  The oracle's grid
    search (pinned against brute force in test_oracle_knn.py) gives the expected sets."""
    pos, radius, valid, q = make_entries(3_000_000, seed=5)
    q = q[:4000]
    assert int(valid.sum()) > 2048 * 1024
    io, do, co = orc.entries_query(pos, radius, valid, q, 8, brute=False)
    E = cx_runtime.Entries(cx_ctx, pos.shape[0])
    E.build(pos, radius, valid, pos.min(0), pos.max(0))
    ig, dg, cg = E.query(q, 8)
    print(f"3 M entries: mean neighbours {co.mean():.2f}, full {np.mean(co == 8):.3f}")
    assert co.mean() > 7.5
    assert np.array_equal(co, cg)
    for j in range(q.shape[0]):
        c = co[j]
        assert np.array_equal(io[j, :c], ig[j, :c]), j
        assert np.array_equal(do[j, :c].view(np.uint32), dg[j, :c].view(np.uint32)), j


def test_empty_and_all_invalid(cx_runtime, cx_ctx):
    pos = np.zeros((10, 3), np.float32)
    E = cx_runtime.Entries(cx_ctx, 10)
    E.build(pos, np.ones(10, np.float32), np.zeros(10, np.uint8), np.zeros(3), np.ones(3))
    _, _, c = E.query(np.zeros((5, 3), np.float32), 4)
    assert (c == 0).all()


@pytest.mark.parametrize("n", [1, 8, 9, 17, 2048, 2049, 4097, 300_000])
@pytest.mark.parametrize("k", [1, 7, 8, 9, 31])
def test_sizes_ties_and_extremes(n, k, orc, cx_runtime, cx_ctx):
    """Entry counts at the edges of a leaf, of the range tree's levels per launch (2048 entries are
    256 groups) and of the kernel's k; ties (equal positions, queries on entries: distance zero),
    distances whose squares underflow, infinite, zero, negative and NaN radii, non-finite queries.
    Slots beyond a query's count hold the index 0xFFFFFFFF and the distance 0."""
    pos, radius, _, q = make_entries(max(n, 64), seed=n + k)
    pos, radius, q = pos[:n], radius[:n], np.resize(q, (256, 3))
    rng = np.random.default_rng(n * 100 + k)
    same = rng.integers(0, n, n // 4)
    pos[rng.integers(0, n, n // 4)] = pos[same]                          # ties by index
    near = rng.integers(0, n, n // 8)
    pos[near] = (rng.choice([0.0, 1e-20, 3e-23, 1e-30, 1e-38], (len(near), 3))).astype(np.float32)
    radius[rng.integers(0, n, n // 10)] = np.inf
    radius[rng.integers(0, n, n // 10)] = 0.0
    radius[rng.integers(0, n, n // 10)] = 1e-22
    radius[rng.integers(0, n, n // 20)] = -1.0
    radius[rng.integers(0, n, n // 20)] = np.nan
    q[:64] = pos[rng.integers(0, n, 64)]
    q[64:96] = rng.choice([0.0, 1e-20, 2e-23, 1e-38], (32, 3))
    q[96:104] = np.array([1e30, -1e25, 1e19])
    q[104] = np.inf
    q[105] = np.nan
    valid = np.ones(n, np.uint8)
    # a NaN radius or query is no candidate on the device; the oracle is asked without them
    io, do, co = orc.entries_query(pos, np.nan_to_num(radius, nan=0.0, posinf=np.inf),
                                   (~np.isnan(radius)).astype(np.uint8), np.nan_to_num(q, posinf=np.inf), k, brute=True)
    co[np.isnan(q).any(1)] = 0
    E = cx_runtime.Entries(cx_ctx, n)
    E.build(pos, radius, valid, pos.min(0), pos.max(0))
    ig, dg, cg = E.query(q, k)
    assert np.array_equal(co, cg), np.nonzero(co != cg)
    held = np.arange(k)[None, :] < co[:, None]
    assert np.array_equal(io[held], ig[held])
    assert np.array_equal(do[held].view(np.uint32), dg[held].view(np.uint32))
    assert np.all(ig[~held] == 0xFFFFFFFF) and np.all(dg[~held].view(np.uint32) == 0)


@pytest.mark.parametrize("k", [8, 31])
def test_entries_without_a_reach_are_left_out_by_node(k, cx_runtime, cx_ctx):
    """Entries of negative, NaN or -inf radius are no candidates, and a query does not visit them one
    by one: with no other entries it finds nothing, in no more time than it takes to find its k among
    entries of a usual radius (it took 3 to 250 times as long where a square lost the radius's sign)."""
    import time
    n = 100_000
    pos, radius, _, q = make_entries(n, seed=3)
    q = np.resize(q, (40_000, 3))
    E = cx_runtime.Entries(cx_ctx, n)

    def best(radius):
        E.build(pos, radius, np.ones(n, np.uint8), pos.min(0), pos.max(0))
        t = []
        for _ in range(5):
            t0 = time.perf_counter()
            count = E.query(q, k)[2]
            t.append(time.perf_counter() - t0)
        return min(t), count

    plain, count = best(radius)
    assert count.any()
    for r in (-1.0, -np.inf, np.nan):
        took, count = best(np.full(n, r, np.float32))
        print(f"k {k} radius {r}: {took * 1e3:.2f} ms against {plain * 1e3:.2f}", flush=True)
        assert not count.any()
        assert took < 1.5 * plain + 1e-3
