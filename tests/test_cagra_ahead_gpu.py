"""GPU: graph search of small batches (rows gathered for several parents at a
time) against the search of large ones.

A query's result does not depend on the batch it is in (its position apart,
which picks the hashed seeds), so the first queries of a batch large enough
for one parent at a time must give the same ids, distances, evaluation and
iteration counts, bit for bit, as the same queries in a
batch of their own.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BIG = 513  # queries (x teams) from which the search takes one parent at a time


def graph_of(rng, oracle, base, degree, kind):
    n = len(base)
    if kind == "knn":
        return oracle.knn_graph(base, degree, threads=16)
    g = rng.integers(0, n, (n, degree), dtype=np.uint32)
    if kind == "holes":  # empty and out-of-range slots, repeated neighbours
        g[rng.random(g.shape) < 0.2] = 0xFFFFFFFF
        g[rng.random(g.shape) < 0.02] = n
        g[:, 1] = g[:, 0]
    return g


def search(ctx, cvs, idx, qs, k, knobs):
    q = len(qs)
    nbr, dist = cvs.DeviceArray(ctx, (q, k), np.uint32), cvs.DeviceArray(ctx, (q, k), np.float32)
    st = cvs.DeviceArray(ctx, (q, 2), np.uint32)
    queries = cvs.DeviceArray.from_host(ctx, qs)
    idx.search_async(queries, k, nbr, dist, stats=st, **knobs)
    ctx.synchronize()
    return nbr.to_host(), dist.to_host(), st.to_host()


@pytest.mark.parametrize("n,d,degree,kind,itopk,width,iters", [
    (3000, 128, 64, "knn", 64, 1, 0),
    (3000, 100, 33, "knn", 512, 1, 0),
    (2049, 64, 16, "random", 65, 3, 0),
    (1000, 257, 64, "holes", 128, 8, 0),
    (40, 24, 8, "random", 200, 2, 0),        # fewer rows than list entries
    (5000, 1024, 64, "knn", 10, 1, 0),       # a list shorter than the parents gathered ahead
    (3000, 128, 32, "random", 300, 4, 7),    # cut off by max_iterations
    (1, 16, 1, "random", 32, 1, 0),
    # Narrow iterations, part-filled chunks, too few rows, cut off, with lists
    # long enough for the kernel.
    (2049, 64, 48, "random", 65, 8, 0),
    (2049, 64, 33, "holes", 192, 3, 0),
    (3000, 100, 32, "knn", 256, 2, 0),
    (40, 24, 33, "random", 512, 2, 0),
    (3000, 128, 64, "random", 300, 4, 7),
    (1, 16, 1, "random", 512, 1, 0),
    # Hundreds of new keys in one step, again and again: the pool's buffer has
    # to hold up to 999 keys.  Every list length; wide steps and runs of single
    # parents.
    (20000, 32, 64, "random", 64, 8, 0),
    (20000, 32, 64, "random", 128, 4, 0),
    (20000, 32, 64, "random", 256, 1, 0),
    (20000, 32, 64, "random", 256, 8, 0),
    (20000, 32, 64, "random", 512, 1, 0),
    (20000, 32, 64, "random", 512, 8, 0),
    (20000, 32, 64, "knn", 128, 4, 0),
    (20000, 32, 64, "knn", 512, 1, 0),
])
@pytest.mark.parametrize("bits", [32, 16])
def test_small_batches_equal_large(ctx, cvs, oracle, n, d, degree, kind, itopk, width, iters, bits):
    rng = np.random.default_rng(n + d + degree + itopk)
    centres = rng.standard_normal((8, d)).astype(np.float32)
    base = centres[rng.integers(0, 8, n)] + 0.4 * rng.standard_normal((n, d)).astype(np.float32)
    base = np.rint(base * 8) / 8  # equal distances are common
    qs = centres[rng.integers(0, 8, BIG)] + 0.4 * rng.standard_normal((BIG, d)).astype(np.float32)
    graph = graph_of(rng, oracle, base, degree, kind) if n > degree else np.zeros((n, degree), np.uint32)
    k = min(itopk, 10)
    knobs = dict(itopk_size=itopk, search_width=width, max_iterations=iters)
    idx = ctx.cagra_index(base, graph, cvs.cagra_nav_nodes(n), traversal_bits=bits)
    try:
        ref = search(ctx, cvs, idx, qs, k, knobs)
        for q in (1, 128, 129):  # eight and four waves per query
            for got, want, what in zip(search(ctx, cvs, idx, qs[:q], k, knobs), ref, ("ids", "distances", "stats")):
                np.testing.assert_array_equal(got, want[:q], err_msg=f"{what}, batch of {q}")
    finally:
        idx.close()


@pytest.mark.parametrize("n,itopk,width", [(262_144, 512, 1), (262_144, 512, 8), (262_144, 65, 2)])
@pytest.mark.parametrize("bits", [32, 16])
def test_most_rows(ctx, cvs, n, itopk, width, bits):
    """The largest visited set of the small-batch kernel (with the longest list
    and fp16 traversal, more than 64 KiB of LDS) against the same search with
    its evaluations recorded, which takes one parent at a time."""
    rng = np.random.default_rng(itopk + width)
    base = rng.integers(-20, 21, (n, 16)).astype(np.float32)
    qs = rng.integers(-20, 21, (3, 16)).astype(np.float32)
    graph = rng.integers(0, n, (n, 64), dtype=np.uint32)
    idx = ctx.cagra_index(base, graph, cvs.cagra_nav_nodes(n), traversal_bits=bits)
    try:
        got = search(ctx, cvs, idx, qs, 10, dict(itopk_size=itopk, search_width=width))
        nbr, dist = cvs.DeviceArray(ctx, (3, 10), np.uint32), cvs.DeviceArray(ctx, (3, 10), np.float32)
        st, rec = cvs.DeviceArray(ctx, (3, 2), np.uint32), cvs.DeviceArray(ctx, (3, 64), np.uint32)
        idx.search_record_async(cvs.DeviceArray.from_host(ctx, qs), 10, nbr, dist, st, rec, itopk_size=itopk,
                                search_width=width)
        ctx.synchronize()
        for g, want, what in zip(got, (nbr, dist, st), ("ids", "distances", "stats")):
            np.testing.assert_array_equal(g, want.to_host(), err_msg=what)
    finally:
        idx.close()
