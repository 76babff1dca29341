"""GPU parity of the fused brute-force path (C ABI: cvs_bf_search) against the
oracle and the reference's golden outputs.

Gate (stated by the target): top-k id sets equal to the reference's except
where the k-th and (k+1)-th reference distances are within 1e-3 relative;
distances within 1e-3 relative.  Integer-valued inputs must match exactly.
"""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(__file__), "golden")
REL_TOL = 1e-3


def assert_parity(nbr, dist, ref_nbr, ref_dist_k1, k):
    """ref_dist_k1: reference distances for k+1 results (sorted)."""
    q = nbr.shape[0]
    ref_dist = ref_dist_k1[:, :k]
    finite = np.isfinite(ref_dist)
    np.testing.assert_array_equal(np.isfinite(dist), finite)
    scale = np.maximum(np.abs(ref_dist), 1e-30)
    err = np.where(finite, np.abs(dist - ref_dist) / scale, 0)
    assert err.max() <= REL_TOL, f"distance error {err.max()}"
    for i in range(q):
        dk = ref_dist_k1[i, k - 1]
        dk1 = ref_dist_k1[i, k] if ref_dist_k1.shape[1] > k else np.inf
        near_tie = np.isfinite(dk1) and abs(dk1 - dk) <= REL_TOL * max(abs(dk), 1e-30)
        if not near_tie:
            assert set(nbr[i].tolist()) == set(ref_nbr[i, :k].tolist()), f"query {i}"
    # rows sorted by (distance, id)
    for i in range(q):
        for j in range(1, k):
            assert dist[i, j - 1] < dist[i, j] or (dist[i, j - 1] == dist[i, j] and nbr[i, j - 1] < nbr[i, j]) \
                or not np.isfinite(dist[i, j])


def check_against_oracle(ctx, oracle, base, queries, k, threads=8):
    ds = ctx.dataset(base)
    nbr, dist = ds.bf_search(queries, k)
    ref_nbr, ref_dist = oracle.bf_exact(base, queries, k + 1, threads=threads)
    assert_parity(nbr, dist, ref_nbr, ref_dist, k)
    return nbr, dist


def test_faiss_known_answers(ctx):
    db = np.array([[0, 0], [10, 0], [0, 10], [2, 2]], np.float32)
    qs = np.array([[0, 0], [9, 1]], np.float32)
    ds = ctx.dataset(db)
    nbr, dist = ds.bf_search(qs, 2)
    assert nbr.tolist() == [[0, 3], [1, 3]]
    assert dist.tolist() == [[0.0, 8.0], [2.0, 50.0]]
    nbr, dist = ds.bf_search(qs[:1], 4)
    assert nbr.tolist() == [[0, 3, 1, 2]] and dist.tolist() == [[0.0, 8.0, 100.0, 100.0]]
    nbr, dist = ds.bf_search(qs, 5)
    assert nbr[:, 4].tolist() == [0xFFFFFFFF] * 2 and np.isinf(dist[:, 4]).all()
    assert nbr[:, :4].tolist() == [[0, 3, 1, 2], [1, 3, 0, 2]]


def test_dispatch_test_inputs_run_on_gpu(ctx, cvs):
    base = np.zeros((64, 8), np.float32)
    for i in range(64):
        base[i, i % 8] = i
    qs = np.zeros((4, 8), np.float32)
    for j in range(4):
        qs[j, j % 8] = 1
    ds = ctx.dataset(base)
    cvs.reset_dispatch_count()
    nbr, dist = ds.bf_search(qs, 4)
    assert cvs.dispatch_count() > 0
    assert nbr.tolist() == [[0, 1, 2, 3], [1, 0, 2, 3], [0, 2, 1, 3], [0, 1, 3, 2]]
    assert dist.tolist() == [[1, 2, 5, 10], [0, 1, 5, 10], [1, 1, 2, 10], [1, 2, 4, 5]]


@pytest.mark.parametrize("name", ["random", "ties", "kbig", "wide"])
def test_reference_golden(ctx, oracle, name):
    g = np.load(os.path.join(GOLDEN, "bf_ref.npz"))
    base, qs, k = g[f"{name}_base"], g[f"{name}_queries"], int(g[f"{name}_k"])
    nbr, dist = ctx.dataset(base).bf_search(qs, k)
    if name in ("ties", "kbig"):
        if name == "ties":  # integer data: every quantity is exact
            np.testing.assert_array_equal(nbr, g[f"{name}_nbr"])
            np.testing.assert_array_equal(dist, g[f"{name}_dist"])
        else:
            np.testing.assert_array_equal(nbr, g[f"{name}_nbr"])
            np.testing.assert_allclose(dist, g[f"{name}_dist"], rtol=REL_TOL)
    else:
        _, ref_dist = oracle.bf_exact(base, qs, k + 1)
        assert_parity(nbr, dist, g[f"{name}_nbr"], ref_dist, k)


@pytest.mark.parametrize("n,d,q,k", [
    (1, 1, 1, 1),
    (7, 5, 3, 10),        # k > n: padded slots
    (100, 64, 130, 10),   # two query blocks
    (1000, 96, 17, 48),   # largest k of the LDS lists
    (1000, 96, 17, 49),   # smallest k of the global-memory lists (kp = 128)
    (20000, 128, 300, 100),
    (3000, 64, 40, 112),  # largest k
    (100, 32, 5, 112),    # k > n with global-memory lists
    (5000, 256, 33, 24),
    (4000, 300, 50, 10),    # 32 k-steps per tile (k-split scan, one stage per tile)
    (2500, 512, 130, 100),  # 32 k-steps, two query blocks, global-memory lists
    (6000, 384, 20, 40),
    (2000, 1024, 5, 1),
    (3333, 1000, 9, 16),  # d not a power of two
    (40000, 128, 129, 10),
])
def test_random_shapes(ctx, oracle, n, d, q, k):
    rng = np.random.default_rng(n * 31 + d)
    base = rng.standard_normal((n, d)).astype(np.float32)
    qs = rng.standard_normal((q, d)).astype(np.float32)
    check_against_oracle(ctx, oracle, base, qs, k)


@pytest.mark.parametrize("q", [1, 250, 252])
def test_blocking_calls_on_both_sides_of_the_pinned_limit(ctx, cvs, q):
    """250 queries of 1,024 columns with 10 results each fit the pinned
    staging (1 MiB), 252 do not; a refused call in between leaves nothing
    behind."""
    rng = np.random.default_rng(q)
    base = rng.integers(-6, 7, (3000, 1024)).astype(np.float32)
    qs = rng.integers(-6, 7, (q, 1024)).astype(np.float32)
    ds = ctx.dataset(base)
    with pytest.raises(ValueError):
        ds.bf_search(qs[:1], 1025)
    nbr, dist = ds.bf_search(qs, 10)
    queries = cvs.DeviceArray.from_host(ctx, qs)
    want_nbr, want_dist = cvs.DeviceArray(ctx, (q, 10), np.uint32), cvs.DeviceArray(ctx, (q, 10), np.float32)
    ds.bf_search_async(queries, 10, want_nbr, want_dist)
    ctx.synchronize()
    np.testing.assert_array_equal(nbr, want_nbr.to_host())
    np.testing.assert_array_equal(dist, want_dist.to_host())


@pytest.mark.parametrize("copies,k", [(0, 49), (300, 100), (4000, 112), (9000, 100)])
@pytest.mark.parametrize("d", [20, 128, 132, 515, 1024])
def test_merge_of_long_lists(ctx, d, copies, k):
    """kp = 128: the candidates are selected among the listed keys (equal
    distances cut by the row id), or, when more keys lie within the bound than
    the merge's buffer holds (9,000 copies of one row), from running lists.
    Whole numbers: ids and distances equal those of a sort by (distance, id).
    The dimensions cover the exact re-rank's forms: half a wave a row, one to
    four chunks of 256 columns, unaligned rows."""
    rng = np.random.default_rng(d + copies)
    n, q = 40_000, 7
    base = rng.integers(-5, 6, (n, d)).astype(np.float32)
    base[rng.choice(n, copies, replace=False)] = base[0]
    qs = np.concatenate([base[:1], rng.integers(-5, 6, (q - 1, d)).astype(np.float32)])
    nbr, dist = ctx.dataset(base).bf_search(qs, k)
    key = ((qs.astype(np.float64) ** 2).sum(1)[:, None] - 2.0 * (qs.astype(np.float64) @ base.T.astype(np.float64))
           + (base.astype(np.float64) ** 2).sum(1)[None, :]).astype(np.int64) * n + np.arange(n)[None, :]
    near = np.sort(np.partition(key, k - 1, axis=1)[:, :k], axis=1)
    np.testing.assert_array_equal(nbr, near % n)
    np.testing.assert_array_equal(dist, near // n)


@pytest.mark.parametrize("d", [65, 128, 160, 256, 320])
@pytest.mark.parametrize("n,q,k", [
    (2500, 1025, 10),    # one query past the limit; part-filled last workgroup and query tile
    (20001, 1600, 24),
    (9000, 1281, 48),
    (70, 1100, 100),     # k > n, most ranges empty
    (30000, 1030, 112),
    (40001, 1025, 10), (4100, 5201, 7), (2000, 8250, 3),  # 16-key lists: fewer rows or queries take the other scan
    (36001, 1030, 24), (2100, 6001, 20),                  # 32-key lists
    (2500, 1100, 48), (1500, 3000, 30), (1499, 1100, 48),  # 64-key lists
])
def test_narrow_large_batches(ctx, d, n, q, k):
    """The large-batch scan over 8 to 20 k-steps, every list geometry.  Rows
    in order of falling distance to the queries, so that keys keep passing and
    lists are compacted; whole numbers, so ids equal those of a sort by
    (distance, id)."""
    rng = np.random.default_rng(d + n)
    base = rng.integers(-6, 7, (n, d)).astype(np.float32)
    base[:, 0] = np.rint(np.linspace(200, 0, n))
    qs = rng.integers(-6, 7, (q, d)).astype(np.float32)
    nbr, dist = ctx.dataset(base).bf_search(qs, k)
    key = ((qs.astype(np.float64) ** 2).sum(1)[:, None] - 2.0 * (qs.astype(np.float64) @ base.T.astype(np.float64))
           + (base.astype(np.float64) ** 2).sum(1)[None, :]).astype(np.int64) * n + np.arange(n)[None, :]
    m = min(k, n)
    near = np.sort(np.partition(key, m - 1, axis=1)[:, :m], axis=1)
    np.testing.assert_array_equal(nbr[:, :m], near % n)
    np.testing.assert_array_equal(dist[:, :m], near // n)
    assert (nbr[:, m:] == 0xFFFFFFFF).all() and np.isinf(dist[:, m:]).all()


@pytest.mark.parametrize("d,q,k", [(256, 131_072, 10), (256, 65_536, 10), (128, 196_608, 24)])
def test_narrow_batches_of_many_queries(ctx, cvs, d, q, k):
    """Query counts that fill the chip with one or two ranges of the dataset:
    there have to be enough candidate lists all the same for the certificate to
    hold (with one list of 16 keys 29% of these queries at K = 10 fail it, each
    then re-ranked over every row)."""
    rng = np.random.default_rng(d + q)
    n = 20_000
    centres = rng.standard_normal((64, d)).astype(np.float32)
    def points(m):
        x = centres[rng.integers(0, 64, m)] + 0.1 * rng.standard_normal((m, d), dtype=np.float32)
        return x / np.linalg.norm(x, axis=1, keepdims=True)
    base, qs = points(n), points(q)
    ds = ctx.dataset(base)
    ctx.bf_escalations(reset=True)
    nbr, dist = ds.bf_search(qs, k)
    escalated, _ = ctx.bf_escalations(reset=True)
    assert escalated <= q // 1000
    some = rng.choice(q, 500, replace=False)
    want_nbr, want_dist = ds.bf_search(qs[some], k)  # the scan of small batches
    np.testing.assert_array_equal(nbr[some], want_nbr)
    np.testing.assert_array_equal(dist[some], want_dist)


@pytest.mark.parametrize("d,q,k", [(128, 1100, 48), (200, 1100, 25), (128, 1100, 24), (128, 2900, 48)])
def test_narrow_large_batches_with_long_lists(ctx, d, q, k):
    """Full candidate lists, 64 (the last row) to 128 a query: the nearest rows
    lie where the threshold sample does not look (it takes every third unit of
    256 rows, or 128 beyond 128 columns), so that two thirds of the rows pass its threshold.  No query may
    need an escalation for it."""
    rng = np.random.default_rng(d + q + k)
    n = 100_000
    base = rng.standard_normal((n, d), dtype=np.float32)
    base[np.arange(n) // (256 if d <= 128 else 128) % 3 == 0] *= 1.6
    qs = rng.standard_normal((q, d), dtype=np.float32)
    ds = ctx.dataset(base)
    ctx.bf_escalations(reset=True)
    nbr, dist = ds.bf_search(qs, k)
    assert ctx.bf_escalations(reset=True)[0] == 0
    want_nbr, want_dist = ds.bf_search(qs[:500], k)  # the scan of small batches
    np.testing.assert_array_equal(nbr[:500], want_nbr)
    np.testing.assert_array_equal(dist[:500], want_dist)


@pytest.mark.parametrize("q,k", [(2000, 10), (1100, 24)])
def test_narrow_large_batches_without_allocation(ctx, cvs, q, k):
    """The fixed scratch of the allocation-free call is too small for that
    scan's lists at some sizes it takes: it then runs another scan."""
    rng = np.random.default_rng(q + k)
    base = rng.integers(-6, 7, (30_000, 128)).astype(np.float32)
    qs = rng.integers(-6, 7, (q, 128)).astype(np.float32)
    ds = ctx.dataset(base)
    want_nbr, want_dist = ds.bf_search(qs, k)
    queries = cvs.DeviceArray.from_host(ctx, qs)
    nbr, dist = cvs.DeviceArray(ctx, (q, k), np.uint32), cvs.DeviceArray(ctx, (q, k), np.float32)
    ds.bf_search_noalloc(queries, k, nbr, dist)
    ctx.synchronize()
    np.testing.assert_array_equal(nbr.to_host(), want_nbr)
    np.testing.assert_array_equal(dist.to_host(), want_dist)


@pytest.mark.parametrize("d", [129, 192, 193, 320, 321, 384, 385, 448, 449, 640, 641, 768, 769, 896, 897])
@pytest.mark.parametrize("n,q,k", [
    (17000, 33, 10), (9001, 130, 24), (6002, 5, 48), (4003, 20, 100),  # one list geometry each
    (4100, 1100, 60),                                                  # the register-blocked scan
    (2000, 3, 120),                                                    # the keys-matrix path
])
def test_every_padded_dimension(ctx, d, n, q, k):
    """First and last dimension of each k-step count that is no power of two:
    whole-number rows, so that distances are exact and ids equal those of a
    sort by (distance, id)."""
    rng = np.random.default_rng(d * 7 + n)
    base = rng.integers(-8, 9, (n, d)).astype(np.float32)
    qs = rng.integers(-8, 9, (q, d)).astype(np.float32)
    nbr, dist = ctx.dataset(base).bf_search(qs, k)
    key = ((qs.astype(np.float64) ** 2).sum(1)[:, None] - 2.0 * (qs.astype(np.float64) @ base.T.astype(np.float64))
           + (base.astype(np.float64) ** 2).sum(1)[None, :]).astype(np.int64) * n + np.arange(n)[None, :]
    near = np.sort(np.partition(key, k - 1, axis=1)[:, :k], axis=1)
    np.testing.assert_array_equal(nbr, near % n)
    np.testing.assert_array_equal(dist, near // n)


@pytest.mark.parametrize("n,d,q,k", [
    (30000, 64, 1500, 10),    # > 8 query blocks: range-major launch, LDS lists
    (30000, 64, 1500, 100),   # range-major launch, global-memory lists (8 k-steps or fewer)
    (8000, 1024, 1100, 64),   # register-blocked scan (bf_gemm.hip): 3 query blocks
    (3000, 128, 2000, 100),   # 8 k-steps, one 128-row block per span
    (500, 256, 1200, 100),    # half the spans empty
    (20000, 1000, 1500, 100), # d padded to 1024
    (20000, 512, 5000, 112),  # 10 query blocks: two per XCD for XCDs 0 and 1, largest k
    (12000, 1024, 1300, 10),  # range-major pipelined scan (64 k-steps), kp = 16 LDS lists
    (12000, 512, 1100, 40),   # range-major pipelined scan (32 k-steps), kp = 64 LDS lists
    (7000, 384, 1100, 100),   # 24 k-steps
    (5000, 640, 1030, 50),    # 40 k-steps; the last 512-query block holds one 32-query tile
    (9000, 768, 1200, 112),   # 48 k-steps, largest k
    (3000, 896, 2100, 77),    # 56 k-steps, 5 query blocks
])
def test_large_batches(ctx, oracle, n, d, q, k):
    rng = np.random.default_rng(q + k)
    centers = rng.standard_normal((32, d)).astype(np.float32)
    base = centers[rng.integers(0, 32, n)] + 0.3 * rng.standard_normal((n, d)).astype(np.float32)
    qs = centers[rng.integers(0, 32, q)] + 0.3 * rng.standard_normal((q, d)).astype(np.float32)
    check_against_oracle(ctx, oracle, base, qs, k)


def test_duplicate_rows_tie_break_by_id(ctx, oracle):
    rng = np.random.default_rng(5)
    uniq = rng.standard_normal((50, 48)).astype(np.float32)
    base = np.repeat(uniq, 20, axis=0)   # every vector 20 times
    qs = uniq[:6] + 0.01 * rng.standard_normal((6, 48)).astype(np.float32)
    nbr, dist = ctx.dataset(base).bf_search(qs, 25)
    ref_nbr, ref_dist = oracle.bf_exact(base, qs, 25)
    # the 20 copies of the nearest vector come first, in id order
    np.testing.assert_array_equal(nbr[:, :20], ref_nbr[:, :20])
    np.testing.assert_allclose(dist, ref_dist, rtol=REL_TOL)


def test_c1_clustered_config(ctx, cvs, oracle):
    """N=10,000, Q=100, D=1024, K=10 on the clustered distribution."""
    base = cvs.synth_clustered(12345, cvs.STREAM_BASE, 10000, 1024)
    qs = cvs.synth_clustered(12345, cvs.STREAM_QUERIES, 100, 1024)
    check_against_oracle(ctx, oracle, base, qs, 10)


def test_async_matches_sync(ctx, cvs):
    rng = np.random.default_rng(9)
    base = rng.standard_normal((3000, 200)).astype(np.float32)
    qs = rng.standard_normal((40, 200)).astype(np.float32)
    ds = ctx.dataset(base)
    nbr, dist = ds.bf_search(qs, 10)
    dq = cvs.DeviceArray.from_host(ctx, qs)
    dn = cvs.DeviceArray(ctx, (40, 10), np.uint32)
    dd = cvs.DeviceArray(ctx, (40, 10), np.float32)
    ds.bf_search_async(dq, 10, dn, dd)
    ctx.synchronize()
    np.testing.assert_array_equal(dn.to_host(), nbr)
    np.testing.assert_array_equal(dd.to_host(), dist)
    # repeated calls reuse workspaces and give identical results
    for _ in range(3):
        ds.bf_search_async(dq, 10, dn, dd)
    ctx.synchronize()
    np.testing.assert_array_equal(dn.to_host(), nbr)


def test_dataset_from_device_rows(ctx, cvs):
    rng = np.random.default_rng(13)
    base = rng.standard_normal((500, 40)).astype(np.float32)
    qs = rng.standard_normal((3, 40)).astype(np.float32)
    a = ctx.dataset(base).bf_search(qs, 7)
    b = ctx.dataset(cvs.DeviceArray.from_host(ctx, base)).bf_search(qs, 7)
    np.testing.assert_array_equal(a[0], b[0])
    np.testing.assert_array_equal(a[1], b[1])


def test_argument_errors(ctx):
    ds = ctx.dataset(np.ones((10, 4), np.float32))
    with pytest.raises(ValueError):
        ds.bf_search(np.ones((2, 4), np.float32), 0)
    with pytest.raises(ValueError):
        ds.bf_search(np.ones((2, 4), np.float32), 1025)
    with pytest.raises(ValueError):
        ds.bf_search(np.ones((2, 5), np.float32), 3)
    with pytest.raises(ValueError):
        ctx.dataset(np.ones((10, 16385), np.float32)).bf_search(np.ones((1, 16385), np.float32), 3)
    with pytest.raises(ValueError):
        ctx.dataset(np.ones((0, 4), np.float32))


def exact_topk_numpy(base, qs, k, extra=64):
    """fp32 GEMM candidates re-scored in fp64 (ground truth at full size)."""
    cross = qs @ base.T
    norms = np.einsum("ij,ij->i", base, base)
    approx = norms[None, :] - 2 * cross
    cand = np.argpartition(approx, k + extra, axis=1)[:, :k + extra]
    out_i = np.empty((qs.shape[0], k + 1), np.int64)
    out_d = np.empty((qs.shape[0], k + 1), np.float64)
    for i in range(qs.shape[0]):
        c = cand[i]
        d = ((base[c].astype(np.float64) - qs[i].astype(np.float64)) ** 2).sum(1)
        o = np.lexsort((c, d))[:k + 1]
        out_i[i], out_d[i] = c[o], d[o]
    return out_i, out_d


def test_c3_full_size_large_batch(ctx, cvs):
    """N=1,000,000, D=1024, Q=10,000, K=100 in one call: ids and distances
    of 200 sampled queries against the exact ground truth (same gates)."""
    n, d, q, k = 1_000_000, 1024, 10_000, 100
    base = cvs.synth_clustered(12345, cvs.STREAM_BASE, n, d)
    qs = cvs.synth_clustered(12345, cvs.STREAM_QUERIES, q, d)
    nbr, dist = ctx.dataset(base).bf_search(qs, k)
    sample = np.random.default_rng(0).choice(q, 200, replace=False)
    gt_i, gt_d = exact_topk_numpy(base, qs[sample], k)
    assert_parity(nbr[sample], dist[sample], gt_i.astype(np.uint32), gt_d, k)
    recall = np.mean([len(set(nbr[s].tolist()) & set(gt_i[j, :k].tolist())) / k for j, s in enumerate(sample)])
    assert recall >= 0.999, recall


def test_c2_full_size_recall(ctx, cvs):
    """N=1,000,000, D=1024, Q=100, K=10: recall@10 = 1.0 vs exact (up to
    near-ties), distances within 1e-3."""
    n, d, q, k = 1_000_000, 1024, 100, 10
    base = cvs.synth_clustered(12345, cvs.STREAM_BASE, n, d)
    qs = cvs.synth_clustered(12345, cvs.STREAM_QUERIES, q, d)
    ds = ctx.dataset(base)
    nbr, dist = ds.bf_search(qs, k)
    gt_i, gt_d = exact_topk_numpy(base, qs, k)
    assert_parity(nbr, dist, gt_i.astype(np.uint32), gt_d, k)
    recall = np.mean([len(set(nbr[i]) & set(gt_i[i, :k])) / k for i in range(q)])
    assert recall >= 0.999
