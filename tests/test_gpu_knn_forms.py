"""The forms of the exact-kNN call (a few queries; tiles) against each other and the oracle.  All of them multiply on the
matrix cores in one order, so a query's answer has the same bits whatever batch it is in; against the oracle's float32
sums the order differs, hence the tolerance of test_knn_exact (rtol 1e-5 / atol 1e-6: a few ulp of sums below 1)."""
import numpy as np
import pytest
import torch

from oracle import oracle as orc

pytestmark = pytest.mark.gpu

DEV = "cuda"


def rows(rng, n, dim):
    v = rng.standard_normal((n, dim)).astype(np.float32)
    return v / np.linalg.norm(v, axis=1, keepdims=True)


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


# tiles of 32 vectors and 32 queries, chunk pairs of 8 columns (a lone last chunk when dim % 8 == 4), one tile per
# wavefront up to 65,536 vectors and several beyond, every list length
@pytest.mark.parametrize("n,dim,nq,k,metric", [
    (1, 4, 1, 1, "cosine"), (31, 12, 2, 16, "cosine"), (32, 8, 31, 4, "l2"), (33, 20, 32, 10, "cosine"),
    (1000, 64, 33, 16, "l2"), (4097, 68, 128, 12, "cosine"), (65_541, 16, 5, 16, "cosine"), (140_000, 36, 40, 8, "l2"),
    (70_000, 132, 1, 10, "cosine")])
def test_a_few_queries(n, dim, nq, k, metric):
    print(f"a few queries n={n} dim={dim} nq={nq} k={k} {metric}", flush=True)
    from vectorlink_gpu.kernels import knn_exact

    rng = np.random.default_rng(n + dim)
    v, q = rows(rng, n, dim), rows(rng, nq, dim)
    q[0] = v[n // 2]
    (gi, gd) = knn_exact(dev(q), dev(v), k, metric)
    # the same queries in a batch that the tiles take
    many = np.concatenate([q, rows(rng, 150, dim)])
    (ti, td) = knn_exact(dev(many), dev(v), k, metric)
    assert torch.equal(gi, ti[:nq]) and torch.equal(gd, td[:nq])
    gi, gd = gi.cpu().numpy(), gd.cpu().numpy()
    have = min(k, n)
    assert (gi[:, have:] == orc.MAXINT).all() and (gd[:, have:] == np.float32(orc.MAXFLOAT)).all()
    s = q.astype(np.float64) @ v.astype(np.float64).T
    true = np.clip((1 - s) / 2, 0, 1) if metric == "cosine" else np.maximum(
        (q.astype(np.float64) ** 2).sum(1)[:, None] + (v.astype(np.float64) ** 2).sum(1)[None] - 2 * s, 0)
    want = np.sort(true, axis=1)[:, :have]
    assert np.allclose(gd[:, :have], want, rtol=1e-5, atol=1e-6)
    assert np.allclose(np.take_along_axis(true, gi[:, :have].astype(np.int64), 1), want, rtol=1e-5, atol=2e-6)
    assert all(len(set(r)) == have for r in gi[:, :have].tolist())


@pytest.mark.parametrize("n,nq", [(3000, 3), (70_000, 2)])
def test_a_few_queries_among_equal_rows(n, nq):
    """Every row the same: all keys are as close as the best one (more than the selection's pool holds) and the ids decide."""
    print(f"equal rows n={n} nq={nq}", flush=True)
    from vectorlink_gpu.kernels import knn_exact

    rng = np.random.default_rng(n)
    v = np.repeat(rows(rng, 1, 24), n, axis=0)
    q = rows(rng, nq, 24)
    (gi, gd) = knn_exact(dev(q), dev(v), 16)
    assert np.array_equal(gi.cpu().numpy(), np.tile(np.arange(16, dtype=np.int32), (nq, 1)))
    assert all(len(set(r)) == 1 for r in gd.cpu().numpy().tolist())


# the bfloat16 filter: tiles of 256 x 256 and stages of 64 columns with remainders, an odd number of stages, three more
# columns for L2, rows of very different lengths, and more than one converted piece of the table (2 GiB of 64 columns)
@pytest.mark.parametrize("n,dim,nq,k,metric", [
    (4096, 64, 129, 10, "cosine"), (4097, 4, 256, 16, "cosine"), (5000, 60, 257, 4, "l2"), (6000, 64, 300, 1, "l2"),
    (40_000, 192, 700, 16, "cosine"), (33_000, 196, 513, 12, "l2"), (17_000_000, 4, 150, 4, "cosine")])
def test_the_filter_and_a_few_queries_agree(n, dim, nq, k, metric):
    print(f"filter n={n} dim={dim} nq={nq} k={k} {metric}", flush=True)
    from vectorlink_gpu.kernels import knn_exact

    gen = torch.Generator(device=DEV).manual_seed(n + dim)
    v = torch.randn((n, dim), generator=gen, device=DEV)
    q = torch.randn((nq, dim), generator=gen, device=DEV)
    if metric == "cosine":
        v, q = torch.nn.functional.normalize(v, dim=1), torch.nn.functional.normalize(q, dim=1)
    else:
        v *= torch.rand((n, 1), generator=gen, device=DEV) * 4
    v[n - 1] = q[nq - 1]
    v[n // 3] = v[n - 1]  # a tie that the ids decide
    (gi, gd) = knn_exact(q, v, k, metric)
    for s in range(0, nq, 32):
        (fi, fd) = knn_exact(q[s:s + 32].contiguous(), v, k, metric)
        assert torch.equal(gi[s:s + 32], fi) and torch.equal(gd[s:s + 32], fd)
    assert int(gi[nq - 1, 0]) == n // 3


@pytest.mark.parametrize("bad", ["equal rows", "an infinite row"])
def test_what_the_filter_leaves_to_the_tiles(bad):
    """More rows within the rounding of each other than a query's buffer holds, or no bound at all."""
    print(f"filter with {bad}", flush=True)
    from vectorlink_gpu.kernels import knn_exact

    rng = np.random.default_rng(8)
    v = rows(rng, 9000, 32)
    if bad == "equal rows":
        v[:5000] = v[0]
    q = rows(rng, 300, 32)
    q[:200] = v[0] + 0.01 * q[:200]
    gv = dev(v)
    if bad != "equal rows":
        gv[4321, 5] = float("inf")
    gq = dev(q)
    (gi, gd) = knn_exact(gq, gv, 10)
    for s in range(0, 300, 32):
        (fi, fd) = knn_exact(gq[s:s + 32].contiguous(), gv, 10)
        assert torch.equal(gi[s:s + 32], fi) and torch.equal(gd[s:s + 32], fd)
    if bad == "equal rows":
        assert np.array_equal(gi[:200].cpu().numpy(), np.tile(np.arange(10, dtype=np.int32), (200, 1)))


@pytest.mark.parametrize("n,dim,nq,k,metric", [(9000, 32, 300, 10, "cosine"), (40_000, 64, 130, 16, "l2"), (70_000, 16, 3, 4, "l2")])
def test_a_workspace_for_the_tiles_alone(n, dim, nq, k, metric):
    """The tiles want at most 256 lists of 16 keys a query, two words a query and one a vector; a call that brings no more
    than that is answered by them, with the same bits."""
    print(f"small workspace n={n} dim={dim} nq={nq} k={k} {metric}", flush=True)
    from vectorlink_gpu import _native as nv
    from vectorlink_gpu.kernels import knn_exact

    rng = np.random.default_rng(n)
    v, q = dev(rows(rng, n, dim)), dev(rows(rng, nq, dim))
    (wi, wd) = knn_exact(q, v, k, metric)
    most = nv.lib().vl_knn_workspace_bytes(nq, n, dim, k)
    small = nq * 256 * 16 * 8 + (2 * nq + n) * 4 + 16
    if nq > 128:
        small = min(small, most - 1)  # one byte less than the filter's
    ws = torch.empty(small, dtype=torch.uint8, device=DEV)
    ids = torch.empty((nq, k), dtype=torch.int32, device=DEV)
    d = torch.empty((nq, k), dtype=torch.float32, device=DEV)
    nv.check(nv.lib().vl_knn_exact_metric(nv.ptr(q), nq, nv.ptr(v), n, dim, k, nv.metric_code(metric), nv.ptr(ids),
                                          nv.ptr(d), nv.ptr(ws), ws.numel(), nv.stream()))
    assert torch.equal(ids, wi) and torch.equal(d, wd)


@pytest.mark.parametrize("metric", ["cosine", "l2"])
def test_more_queries_than_the_filter_takes_at_a_time(metric):
    """65,536 at a time: a second piece of 200, with its own block flags."""
    print(f"two pieces of queries {metric}", flush=True)
    from vectorlink_gpu.kernels import knn_exact

    gen = torch.Generator(device=DEV).manual_seed(4)
    v = torch.nn.functional.normalize(torch.randn((4096, 16), generator=gen, device=DEV), dim=1)
    q = torch.nn.functional.normalize(torch.randn((65_736, 16), generator=gen, device=DEV), dim=1)
    (gi, gd) = knn_exact(q, v, 4, metric)
    for s in (0, 65_408, 65_536, 65_636):
        (fi, fd) = knn_exact(q[s:s + 100].contiguous(), v, 4, metric)
        assert torch.equal(gi[s:s + 100], fi) and torch.equal(gd[s:s + 100], fd)


@pytest.mark.parametrize("metric", ["cosine", "l2"])
@pytest.mark.parametrize("bad", ["nan", "inf", "long"])
def test_no_bound_in_a_short_last_piece_of_the_table(bad, metric):
    """2 GiB of 64 columns are 16,777,216 rows: the second piece of the table is 100 rows of a tile of 256, and one of them
    takes that piece's error bound beyond every value.  The 156 places behind the last row must not become candidates."""
    print(f"short last piece with {bad} {metric}", flush=True)
    from vectorlink_gpu.kernels import knn_exact

    gen = torch.Generator(device=DEV).manual_seed(5)
    n = (1 << 24) + 100
    v = torch.nn.functional.normalize(torch.randn((n, 4), generator=gen, device=DEV), dim=1)
    q = torch.nn.functional.normalize(torch.randn((150, 4), generator=gen, device=DEV), dim=1)
    if bad == "long":
        v[n - 7] *= 1e6
    else:
        v[n - 7, 2] = float(bad)
    (gi, gd) = knn_exact(q, v, 4, metric)
    assert int(gi.max()) < n and int(gi.min()) >= 0
    for s in range(0, 150, 32):
        (fi, fd) = knn_exact(q[s:s + 32].contiguous(), v, 4, metric)
        assert torch.equal(gi[s:s + 32], fi) and torch.equal(gd[s:s + 32], fd)


@pytest.mark.parametrize("metric", ["cosine", "l2"])
@pytest.mark.parametrize("k", [1, 10, 13, 16])
@pytest.mark.parametrize("n", [20, 1000, 9000, 70_000])
def test_values_that_are_not_finite(n, k, metric):
    """A distance that is not finite is nobody's neighbour: a NaN query has no neighbours under the cosine, a NaN row is
    none; all forms agree (a few queries with one and with several tiles per wavefront; a batch of 150)."""
    print(f"not finite n={n} k={k} {metric}", flush=True)
    from vectorlink_gpu.kernels import knn_exact

    rng = np.random.default_rng(n + k)
    v, q = rows(rng, n, 20), rows(rng, 150, 20)
    v[5, 3], v[6, 2], v[7, 0], v[8] = np.nan, np.inf, -np.inf, 3e38
    q[1, 1], q[2, 4], q[3, 0], q[4] = np.nan, -np.inf, np.inf, 3e38
    (gv, gq) = (dev(v), dev(q))
    (mi, md) = knn_exact(gq, gv, k, metric)
    (fi, fd) = knn_exact(gq[:30].contiguous(), gv, k, metric)
    assert torch.equal(mi[:30], fi) and torch.equal(md[:30], fd)
    assert not md.isnan().any()
    assert ((md == orc.MAXFLOAT) == (mi == orc.MAXINT)).all()
    if metric == "cosine":
        assert (fi[1] == orc.MAXINT).all() and (fi != 5).all()


def call(q, v, k, metric="cosine"):
    """(ids, distances, the queries left to the tiles or None if the filter does not take the call), whatever the sizes."""
    from vectorlink_gpu import _native as nv

    (nq, dim) = q.shape
    code = nv.metric_code(metric) + nv.KNN_ANY_SIZE
    sizes = (nq, v.shape[0], dim, k, code)
    ws = torch.empty(nv.lib().vl_knn_metric_workspace_bytes(*sizes), dtype=torch.uint8, device=DEV)
    ids = torch.empty((nq, k), dtype=torch.int32, device=DEV)
    d = torch.empty((nq, k), dtype=torch.float32, device=DEV)
    nv.check(nv.lib().vl_knn_exact_metric(nv.ptr(q), nq, nv.ptr(v), v.shape[0], dim, k, code, nv.ptr(ids),
                                          nv.ptr(d), nv.ptr(ws), ws.numel(), nv.stream()))
    if nv.lib().vl_knn_form(*sizes, ws.numel()) != 2:
        return ids, d, None
    at = nv.lib().vl_knn_left_offset(*sizes, ws.numel())
    words = ws[at:at + 4 * (1 + nq)].view(torch.int32).cpu()
    return ids, d, words[1:1 + int(words[0])].tolist()


def agrees_with_a_few_queries(q, v, k, metric, ids, d):
    from vectorlink_gpu.kernels import knn_exact

    for s in range(0, q.shape[0], 32):
        (fi, fd) = knn_exact(q[s:s + 32].contiguous(), v, k, metric)
        assert torch.equal(ids[s:s + 32], fi) and torch.equal(d[s:s + 32], fd)


@pytest.mark.parametrize("n,dim,nq,k,metric,crowded", [
    (60_000, 64, 1000, 10, "cosine", [0, 130, 131, 511, 999]), (40_000, 128, 2500, 16, "l2", [2499]),
    (20_000, 64, 700, 4, "cosine", list(range(100, 400))), (9000, 256, 300, 12, "cosine", list(range(300)))])
def test_only_the_queries_that_overflow_are_left_to_the_tiles(n, dim, nq, k, metric, crowded):
    """3,000 rows within the rounding of each other around some of the queries; the others are answered by the filter."""
    print(f"crowded queries n={n} dim={dim} nq={nq} k={k} {metric}", flush=True)
    gen = torch.Generator(device=DEV).manual_seed(n)
    v = torch.nn.functional.normalize(torch.randn((n, dim), generator=gen, device=DEV), dim=1)
    q = torch.nn.functional.normalize(torch.randn((nq, dim), generator=gen, device=DEV), dim=1)
    centre = q[crowded[0]].clone()
    q = torch.nn.functional.normalize(q - (q @ centre)[:, None] * centre, dim=1)  # the others: none of the 3,000 near them
    at = torch.randperm(n, generator=gen, device=DEV)[:3000]
    v[at] = torch.nn.functional.normalize(centre + 1e-4 * torch.randn((3000, dim), generator=gen, device=DEV), dim=1)
    for c in crowded:
        q[c] = torch.nn.functional.normalize(centre + 1e-4 * q[c], dim=0)
    (ids, d, left) = call(q, v, k, metric)
    assert left == crowded
    agrees_with_a_few_queries(q, v, k, metric, ids, d)


@pytest.mark.parametrize("metric", ["cosine", "l2"])
@pytest.mark.parametrize("order", ["random", "by cluster", "in turn"])
@pytest.mark.parametrize("n,dim,members,nq,k", [(60_000, 128, 200, 600, 10), (9000, 64, 90, 300, 16), (131_075, 256, 500, 400, 1)])
def test_the_order_of_the_rows_does_not_matter(n, dim, members, nq, k, order, metric):
    """Clusters whose rows follow each other, or come one from each in turn: the sample that bounds are taken from meets all
    of them, and no query has more candidates than its buffer holds."""
    print(f"order {order} n={n} dim={dim} members={members} nq={nq} k={k} {metric}", flush=True)
    gen = torch.Generator(device=DEV).manual_seed(n + k)
    count = n // members
    at = torch.arange(n, device=DEV)
    group = {"random": at[torch.randperm(n, generator=gen, device=DEV)] % count, "by cluster": at * count // n,
             "in turn": at % count}[order]
    centres = torch.randn((count, dim), generator=gen, device=DEV)
    v = centres[group] + 0.15 * torch.randn((n, dim), generator=gen, device=DEV)
    q = centres[torch.randint(0, count, (nq,), generator=gen, device=DEV)] + 0.15 * torch.randn((nq, dim), generator=gen, device=DEV)
    (v, q) = (torch.nn.functional.normalize(x, dim=1) for x in (v, q))
    (ids, d, left) = call(q, v, k, metric)
    assert left == []
    agrees_with_a_few_queries(q, v, k, metric, ids, d)


# candidates of a query around the wavefronts' shares of 8, 16, 32 and 64 rows, one round of a workgroup and several;
# rows that end within a line of 32 columns, with and without a chunk on its own
@pytest.mark.parametrize("nq", [200, 600])
@pytest.mark.parametrize("members,dim,k,metric", [
    (3, 20, 16, "cosine"), (9, 64, 1, "cosine"), (17, 36, 10, "l2"), (33, 132, 4, "cosine"), (64, 256, 16, "cosine"),
    (65, 28, 12, "l2"), (129, 60, 10, "cosine"), (300, 300, 16, "cosine"), (1025, 768, 10, "cosine"), (1900, 4, 8, "l2")])
def test_candidates_of_every_number(members, dim, k, metric, nq):
    """Rows close to each other in groups: a query has its whole group to evaluate."""
    print(f"candidates members={members} dim={dim} nq={nq} k={k} {metric}", flush=True)
    gen = torch.Generator(device=DEV).manual_seed(members)
    n = 12_007 if members < 1000 else 80_003  # (in a short table the tiles take queries with so many)
    count = n // members
    group = torch.arange(n, device=DEV) % count
    centres = torch.randn((count, dim), generator=gen, device=DEV)
    v = centres[group] + 1e-3 * torch.randn((n, dim), generator=gen, device=DEV)
    q = centres[torch.randint(0, count, (nq,), generator=gen, device=DEV)] + 1e-3 * torch.randn((nq, dim), generator=gen, device=DEV)
    if metric == "cosine":
        (v, q) = (torch.nn.functional.normalize(x, dim=1) for x in (v, q))
    v[n // 2] = v[n // 3]  # a tie that the ids decide
    (ids, d, left) = call(q, v, k, metric)
    assert left == [] or dim == 4  # (groups of 4 columns lie on top of each other)
    agrees_with_a_few_queries(q, v, k, metric, ids, d)


@pytest.mark.parametrize("n,dim,members,nq,k", [(16_384, 1536, 977, 1000, 10), (100_000, 64, 20_000, 300, 1), (9000, 128, 3000, 513, 16)])
def test_queries_that_the_tiles_answer_sooner_are_left_to_them(n, dim, members, nq, k):
    """The sample shows that a query has more candidates than are worth evaluating one by one; half the queries have few."""
    print(f"expected candidates n={n} dim={dim} members={members} nq={nq} k={k}", flush=True)
    gen = torch.Generator(device=DEV).manual_seed(n)
    v = torch.nn.functional.normalize(torch.randn((n, dim), generator=gen, device=DEV), dim=1)
    q = torch.nn.functional.normalize(torch.randn((nq, dim), generator=gen, device=DEV), dim=1)
    crowd = torch.nn.functional.normalize(torch.randn((1, dim), generator=gen, device=DEV), dim=1)
    q -= (q @ crowd.T) * crowd
    at = torch.randperm(n, generator=gen, device=DEV)[:members]
    v[at] = crowd + 1e-3 * v[at]
    q[::2] = crowd + 1e-3 * q[::2]
    (v, q) = (torch.nn.functional.normalize(x, dim=1) for x in (v, q))
    (ids, d, left) = call(q, v, k)
    assert left == list(range(0, nq, 2))
    agrees_with_a_few_queries(q, v, k, "cosine", ids, d)


@pytest.mark.parametrize("n,dim,nq,k,metric", [
    (4096, 64, 129, 10, "cosine"), (4097, 4, 256, 16, "cosine"), (5000, 60, 257, 4, "l2"), (6000, 64, 300, 1, "l2"),
    (4096, 1536, 1, 1, "cosine"), (8191, 132, 33, 12, "l2"), (33_000, 196, 513, 12, "l2"), (40_000, 192, 700, 16, "cosine")])
def test_the_filter_against_float64(n, dim, nq, k, metric):
    """Calls of every size through the filter: no query is left to the tiles, and the answers are those of the other forms
    and, to the rounding of float32 sums (as in test_a_few_queries), those of 64 bits."""
    print(f"filter against float64 n={n} dim={dim} nq={nq} k={k} {metric}", flush=True)
    rng = np.random.default_rng(n + dim)
    (v, q) = (rows(rng, n, dim), rows(rng, nq, dim))
    q[nq // 2] = v[n - 1]
    (ids, d, left) = call(dev(q), dev(v), k, metric)
    assert left == []
    agrees_with_a_few_queries(dev(q), dev(v), k, metric, ids, d)
    s = q.astype(np.float64) @ v.astype(np.float64).T
    true = np.clip((1 - s) / 2, 0, 1) if metric == "cosine" else np.maximum(
        (q.astype(np.float64) ** 2).sum(1)[:, None] + (v.astype(np.float64) ** 2).sum(1)[None] - 2 * s, 0)
    want = np.sort(true, axis=1)[:, :k]
    assert np.allclose(d.cpu().numpy(), want, rtol=1e-5, atol=1e-6)
    assert np.allclose(np.take_along_axis(true, ids.cpu().numpy().astype(np.int64), 1), want, rtol=1e-5, atol=2e-6)


@pytest.mark.parametrize("metric", ["cosine", "l2"])
@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
def test_the_filter_of_a_short_table_with_values_that_are_not_finite(value, metric):
    print(f"filter of a short table with {value} {metric}", flush=True)
    rng = np.random.default_rng(3)
    (v, q) = (rows(rng, 5000, 20), rows(rng, 200, 20))
    q[3, 7] = value
    for bad in (False, True):
        if bad:
            v[4999, 2] = value
        (ids, d, left) = call(dev(q), dev(v), 10, metric)
        assert left == (list(range(200)) if bad else [3])
        agrees_with_a_few_queries(dev(q), dev(v), 10, metric, ids, d)


@pytest.mark.parametrize("nq,share,want", [(300, 3, "none"), (300, 1.5, "all"), (512, 1.9, "all"), (513, 1.9, "crowd"), (1000, 1.5, "crowd"), (1000, 3, "none")])
def test_what_a_batch_leaves_to_the_tiles_before_the_pass(nq, share, want):
    """Queries with 1,100 candidates, somewhat more than cost what the tiles do for one (858): a small batch is left as a
    whole or not at all, a large one leaves them if they are many."""
    print(f"left before the pass nq={nq} share={share}", flush=True)
    (n, dim) = (32_768, 256)
    gen = torch.Generator(device=DEV).manual_seed(nq)
    v = torch.nn.functional.normalize(torch.randn((n, dim), generator=gen, device=DEV), dim=1)
    q = torch.nn.functional.normalize(torch.randn((nq, dim), generator=gen, device=DEV), dim=1)
    crowd = torch.nn.functional.normalize(torch.randn((1, dim), generator=gen, device=DEV), dim=1)
    q -= (q @ crowd.T) * crowd
    v[torch.randperm(n, generator=gen, device=DEV)[:1100]] = crowd + 1e-3 * torch.randn((1100, dim), generator=gen, device=DEV)
    at = torch.randperm(nq, generator=gen, device=DEV)[:int(nq / share)].sort().values
    q[at] = crowd + 1e-3 * q[at]
    (v, q) = (torch.nn.functional.normalize(x, dim=1) for x in (v, q))
    (ids, d, left) = call(q, v, 1)
    assert left == {"none": [], "all": list(range(nq)), "crowd": at.tolist()}[want]
    agrees_with_a_few_queries(q, v, 1, "cosine", ids, d)
