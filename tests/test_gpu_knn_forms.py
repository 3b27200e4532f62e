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
