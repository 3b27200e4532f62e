"""The search queue that a search starts from, made in one launch (csrc/seed.hip), against the oracle's seeds, distances and
queue insert."""
import numpy as np
import pytest
import torch

from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")


# seeds on both sides of what a wavefront takes and of the powers of two that are sorted; row lengths of every form, aligned
# and not; fewer vectors than seeds (copies of an id), more rows than vectors (numbers that wrap round)
@pytest.mark.parametrize("metric", ["cosine", "l2"])
@pytest.mark.parametrize("rows,n,dim,k,more", [(1, 50, 3, 1, 1), (3, 50, 4, 4, 0), (2, 300, 50, 16, 5), (5, 40, 64, 63, 100),
                                               (70, 20, 128, 64, 1), (1, 500, 130, 65, 300), (4, 500, 300, 127, 1),
                                               (9, 500, 768, 128, 384), (2, 900, 1030, 255, 1), (2, 900, 1536, 257, 300),
                                               (1, 1200, 2049, 965, 100), (300, 600, 7, 72, 96)])
def test_seeded_queue_is_the_first_insert(rows, n, dim, k, more, metric):
    print(f"seeded queue rows={rows} n={n} dim={dim} k={k} {metric}", flush=True)
    from vectorlink_gpu import Queue
    from vectorlink_gpu.utils import primes

    rng = np.random.default_rng(rows + n + dim)
    v = rng.standard_normal((n, dim)).astype(np.float32)
    q = rng.standard_normal((rows, dim)).astype(np.float32)
    (length, cap) = (k, 2 * k + more)
    names = rng.permutation(n)[: max(1, n // 2)].astype(np.int32)
    places = rng.integers(0, names.size, (rows, k)).astype(np.int32)
    ids = rng.integers(0, n, (rows, k)).astype(np.int32)
    ids[rng.random((rows, k)) < 0.1] = 0x7FFFFFFF
    with orc.metric(metric):
        for (got, seeds) in (
                (Queue.seeded(length, cap, dev(q), dev(v), primes(k, "cuda:0"), metric), orc.generate_queue_circulants(rows, n, orc.primes(k))),
                (Queue.seeded(length, cap, dev(q), dev(v), dev(places), metric, names=dev(names)), names[places]),
                (Queue.seeded(length, cap, dev(q), dev(v), dev(ids), metric), ids)):
            want = orc.Queue(rows, length, cap)
            want.insert(seeds, orc.gather_distances(q, v, seeds))
            assert got.length == length and got.indices.size() == (rows, cap)
            assert np.array_equal(got.indices.cpu().numpy(), want.indices)
            assert np.array_equal(got.distances.cpu().numpy().view(np.uint32), want.distances.view(np.uint32))


@pytest.mark.parametrize("value", [np.inf, np.nan, 1e25])
def test_seeds_at_no_ordinary_distance(value):
    from vectorlink_gpu import Queue

    v = np.random.default_rng(1).standard_normal((40, 24)).astype(np.float32)
    v[7, 3] = value
    v[9, 20] = value
    seeds = np.tile(np.array([3, 7, 9, 7, 20, 0x7FFFFFFF, 9, 1], dtype=np.int32), (5, 1))
    (q, cap) = (v[:5], 21)
    with orc.metric("l2"):
        want = orc.Queue(5, 8, cap)
        want.insert(seeds, orc.gather_distances(q, v, seeds))
    got = Queue.seeded(8, cap, dev(q), dev(v), dev(seeds), "l2")
    assert np.array_equal(got.indices.cpu().numpy(), want.indices)
    assert np.array_equal(got.distances.cpu().numpy(), want.distances, equal_nan=True)


def test_what_does_not_fit_is_refused():
    from vectorlink_gpu import Queue

    v = torch.zeros((10, 4), device="cuda:0")
    with pytest.raises(ValueError, match="do not fit"):
        Queue.seeded(6, 10, v, v, torch.zeros((10, 5), dtype=torch.int32, device="cuda:0"))
    assert Queue.seeded(4, 9, v[:0], v, torch.zeros((0, 4), dtype=torch.int32, device="cuda:0")).indices.size() == (0, 9)


def test_entry_points_from_every_other_id_of_a_list():
    from vectorlink_gpu.ann import dense_search_queue

    rng = np.random.default_rng(3)
    v = rng.standard_normal((400, 32)).astype(np.float32)
    v /= np.linalg.norm(v, axis=1, keepdims=True)
    ids = rng.permutation(400)[:200].astype(np.int32)
    c = dict(orc.DEFAULT_CONFIG, beam_size=8)
    entry = dev(v[ids[::2]])
    want = dense_search_queue(dev(v), dev(v[:9]), c, dev(ids[::2]), entry)
    got = dense_search_queue(dev(v), dev(v[:9]), c, dev(ids)[::2], entry)
    assert torch.equal(got.indices, want.indices) and torch.equal(got.distances, want.distances)
