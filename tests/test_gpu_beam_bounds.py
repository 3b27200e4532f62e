"""The beam loop with bounds from the products of all queries and vectors (csrc/near_products.h, knn_filter.hip) against the loop
without them and the oracle's.  A bound that is wrong by more than it says drops a candidate that belongs into a queue."""
import ctypes as C

import numpy as np
import pytest
import torch

from oracle import oracle as orc
from test_gpu_beam_table import config, dev, oracle, same, search, vectors

pytestmark = pytest.mark.gpu


def both(v, rows, beams, seeds, c, exclude=True, flags=0):
    """Results with the bounds and without bounds and sketch, and what was counted in a third run, with the bounds."""
    from vectorlink_gpu import Queue, _native as nv
    from vectorlink_gpu.ann import BEAM_BOUNDS, BEAM_NO_TABLE, BEAM_USES_SKETCH, _beam_params
    from vectorlink_gpu.kernels import build_sketch

    g = dev(v)
    length = seeds.shape[1]
    q = Queue(rows, length, length + max(length, beams.size(1) * c["parallel_visit_count"]))
    p = _beam_params(rows, v.shape[1], v.shape[0], beams.size(1), q, c, int(exclude), BEAM_BOUNDS | BEAM_USES_SKETCH | flags)
    assert nv.lib().vl_beam_ahead(C.byref(p)) == BEAM_BOUNDS  # (a call that took the distances would show nothing)
    sketch = build_sketch(g)
    want = search(g, rows, beams, seeds, c, exclude, BEAM_NO_TABLE | flags)
    got = search(g, rows, beams, seeds, c, exclude, BEAM_NO_TABLE | flags, sketch=sketch)
    same(got, want)
    got = search(g, rows, beams, seeds, c, exclude, BEAM_BOUNDS | flags, sketch=sketch)
    out = (C.c_double * 9)()
    nv.lib().vl_beam_profile(1, 1, out)
    try:
        again = search(g, rows, beams, seeds, c, exclude, BEAM_BOUNDS | flags, sketch=sketch)
    finally:
        nv.lib().vl_beam_profile(0, 1, out)
    same(again, want)
    return got, want, out


# remainders of the 64 columns of a stage, one to eight chunks of the sketch's shapes, tiles of 256 queries and vectors, classes of
# columns with and without a rest
@pytest.mark.parametrize("rows,n,dim", [(130, 3000, d) for d in (4, 60, 64, 68, 256, 260, 384, 512, 516, 768, 1024, 1028, 1536, 2048)] +
                         [(r, n, 128) for r in (1, 255, 256, 257, 513) for n in (1530, 1536, 1537, 3071)])
def test_same_queues(rows, n, dim):
    print(f"bounds {rows} x {n} x {dim}", flush=True)
    v = vectors(n, dim)
    beams = dev(orc.generate_circulant_beams(n, orc.primes(48)))
    seeds = orc.generate_circulant_beams(n, orc.primes(48))[:rows]
    (got, want, _) = both(v, rows, beams, seeds, config(beam_size=24))
    same(got, want)


def test_against_the_oracle_and_what_is_fetched():
    (n, rows, dim) = (6000, 40, 256)
    v = vectors(n, dim)
    ids = orc.generate_circulant_beams(n, orc.primes(64))
    c = config(beam_size=32)
    (got, _, out) = both(v, rows, dev(ids), ids[:rows], c)
    same(got, oracle(v, rows, ids, ids[:rows], c, True))
    (evals, wanted, sketched) = (out[4], out[7], out[8])
    assert sketched == 0 and 0 < evals < 0.5 * wanted


@pytest.mark.parametrize("kind", ["lengths", "duplicates", "nan", "inf", "huge", "zero"])
def test_rows_that_are_not_unit_vectors(kind):
    """Norms from 1e-3 to 50, equal rows (ties, distances of 0), a row whose products are no halves or no numbers."""
    (n, rows, dim) = (2500, 300, 256)
    v = vectors(n, dim)
    if kind == "lengths":
        v *= np.exp(np.random.default_rng(2).uniform(np.log(1e-3), np.log(50.0), (n, 1))).astype(np.float32)
    elif kind == "duplicates":
        v[:] = v[np.arange(n) % 400]
    elif kind == "zero":
        v[100:200] = 0
    else:
        v[77, 5] = {"nan": np.nan, "inf": np.inf, "huge": 1e25}[kind]
    beams = dev(orc.generate_circulant_beams(n, orc.primes(32)))
    seeds = orc.generate_circulant_beams(n, orc.primes(32))[:rows]
    (got, want, _) = both(v, rows, beams, seeds, config(beam_size=16))
    same(got, want)


def test_near_neighbours_and_the_stop_of_each_row():
    """A graph of near neighbours in clusters (rows give bounds up), lists that fill up, every row stopping on its own."""
    from vectorlink_gpu.ann import BEAM_PER_QUERY_STOP

    (n, rows, dim) = (3000, 280, 256)
    rng = np.random.default_rng(4)
    v = rng.standard_normal((10, dim))[rng.integers(0, 10, n)] + 0.15 * rng.standard_normal((n, dim))
    v = (v / np.linalg.norm(v, axis=1, keepdims=True)).astype(np.float32)
    sim = v @ v.T
    np.fill_diagonal(sim, -2)
    beams = dev(np.argsort(-sim, axis=1)[:, :32].astype(np.int32))
    seeds = orc.generate_circulant_beams(n, orc.primes(64))[:rows]
    for (c, flags) in ((config(beam_size=32), 0), (config(beam_size=32, exclude_factor=2), 0), (config(beam_size=32), BEAM_PER_QUERY_STOP)):
        (got, want, _) = both(v, rows, beams, seeds, c, True, flags)
        same(got, want)


def test_what_takes_the_bounds_and_what_does_not():
    """By the bytes that a call asks for."""
    from vectorlink_gpu import Queue, _native as nv
    from vectorlink_gpu.ann import BEAM_MANY_ITERATIONS, BEAM_NO_CACHE, BEAM_NO_TABLE, BEAM_USES_SKETCH, _beam_params

    def asks(rows, n, dim, flags, exclude, beam=64, width=128, metric="cosine"):
        q = Queue(rows, 128, 128 + 4 * width)
        c = config(beam_size=beam, metric=metric)

        def need(f):
            f |= BEAM_NO_CACHE | BEAM_MANY_ITERATIONS
            return nv.check(nv.lib().vl_beam_workspace_bytes(C.byref(_beam_params(rows, dim, n, width, q, c, exclude, f))))
        return need(flags) > need(flags | BEAM_NO_TABLE)

    assert asks(10_000, 1_000_000, 768, BEAM_USES_SKETCH, 1)
    assert not asks(10_000, 1_000_000, 768, 0, 1)                       # brings no sketch
    assert not asks(10_000, 1_000_000, 768, BEAM_USES_SKETCH, 0)        # a search
    assert not asks(10_000, 1_000_000, 768, BEAM_USES_SKETCH, 1, metric="l2")
    assert not asks(10_000, 1_000_000, 256, BEAM_USES_SKETCH, 1, 32, 64)  # more products than the iterations are worth
    assert not asks(10_000, 1_500_000, 768, BEAM_USES_SKETCH, 1)        # more than 24 GiB


def test_a_workspace_without_room_for_the_bounds():
    from vectorlink_gpu import Queue, _native as nv
    from vectorlink_gpu.ann import BEAM_BOUNDS, BEAM_NO_TABLE, BEAM_USES_SKETCH, _beam_params
    from vectorlink_gpu.kernels import build_sketch

    (n, rows, dim, length) = (20_000, 300, 256, 32)
    v = vectors(n, dim)
    (gv, gb) = (dev(v), dev(orc.generate_circulant_beams(n, orc.primes(16))))
    sketch = build_sketch(gv)
    seeds = orc.generate_circulant_beams(n, orc.primes(length))[:rows]
    d = dev(orc.gather_distances(v[:rows], v, seeds))
    c = config(beam_size=16)
    results = []
    for (flags, sized) in ((BEAM_BOUNDS, BEAM_BOUNDS), (BEAM_BOUNDS, BEAM_NO_TABLE), (BEAM_NO_TABLE, BEAM_NO_TABLE)):
        q = Queue(rows, length, length + 64)
        q.insert(dev(seeds), d)
        have = nv.lib().vl_beam_workspace_bytes(C.byref(_beam_params(rows, dim, n, 16, q, c, 0, sized | BEAM_USES_SKETCH)))
        p = _beam_params(rows, dim, n, 16, q, c, 0, flags | BEAM_USES_SKETCH)
        assert nv.lib().vl_beam_workspace_bytes(C.byref(p)) >= have
        ws = torch.full((have + 256,), 0xA5, dtype=torch.uint8, device="cuda:0")
        rc = nv.lib().vl_closest_vectors_with_sketch(C.byref(p), nv.ptr(gv), nv.ptr(gv), nv.ptr(sketch), nv.ptr(gb), nv.ptr(q.indices),
                                                     nv.ptr(q.distances), None, nv.ptr(ws), have, nv.stream())
        assert bool((ws[have:] == 0xA5).all())
        results.append((rc, q.indices.cpu().numpy()[:, :length], q.distances.cpu().numpy()[:, :length].view(np.uint32)))
    assert results[0][0] > 0
    same(results[1], results[0])
    same(results[2], results[0])
