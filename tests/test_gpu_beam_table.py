"""The beam loop with the distances of all queries and vectors ahead of it (csrc/pair_table.hip, beam_table.hip) against the
oracle's loop.  Distances are looked up as the bits that the products' kernel left, so a wrong sum, column or order of
additions shows as other bits; the loop itself is compared over queue lengths, candidates and visits around the sets of 64."""
import ctypes as C

import numpy as np
import pytest
import torch

from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")


def bits(t):
    return t.cpu().numpy().view(np.uint32)


def vectors(n, dim, metric="cosine", seed=0):
    v = np.random.default_rng(seed + n + dim).standard_normal((n, dim)).astype(np.float32)
    return v if metric == "l2" else v / np.linalg.norm(v, axis=1, keepdims=True)


def config(**kw):
    c = dict(orc.DEFAULT_CONFIG)
    c.update(kw)
    return c


def ahead(rows, n, dim, beams, queue, c, exclude, flags):
    """What the sizes and the flags give a call ahead of its loop (include/vlgpu.h: vl_beam_ahead)."""
    from vectorlink_gpu import _native as nv
    from vectorlink_gpu.ann import _beam_params

    p = _beam_params(rows, dim, n, beams.size(1), queue, c, int(exclude), flags)
    return nv.check(nv.lib().vl_beam_ahead(C.byref(p))), nv.check(nv.lib().vl_beam_workspace_bytes(C.byref(p)))


def search(v, rows, beams, seeds, c, exclude, flags, sketch=None, table=True):
    """(iterations, ids, distance bits) of rows 0 .. rows - 1 searched from seeds (ids).  A call that asks for the table is given
    it, and finds the room (table=False: is expected not to find it)."""
    from vectorlink_gpu import Queue
    from vectorlink_gpu.ann import BEAM_TABLE, BEAM_USES_SKETCH, _workspace, closest_vectors, excluding_self
    from vectorlink_gpu.kernels import gather_distances

    length = seeds.shape[1]
    q = Queue(rows, length, length + max(length, beams.size(1) * c["parallel_visit_count"]))
    ids = dev(seeds)
    q.insert(ids, gather_distances(v[:rows], v, ids, metric=c.get("metric", "cosine")))
    t = closest_vectors(v[:rows], q, v, beams, c, excluding_self(0, rows) if exclude else None, flags=flags, sketch=sketch)
    if flags & BEAM_TABLE:
        (given, need) = ahead(rows, v.size(0), v.size(1), beams, q, c, exclude, flags | (BEAM_USES_SKETCH if sketch is not None else 0))
        assert given == BEAM_TABLE
        assert _workspace(v.device).has(need) == table
    return t, q.indices.cpu().numpy()[:, :length], bits(q.distances)[:, :length]


def oracle(v, rows, beams, seeds, c, exclude, per_query=False):
    length = seeds.shape[1]
    q = orc.Queue(rows, length, length + max(length, beams.shape[1] * c["parallel_visit_count"]))
    with orc.metric(c.get("metric", "cosine")):
        q.insert(seeds, orc.gather_distances(v[:rows], v, seeds))
        run = orc.closest_vectors_per_query if per_query else orc.closest_vectors
        t = run(v[:rows], q, v, beams, c, orc.excluding_self(0, rows) if exclude else None)
    return t, q.indices[:, :length], q.distances[:, :length].view(np.uint32)


def same(got, want):
    assert got[0] == want[0]
    assert np.array_equal(got[1], want[1])
    assert np.array_equal(got[2], want[2])


# every length of a row's last chunk and last set of 16, 32 and 64 partial sums; tiles of 64 queries and vectors and their
# neighbours; the classes of columns with and without a rest
@pytest.mark.parametrize("metric", ["cosine", "l2"])
@pytest.mark.parametrize("rows,n,dim", [(1, 65, d) for d in (1, 2, 3, 4, 5, 61, 63, 64, 65, 66, 127, 128, 129, 130, 255, 256, 257, 260,
                                                            383, 384, 511, 512, 513, 768, 1023, 1027, 1536, 2045, 2048)] +
                         [(r, n, 20) for r in (1, 63, 64, 65, 129) for n in (129, 191, 192, 193, 384, 385)])
def test_distances_have_the_bits_of_the_sums(rows, n, dim, metric):
    print(f"table distances {rows} x {n} x {dim} {metric}", flush=True)
    from vectorlink_gpu.ann import BEAM_TABLE

    v = vectors(n, dim, metric)
    c = config(beam_size=16, exclude_factor=30, metric=metric)
    beams = orc.generate_circulant_beams(n, orc.primes(32))
    seeds = np.random.default_rng(n).permuted(np.tile(np.arange(n, dtype=np.int32), (rows, 1)), axis=1)[:, :48]
    got = search(dev(v), rows, dev(beams), seeds, c, False, BEAM_TABLE)
    same(got, oracle(v, rows, beams, seeds, c, False))


# queue and visit-queue lengths on both sides of 64 and 128, candidates on both sides of 64, 128, 256 and 512, one to eight
# visits, queues longer and shorter than the visit queue, lists that fill up (exclude_factor 2) and do not
@pytest.mark.parametrize("beam,length,width,visits,ef", [
    (4, 3, 5, 1, 5), (21, 63, 64, 1, 5), (21, 64, 65, 1, 2), (22, 65, 63, 2, 5), (24, 72, 24, 4, 5), (32, 64, 64, 4, 5),
    (32, 127, 32, 4, 2), (42, 128, 43, 3, 5), (43, 129, 64, 4, 5), (48, 96, 96, 4, 2), (64, 191, 64, 8, 5), (64, 192, 128, 4, 2),
    (64, 10, 128, 4, 5), (8, 190, 20, 5, 20)])
@pytest.mark.parametrize("per_query", [False, True])
def test_queues_around_the_sets_of_64(beam, length, width, visits, ef, per_query):
    print(f"table queues beam={beam} length={length} width={width} visits={visits} {per_query}", flush=True)
    from vectorlink_gpu.ann import BEAM_PER_QUERY_STOP, BEAM_TABLE

    (n, dim, rows) = (1500, 12, 90)
    v = vectors(n, dim)
    c = config(beam_size=beam, parallel_visit_count=visits, exclude_factor=ef)
    rng = np.random.default_rng(beam + length + width)
    beams = rng.integers(0, n, (n, width)).astype(np.int32)  # ids anywhere: several times in a list, in several lists
    beams[rng.random((n, width)) < 0.1] = 0x7FFFFFFF         # and empty slots
    seeds = rng.permuted(np.tile(np.arange(n, dtype=np.int32), (rows, 1)), axis=1)[:, :length]
    flags = BEAM_TABLE | (BEAM_PER_QUERY_STOP if per_query else 0)
    for exclude in (False, True):
        got = search(dev(v), rows, dev(beams), seeds, c, exclude, flags)
        same(got, oracle(v, rows, beams, seeds, c, exclude, per_query))


@pytest.mark.parametrize("sketched", [False, True])
def test_distances_are_looked_up_and_not_fetched(sketched):
    """What a profiled call counts: candidates, and none of them a row that was read."""
    from vectorlink_gpu import _native as nv
    from vectorlink_gpu.ann import BEAM_TABLE
    from vectorlink_gpu.kernels import build_sketch

    (n, rows) = (900, 300)
    v = dev(vectors(n, 256))
    ids = orc.generate_circulant_beams(n, orc.primes(32))
    out = (C.c_double * 9)()
    nv.lib().vl_beam_profile(1, 1, out)
    try:
        search(v, rows, dev(ids), ids[:rows], config(beam_size=16, exclude_factor=30), True, BEAM_TABLE,
               sketch=build_sketch(v) if sketched else None)
    finally:
        nv.lib().vl_beam_profile(0, 1, out)
    (evals, wanted, through_sketch) = (out[4], out[7], out[8])
    assert evals == through_sketch == 0 and wanted > 4 * 32 * rows


def test_many_rows_and_the_sketch():
    """More rows than the chip holds at once, visited lists that fill up, a sketch that only calls without the table use."""
    from vectorlink_gpu.ann import BEAM_NO_TABLE, BEAM_TABLE
    from vectorlink_gpu.kernels import build_sketch

    (n, rows) = (9000, 8700)
    v = dev(vectors(n, 256))
    beams = dev(orc.generate_circulant_beams(n, orc.primes(32)))
    seeds = orc.generate_circulant_beams(n, orc.primes(32))[:rows]
    c = config(beam_size=16, exclude_factor=2)
    sketch = build_sketch(v)
    want = search(v, rows, beams, seeds, c, True, BEAM_NO_TABLE)
    for s in (None, sketch):
        same(search(v, rows, beams, seeds, c, True, BEAM_TABLE, sketch=s), want)


@pytest.mark.parametrize("metric,value", [("cosine", np.nan), ("cosine", np.inf), ("l2", np.inf), ("l2", -1e30), ("l2", np.nan)])
def test_distances_that_are_no_ordinary_numbers(metric, value):
    """One vector has them: the loop leaves the table alone, and what it had not begun it ends without."""
    from vectorlink_gpu.ann import BEAM_NO_TABLE, BEAM_TABLE
    from vectorlink_gpu.kernels import build_sketch

    (n, rows, dim) = (700, 130, 256)
    v = vectors(n, dim, metric)
    v[333, 5] = value
    g = dev(v)
    beams = dev(orc.generate_circulant_beams(n, orc.primes(32)))
    seeds = orc.generate_circulant_beams(n, orc.primes(32))[:rows]
    c = config(beam_size=16, metric=metric)
    for sketch in (None, build_sketch(g)):
        want = search(g, rows, beams, seeds, c, True, BEAM_NO_TABLE, sketch=sketch)
        same(search(g, rows, beams, seeds, c, True, BEAM_TABLE, sketch=sketch), want)


# The launch behind the refused one is an ordinary one: lists with room for one stretch between two progress checks and not for two
# (24 ids of 4 a time in stretches of 5; 360 in stretches of 50).  Profiled calls wait for a check before they go on, others do not.
@pytest.mark.parametrize("metric,value", [("cosine", np.nan), ("cosine", np.inf), ("l2", np.inf), ("l2", 1e19), ("l2", np.nan)])
@pytest.mark.parametrize("beam,ef,ra", [(8, 1, 5), (24, 5, 50)])
@pytest.mark.parametrize("per_query", [False, True])
def test_refused_where_the_lists_fill_up_in_the_next_launch(beam, ef, ra, metric, value, per_query):
    print(f"table refused beam={beam} ra={ra} {metric} {value} {per_query}", flush=True)
    from vectorlink_gpu import _native as nv
    from vectorlink_gpu.ann import BEAM_PER_QUERY_STOP, BEAM_TABLE
    from vectorlink_gpu.kernels import build_sketch

    (n, rows, dim) = (700, 130, 256)
    v = vectors(n, dim, metric)
    v[333, 5] = value
    g = dev(v)
    ids = orc.generate_circulant_beams(n, orc.primes(2 * beam))
    c = config(beam_size=beam, exclude_factor=ef, speculative_readahead=ra, metric=metric)
    flags = BEAM_TABLE | (BEAM_PER_QUERY_STOP if per_query else 0)
    want = oracle(v, rows, ids, ids[:rows], c, True, per_query)
    assert not np.array_equal(np.sort(want[1], axis=1), np.sort(ids[:rows], axis=1))  # (a call that does nothing is not right by chance)

    def check(sketch=None):
        got = search(g, rows, dev(ids), ids[:rows], c, True, flags, sketch=sketch)
        assert got[0] == want[0] and np.array_equal(got[1], want[1])
        assert np.array_equal(got[2].view(np.float32), want[2].view(np.float32), equal_nan=True)

    check()
    check(build_sketch(g))
    if ra <= 64:
        nv.lib().vl_beam_profile(1, 1, None)
        try:
            check()
        finally:
            nv.lib().vl_beam_profile(0, 1, None)


def test_a_workspace_without_room_for_the_table():
    from vectorlink_gpu import Queue, _native as nv
    from vectorlink_gpu.ann import BEAM_NO_TABLE, BEAM_TABLE, _beam_params

    (n, rows, dim, length) = (40_000, 300, 24, 32)
    v = vectors(n, dim)
    (gv, gb) = (dev(v), dev(orc.generate_circulant_beams(n, orc.primes(16))))
    seeds = orc.generate_circulant_beams(n, orc.primes(length))[:rows]
    d = dev(orc.gather_distances(v[:rows], v, seeds))
    c = config(beam_size=16)
    results = []
    for (flags, sized) in ((BEAM_TABLE, BEAM_TABLE), (BEAM_TABLE, BEAM_NO_TABLE), (BEAM_NO_TABLE, BEAM_NO_TABLE)):
        q = Queue(rows, length, length + 64)
        q.insert(dev(seeds), d)
        have = nv.lib().vl_beam_workspace_bytes(C.byref(_beam_params(rows, dim, n, 16, q, c, 0, sized)))
        p = _beam_params(rows, dim, n, 16, q, c, 0, flags)
        assert nv.lib().vl_beam_workspace_bytes(C.byref(p)) >= have
        ws = torch.full((have + 256,), 0xA5, dtype=torch.uint8, device="cuda:0")
        rc = nv.lib().vl_closest_vectors(C.byref(p), nv.ptr(gv), nv.ptr(gv), nv.ptr(gb), nv.ptr(q.indices), nv.ptr(q.distances),
                                         None, nv.ptr(ws), have, nv.stream())
        assert bool((ws[have:] == 0xA5).all())
        results.append((rc, q.indices.cpu().numpy()[:, :length], bits(q.distances)[:, :length]))
    assert results[0][0] > 0
    same(results[1], results[0])
    same(results[2], results[0])


def test_what_takes_the_table_and_what_does_not():
    """By the bytes that a call asks for: the rule on sizes and on what a call says of itself."""
    from vectorlink_gpu import Queue, _native as nv
    from vectorlink_gpu.ann import BEAM_MANY_ITERATIONS, BEAM_NO_CACHE, BEAM_NO_TABLE, _beam_params

    def asks(rows, n, dim, flags, exclude, metric="cosine", beam=64, width=128):
        q = Queue(rows, 128, 128 + 4 * width)
        c = config(beam_size=beam, metric=metric)

        def need(f):
            f |= BEAM_NO_CACHE  # (the table lies where the cache would)
            return nv.check(nv.lib().vl_beam_workspace_bytes(C.byref(_beam_params(rows, dim, n, width, q, c, exclude, f))))
        return need(flags) > need(BEAM_NO_TABLE)

    assert asks(10_000, 150_000, 768, BEAM_MANY_ITERATIONS, 1)
    assert not asks(10_000, 450_000, 64, BEAM_MANY_ITERATIONS, 1)     # more than 16 GiB of distances
    assert not asks(1_000, 1_000_000, 768, BEAM_MANY_ITERATIONS, 1)   # more products than the iterations are worth
    assert asks(64, 4_096, 128, BEAM_MANY_ITERATIONS, 0)
    assert not asks(64, 4_096, 128, 0, 0)                             # asks for a small workspace and says nothing else


def test_no_memory_for_the_table(monkeypatch):
    """The workspace with the table cannot be had: the call runs without it."""
    from vectorlink_gpu import ann

    (n, rows) = (3000, 200)
    v = dev(vectors(n, 24))
    beams = dev(orc.generate_circulant_beams(n, orc.primes(32)))
    seeds = orc.generate_circulant_beams(n, orc.primes(32))[:rows]
    c = config(beam_size=16, exclude_factor=2)
    want = search(v, rows, beams, seeds, c, True, ann.BEAM_NO_TABLE | ann.BEAM_NO_CACHE)
    (asked, reserve) = ([], ann._Workspace.reserve)

    def refuse_first(self, nbytes, device):
        asked.append(nbytes)
        if len(asked) == 1:
            raise torch.OutOfMemoryError("no room")
        return reserve(self, nbytes, device)

    ann.release_workspaces()
    monkeypatch.setattr(ann._Workspace, "reserve", refuse_first)
    same(search(v, rows, beams, seeds, c, True, ann.BEAM_TABLE | ann.BEAM_NO_CACHE, table=False), want)
    assert len(asked) == 2 and asked[1] < asked[0]


@pytest.mark.parametrize("circulant", [True, False])
def test_a_batch_of_a_build_that_comes_without_a_word(circulant):
    """Rows that exclude themselves: the graph is looked at, on the last node's list as on the others (it wraps round)."""
    (n, rows) = (70_001, 400)
    v = dev(vectors(n, 64))
    ids = orc.generate_circulant_beams(n, orc.primes(64))
    if not circulant:
        ids = np.random.default_rng(5).integers(0, n, ids.shape).astype(np.int32)
    seeds = orc.generate_circulant_beams(n, orc.primes(64))[:rows]
    c = config(beam_size=32)
    from vectorlink_gpu import Queue
    from vectorlink_gpu.ann import BEAM_MANY_ITERATIONS, BEAM_NO_TABLE, BEAM_TABLE, _circulant_graph

    q = Queue(rows, 64, 64 + 256)
    assert ahead(rows, n, 64, dev(ids), q, c, True, 0)[0] == BEAM_MANY_ITERATIONS and _circulant_graph(dev(ids)) == circulant
    assert ahead(rows, n, 64, dev(ids), q, c, True, BEAM_MANY_ITERATIONS)[0] == BEAM_TABLE
    same(search(v, rows, dev(ids), seeds, c, True, 0), search(v, rows, dev(ids), seeds, c, True, BEAM_NO_TABLE))
