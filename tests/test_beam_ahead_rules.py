"""Which calls of the beam loop are given the distances or bounds of all their queries and vectors, by the bytes of workspace that
they ask for and by vl_beam_ahead (include/vlgpu.h); nothing is launched."""
import ctypes as C

import pytest

NO_CACHE, SKETCH, MANY, TABLE, NO_TABLE, BOUNDS, KNOWN = 8, 16, 128, 256, 512, 1024, 2048  # VL_BEAM_*


def params(flags, rows=10_000, n=1_000_000, dim=768, width=128, beam=64, visits=4, ef=5, readahead=5, excl=1, metric=0,
           length=128):
    from vectorlink_gpu import _native as nv

    return nv.BeamParams(n_rows=rows, dim=dim, n_vectors=n, width=width, queue_capacity=length + max(length, visits * width), queue_length=length,
                         beam_size=beam, parallel_visit_count=visits, visit_queue_factor=3, exclude_factor=ef,
                         speculative_readahead=readahead, excl_cols=excl, flags=flags, metric=metric)


def need(flags, **kw):
    from vectorlink_gpu import _native as nv

    return nv.check(nv.lib().vl_beam_workspace_bytes(C.byref(params(flags, **kw))))


def asks(flags, **kw):
    """Bytes beyond those of the same call without distances and bounds (and without the cache, which they may lie over)."""
    flags |= NO_CACHE
    return need(flags, **kw) - need((flags | NO_TABLE) & ~(TABLE | BOUNDS), **kw)


def ahead(flags, **kw):
    from vectorlink_gpu import _native as nv

    return nv.check(nv.lib().vl_beam_ahead(C.byref(params(flags, **kw))))


@pytest.mark.parametrize("n", [1, 2, 63])
@pytest.mark.parametrize("flags", [SKETCH, SKETCH | MANY, SKETCH | BOUNDS, TABLE])
def test_a_few_vectors_have_neither(n, flags):
    """(The look at the graph reads the lists of a node and of the next one.)"""
    assert asks(flags, n=n) == 0 == ahead(flags, n=n)


@pytest.mark.parametrize("rows,n,dim", [(8, 70_000_000, 4), (1, 600_000_000, 4)])
def test_sizes_beyond_the_grid_of_the_distances_do_without(rows, n, dim):
    """(The kernels' launcher refuses them.)"""
    assert asks(TABLE, rows=rows, n=n, dim=dim) == 0
    assert asks(TABLE, rows=rows, n=60_000_000, dim=dim) > 0


def test_a_call_that_does_not_say_that_it_is_long_asks_for_no_more_than_without():
    """Rows that exclude their own ids, 10,000 of 1M x 768 (bounds, 20 GiB) and of 150,000 x 768 (distances, 6 GiB)."""
    for (sketch, n, given) in ((SKETCH, 1_000_000, BOUNDS), (0, 150_000, TABLE)):
        assert need(sketch, n=n) == need(sketch | NO_TABLE, n=n)
        assert need(sketch | MANY, n=n) > need(sketch | NO_TABLE, n=n)
        assert ahead(sketch | MANY, n=n) == given
        assert ahead(sketch, n=n) == MANY                                            # the graph is worth a look
        assert ahead(sketch | KNOWN, n=n) == 0 == ahead(sketch | NO_TABLE, n=n)
        assert ahead(sketch | NO_CACHE, n=n) == 0 == ahead(sketch, n=n, excl=0)      # a small workspace; a search
        assert ahead(sketch, n=n, rows=255) == 0


def test_a_small_table_needs_no_word():
    small = dict(rows=4096, n=4096, dim=128, width=64, beam=32)
    assert ahead(0, **small) == TABLE == ahead(KNOWN, **small) and asks(TABLE, **small) > 0


# (rows, vectors, columns, degree, queue): where storing the distances takes longer than looking at them saves, and where it does not
@pytest.mark.parametrize("given,sizes", [
    (0, (10_000, 100_000, 4, 64, 10)), (0, (10_000, 60_000, 24, 64, 10)), (0, (10_000, 60_000, 25, 64, 128)), (0, (10_000, 20_011, 64, 64, 10)),
    (TABLE, (10_000, 4_096, 24, 64, 10)), (TABLE, (10_000, 20_011, 24, 64, 10)), (TABLE, (10_000, 20_011, 64, 64, 128)),
    (TABLE, (2_000, 10_000, 24, 64, 10))])
def test_searches_that_say_nothing_pay_for_the_stores(given, sizes):
    (rows, n, dim, degree, length) = sizes
    assert ahead(0, rows=rows, n=n, dim=dim, width=degree, beam=degree, excl=0, length=length) == given


@pytest.mark.parametrize("given,sizes", [
    (0, (10_000, 400_000, 4, 24, 0)), (0, (10_000, 150_000, 4, 24, 0)), (0, (300, 400_000, 4, 32, 0)),
    (TABLE, (10_000, 60_000, 16, 24, 0)), (TABLE, (10_000, 60_000, 64, 64, 0)), (TABLE, (37, 20_011, 50, 24, 0)),
    (0, (10_000, 400_000, 16, 24, 1)), (TABLE, (10_000, 150_000, 50, 24, 1)), (TABLE, (10_000, 100_000, 128, 32, 1)),
    (TABLE, (10_000, 20_011, 768, 64, 1))])
def test_long_calls_pay_for_the_stores(given, sizes):
    (rows, n, dim, degree, first_loop) = sizes
    assert ahead(MANY, rows=rows, n=n, dim=dim, width=degree * (1 + first_loop), beam=degree, excl=first_loop, length=2 * degree) == given


def test_bounds_where_they_are_asked_for():
    """... and the sizes would have the distances: of rows that exclude their own ids and of a small table."""
    for kw in (dict(rows=300, n=2500, dim=256, width=32, beam=16), dict(rows=257, n=1530, dim=128, width=48, beam=24),
               dict(rows=4096, n=4096, dim=128, width=64, beam=32)):
        for said in (0, MANY):
            assert ahead(SKETCH | BOUNDS | said, **kw) == BOUNDS
            assert ahead(SKETCH | BOUNDS | TABLE | said, **kw) == TABLE
            assert ahead(BOUNDS | said, **kw) == ahead(said, **kw)  # brings no sketch


def test_bounds_that_no_launch_could_use_are_not_asked_for():
    """Lists that fill up before the first progress check run one iteration per launch, which the bounds are not built for."""
    assert ahead(SKETCH | MANY, readahead=200) == BOUNDS                  # 960 ids, 800 of them
    assert ahead(SKETCH | MANY, readahead=241) == 0 == asks(SKETCH | BOUNDS, readahead=241)
