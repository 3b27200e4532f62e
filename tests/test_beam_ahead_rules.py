"""Which calls of the beam loop ask for the distances or bounds of all their queries and vectors, by the bytes of workspace that
they ask for (include/vlgpu.h); nothing is launched."""
import ctypes as C

import pytest

NO_CACHE, SKETCH, MANY, TABLE, NO_TABLE, BOUNDS = 8, 16, 128, 256, 512, 1024  # VL_BEAM_*


def asks(flags, rows=10_000, n=1_000_000, dim=768, width=128, beam=64, visits=4, ef=5, readahead=5, excl=1, metric=0):
    """Bytes beyond those of the same call without distances and bounds (and without the cache, which they may lie over)."""
    from vectorlink_gpu import _native as nv

    def need(f):
        p = nv.BeamParams(n_rows=rows, dim=dim, n_vectors=n, width=width, queue_capacity=128 + visits * width, queue_length=128,
                          beam_size=beam, parallel_visit_count=visits, visit_queue_factor=3, exclude_factor=ef,
                          speculative_readahead=readahead, excl_cols=excl, flags=f | NO_CACHE, metric=metric)
        return nv.check(nv.lib().vl_beam_workspace_bytes(C.byref(p)))
    return need(flags) - need((flags | NO_TABLE) & ~(TABLE | BOUNDS))


@pytest.mark.parametrize("n", [1, 2, 63])
@pytest.mark.parametrize("flags", [SKETCH, SKETCH | MANY, SKETCH | BOUNDS, TABLE])
def test_a_few_vectors_have_neither(n, flags):
    """(The look at the graph reads the lists of a node and of the next one.)"""
    assert asks(flags, n=n) == 0


@pytest.mark.parametrize("rows,n,dim", [(8, 70_000_000, 4), (1, 600_000_000, 4)])
def test_sizes_beyond_the_grid_of_the_distances_do_without(rows, n, dim):
    """(The kernels' launcher refuses them.)"""
    assert asks(TABLE, rows=rows, n=n, dim=dim) == 0
    assert asks(TABLE, rows=rows, n=60_000_000, dim=dim) > 0
