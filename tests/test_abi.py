"""The C ABI without a GPU: the library loads, exports every function that
include/vlgpu.h declares, the Python binding table covers them all, and shape
validation rejects bad calls on the host before anything is launched."""
import ctypes as C
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "vlgpu.h")


def declared_functions():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(vl_[a-z0-9_]+)\s*\(", text)))


@pytest.fixture(scope="module")
def lib():
    from vectorlink_gpu import _native

    if not os.path.exists(_native.LIB_PATH):
        import __graft_entry__

        __graft_entry__.build()
    return _native.lib()


def test_header_symbols_are_exported(lib):
    names = declared_functions()
    assert len(names) >= 20
    for n in names:
        assert hasattr(lib, n), f"{n} is declared in vlgpu.h but not exported"


def test_binding_table_matches_header():
    from vectorlink_gpu import _native

    assert sorted(_native._SIGNATURES) == declared_functions()


def test_sentinels_match_reference_constants():
    from vectorlink_gpu.constants import MAXFLOAT, MAXINT, PRIMES_HOST

    text = open(HEADER).read()
    assert f"#define VL_MAXINT {MAXINT}" in text
    assert "#define VL_MAXFLOAT 3.4028e37f" in text and MAXFLOAT == 3.4028e37
    assert "#define VL_ERR_STATE (-4)" in text
    assert PRIMES_HOST.numel() == 965 and int(PRIMES_HOST[0]) == 10000349 and int(PRIMES_HOST[964]) == 1999


def test_host_side_validation(lib):
    from vectorlink_gpu import _native as nv

    one = C.c_void_p(256)  # never dereferenced: every call below is rejected on the host
    # insert that does not fit the queue
    rc = lib.vl_queue_insert(one, one, 4, 10, 8, one, one, 5, None, 0, None, None)
    assert rc == -1 and b"does not fit" in lib.vl_last_error()
    with pytest.raises(ValueError):
        nv.check(rc)
    # rows beyond what the LDS sort holds
    assert lib.vl_queue_sort(one, one, 4, 5000, None) == -1
    # negative sizes, null pointers
    assert lib.vl_gather_distances(one, -1, one, 10, 8, one, 4, one, None) == -1
    assert lib.vl_gather_distances(None, 3, one, 10, 8, one, 4, one, None) == -1
    assert lib.vl_prune(one, one, 10, 4, one, one, None) == -1  # in-place prune is refused
    # beam parameters: queue too small for one round of candidates, workspace too small
    p = nv.BeamParams(n_rows=10, dim=8, n_vectors=100, width=8, queue_capacity=20, queue_length=8, beam_size=4,
                      parallel_visit_count=4, visit_queue_factor=3, exclude_factor=5, speculative_readahead=5,
                      excl_cols=0, flags=0)
    assert lib.vl_beam_workspace_bytes(C.byref(p)) == -1
    p.queue_capacity = 8 + 32
    need = lib.vl_beam_workspace_bytes(C.byref(p))
    assert need > 0 and need % 256 == 0
    rc = lib.vl_closest_vectors(C.byref(p), one, one, one, one, one, None, one, need - 1, None)
    assert rc == -3 and b"workspace" in lib.vl_last_error()
    # exact kNN limits
    assert lib.vl_knn_workspace_bytes(10, 100, 8, 17) == -1
    assert lib.vl_knn_workspace_bytes(10, 100, 6, 10) == -1
    assert lib.vl_knn_workspace_bytes(10, 100, 8, 10) > 0
    # empty problems succeed without touching a device
    assert lib.vl_queue_sort(None, None, 0, 16, None) == 0
    assert lib.vl_search_from_seeds(None, 0, 8, None, 4, None, 10, 4, None, 10, None, None, None) == 0


def test_knn_workspace_of_many_queries(lib):
    """The buffers of the bfloat16 filter (16 KB a query and more) are for a bounded number of queries."""
    few, many = (lib.vl_knn_workspace_bytes(n, 1_000_000, 768, 10) for n in (1 << 17, 1 << 23))
    assert 0 < few and many - few < 1024 * ((1 << 23) - (1 << 17))  # 4 lists of 10 keys and two words a query


@pytest.mark.parametrize("metric", [0, 1])
def test_knn_workspace_serves_both_metrics(lib, metric):
    """What vl_knn_workspace_bytes asks for admits the form that a call with any amount of it would take."""
    import random

    rng = random.Random(11)
    sizes = [(200, 3_000_000, 512, 10), (500, 3_000_000, 512, 10), (200, 9_000_000, 128, 10), (200, 9_000_000, 256, 10),
             (200, 9_000_000, 320, 4)]
    sizes += [(rng.randint(1, 20_000), rng.randint(100, 20_000_000), 4 * rng.randint(1, 600), rng.randint(1, 16))
              for _ in range(300)]
    for s in sizes:
        assert lib.vl_knn_form(*s, metric, lib.vl_knn_workspace_bytes(*s)) == lib.vl_knn_form(*s, metric, 1 << 60), s


def test_calls_that_cannot_use_the_sketch_are_sized_as_without_it(lib):
    """The distance cache of rows that meet most vectors again is larger, and with the sketch they have to ask for more of
    them.  A call whose metric, row length or form rules the sketch out is judged as one without it: the sketch's own part of
    the workspace is all that the flag adds, for tables of every size."""
    from vectorlink_gpu import _native as nv

    def size(n, flags, **kw):
        p = dict(n_rows=100, dim=64, n_vectors=n, width=64, queue_capacity=64 + 256, queue_length=64, beam_size=64,
                 parallel_visit_count=4, visit_queue_factor=3, exclude_factor=5, speculative_readahead=5, excl_cols=0,
                 flags=flags, metric=0)
        p.update(kw)
        return lib.vl_beam_workspace_bytes(C.byref(nv.BeamParams(**p)))

    for kw, flags in ((dict(metric=1), 0), (dict(dim=50), 0), (dict(), 1), (dict(), 2)):
        adds = {size(n, 16 | flags, **kw) - size(n, flags, **kw) for n in (500, 5000, 15_000, 18_000, 24_000, 60_000, 1_000_000)}
        assert len(adds) == 1 and adds.pop() > 0, (kw, flags)


def test_the_filter_is_left_out_where_the_tiles_are_sooner(lib):
    """Short calls stay with the float32 tiles; long ones go through the filter, and so does any if asked for."""
    few, tiles, filt = 1, 0, 2
    form = lambda *s: lib.vl_knn_form(*s, 0, 1 << 60)
    assert form(300, 4096, 64, 10) == tiles and form(10_000, 4096, 64, 10) == tiles
    assert form(1500, 6000, 768, 10) == tiles and form(300, 32_768, 64, 1) == tiles and form(129, 12_000, 20, 16) == tiles
    assert form(10_000, 32_768, 64, 4) == filt and form(1000, 32_768, 1536, 16) == filt
    assert form(10_000, 1_000_000, 768, 10) == filt and form(300, 150_000, 64, 10) == filt and form(10_000, 6000, 768, 10) == filt
    assert form(32, 32_768, 64, 1) == few
    for s in [(300, 4096, 64, 10), (32, 32_768, 64, 1), (1, 4096, 4, 1)]:
        for metric in (0, 1):
            need = lib.vl_knn_metric_workspace_bytes(*s, metric + 256)
            assert lib.vl_knn_form(*s, metric + 256, need) == filt and lib.vl_knn_form(*s, metric + 256, need - 1) != filt
    assert lib.vl_knn_form(300, 4000, 64, 10, 256, 1 << 60) == tiles
    for metric in (2, 255, 258, -1, 512):
        assert lib.vl_knn_form(300, 4096, 64, 10, metric, 1 << 60) < 0
        assert lib.vl_knn_metric_workspace_bytes(300, 4096, 64, 10, metric) < 0


def test_cpu_tensors_are_refused():
    import torch

    from vectorlink_gpu import Queue
    from vectorlink_gpu.kernels import calculate_distances

    v = torch.zeros((4, 8), dtype=torch.float32)
    b = torch.zeros((4, 2), dtype=torch.int32)
    with pytest.raises(RuntimeError):
        calculate_distances(v, b)
    q = Queue(2, 2, 6, device="cpu")
    with pytest.raises(RuntimeError):
        q.insert(torch.zeros((2, 2), dtype=torch.int32), torch.zeros((2, 2), dtype=torch.float32))


def test_library_is_not_older_than_its_sources():
    """The built library travels with the tree; one that predates an edit of its sources would be
    tested in their place."""
    from vectorlink_gpu import _native

    built = os.path.getmtime(_native.LIB_PATH)
    csrc = os.path.join(ROOT, "vectorlink-gpu_amd", "csrc")
    sources = [os.path.join(csrc, f) for f in os.listdir(csrc)] + [HEADER]
    stale = [os.path.basename(s) for s in sources if os.path.getmtime(s) > built]
    assert not stale, f"rebuild libvlgpu.so (python vectorlink-gpu_amd/build.py): newer sources {stale}"
