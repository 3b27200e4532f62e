"""The forms of the fused beam step against the oracle's loop: one iteration per launch, several per launch, and whatever
the library picks.  A launch's LDS depends on the rows of the call and on the iteration, so the row counts go from one
workgroup on the chip to more than it holds at once.  A row has 256 threads up to two rows per compute unit (512), where it
is aligned with at most 128 candidates, up to six (1,536) otherwise (four, 1,024, from 769 columns on), and with more than
320 candidates in an iteration; beyond that it has 128, and then a wavefront looks at its candidates in every second set of
64 instead of every fourth."""
import numpy as np
import pytest
import torch

from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")


def bits(t):
    return t.cpu().numpy().view(np.uint32)


# rows of the call, vectors, columns, degree, build queue factor, visited-list factor
SHAPES = [
    (1, 300, 24, 6, 2, 5),
    (257, 700, 52, 8, 2, 5),      # one row more than compute units
    (700, 700, 256, 16, 2, 5),    # rows of 1 KiB: the sketch
    (900, 900, 16, 24, 3, 2),     # 288 candidates in 256 threads, a visited list that fills up
    (1600, 1600, 16, 24, 3, 2),   # the same in 128 threads
    (1600, 1600, 12, 65, 1, 2),   # 260 and 320 candidates in 128 threads: a second and third pass over two sets of 64, begun and full
    (1600, 1600, 12, 40, 2, 2),
    (1600, 1600, 10, 65, 1, 2),   # the same, rows that are not aligned
    (1600, 1600, 10, 40, 2, 2),
    (2300, 2300, 12, 4, 2, 5),    # more rows than the chip holds at once
    (40, 1200, 8, 64, 2, 5),      # 512 candidates, 256 threads
    (40, 1200, 8, 129, 1, 2),     # 516, 580 and 640 in 256 threads: a second pass, with one set of it and with both
    (40, 1200, 9, 145, 1, 2),
    (40, 1200, 8, 80, 2, 2),
    (40, 1200, 9, 80, 2, 2),
]


@pytest.mark.parametrize("rows,n,dim,beam,bqf,ef", SHAPES)
def test_forms_agree_with_the_oracle(rows, n, dim, beam, bqf, ef):
    print(f"beam forms rows={rows} n={n} dim={dim} beam={beam}", flush=True)
    from vectorlink_gpu import Queue
    from vectorlink_gpu.ann import BEAM_NO_WINDOWS, BEAM_WINDOWS, closest_vectors, excluding_self
    from vectorlink_gpu.kernels import build_sketch

    rng = np.random.default_rng(rows + dim)
    v = rng.standard_normal((n, dim)).astype(np.float32)
    v /= np.linalg.norm(v, axis=1, keepdims=True)
    c = dict(orc.DEFAULT_CONFIG)
    c.update(beam_size=beam, beam_queue_factor=bqf, exclude_factor=ef)
    ql = beam * bqf
    beams = orc.generate_circulant_beams(n, orc.primes(ql))
    d = orc.calculate_distances(v, beams)
    want = orc.Queue(rows, ql, ql + ql * 4)
    want.insert(beams[:rows], d[:rows])
    t_want = orc.closest_vectors(v[:rows], want, v, beams, c, orc.excluding_self(0, rows))
    gv, gb, gd = dev(v), dev(beams), dev(d)
    for sketch in ([None, build_sketch(gv)] if dim >= 256 else [None]):
        for flags in (0, BEAM_NO_WINDOWS, BEAM_WINDOWS):
            q = Queue(rows, ql, ql + ql * 4)
            q.insert(gb[:rows], gd[:rows])
            t = closest_vectors(gv[:rows], q, gv, gb, c, excluding_self(0, rows), flags=flags, sketch=sketch)
            assert t == t_want, (flags, sketch is not None)
            assert np.array_equal(q.indices.cpu().numpy()[:, :ql], want.indices[:, :ql]), (flags, sketch is not None)
            assert np.array_equal(bits(q.distances)[:, :ql], want.distances[:, :ql].view(np.uint32)), flags


@pytest.mark.parametrize("rows,width,dim",
                         [(70, w, d) for d in (40, 128, 130, 300) for w in (1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 96, 97)] +
                         [(70, w, d) for d in (40, 130) for w in (127, 129, 145, 160, 161)] +
                         [(1600, w, d) for d in (40, 130) for w in (15, 16, 17, 32, 33, 64, 65, 79, 80)])
def test_candidate_counts_around_the_sets_of_64(rows, width, dim):
    """Four neighbour lists of `width` ids: the last set of 64 candidates of a wavefront, and its last pair of sets, full,
    short by one and begun; 70 rows have 256 threads, 1,600 have 128.  Lists share ids and have empty places, so what is left to
    fetch lies unevenly among the sets."""
    print(f"beam candidates rows={rows} width={width} dim={dim}", flush=True)
    from vectorlink_gpu import Queue
    from vectorlink_gpu.ann import BEAM_NO_CACHE, BEAM_NO_WINDOWS, closest_vectors

    rng = np.random.default_rng(width * 1000 + dim)
    (n, length) = (max(500, rows), 24)
    v = rng.standard_normal((n, dim)).astype(np.float32)
    v /= np.linalg.norm(v, axis=1, keepdims=True)
    table = rng.integers(0, n, (n, width)).astype(np.int32)
    table[rng.random((n, width)) < 0.1] = orc.MAXINT
    table[::7, : width // 2] = table[0, : width // 2]
    c = dict(orc.DEFAULT_CONFIG)
    c.update(beam_size=12)
    seeds = np.stack([rng.choice(n, length, replace=False) for _ in range(rows)]).astype(np.int32)
    d = orc.gather_distances(v[:rows], v, seeds)
    want = orc.Queue(rows, length, length + 4 * max(width, 6))
    want.insert(seeds, d)
    t_want = orc.closest_vectors(v[:rows], want, v, table, c, None)
    for flags in (0, BEAM_NO_WINDOWS, BEAM_NO_CACHE):
        q = Queue(rows, length, length + 4 * max(width, 6))
        q.insert(dev(seeds), dev(d))
        assert closest_vectors(dev(v[:rows]), q, dev(v), dev(table), c, flags=flags) == t_want, flags
        assert np.array_equal(q.indices.cpu().numpy()[:, :length], want.indices[:, :length]), flags
        assert np.array_equal(bits(q.distances)[:, :length], want.distances[:, :length].view(np.uint32)), flags


# lengths around a multiple of 4 at the edges of the shapes (16, 32, 64, 96, 128, 192, 256, 320, 384, 448, 512 chunks)
ODD_DIMS = [1, 3, 5, 50, 62, 65, 127, 130, 253, 259, 383, 386, 511, 514, 766, 1022, 1026, 1279, 1534, 1790, 2045, 2049]


@pytest.mark.parametrize("n,dim,metric", [(90, d, m) for d in ODD_DIMS for m in ("cosine", "l2")] +
                         [(1600, d, "cosine" if i % 2 else "l2") for i, d in
                          enumerate([3, 50, 62, 65, 127, 130, 253, 383, 511, 766, 1022, 1279, 1534, 1790, 2045, 2049])])
def test_rows_of_odd_length(n, dim, metric):
    """Distances and the loop on rows that do not start on 16-byte boundaries; the last row ends with the table.  90 rows have
    256 threads, 1,600 have 128."""
    print(f"odd rows n={n} dim={dim} {metric}", flush=True)
    from vectorlink_gpu import Queue
    from vectorlink_gpu.ann import closest_vectors, excluding_self
    from vectorlink_gpu.kernels import gather_distances

    rng = np.random.default_rng(dim)
    beam = 6
    v = rng.standard_normal((n, dim)).astype(np.float32)
    if metric == "cosine":
        v /= np.linalg.norm(v, axis=1, keepdims=True)
    c = dict(orc.DEFAULT_CONFIG)
    c.update(beam_size=beam, beam_queue_factor=2, metric=metric)
    ql = 2 * beam
    beams = orc.generate_circulant_beams(n, orc.primes(ql))
    ids = np.concatenate([beams, np.full((n, 1), n - 1, np.int32)], axis=1)
    with orc.metric(metric):
        d = orc.gather_distances(v, v, ids)
        want = orc.Queue(n, ql, ql + ql * 4)
        want.insert(beams, np.ascontiguousarray(d[:, :ql]))
        t_want = orc.closest_vectors(v, want, v, beams, c, orc.excluding_self(0, n))
    assert np.array_equal(bits(gather_distances(dev(v), dev(v), dev(ids), metric=metric)), d.view(np.uint32))
    q = Queue(n, ql, ql + ql * 4)
    q.insert(dev(beams), dev(d[:, :ql]))
    assert closest_vectors(dev(v), q, dev(v), dev(beams), c, excluding_self(0, n)) == t_want
    assert np.array_equal(q.indices.cpu().numpy()[:, :ql], want.indices[:, :ql])
    assert np.array_equal(bits(q.distances)[:, :ql], want.distances[:, :ql].view(np.uint32))


@pytest.mark.parametrize("rows,dim", [(r, d) for r in (2560, 2561, 3072, 3073) for d in (390, 902)] +
                         [(3073, d) for d in (602, 1182, 1410, 1702, 2045)])
def test_rows_of_odd_length_in_one_round(rows, dim):
    """From 385 columns on, ten, eleven, twelve and thirteen rows per compute unit take different forms of the fetch."""
    print(f"odd rows dim={dim} rows={rows}", flush=True)
    from vectorlink_gpu import Queue
    from vectorlink_gpu.ann import BEAM_NO_WINDOWS, closest_vectors, excluding_self

    rng = np.random.default_rng(rows + dim)
    (beam, ql) = (3, 6)
    v = rng.standard_normal((rows, dim)).astype(np.float32)
    v /= np.linalg.norm(v, axis=1, keepdims=True)
    c = dict(orc.DEFAULT_CONFIG)
    c.update(beam_size=beam, beam_queue_factor=2, exclude_factor=3)
    beams = orc.generate_circulant_beams(rows, orc.primes(ql))
    d = orc.calculate_distances(v, beams)
    want = orc.Queue(rows, ql, ql + ql * 4)
    want.insert(beams, d)
    t_want = orc.closest_vectors(v, want, v, beams, c, orc.excluding_self(0, rows))
    for flags in (0, BEAM_NO_WINDOWS):
        q = Queue(rows, ql, ql + ql * 4)
        q.insert(dev(beams), dev(d))
        assert closest_vectors(dev(v), q, dev(v), dev(beams), c, excluding_self(0, rows), flags=flags) == t_want
        assert np.array_equal(q.indices.cpu().numpy()[:, :ql], want.indices[:, :ql])
        assert np.array_equal(bits(q.distances)[:, :ql], want.distances[:, :ql].view(np.uint32))


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
def test_odd_rows_with_values_that_are_not_finite(value):
    """A row of 7 elements is read as elements 0-3 and 3-6: element 3 counts once, whatever it is."""
    from vectorlink_gpu.kernels import gather_distances

    v = np.linspace(-1, 1, 63, dtype=np.float32).reshape(9, 7)
    v[4, 3] = value
    ids = np.tile(np.arange(9, dtype=np.int32), (9, 1))
    want = orc.gather_distances(v, v, ids)
    got = gather_distances(dev(v), dev(v), dev(ids)).cpu().numpy()
    assert np.array_equal(got, want, equal_nan=True)


@pytest.mark.parametrize("n,dim,windows", [(45_000, 768, True), (45_000, 772, False), (20_000, 768, False)])
def test_which_calls_with_a_sketch_take_several_iterations_per_launch(n, dim, windows):
    """More than 32 MiB of sketch and at most 768 columns: the launches of a call tell."""
    print(f"sketch windows n={n} dim={dim}", flush=True)
    from vectorlink_gpu import Queue, _native
    from vectorlink_gpu.ann import closest_vectors, excluding_self
    from vectorlink_gpu.kernels import build_sketch, calculate_distances
    from vectorlink_gpu.utils import generate_circulant_beams, primes

    gen = torch.Generator(device="cuda").manual_seed(n + dim)
    v = torch.nn.functional.normalize(torch.randn((n, dim), generator=gen, device="cuda"), dim=1)
    (rows, ql) = (64, 32)
    beams = generate_circulant_beams(n, primes(ql, "cuda"))
    q = Queue(rows, ql, ql + ql * 4, device="cuda")
    q.insert(beams[:rows], calculate_distances(v, beams)[:rows])
    c = dict(orc.DEFAULT_CONFIG)
    c.update(beam_size=16, beam_queue_factor=2)
    before = _native.lib().vl_beam_launches()
    t = closest_vectors(v[:rows], q, v, beams, c, excluding_self(0, rows, ql, "cuda"), sketch=build_sketch(v))
    launches = _native.lib().vl_beam_launches() - before
    assert t >= 10  # (one launch more than needed is on its way when the loop ends, of five iterations or of one)
    assert (launches < t) == windows, (launches, t)


# the cache's size: a slot for every vector and a quarter (819 vectors fit 1,024 slots, 820 do not), 1,024 slots for 3,000
# vectors of up to 128 columns, which collide; 128 threads a row up to iteration 25 and 256 from there on (eleven rows per
# compute unit, of which LDS holds eleven, then ten), 256 throughout (twelve), 128 up to iteration 5 (fourteen, and LDS for ten,
# then nine)
@pytest.mark.parametrize("rows,n,dim,beam,ef", [(60, 819, 40, 16, 5), (60, 820, 40, 16, 5), (60, 3000, 128, 4, 2),
                                                (60, 3000, 132, 4, 2), (2816, 2817, 8, 64, 1), (2817, 2817, 8, 64, 1),
                                                (3400, 3401, 8, 72, 1)])
def test_cache_sizes_and_threads_per_row(rows, n, dim, beam, ef):
    print(f"beam cache and threads rows={rows} n={n} dim={dim} beam={beam}", flush=True)
    from vectorlink_gpu import Queue
    from vectorlink_gpu.ann import BEAM_NO_CACHE, BEAM_NO_WINDOWS, closest_vectors

    rng = np.random.default_rng(n + dim)
    v = rng.standard_normal((n, dim)).astype(np.float32)
    v /= np.linalg.norm(v, axis=1, keepdims=True)
    c = dict(orc.DEFAULT_CONFIG)
    c.update(beam_size=beam, exclude_factor=ef)
    (length, cap) = (2 * beam, 2 * beam + 4 * beam)
    beams = orc.generate_circulant_beams(n, orc.primes(beam))
    seeds = np.ascontiguousarray(orc.generate_circulant_beams(n, orc.primes(length))[:rows])
    d = orc.gather_distances(v[:rows], v, seeds)
    want = orc.Queue(rows, length, cap + length)
    want.insert(seeds, d)
    t_want = orc.closest_vectors(v[:rows], want, v, beams, c, None)
    for flags in (0, BEAM_NO_WINDOWS, BEAM_NO_CACHE):
        q = Queue(rows, length, cap + length)
        q.insert(dev(seeds), dev(d))
        assert closest_vectors(dev(v[:rows]), q, dev(v), dev(beams), c, flags=flags) == t_want, flags
        assert np.array_equal(q.indices.cpu().numpy()[:, :length], want.indices[:, :length]), flags
        assert np.array_equal(bits(q.distances)[:, :length], want.distances[:, :length].view(np.uint32)), flags


# sized for a table of fewer vectors, of more vectors (whose rows of up to 128 columns meet few vectors again and take a small
# cache), of longer rows; and by what a table of one vector needs
@pytest.mark.parametrize("dim,sized", [(768, dict(n_vectors=3000)), (768, dict(n_vectors=1)), (64, dict(n_vectors=1_000_000)),
                                       (64, dict(dim=100, n_vectors=400_000)), (132, dict(dim=64, n_vectors=1_000_000))])
def test_a_workspace_sized_for_another_table_serves(dim, sized):
    print(f"workspace of another table dim={dim} {sized}", flush=True)
    import ctypes as C

    from vectorlink_gpu import Queue, _native as nv
    from vectorlink_gpu.ann import _beam_params

    rng = np.random.default_rng(dim)
    (n, rows, beam) = (4000, 30, 32)
    v = rng.standard_normal((n, dim)).astype(np.float32)
    v /= np.linalg.norm(v, axis=1, keepdims=True)
    c = dict(orc.DEFAULT_CONFIG)
    c.update(beam_size=beam)
    (length, cap) = (2 * beam, 6 * beam)
    gv, gb = dev(v), dev(orc.generate_circulant_beams(n, orc.primes(beam)))
    seeds = orc.generate_circulant_beams(n, orc.primes(length))[:rows]
    d = dev(orc.gather_distances(v[:rows], v, seeds))

    def run(give):
        """Result of a call with `give` of the bytes that its own parameters ask for, and what lies behind them."""
        q = Queue(rows, length, cap + length)
        q.insert(dev(seeds), d)
        p = _beam_params(rows, dim, n, beam, q, c, 0, 0)
        need = nv.lib().vl_beam_workspace_bytes(C.byref(p))
        have = give(p) or need
        ws = torch.full((max(have, need) + 256,), 0xA5, dtype=torch.uint8, device="cuda:0")
        rc = nv.lib().vl_closest_vectors(C.byref(p), nv.ptr(gv), nv.ptr(gv), nv.ptr(gb), nv.ptr(q.indices),
                                         nv.ptr(q.distances), None, nv.ptr(ws), have, nv.stream())
        assert bool((ws[have:] == 0xA5).all())
        return have, need, (rc, q.indices.cpu().numpy()[:, :length], bits(q.distances)[:, :length])

    def other(p, **kw):
        o = type(p)(**{f: getattr(p, f) for f, _ in p._fields_})
        for k, x in kw.items():
            setattr(o, k, x)
        return nv.lib().vl_beam_workspace_bytes(C.byref(o))

    want = run(lambda p: None)[2]
    have, need, got = run(lambda p: other(p, **sized))
    assert have < need and got[0] == want[0] > 0
    assert np.array_equal(got[1], want[1]) and np.array_equal(got[2], want[2])
    assert run(lambda p: other(p, n_vectors=1) - 1)[2][0] == -3
