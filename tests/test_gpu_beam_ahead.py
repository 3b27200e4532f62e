"""What closest_vectors gives a call ahead of its loop: the look at the graph, the workspace, and builds that say what their loops
are (vectorlink_gpu/ann.py)."""
import numpy as np
import pytest
import torch

from oracle import oracle as orc
from test_gpu_beam_table import config, dev, same, search, vectors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,width", [(2, 1), (3, 2), (64, 5), (65, 24), (1000, 64), (5003, 128)])
def test_the_graph_that_builds_start_from(n, width):
    from vectorlink_gpu.ann import _circulant_graph

    ids = orc.generate_circulant_beams(n, orc.primes(width))
    assert _circulant_graph(dev(ids))
    for (node, k) in ((0, 0), ((63 * (n - 1)) // 64 + 1, width - 1)):  # the first and the last list that are read
        other = ids.copy()
        other[node, k] = (other[node, k] + 1) % n if n > 2 else 7
        assert not _circulant_graph(dev(other))
    empty = ids.copy()
    empty[:, 0] = 0x7FFFFFFF
    assert not _circulant_graph(dev(empty)) and not _circulant_graph(dev(ids[:1]))


def test_a_captured_call_is_not_looked_at(monkeypatch):
    """It is refused by the loop, which says why; waiting for the stream would end the capture."""
    from vectorlink_gpu import _native as nv
    from vectorlink_gpu.ann import _circulant_graph

    beams = dev(orc.generate_circulant_beams(100, orc.primes(8)))
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    monkeypatch.setattr(nv, "lib", None)  # (no launch)
    assert not _circulant_graph(beams)


def test_only_the_graph_of_a_first_loop_is_given_the_large_workspace(monkeypatch):
    from vectorlink_gpu import ann

    (n, rows) = (70_001, 400)
    v = dev(vectors(n, 64))
    c = config(beam_size=32)
    ids = orc.generate_circulant_beams(n, orc.primes(64))
    other = np.random.default_rng(5).integers(0, n, ids.shape).astype(np.int32)
    (asked, reserve) = ([], ann._Workspace.reserve)
    monkeypatch.setattr(ann._Workspace, "reserve", lambda self, nbytes, device: asked.append(nbytes) or reserve(self, nbytes, device))
    for beams in (ids, other):
        same(search(v, rows, dev(beams), ids[:rows], c, True, 0), search(v, rows, dev(beams), ids[:rows], c, True, ann.BEAM_NO_TABLE))
    assert asked[0] > asked[1] == asked[2] == asked[3]


def test_later_loops_of_a_build_are_not_looked_at(monkeypatch):
    from vectorlink_gpu import ann

    (looked, flags, search_) = ([], [], ann.closest_vectors)
    monkeypatch.setattr(ann, "_circulant_graph", lambda beams: looked.append(1))
    monkeypatch.setattr(ann, "ann_calculate_recall", lambda *a, **k: (0, 0.0))  # (a recall of 1 ends a build)
    monkeypatch.setattr(ann, "closest_vectors", lambda *a, **k: flags.append(k["flags"]) or search_(*a, **k))
    ann.ANN(dev(vectors(6007, 384)), beam_size=48, beam_queue_factor=2)
    assert flags == [ann.BEAM_MANY_ITERATIONS | ann.BEAM_NO_CACHE, ann.BEAM_KNOWN_GRAPH, ann.BEAM_KNOWN_GRAPH]
    assert not looked


def test_a_size_that_cannot_be_had_is_asked_for_once(monkeypatch):
    """... until the workspaces are let go; the smaller block stays where it is meanwhile."""
    from vectorlink_gpu import ann

    (n, rows) = (3000, 200)
    v = dev(vectors(n, 24))
    beams = dev(orc.generate_circulant_beams(n, orc.primes(32)))
    seeds = orc.generate_circulant_beams(n, orc.primes(32))[:rows]
    c = config(beam_size=16, exclude_factor=2)
    want = search(v, rows, beams, seeds, c, True, ann.BEAM_NO_TABLE | ann.BEAM_NO_CACHE)
    (made, most, empty) = ([], 1 << 21, torch.empty)
    ann.release_workspaces()

    def no_room(size, *a, **k):
        if k.get("dtype") == torch.uint8:
            made.append(size)
            if size > most:
                raise torch.OutOfMemoryError("no room")
        return empty(size, *a, **k)

    monkeypatch.setattr(ann.torch, "empty", no_room)
    for _ in range(3):
        same(search(v, rows, beams, seeds, c, True, ann.BEAM_TABLE | ann.BEAM_NO_CACHE, table=False), want)
    assert len(made) == 2 and made[1] <= most < made[0]
    ann.release_workspaces()
    same(search(v, rows, beams, seeds, c, True, ann.BEAM_TABLE | ann.BEAM_NO_CACHE, table=False), want)
    assert made[2:] == made[:2]
    ann.release_workspaces()


def test_as_much_again_is_left_for_others(monkeypatch):
    """10,000 of 100,000 x 64: 4 GiB of distances."""
    from vectorlink_gpu import ann

    (n, rows) = (100_000, 10_000)
    v = dev(vectors(n, 64))
    c = config(beam_size=8, beam_queue_factor=2, exclude_factor=1)
    beams = dev(orc.generate_circulant_beams(n, orc.primes(16)))
    seeds = orc.generate_circulant_beams(n, orc.primes(16))[:rows]
    want = search(v, rows, beams, seeds, c, True, ann.BEAM_NO_TABLE)
    stream = torch.cuda.current_stream()

    def block(room, table=False):
        ann.release_workspaces()
        monkeypatch.setattr(ann, "_room", lambda device: room)
        same(search(v, rows, beams, seeds, c, True, ann.BEAM_TABLE, table=table), want)
        return ann._WORKSPACES[("cuda:0", int(stream.cuda_stream))].tensor.numel()

    large = block(1 << 40, True)
    small = block(0)
    assert large - small > 3 << 30
    assert block(small + 2 * (large - small), True) == large and block(small + 2 * (large - small) - 1) == small
    # a block that is there counts: it goes before a larger one is asked for
    monkeypatch.setattr(ann, "_room", lambda device: 2 * (large - small))
    same(search(v, rows, beams, seeds, c, True, ann.BEAM_TABLE), want)
    assert ann._WORKSPACES[("cuda:0", int(stream.cuda_stream))].tensor.numel() == large
    ann.release_workspaces()


def test_room_is_what_is_free_and_what_torch_keeps():
    from vectorlink_gpu import ann

    device = torch.device("cuda:0")
    torch.cuda.synchronize()
    before = ann._room(device)
    x = torch.empty(3 << 30, dtype=torch.uint8, device=device)
    assert abs(before - (3 << 30) - ann._room(device)) < 64 << 20
    del x
    assert abs(before - ann._room(device)) < 64 << 20  # (torch keeps the block)
