"""The record layout and cell tables made on the device against the host's
(``navi_relayout_leaves``, ``navi_build_cell_table``), bit for bit, and the DAGs that the
device leaves to the host."""

import ctypes

import numpy as np
import pytest
import torch

from navi_amd import _native, multiscene
from navi_amd import scenes as S
from navi_amd.multiscene import ResidentScenes

pytestmark = pytest.mark.gpu

LEAF = 1 << 63
VOID = 0


def _leaf(semantic, bits):
    return LEAF | semantic << 16 | bits


def _node(mask, base):
    return mask << 55 | base


def _chain(records, last):
    """A chain of ``records`` nodes, each the only child of the one above, over ``last``."""
    words = []
    for k in range(records):
        words += [_node(1 << (k % 8), 2 * k + 1), 2 * k + 2]
    return words + [last]


def _hand_made():
    leaf = _leaf(3, 0x2E66)
    return {
        # every octant a leaf, void octants, a child index and a table word past the end
        "one_record": [_node(0xFF, 1), *[9] * 8, leaf],
        "void_octants": [_node(0b10010010, 1), 4, 4, 4, leaf],
        "no_children": [_node(0, 1)],
        "bad_child": [_node(0b11, 1), 3, 77, leaf],
        "bad_table": [_node(0xFF, 1), 3, 3, leaf],
        "negative_leaf": [_node(0b11, 1), 3, 4, leaf, _leaf(0, 0x8001)],
        # one level's children named by several parents, the first in octant order wins
        "shared": [_node(0b1011, 1), 6, 4, 6, _node(0b1, 8), 0, _node(0b101, 9), 0, 12, 11, 12, _node(0b1, 8), leaf],
        "levels_31": _chain(31, leaf),
        # left to the host
        "levels_32": _chain(32, leaf),
        "one_leaf": [leaf],
        "table_leaf": [_node(0b11, 1), 3, 4, leaf, _leaf(0x7FFF, 0x2E66)],
        "table_leaf_high": [_node(0b11, 1), 3, 4, leaf, _leaf(0x8001, 0x2E66)],
        "cycle": [_node(0b11, 1), 3, 0, leaf],
        "two_depths": [_node(0b11, 1), 3, 5, _node(0b1, 7), 0, _node(0b1, 8), 0, 5, 9, leaf],
    }


HOST_ONLY = ("levels_32", "one_leaf", "table_leaf", "table_leaf_high", "cycle", "two_depths")


def _compare(scenes, monkeypatch, on_device, **kw):
    want = ResidentScenes(scenes, "cpu", **kw)
    monkeypatch.setattr(multiscene, "DEVICE_MIN_WORDS", 0)
    if on_device:
        def refuse(self, *a):
            raise AssertionError("converted on the host")
        monkeypatch.setattr(ResidentScenes, "_layout_on_host", refuse)
    else:
        layout = ResidentScenes._layout_on_device
        monkeypatch.setattr(ResidentScenes, "_layout_on_device",
                            lambda self, *a: pytest.fail("converted on the device") if layout(self, *a) else False)
    for source in (lambda w: w, lambda w: torch.from_numpy(w.view(np.int64)).cuda()):
        got = ResidentScenes([(source(w), lo, hi) for w, lo, hi in scenes], "cuda", **kw)
        assert got.relaid_ok and got.table_depth == want.table_depth and got.n_records == want.n_records
        assert got.record_counts == want.record_counts and got.word_counts == want.word_counts
        for name in ("records", "cell_tables", "relaid_table", "table", "pool", "leaves"):
            a, b = getattr(got, name), getattr(want, name)
            assert (a is None) == (b is None) and (a is None or torch.equal(a.cpu(), b)), name


@pytest.mark.parametrize("name", list(_hand_made()))
def test_hand_made_dags(name, monkeypatch):
    words = np.array(_hand_made()[name], np.uint64)
    _compare([(words, [0.0] * 3, [1.0] * 3)], monkeypatch, name not in HOST_ONLY)


@pytest.mark.parametrize("depth", [4, 5, 6, 7, None])
def test_compiled_scenes(depth, monkeypatch):
    """Pools of scenes whose levels fill less than one workgroup's round and many rounds
    (512^3: 100 K records on the last level, 800 K candidates on 1024 workgroups)."""
    scenes = []
    for family, seed, resolution in (("box_room", 1, 64), ("rooms", 2, 256), ("cluttered", 3, 512)):
        scene = getattr(S, family)(seed=seed, resolution=resolution)
        scene.compile(threads=8)
        scenes.append((scene.words, scene.bbox_min_list, list(scene.bbox_max)))
    _compare(scenes, monkeypatch, True, table_depth=depth)


@pytest.mark.parametrize("names", [("table_leaf", "room", "shared", "room"), ("room", "one_leaf", "two_depths", "room"),
                                   ("one_record", "table_leaf", "room", "table_leaf_high"), ("one_leaf", "one_leaf"),
                                   ("cycle", "table_leaf_high")])
def test_pools_of_both_conversions(names, monkeypatch):
    """A pool whose scenes are covered by the device, left to the host, or both: the same
    arrays as an all-host pool, and the host converts only what is left to it."""
    room = S.box_room(seed=1, resolution=64)
    room.compile(threads=8)
    dags = {k: np.array(w, np.uint64) for k, w in _hand_made().items()} | {"room": room.words}
    scenes = [(dags[name], [0.0] * 3, [1.0 + k] * 3) for k, name in enumerate(names)]
    want = ResidentScenes(scenes, "cpu")
    monkeypatch.setattr(multiscene, "DEVICE_MIN_WORDS", 0)
    host = ResidentScenes._layout_on_host
    converted = []
    monkeypatch.setattr(ResidentScenes, "_layout_on_host",
                        lambda self, entry, chunk, *a: converted.append(1) or host(entry, chunk, *a))
    for keep_words in (False, True):
        converted.clear()
        got = ResidentScenes(scenes, "cuda", keep_words=keep_words)
        assert len(converted) == sum(name in HOST_ONLY for name in names)
        assert got.relaid_ok and got.n_records == want.n_records and got.n_leaves == want.n_leaves
        assert got.record_counts == want.record_counts and got.table_depth == want.table_depth
        for name in ("records", "cell_tables", "relaid_table", "table", "leaves"):
            a, b = getattr(got, name), getattr(want, name)
            assert (a is None) == (b is None) and (a is None or torch.equal(a.cpu(), b)), name


@pytest.mark.parametrize("n,on_host", [(1, True), ((1 << 14) - 1, True), (1 << 14, False)])
def test_small_scenes_are_converted_on_the_host(n, on_host, monkeypatch):
    host = ResidentScenes._layout_on_host
    converted = []
    monkeypatch.setattr(ResidentScenes, "_layout_on_host",
                        lambda self, entry, chunk, *a: converted.append(1) or host(entry, chunk, *a))
    words = np.zeros(n, np.uint64)
    words[0] = _node(0, 1)
    for source in (words, torch.from_numpy(words.view(np.int64)).cuda()):
        converted.clear()
        got = ResidentScenes([(source, [0.0] * 3, [1.0] * 3)], "cuda")
        assert bool(converted) == on_host and got.n_records == 1
        assert bool((got.records.cpu() == 0x7FFFFFFF).all())


@pytest.mark.parametrize("keep_words", [False, True])
def test_device_words_of_any_stride(keep_words, monkeypatch):
    """Words that lie apart in their tensor, or are one word expanded, convert as their
    copies do."""
    monkeypatch.setattr(multiscene, "DEVICE_MIN_WORDS", 0)
    scene = S.box_room(seed=1, resolution=64)
    scene.compile(threads=8)
    plain = torch.from_numpy(scene.words.view(np.int64)).cuda()
    apart = torch.full((plain.numel(), 3), -1, dtype=torch.int64, device="cuda")
    apart[:, 1] = plain
    node = torch.tensor([_node(0, 1)], dtype=torch.int64, device="cuda")
    for words, copy in ((apart[:, 1], plain), (node.expand(5), node.repeat(5))):
        assert not words.is_contiguous()
        got, want = (ResidentScenes([(w, scene.bbox_min_list, scene.bbox_max)], "cuda", keep_words=keep_words)
                     for w in (words, copy))
        assert got.n_records == want.n_records
        for name in ("records", "cell_tables", "relaid_table", "pool"):
            a, b = getattr(got, name), getattr(want, name)
            assert (a is None) == (b is None) and (a is None or torch.equal(a, b)), name


def test_refused_while_capturing():
    """The conversion waits for its stream, so a capturing stream is an error that leaves
    the capture as it is."""
    words = torch.from_numpy(np.array(_hand_made()["one_record"], np.uint64).view(np.int64)).cuda()
    scratch = torch.zeros(2 * words.numel() + _native.RELAYOUT_STATE_WORDS, dtype=torch.int32, device="cuda")
    layout = _native.DeviceLayout()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        scratch.fill_(7)
        p = scratch.data_ptr()
        code = _native.lib().navi_relayout_device(words.data_ptr(), words.numel(), p, p + 4 * words.numel(),
                                                  p + 8 * words.numel(), ctypes.byref(layout),
                                                  torch.cuda.current_stream().cuda_stream)
    assert code == _native.NAVI_E_LAUNCH and layout.converted == 0
    graph.replay()
    torch.cuda.synchronize()
    assert bool((scratch == 7).all())
