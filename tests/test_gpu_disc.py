"""GPU: the LDS shortest search where it could go wrong, against the oracle: exact ties everywhere,
rows of one to four blocks and beyond, one-way and parallel edges, streets cut into short pieces, a
single very short edge (nodes that settle alone), either result by itself, more thresholds than one
variant's registers, source subsets, and searches that outgrow the room the probed sources asked for. And which
calls that search takes."""

from __future__ import annotations

import numpy as np
import pytest

from cityseer import _native
from cityseer.batch import CentralityBatch
from cityseer.rustalgos.graph import NetworkStructure
from cityseer.tools import mock
import oracle.oracle as O
from oracle.oracle import OracleGraph
from test_gpu_angular_wave import _grid, _star
from test_gpu_shortest import SHORTEST_KEYS, assert_close, say, stack

pytestmark = pytest.mark.gpu


def _knot(side=60, size=14):
    """A lattice at 100 m with one size x size lattice at 4 m hung on its corner: the searches there reach
    many times as many nodes as the rest."""
    a, b = mock.perturbed_lattice(side, seed=5), mock.perturbed_lattice(size, spacing=4.0, jitter=1.0, seed=6)
    k = len(a.x)
    return mock.Lattice(x=np.concatenate([a.x, b.x + a.x[0] - 100.0]), y=np.concatenate([a.y, b.y + a.y[0] - 100.0]),
                        edges=np.concatenate([a.edges, b.edges + k, [[0, k]]]),
                        length=np.concatenate([a.length, b.length, [np.float32(60.0)]]).astype(np.float32))


def _directed(lat, seed):
    """The lattice with a third of its streets one-way, a tenth doubled and a few loops."""
    rng = np.random.default_rng(seed)
    ns = NetworkStructure()
    n, m = lat.n_nodes, lat.n_edges
    ns.add_street_nodes_bulk(None, lat.x, lat.y)
    way = rng.integers(0, 3, m)
    a = np.concatenate([lat.edges[way != 2, 0], lat.edges[way != 1, 1], lat.edges[:m // 10, 0], [3, 7]])
    b = np.concatenate([lat.edges[way != 2, 1], lat.edges[way != 1, 0], lat.edges[:m // 10, 1], [3, 7]])
    length = np.concatenate([lat.length[way != 2], lat.length[way != 1], lat.length[:m // 10] * np.float32(1.00003),
                             np.float32([30.0, 40.0])])
    key = np.concatenate([np.zeros(len(a) - m // 10 - 2), np.ones(m // 10), [0, 0]]).astype(np.uint32)
    ns.add_street_edges_bulk(a, b, key, length)
    return ns


def _short_edge():
    lat = mock.perturbed_lattice(16, seed=83)
    lat.length[::37] = np.float32(0.05)
    return lat


@pytest.mark.parametrize("name,distances,kw", [
    ("grid", [250, 700, 1500], {}),
    ("star8", [150, 450], {}), ("star16", [300], {}), ("star18", [300], {}),
    ("pieces", [120, 400, 900], {}),
    ("directed", [300, 800], {}),
    ("short edge", [400, 2500], {}),
    ("five", [200, 300, 400, 500, 3000], {}),
    ("one", [5000], {}),
    ("knot", [150, 300], {}),
    ("five", [350, 800], {"compute_betweenness": False}),
    ("five", [350, 800], {"compute_closeness": False}),
    ("five", [600], {"source_indices": [0, 5, 17, 60, 61, 62]}),
])
def test_matches_oracle(name, distances, kw):
    O.set_heap_mode(False)
    make = {"grid": lambda: _grid(11), "star8": lambda: _star(8, 4, 1.0), "star16": lambda: _star(16, 3, 1.0),
            "star18": lambda: _star(18, 3, 1.0), "pieces": lambda: mock.decompose_lattice(mock.perturbed_lattice(9, seed=81), 15.0),
            "short edge": _short_edge, "five": lambda: mock.perturbed_lattice(13, seed=82, diag_frac=0.4),
            "one": lambda: mock.perturbed_lattice(5, seed=84), "knot": _knot}
    if name == "directed":
        ns = _directed(mock.perturbed_lattice(14, seed=85, diag_frac=0.1), 85)
    else:
        ns = mock.network_structure_from_lattice(make[name]())
    say(f"shortest search, {name}: {ns.node_count()} nodes, {distances} m {kw}")
    res = ns.centrality_shortest(distances=distances, **kw)
    stats, in_lds = _native.last_stats(), _native.last_lds_searches()
    plan = ns._sampling_plan(None, None, None, kw.get("source_indices"))
    ref, _ = OracleGraph.from_network_structure(ns).centrality_shortest(
        distances, closeness=kw.get("compute_closeness", True), betweenness=kw.get("compute_betweenness", True),
        sources=plan["sources"], eligible=plan["eligible"], scale=plan["scale"])
    got = stack(res, SHORTEST_KEYS, distances)
    assert np.array_equal(got[0], ref[0])
    assert_close(got, ref, name)
    # which search ran: rows of more than 16 neighbours have no place in LDS
    assert in_lds == (0 if name == "star18" else stats["sources"])
    if name == "knot":
        assert stats["retries"] > 0


@pytest.mark.parametrize("n_src,closeness,betweenness,in_lds", [
    (300, True, True, True),     # one source a workgroup at once
    (1600, True, True, False),   # dependencies of 6,000 nodes leave two workgroups a CU: they would take turns
    (1600, True, False, True),   # without them the turns are short
])
def test_which_search(n_src, closeness, betweenness, in_lds):
    O.set_heap_mode(False)
    ns = mock.network_structure_from_lattice(mock.perturbed_lattice(110, seed=88))
    src = np.linspace(0, ns.node_count() - 1, n_src).astype(int).tolist()
    say(f"shortest search to 7,200 m, {n_src} sources, betweenness {betweenness}")
    res = ns.centrality_shortest(distances=[800, 7200], source_indices=src, compute_closeness=closeness,
                                 compute_betweenness=betweenness)
    assert _native.last_lds_searches() == (n_src if in_lds else 0)
    assert _native.last_stats()["retries"] == 0
    plan = ns._sampling_plan(None, None, None, src)
    ref, _ = OracleGraph.from_network_structure(ns).centrality_shortest(
        [800, 7200], closeness=closeness, betweenness=betweenness, sources=plan["sources"], eligible=plan["eligible"],
        scale=plan["scale"], n_threads=8)
    got = stack(res, SHORTEST_KEYS, [800, 7200])
    assert np.array_equal(got[0], ref[0])
    assert_close(got, ref, "which search")


def test_city_is_searched_once():
    """Room up to what costs no resident workgroup: no source of a large even network runs out of it."""
    ns = mock.network_structure_from_lattice(mock.perturbed_lattice(200, seed=1, diag_frac=0.05))
    say(f"shortest search, {ns.node_count()} nodes to 5,000 m")
    ns.centrality_shortest(distances=[5000])
    assert _native.last_stats()["retries"] == 0 and _native.last_lds_searches() == ns.node_count()


def test_waves_of_a_town_as_wide_as_its_searches():
    """Two waves a workgroup: only the town's middle has a front past their line (100), its spread sources none."""
    ns = mock.network_structure_from_lattice(mock.perturbed_lattice(56, seed=2, diag_frac=0.05))
    n = ns.node_count() // 2  # all at once: 2 waves each, 4 by the middle's front
    src = np.linspace(0, ns.node_count() - 1, n).astype(int).tolist()
    say(f"{ns.node_count()} nodes, {n} sources to 2,750 m")
    ns.centrality_shortest(distances=[2750], source_indices=src)
    stats = _native.last_stats()
    assert _native.last_lds_searches() == n and stats["waves"] == 2 * n, stats


def test_large_reach_is_searched_once():
    """Too large for a workgroup's LDS and for the usual records of a wave: no source is searched twice."""
    O.set_heap_mode(False)
    ns = mock.network_structure_from_lattice(mock.decompose_lattice(mock.perturbed_lattice(46, seed=86), 20.0))
    n = ns.node_count()
    src = list(range(0, n, n // 270))
    say(f"shortest search, large reach: {n} nodes, {len(src)} sources")
    res = ns.centrality_shortest(distances=[600, 9000], source_indices=src)
    stats = _native.last_stats()
    assert _native.last_lds_searches() == 0
    assert stats["nodes_reached"] > 16384 * len(src) and stats["retries"] == 0
    plan = ns._sampling_plan(None, None, None, src)
    ref, _ = OracleGraph.from_network_structure(ns).centrality_shortest(
        [600, 9000], sources=plan["sources"], eligible=plan["eligible"], scale=plan["scale"])
    got = stack(res, SHORTEST_KEYS, [600, 9000])
    assert np.array_equal(got[0], ref[0])
    assert_close(got, ref, "large reach")


def test_batch_mixes_searches_and_replays():
    """One batch of searches in LDS, of two sizes, some out of room, and in scratch; every replay the same.
    (The knot is a twentieth of its network's node order, before its first probed source, and its 1,296
    nodes are past 1.3 times the 400 or so that any probed source of the batch reaches.)"""
    nets = [mock.network_structure_from_lattice(x) for x in
            (_knot(160, 36), _star(18, 3, 1.0), mock.perturbed_lattice(13, seed=82), mock.perturbed_lattice(50, seed=87))]
    asked = [[150, 300], [300], [200, 500], [1500]]
    alone = [stack(ns.centrality_shortest(distances=d), SHORTEST_KEYS, d) for ns, d in zip(nets, asked)]
    with CentralityBatch() as batch:
        for ns, d in zip(nets, asked):
            batch.add_shortest(ns, distances=d)
        for k in range(3):
            say(f"batch of {len(nets)} networks, run {k}")
            stats = batch.run()
            assert stats["retries"] > 0
            in_lds = _native.last_lds_searches()
            assert 0 < in_lds < stats["sources"] - nets[1].node_count()
            for i, (res, d) in enumerate(zip(batch.results(), asked)):
                got = stack(res, SHORTEST_KEYS, d)
                assert np.array_equal(got[0], alone[i][0])
                assert_close(got, alone[i], f"network {i}, run {k}")
            nets[2].centrality_shortest(distances=[400])


def test_batch_of_small_towns_is_one_launch():
    """Towns of very different sizes whose sources all run at once: a workgroup for each, in one launch."""
    nets = [mock.network_structure_from_lattice(mock.perturbed_lattice(s, seed=90 + s)) for s in (9, 11, 13, 16, 19, 23, 28)]
    alone = [stack(ns.centrality_shortest(distances=[400, 1200]), SHORTEST_KEYS, [400, 1200]) for ns in nets]
    with CentralityBatch() as batch:
        for ns in nets:
            batch.add_shortest(ns, distances=[400, 1200])
        for k in range(2):
            say(f"batch of {len(nets)} small towns, run {k}")
            stats = batch.run()
            assert _native.last_lds_searches() == stats["sources"] and stats["waves"] >= stats["sources"]
            for i, res in enumerate(batch.results()):
                got = stack(res, SHORTEST_KEYS, [400, 1200])
                assert np.array_equal(got[0], alone[i][0])
                assert_close(got, alone[i], f"town {i}, run {k}")


@pytest.mark.parametrize("size", [14, 24, 36])
def test_what_outgrows_its_room_is_searched_few_times(size):
    """A knot of a hundredth to a twentieth of the sources, up to seventeen times the probed reach: a second
    try has room for all of it or all of LDS, and later calls, which may start with that room, try no more."""
    ns = mock.network_structure_from_lattice(_knot(160, size))
    seen = []
    for k in range(4):
        say(f"call {k} on a network with a {size} x {size} knot")
        res = stack(ns.centrality_shortest(distances=[150, 300]), SHORTEST_KEYS, [150, 300])
        seen.append((_native.last_stats()["retries"], res))
        assert np.array_equal(res[0], seen[0][1][0])
        assert_close(res, seen[0][1], f"call {k}")
    tries = [r for r, _ in seen]
    assert 0 < tries[0] <= 2 * (size * size + 10) and tries == sorted(tries, reverse=True), tries


def test_batch_learns_the_room_its_searches_take():
    """Runs of a batch whose knot outgrows the probed searches (1,296 nodes to their 75): each plans the next
    with more room, until none searches twice; every run the same."""
    ns = mock.network_structure_from_lattice(_knot(160, 36))
    want = stack(ns.centrality_shortest(distances=[150, 300]), SHORTEST_KEYS, [150, 300])
    with CentralityBatch() as batch:
        batch.add_shortest(ns, distances=[150, 300])
        retries = []
        while not retries or retries[-1] > 0 and len(retries) < 24:
            say(f"batch with a knot, run {len(retries)}")
            retries.append(batch.run()["retries"])
            got = stack(batch.results()[0], SHORTEST_KEYS, [150, 300])
            assert np.array_equal(got[0], want[0])
            assert_close(got, want, f"run {len(retries)}")
    assert retries[0] > 0 and retries[-1] == 0, retries
