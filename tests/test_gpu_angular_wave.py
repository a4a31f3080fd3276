"""GPU: the LDS angular search where it could go wrong, against the oracle: exactly equal routes
everywhere (one at a time, and many at one route), streets cut into short straight pieces (no two
states safe together), crossings of more than four streets (longer rows than one state's lanes),
more thresholds than one back-propagation pass holds, and searches that outgrow the room the
probed sources asked for (a dense knot in a sparse network; many dense cores, where searches run out
of pages at a run of nodes met for the first time and their waves go on to other sources). And which
calls that search takes: it and one lane per source give the same results."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

from cityseer import _native
from cityseer.serving import CentralityServer
from cityseer.tools import mock
import oracle.oracle as O
from oracle.oracle import OracleGraph
from test_gpu_shortest import assert_close, say, stack

pytestmark = pytest.mark.gpu

SIMPLEST = ("node_density", "node_farness", "node_harmonic", "node_betweenness")


def _grid(side):
    """Unjittered square grid: every turn 0 or 90 degrees, every length 100."""
    return mock.perturbed_lattice(side, jitter=0.0, drop_frac=0.0, len_range=(1.0, 1.0), seed=0)


def _star(arms, rings, jitter):
    """`arms` radial streets through one crossing, joined by rings: a crossing of `arms` streets."""
    rng = np.random.default_rng(arms)
    ang = 2 * np.pi * (np.arange(arms) + jitter * rng.uniform(-0.3, 0.3, arms)) / arms
    x, y, edges = [0.0], [0.0], []
    for r in range(1, rings + 1):
        for a in range(arms):
            x.append(100.0 * r * np.cos(ang[a]))
            y.append(100.0 * r * np.sin(ang[a]))
            me = 1 + (r - 1) * arms + a
            edges.append((0 if r == 1 else me - arms, me))
            edges.append((me, 1 + (r - 1) * arms + (a + 1) % arms))
    x, y, edges = np.array(x), np.array(y), np.array(edges)
    length = np.hypot(x[edges[:, 1]] - x[edges[:, 0]], y[edges[:, 1]] - y[edges[:, 0]]).astype(np.float32)
    return mock.Lattice(x=x, y=y, edges=edges, length=length)


def _knot():
    """A lattice at 100 m with one 9 x 9 lattice at 4 m hung on its corner: the searches there reach
    several times as many nodes as the rest."""
    a, b = mock.perturbed_lattice(40, seed=5), mock.perturbed_lattice(9, spacing=4.0, jitter=1.0, seed=6)
    k = len(a.x)
    return mock.Lattice(x=np.concatenate([a.x, b.x + a.x[0] - 100.0]), y=np.concatenate([a.y, b.y + a.y[0] - 100.0]),
                        edges=np.concatenate([a.edges, b.edges + k, [[0, k]]]),
                        length=np.concatenate([a.length, b.length, [np.float32(60.0)]]).astype(np.float32))


@pytest.mark.parametrize("name,distances", [
    ("grid", [400, 900]), ("star8", [300, 700]), ("star9 even", [250, 600]), ("pieces", [150, 400, 700]),
    ("five", [200, 300, 400, 500, 600]), ("one", [350]), ("knot", [150, 300])])
def test_matches_oracle(name, distances):
    O.set_heap_mode(False)
    primal = {"grid": lambda: _grid(9), "star8": lambda: _star(8, 4, 1.0), "star9 even": lambda: _star(9, 3, 0.0),
              "pieces": lambda: mock.decompose_lattice(mock.perturbed_lattice(8, seed=71), 15.0),
              "five": lambda: mock.perturbed_lattice(12, seed=72, diag_frac=0.2),
              "one": lambda: mock.perturbed_lattice(5, seed=73), "knot": _knot}[name]()
    ns = mock.network_structure_from_lattice(mock.lattice_dual(primal))
    say(f"angular search, {name}: {ns.node_count()} dual nodes, {distances} m")
    got = stack(ns.centrality_simplest(distances=distances), SIMPLEST, distances)
    stats = _native.last_stats()
    assert _native.last_lds_searches() == stats["sources"]
    ref, _ = OracleGraph.from_network_structure(ns).centrality_simplest(distances)
    assert np.array_equal(got[0], ref[0])
    assert_close(got, ref, name)
    if name == "knot":
        assert stats["retries"] > 0


def _cores(side, across, size):
    """A lattice at 100 m with across x across lattices at 4 m hung on it."""
    a = mock.perturbed_lattice(side, seed=5)
    x, y, edges, length, k = [a.x], [a.y], [a.edges], [a.length], len(a.x)
    for i in range(across):
        for j in range(across):
            b = mock.perturbed_lattice(size, spacing=4.0, jitter=1.0, seed=6 + across * i + j)
            c = int(np.argmin(np.hypot(a.x - 100.0 * side * (i + 0.5) / across, a.y - 100.0 * side * (j + 0.5) / across)))
            x.append(b.x + a.x[c] + 20.0)
            y.append(b.y + a.y[c] + 20.0)
            edges += [b.edges + k, np.array([[c, k]])]
            length += [b.length, np.float32([30.0])]
            k += len(b.x)
    return mock.Lattice(x=np.concatenate(x), y=np.concatenate(y), edges=np.concatenate(edges),
                        length=np.concatenate(length).astype(np.float32))


def test_waves_search_on_after_running_out_of_pages():
    """12,518 dual nodes, three sources a wave: by the layout's arithmetic (the probed sources reach 448
    nodes: 74 pages, 16 runs of 64 nodes) two thirds run out of pages, some 360 of them at a run of
    nodes met for the first time."""
    O.set_heap_mode(False)
    ns = mock.network_structure_from_lattice(mock.lattice_dual(_cores(70, 4, 12)))
    say(f"angular search, dense cores: {ns.node_count()} dual nodes")
    ref, _ = OracleGraph.from_network_structure(ns).centrality_simplest([1200], n_threads=8)
    retries = []
    for k in range(6):
        got = stack(ns.centrality_simplest(distances=[1200]), SIMPLEST, [1200])
        retries.append(_native.last_stats()["retries"])
        assert np.array_equal(got[0], ref[0])
        assert_close(got, ref, f"dense cores, call {k}")
    assert retries[0] > 1000
    assert retries[-1] * 32 <= ns.node_count(), retries  # (later calls have room for them)


def _pieces(side, seed):
    """A dual of streets cut into 20 m pieces, where nearly every state settles alone."""
    return mock.network_structure_from_lattice(
        mock.lattice_dual(mock.decompose_lattice(mock.perturbed_lattice(side, seed=seed), 20.0)))


@pytest.mark.parametrize("side,distances,n_src,in_lds", [
    (22, [900], 60, True),      # few long searches: a wave each
    (22, [1800], 5254, False),  # many: they would take turns, a lane each does not
    (40, [2600], 12, False),    # more states than a state word has positions for
])
def test_which_search(side, distances, n_src, in_lds):
    O.set_heap_mode(False)
    ns = _pieces(side, seed=75)
    src = np.linspace(0, ns.node_count() - 1, n_src).astype(int).tolist()
    say(f"{ns.node_count()} dual nodes in 20 m pieces, {n_src} sources, {distances} m")
    got = stack(ns.centrality_simplest(distances=distances, source_indices=src), SIMPLEST, distances)
    assert _native.last_lds_searches() == (n_src if in_lds else 0)
    plan = ns._sampling_plan(None, None, None, src)
    ref, _ = OracleGraph.from_network_structure(ns).centrality_simplest(
        distances, sources=plan["sources"], eligible=plan["eligible"], scale=plan["scale"], n_threads=8)
    assert np.array_equal(got[0], ref[0])
    assert_close(got, ref, "pieces")


def test_requests_of_all_sizes_served_together():
    """Served slices whose requests go to several launches in LDS, to lanes, and to both."""
    nets = [mock.network_structure_from_lattice(mock.lattice_dual(x)) for x in
            (mock.perturbed_lattice(50, seed=76), _star(9, 3, 1.0), _cores(40, 2, 9))] + [_pieces(22, seed=77)]
    some = np.linspace(0, nets[3].node_count() - 1, 5000).astype(int).tolist()
    mix = [(nets[0], dict(distances=[400])), (nets[3], dict(distances=[1800], source_indices=some)),
           (nets[1], dict(distances=[250, 600])), (nets[2], dict(distances=[300, 900])),
           (nets[3], dict(distances=[300], source_indices=some[::100])), (nets[0], dict(distances=[700, 1500])),
           (nets[2], dict(distances=[500], compute_betweenness=False)),
           (nets[1], dict(distances=[400], tolerance=0.03))]
    alone = [ns.centrality_simplest(**kw) for ns, kw in mix]
    say(f"{len(mix)} simplest requests at once")
    with CentralityServer(slice_ms=50.0) as srv:
        reqs = [srv.submit_simplest(ns, **kw) for ns, kw in mix]
        for k, ((ns, kw), r, want) in enumerate(zip(mix, reqs, alone)):
            r.wait()
            x, y = (stack(v, SIMPLEST, kw["distances"]) for v in (r.result(), want))
            assert np.array_equal(x[0], y[0]), f"request {k}"
            assert_close(x, y, f"request {k}")


def test_lane_workspace_does_not_creep():
    """A network whose lanes are as many as a share of the memory holds: repeated calls run the same number
    of waves, in the same workspace."""
    ns = mock.network_structure_from_lattice(mock.lattice_dual(mock.perturbed_lattice(240, seed=74)))
    lib, tuning = _native.load(), _native.CsTuning()
    _native.check(lib.cs_get_tuning(ctypes.byref(tuning)))
    lanes, tuning.simplest_lanes = tuning.simplest_lanes, 64
    _native.check(lib.cs_set_tuning(ctypes.byref(tuning)))
    try:
        waves = []
        for k in range(3):
            say(f"{ns.node_count()} dual nodes, one lane per source, call {k}")
            ns.centrality_simplest(distances=[150])
            waves.append(_native.last_stats()["waves"])
    finally:
        tuning.simplest_lanes = lanes
        _native.check(lib.cs_set_tuning(ctypes.byref(tuning)))
        _native.check(lib.cs_release_workspaces())
    assert waves[0] * 64 < ns.node_count()
    assert waves[1:] == waves[:-1]
