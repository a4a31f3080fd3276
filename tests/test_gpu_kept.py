"""GPU: device buffers and streams kept between calls: calls of growing and shrinking sizes from several
threads at once, before and after the kept memory is given back, equal the same calls one by one; and what
a graph keeps of its first call, when that call is a batch's first run and a direct call at once."""

from __future__ import annotations

import threading

import numpy as np
import pytest

from cityseer import _native
from cityseer.batch import CentralityBatch
from cityseer.tools import mock
from test_gpu_shortest import SHORTEST_KEYS, assert_close, say, stack

pytestmark = pytest.mark.gpu


def test_threads_and_sizes():
    nets = [mock.network_structure_from_lattice(mock.perturbed_lattice(s, seed=90 + s)) for s in (5, 31, 12, 48)]
    calls = [(ns, d) for d in ([300], [200, 400, 900]) for ns in nets]

    def run(ns, d):
        return stack(ns.centrality_shortest(distances=d, sample_probability=0.5, random_seed=3), SHORTEST_KEYS, d)

    alone = [run(ns, d) for ns, d in calls]
    for rep in range(2):
        say(f"4 threads x {len(calls)} calls, pass {rep}")
        wrong: list[str] = []

        def work(k):
            try:
                for i in range(len(calls)):
                    j = (i + 3 * k) % len(calls)
                    got = run(*calls[j])
                    assert np.array_equal(got[0], alone[j][0])
                    assert_close(got, alone[j], f"thread {k}, call {j}")
            except BaseException as e:  # reported by the test itself
                wrong.append(repr(e))

        ts = [threading.Thread(target=work, args=(k,)) for k in range(4)]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
        assert not wrong, wrong
        _native.check(_native.load().cs_release_workspaces())


@pytest.mark.parametrize("side", [4, 24, 60])  # 24 and below: every source at once, no probed searches
def test_first_batch_run_beside_a_first_call(side):
    lat = mock.perturbed_lattice(side, seed=70 + side)
    want = stack(mock.network_structure_from_lattice(lat).centrality_shortest(distances=[300, 600]), SHORTEST_KEYS, [300, 600])
    for rep in range(8):
        say(f"side {side}, fresh network {rep}")
        ns = mock.network_structure_from_lattice(lat)
        ns.upload()
        got: dict = {}
        start = threading.Barrier(2)

        def batch():
            with CentralityBatch() as b:
                b.add_shortest(ns, distances=[300, 600])
                start.wait()
                b.run()
                got["batch"] = b.results()[0]

        def call():
            start.wait()
            got["call"] = ns.centrality_shortest(distances=[300, 600])

        ts = [threading.Thread(target=f) for f in (batch, call)]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
        for name in ("batch", "call"):
            x = stack(got[name], SHORTEST_KEYS, [300, 600])
            assert np.array_equal(x[0], want[0])
            assert_close(x, want, name)
