"""GPU: sources put in device order on the device, around the edges of its blocks (2,048 nodes, 256 sources)
and of its use (1,024 sources), in any listing, some named twice: the same results as a network kept in its
original order, which needs none of it."""

from __future__ import annotations

import numpy as np
import pytest

from cityseer.tools import mock
from test_gpu_node_order import pair, shuffled
from test_gpu_shortest import SEGMENT_KEYS, SHORTEST_KEYS, assert_close, say, stack

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("side,n_src,twice", [
    (32, 1023, 0), (32, 1024, 0), (33, 1025, 40), (46, 2116, 0), (64, 4096, 0), (65, 3000, 700), (91, 8281, 0)])
def test_any_listing_equals_original_order(side, n_src, twice):
    a, b = pair(shuffled(mock.perturbed_lattice(side, seed=side), seed=side + 1))
    rng = np.random.default_rng(n_src)
    src = rng.permutation(a.node_count())[:n_src - twice]
    src = rng.permutation(np.concatenate([src, src[:twice]])).tolist()
    say(f"{a.node_count()} nodes, {len(src)} sources, {twice} named twice")
    got, want = (stack(ns.centrality_shortest(distances=[300, 700], source_indices=src), SHORTEST_KEYS, [300, 700])
                 for ns in (a, b))
    assert np.array_equal(got[0], want[0])
    assert_close(got, want, "shortest")
    got, want = (stack(ns.segment_centrality(distances=[400]), SEGMENT_KEYS, [400]) for ns in (a, b))
    assert_close(got, want, "segment")
