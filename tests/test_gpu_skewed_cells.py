"""Neighbor lists of strongly sheared cells, which are binned by a shorter basis of the same lattice: the shifts have to come
out in the lattice vectors that were given, for every pattern of periodic axes and for atoms outside their cell."""

import numpy as np
import pytest

from _systems import ptr_from_counts
from test_gpu_neighbor_list import check_against_oracle, sort_path  # noqa: F401

pytestmark = pytest.mark.gpu


def sheared(rng, k, length):
    """A nearly cubic cell with multiples ``k`` of its vectors added to one another."""
    h = np.eye(3) * length + rng.uniform(-0.1, 0.1, (3, 3)) * length
    h[0] += k[0] * h[1]
    h[1] += k[1] * h[2]
    h[2] += k[2] * h[0]
    return h


@pytest.mark.parametrize("pbc", [(1, 1, 1), (1, 1, 0), (0, 1, 1), (1, 0, 1), (0, 1, 0), (0, 0, 1), (0, 0, 0)])
@pytest.mark.parametrize("k", [(1, 0, 0), (-2, 1, 0), (3, -1, 1)])
def test_sheared_cells_match_brute_force(k, pbc):
    rng = np.random.default_rng(11)
    # (one atom; a cell narrower than the cutoff; two and three cells per axis; more than one tile of candidates)
    counts, lengths = [1, 12, 90, 300, 700], [4.0, 5.3, 10.5, 16.0, 16.0]
    C = np.stack([sheared(rng, k, length) for length in lengths])
    pos = []
    for n, h in zip(counts, C):
        outside = rng.integers(-1, 2, (n, 3)) * np.array(pbc)
        pos.append((rng.uniform(0, 1, (n, 3)) + outside) @ h)
    P = np.concatenate(pos).astype(np.float32)
    pb = np.tile(np.array(pbc, dtype=bool), (len(counts), 1))
    check_against_oracle(P, C.astype(np.float32), pb, ptr_from_counts(counts), 5.0)
