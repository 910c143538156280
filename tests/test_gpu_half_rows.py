"""The half-list pair kernel at the edges of its decomposition (rows per workgroup, systems in a window, systems larger
than a window, more systems than it collects in LDS, rows that are not 16-byte words, pairs that join systems) against
the numpy oracle."""

import numpy as np
import pytest
import torch

import oracle
from _systems import ptr_from_counts

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def batch(counts, rc):
    rng = np.random.default_rng(sum(counts))
    pos, cells = [], []
    for n in counts:
        m = int(np.ceil(n ** (1 / 3)))
        length = max(m * 1.1, 2.6)
        g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)
        g = g[rng.permutation(m**3)[:n]]
        pos.append((g + 0.5 + rng.uniform(-0.1, 0.1, (n, 3))) * length / m)
        cells.append(np.eye(3) * length)
    return np.concatenate(pos).astype(np.float32), np.stack(cells).astype(np.float32), ptr_from_counts(counts)


def check(P, C, nm, sh, nn, bi, rc, switch, virial):
    from nvalchemi_amd.models._ops.lj import lj_energy_forces_system_batch

    dev = lambda x: None if x is None else torch.from_numpy(np.ascontiguousarray(x)).to(DEV)  # noqa: E731
    N, B = len(P), len(C)
    e, f, es, w = lj_energy_forces_system_batch(dev(P), dev(C), dev(nm), dev(sh), dev(nn), dev(bi), N, 1.0, 1.0, rc, switch,
                                                True, compute_virial=virial)
    ref = oracle.lj_matrix(P, C, nm, sh, nn, bi, N, 1.0, 1.0, rc, half=True, virial=virial, switch_width=switch)

    def close(got, want, sums=1):
        # double sums rounded to float32 once (a system's energy: the float32 energies of its atoms, summed)
        want = np.asarray(want, dtype=np.float64).reshape(tuple(got.shape))
        assert np.all(np.abs(got.cpu().numpy() - want) <= 1.2e-7 * sums * max(1.0, float(np.abs(want).max())))

    close(e, ref["atomic_energies"])
    close(f, ref["forces"])
    close(es, ref["energy"], sums=2)
    if virial:
        close(w, ref["virials"], sums=2)


# (one atom; a remainder of a pass of 64 rows; twenty systems in one workgroup; windows that end inside a run of rows;
# 1792 and 1793 atoms: the largest window, and one atom past it; systems in two windows)
@pytest.mark.parametrize("counts", [[1], [65], [5] * 60, [900, 3, 800, 200, 1], [1792], [1793, 40], [4200, 7], [300] * 25])
@pytest.mark.parametrize("periodic", [False, True])
@pytest.mark.parametrize("width,switch,virial", [(64, 0.0, True), (67, 0.4, True), (64, 0.4, False)])
def test_half_rows_match_the_oracle(counts, periodic, width, switch, virial):
    rc = 2.2
    P, C, ptr = batch(counts, rc)
    pb = np.ones((len(counts), 3), bool)
    nm, nn, sh = oracle.nl_cell(P, C if periodic else None, pb if periodic else None, ptr, rc, width, half=True)
    assert nn.max() < width
    check(P, C, nm, sh, nn, oracle.batch_idx_from_ptr(ptr), rc, switch, virial)


def test_pairs_that_join_systems():
    """A list may name any atom as a partner, near or far in memory."""
    rc, counts = 2.2, [1500, 1500, 1500]
    P, C, ptr = batch(counts, rc)
    rng = np.random.default_rng(3)
    N = len(P)
    nm = rng.integers(0, N, (N, 24)).astype(np.int32)
    nm[nm == np.arange(N)[:, None]] += 1
    nm[nm == N] = 0
    nn = rng.integers(0, 25, N).astype(np.int32)
    # a potential that stays finite at the distances of strangers
    bi = oracle.batch_idx_from_ptr(ptr)
    P += (np.arange(N, dtype=np.float32) * 0.05)[:, None]
    check(P, C, nm, None, nn, bi, 400.0, 0.0, True)
