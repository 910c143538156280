"""The float64 pair kernel at the edges of its decomposition (rows per workgroup, systems collected in LDS, entries per
lane) against the numpy oracle in double, and the float64 sort with systems kept in registers and not."""

import numpy as np
import pytest
import torch

import oracle
from oracle import f64 as oracle64
from _systems import ptr_from_counts

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# (one atom; a remainder of a pass of 32 rows; twenty systems in one workgroup, more than it collects in LDS; a system
# larger than a workgroup's run; 2049 and 4097 atoms: the sort with eight atoms per lane, and one past it)
@pytest.mark.parametrize("counts", [[1], [33], [3] * 20, [1, 700, 2], [2049], [4097, 5]])
@pytest.mark.parametrize("periodic", [False, True])
@pytest.mark.parametrize("virial", [False, True])
def test_float64_rows_match_the_oracle(counts, periodic, virial):
    from nvalchemi_amd._neighbor_ops import neighbor_list
    from nvalchemi_amd.models._ops.lj import lj_energy_forces_system_batch

    rng = np.random.default_rng(sum(counts))
    rc, pos, cells = 2.5, [], []
    for n in counts:
        m = int(np.ceil(n ** (1 / 3)))
        length = max(m * 1.1, 2.6)
        g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
        pos.append((g + 0.5 + rng.uniform(-0.1, 0.1, (n, 3))) * length / m)
        cells.append(np.eye(3) * length)
    # (values that float32 holds exactly: the float32 oracle then decides every pair as the double build has to)
    P32, C32, ptr = np.concatenate(pos).astype(np.float32), np.stack(cells).astype(np.float32), ptr_from_counts(counts)
    P, C = P32.astype(np.float64), C32.astype(np.float64)
    N, B = len(P), len(counts)
    bi = oracle.batch_idx_from_ptr(ptr)
    pb = np.ones((B, 3), bool)
    dev = lambda x, t: torch.from_numpy(np.ascontiguousarray(x)).to(DEV, t)  # noqa: E731
    nm, nn, sh = neighbor_list(dev(P, torch.float64), rc, dev(C, torch.float64) if periodic else None,
                               dev(pb, torch.bool) if periodic else None, 128, False, dev(ptr, torch.int32),
                               dev(bi, torch.int32))
    want = oracle.nl_cell(P32, C32 if periodic else None, pb if periodic else None, ptr, rc, 128)
    got = [None if t is None else t.cpu().numpy() for t in (nm, nn, sh)]
    assert np.array_equal(got[1], want[1])
    assert np.array_equal(oracle.matrix_to_edges(*got), oracle.matrix_to_edges(*want))
    e, f, es, w = lj_energy_forces_system_batch(dev(P, torch.float64), dev(C, torch.float64), nm, sh, nn,
                                                dev(bi, torch.int32), N, 1.0, 1.0, rc, 0.0, False, compute_virial=virial)
    ref = oracle64.lj_matrix(P, C, got[0], got[2], got[1], bi, N, 1.0, 1.0, rc, virial=virial)

    def close(got, want):
        # a double sum of at most a few thousand terms in another order: their number times a rounding of the largest
        want = np.asarray(want).reshape(tuple(got.shape))
        assert np.all(np.abs(got.cpu().numpy() - want) <= 1e-12 * max(1.0, float(np.abs(want).max())))

    close(e, ref["atomic_energies"])
    close(f, ref["forces"])
    close(es, np.bincount(bi, weights=ref["atomic_energies"], minlength=B))
    if virial:
        close(w, ref["virials"])
