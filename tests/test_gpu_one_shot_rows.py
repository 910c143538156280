"""Rows that are padded after the build: row widths around the 16-byte stores, full and empty rows, no shifts; the summary of
a build at the sizes of its grid; a one-shot list in memory that held something else; the stress from the virial."""

import numpy as np
import pytest
import torch

import oracle
from _systems import periodic_batch
from test_gpu_dynamics import make_batch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("K", [1, 2, 3, 4, 5, 63, 64, 65, 255, 256, 257, 784])
@pytest.mark.parametrize("shifted", [True, False])
def test_pad_rows(K, shifted):
    from nvalchemi_amd import _lib

    N = 13
    nn = np.random.default_rng(K).integers(0, K + 1, N).astype(np.int32)
    nn[:3] = 0, K, K + 2  # (a count past K: nothing to pad)
    nm = torch.full((N, K), -7, dtype=torch.int32, device=DEV)
    sh = torch.full((N, K, 3), -7, dtype=torch.int32, device=DEV)
    _lib.nl_pad_rows(torch.as_tensor(nn, device=DEV), N, nm, sh if shifted else None)
    padding = np.arange(K)[None, :] >= nn[:, None]
    assert np.array_equal(nm.cpu().numpy(), np.where(padding, N, -7))
    assert np.array_equal(sh.cpu().numpy(), np.where(padding[..., None] & shifted, 0, -7) * np.ones((1, 1, 3), int))


@pytest.mark.parametrize("N", [1, 63, 1023, 1024, 1025, 600_001])
def test_summary(N):
    from nvalchemi_amd import _lib

    _lib.nl_status(N, 1, DEV, clear=True)
    counts = torch.randint(0, 5000, (N,), dtype=torch.int32, device=DEV)
    counts[-1] = 5001
    assert _lib.nl_summary(counts, 1) == (5001, int(counts.long().sum()), 0, 0)


@pytest.mark.parametrize("K", [16, None, 200])
@pytest.mark.parametrize("half", [False, True])
def test_nothing_of_the_memory_underneath_is_left(K, half):
    from nvalchemi_amd.models.base import NeighborListFormat
    from nvalchemi_amd.neighbors import compute_neighbors

    P, C, pb, ptr = periodic_batch(29, 5, 1, 150, 0.5)
    N = len(P)
    for fmt in (NeighborListFormat.MATRIX, NeighborListFormat.COO):
        batch = make_batch(P, np.ones(N, np.int64), np.ones(N, np.float32), C, pb, ptr)
        junk = [torch.full((N * w * 3,), 77, dtype=torch.int32, device=DEV) for w in (16, 32, 64, 100, 200, 200)]
        del junk
        compute_neighbors(batch, 2.5, format=fmt, max_neighbors=K, half_list=half)
        if fmt == NeighborListFormat.COO:
            edges = np.concatenate([batch.neighbor_list.cpu().numpy(), batch.neighbor_list_shifts.cpu().numpy()], 1)
        else:
            nm, sh, nn = (t.cpu().numpy() for t in (batch.neighbor_matrix, batch.neighbor_matrix_shifts, batch.num_neighbors))
            padding = np.arange(nm.shape[1])[None, :] >= nn[:, None]
            assert nm.shape[1] > nn.max() and (nm[padding] == N).all() and (sh[padding] == 0).all()
            edges = oracle.matrix_to_edges(nm, nn, sh)
        if half:
            mirrored = np.concatenate([edges[:, [1, 0]], -edges[:, 2:]], 1)
            edges = np.concatenate([edges, mirrored])
        assert np.array_equal(oracle.canonical_edges(edges), oracle.nl_brute(P, C, pb, ptr, 2.5))


@pytest.mark.parametrize("B", [1, 28, 29, 300])
def test_stress(B):
    from nvalchemi_amd import _lib

    rng = np.random.default_rng(B)
    cell = (rng.normal(0, 1, (B, 3, 3)) + 4 * np.eye(3)).astype(np.float32)
    virial = rng.normal(0, 1, (B, 3, 3)).astype(np.float32)
    got = _lib.stress_from_virial(torch.as_tensor(virial, device=DEV), torch.as_tensor(cell, device=DEV)).cpu().numpy()
    want = -virial.astype(np.float64) / np.abs(np.linalg.det(cell.astype(np.float64)))[:, None, None]
    # (the volume rounded, then the quotient: half a unit in the last place each)
    assert np.all(np.abs(got - want) <= 2 * 2.0**-24 * 1.01 * np.abs(want) + 1e-45)
