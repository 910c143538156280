"""The row filter and the matrix-to-edge-list conversion at the edges of their decomposition: rows around the 64 and 256
slots that the filter has in flight and the 48 entries that the conversion has, rows that do not begin on a 16-byte
boundary, rows that are full, empty or padded in the middle, and an edge list that is too short for all edges."""

import numpy as np
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def T(a):
    return torch.as_tensor(np.ascontiguousarray(a), device=DEV)


def rows(N, K, full):
    """Rows with padding (and shifts that padding should not have) in between, the last one full, the first one empty."""
    rng = np.random.default_rng(100 * K + N)
    pos = rng.uniform(0.0, 6.0, (N, 3)).astype(np.float32)
    nm = rng.integers(0, N, (N, K)).astype(np.int32)
    if not full:
        nm[rng.random((N, K)) < 0.5] = N
        nm[0] = N
    sh = rng.integers(-1, 2, (N, K, 3)).astype(np.int32)
    return pos, nm, sh


@pytest.mark.parametrize("full", [False, True])
@pytest.mark.parametrize("K", [1, 3, 15, 63, 64, 65, 255, 256, 257, 530])
def test_filter_rows(K, full):
    from nvalchemi_amd.models._ops import neighbor_filter as nf

    pos, nm, sh = rows(9, K, full)
    cell = (6.0 * np.eye(3)).astype(np.float32)
    nn = (nm < 9).sum(1).astype(np.int32)
    for shifts, c in ((sh, cell), (sh, None), (None, None)):
        got = nf.filter_neighbor_matrix(T(pos), 4.0, T(nm), T(nn), 9, cell=None if c is None else T(c),
                                        neighbor_matrix_shifts=None if shifts is None else T(shifts))
        want = oracle.filter_neighbor_matrix(pos, 4.0, nm, nn, 9, cell=c, neighbor_matrix_shifts=shifts)
        for g, w in zip(got, want):
            assert (g is None and w is None) or np.array_equal(g.cpu().numpy(), w)


@pytest.mark.parametrize("K", [1, 15, 16, 17, 47, 48, 49, 97, 160])
@pytest.mark.parametrize("offset", [0, 1])
def test_coo_rows(K, offset):
    from nvalchemi_amd import _lib

    N = 21
    _, nm, sh = rows(N, K, True)
    nn = np.random.default_rng(K).integers(0, K + 3, N).astype(np.int32)  # (counts past K: rows that overflowed)
    nn[0], nn[-1] = 0, K
    kept = np.minimum(nn, K)
    total = int(kept.sum())
    ii, kk = np.nonzero(np.arange(K)[None, :] < kept[:, None])
    for cap in (total, total + 5, max(total - 2, 1)):
        # (offset 1: an edge list that begins in the middle of an 8-byte word)
        edges = torch.full((2 * cap + 8,), -7, dtype=torch.int32, device=DEV)
        shifts = torch.full((cap + 4, 3), -7, dtype=torch.int32, device=DEV)
        ptr = torch.empty(N + 1, dtype=torch.int32, device=DEV)
        counts = torch.empty(2, dtype=torch.int32, device=DEV)
        view = edges[offset: offset + 2 * cap].view(cap, 2)
        _lib.nl_coo_from_matrix(T(nm), T(sh), T(nn), ptr, view, shifts[:cap], counts)
        n = min(total, cap)
        assert counts.tolist() == [total, int(total > cap)]
        assert np.array_equal(ptr.cpu().numpy(), np.concatenate([[0], np.cumsum(kept)]))
        assert np.array_equal(view[:n].cpu().numpy(), np.stack([ii, nm[ii, kk]], 1)[:n])
        assert np.array_equal(shifts[:n].cpu().numpy(), sh[ii, kk][:n])
        assert (edges[offset + 2 * n:] == -7).all() and (edges[:offset] == -7).all() and (shifts[n:] == -7).all()
