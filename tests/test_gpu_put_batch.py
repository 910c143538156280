"""A put of a whole batch in one plan and one copy against the same put level by level and tensor by tensor (which the other
tests hold to the oracle): every tensor, boundary, mask and count must come out the same."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def source(n, edges, seed):
    """``n`` systems of 0 to 40 atoms with rows of 1 to 36 bytes."""
    from nvalchemi_amd.data.batch import Batch, SegmentedGroup, UniformGroup

    g = torch.Generator().manual_seed(seed)
    sizes = torch.randint(0, 41, (n,), generator=g)
    N = int(sizes.sum())
    atoms = {"positions": torch.randn(N, 3, generator=g), "atomic_numbers": torch.randint(1, 90, (N,), generator=g),
             "flag": torch.rand(N, generator=g) < 0.5, "wide": torch.randn(N, 3, 3, generator=g, dtype=torch.float64)}
    groups = {"atoms": SegmentedGroup({k: v.to(DEV) for k, v in atoms.items()}, sizes, DEV)}
    if edges:
        per = torch.randint(0, 9, (n,), generator=g) * (sizes > 0)
        E = int(per.sum())
        owner = torch.repeat_interleave(torch.arange(n), per)
        first = torch.cumsum(sizes, 0) - sizes
        nl = first[owner].unsqueeze(1) + (torch.rand(E, 2, generator=g) * sizes[owner].unsqueeze(1)).long()
        groups["edges"] = SegmentedGroup({"neighbor_list": nl.to(torch.int32).to(DEV), "kind": (torch.rand(E, generator=g) < 0.5).to(DEV)},
                                         per, DEV)
    system = {"energy": torch.randn(n, 1, generator=g), "pbc": torch.rand(n, 3, generator=g) < 0.5,
              "system_id": torch.arange(n).unsqueeze(1)}
    groups["system"] = UniformGroup({k: v.to(DEV) for k, v in system.items()}, n, DEV)
    return Batch._construct(DEV, groups)


def state(b):
    out = {}
    for name, g in b._storage.groups.items():
        for k, v in g.items():
            out[name, k] = v.clone()
        if name != "system":
            out[name, "ptr"], out[name, "lengths"] = g._ptr_store().clone(), g.segment_lengths.clone()
            out[name, "host"] = torch.tensor(list(g.lengths_list()))
        out[name, "n"] = torch.tensor(len(g))
    return out


def same(a, b):
    assert a.keys() == b.keys()
    for k in a:
        assert a[k].shape == b[k].shape and a[k].dtype == b[k].dtype and torch.equal(a[k], b[k]), k


@pytest.mark.parametrize("n, edges, room", [(1, False, 1.0), (5, True, 0.4), (64, True, 1.0), (300, False, 0.5), (1023, True, 0.7),
                                            (1025, True, 1.0), (2100, False, 0.3)])
def test_one_plan_moves_what_the_levels_move(n, edges, room, monkeypatch):
    from nvalchemi_amd.data.batch import Batch

    def run(together):
        taken = []
        general = Batch._put_together
        with monkeypatch.context() as m:
            def put(self, *a, **k):
                taken.append(general(self, *a, **k) if together else None)
                return taken[-1]
            m.setattr(Batch, "_put_together", put)
            rng = np.random.default_rng(n)
            cap = max(2, int(n * room) + 2)
            src = source(n, edges, n)
            buf = Batch.empty(num_systems=cap, num_nodes=max(int(room * src.num_nodes), 8), num_edges=int(4 * n * room) + 8,
                              template=src, device=DEV)
            slots = torch.zeros(cap, dtype=torch.bool, device=DEV)
            # (the first slots are taken and so are some in between: a put fills from the first free one on)
            slots[: cap // 8] = True
            slots[cap // 2 : cap // 2 + cap // 8] = True
            out = []
            for k, share in enumerate((0.3, 0.0, 1.0, 0.5)):
                s = source(n, edges, n + k)
                for g in (buf._atoms_group, buf._edges_group):
                    if g is not None and k < 3:  # the last put meets boundaries without headroom
                        store = torch.zeros(len(g) + n + 2, dtype=torch.int32, device=DEV)
                        store[: len(g) + 1] = g.batch_ptr
                        g._batch_ptr = store
                mask = torch.from_numpy(rng.random(n) < share).to(DEV)
                copied = torch.zeros(n, dtype=torch.bool, device=DEV) if k % 2 else None
                buf.put(s, mask, copied_mask=copied, dest_mask=slots if k != 1 else None)
                out.append({**state(buf), ("mask", ""): (copied if copied is not None else s._copied_mask).clone(),
                            ("slots", ""): slots.clone()})
        if together:
            assert [t is not None for t in taken] == [True, True, True, False]
        return out

    for a, b in zip(run(True), run(False)):
        same(a, b)


def test_buffer_round_trips_and_refusals(monkeypatch):
    from nvalchemi_amd.data.batch import Batch
    from nvalchemi_amd.dynamics.sinks import GPUBuffer

    def run(together):
        out = []
        with monkeypatch.context() as m:
            if not together:
                m.setattr(Batch, "_put_together", lambda self, *a, **k: None)
            buf = GPUBuffer(capacity=12, max_atoms=30, max_edges=8)
            for k in range(8):
                src = source(20, True, k)
                sizes = src.num_nodes_per_graph
                mask = (torch.arange(20, device=DEV) % (3 + k % 3) == 0)
                if k != 4:
                    mask &= sizes <= 30  # (pass 4 is refused for its atoms unless its buffer is full)
                try:
                    buf.write(src, mask)
                except RuntimeError as e:
                    out.append(str(e))
                if len(buf):
                    out.append(state(buf.read()))
                if k in (2, 5):
                    out.append(state(buf.drain()))
                    assert len(buf) == 0
                out.append(state(buf._buffer))
                out.append({("slots", ""): buf._dest_mask.clone()})
        return out

    a, b = run(True), run(False)
    assert len(a) == len(b) and any(isinstance(x, str) for x in a)
    for x, y in zip(a, b):
        assert x == y if isinstance(x, str) else same(x, y) is None


def test_ranges_at_odd_addresses():
    from nvalchemi_amd import _lib

    base = torch.randint(0, 255, (300_000,), dtype=torch.uint8, device=DEV)
    cases = [(0, 1), (1, 17), (15, 15), (16, 16), (31, 64), (100, 5), (112, 4096), (5000, 100_003), (110_004, 70_000), (190_000, 0)]
    for shift in (0, 1, 4, 16):
        dst = torch.full_like(base, 7)
        want = dst.clone()
        src = [base[o: o + n] for o, n in cases]
        put = [dst[o + shift: o + shift + n] for o, n in cases]
        for s, (o, n) in zip(src, cases):
            want[o + shift: o + shift + n] = s
        # (the ranges do not overlap: with a shift some would, so one call for each then)
        for s, d in zip(src, put):
            _lib.copy_tensors([s], [d])
        assert torch.equal(dst, want)
        for o, n in cases:
            want[o + shift: o + shift + n] = 0
        _lib.zero_tensors(put)
        assert torch.equal(dst, want)
