"""The count pass's row words and the expansion's blocks at their edges: stencil rows of as many
candidates as one word, one sweep piece or one mask hold, and one more; pairs at distances around
the exclusion of coincident atoms; target ids that start anywhere in a 128-byte line, and tiles
that start and end anywhere in a block.  Results are whole numbers, compared with the CPU oracle
(or, byte for byte, with the aligned build)."""
import numpy as np
import pytest
import torch

import oracle
import plan_model
from dynamis_amd import _lib as L
from dynamis_amd import configs
from dynamis_amd.dynamis_state import dynamis_state_impl as impl

pytestmark = pytest.mark.gpu


def _parity(pos, cell, pbc, r, dev, targets=None):
    tg = None if targets is None else torch.from_numpy(targets).to(dev)
    ei, co, _, cnt = impl.radius_graph_pbc_ex(torch.from_numpy(pos).to(dev), torch.from_numpy(cell),
                                              torch.tensor(pbc), r, 0, False, tg)
    torch.cuda.synchronize()
    used = cell.astype(pos.dtype).astype(np.float64)
    o = oracle.radius_graph(pos, used, pbc, float(np.float32(r)), targets)
    assert np.array_equal(cnt.cpu().numpy(), o["counts"])
    got = oracle.canonical_sort(ei[0].cpu().numpy(), ei[1].cpu().numpy(), co.cpu().numpy().astype(np.int64))
    for a, b in zip(got, oracle.canonical_sort(o["src"], o["dst"], o["shift"])):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("cell", ["cubic", "sheared", "general"])
@pytest.mark.parametrize("k", [1, 2, 4, 5, 19, 20, 21, 27, 28, 29, 40, 41, 56, 57, 130])
def test_rows_of_k_candidates(cuda, cell, k):
    """k atoms side by side along x (one stencil row holds them all) among a few others."""
    print(f"\n[case] rows k={k} {cell}", flush=True)
    rng = np.random.default_rng(k)
    pos = rng.uniform(0.0, 30.0, (60, 3))
    line = np.full((k, 3), 15.0) + rng.uniform(-0.05, 0.05, (k, 3))
    line[:, 0] += rng.permutation(np.linspace(-1.0, 1.0, k))
    C = np.eye(3) * 30.0
    if cell == "sheared":
        C[1, 0], C[2, 0], C[2, 1] = 6.0, -4.0, 5.0
    elif cell == "general":
        C[0, 1], C[1, 2], C[2, 0] = 5.0, -4.0, 3.0
    pos = np.concatenate([pos, line])[rng.permutation(60 + k)].astype(np.float32)
    _parity(pos, C, (True, True, True), 5.0, cuda)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_close_pairs(cuda, dtype):
    """Pairs at distances around 1e-4 (the exclusion of coincident atoms), duplicates included,
    inside a bin and across bins and cell faces."""
    print(f"\n[case] close pairs {np.dtype(dtype)}", flush=True)
    rng = np.random.default_rng(3)
    base = rng.uniform(0.0, 24.0, (200, 3))
    base[:8, 0] = 0.0
    base[8:16] = np.round(base[8:16] / 2.4) * 2.4
    seps = np.array([0.0, 1e-6, 5e-5, 9.9e-5, 1e-4, 1.01e-4, 2e-4, 1e-3, 3e-3, 1e-2])
    d = rng.normal(size=(200, 3))
    d *= (seps[np.arange(200) % len(seps)] / np.linalg.norm(d, axis=1))[:, None]
    pos = np.concatenate([base, base + d]).astype(dtype)
    _parity(pos, np.eye(3) * 24.0, (True, True, True), 5.0, cuda)


def _vectors_agree(pos, cell, r, dev):
    """The build with vectors and distances: the same edges, and their vectors in 64 bits."""
    p, c, b = torch.from_numpy(pos).to(dev), torch.from_numpy(cell), torch.tensor([True] * 3)
    ei, co, _, cnt = impl.radius_graph_pbc_ex(p, c, b, r, 0, False)
    ei2, co2, _, cnt2, vec, dist = impl.radius_graph_pbc_vectors(p, c, b, r)
    assert torch.equal(ei2, ei) and torch.equal(co2, co) and torch.equal(cnt2, cnt)
    used = c.to(p.dtype).double().to(dev)
    v = p.double()[ei[0]] - p.double()[ei[1]] + co.double() @ used
    # (a vector is a 64-bit result: three products and sums of at most 400 A, rounded once more
    # where the outputs are 32-bit)
    tol = 400 * 2.0 ** -50 + (5.0 * 2.0 ** -24 if vec.dtype == torch.float32 else 0.0)
    assert float((vec.double() - v).abs().max()) <= tol
    assert float((dist.double() - v.norm(dim=1)).abs().max()) <= 2 * tol


def _build(pos, cell, dev, r, cap, skew):
    """dg_graph_build with the target ids `skew` entries into an array that starts on a line, and
    guard values around every output."""
    lib = L.lib()
    d = impl._desc(pos, cell, torch.tensor([True, True, True]), impl._r32(r), None)
    wsb = lib.dg_graph_workspace_size(d)
    ws = torch.empty(wsb, dtype=torch.uint8, device=dev)
    cnt = torch.empty(pos.size(0), dtype=torch.int32, device=dev)
    src = torch.full((cap + 64,), -7, dtype=torch.int64, device=dev)
    dst = torch.full((cap + 64,), -7, dtype=torch.int64, device=dev)
    sh = torch.full((cap + 64, 3), -7.0, dtype=torch.float32, device=dev)
    st = lib.dg_graph_build(d, L.ptr(pos), None, L.ptr(ws), wsb, cap, L.ptr(cnt), L.ptr(src),
                            L.ctypes.c_void_p(dst.data_ptr() + 8 * skew), L.ptr(sh), None, None, L.DG_F32,
                            L.stream_of(dev))
    L.check(st, "dg_graph_build")
    E, fl = L._i64(0), L._i64(0)
    L.check(lib.dg_graph_read_totals(d, L.ptr(ws), E, fl, L.stream_of(dev)), "totals")
    return int(E.value), src, dst, sh


@pytest.mark.parametrize("n", [40, 700, 3001, 20011])
def test_target_ids_anywhere_in_a_line(cuda, n):
    print(f"\n[case] skewed target ids n={n}", flush=True)
    b = configs.uniform(n, density=0.08, seed=n, dtype=np.float32, radius=5.0)
    pos, cell = torch.from_numpy(b.pos).to(cuda), torch.from_numpy(b.cell)
    E, src0, dst0, sh0 = _build(pos, cell, cuda, b.radius, 200 * n, 0)
    assert E > 0 and bool((src0[E:] == -7).all()) and bool((dst0[E:] == -7).all()) and bool((sh0[E:] == -7).all())
    for skew in range(1, 17):
        e, src, dst, sh = _build(pos, cell, cuda, b.radius, 200 * n, skew)
        assert e == E
        assert torch.equal(src, src0) and torch.equal(sh, sh0)
        assert torch.equal(dst[skew:skew + E], dst0[:E])
        assert bool((dst[:skew] == -7).all()) and bool((dst[skew + E:] == -7).all())


@pytest.mark.parametrize("seed", range(8))
def test_batch_of_ghosts_inside_a_tile(cuda, seed):
    """Targets 0 .. nt - 1 of a tile that holds over 512 atoms: 256 or more ghosts lie between its
    first targets and its last, so that a batch of 256 lanes has no edges at all while the batches
    before and behind it have.  The expansion skips it."""
    rng = np.random.default_rng(seed)
    r, side = 5.0, 40.0  # 15 bins an axis, tiles of 5
    own, ghosts = [], []
    for k in range(6):  # six tiles, none in the reach of another
        lo, mid, hi = rng.integers(40, 250), rng.integers(520, 600), rng.integers(40, 250)
        low = np.array([26.7 * (k & 1), 26.7 * (k >> 1 & 1), 26.7 * (k >> 2)])
        for zlo, zhi, m, out in [(0.2, 2.5, lo, own), (2.8, 10.5, mid, ghosts), (10.8, 13.1, hi, own)]:
            out.append(low + rng.uniform([0.1, 0.1, zlo], [13.2, 13.2, zhi], (m, 3)))
    nt = sum(map(len, own))
    pos = np.concatenate(own + ghosts)
    pos[:nt] = pos[rng.permutation(nt)]
    cell = np.eye(3) * side
    plan = plan_model.plan(cell, (0, 0, 0), r, len(pos), nt)
    assert plan.nb == [15] * 3 and plan.T == [5] * 3
    # the tile's order: bin by bin, x fastest; batches of 256 with and without targets
    b = np.minimum((pos / side * 15).astype(int), 14)
    tile, l = (b // 5) @ [1, 3, 9], (b % 5) @ [1, 5, 25]
    empty = 0
    for t in np.unique(tile):
        order = np.flatnonzero(tile == t)[np.argsort(l[tile == t], kind="stable")]
        has = [bool((order[k:k + 256] < nt).any()) for k in range(0, len(order), 256)]
        empty += sum(not h and any(has[:k]) and any(has[k:]) for k, h in enumerate(has))
    assert empty > 0
    print(f"\n[case] batch of ghosts seed={seed}: {empty} batches without edges", flush=True)
    for dt in (np.float32, np.float64):
        _parity(pos.astype(dt), cell, (False,) * 3, r, cuda, np.arange(nt))


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("spill,xs", [("one pool full", (5, 6)), ("all pools full", (4, 6))])
def test_region_map_spills(cuda, spill, xs, dtype):
    """A column of atoms along z, in every other stretch of 20 bins of 156 and in those bins along x
    and y that most tiles' regions hold: all tiles ask one of the map's two pools, which has not
    the room.  The others' entries go to the second pool, or, where that fills too, their tiles to
    the fix-up pass; the edges and their vectors are the same."""
    n, r, cell = 2400, 5.0, np.diag([15.6, 15.6, 391.5])  # 6 x 6 x 156 bins
    rng = np.random.default_rng(1)
    f = rng.uniform(0.0, 1.0, (n, 3))
    f[:, 0] = (xs[0] + f[:, 0] * (xs[1] - xs[0])) / 6
    f[:, 1] = (4 + 2 * f[:, 1]) / 6
    f[:, 2] = (40 * rng.integers(0, 4, n) + 20 * f[:, 2]) / 156
    pos = (f @ cell).astype(dtype)
    plan = plan_model.plan(cell, (1, 1, 1), r, n, f64=dtype is np.float64)
    words, pools = plan_model.row_words(pos, cell, (1, 1, 1), r)
    assert plan.npools == 2 and words.max() <= plan.Kw  # (no target goes to the fix-up pass by itself)
    assert pools[0] > 1.1 * plan.mapcap / 2 and pools[1] == 0
    assert pools[0] > 1.1 * plan.mapcap if spill == "all pools full" else pools[0] < 0.9 * plan.mapcap
    print(f"\n[case] region map, {spill} {np.dtype(dtype)}", flush=True)
    _parity(pos, cell, (True,) * 3, r, cuda)
    _vectors_agree(pos, cell, r, cuda)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("shape", ["cubic", "sheared"])
def test_targets_past_their_list(cuda, shape, dtype):
    """A dense clump in an even box: its targets have more row words than their lists hold and go
    to the fix-up pass, in tiles whose other targets the expansion writes."""
    rng = np.random.default_rng(13)
    pos = rng.uniform(0.0, 40.0, (6000, 3))
    pos[:400] = 20.0 + rng.uniform(-1.2, 1.2, (400, 3))
    cell = np.eye(3) * 40.0
    if shape == "sheared":
        cell[1, 0], cell[2, 0], cell[2, 1] = 6.0, -4.0, 5.0
    pos, r = pos.astype(dtype), 5.0
    plan = plan_model.plan(cell, (1, 1, 1), r, len(pos), f64=dtype is np.float64)
    words, _ = plan_model.row_words(pos, cell, (1, 1, 1), r)
    assert 100 < int((words > plan.Kw).sum()) < 1000
    print(f"\n[case] targets past their list {shape} {np.dtype(dtype)}", flush=True)
    _parity(pos, cell, (True,) * 3, r, cuda)
    _vectors_agree(pos, cell, r, cuda)
