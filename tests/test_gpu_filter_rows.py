"""The two-pass filter (dg_filter_rows) at the edges of its tiles and of a wave's chunks, with
chunks that keep everything, nothing and some of their edges, against numpy."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["float32", "float64", "int32", "int64"])
@pytest.mark.parametrize("E", [1, 511, 513, 4095, 4096, 4097, 70000, 1200001])
def test_filter_rows(E, dtype):
    import torch
    from dynamis_amd import _lib as L
    if not torch.cuda.is_available():
        pytest.skip("needs the GPU")
    n, r = 500, 2.0
    g = np.random.default_rng(E)
    # multiples of 1/8 (shifts whole): the products, sums and squares below are exact in fp32 and
    # fp64, so the kept set is the same however they are rounded
    pos = (g.integers(0, 80, (n, 3)) / 8).astype("float64" if dtype == "float64" else "float32")
    cell = np.diag([10.0, 10.0, 10.0])
    src, dst = g.integers(0, n, E), g.integers(0, n, E)
    shift = g.integers(-1, 2, (E, 3))
    # three of four edges close to their source, in runs of all, none and some kept
    close = g.random(E) < np.where(np.arange(E) // 5000 % 3 == 0, 0.0, np.where(np.arange(E) // 5000 % 3 == 1, 1.0, 0.75))
    dst, shift = np.where(close, src, dst), np.where(close[:, None], 0, shift)
    d = pos[src].astype("f8") - pos[dst] + shift @ cell
    keep = (d * d).sum(1) <= r * r
    dev = torch.device("cuda")
    lib = L.lib()
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)
    p, s, e, sh = t(pos), t(src), t(dst), t(shift.astype(dtype))
    code = {"float32": L.DG_F32, "float64": L.DG_F64, "int32": L.DG_I32, "int64": L.DG_I64}[dtype]
    oe, osh = torch.full((2 * E,), -5, dtype=torch.int64, device=dev), torch.full_like(sh, -5)
    nk = torch.empty(1, dtype=torch.int64, device=dev)
    wsb = lib.dg_filter_rows_workspace_size(E)
    ws = torch.empty(wsb, dtype=torch.uint8, device=dev)
    cbuf = (L.ctypes.c_double * 9)(*cell.reshape(-1).tolist())

    def run(n_atoms):
        L.check(lib.dg_filter_rows(L.ptr(p), L.DG_F64 if dtype == "float64" else L.DG_F32, n_atoms, cbuf, r,
                                   L.ptr(s), L.ptr(e), L.ptr(sh), code, E, L.ptr(oe), L.ptr(osh), L.ptr(nk),
                                   L.ptr(ws), wsb, L.stream_of(dev)), "filter")
        return int(nk.item())

    k = run(n)
    assert k == int(keep.sum())
    np.testing.assert_array_equal(oe[:2 * k].cpu().numpy(), np.concatenate([src[keep], dst[keep]]))
    np.testing.assert_array_equal(osh[:k].cpu().numpy(), shift[keep].astype(dtype))
    assert bool((oe[2 * k:] == -5).all()) and bool((osh[k:] == -5).all())
    assert run(0) == -1  # no atoms: every edge names one outside
