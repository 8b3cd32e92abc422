"""The row-word lists and the region map hold what structures need whose atoms fill a part of their
cell only (slabs, droplets), and small and large even boxes: a model of the count pass (its rows,
quarter-bin ends, pieces and words: tests/plan_model.cpp) on the library's own plan.  A target past
its list, or a tile past the map, is swept again by the fix-up pass, at several times the cost."""
import numpy as np
import pytest

import plan_model

SHEAR = np.array([[1.0, 0.0, 0.0], [0.25, 0.95, 0.0], [0.1, 0.15, 0.8]])


def _slab(n, rho, fill, shape=None, axis=2, at=0.0):
    shape = np.eye(3) if shape is None else shape
    cell = shape * (n / (fill * rho * np.linalg.det(shape))) ** (1.0 / 3.0)
    f = np.random.default_rng(n).uniform(0.0, 1.0, (n, 3))
    f[:, axis] = at + fill * f[:, axis]
    return f % 1.0 @ cell, cell


def _droplet(n, rho, widths):
    rad = (3.0 * n / (4.0 * np.pi * rho)) ** (1.0 / 3.0)
    q = np.random.default_rng(n).uniform(-rad, rad, (3 * n, 3))
    q = q[(q * q).sum(1) < rad * rad][:n]
    return q + widths * rad, np.eye(3) * (2.0 * widths * rad)


CASES = (
    [("slab %g rho=%g r=%g" % c, _slab, (20_000, c[1], c[0]), c[2])
     for c in [(0.2, 0.05, 4.5), (0.3, 0.04, 5.0), (0.1, 0.08, 6.0), (0.2, 0.1, 6.0), (0.5, 0.1, 6.0),
               (0.3, 0.05, 8.0)]]
    + [("slab x at %g" % at, _slab, (n, 0.06, 0.25, None, 0, at), 5.0) for n in (3000, 20_000) for at in (0.4, 0.9)]
    + [("sheared slab rho=%g r=%g fill=%g" % c, _slab, (9973, c[0], c[2], SHEAR), c[1])
       for c in [(0.08, 5.0, 0.6), (0.05, 4.5, 0.2), (0.1, 6.0, 0.2)]]
    + [("droplet rho=%g r=%g" % c, _droplet, (20_000, c[0], 2.0), c[1])
       for c in [(0.085, 5.0), (0.1, 6.0), (0.04, 4.5)]]
    + [("even n=%d rho=%g r=%g" % (n, *c), _slab, (n, c[0], 1.0), c[1])
       for n in (100, 300, 1000, 2000, 10_007) for c in [(0.04, 4.5), (0.1, 6.0), (0.1, 8.0), (0.1, 10.0), (0.1, 12.0)]])


@pytest.mark.parametrize("name,make,args,r", CASES, ids=[f"{c[0]} {c[2][0]}" for c in CASES])
def test_lists_hold_every_target(name, make, args, r):
    pos, cell = make(*args)
    plan = plan_model.plan(cell, (1, 1, 1), r, len(pos))
    words, pools = plan_model.row_words(pos, cell, (1, 1, 1), r)
    assert words.max() > 0
    # (the fullest list of 20,000 leaves a fifth: no structure of its kind is near the end)
    assert words.max() <= 0.8 * plan.Kw
    assert pools.sum() <= 0.96 * plan.mapcap


@pytest.mark.parametrize("r,rho", [(4.5, 0.02), (5.0, 0.05), (6.0, 0.1), (10.0, 0.1)])
def test_the_lists_end_at_the_static_workspace(r, rho):
    """No build leaves the 64 MiB of the allocation-free build for its lists: past the atoms where
    the workspace reaches it, it stays there until the least lists need more."""
    _ends_at(64 << 20, 2e4, 6e5, r, rho)


@pytest.mark.parametrize("r,rho", [(4.5, 0.02), (5.0, 0.05)])
def test_the_lists_of_the_largest_builds(r, rho):
    """Nor do they take a build past 64 GiB, and one that is past it has the least lists: what fitted
    the card before still does."""
    _ends_at(64 << 30, 1e8, 4e8, r, rho)
    n = 500_000_000
    plan = plan_model.plan(np.eye(3) * (n / rho) ** (1.0 / 3.0), (1, 1, 1), r, n)
    assert plan.ws_bytes == plan.least_bytes > 64 << 30


def _ends_at(limit, lo, hi, r, rho):
    sizes = []
    for n in np.unique(np.geomspace(lo, hi, 400).astype(int)):
        cell = np.eye(3) * (n / rho) ** (1.0 / 3.0)
        sizes.append((n, plan_model.plan(cell, (1, 1, 1), r, int(n)).ws_bytes))
    below = [s for _, s in sizes if s <= limit]
    assert below and max(below) > 0.99 * limit
    # and the two ways a size is reached meet: none is above the limit by the lists' growth alone
    first = next(n for n, s in sizes if s > limit)
    least = plan_model.plan(np.eye(3) * (first / rho) ** (1.0 / 3.0), (1, 1, 1), r, int(first)).least_bytes
    assert least > limit
