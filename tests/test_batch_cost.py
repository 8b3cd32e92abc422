"""The batch wrapper's image counts as one array expression, against the definition cell by cell."""
import importlib

import numpy as np
import pytest

wrap = importlib.import_module("dynamis_amd.dynamis_state.radius_graph_pbc_cuda")


def _images(cell, pbc, radius):
    vol = abs(float(np.dot(cell[0], np.cross(cell[1], cell[2]))))
    img = 1.0
    for d in range(3):
        if pbc[d]:
            area = float(np.linalg.norm(np.cross(cell[(d + 1) % 3], cell[(d + 2) % 3])))
            if not (vol > 0.0 and area > 0.0):
                return float("inf")
            img *= 2.0 * radius / (vol / area) + 1.0
    return img


@pytest.mark.parametrize("pbc", [(True, True, True), (True, False, True), (False, False, False)])
def test_images_of_a_batch(pbc):
    rng = np.random.default_rng(5)
    cells = rng.normal(size=(50, 3, 3)) * 8.0
    cells[7] = 0.0                    # singular
    cells[8, 1] = cells[8, 0]         # flat
    cells[9] = np.diag([9.0, 9.0, np.nan])
    got = wrap._images_per_pair(cells, pbc, 6.0)
    want = np.array([_images(c, pbc, 6.0) for c in cells])
    assert got.shape == (50,)
    fin = np.isfinite(want)
    assert np.array_equal(np.isinf(got), ~fin)
    # a handful of roundings in 64 bits each (determinants of random cells lose a few digits)
    np.testing.assert_allclose(got[fin], want[fin], rtol=1e-10)
    assert wrap._images_per_pair(cells[0], pbc, 6.0) == pytest.approx(want[0], rel=1e-10)


@pytest.mark.parametrize("natoms", [[10, 10], [8000, 8000], [250] * 128])
def test_cells_of_a_padded_batch(natoms):
    """More cells than structures: the first ones count, as in the loop over the structures."""
    cells = np.repeat(np.eye(3)[None] * 46.0, len(natoms), axis=0)
    want = wrap._batch_in_one_pass(natoms, cells, [True] * 3, 6.0)
    for more in (1, 3):
        padded = np.concatenate([cells, np.eye(3)[None].repeat(more, axis=0) * 30.0])
        assert wrap._batch_in_one_pass(natoms, padded, [True] * 3, 6.0) == want
