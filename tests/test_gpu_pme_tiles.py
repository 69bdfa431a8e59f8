"""The tiles and bins of the PME charge grid at their edges, against the
oracle's k-space sum with the bars of test_gpu_pme: grids as small as the
B-spline order (every stencil wraps onto all points), tiles and bins cut by
the grid's end, atoms beyond a bin's bucket and a tile's list, and charges
beyond the range of the fast fixed-point conversion."""
import numpy as np
import pytest

from protomoladdon_amd import systems
from tests.test_gpu_pme import check, run_device

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order,grid", [
    (2, (2, 3, 4)), (4, (4, 5, 9)), (8, (8, 8, 8)), (8, (9, 11, 13)),
    (6, (17, 8, 10)), (4, (25, 16, 7)), (2, (33, 31, 15))])
def test_grid_edges(order, grid):
    check(systems.small_water(n_mol=200, elec="coulomb"), grid, order, 0.35)


@pytest.mark.parametrize("order", [2, 4, 8])
def test_atoms_beyond_their_bucket(order):
    w = systems.small_water(n_mol=300, elec="coulomb")
    w.positions = 0.2 * w.positions
    check(w, (24, 24, 24), order, 0.35)
    outs, _ = run_device(w, (24, 24, 24), order, 0.35, repeat=3)
    for f, o in outs[1:]:
        assert np.array_equal(f, outs[0][0]) and np.array_equal(o, outs[0][1])


def test_large_charges():
    w = systems.small_water(n_mol=100, elec="coulomb")
    w.topology.scaled_charges *= 1e3
    w.topology.touch()
    check(w, (20, 20, 20), 4, 0.35)


@pytest.mark.parametrize("order", [2, 4, 8])
@pytest.mark.parametrize("squeeze", [0.02, 0.5])
def test_atoms_in_a_part_of_the_box(order, squeeze):
    """Far more atoms than a bucket and a tile's list hold, in a few bins."""
    w = systems.small_water(n_mol=1000, elec="coulomb")
    w.positions = squeeze * w.positions
    check(w, (24, 27, 30), order, 0.35)
    outs, _ = run_device(w, (24, 27, 30), order, 0.35, repeat=3)
    for f, o in outs[1:]:
        assert np.array_equal(f, outs[0][0]) and np.array_equal(o, outs[0][1])


@pytest.mark.parametrize("order,grid", [(2, (2, 3, 4)), (4, (4, 5, 9)),
                                        (8, (8, 8, 8)), (6, (17, 8, 10))])
@pytest.mark.parametrize("n_mol", [20, 500])
def test_few_tiles(order, grid, n_mol):
    """Grids of one to six tiles, by tiles (60 atoms) and by atomics in memory
    (1,500 atoms: more than 64 a tile), which repeat bit for bit."""
    w = systems.small_water(n_mol=n_mol, elec="coulomb")
    check(w, grid, order, 0.35)
    outs, _ = run_device(w, grid, order, 0.35, repeat=3)
    for f, o in outs[1:]:
        assert np.array_equal(f, outs[0][0]) and np.array_equal(o, outs[0][1])
