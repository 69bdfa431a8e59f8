"""The tiles of the k-space matrix products at their edges, against the
oracle's sums: no k-vector at all, fewer orders than a tile, atoms one past a
block's, more orders than one pass holds, and unequal axes.  Bars as in
test_gpu_ewald (forces and virial 1e-10 of the largest, the sums differ in
order only); the energy within 1e-12 of the self energy, whose rounding the
oracle's running sum over up to 1.4e5 k-vectors carries."""
import numpy as np
import pytest

from oracle import oracle as O
from protomoladdon_amd import systems
from tests.test_gpu_ewald import run_device
from tests.test_gpu_pairs import stretched

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("make,alpha,acc", [
    (lambda: systems.small_water(n_mol=7, elec="coulomb"), 0.05, 0.5),
    (lambda: systems.small_water(n_mol=20, elec="coulomb"), 0.3, 0.05),
    (lambda: systems.small_water(n_mol=43, elec="coulomb"), 0.6, 1e-5),
    (lambda: systems.small_water(n_mol=21, elec="coulomb"), 3.5, 1e-8),
    (lambda: stretched(1.7, 1.0, 0.6, n_mol=100), 0.5, 1e-6),
    (lambda: stretched(0.5, 0.8, 2.5, n_mol=100), 0.9, 1e-9),
], ids=["no_kvectors", "few_orders", "atoms129", "two_passes", "flat", "tall"])
def test_tile_edges(make, alpha, acc):
    w = make()
    fr, er, vr, info = O.ewald_kspace(O.System.from_workload(w, flags=1), alpha,
                                      acc)
    fd, od, dinfo = run_device(w, alpha, acc)
    print("nk %d" % dinfo[3], flush=True)
    assert dinfo[3] == int(info[3])
    assert np.abs(fd - fr).max() <= 1e-10 * np.abs(fr).max()
    q = w.topology.scaled_charges
    scale = abs(er) + np.sum(q * q) * dinfo[0] / np.sqrt(np.pi)
    assert abs(od[1] - er) <= 1e-12 * scale
    assert np.abs(od[2:11] - vr).max() <= 1e-10 * np.abs(vr).max()
