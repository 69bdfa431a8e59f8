"""Systems whose atoms do not fill their box evenly, against the FP64 oracle
with the bars of test_gpu_parity (pair sets bit for bit, FP64 forces within
1e-11 of the largest component, mixed forces within 1e-5 RMS): the cell grid
is laid out from the box and the number of atoms alone, the atoms may be
anywhere in it."""
import numpy as np
import pytest

from protomoladdon_amd import systems
from tests.test_gpu_parity import check_fp64, check_mixed

pytestmark = pytest.mark.gpu


def dimers(n_pairs, L):
    """Pairs of waters, oxygens 2.8 to 3.2 A or 8.9 to 9.1 A apart (the
    cutoff is 9 A), far from all other pairs."""
    w = systems.water_workload("dimers", 2 * n_pairs, L, 6, 9.0, 7.5, "ewald",
                               0.32, cell_size=50.0)
    rng = np.random.default_rng(7)
    k = int(np.ceil(n_pairs ** (1 / 3)))
    site = np.stack(np.unravel_index(np.arange(n_pairs), (k, k, k)), 1)
    O = (site + 0.5) * (L / k) + rng.uniform(-9, 9, (n_pairs, 3))
    d = rng.normal(size=(n_pairs, 3))
    d /= np.linalg.norm(d, axis=1)[:, None]
    r = np.where(np.arange(n_pairs) % 2, rng.uniform(2.8, 3.2, n_pairs),
                 rng.uniform(8.9, 9.1, n_pairs))
    p = w.positions.reshape(-1, 3, 3)
    p = p - p[:, :1]
    p[0::2] += O[:, None]
    p[1::2] += (O + d * r[:, None])[:, None]
    w.positions = p.reshape(-1, 3)
    return w


def test_dimers_in_a_wide_box():
    """2,400 A: with columns and cells far wider than the cutoff the FP32
    offsets in a cell lose the pairs near the cutoff."""
    check_fp64(dimers(300, 2400.0))
    check_mixed(dimers(300, 2400.0))
