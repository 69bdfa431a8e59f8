"""The adjoint at the edges of the pair kernel's ranges: wrapped and plain
axes, one to four LJ types, every electrostatic term, far exclusions.  Bars:
the FP64 adjoint's dL/dx along a random direction equals the central
difference (h = 1e-5 A) of the FP64 forces within 1e-6 of the product of the
norms (truncation and rounding of the difference are below 1e-7 of it); the
mixed adjoint within test_gpu_grad's 1e-4 (positions, charges) and 1e-3 (LJ
table) RMS of the FP64 one."""
import numpy as np
import pytest

from protomoladdon_amd import systems
from tests.test_gpu_grad import adjoint, rms_rel
from tests.test_gpu_pairs import far_exclusions, stretched, types
from tests.test_gpu_parity import run_gpu

pytestmark = pytest.mark.gpu

CASES = {
    "one_type": lambda: types(1), "three_types": lambda: types(3),
    "four_types": lambda: types(4),
    "coulomb": lambda: systems.small_water(n_mol=400, elec="coulomb"),
    "no_electrostatics": lambda: systems.small_water(n_mol=200, elec="none"),
    "four_columns_x": lambda: stretched(0.85, 1.2, 1.0),
    "two_columns_y_flat_z": lambda: stretched(1.2, 0.73, 0.75),
    "far_exclusions": far_exclusions,
}


@pytest.mark.parametrize("case", list(CASES))
def test_adjoint_edges(case):
    w = CASES[case]()
    rng = np.random.default_rng(3)
    g = rng.normal(size=(w.n_atoms, 3))
    v = rng.normal(size=(w.n_atoms, 3))
    x64, q64, t64 = adjoint(w, "fp64", g)
    h = 1e-5
    fp = run_gpu(w, "fp64", 0, positions=w.positions + h * v, with_pairs=False)[0]
    fm = run_gpu(w, "fp64", 0, positions=w.positions - h * v, with_pairs=False)[0]
    lhs = np.sum((fp - fm) / (2 * h) * g)
    assert abs(lhs - np.sum(x64 * v)) <= 1e-6 * np.linalg.norm(x64) * \
        np.linalg.norm(v)
    x32, q32, t32 = adjoint(w, "mixed", g)
    assert rms_rel(x32, x64) <= 1e-4
    if w.elec != "none":
        assert rms_rel(q32, q64) <= 1e-4
    assert rms_rel(t32, t64) <= 1e-3


def test_nan_gradient_stays_with_its_neighbours():
    """A non-finite dL/dF of one atom reaches the atoms within the cutoff of
    it and no others."""
    w = systems.small_water(n_mol=1500)
    g = np.random.default_rng(4).normal(size=(w.n_atoms, 3))
    g[0] = np.nan
    gx, _, _ = adjoint(w, "mixed", g)
    L = w.topology.boundary_conditions.lengths()[0]
    d = w.positions - w.positions[0]
    d -= L * np.rint(d / L)
    far = np.sum(d * d, axis=1) > 9.0 ** 2 + 1e-6
    assert far.any() and np.isfinite(gx[far]).all()
