"""The tile path's cell build and pair kernel at the edges of their ranges,
against the FP64 oracle, with the bars of test_gpu_parity: pair sets bit for
bit, FP64 forces within 1e-11 of the largest component, mixed forces within
1e-5 RMS."""
import numpy as np
import pytest

from oracle import oracle as O
from protomoladdon_amd import systems
from protomoladdon_amd.batch import BatchedCutoffForce
from protomoladdon_amd.topology import (EXCLUSION_FULL, EXCLUSION_MODIFIED,
                                        PeriodicBoundaryConditions)
from protomoladdon_amd.topology import ScalarStructure as SS
from tests.test_gpu_batch import batch_eval
from tests.test_gpu_parity import check_fp64, check_mixed, rms_rel, run_gpu

pytestmark = pytest.mark.gpu


def types(n):
    """n LJ types: 8 fit the kernel's LDS table, 9 .. 256 are read from
    memory, 257 take the general path."""
    return systems.many_type_chains(n_chains=45, n_types=n)


def stretched(sx, sy, sz, n_mol=500):
    """Water in a box of sx, sy, sz times the cube's side (25 A at 500):
    columns are 4.5 A wide, so an axis below 18 A has fewer than four and
    takes the minimum image of every pair, one below 22.5 A has four."""
    w = systems.small_water(n_mol=n_mol)
    L = float(w.topology.boundary_conditions.lengths()[0])
    s = np.array([sx, sy, sz])
    w.positions = w.positions * s
    a, b, c = L * s
    w.topology.boundary_conditions = PeriodicBoundaryConditions(
        (a, 0, 0), (0, b, 0), (0, 0, c), (0.5 * a, 0.5 * b, 0.5 * c))
    w.name = "water_%g_%g_%g" % (sx, sy, sz)
    return w


def side_lengths(a, b, c):
    w = systems.small_water(n_mol=300)
    L = float(w.topology.boundary_conditions.lengths()[0])
    return stretched(a / L, b / L, c / L, n_mol=300)


def gas(n_mol, L):
    """A thin gas, without one pair (tests/test_gpu_density.py has gases
    with pairs)."""
    return systems.water_workload("gas", n_mol, L, 5, 9.0, 7.5, "ewald", 0.32)


def far_exclusions():
    """FULL and MODIFIED pairs at index distances of 1 .. 64 (15 is the last
    held in the code word, 64 the last in the masks)."""
    w = systems.small_chains(n_chains=60)
    n = w.n_atoms
    w.topology.molecules[:] = np.arange(n) // 100
    x = w.topology.exclusions
    for k, d in enumerate((14, 15, 16, 31, 63, 64)):
        a = np.arange(k, n - d, 7)
        a = a[a // 100 == (a + d) // 100]
        x.add_many(np.stack([a, a + d], 1),
                   EXCLUSION_FULL if k % 2 else EXCLUSION_MODIFIED)
    w.topology.touch()
    return w


CASES = {
    "types1": lambda: types(1), "types8": lambda: types(8),
    "types9": lambda: types(9), "types256": lambda: types(256),
    "types257": lambda: types(257),
    "four_columns_x": lambda: stretched(0.85, 1.2, 1.0),
    "two_columns_y_flat_z": lambda: stretched(1.2, 0.73, 0.75),
    # 18 A and what the band of the cutoff adds is the shortest axis whose
    # fourth column is taken at two images
    "four_columns_shortest": lambda: side_lengths(18.0003, 18.0001, 22.0),
    "four_columns_short": lambda: side_lengths(18.0001, 18.01, 18.02),
    "four_columns_long": lambda: side_lengths(18.3, 22.49, 31.0),
    "gas": lambda: gas(600, 120.0), "gas_no_pairs": lambda: gas(60, 90.0),
    "gas_three_molecules": lambda: gas(3, 200.0),
    "dense_column": lambda: stretched(0.8, 0.8, 12.0, n_mol=900),
    "far_exclusions": far_exclusions,
}


@pytest.mark.parametrize("case", list(CASES))
def test_pairs_match_oracle(case):
    ref = check_fp64(CASES[case](), flags=3)
    if ref.n_pairs:
        check_mixed(CASES[case](), flags=1)
    else:
        f, _, npairs, _ = run_gpu(CASES[case](), "mixed", 1, with_pairs=False)
        assert npairs == 0 and not f.any()


@pytest.mark.parametrize("precision,shapes", [("mixed", 3), ("fp64", 2)])
def test_shapes_give_the_same_bits(precision, shapes):
    """A wave per item or a block per item, mixed sizes in one batch."""
    ws = [systems.config3_replica(0, 167), systems.config3_replica(1, 40),
          systems.config3_replica(2, 700)]
    bf = BatchedCutoffForce.from_workloads(ws, precision=precision)
    res = []
    for shape in range(shapes):
        bf.set_shape(shape)
        res.append(batch_eval(bf, ws)[1:])
    bf.close()
    for f, out in res[1:]:
        np.testing.assert_array_equal(f, res[0][0])
        np.testing.assert_array_equal(out, res[0][1])


@pytest.mark.parametrize("precision", ["mixed", "fp64"])
@pytest.mark.parametrize("bad", [np.nan, -np.nan, np.inf])
def test_atoms_without_a_position_have_no_pairs(precision, bad):
    """The other atoms' forces are those without them: the two atoms carry
    no charge and the oxygens' type of a hydrogen, so at any position they
    give no force."""
    w = systems.small_water(n_mol=300)
    t = w.topology
    t.scaled_charges[[4, 5]] = 0.0
    t.touch()
    ref = run_gpu(w, "fp64", 0, with_pairs=False)
    p = w.positions.copy()
    p[4] = bad
    p[5, 1] = bad
    f, _, npairs, _ = run_gpu(w, precision, 0, positions=p, with_pairs=False)
    rest = np.setdiff1d(np.arange(w.n_atoms), [4, 5])
    assert npairs < ref[2]
    assert np.isfinite(f).all()
    assert rms_rel(f[rest], ref[0][rest]) <= (
        1e-5 if precision == "mixed" else 1e-12)


@pytest.mark.parametrize("precision", ["mixed", "fp64"])
@pytest.mark.parametrize("n_mol", [60, 500])
def test_no_atom_has_a_position(precision, n_mol):
    """Work items without one finite position, in a box that wraps per pair
    (60 waters) and one that does not."""
    w = systems.small_water(n_mol=n_mol)
    p = np.full_like(w.positions, np.nan)
    f, _, npairs, _ = run_gpu(w, precision, 0, positions=p, with_pairs=False)
    assert npairs == 0 and not f.any()


def test_lj_parameters_are_the_users():
    """Two oxygens 2 A apart without electrostatics, in a box whose columns and
    cells are whole multiples of 1.5 A: every number on the way to A / r^12 -
    B / r^6 is a power of two times the table's A or B, so the mixed energy is
    that of their FP32 values exactly."""
    w = systems.small_water(n_mol=2, elec="none")
    w.topology.boundary_conditions = PeriodicBoundaryConditions(
        (72, 0, 0), (0, 72, 0), (0, 0, 72), (36, 36, 36))
    t = w.topology.lennard_jones_parameters.table
    p = w.positions.copy()
    p[:3] += (8.0, 8.0, 8.0) - p[0]
    p[3:] += (10.0, 8.0, 8.0) - p[3]
    for A, B in ((8191.0, 0.0), (0.0, 64.0), (1048575.0, 0.0), (0.0, 594.83)):
        t[...] = 0.0
        t[0, 0, 0], t[0, 0, 1] = A, B
        w.topology.touch()
        e = run_gpu(w, "mixed", 0, positions=p, with_pairs=False)[1]
        assert e[SS.LENNARDJONES] == (float(np.float32(A)) / 2.0 ** 12 -
                                      float(np.float32(B)) / 2.0 ** 6)


def test_virial_over_tables_and_positions():
    """With electrostatics the mean error of the virial's trace over boxes of
    water and LJ tables is below 6e-7 kcal/mol an atom: without the factors of
    the FP32 records it is 9e-7, with them 2e-7, each 1e-7 uncertain."""
    rng = np.random.default_rng(12)
    err = []
    for k in range(48):
        w = systems.config3_replica(k, 700)
        t = w.topology.lennard_jones_parameters.table
        s = np.sqrt(rng.uniform(0.7, 1.4, t.shape[0]))
        u = np.sqrt(rng.uniform(0.9, 1.1, t.shape[0]))
        s, u = np.outer(s, s), np.outer(u, u)
        for c in range(4):
            t[..., c] *= s * u if c % 2 else s * u * u
        w.topology.touch()
        tr = [run_gpu(w, p, 1, with_pairs=False)[1].table[7:16:4].sum()
              for p in ("fp64", "mixed")]
        err.append((tr[1] - tr[0]) / w.n_atoms)
    print("mean %.3g, scatter %.3g" % (np.mean(err), np.std(err)), flush=True)
    assert abs(np.mean(err)) <= 6e-7


@pytest.mark.parametrize("elec", ["coulomb", "ewald"])
@pytest.mark.parametrize("switch", ["C2", "other C2", "C1"])
@pytest.mark.parametrize("who", [(0, 3), (0, 4)])
def test_coincident_atoms_fp64(elec, switch, who):
    """The electrostatic energy of two atoms in one place is infinite, of
    their charges' sign; their forces and the LJ energy are NaN, as the
    reference's arithmetic gives them."""
    w = systems.small_water(n_mol=300, elec=elec)
    if switch == "other C2":
        w.elec_switch = (7.0, 9.0)
    elif switch == "C1":
        w.elec_switch = ("C1", 9.0)
    p = w.positions.copy()
    p[who[0]] = p[who[1]]
    ref = O.evaluate(O.System.from_workload(w, positions=p, flags=0))
    f, e, _, _ = run_gpu(w, "fp64", 0, positions=p, with_pairs=False)
    assert np.isinf(ref.energies[1])
    assert e[SS.COULOMB] == ref.energies[1]
    assert np.isnan(e[SS.LENNARDJONES]) and np.isnan(ref.energies[0])
    np.testing.assert_array_equal(np.isnan(f), np.isnan(ref.forces))
