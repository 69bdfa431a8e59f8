"""Parity of the HIP path (through the C ABI) with the FP64 oracle and the
reference's golden outputs.

Bars: pair sets bit-exact; FP64 forces within 1e-12 of the largest oracle
force component (different summation order only) and energies/virials
within 1e-11 relative; mixed precision RMS relative force error <= 1e-5
(the stated accuracy target), energies and virials within 2e-5 relative."""
import numpy as np
import pytest

from oracle import oracle as O
from protomoladdon_amd import systems
from protomoladdon_amd.topology import ScalarStructure as SS
from tests import fixtures_lib as FX

pytestmark = pytest.mark.gpu


def rms_rel(f, ref):
    return float(np.sqrt(np.mean(np.sum((f - ref) ** 2, axis=1)) /
                         np.mean(np.sum(ref ** 2, axis=1))))


def run_gpu(w, precision, flags=0, positions=None, with_pairs=True,
            force_pairs=False):
    """Forces, energies, pair count; with_pairs adds the FP64 pair-set
    kernel's set, force_pairs the set the force kernel itself evaluated."""
    from protomoladdon_amd.topology import ScalarStructure
    force = w.make_force(precision)
    pos = w.positions if positions is None else positions
    f = np.zeros((w.n_atoms, 3))
    e = ScalarStructure(virial=bool(flags & 1), molecular_virial=bool(flags & 2))
    force.evaluate(w.topology, pos, f, e)
    npairs = force.last_pair_count()
    pairs = force.pair_set(w.topology, pos) if with_pairs else None
    if force_pairs:
        pairs = (pairs, force.force_pairs(w.topology, pos))
    force.close()
    return f, e, npairs, pairs


def check_fp64(w, flags=3, positions=None):
    s = O.System.from_workload(w, positions=positions, flags=flags)
    ref = O.evaluate(s, record_pairs=True)
    f, e, npairs, (pairs, fpairs) = run_gpu(w, "fp64", flags, positions,
                                            force_pairs=True)
    print(w.name, "n", w.n_atoms, "pairs", ref.n_pairs, flush=True)
    ref_pairs = O.sorted_pairs(ref.pairs)
    np.testing.assert_array_equal(pairs, ref_pairs)
    # the pairs the FP64 force kernel itself evaluated, with their classes
    np.testing.assert_array_equal(fpairs, ref_pairs)
    assert npairs == ref.n_pairs
    scale = max(1.0, np.abs(ref.forces).max())
    assert np.abs(f - ref.forces).max() <= 1e-12 * scale * 10
    np.testing.assert_allclose([e[SS.LENNARDJONES], e[SS.COULOMB]], ref.energies, rtol=1e-11,
                               atol=1e-9)
    if flags & 3:
        vir = e.table[7:16]
        np.testing.assert_allclose(vir, ref.virial, rtol=1e-11,
                                   atol=1e-9 * np.abs(ref.virial).max())
    if flags & 2:
        mv = e.table[16:25]
        np.testing.assert_allclose(mv, ref.molvirial, rtol=1e-11,
                                   atol=1e-9 * np.abs(ref.molvirial).max())
    return ref


def check_mixed(w, flags=1):
    s = O.System.from_workload(w, flags=flags)
    ref = O.evaluate(s, record_pairs=True)
    f, e, npairs, (_, fpairs) = run_gpu(w, "mixed", flags, with_pairs=False,
                                        force_pairs=True)
    err = rms_rel(f, ref.forces)
    print(w.name, "mixed rms rel force err", err, flush=True)
    assert err <= 1e-5
    assert npairs == ref.n_pairs
    # the pairs the mixed kernel evaluated (FP32 test, FP64 re-decision
    # within `band` of the cutoff) are the FP64 oracle's, pair by pair
    np.testing.assert_array_equal(fpairs, O.sorted_pairs(ref.pairs))
    # FP32 pair energies summed in FP64: the totals carry the per-pair FP32
    # error amplified by cancellation between positive and negative terms
    # (the LJ total is a small difference of large sums), so energies and
    # virials are held to 2e-5 relative.
    np.testing.assert_allclose([e[SS.LENNARDJONES], e[SS.COULOMB]],
                               ref.energies, rtol=2e-5, atol=1e-6)
    if flags & 1:
        np.testing.assert_allclose(e.table[7:16], ref.virial, rtol=2e-5,
                                   atol=2e-5 * np.abs(ref.virial).max())
    return err


def slab_water():
    """600 waters with z compressed to 0.7 of the box: two columns in x and
    y, and a z axis the cutoff spans completely (the single-system tile
    kernel then takes the minimum image along z per pair)."""
    from protomoladdon_amd.topology import PeriodicBoundaryConditions
    w = systems.small_water(n_mol=600)
    L = float(w.topology.boundary_conditions.lengths()[0])
    Lz = 0.7 * L
    w.positions = w.positions * np.array([1.0, 1.0, 0.7])
    w.topology.boundary_conditions = PeriodicBoundaryConditions(
        (L, 0, 0), (0, L, 0), (0, 0, Lz), (0.5 * L, 0.5 * L, 0.5 * Lz))
    w.name = "water_slab"
    return w


# ------------------------------------------------------------------ FP64
@pytest.mark.parametrize("make", [
    systems.config0,
    lambda: systems.small_water(n_mol=400),
    lambda: systems.small_chains(n_chains=120),
    lambda: systems.config3_replica(0, 167),
    lambda: systems.config3_replica(7, 2667),
    slab_water,
], ids=["config0", "water_ewald", "chains", "replica_small", "replica_large",
        "water_slab"])
def test_fp64_matches_oracle(make):
    check_fp64(make())


def test_fp64_golden_reference_vectors():
    for name, make in (("config0", systems.config0),
                       ("chains2k", lambda: systems.small_chains(n_chains=100)),
                       ("replica167", lambda: systems.config3_replica(0, 167))):
        g = FX.load("ref_%s.npz" % name)
        w = make()
        f, e, npairs, pairs = run_gpu(w, "fp64", 3)
        assert npairs == int(g["n_pairs"])
        from tests.golden.make_fixtures import pair_hash
        assert pair_hash(pairs) == str(g["pair_sha256"])
        scale = max(1.0, np.abs(g["forces"]).max())
        assert np.abs(f - g["forces"]).max() <= 1e-11 * scale
        np.testing.assert_allclose([e[SS.LENNARDJONES], e[SS.COULOMB]], g["energies"], rtol=1e-11)


def test_fp64_water423_reference_output():
    # the reference's own regression case, Coulomb with C1 switching
    w, d = FX.water423()
    f, e, _, _ = run_gpu(w, "fp64", 0)
    assert abs(e[SS.LENNARDJONES] - d["energy_row0"][9]) < 6e-5
    assert abs(e[SS.COULOMB] - d["energy_row0"][10]) < 6e-5
    fb, _, _ = FX.harmonic_bonded_forces(
        w.positions, d["bonds"], d["angles"], d["bond_k_r0"][0],
        d["bond_k_r0"][1], d["angle_k_theta0"][0], d["angle_k_theta0"][1],
        d["box"])
    assert np.abs(f + fb - d["forces_frame0"]).max() < 1e-6


def test_fp64_pentane_reference_output():
    w, d = FX.pentane320()
    f, e, _, _ = run_gpu(w, "fp64", 0)
    assert abs(e[SS.LENNARDJONES] - d["energy_row0"][9]) < 6e-6


def test_fp64_edge_positions():
    # atoms on box faces, far images and a non-zero origin
    w = systems.small_water(n_mol=300)
    L = w.topology.boundary_conditions.lengths()[0]
    p = w.positions.copy()
    p[0] = (0.0, L, L / 2)
    p[3] = (L, 0.0, np.nextafter(L, 0))
    p[6] += (-L, 2 * L, 3 * L)
    p[9] += (5 * L, 0.0, -7 * L)
    check_fp64(w, positions=p)
    bc = w.topology.boundary_conditions
    bc.set(bc.e1, bc.e2, bc.e3, (6.8, 7.3, 8.2))
    w.topology.touch()
    check_fp64(w)


def test_fp64_empty_and_tiny_systems():
    from protomoladdon_amd.topology import ScalarStructure
    w = systems.small_water(n_mol=1)
    check_fp64(w)
    # zero atoms
    t = w.topology
    from protomoladdon_amd.topology import ExclusionTable, Topology
    t0 = Topology(np.zeros(0, np.int32), np.zeros(0), np.zeros(0, np.int32),
                  t.lennard_jones_parameters, ExclusionTable(0),
                  t.boundary_conditions, t.cell_manager)
    force = w.make_force("fp64")
    f = np.zeros((0, 3))
    e = ScalarStructure()
    force.evaluate(t0, np.zeros((0, 3)), f, e)
    assert e[SS.COULOMB] == 0.0 and e[SS.LENNARDJONES] == 0.0
    assert len(force.pair_set(t0, np.zeros((0, 3)))) == 0


def test_fp64_is_deterministic_and_accumulates():
    from protomoladdon_amd.topology import ScalarStructure
    w = systems.small_water(n_mol=500)
    force = w.make_force("fp64")
    f1 = np.zeros((w.n_atoms, 3))
    e1 = ScalarStructure(virial=True)
    force.evaluate(w.topology, w.positions, f1, e1)
    f2 = np.ones((w.n_atoms, 3))
    e2 = ScalarStructure(virial=True)
    e2[SS.COULOMB] = 5.0
    force.evaluate(w.topology, w.positions, f2, e2)
    np.testing.assert_array_equal(f2, 1.0 + f1)
    assert e2[SS.COULOMB] == 5.0 + e1[SS.COULOMB]
    f3 = np.zeros((w.n_atoms, 3))
    e3 = ScalarStructure(virial=True)
    force.evaluate(w.topology, w.positions, f3, e3)
    np.testing.assert_array_equal(f3, f1)
    np.testing.assert_array_equal(e3.table, e1.table)


def dense_cell_water(n_mol, seed=11):
    """Water in a 60 A box with every molecule moved rigidly so that its
    oxygen lies in 7 x 7 x 1.6 A at the origin corner: one cell of the tile
    grid holds far more atoms than its bucket row (the mean occupancy is
    below one atom, so a row has 64 slots), and the gather reads that cell
    back from the cell index of every atom (in LDS up to 512 atoms, beyond
    in the cell's segment)."""
    w = systems.water_workload("water_dense_cell", n_mol, 60.0, seed, 9.0,
                               7.5, "ewald", 0.32)
    rng = np.random.default_rng(seed)
    X = w.positions.reshape(n_mol, 3, 3).copy()
    o_new = rng.uniform([0.5, 0.5, 0.35], [7.5, 7.5, 1.95], size=(n_mol, 3))
    X += (o_new - X[:, 0, :])[:, None, :]
    return w, np.ascontiguousarray(X.reshape(-1, 3))


@pytest.mark.parametrize("n_mol", [100, 300])
def test_fp64_cell_beyond_its_bucket(n_mol):
    w, pos = dense_cell_water(n_mol)
    check_fp64(w, flags=1, positions=pos)


def test_mixed_pair_set_of_a_cell_beyond_its_bucket():
    w, pos = dense_cell_water(100)
    s = O.System.from_workload(w, positions=pos, flags=1)
    ref = O.evaluate(s, record_pairs=True)
    _, _, npairs, (pairs, fpairs) = run_gpu(w, "mixed", 1, pos,
                                            force_pairs=True)
    ref_pairs = O.sorted_pairs(ref.pairs)
    np.testing.assert_array_equal(pairs, ref_pairs)
    np.testing.assert_array_equal(fpairs, ref_pairs)
    assert npairs == ref.n_pairs


@pytest.mark.parametrize("n_mol,threads", [
    (1500, None),   # below the chunked staging: the caller's thread alone
    (8000, None),   # 24,000 atoms: chunked copy and add on the host threads
    (8000, "1"),
    (8000, "3"),
])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_host_entry_equals_device_entry_on_changing_positions(
        precision, n_mol, threads, monkeypatch):
    """pmnb_evaluate (host arrays; the tile path writes its results into
    mapped host memory) against pmnb_evaluate_device on the same context,
    bit for bit, over calls whose positions change every time, so that a
    result left over from an earlier call cannot pass; forces and energies
    are added to what the caller's arrays already hold.  threads: the host
    threads that share the staging copy and the force add
    (PMNB_HOST_THREADS, read when a context first stages a large system)."""
    import torch
    from protomoladdon_amd.topology import ScalarStructure
    if threads is None:
        monkeypatch.delenv("PMNB_HOST_THREADS", raising=False)
    else:
        monkeypatch.setenv("PMNB_HOST_THREADS", threads)
    w = systems.small_water(n_mol=n_mol)
    force = w.make_force(precision)
    rng = np.random.default_rng(7)
    dev = torch.device("cuda:0")
    for k in range(4):
        pos = w.positions + rng.normal(0.0, 0.02, w.positions.shape)
        print("call", k, precision, n_mol, threads, flush=True)
        fh = np.full((w.n_atoms, 3), 0.25)
        e = ScalarStructure(virial=True)
        e[SS.COULOMB] = 3.0
        force.evaluate(w.topology, pos, fh, e)
        n_host = force.last_pair_count()
        x = torch.tensor(pos, dtype=torch.float64, device=dev)
        fd = torch.zeros_like(x)
        out = torch.zeros(20, dtype=torch.float64, device=dev)
        force.evaluate_device(w.topology, x, fd, out, 1)
        torch.cuda.synchronize()
        n_dev = force.last_pair_count()
        o = out.cpu().numpy()
        np.testing.assert_array_equal(fh, 0.25 + fd.cpu().numpy())
        assert e[SS.LENNARDJONES] == o[0] and e[SS.COULOMB] == 3.0 + o[1]
        np.testing.assert_array_equal(e.table[7:16], o[2:11])
        assert n_host == n_dev > 0
    force.close()


# ----------------------------------------------------------------- mixed
@pytest.mark.parametrize("make", [
    systems.config0,
    lambda: systems.small_water(n_mol=400),
    lambda: systems.small_chains(n_chains=120),
    lambda: systems.config3_replica(0, 167),
    slab_water,
], ids=["config0", "water_ewald", "chains", "replica_small", "water_slab"])
def test_mixed_matches_oracle(make):
    check_mixed(make())


def test_mixed_pair_set_and_determinism():
    from protomoladdon_amd.topology import ScalarStructure
    w = systems.small_water(n_mol=600)
    force = w.make_force("mixed")
    out = []
    for _ in range(2):
        f = np.zeros((w.n_atoms, 3))
        e = ScalarStructure(virial=True)
        force.evaluate(w.topology, w.positions, f, e)
        out.append((f, e.table.copy(), force.last_pair_count()))
    np.testing.assert_array_equal(out[0][0], out[1][0])
    np.testing.assert_array_equal(out[0][1], out[1][1])
    ref = O.evaluate(O.System.from_workload(w))
    assert out[0][2] == ref.n_pairs


@pytest.mark.parametrize("which", [1, 2])
def test_large_config_properties(which):
    """Full-size configs: FP64 GPU vs the oracle (bit-exact pair count,
    forces) and mixed RMS error; sizes the oracle runs in seconds."""
    w = systems.config1() if which == 1 else systems.config2()
    s = O.System.from_workload(w)
    ref = O.evaluate(s, record_pairs=True)
    ref_pairs = O.sorted_pairs(ref.pairs)
    f, e, npairs, (_, fp) = run_gpu(w, "fp64", 0, with_pairs=False,
                                    force_pairs=True)
    print(w.name, "pairs", ref.n_pairs, flush=True)
    assert npairs == ref.n_pairs
    np.testing.assert_array_equal(fp, ref_pairs)
    del fp
    scale = max(1.0, np.abs(ref.forces).max())
    assert np.abs(f - ref.forces).max() <= 1e-11 * scale
    fm, em, npm, (_, fpm) = run_gpu(w, "mixed", 0, with_pairs=False,
                                    force_pairs=True)
    assert npm == ref.n_pairs
    np.testing.assert_array_equal(fpm, ref_pairs)
    del fpm
    err = rms_rel(fm, ref.forces)
    print(w.name, "mixed rms rel err", err, flush=True)
    assert err <= 1e-5
    # Newton's third law holds to the fixed-point resolution
    assert np.abs(fm.sum(axis=0)).max() < 1e-6 * np.abs(fm).sum() + 1e-3


def test_single_system_of_many_cells():
    """A single system of many small tile cells (27,000 waters with a 5 A
    cutoff: 37 x 37 columns of 60 z cells, more than one atom in few of them):
    the pair record of both precisions equals the oracle's pair set, FP64
    forces within 1e-11, mixed RMS within 1e-5."""
    w = systems.small_water(n_mol=27000, rc=5.0, rs=4.0)
    L = (27000 / systems.WATER_DENSITY) ** (1.0 / 3.0)
    assert int(L / 5.0) ** 2 * int(L / (5.0 / 3.0)) > 16384
    fc = w.make_force("mixed")
    assert fc.pair_path(w.topology) == "tile"
    fc.close()
    ref = O.evaluate(O.System.from_workload(w), record_pairs=True)
    ref_pairs = O.sorted_pairs(ref.pairs)
    print(w.name, w.n_atoms, "atoms, pairs", ref.n_pairs, flush=True)
    for precision in ("fp64", "mixed"):
        f, e, npairs, (_, fp) = run_gpu(w, precision, 0, with_pairs=False,
                                        force_pairs=True)
        print(precision, "pairs", npairs, flush=True)
        assert npairs == ref.n_pairs
        np.testing.assert_array_equal(fp, ref_pairs)
        if precision == "fp64":
            scale = max(1.0, np.abs(ref.forces).max())
            assert np.abs(f - ref.forces).max() <= 1e-11 * scale
        else:
            assert rms_rel(f, ref.forces) <= 1e-5


# ------------------------------------------------------------ general path
# Algorithm cutoff below the switching cutoff (the pair set is the one the
# reference's cell grid and delta list reach:
# CellListEnumeratorPeriodicBoundaries.h:46-83,114-134, CubicCellManager.cpp
# :53-59), and systems whose LJ table does not fit the tile kernel's LDS.  The
# oracle is bitwise equal to the reference's own build on these cases but the
# last (tests/test_oracle.py).
GENERAL = {
    # 6.5 A cell reach, 9 A C2 cutoff, 3 A cells: neighbour-list kernels
    "water_acut": (lambda: systems.with_algorithm(
        systems.small_water(n_mol=400), 6.5, 3.0), "list"),
    # 17.1 A box, 2.14 A cells: fewer cells than the reach spans, per-pair
    # minimum image in the list kernels
    "replica_acut": (lambda: systems.with_algorithm(
        systems.config3_replica(0, 167), 6.5, 2.0), "list"),
    # more than 512 cell offsets: the direct-scan kernels
    "water_scan": (lambda: systems.with_algorithm(
        systems.small_water(n_mol=300), 8.9, 1.5), "scan"),
    # 12 LJ types with 1-4 pairs: the tile kernel with its table in memory
    "chains_12types": (lambda: systems.many_type_chains(), "tile"),
    # the same with the first case's reach: neighbour-list kernels
    "chains_12types_acut": (lambda: systems.with_algorithm(
        systems.many_type_chains(), 6.5, 3.0), "list"),
}


@pytest.mark.parametrize("case", list(GENERAL))
def test_general_path_fp64(case):
    make, path = GENERAL[case]
    w = make()
    f = w.make_force("fp64")
    assert f.pair_path(w.topology) == path
    f.close()
    check_fp64(w)


@pytest.mark.parametrize("case", list(GENERAL))
def test_general_path_mixed(case):
    make, path = GENERAL[case]
    w = make()
    f = w.make_force("mixed")
    assert f.pair_path(w.topology) == path
    f.close()
    check_mixed(w)


def test_tile_path_is_taken_for_the_workloads():
    for w in (systems.config0(), systems.small_chains(n_chains=60),
              systems.config3_replica(0, 167), slab_water()):
        f = w.make_force("mixed")
        assert f.pair_path(w.topology) == "tile", w.name
        f.close()
