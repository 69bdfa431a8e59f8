"""Systems whose atoms do not fill their box evenly, against the FP64 oracle
with the bars of test_gpu_parity (pair sets bit for bit, FP64 forces within
1e-11 of the largest component, mixed forces within 1e-5 RMS): the cell grid
is laid out from the box and the number of atoms alone, the atoms may be
anywhere in it."""
import time

import numpy as np
import pytest

from oracle import oracle as O
from protomoladdon_amd import systems
from protomoladdon_amd._lib import PmnbError
from protomoladdon_amd.batch import BatchedCutoffForce
from protomoladdon_amd.topology import PeriodicBoundaryConditions
from tests.test_gpu_batch import batch_eval, single_eval
from tests.test_gpu_parity import check_fp64, check_mixed, rms_rel

pytestmark = pytest.mark.gpu


def dimers(n_pairs, L, cell_size=50.0):
    """Pairs of waters, oxygens 2.8 to 3.2 A or 8.9 to 9.1 A apart (the
    cutoff is 9 A), far from all other pairs."""
    w = systems.water_workload("dimers", 2 * n_pairs, L, 6, 9.0, 7.5, "ewald",
                               0.32, cell_size=cell_size)
    rng = np.random.default_rng(7)
    k = int(np.ceil(n_pairs ** (1 / 3)))
    site = np.stack(np.unravel_index(np.arange(n_pairs), (k, k, k)), 1)
    room = min(9.0, 0.5 * (L / k - 15.0))
    O = (site + 0.5) * (L / k) + rng.uniform(-room, room, (n_pairs, 3))
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


@pytest.mark.parametrize("n_pairs,L", [(300, 2400.0), (400, 150.0)])
def test_dimers_in_a_wide_box(n_pairs, L):
    """2,400 A: with columns and cells far wider than the cutoff the FP32
    offsets in a cell lose the pairs near the cutoff.  150 A: work items whose
    atoms spread beyond the expanded distance test."""
    check_fp64(dimers(n_pairs, L))
    check_mixed(dimers(n_pairs, L))


def test_box_beyond_the_tile_grid():
    """3,800 A are more than 2^26 cells of a 9 A cutoff: one system takes the
    cell grid of its cell size, a batch refuses the box."""
    w = dimers(200, 3800.0, 16.0)
    f = w.make_force("mixed")
    assert f.pair_path(w.topology) != "tile"
    f.close()
    check_fp64(w)
    check_mixed(w)
    bf = BatchedCutoffForce.from_workloads([w], precision="mixed")
    with pytest.raises(PmnbError) as e:
        batch_eval(bf, [w])
    assert e.value.code == 3  # PMNB_ERR_UNSUPPORTED
    bf.close()


def dense_in_wide_box(n_mol, L, squeeze):
    """A cube of water, squeezed by `squeeze` per axis, in a corner of a box
    of L."""
    w = systems.small_water(n_mol=n_mol)
    w.positions = w.positions * squeeze
    w.topology.boundary_conditions = PeriodicBoundaryConditions(
        (L, 0, 0), (0, L, 0), (0, 0, L), (0.5 * L,) * 3)
    return w


@pytest.mark.parametrize("n_mol,L,squeeze", [
    (700, 60.0, 0.62),    # no bin beyond what a block sorts in LDS
    (2500, 150.0, 0.5),   # bins of over 1,024 atoms
    (1500, 150.0, 0.12),  # z cells of over 256 atoms
    (2000, 2400.0, 1.0),  # bucket rows shorter than the bins' atoms
])
def test_dense_part_of_a_box(n_mol, L, squeeze):
    w = dense_in_wide_box(n_mol, L, squeeze)
    check_fp64(systems.with_algorithm(w, 9.0, max(4.5, L / 48)))


@pytest.mark.parametrize("precision", ["mixed", "fp64"])
def test_replicas_of_many_bins(precision):
    """Replicas whose bins are counted by groups between others, each as it
    gives alone."""
    ws = [systems.config3_replica(i, n) for i, n in enumerate((40, 300, 700, 90))]
    for w, L in ((ws[1], 640.0), (ws[2], 620.0)):
        w.topology.boundary_conditions = PeriodicBoundaryConditions(
            (L, 0, 0), (0, L, 0), (0, 0, 1.5 * L), (0.5 * L,) * 3)
    bf = BatchedCutoffForce.from_workloads(ws, precision=precision)
    frc, out = batch_eval(bf, ws)[1:]
    n = bf.pair_count()
    total = 0
    for r, w in enumerate(ws):
        f1, o1, n1 = single_eval(w, precision)
        ref = O.evaluate(O.System.from_workload(w, flags=1))
        total += n1
        assert n1 == ref.n_pairs
        a, b = bf.offsets[r], bf.offsets[r + 1]
        np.testing.assert_array_equal(frc[a:b], f1)
        np.testing.assert_array_equal(out[r], o1)
        assert rms_rel(f1, ref.forces) <= (1e-5 if precision == "mixed" else
                                           1e-12)
    bf.close()
    assert n == total


@pytest.mark.parametrize("precision", ["mixed", "fp64"])
def test_no_finite_position_takes_no_time(precision):
    """All atoms in one z cell of one bin: sorted in linear time (a sort by
    comparison of all pairs of 30,000 atoms takes seconds)."""
    import torch
    w = systems.small_water(n_mol=10000)
    f = w.make_force(precision)
    x = torch.full((w.n_atoms, 3), float("nan"), dtype=torch.float64,
                   device="cuda")
    frc = torch.zeros_like(x)
    out = torch.zeros(20, dtype=torch.float64, device="cuda")
    f.evaluate_device(w.topology, x, frc, out, 0)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    f.evaluate_device(w.topology, x, frc, out, 0)
    torch.cuda.synchronize()
    ms = 1e3 * (time.perf_counter() - t0)
    n = f.last_pair_count()
    f.close()
    print("%d atoms %.2f ms" % (w.n_atoms, ms), flush=True)
    assert n == 0 and not frc.abs().max().item()
    assert ms < 100.0
