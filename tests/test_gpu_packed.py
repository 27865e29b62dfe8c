"""The wave engine (ktt_amd/kernels/coulomb_wave.h) against the FP64 oracle at every point, where it
can go wrong: sides whose rows wrap within a wave, end inside one or are shorter than a lane's run; atom
counts around a wave's 64-atom tile and the unrolled step; one wave, waves without atoms, and splits that
meet in several passes over the LDS. Wide blocks and large sides at sampled points.

Bars as for every form: 1e-5 plain, 1e-6 compensated, normalised by sum_i |q_i| / r_i."""

from __future__ import annotations

import numpy as np
import pytest

from ktt_amd import workloads
from oracle import coulomb_oracle as oracle

pytestmark = pytest.mark.gpu

BARS = {0: 1e-5, 1: 1e-6}


def run_guarded(capi, atoms, spacing, grid, form, config):
    """The map added onto zeros, with a guard behind it that must stay as it was."""
    atoms_buffer = capi.DeviceBuffer.from_array(atoms)
    start = np.zeros(grid ** 3 + 256, dtype=np.float32)
    start[grid ** 3:] = 7.0
    energy = capi.DeviceBuffer.from_array(start)
    capi.coulomb3d(atoms_buffer, atoms.shape[0], spacing, grid, energy, form=form, config=config)
    out = energy.download((grid ** 3 + 256,))
    assert (out[grid ** 3:] == 7.0).all()
    return out[:grid ** 3]


def check(capi, grid, count, form, config, spacing=0.5):
    atoms = workloads.uniform_atoms(1000 * grid + count, count, box=max(grid, 4) * spacing)
    z, y, x = np.meshgrid(*(np.arange(grid),) * 3, indexing="ij")
    points = np.stack([x.ravel(), y.ravel(), z.ravel()], axis=1).astype(np.int32)
    print(f"grid {grid} atoms {count} form {form} config {config}", flush=True)
    values, norms = oracle.points_f64(atoms, spacing, points)
    worst, rms = oracle.normalised_error(run_guarded(capi, atoms, spacing, grid, form, config), values, norms)
    assert worst <= BARS[form], (worst, rms)


def check_sampled(capi, grid, count, form, config, spacing=0.5):
    """As check, at sampled points, the grid's last row among them."""
    atoms = workloads.uniform_atoms(1000 * grid + count, count, box=grid * spacing)
    points = np.concatenate([workloads.sample_points(grid, 2048, grid),
                             np.array([[x, grid - 1, grid - 1] for x in range(grid)], dtype=np.int32)])
    print(f"grid {grid} atoms {count} form {form} config {config}", flush=True)
    values, norms = oracle.points_f64(atoms, spacing, points)
    out = run_guarded(capi, atoms, spacing, grid, form, config).reshape(grid, grid, grid)
    worst, rms = oracle.normalised_error(out[points[:, 2], points[:, 1], points[:, 0]], values, norms)
    assert worst <= BARS[form], (worst, rms)


@pytest.mark.parametrize("form", [0, 1])
@pytest.mark.parametrize("grid", [1, 2, 3, 6, 7, 16, 31, 33, 48, 65, 70])
def test_default_shapes(capi, grid, form):
    for count in (1, 64, 203):
        check(capi, grid, count, form, None)


@pytest.mark.parametrize("form", [0, 1])
@pytest.mark.parametrize("shape", ["POINTS_X=2,ROWS_PER_THREAD=8", "POINTS_X=1,ROWS_PER_THREAD=8", "POINTS_X=1,ROWS_PER_THREAD=4",
                                   "POINTS_X=3,ROWS_PER_THREAD=4"])
@pytest.mark.parametrize("waves,count", [(1, 7), (1, 65), (3, 257), (4, 521), (16, 9), (16, 1025)])
def test_splits(capi, shape, waves, count, form):
    check(capi, 45, count, form, f"WAVE_SPLIT={waves},{shape}")


@pytest.mark.parametrize("form", [0, 1])
@pytest.mark.parametrize("shape", ["POINTS_X=3,ROWS_PER_THREAD=8", "POINTS_X=4,ROWS_PER_THREAD=4", "POINTS_X=4,ROWS_PER_THREAD=8"])
@pytest.mark.parametrize("waves,count", [(1, 65), (16, 1025)])
def test_wide_blocks(capi, shape, waves, count, form):
    """The widest blocks a configuration may name (4 x 8 points spill registers), on rows they do not divide."""
    check_sampled(capi, 91, count, form, f"WAVE_SPLIT={waves},{shape}")


@pytest.mark.parametrize("form", [0, 1])
@pytest.mark.parametrize("grid,count", [(257, 100), (300, 1000), (513, 300)])
def test_default_above_256(capi, grid, count, form):
    """The default of sides above 256, up to 1,024, that 256 does not divide."""
    assert capi.coulomb3d_launch_plan(count, grid, form=form)["block"][1] == 1
    check_sampled(capi, grid, count, form, None)


@pytest.mark.parametrize("form", [0, 1])
def test_odd_spacings_and_far_atoms(capi, form):
    """A spacing that FP32 rounds, and atoms outside the box on both sides, some so far that their grid
    index passes 2^23 (where the compensated x offset is clamped)."""
    grid, spacing = 27, 0.49
    atoms = workloads.uniform_atoms(77, 90, box=20.0)
    atoms[:30, :3] -= 15.0
    atoms[30:33, 0] += np.float32(6.0e6)
    atoms[33:36, 0] -= np.float32(6.0e6)
    z, y, x = np.meshgrid(*(np.arange(grid),) * 3, indexing="ij")
    points = np.stack([x.ravel(), y.ravel(), z.ravel()], axis=1).astype(np.int32)
    values, norms = oracle.points_f64(atoms, spacing, points)
    for config in (None, "WAVE_SPLIT=4,POINTS_X=2,ROWS_PER_THREAD=8"):
        result = run_guarded(capi, atoms, spacing, grid, form, config)
        assert oracle.normalised_error(result, values, norms)[0] <= BARS[form]


def test_plain_coordinates_round_as_the_reference_does(capi):
    """A spacing FP32 rounds, atoms at float32(h * i): the reference generator forms the same rounded
    coordinate and finds distance 0 there (+-inf); so must the plain form's default launch."""
    grid, spacing = 30, np.float32(0.49)
    atoms = workloads.uniform_atoms(79, 60, box=14.0)
    cells = [(3, 17, 28), (29, 5, 11), (7, 7, 23)]
    for k, (x, y, z) in enumerate(cells):
        atoms[10 * k] = [spacing * np.float32(x), spacing * np.float32(y), spacing * np.float32(z), -0.5 if k else 0.5]
    cpu = oracle.coulomb3d_f32(atoms, spacing, grid)
    result = run_guarded(capi, atoms, float(spacing), grid, 0, None).reshape(grid, grid, grid)
    for x, y, z in cells:
        assert np.isinf(cpu[z, y, x]) and result[z, y, x] == cpu[z, y, x]
    finite = np.isfinite(cpu)
    assert np.array_equal(finite, np.isfinite(result))
    assert np.max(np.abs(result[finite] - cpu[finite])) <= 0.01


def test_repeats_are_bitwise_equal_and_bad_shapes_are_refused(capi):
    atoms = workloads.uniform_atoms(78, 700, box=20.0)
    for form in (0, 1):
        first = run_guarded(capi, atoms, 0.5, 40, form, "WAVE_SPLIT=16,POINTS_X=1,ROWS_PER_THREAD=4")
        second = run_guarded(capi, atoms, 0.5, 40, form, "WAVE_SPLIT=16,POINTS_X=1,ROWS_PER_THREAD=4")
        np.testing.assert_array_equal(first, second)
    for config in ("WAVE_SPLIT=17", "WAVE_SPLIT=0", "WAVE_SPLIT=2,POINTS_X=5", "WAVE_SPLIT=2,ROWS_PER_THREAD=6"):
        with pytest.raises(capi.KttHipError, match="WAVE_SPLIT"):
            run_guarded(capi, atoms, 0.5, 40, 0, config)


@pytest.mark.parametrize("grid_x,grid_y,count,config", [
    (64, 16, 1, None), (64, 16, 255, None), (128, 48, 257, None), (192, 32, 3000, None),
    (50, 37, 100, "WAVE_SPLIT=2,POINTS_X=2,ROWS_PER_THREAD=8,ATOM_BLOCKS=3"),
    (50, 37, 100, "WAVE_SPLIT=16,POINTS_X=1,ROWS_PER_THREAD=4"),
])
def test_slices(capi, grid_x, grid_y, count, config):
    """One slice (dz^2 in .z): the default launch of small slices, one and several atom blocks, and a grid
    that no workgroup tiles."""
    spacing = 0.5
    atoms = workloads.slice_dz2(workloads.uniform_atoms(80 + count, count, box=grid_x * spacing), 7.3)
    start = np.full(grid_x * grid_y + 64, 7.0, dtype=np.float32)
    start[:grid_x * grid_y] = 0.0
    energy = capi.DeviceBuffer.from_array(start)
    print(f"slice {grid_x} x {grid_y} atoms {count} config {config}", flush=True)
    capi.coulomb2d(capi.DeviceBuffer.from_array(atoms), count, spacing, grid_x, grid_y, energy, config=config)
    out = energy.download((grid_x * grid_y + 64,))
    assert (out[grid_x * grid_y:] == 7.0).all()
    y, x = np.meshgrid(np.arange(grid_y), np.arange(grid_x), indexing="ij")
    points = np.stack([x.ravel(), y.ravel()], axis=1).astype(np.int32)
    values, norms = oracle.points2d_f64(atoms, spacing, points)
    assert oracle.normalised_error(out[:grid_x * grid_y], values, norms)[0] <= BARS[0]


def test_slice_calls_take_wave_split(capi):
    """WAVE_SPLIT in the two iterative entry points: the planes of the volume launch that ktt_coulomb3d makes of the
    same configuration, bit for bit, and its refusals; sides the slice kernels do not tile stay refused."""
    grid, spacing = 128, 0.5
    atoms = workloads.uniform_atoms(81, 700, box=grid * spacing)
    atoms_buffer = capi.DeviceBuffer.from_array(atoms)
    energy = capi.DeviceBuffer(4 * grid ** 3)
    for config in ("WAVE_SPLIT=4,POINTS_X=1,ROWS_PER_THREAD=8", "WAVE_SPLIT=2"):
        volume = run_guarded(capi, atoms, spacing, grid, 0, config).reshape(grid, grid, grid)
        energy.zero()
        capi.coulomb3d_slices(atoms_buffer, atoms.shape[0], spacing, grid, energy, config=config)
        np.testing.assert_array_equal(energy.download((grid,) * 3), volume)
        energy.zero()
        capi.coulomb3d_iterative(atoms, spacing, grid, energy, config=config)
        np.testing.assert_array_equal(energy.download((grid,) * 3), volume)
    for config in ("WAVE_SPLIT=17", "WAVE_SPLIT=2,ROWS_PER_THREAD=6"):
        for call in (lambda: capi.coulomb3d_slices(atoms_buffer, atoms.shape[0], spacing, grid, energy, config=config),
                     lambda: capi.coulomb3d_iterative(atoms, spacing, grid, energy, config=config)):
            with pytest.raises(capi.KttHipError):
                call()
    for config in (None, "WAVE_SPLIT=4"):
        with pytest.raises(capi.KttHipError, match="multiple of the workgroup span"):
            capi.coulomb3d_slices(atoms_buffer, atoms.shape[0], spacing, 100, energy, config=config)


@pytest.mark.parametrize("grid,count", [(1, 5), (6, 30), (9, 100), (24, 700), (43, 600), (45, 300), (59, 600), (63, 64), (63, 600), (64, 300),
                                        (70, 3000), (76, 300), (100, 501), (127, 5)])
def test_no_alloc_entry_point_takes_the_same_shapes(capi, grid, count):
    """ktt_coulomb3d_compensated_noalloc at sides that run the wave engine, at least one for each of its
    precompiled kernels (ktt_core_tests checks that these sizes reach every one), against FP64 and ktt_coulomb3d."""
    spacing = 0.5
    atoms = workloads.uniform_atoms(90 + grid, count, box=max(grid, 4) * spacing)
    start = np.zeros(grid ** 3 + 64, dtype=np.float32)
    start[grid ** 3:] = 7.0
    energy = capi.DeviceBuffer.from_array(start)
    print(f"no-alloc grid {grid} atoms {count}", flush=True)
    capi.coulomb3d_compensated_noalloc(capi.DeviceBuffer.from_array(atoms), count, spacing, grid, energy)
    capi.synchronize()
    out = energy.download((grid ** 3 + 64,))
    assert (out[grid ** 3:] == 7.0).all()
    points = workloads.sample_points(91, 2048, grid)
    values, norms = oracle.points_f64(atoms, spacing, points)
    index = (points[:, 2].astype(np.int64) * grid + points[:, 1]) * grid + points[:, 0]
    assert oracle.normalised_error(out[index], values, norms)[0] <= BARS[1]
    other = run_guarded(capi, atoms, spacing, grid, 1, None)
    assert (np.abs(out[index].astype(np.float64) - other[index]) / norms).max() <= BARS[1]


@pytest.mark.parametrize("config", [None, "WAVE_SPLIT=1", "WAVE_SPLIT=5"])
@pytest.mark.parametrize("sides", [(3, 24, 31, 33, 66), (32, 48, 63, 64, 128), (7,), (6, 7, 48)])
def test_batches(capi, sides, config):
    """Batches whose sides fall into each class of points per lane, ragged and not, with no atoms in one
    system, against FP64 at sampled points; eager and graph launches agree bit for bit."""
    systems = []
    for k, side in enumerate(sides * 2):
        count = (0, 1, 65, 300, 701)[k % 5] if k else 513
        systems.append(workloads.BatchSystem(workloads.uniform_atoms(300 + k, count, box=max(side, 4) * 0.49), side, 0.49))
    batch = capi.Batch(systems, config=config)
    print("batch", sides, config, batch.info()["items"], batch.info()["shapes"], flush=True)
    batch.zero()
    batch.run(use_graph=False)
    grids = batch.grids()
    for k, (system, grid) in enumerate(zip(systems, grids)):
        if system.atoms.shape[0] == 0:
            assert (grid == 0.0).all()
            continue
        points = workloads.sample_points(400 + k, 500, system.grid)
        values, norms = oracle.points_f64(system.atoms, system.spacing, points)
        assert oracle.normalised_error(grid[points[:, 2], points[:, 1], points[:, 0]], values, norms)[0] <= BARS[1]
    for _ in range(2):
        batch.zero()
        batch.run(use_graph=True)
        for first, again in zip(grids, batch.grids()):
            np.testing.assert_array_equal(first, again)


@pytest.mark.parametrize("form", [0, 1])
@pytest.mark.parametrize("grid,count", [(117, 16), (127, 64), (251, 12), (255, 16)])
def test_few_atoms(capi, grid, count, form):
    """Sides of the wave engine whose few atoms run on the workgroup shapes in the plain form: the plan says so,
    and the map meets the bar at sampled points."""
    plan = capi.coulomb3d_launch_plan(count, grid, form=form)
    assert (plan["block"][1] > 1) == (form == 0), plan
    assert plan["scratch_bytes"] == 0
    atoms = workloads.uniform_atoms(500 + grid, count, box=grid * 0.5)
    print(f"few atoms: grid {grid} atoms {count} form {form}", flush=True)
    out = run_guarded(capi, atoms, 0.5, grid, form, None).reshape(grid, grid, grid)
    points = workloads.sample_points(501, 2048, grid)
    values, norms = oracle.points_f64(atoms, 0.5, points)
    assert oracle.normalised_error(out[points[:, 2], points[:, 1], points[:, 0]], values, norms)[0] <= BARS[form]
