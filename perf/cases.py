"""Performance cases of the Coulomb and N-body paths, through the package's public entry points.

Each case is one call a user's program makes: a potential map of a molecule on a cubic grid (the
whole volume in either form, slice by slice with dz^2 formed on the device or on the host, or one
slice alone), a batch of independent systems, or one step of the N-body sibling. A pass clears
the output map and adds the potential into it, as every caller has to (the kernels add).

Inputs are the seeded generators of ktt_amd.workloads: uniform atoms with charges of both signs,
or the reference example's own workload. ``exact`` sums the same inputs in 64 bits.
"""

from __future__ import annotations

import math

import numpy as np
import torch

from ktt_amd import capi, workloads

# Examples/Nbody/Nbody.cpp:71-73
NBODY_DT, NBODY_DAMPING, NBODY_SOFT2 = 0.001, 0.5, 0.01

# Most grid-point x atom interactions of one case: the 256^3 x 65,536 map.
MOST_INTERACTIONS = 256 ** 3 * 65536


def listed() -> list[dict]:
    return [
        # The smallest system of the mixed batches, called alone: launch cost and latency.
        {"name": "volume_32_plain", "kind": "volume", "form": "plain", "grid": 32, "atoms": 200, "spacing": 0.5},
        # One small molecule, compensated.
        {"name": "volume_64_comp", "kind": "volume", "form": "compensated", "grid": 64, "atoms": 5000, "spacing": 0.5},
        # A grid side and an atom count that no tile divides.
        {"name": "volume_99_plain", "kind": "volume", "form": "plain", "grid": 99, "atoms": 3001, "spacing": 0.5},
        {"name": "volume_150_comp", "kind": "volume", "form": "compensated", "grid": 150, "atoms": 20011, "spacing": 0.49},
        # The reference CoulombSum3d example's own workload (CoulombSum3d.cpp:67-98).
        {"name": "reference_example", "kind": "volume", "form": "plain", "grid": 256, "atoms": 64, "spacing": 0.5, "box": 20.0,
         "positive": True},
        # The benchmark's headline map: the largest case.
        {"name": "volume_256_comp", "kind": "volume", "form": "compensated", "grid": 256, "atoms": 65536, "spacing": 0.5},
        # The entry point that allocates nothing, on the size its callers test with.
        {"name": "noalloc_160", "kind": "noalloc", "grid": 160, "atoms": 600, "spacing": 0.5},
        # CoulombSum2d: one slice of the example's size.
        {"name": "slice_256", "kind": "slice2d", "grid_x": 256, "grid_y": 256, "atoms": 4000, "spacing": 0.5},
        # CoulombSum3dIterative with dz^2 formed on the device, and with the reference launcher's host dz^2.
        {"name": "slices_128", "kind": "slices", "grid": 128, "atoms": 8192, "spacing": 0.5},
        {"name": "iterative_128", "kind": "iterative", "grid": 128, "atoms": 2000, "spacing": 0.5},
        # Many independent systems of mixed sizes (the benchmark's distribution, fewer of them).
        {"name": "batch_128", "kind": "batch", "systems": 128, "sides": "32,48,64,96,128", "min_atoms": 200, "max_atoms": 20000,
         "spacing": 0.5},
        # One step of the N-body sibling, between the tests' 4,096 and the example's 131,072 bodies.
        {"name": "nbody_16384", "kind": "nbody", "bodies": 16384},
    ]


def _log_int(rng, low: int, high: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng) -> dict:
    """One more case of the same kinds and ranges; sides and atom counts over their logarithm."""
    while True:
        kind = rng.choice(["volume", "volume", "volume", "noalloc", "slice2d", "slices", "iterative", "batch", "nbody"])
        spacing = rng.choice([0.25, 0.49, 0.5, 1.0])
        if kind == "nbody":
            return {"kind": kind, "bodies": 1024 * _log_int(rng, 1, 128)}
        if kind == "batch":
            sides = sorted(rng.sample(range(24, 129), rng.randint(1, 5)))
            return {"kind": kind, "systems": _log_int(rng, 8, 160), "sides": ",".join(str(s) for s in sides), "min_atoms": 200,
                    "max_atoms": _log_int(rng, 500, 20000), "spacing": spacing}
        atoms = _log_int(rng, 64, 65536)
        if kind == "slice2d":
            return {"kind": kind, "grid_x": 64 * rng.randint(1, 8), "grid_y": 16 * rng.randint(2, 32), "atoms": atoms, "spacing": spacing}
        if kind in ("slices", "iterative"):
            # The slice kernels need rows that their workgroups tile.
            case = {"kind": kind, "grid": 64 * rng.randint(1, 4), "atoms": min(atoms, 16384), "spacing": spacing}
        else:
            case = {"kind": kind, "grid": _log_int(rng, 24, 256), "atoms": atoms, "spacing": spacing}
            if kind == "volume":
                case["form"] = rng.choice(["plain", "compensated"])
        if case["grid"] ** 3 * case["atoms"] <= MOST_INTERACTIONS:
            return case


def _box(case: dict) -> float:
    return float(case.get("box", case["spacing"] * case.get("grid", case.get("grid_x", 0))))


def _host_atoms(case: dict, seed: int) -> np.ndarray:
    """float4 atoms (x, y, z, q) in the grid's box; a slice's atoms hold dz^2 to its middle plane in z."""
    atoms = workloads.uniform_atoms(seed, case["atoms"], _box(case))
    if case.get("positive"):  # q = U[0, 20) / 40, as the example draws it
        atoms[:, 3] = workloads.uniform01(seed, case["atoms"], stream=1) * np.float32(0.5)
    if case["kind"] == "slice2d":
        atoms = workloads.slice_dz2(atoms, 0.5 * _box(case))
    return atoms


def _systems(case: dict, seed: int) -> list:
    sides = tuple(int(s) for s in case["sides"].split(","))
    # Counts and sides by the case alone, so that every seed is the same work; atoms by the seed.
    systems = workloads.batch(systems=case["systems"], min_atoms=case["min_atoms"], max_atoms=case["max_atoms"],
                              spacing=case["spacing"], sides=sides)
    for k, system in enumerate(systems):
        system.atoms = workloads.uniform_atoms(seed * 1000003 + k, system.atoms.shape[0], system.grid * system.spacing, stream=3)
    return systems


def _bodies(case: dict, seed: int) -> tuple[np.ndarray, np.ndarray]:
    n = case["bodies"]
    position = workloads.uniform01(seed, 4 * n, stream=1).reshape(n, 4) * np.float32(20.0)  # x, y, z, mass
    velocity = workloads.uniform01(seed, 4 * n, stream=2).reshape(n, 4) * np.float32(20.0)
    velocity[:, 3] = 0.0
    return position, velocity


class _View:
    """Device memory for a torch tensor without a copy; the tensor keeps the view and so the owner."""

    def __init__(self, owner, pointer: int, shape: tuple):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f4", "data": (pointer, False), "version": 2}


def _tensor(owner, pointer: int, shape: tuple) -> torch.Tensor:
    return torch.as_tensor(_View(owner, pointer, shape), device="cuda")


def _points_shape(case: dict) -> tuple:
    if case["kind"] == "slice2d":
        return (case["grid_y"], case["grid_x"])
    return (case["grid"],) * 3


def prepare(case: dict, seed: int) -> dict:
    state = {"case": case}
    if case["kind"] == "batch":
        batch = capi.Batch(_systems(case, seed))
        info = batch.info()
        state.update(batch=batch, out=_tensor(batch, info["grids"].value, (info["points"],)))
    elif case["kind"] == "nbody":
        n = case["bodies"]
        position, velocity = _bodies(case, seed)
        state.update(bodies=capi.DeviceBuffer.from_array(position), velocity=capi.DeviceBuffer.from_array(velocity),
                     new_bodies=capi.DeviceBuffer(16 * n), new_velocity=capi.DeviceBuffer(16 * n))
        state["out"] = {key: _tensor(state[key], state[key].ptr.value, (n, 4)) for key in ("new_bodies", "new_velocity")}
    else:
        atoms = _host_atoms(case, seed)
        shape = _points_shape(case)
        # The host launcher takes the atoms from host memory on every call; the others from the device.
        state["atoms"] = atoms if case["kind"] == "iterative" else capi.DeviceBuffer.from_array(atoms)
        state["energy"] = capi.DeviceBuffer(4 * int(np.prod(shape)))
        state["out"] = _tensor(state["energy"], state["energy"].ptr.value, shape)
    return state


def run(state: dict):
    case = state["case"]
    kind = case["kind"]
    if kind == "batch":
        state["batch"].zero()
        state["batch"].run(use_graph=True, timed=False)
        return state["out"]
    if kind == "nbody":
        capi.nbody_step(state["bodies"], state["velocity"], case["bodies"], NBODY_DT, NBODY_DAMPING, NBODY_SOFT2,
                        state["new_bodies"], state["new_velocity"])
        return state["out"]
    atoms, energy, n, h = state["atoms"], state["energy"], case["atoms"], case["spacing"]
    energy.zero()
    if kind == "volume":
        form = capi.COMPENSATED if case["form"] == "compensated" else capi.PLAIN
        capi.coulomb3d(atoms, n, h, case["grid"], energy, form=form, timed=False)
    elif kind == "noalloc":
        capi.coulomb3d_compensated_noalloc(atoms, n, h, case["grid"], energy)
    elif kind == "slice2d":
        capi.coulomb2d(atoms, n, h, case["grid_x"], case["grid_y"], energy, timed=False)
    elif kind == "slices":
        capi.coulomb3d_slices(atoms, n, h, case["grid"], energy, timed=False)
    else:
        capi.coulomb3d_iterative(atoms, h, case["grid"], energy)
    return state["out"]


def work(case: dict) -> dict:
    """Each atom read once, each point written once; 11 operations per interaction (3 sub, 3 mul and 2
    add for r^2, the inverse square root, the product with q and its addition), 20 for N-body."""
    if case["kind"] == "nbody":
        return {"bytes": 64 * case["bodies"], "flops": 20 * case["bodies"] ** 2}
    if case["kind"] == "batch":
        systems = _systems(case, 0)
        return {"bytes": sum(16 * s.atoms.shape[0] + 4 * s.grid ** 3 for s in systems),
                "flops": 11 * sum(s.interactions for s in systems)}
    points = int(np.prod(_points_shape(case)))
    return {"bytes": 16 * case["atoms"] + 4 * points, "flops": 11 * points * case["atoms"]}


def tolerance(case: dict) -> dict:
    # Four times the largest errors against exact() over these ranges. A step adds a small update to
    # each body: 9e-8 and 8e-7. A map sums up to 65,536 terms of both signs in 32 bits, and a point
    # close to an atom carries the rounding of its coordinates: 3.4e-6 and 3.1e-4.
    if case["kind"] == "nbody":
        return {"rel": 4e-7, "max": 4e-6}
    return {"rel": 1.4e-5, "max": 1.2e-3}


def _potential64(atoms: np.ndarray, h: float, grid_x: int, planes: list, rows: int) -> torch.Tensor:
    """V of one system in 64 bits over rows x grid_x points of every plane; planes holds each plane's
    dz^2 to every atom, or its z coordinate."""
    device = torch.device("cuda")
    a = torch.from_numpy(atoms).to(device, torch.float64)
    x, y, z, q = a.unbind(1)
    dx2 = (h * torch.arange(grid_x, device=device, dtype=torch.float64)[:, None] - x) ** 2
    dy2 = (h * torch.arange(rows, device=device, dtype=torch.float64)[:, None] - y) ** 2
    out = torch.empty(len(planes), rows, grid_x, device=device, dtype=torch.float64)
    step = max(1, (1 << 28) // max(1, grid_x * len(atoms)))
    for k, plane in enumerate(planes):
        dz2 = z if plane is None else (plane - z) ** 2
        for first in range(0, rows, step):
            bracket = dy2[first:first + step] + dz2
            r = (bracket[:, None, :] + dx2[None, :, :]).rsqrt_()
            out[k, first:first + step] = r.reshape(-1, len(atoms)).mv(q).reshape(-1, grid_x)
    return out


def exact(case: dict, seed: int):
    h = float(np.float32(case.get("spacing", 0.0)))
    if case["kind"] == "batch":
        return torch.cat([_potential64(s.atoms, h, s.grid, [h * k for k in range(s.grid)], s.grid).reshape(-1)
                          for s in _systems(case, seed)])
    if case["kind"] == "nbody":
        position, velocity = (torch.from_numpy(v).to("cuda", torch.float64) for v in _bodies(case, seed))
        acceleration = torch.empty_like(position[:, :3])
        for first in range(0, case["bodies"], 1024):
            d = position[None, :, :3] - position[first:first + 1024, None, :3]
            s = position[:, 3] * (d.square().sum(2) + NBODY_SOFT2) ** -1.5
            acceleration[first:first + 1024] = (d * s[:, :, None]).sum(1)
        moved, faster = position.clone(), torch.zeros_like(velocity)
        moved[:, :3] += NBODY_DT * velocity[:, :3] + NBODY_DAMPING * NBODY_DT ** 2 * acceleration
        faster[:, :3] = velocity[:, :3] + NBODY_DT * acceleration
        return {"new_bodies": moved, "new_velocity": faster}
    atoms = _host_atoms(case, seed)
    if case["kind"] == "slice2d":
        return _potential64(atoms, h, case["grid_x"], [None], case["grid_y"])[0]
    return _potential64(atoms, h, case["grid"], [h * k for k in range(case["grid"])], case["grid"])
