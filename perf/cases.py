"""The workloads that this framework's speed is measured on.

Each case is one thing a user's program has the framework do, called as such a
program calls it: a surface or solid voxelization of a resident mesh
(``path`` "call"), the reference's synchronous drop-in form on a table that the
caller zeroes ("dropin"), a graph batch of many meshes ("batch"), and a mesh in
host memory taken all the way to the bytes of an output file ("file").

Meshes are the package's own workload shapes (cuda_voxelizer_amd/meshgen.py),
generated on the GPU from the seed: jittered icospheres and tori, displaced
spheres, tori with slivers, random triangle soups.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

import cuda_voxelizer_amd as V
from cuda_voxelizer_amd import io as vio
from cuda_voxelizer_amd import meshgen

DEVICE = "cuda:0"


def listed() -> list[dict]:
    return [
        # The smallest configuration: one call on a 64^3 grid, where launches and one
        # workgroup's chain of work are all there is.
        dict(name="surface_64_icosphere", path="call", mesh="icosphere", n=5_120, grid=64, morton=False, solid=False),
        # A grid edge that is no multiple of 32 and a ragged triangle count.
        dict(name="surface_200_torus", path="call", mesh="torus", n=26_866, grid=200, morton=False, solid=False),
        # Unordered triangles of very uneven sizes (broken scans, CAD soups).
        dict(name="surface_256_soup", path="call", mesh="soup", n=100_003, grid=256, morton=False, solid=False),
        # One million triangles, some degenerate, into the Morton layout.
        dict(name="surface_512_torus_morton", path="call", mesh="slivers", n=1_048_576, grid=512, morton=True,
             solid=False),
        # The headline: the same mesh at 1024^3, linear.
        dict(name="surface_1024_torus", path="call", mesh="slivers", n=1_048_576, grid=1024, morton=False, solid=False),
        # The largest grid of the reference's published table, with its mesh size (about 70k triangles).
        dict(name="surface_2048_sphere", path="call", mesh="displaced", n=81_920, grid=2048, morton=False, solid=False),
        # Solid fill of a coarse model: few triangles, each over many columns.
        dict(name="solid_256_coarse", path="call", mesh="icosphere", n=1_280, grid=256, morton=False, solid=True),
        # Solid fill into the Morton layout.
        dict(name="solid_512_sphere_morton", path="call", mesh="displaced", n=327_680, grid=512, morton=True, solid=True),
        # The largest single-grid configuration: 1.3 million triangles, solid, 1024^3.
        dict(name="solid_1024_sphere", path="call", mesh="displaced", n=1_310_720, grid=1024, morton=False, solid=True),
        # The reference's own calling convention: zero the table, voxelize into it, wait.
        dict(name="dropin_256_solid", path="dropin", mesh="icosphere", n=81_920, grid=256, morton=False, solid=True),
        # Many meshes of uneven sizes and grids in one graph launch.
        dict(name="batch_48_mixed", path="batch", count=48),
        # What the command line does: a mesh in host memory to the bytes of a .binvox file.
        dict(name="file_256_binvox", path="file", mesh="displaced", n=81_920, grid=256, morton=False, solid=False,
             fmt="binvox"),
    ]


def _log_uniform(rng, lo: float, hi: float) -> float:
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng) -> dict:
    path = rng.choice(["call"] * 7 + ["dropin", "batch", "file"])
    if path == "batch":
        return dict(path="batch", count=rng.randint(8, 48))
    solid = rng.random() < 0.45
    # soups are not closed, so they are surfaces; their triangles are large, so grids stay at 256
    mesh = rng.choice(["icosphere", "torus", "displaced"] if solid else ["icosphere", "torus", "displaced", "slivers",
                                                                         "soup"])
    morton = rng.random() < 0.3
    top = 256 if mesh == "soup" or path == "file" else 1024
    if morton:
        grid = 1 << rng.randint(5, int(math.log2(top)))
    else:
        grid = int(round(_log_uniform(rng, 32, top)))
        if rng.random() < 0.7:
            grid = max(32, grid // 32 * 32)
    # from coarse models (a triangle over some thousand voxels) up to the finest scans
    n = int(round(_log_uniform(rng, max(500, grid * grid / 64), 100_003 if mesh == "soup" else 1_310_720)))
    case = dict(path=path, mesh=mesh, n=n, grid=grid, morton=morton, solid=solid)
    if path == "file":
        case["fmt"] = "binvox" if solid or mesh == "soup" else rng.choice(["binvox", "binvox", "obj_points"])
    return case


# ---- meshes (float32 [n, 3, 3] on the GPU) ----------------------------------------------
@functools.lru_cache(maxsize=None)
def _icosphere(level: int):
    v, f = meshgen.icosphere(level)
    return torch.from_numpy(v).to(DEVICE), torch.from_numpy(f).to(DEVICE)


def _level(n: int) -> int:
    return max(0, min(8, round(math.log(max(n, 20) / 20.0, 4))))


def _torus_shape(n: int) -> tuple[int, int]:
    nu = max(3, round(math.sqrt(n)))
    return nu, max(3, round(n / (2 * nu)))


def triangles(mesh: str, n: int) -> int:
    if mesh in ("icosphere", "displaced"):
        return 20 * 4 ** _level(n)
    if mesh in ("torus", "slivers"):
        nu, nv = _torus_shape(n)
        return 2 * nu * nv
    return n


def _indexed(mesh: str, n: int, g: torch.Generator):
    """(float64 vertices, faces) of a closed mesh, in the order its generator makes them."""
    if mesh in ("icosphere", "displaced"):
        v, f = _icosphere(_level(n))
        if mesh == "icosphere":  # every vertex moved radially by up to 2 %
            r = 0.98 + 0.04 * torch.rand(v.shape[0], 1, generator=g, device=DEVICE, dtype=torch.float64)
        else:  # a low-frequency radial field, 0.85 .. 1.15
            w = 3.0 * torch.randn(3, 8, generator=g, device=DEVICE, dtype=torch.float64)
            a = torch.rand(8, generator=g, device=DEVICE, dtype=torch.float64) + 0.2
            p = 6.3 * torch.rand(8, generator=g, device=DEVICE, dtype=torch.float64)
            r = 1.0 + 0.15 * ((torch.sin(v @ w + p) * (a / a.sum())).sum(1, keepdim=True))
        return v * r, f
    nu, nv = _torus_shape(n)
    u = torch.arange(nu, device=DEVICE, dtype=torch.float64)[:, None] * (2.0 * math.pi / nu)
    w = torch.arange(nv, device=DEVICE, dtype=torch.float64)[None, :] * (2.0 * math.pi / nv)
    rad = 1.0 + 0.35 * torch.cos(w)
    v = torch.stack([rad * torch.cos(u), rad * torch.sin(u), (0.35 * torch.sin(w)).expand(nu, nv)], -1).reshape(-1, 3)
    v = v + 0.00035 * torch.randn(v.shape, generator=g, device=DEVICE, dtype=torch.float64)
    i = torch.arange(nu, device=DEVICE)[:, None]
    j = torch.arange(nv, device=DEVICE)[None, :]
    a, b = i * nv + j, (i + 1) % nu * nv + j
    c, d = (i + 1) % nu * nv + (j + 1) % nv, i * nv + (j + 1) % nv
    f = torch.stack([torch.stack([a, b, c], -1), torch.stack([a, c, d], -1)], 2).reshape(-1, 3)
    return v, f


def _aos(mesh: str, n: int, grid: int, g: torch.Generator) -> torch.Tensor:
    if mesh == "soup":
        t = torch.rand(n, 1, 3, generator=g, device=DEVICE, dtype=torch.float64).repeat(1, 3, 1)
        d = torch.randn(n, 2, 3, generator=g, device=DEVICE, dtype=torch.float64)
        d = d / d.norm(dim=2, keepdim=True)
        t[:, 1:] += d * torch.exp(torch.randn(n, 2, 1, generator=g, device=DEVICE, dtype=torch.float64) - 3.0)
    else:
        v, f = _indexed(mesh, n, g)
        t = v[f]
        if mesh == "slivers":  # every tenth triangle: one edge of 1e-4 voxels
            pick = torch.rand(t.shape[0], generator=g, device=DEVICE) < 0.1
            d = torch.randn(t.shape[0], 3, generator=g, device=DEVICE, dtype=torch.float64)
            unit = (v.amax(0) - v.amin(0)).max() / grid
            t[:, 1] = torch.where(pick[:, None], t[:, 0] + d / d.norm(dim=1, keepdim=True) * (1e-4 * unit), t[:, 1])
    return t.to(torch.float32).contiguous()


def _info(tris: torch.Tensor, grid: int):
    p = tris.reshape(-1, 3)
    box = V.AABox(p.amin(0).cpu().numpy(), p.amax(0).cpu().numpy())
    return V.VoxInfo(V.create_mesh_bbox_cube(box), (grid, grid, grid), tris.shape[0])


# ---- the batch's jobs: sizes from the case, the same for every seed ---------------------
def _batch_jobs(count: int) -> list[tuple[str, int, int]]:
    rng = np.random.Generator(np.random.PCG64(count))
    jobs = []
    for i in range(count):
        n = int(round(math.exp(rng.uniform(math.log(500), math.log(500_000)))))
        jobs.append((("icosphere", "torus", "soup")[i % 3], n, int(rng.choice((32, 64, 128, 256)))))
    return jobs


def prepare(case: dict, seed: int):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(int(seed))
    if case["path"] == "batch":
        jobs = []
        for mesh, n, grid in _batch_jobs(case["count"]):
            t = _aos(mesh, n, grid, g)
            table = torch.empty(V.table_words(grid), dtype=torch.int32, device=DEVICE)
            jobs.append(V.BatchJob(_info(t, grid), t.reshape(-1), table, solid=mesh != "soup"))
        return dict(case=case, jobs=jobs, batch=V.Batch(jobs))
    if case["path"] == "file":
        if case["mesh"] in ("soup", "slivers"):  # unshared vertices, as an STL file has them
            t = _aos(case["mesh"], case["n"], case["grid"], g)
            v, f = t.reshape(-1, 3), torch.arange(3 * t.shape[0], device=DEVICE).reshape(-1, 3)
        else:
            v, f = _indexed(case["mesh"], case["n"], g)
        # the file's image in memory, as large as such a mesh can need: the body's length depends on the mesh
        G = case["grid"]
        room = G ** 3 // 2 if case["mesh"] == "soup" else (768 if case["fmt"] == "obj_points" else 40) * G * G
        return dict(case=case, vertices=v.to(torch.float32).cpu().numpy(), faces=f.to(torch.int32).cpu().numpy(),
                    encoder=vio.Encoder(), file=np.zeros(room + 4096, np.uint8))
    tris = _aos(case["mesh"], case["n"], case["grid"], g)
    state = dict(case=case, info=_info(tris, case["grid"]), tris=tris.reshape(-1))
    if case["path"] == "dropin":
        state["table"] = torch.empty(V.table_words(case["grid"]), dtype=torch.int32, device=DEVICE)
    return state


def run(state):
    case = state["case"]
    if case["path"] == "batch":
        state["batch"].launch()
        return [j.table for j in state["jobs"]]
    if case["path"] == "file":
        info, tris = V.prepare_mesh(state["vertices"], state["faces"], case["grid"])
        voxelize = V.voxelize_solid_table if case["solid"] else V.voxelize_surface
        table = voxelize(info, tris, morton=case["morton"])
        body = state["encoder"].encode(table, case["grid"], case["morton"], vio.FORMATS[case["fmt"]])
        head = vio.binvox_header(info) if case["fmt"] == "binvox" else b""
        file = state["file"]
        file[:len(head)] = np.frombuffer(head, np.uint8)
        file[len(head):len(head) + len(body)] = np.frombuffer(body, np.uint8)
        return file
    if case["path"] == "dropin":
        table = state["table"]
        table.zero_()
        if case["solid"]:
            V.voxelize_solid(state["info"], state["tris"], table, morton_code=case["morton"])
        else:
            V.voxelize(state["info"], state["tris"], table, morton_code=case["morton"])
        return table
    voxelize = V.voxelize_solid_table if case["solid"] else V.voxelize_surface
    return voxelize(state["info"], state["tris"], morton=case["morton"])


def _one(mesh: str, n: int, grid: int) -> tuple[int, int]:
    """(bytes, float operations): triangles read, table written; each triangle's planes and edges set up once."""
    t = triangles(mesh, n)
    return 36 * t + (grid ** 3 + 31) // 32 * 4, 160 * t


def work(case: dict) -> dict:
    if case["path"] == "batch":
        parts = [_one(*j) for j in _batch_jobs(case["count"])]
        return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}
    b, f = _one(case["mesh"], case["n"], case["grid"])
    if case["path"] == "file":
        # the indexed mesh uploaded (about half as many vertices as faces), packed, voxelized, and the
        # table read into a body: a pair per 255 equal voxels and two per crossing of the shell
        t, G = triangles(case["mesh"], case["n"]), case["grid"]
        b += 18 * t + 36 * t + G ** 3 // 8 + 2 * (G ** 3 // 255 + 2 * G * G)
    return {"bytes": b, "flops": f}


def exact(case: dict, seed: int):
    """Tables and files are whole numbers and bytes, so there is nothing to compute more exactly."""
    return None
