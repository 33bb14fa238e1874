"""GPU parity of the work shapes of a batch's jobs: triangles shared by 1 to 16 lanes
and by further parts, in every layout's form of the chunk kernel and in the marker
kernel, and the shapes that jobs have beside one of more than 1.6 million
triangles.  Bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (triangles, grid, Morton, solid, waves): 50, 75: layout-generic; 128, 256: blocked; 4096 and
# 65536 >> k: the last mesh that 16, 8, .. lanes share
JOBS = [(300, 64, False, False, 0), (300, 64, True, False, 0), (2000, 128, False, False, 0), (2000, 128, True, False, 0),
        (60, 50, False, False, 0), (60, 75, False, False, 1), (60, 75, False, False, 2), (1, 256, False, False, 0),
        (8192, 256, False, False, 0), (8193, 256, False, False, 0), (20480, 256, False, False, 0),
        (70000, 40, False, False, 0), (3, 33, False, False, 0),
        (300, 64, False, True, 0), (2000, 128, False, True, 0), (4096, 96, False, True, 0), (4097, 96, False, True, 0),
        (32768, 64, False, True, 0), (32769, 128, False, True, 0), (1, 96, False, True, 0), (9000, 128, True, True, 0)]


@pytest.mark.parametrize("beside", [0, 1_600_000])
@pytest.mark.parametrize("use_graph", [True, False])
def test_work_shapes(oracle, gpu, beside, use_graph):
    import cuda_voxelizer_amd as V
    import torch
    from cuda_voxelizer_amd import _capi, meshgen
    jobs, exp = [], []
    for k, (n, grid, morton, solid, waves) in enumerate(JOBS + ([(beside, 32, False, False, 0)] if beside else [])):
        mu = -2.0 if n < 3000 else (-3.5 if n < 100_000 else -6.0)
        tris = np.ascontiguousarray(meshgen.triangle_soup(n, seed=k, mu=mu, sigma=0.6), np.float32)
        info = V.voxinfo_for_mesh(tris.reshape(-1, 3), grid, n)
        oinfo = oracle.info_from_bytes(info.as_bytes())
        exp.append((oracle.solid if solid else oracle.surface)(oinfo, tris, morton=morton)[0])
        jobs.append(V.BatchJob(info, torch.from_numpy(tris.reshape(-1)).to(gpu),
                               torch.full((exp[-1].size,), -1, dtype=torch.int32, device=gpu), morton=morton,
                               solid=solid, tune=_capi.tune_waves(waves)))
    batch = V.Batch(jobs, use_graph=use_graph)
    for _ in range(2):
        batch.launch()
        torch.cuda.synchronize()
        for k, (j, e) in enumerate(zip(jobs, exp)):
            assert (j.table.cpu().numpy().view(np.uint32) == e).all(), JOBS[k] if k < len(JOBS) else beside
            j.table.fill_(-1)
    batch.close()
