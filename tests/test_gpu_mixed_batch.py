"""GPU parity of batch jobs that share one launch of the layout-generic chunk
kernel: jobs whose workgroups loop over several chunks (dense tables of many
triangles) beside jobs whose chunks are split into parts (coarse meshes on grids
whose rows are no whole words).  Bit for bit, as a graph, as plain launches and
through a runner."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# 32 and 40: loops over two and more chunks; 50, 75 and 700: coarse, not blocked in a batch
LOOPING = [(70_000, 32), (140_003, 40)]
SPLIT = [(500, 50), (130, 75), (3000, 700)]


def _jobs(oracle, gpu, sizes):
    import cuda_voxelizer_amd as V
    import torch
    from cuda_voxelizer_amd import meshgen
    jobs, exp = [], []
    for k, (n, grid) in enumerate(sizes):
        tris = np.ascontiguousarray(meshgen.triangle_soup(n, seed=40 + k, mu=-2.0, sigma=0.6), np.float32)
        info = V.voxinfo_for_mesh(tris.reshape(-1, 3), grid, n)
        exp.append(oracle.surface(oracle.info_from_bytes(info.as_bytes()), tris, morton=False)[0])
        table = torch.full((exp[-1].size,), -1, dtype=torch.int32, device=gpu)
        jobs.append(V.BatchJob(info, torch.from_numpy(tris.reshape(-1)).to(gpu), table))
    return jobs, exp


def _check(jobs, exp):
    import torch
    torch.cuda.synchronize()
    for j, e in zip(jobs, exp):
        assert (j.table.cpu().numpy().view(np.uint32) == e).all(), (j.info.n_triangles, j.info.grid)
        j.table.fill_(-1)


@pytest.mark.parametrize("sizes", [SPLIT, LOOPING + SPLIT, SPLIT + LOOPING], ids=["split", "loop+split", "split+loop"])
@pytest.mark.parametrize("use_graph", [True, False])
def test_looping_jobs_beside_split_ones(oracle, gpu, sizes, use_graph):
    import cuda_voxelizer_amd as V
    jobs, exp = _jobs(oracle, gpu, sizes)
    batch = V.Batch(jobs, use_graph=use_graph)
    for _ in range(2):
        batch.launch()
        _check(jobs, exp)
    batch.close()


def test_looping_jobs_beside_split_ones_in_a_runner(oracle, gpu, capi):
    import torch
    from cuda_voxelizer_amd import _capi
    jobs, exp = _jobs(oracle, gpu, LOOPING + SPLIT)
    items = (_capi.vox_batch_item * len(jobs))()
    for it, j in zip(items, jobs):
        ctypes.memmove(ctypes.addressof(it.info), ctypes.addressof(j.info._c), 64)
        it.d_tris, it.d_table = j.tris.data_ptr(), j.table.data_ptr()
    h = ctypes.c_void_p()
    _capi.check(capi.vox_runner_create(torch.cuda.current_stream().cuda_stream, ctypes.byref(h)))
    try:
        for _ in range(2):
            _capi.check(capi.vox_runner_launch(h, items, len(jobs)))
            _check(jobs, exp)
    finally:
        torch.cuda.synchronize()
        capi.vox_runner_destroy(h)
