"""Batches and runners on a device without room for their scratch tables: they
work in the jobs' tables.  Bit for bit."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MB = 1 << 20
JOBS = 40  # at 512^3: 640 MB of scratch tables


@pytest.fixture
def jobs(oracle, gpu):
    import cuda_voxelizer_amd as V
    import torch
    from cuda_voxelizer_amd import meshgen
    tris = np.ascontiguousarray(meshgen.triangle_soup(300, seed=8, mu=-2.0, sigma=0.6), np.float32)
    info = V.voxinfo_for_mesh(tris.reshape(-1, 3), 512, 300)
    exp = torch.from_numpy(oracle.surface(oracle.info_from_bytes(info.as_bytes()), tris, morton=False)[0].view(np.int32))
    d = torch.from_numpy(tris.reshape(-1)).to(gpu)
    out = [V.BatchJob(info, d, torch.empty(exp.numel(), dtype=torch.int32, device=gpu)) for _ in range(JOBS)]
    yield out, exp.to(gpu)
    out.clear()
    torch.cuda.empty_cache()


def _check(jobs, exp):
    import torch
    torch.cuda.synchronize()
    for k, j in enumerate(jobs):
        assert torch.equal(j.table, exp), k
        j.table.fill_(-1)
    torch.cuda.synchronize()


def _fill_device(gpu):
    """All but 400 MB of the device's memory."""
    import torch
    torch.cuda.synchronize()
    held = [torch.empty(torch.cuda.mem_get_info()[0] - 2000 * MB, dtype=torch.uint8, device=gpu)]
    while torch.cuda.mem_get_info()[0] > 400 * MB:  # what is free after a large allocation is not the difference
        held.append(torch.empty(64 * MB, dtype=torch.uint8, device=gpu))
    return held


@pytest.mark.parametrize("use_graph", [True, False])
def test_batch_without_room(jobs, gpu, use_graph):
    import cuda_voxelizer_amd as V
    jobs, exp = jobs
    for full in (False, True, False):
        room = _fill_device(gpu) if full else None
        batch = V.Batch(jobs, use_graph=use_graph)
        assert (batch.info()["workspace_bytes"] >= JOBS * 16 * MB) == (not full)
        for _ in range(2):
            batch.launch()
            _check(jobs, exp)
        batch.close()
        del room
        _empty()


def _empty():
    import torch
    torch.cuda.empty_cache()


def test_runner_without_room(jobs, gpu, capi):
    import torch
    from cuda_voxelizer_amd import _capi
    jobs, exp = jobs
    items = (_capi.vox_batch_item * JOBS)()
    for it, j in zip(items, jobs):
        ctypes.memmove(ctypes.addressof(it.info), ctypes.addressof(j.info._c), 64)
        it.d_tris, it.d_table = j.tris.data_ptr(), j.table.data_ptr()
    stream = torch.cuda.current_stream().cuda_stream
    for full in (False, True):
        h = ctypes.c_void_p()
        _capi.check(capi.vox_runner_create(stream, ctypes.byref(h)))
        _capi.check(capi.vox_runner_launch(h, items, 10))  # 160 MB of scratch
        _check(jobs[:10], exp)
        room = _fill_device(gpu) if full else None
        try:
            for _ in range(2):
                _capi.check(capi.vox_runner_launch(h, items, JOBS))
                _check(jobs, exp)
        finally:
            torch.cuda.synchronize()
            capi.vox_runner_destroy(h)
            del room
            _empty()
