"""The scratch tables kept for a device's streams: bounded together, given back on
request and when a thread with a stream of its own has ended, and allocated beside
another thread's graph capture."""
import ctypes
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MB = 1 << 20


def _mesh(gpu, n, grid, seed=3):
    import cuda_voxelizer_amd as V
    import torch
    from cuda_voxelizer_amd import meshgen
    tris = np.ascontiguousarray(meshgen.triangle_soup(n, seed=seed, mu=-2.5, sigma=0.6), np.float32)
    info = V.voxinfo_for_mesh(tris.reshape(-1, 3), grid, n)
    return info, tris, torch.from_numpy(tris.reshape(-1)).to(gpu)


def _free():
    import torch
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def test_tables_are_given_back(oracle, gpu):
    import cuda_voxelizer_amd as V
    import torch
    info, tris, d = _mesh(gpu, 3000, 512)
    table = torch.empty(V.table_words(512), dtype=torch.int32, device=gpu)
    exp = oracle.surface(oracle.info_from_bytes(info.as_bytes()), tris, morton=False)[0]
    streams = [torch.cuda.Stream() for _ in range(8)]
    for s in streams:  # a stream's first kernel takes 2 MB of the runtime's own for good
        with torch.cuda.stream(s):
            V.voxelize_surface(info, d, table=table)
    V.release_scratch()
    before = _free()
    for _ in range(2):
        for s in streams:
            with torch.cuda.stream(s):
                V.voxelize_surface(info, d, table=table)
            s.synchronize()
            assert (table.cpu().numpy().view(np.uint32) == exp).all()
        assert before - _free() >= 8 * 16 * MB
        V.release_scratch()
        assert before - _free() <= 4 * MB


def test_tables_of_ended_threads_are_given_back(gpu, capi):
    import cuda_voxelizer_amd as V
    import torch
    from cuda_voxelizer_amd import _capi
    info, _, d = _mesh(gpu, 500, 1024)  # tables of 128 MB
    table = torch.empty(V.table_words(1024), dtype=torch.int32, device=gpu)
    exp = V.voxelize_surface(info, d).clone()
    V.release_scratch()
    before = _free()

    def work():
        _capi.check(capi.vox_surface(ctypes.byref(info._c), d.data_ptr(), table.data_ptr(), 0, 0, 2))
        torch.cuda.synchronize()

    for _ in range(6):
        t = threading.Thread(target=work)
        t.start()
        t.join()
        assert torch.equal(table, exp)
    assert before - _free() <= 300 * MB  # the last thread's, and the one before at most
    V.release_scratch()


def test_tables_are_bounded(gpu):
    import cuda_voxelizer_amd as V
    import torch
    one = 8192 * MB  # 4096^3 bits; a stream without one works in the caller's table
    info, _, d = _mesh(gpu, 200, 4096)
    table = torch.empty(V.table_words(4096), dtype=torch.int32, device=gpu)
    exp = V.voxelize_solid_table(info, d, table=table, algo="tile").clone()
    total = torch.cuda.mem_get_info()[1]
    streams = [torch.cuda.Stream() for _ in range(total // 8 // one + 2)]
    V.release_scratch()
    assert torch.equal(table, exp)  # and torch has what it keeps for the comparison
    before = _free()
    for k, s in enumerate(streams):
        table.zero_()
        torch.cuda.synchronize()
        with torch.cuda.stream(s):
            V.voxelize_solid_table(info, d, table=table)
        s.synchronize()
        assert torch.equal(table, exp), k
    assert total // 8 - one <= before - _free() <= total // 8 + 256 * MB
    # the others idle: the last stream takes one of their tables
    small, _, sd = _mesh(gpu, 200, 128)
    for _ in range(80):
        V.voxelize_solid_table(small, sd)
    table.zero_()
    torch.cuda.synchronize()
    with torch.cuda.stream(streams[-1]):
        V.voxelize_solid_table(info, d, table=table)
    streams[-1].synchronize()
    assert torch.equal(table, exp)
    assert before - _free() <= total // 8 + 256 * MB
    V.release_scratch()
    assert before - _free() <= 256 * MB


@pytest.mark.parametrize("solid,grid", [(False, 640), (True, 640), (True, 100)])
def test_first_call_beside_a_capture(oracle, gpu, capi, solid, grid):
    import cuda_voxelizer_amd as V
    import torch
    from cuda_voxelizer_amd import _capi
    info, tris, d = _mesh(gpu, 700, grid)
    exp = (oracle.solid if solid else oracle.surface)(oracle.info_from_bytes(info.as_bytes()), tris, morton=False)[0]
    table = torch.empty(exp.size, dtype=torch.int32, device=gpu)
    x = torch.zeros(1000, device=gpu)
    stream = torch.cuda.Stream()
    V.release_scratch()
    errors = []

    def work():
        try:
            ptr = stream.cuda_stream
            if solid:
                _capi.check(capi.vox_solid(ctypes.byref(info._c), d.data_ptr(), table.data_ptr(), 0, 0, None, ptr))
            else:
                _capi.check(capi.vox_surface(ctypes.byref(info._c), d.data_ptr(), table.data_ptr(), 0, 0, ptr))
        except Exception as e:  # noqa: BLE001 - reported by the assertion below
            errors.append(e)

    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        x += 1
        t = threading.Thread(target=work)
        t.start()
        t.join()
        x += 1
    assert not errors
    torch.cuda.synchronize()
    assert (table.cpu().numpy().view(np.uint32) == exp).all()
    graph.replay()
    torch.cuda.synchronize()
    assert float(x[0]) == 2.0
