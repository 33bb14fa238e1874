"""Solid calls recorded into a HIP graph hold none of the library's scratch
tables: replays stay right after larger eager calls on the capture stream have
replaced them.  Linear (16-byte row groups and other whole words), Morton,
accumulating, coarse and fine meshes, runs that leave their row, and a capture
without any earlier call on its stream.  Bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _mesh(gpu, n, grid, seed):
    import cuda_voxelizer_amd as V
    import torch
    from cuda_voxelizer_amd import meshgen
    tris = np.ascontiguousarray(meshgen.triangle_soup(n, seed=seed, mu=-2.0, sigma=0.6), np.float32)
    info = V.voxinfo_for_mesh(tris.reshape(-1, 3), grid, n)
    return info, tris, torch.from_numpy(tris.reshape(-1)).to(gpu)


# 96: rows of 3 words; 500 < grid^2 / 4 <= 5000: a coarse mesh and a fine one
@pytest.mark.parametrize("grid,morton", [(128, False), (128, True), (96, False)])
@pytest.mark.parametrize("accumulate", [False, True])
@pytest.mark.parametrize("n", [500, 5000])
@pytest.mark.parametrize("warm", [True, False])
def test_captured_solid(oracle, gpu, grid, morton, accumulate, n, warm):
    import cuda_voxelizer_amd as V
    import torch
    info, tris, d = _mesh(gpu, n, grid, 7)
    exp, count, _ = oracle.solid(oracle.info_from_bytes(info.as_bytes()), tris, morton=morton)
    big, big_tris, bd = _mesh(gpu, 3000, 256, 8)
    big_exp = oracle.solid(oracle.info_from_bytes(big.as_bytes()), big_tris, morton=morton)[0]
    table = torch.zeros(exp.size, dtype=torch.int32, device=gpu)
    off = torch.zeros(1, dtype=torch.int64, device=gpu)
    s = torch.cuda.Stream()
    if warm:
        with torch.cuda.stream(s):
            V.voxelize_solid_table(info, d, morton=morton, table=table, accumulate=accumulate)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        V.voxelize_solid_table(info, d, morton=morton, table=table, accumulate=accumulate, offrow=off)
    for _ in range(3):
        with torch.cuda.stream(s):
            got = V.voxelize_solid_table(big, bd, morton=morton)
        torch.cuda.synchronize()
        assert (got.cpu().numpy().view(np.uint32) == big_exp).all()
        table.fill_(0x35 if accumulate else -1)
        off.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert (table.cpu().numpy().view(np.uint32) == (exp ^ np.uint32(0x35) if accumulate else exp)).all()
        assert int(off.item()) == count
