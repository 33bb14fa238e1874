"""Coarse solids on large grids whose rows are no whole 16-byte groups run tile from
grid^2 / 24 triangles on: both sides of the line, accumulation, and a captured call
(which holds no workspace that a larger call replaces).  Bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GRID = 1216


@pytest.mark.parametrize("n", [GRID * GRID // 24, GRID * GRID // 24 + 1])
def test_both_sides(oracle, gpu, n):
    import cuda_voxelizer_amd as V
    import torch
    from cuda_voxelizer_amd import meshgen

    def mesh(count, grid):
        tris = np.ascontiguousarray(meshgen.triangle_soup(count, seed=count, mu=-5.0, sigma=0.6), np.float32)
        return V.voxinfo_for_mesh(tris.reshape(-1, 3), grid, count), tris, torch.from_numpy(tris.reshape(-1)).to(gpu)

    info, tris, d = mesh(n, GRID)
    host, count, _ = oracle.solid(oracle.info_from_bytes(info.as_bytes()), tris, morton=False)
    exp = torch.from_numpy(host.view(np.int32)).to(gpu)
    table = torch.full((exp.numel(),), -1, dtype=torch.int32, device=gpu)
    off = torch.zeros(1, dtype=torch.int64, device=gpu)
    for _ in range(2):
        off.zero_()
        V.voxelize_solid_table(info, d, table=table, offrow=off)
        assert torch.equal(table, exp) and int(off.item()) == count
    table.fill_(0x35)
    V.voxelize_solid_table(info, d, table=table, accumulate=True)
    assert torch.equal(table, exp ^ 0x35)
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        V.voxelize_solid_table(info, d, table=table)
    big, _, bd = mesh(2 * n, GRID + 32)
    for _ in range(2):
        with torch.cuda.stream(s):
            V.voxelize_solid_table(big, bd)
        torch.cuda.synchronize()
        table.fill_(-1)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(table, exp)
