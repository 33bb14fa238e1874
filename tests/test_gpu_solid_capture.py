"""Solid calls recorded into a HIP graph hold memory of the graph's own and none of
the stream's scratch: replays stay right after larger eager calls on the capture
stream have replaced that, and beside replays of other graphs of the stream; the
memory goes with the graph.  Linear (16-byte row groups, other whole words and
none), Morton, accumulating, coarse and fine meshes, runs that leave their row, and
a capture without any earlier call on its stream.  Bit for bit."""
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


# 96: rows of 3 words; 100: of no whole words; 500 < grid^2 / 4 <= 5000: a coarse mesh and a fine one
@pytest.mark.parametrize("grid,morton", [(128, False), (128, True), (96, False), (100, False)])
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


@pytest.mark.parametrize("grid,morton,accumulate", [(128, False, False), (128, True, False), (128, False, True),
                                                    (100, False, False), (100, False, True)])
def test_graphs_of_one_stream_beside_each_other(oracle, gpu, grid, morton, accumulate):
    import cuda_voxelizer_amd as V
    import torch
    graphs = []
    capture = torch.cuda.Stream()
    for k in range(3):
        info, tris, d = _mesh(gpu, 800 + 700 * k, grid, 30 + k)
        exp = oracle.solid(oracle.info_from_bytes(info.as_bytes()), tris, morton=morton)[0]
        table = torch.zeros(exp.size, dtype=torch.int32, device=gpu)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=capture):
            V.voxelize_solid_table(info, d, morton=morton, table=table, accumulate=accumulate)
        graphs.append((graph, table, exp, d, torch.cuda.Stream()))
    for _ in range(20):
        for _, table, _, _, _ in graphs:
            table.fill_(0x35)
        torch.cuda.synchronize()
        for graph, _, _, _, s in graphs:
            with torch.cuda.stream(s):
                graph.replay()
        torch.cuda.synchronize()
        for _, table, exp, _, _ in graphs:
            assert (table.cpu().numpy().view(np.uint32) == (exp ^ np.uint32(0x35) if accumulate else exp)).all()


def test_memory_goes_with_the_graph(gpu):
    import gc

    import cuda_voxelizer_amd as V
    import torch
    info, _, d = _mesh(gpu, 3000, 1024, 5)  # marker tables of 128 MB
    table = torch.zeros(V.table_words(1024), dtype=torch.int32, device=gpu)
    exp = V.voxelize_solid_table(info, d, morton=True).clone()

    def capture():
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            V.voxelize_solid_table(info, d, morton=True, table=table)
        return graph

    def free():
        gc.collect()
        torch.cuda.synchronize()
        V.release_scratch()
        return torch.cuda.mem_get_info()[0]

    capture()
    before = free()
    kept = capture()
    for _ in range(4):
        graph = capture()
        for g in (graph, kept):
            table.fill_(-1)
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(table, exp)
        del g, graph
    # the kept graph's table, and what the runtime has not let go yet
    assert before - free() <= (3 * 128 + 64) << 20
    table.fill_(-1)
    kept.replay()
    torch.cuda.synchronize()
    assert torch.equal(table, exp)
