"""One batch launched on several streams and by several threads: its launches share
its scratch tables and workspaces.  Surfaces, solids of every class, an
accumulating job.  Bit for bit."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("use_graph", [True, False])
@pytest.mark.parametrize("threads", [False, True])
def test_launches_on_several_streams(oracle, gpu, use_graph, threads):
    import cuda_voxelizer_amd as V
    import torch
    from cuda_voxelizer_amd import meshgen
    jobs, exp = [], []
    # (triangles, grid, solid, accumulate, algorithm)
    for k, (n, grid, solid, acc, algo) in enumerate([(9000, 256, False, False, "auto"), (33000, 128, False, True, "auto"),
                                                     (2000, 100, False, False, "auto"), (3000, 128, True, False, "auto"),
                                                     (3000, 128, True, False, "tile"), (3000, 128, False, False, "tile")]):
        tris = np.ascontiguousarray(meshgen.triangle_soup(n, seed=60 + k, mu=-2.5, sigma=0.6), np.float32)
        info = V.voxinfo_for_mesh(tris.reshape(-1, 3), grid, n)
        oinfo = oracle.info_from_bytes(info.as_bytes())
        exp.append((oracle.solid if solid else oracle.surface)(oinfo, tris, morton=False)[0])
        jobs.append(V.BatchJob(info, torch.from_numpy(tris.reshape(-1)).to(gpu),
                               torch.zeros(exp[-1].size, dtype=torch.int32, device=gpu), solid=solid, accumulate=acc,
                               algo=algo))
    batch = V.Batch(jobs, use_graph=use_graph)
    streams = [torch.cuda.Stream() for _ in range(3)]
    for _ in range(10):
        for j in jobs:
            j.table.fill_(0 if j.accumulate else -1)
        torch.cuda.synchronize()
        if threads:
            each = [threading.Thread(target=lambda s=s: [batch.launch(stream=s) for _ in range(4)]) for s in streams]
            for t in each:
                t.start()
            for t in each:
                t.join()
        else:
            for k in range(12):
                batch.launch(stream=streams[k % 3])
        torch.cuda.synchronize()
        for k, (j, e) in enumerate(zip(jobs, exp)):
            assert (j.table.cpu().numpy().view(np.uint32) == e).all(), k
    batch.close()


@pytest.mark.parametrize("other_thread", [False, True])
def test_beside_a_capture(oracle, gpu, other_thread):
    """Waits and frees of the library leave a capture under way valid."""
    import cuda_voxelizer_amd as V
    import torch
    from cuda_voxelizer_amd import meshgen
    tris = np.ascontiguousarray(meshgen.triangle_soup(3000, seed=9, mu=-2.5, sigma=0.6), np.float32)
    info = V.voxinfo_for_mesh(tris.reshape(-1, 3), 128, len(tris))
    oinfo = oracle.info_from_bytes(info.as_bytes())
    surface, solid = (f(oinfo, tris, morton=False)[0] for f in (oracle.surface, oracle.solid))
    d = torch.from_numpy(tris.reshape(-1)).to(gpu)
    tables = [torch.zeros(surface.size, dtype=torch.int32, device=gpu) for _ in range(4)]
    streams = [torch.cuda.Stream() for _ in range(3)]
    batch = V.Batch([V.BatchJob(info, d, tables[0]), V.BatchJob(info, d, tables[1], solid=True)])
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()

    def beside():
        for k in range(4):
            batch.launch(stream=streams[k % 2])
        V.release_scratch()

    with torch.cuda.graph(graph, stream=streams[2]):
        V.voxelize_surface(info, d, table=tables[2])
        if other_thread:
            t = threading.Thread(target=beside)
            t.start()
            t.join()
        else:
            beside()
        V.voxelize_solid_table(info, d, table=tables[3])
    for _ in range(3):
        for k in (2, 3):
            tables[k].fill_(-1)
        graph.replay()
        torch.cuda.synchronize()
        for table, exp in zip(tables, (surface, solid, surface, solid)):
            assert (table.cpu().numpy().view(np.uint32) == exp).all()
    batch.close()
