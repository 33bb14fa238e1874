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
