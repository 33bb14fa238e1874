"""VOX_FLAG_NO_SCRATCH: the same tables without a scratch table, and surfaces
without any allocation.  Bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# 96, 128: words and 16-byte groups; 100: ragged; 640: flagged
@pytest.mark.parametrize("grid,morton", [(96, False), (100, False), (128, False), (640, False), (128, True)])
@pytest.mark.parametrize("solid", [False, True])
def test_no_scratch(oracle, gpu, grid, morton, solid):
    import cuda_voxelizer_amd as V
    import torch
    from cuda_voxelizer_amd import _capi, meshgen
    n = 5000
    tris = np.ascontiguousarray(meshgen.triangle_soup(n, seed=grid, mu=-2.5, sigma=0.6), np.float32)
    info = V.voxinfo_for_mesh(tris.reshape(-1, 3), grid, n)
    exp = (oracle.solid if solid else oracle.surface)(oracle.info_from_bytes(info.as_bytes()), tris, morton=morton)[0]
    d = torch.from_numpy(tris.reshape(-1)).to(gpu)
    table = torch.empty(exp.size, dtype=torch.int32, device=gpu)
    call = V.voxelize_solid_table if solid else V.voxelize_surface
    for k in range(2):
        V.release_scratch()
        torch.cuda.synchronize()
        before = torch.cuda.mem_get_info()[0]  # the second time around the runtime has what it loads at first use
        for accumulate in (False, True):
            table.fill_(0x35 if accumulate else -1)
            call(info, d, morton=morton, table=table, accumulate=accumulate, tune=_capi.VOX_FLAG_NO_SCRATCH)
            torch.cuda.synchronize()
            want = exp if not accumulate else (exp ^ np.uint32(0x35) if solid else exp | np.uint32(0x35))
            assert (table.cpu().numpy().view(np.uint32) == want).all()
    # an allocation takes at least 2 MB of the device's; run records are one of 1 MB
    assert before - torch.cuda.mem_get_info()[0] <= (2 << 20 if solid else 0)
    if not solid and not morton:
        batch = V.Batch([V.BatchJob(info, d, table, tune=_capi.VOX_FLAG_NO_SCRATCH)])
        table.fill_(-1)
        torch.cuda.synchronize()
        batch.launch()
        torch.cuda.synchronize()
        assert (table.cpu().numpy().view(np.uint32) == exp).all()
        batch.close()
