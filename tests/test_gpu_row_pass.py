"""GPU parity of the row pass behind surfaces' blocked scratch tables at the edges of
its forms: with and without flags (609 up), rows of any number of words and of no
whole words, last strips that are cut short, streamed rows (1152 up), tables at odd
addresses, accumulation, and a scratch table that is left zero for other sizes.
Bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _mesh(oracle, gpu, n, grid, mu):
    import cuda_voxelizer_amd as V
    import torch
    from cuda_voxelizer_amd import meshgen
    tris = np.ascontiguousarray(meshgen.triangle_soup(n, seed=grid, mu=mu, sigma=0.8), np.float32)
    # corners of the grid, so that the first and the last rows hold bits
    tris[0] = [[0.0, 0.0, 0.0], [0.01, 0.0, 0.0], [0.0, 0.01, 0.0]]
    lo, hi = tris.reshape(-1, 3).min(0), tris.reshape(-1, 3).max(0)
    tris[1] = [hi, hi - [0.02, 0, 0], hi - [0, 0.02, 0]]
    tris[2] = [lo, lo + [0.02, 0, 0], lo + [0, 0, 0.02]]
    info = V.voxinfo_for_mesh(tris.reshape(-1, 3), grid, n)
    exp = oracle.surface(oracle.info_from_bytes(info.as_bytes()), tris, morton=False)[0]
    return info, tris, torch.from_numpy(tris.reshape(-1)).to(gpu), torch.from_numpy(exp.view(np.int32)).to(gpu)


# up to 4096 triangles (32768 up to 160) an accumulating call goes to the table directly, with more through the scratch
# table; 128 to 500 and 607, 608: no flags
@pytest.mark.parametrize("grid", [128, 150, 160, 161, 500, 512, 607, 608, 609, 640, 672, 736, 863, 992, 1023, 1024, 1056,
                                  1120, 1152, 1184, 1312, 1920, 2016, 2048])
def test_row_pass(oracle, gpu, grid):
    import cuda_voxelizer_amd as V
    import torch
    info, tris, d, exp = _mesh(oracle, gpu, 300 if grid <= 1024 else 60, grid, -2.5)
    edge = 32768 if grid <= 160 else 4096
    few, _, few_d, few_exp = _mesh(oracle, gpu, edge, grid, -4.5)
    many, _, many_d, many_exp = _mesh(oracle, gpu, edge + 1, grid, -4.5)
    small = V.voxinfo_for_mesh(tris.reshape(-1, 3), 128, info.n_triangles)
    small_exp = oracle.surface(oracle.info_from_bytes(small.as_bytes()), tris, morton=False)[0]
    room = torch.full((exp.numel() + 8,), 0x1234567, dtype=torch.int32, device=gpu)
    for off in (4, 3):
        t = room[off:off + exp.numel()]
        t.fill_(-1)
        V.voxelize_surface(info, d, table=t)
        assert torch.equal(t, exp)
        for i, tri, e in ((info, d, exp), (few, few_d, few_exp), (many, many_d, many_exp)):
            t.fill_(0x35)
            V.voxelize_surface(i, tri, table=t, accumulate=True)
            assert torch.equal(t, e | 0x35)
        assert int(room[off - 1]) == int(room[off + exp.numel()]) == 0x1234567
        t.fill_(0x1234567)
        assert (V.voxelize_surface(small, d).cpu().numpy().view(np.uint32) == small_exp).all()
