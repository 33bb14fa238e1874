"""Calls of several host threads on one stream share the stream's workspaces: the
tile, slab and region algorithms, surfaces and solids, and the triangle order.
Tables bit for bit; the ordered triangles are a permutation of the input."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _cases(gpu, grids):
    import cuda_voxelizer_amd as V
    import torch
    from cuda_voxelizer_amd import meshgen
    out = []
    for k, grid in enumerate(grids):
        n = 600 + 900 * k
        tris = np.ascontiguousarray(meshgen.triangle_soup(n, seed=70 + k, mu=-2.5, sigma=0.6), np.float32)
        info = V.voxinfo_for_mesh(tris.reshape(-1, 3), grid, n)
        out.append((info, tris, torch.from_numpy(tris.reshape(-1)).to(gpu)))
    return out


def _together(count, work):
    threads = [threading.Thread(target=work, args=(k,)) for k in range(count)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()


@pytest.mark.parametrize("algo", ["tile", "slab", "region"])
@pytest.mark.parametrize("solid", [False, True])
def test_algorithms_on_one_stream(oracle, gpu, algo, solid):
    import cuda_voxelizer_amd as V
    cases = _cases(gpu, (64, 128, 128, 256))
    exp = [(oracle.solid if solid else oracle.surface)(oracle.info_from_bytes(i.as_bytes()), t, morton=False)[0]
           for i, t, _ in cases]
    call = V.voxelize_solid_table if solid else V.voxelize_surface
    bad = []

    def work(k):
        for _ in range(25):
            t = call(cases[k][0], cases[k][2], algo=algo)
            if not (t.cpu().numpy().view(np.uint32) == exp[k]).all():
                bad.append(k)

    _together(len(cases), work)
    assert not bad


def test_triangle_order_on_one_stream(gpu):
    import cuda_voxelizer_amd as V
    cases = _cases(gpu, (64, 128, 256, 512))
    bad = []

    def work(k):
        info, tris, d = cases[k]
        for _ in range(25):
            out, perm = V.sort_triangles(info, d, with_perm=True)
            p = perm.cpu().numpy()
            if not ((np.sort(p) == np.arange(p.size)).all()
                    and (out.cpu().numpy().reshape(tris.shape) == tris[p]).all()):
                bad.append(k)

    _together(len(cases), work)
    assert not bad
