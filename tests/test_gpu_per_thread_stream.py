"""hipStreamPerThread is one handle for a stream of each thread: calls of several
threads on it run at the same time on the device and share no workspace.  The
defaults and every algorithm with a workspace, and the triangle order."""
import ctypes
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PER_THREAD = 2  # hipStreamPerThread


@pytest.mark.parametrize("what", ["surface", "solid", "solid ragged", "solid morton", "tile", "slab", "region", "sort"])
def test_threads_on_their_own_streams(oracle, gpu, capi, what):
    import cuda_voxelizer_amd as V
    import torch
    from cuda_voxelizer_amd import _capi, meshgen
    solid, morton = what != "surface" and what != "sort", what == "solid morton"
    flags = _capi.ALGO_FLAGS[what] if what in _capi.ALGO_FLAGS else 0
    grid = 100 if what == "solid ragged" else 128
    cases = []
    for k in range(4):
        n = 3000 + 100 * k
        tris = np.ascontiguousarray(meshgen.triangle_soup(n, seed=90 + k, mu=-2.5, sigma=0.6), np.float32)
        info = V.voxinfo_for_mesh(tris.reshape(-1, 3), grid, n)
        oinfo = oracle.info_from_bytes(info.as_bytes())
        exp = (oracle.solid if solid else oracle.surface)(oinfo, tris, morton=morton)[0]
        d = torch.from_numpy(tris.reshape(-1)).to(gpu)
        cases.append((info, tris, d, torch.empty(exp.size, dtype=torch.int32, device=gpu),
                      torch.empty_like(d), torch.empty(n, dtype=torch.int32, device=gpu), exp))
    torch.cuda.synchronize()
    bad = []

    def work(k):
        info, tris, d, table, out, perm, exp = cases[k]
        for _ in range(30):
            if what == "sort":
                _capi.check(capi.vox_sort_triangles(ctypes.byref(info._c), d.data_ptr(), out.data_ptr(),
                                                    perm.data_ptr(), PER_THREAD))
            elif solid:
                _capi.check(capi.vox_solid(ctypes.byref(info._c), d.data_ptr(), table.data_ptr(), int(morton), flags,
                                           None, PER_THREAD))
            else:
                _capi.check(capi.vox_surface(ctypes.byref(info._c), d.data_ptr(), table.data_ptr(), 0, flags,
                                             PER_THREAD))
            torch.cuda.synchronize()
            if what == "sort":
                p = perm.cpu().numpy()
                ok = (np.sort(p) == np.arange(p.size)).all() and (out.cpu().numpy().reshape(tris.shape) == tris[p]).all()
            else:
                ok = (table.cpu().numpy().view(np.uint32) == exp).all()
            if not ok:
                bad.append(k)

    for _ in range(2):  # the second time by new threads
        threads = [threading.Thread(target=work, args=(k,)) for k in range(len(cases))]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    assert not bad
