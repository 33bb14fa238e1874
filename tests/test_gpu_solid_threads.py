"""Solid calls of several host threads on one stream share its scratch table and
its spilled runs: linear rows of 16-byte groups, of words and of no whole words,
Morton bricks, markers in blocked and in linear order, growing grids.  The soups
are not closed, so runs leave their rows.  Bit for bit."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FORMS = {"linear": [(128, False), (128, False), (128, False), (128, False)],
         "morton": [(128, True), (128, True), (64, True), (64, True)],
         "ragged": [(100, False), (100, False), (75, False), (123, False)],
         "mixed": [(128, False), (96, False), (100, False), (128, True)],
         "growing": [(64, True), (128, False), (200, False), (256, False)]}


@pytest.mark.parametrize("form", list(FORMS))
@pytest.mark.parametrize("side", [False, True])
def test_threads_on_one_stream(oracle, gpu, form, side):
    import cuda_voxelizer_amd as V
    import torch
    from cuda_voxelizer_amd import meshgen
    cases = []
    for k, (grid, morton) in enumerate(FORMS[form]):
        n = 600 + 100 * k
        tris = np.ascontiguousarray(meshgen.triangle_soup(n, seed=20 + k, mu=-2.0, sigma=0.6), np.float32)
        info = V.voxinfo_for_mesh(tris.reshape(-1, 3), grid, n)
        exp = oracle.solid(oracle.info_from_bytes(info.as_bytes()), tris, morton=morton)[0]
        cases.append((info, torch.from_numpy(tris.reshape(-1)).to(gpu), morton, exp))
    torch.cuda.synchronize()
    stream = torch.cuda.Stream() if side else torch.cuda.current_stream()
    bad = []

    def work(k):
        info, d, morton, exp = cases[k]
        with torch.cuda.stream(stream):
            for _ in range(40):
                t = V.voxelize_solid_table(info, d, morton=morton)
                if not (t.cpu().numpy().view(np.uint32) == exp).all():
                    bad.append(k)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(cases))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
