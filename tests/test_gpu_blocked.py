"""GPU parity of surfaces whose words go through the blocked scratch table
(chunk.hip): row lengths with and without whole 16-byte groups, flagged and
unflagged tables, tables at odd addresses, accumulation, a scratch table left by
calls of other sizes, other streams and graph capture.  Bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _case(gpu, n, grid, seed, mu=-3.0):
    import cuda_voxelizer_amd as V
    import torch
    from cuda_voxelizer_amd import meshgen
    tris = np.ascontiguousarray(meshgen.triangle_soup(n, seed=seed, mu=mu, sigma=0.8), np.float32)
    info = V.voxinfo_for_mesh(tris.reshape(-1, 3), grid, n)
    return info, tris, torch.from_numpy(tris.reshape(-1)).to(gpu)


def _expected(oracle, info, tris):
    return oracle.surface(oracle.info_from_bytes(info.as_bytes()), tris, morton=False)[0]


def _host(t):
    return t.cpu().numpy().view(np.uint32)


# 64: blocked from 16,384 triangles on; 96, 160: rows of 3 and 5 words; 544: 17
# words, no flags; 640 up: flagged; 1408: its rows are streamed
@pytest.mark.parametrize("n,grid", [(16383, 64), (16384, 64), (3000, 96), (5000, 128), (7, 160), (20001, 256),
                                    (4000, 544), (3000, 640), (900, 1024), (300, 1408)])
def test_blocked_tables(oracle, gpu, n, grid):
    import cuda_voxelizer_amd as V
    import torch
    info, tris, d = _case(gpu, n, grid, n + grid)
    exp = _expected(oracle, info, tris)
    for _ in range(2):  # the second call finds the scratch table as the first left it
        assert (_host(V.voxelize_surface(info, d)) == exp).all()
    rng = np.random.default_rng(grid)
    fill = rng.integers(0, 2**32, size=exp.size, dtype=np.uint32)
    room = torch.empty(exp.size + 4, dtype=torch.int32, device=gpu)
    for off in (0, 1):  # 16-byte groups, and a table at an odd address
        t = room[off:off + exp.size]
        V.voxelize_surface(info, d, table=t)
        assert (_host(t) == exp).all()
        t.copy_(torch.from_numpy(fill.view(np.int32)))
        V.voxelize_surface(info, d, table=t, accumulate=True)
        assert (_host(t) == (exp | fill)).all()


def test_calls_of_different_sizes_share_a_stream(oracle, gpu):
    import cuda_voxelizer_amd as V
    import torch
    cases = [_case(gpu, n, g, n) for n, g in ((4000, 128), (1000, 640), (4000, 96), (2000, 1024), (9000, 256))]
    exp = [_expected(oracle, i, t) for i, t, _ in cases]
    side = torch.cuda.Stream()
    for order in (range(5), reversed(range(5)), range(5)):
        got = [(k, V.voxelize_surface(cases[k][0], cases[k][2]),
                V.voxelize_surface(cases[k][0], cases[k][2], stream=side)) for k in order]
        torch.cuda.synchronize()
        for k, a, b in got:
            assert (_host(a) == exp[k]).all() and (_host(b) == exp[k]).all(), k


def test_threads_on_one_stream(oracle, gpu):
    import threading

    import cuda_voxelizer_amd as V
    import torch
    cases = [_case(gpu, 3000 + 100 * k, 128, 50 + k) for k in range(4)]
    exp = [_expected(oracle, i, t) for i, t, _ in cases]
    bad = []

    def work(k):
        for _ in range(40):
            t = V.voxelize_surface(cases[k][0], cases[k][2])
            if not (_host(t) == exp[k]).all():
                bad.append(k)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def test_capture_does_not_hold_the_scratch(oracle, gpu):
    """A captured call is replayed after calls that replace the scratch table."""
    import cuda_voxelizer_amd as V
    import torch
    info, tris, d = _case(gpu, 4000, 128, 9)
    exp = _expected(oracle, info, tris)
    table = torch.zeros(exp.size, dtype=torch.int32, device=gpu)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        V.voxelize_surface(info, d, table=table)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        V.voxelize_surface(info, d, table=table)
    big, _, bd = _case(gpu, 2000, 512, 10)
    for _ in range(3):
        with torch.cuda.stream(s):
            V.voxelize_surface(big, bd)
        torch.cuda.synchronize()
        table.fill_(-1)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert (_host(table) == exp).all()


@pytest.mark.parametrize("use_graph", [True, False])
def test_blocked_batch(oracle, gpu, use_graph):
    """Blocked jobs beside every other class, launched again and again."""
    import cuda_voxelizer_amd as V
    import torch
    jobs, exp = [], []
    for k, (n, grid) in enumerate([(3000, 96), (20000, 64), (500, 128), (800, 32), (1500, 100), (9, 160), (700, 640),
                                   (5000, 256)]):
        info, tris, d = _case(gpu, n, grid, 100 + k)
        e = _expected(oracle, info, tris)
        acc = k % 3 == 2
        table = torch.zeros(e.size, dtype=torch.int32, device=gpu) if acc else \
            torch.full((e.size,), -1, dtype=torch.int32, device=gpu)
        jobs.append(V.BatchJob(info, d, table, accumulate=acc))
        exp.append(e)
    batch = V.Batch(jobs, use_graph=use_graph)
    for _ in range(3):
        batch.launch()
        torch.cuda.synchronize()
        for k, (j, e) in enumerate(zip(jobs, exp)):
            assert (_host(j.table) == e).all(), k
            if not j.accumulate:
                j.table.fill_(0x55)
    batch.close()


# rows of 33 bits up to 31 words and 7 bits; 41^3 and 333^3 bits end inside a word, and
# 41^2, 333^2 rows inside a workgroup's 32
@pytest.mark.parametrize("grid", [33, 41, 63, 100, 127, 200, 333, 999])
@pytest.mark.parametrize("solid", [False, True])
def test_ragged_rows(oracle, gpu, grid, solid):
    import cuda_voxelizer_amd as V
    import torch
    n = 17000 if grid < 100 else (3001 if grid < 500 else 400)
    if solid:  # below G^2, from where small grids run direct
        n = min(n, grid * grid - 1)
    info, tris, d = _case(gpu, n, grid, grid, mu=-2.5)
    words = V.table_words(grid)
    if solid:
        exp, count, _ = oracle.solid(oracle.info_from_bytes(info.as_bytes()), tris, morton=False)
        call = V.voxelize_solid_table
    else:
        exp, call = _expected(oracle, info, tris), V.voxelize_surface
    rng = np.random.default_rng(grid)
    fill = rng.integers(0, 2**32, size=words, dtype=np.uint32)
    guard = torch.full((words + 2,), 0x1234567, dtype=torch.int32, device=gpu)
    t = guard[1:1 + words]
    for _ in range(2):
        call(info, d, table=t)
        assert (_host(t) == exp).all()
        t.copy_(torch.from_numpy(fill.view(np.int32)))
        call(info, d, table=t, accumulate=True)
        assert (_host(t) == (exp ^ fill if solid else exp | fill)).all()
    assert int(guard[0]) == int(guard[-1]) == 0x1234567
    if solid:
        off = torch.zeros(1, dtype=torch.int64, device=gpu)
        V.voxelize_solid_table(info, d, table=t, offrow=off)
        assert int(off.item()) == count


def test_ragged_solid_capture(oracle, gpu):
    import cuda_voxelizer_amd as V
    import torch
    info, tris, d = _case(gpu, 500, 100, 3, mu=-2.0)
    exp = oracle.solid(oracle.info_from_bytes(info.as_bytes()), tris, morton=False)[0]
    table = torch.zeros(exp.size, dtype=torch.int32, device=gpu)
    V.voxelize_solid_table(info, d, table=table)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        V.voxelize_solid_table(info, d, table=table)
    for _ in range(3):
        table.fill_(-1)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert (_host(table) == exp).all()
