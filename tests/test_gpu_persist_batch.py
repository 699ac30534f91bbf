"""The persistent batch (plamatrix_amd/csrc/persist_batch.hip): systems of short,
banded rows solved by teams of workgroups, against the per-kernel batch
(PLAMATRIX_AMD_PERSISTENT=0).  The dot products are summed in another order, so
iteration counts may differ by a step or two and the solutions by what the stop
rule leaves: both end at ||r|| <= rel ||b|| of the recursive residual, so their
difference in the A-norm is of that size; with rel = 1e-10 (FP64) and matrices of
condition below 1e4 that is 1e-6 of x, and 1e-5 * 1e3 = 1e-2 with rel = 1e-5
(FP32, condition below 1e3).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from plamatrix_amd import capi, generators  # noqa: E402


@pytest.fixture(scope="module")
def dev():
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    capi.lib()
    return torch.device("cuda:0")


def diag_system(n):
    return generators.CSRHost(n, n, np.arange(n + 1, dtype=np.int64), np.arange(n, dtype=np.int64),
                              np.linspace(1.0, 3.0, n))


def long_rows(n, seed):
    rng = np.random.default_rng(seed)
    m = rng.standard_normal((n, n)) * 0.1
    m = m @ m.T + np.eye(n) * n * 0.05
    return generators.CSRHost(n, n, np.arange(n + 1, dtype=np.int64) * n, np.tile(np.arange(n, dtype=np.int64), n),
                              m.reshape(-1))


def members(kind):
    lap, box = generators.laplacian2d_csr, generators.diffusion3d_box_csr
    if kind == "edges":  # one workgroup and one row beyond, for 1, 2 and 4 rows per lane; tiny systems; long rows
        return [diag_system(1), lap(8, 8), lap(32, 32), lap(25, 41), lap(64, 32), lap(2049, 1), lap(64, 64),
                lap(17, 241), long_rows(60, 1), diag_system(63)]
    if kind == "teams":  # halos narrower and wider than a piece
        return [lap(150, 90), box(25, 24, 23, seed=1), lap(40, 400), box(60, 50, 4, seed=2), lap(3000, 5)]
    if kind == "alone":  # more workgroups than CUs, most of the systems one workgroup each with 1, 2 or 4 rows per lane
        return [lap(150, 140)] * 45 + [lap(64, 64), lap(60, 68), lap(45, 45), lap(32, 32), lap(20, 20), diag_system(5)] * 20
    # more workgroups than CUs at any rows per lane: several launches
    return [lap(150, 140 + i % 7) for i in range(60)] + [box(30, 30, 30, seed=i) for i in range(6)]


def batch(kind, dtype):
    hosts = [generators.CSRHost(h.rows, h.cols, h.row_offsets, h.col_indices, h.values.astype(dtype)) for h in members(kind)]
    h, begin, end = generators.block_diagonal(hosts, dtype=dtype)
    return h, begin, end


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("kind", ["edges", "teams", "launches", "alone"])
def test_teams_match_the_per_kernel_batch(dev, monkeypatch, kind, dtype):
    h, begin, end = batch(kind, dtype)
    rel, bound = (1e-10, 1e-6) if dtype == np.float64 else (1e-5, 1e-2)
    b = torch.zeros(h.rows, dtype=torch.float64)
    for i, (s, e) in enumerate(zip(begin, end)):
        b[s:e] = torch.from_numpy(generators.rhs_normal(e - s, seed=i).astype(np.float64))
    b = b.to(torch.float32 if dtype == np.float32 else torch.float64).to(dev)
    x0 = 0.1 * torch.ones_like(b)
    for compact, jacobi, refresh, most in ((True, True, 50, 3000), (False, False, 0, 3000), (True, True, 10, 7)):
        a = capi.to_device_csr(h, compact=compact)
        out, storage = {}, {}
        for flag in ("0", "1"):
            monkeypatch.setenv("PLAMATRIX_AMD_PERSISTENT", flag)
            ws = capi.Workspace()
            for _ in range(2):  # the second solve meets the first one's exchange words
                x = x0.clone()
                reps = capi.batch_pcg(a, begin, end, b, x, ws, pol=capi.policy(refresh_interval=refresh),
                                      use_jacobi=jacobi, relative_tolerance=rel, max_iterations=most)
                torch.cuda.synchronize()
                got = [(r.converged, r.iterations, r.status) for r in reps]
                if flag == "1" and flag in out and kind != "edges":
                    assert got == out[flag][0] and torch.equal(x, out[flag][1])  # every system in teams: deterministic
                out[flag] = (got, x.clone(), reps)
            storage[flag] = ws.capacity_bytes
        assert storage["1"] > storage["0"]
        for i, (s, e) in enumerate(zip(begin, end)):
            (c0, n0, s0), (c1, n1, s1) = out["0"][0][i], out["1"][0][i]
            assert (c0, s0) == (c1, s1) and abs(n0 - n1) <= max(2, 0.02 * n0), (i, n0, n1)
            xa, xb = out["0"][1][s:e].double(), out["1"][1][s:e].double()
            assert float((xa - xb).norm()) <= bound * float(xa.norm()), i
            r0, r1 = out["0"][2][i], out["1"][2][i]
            assert abs(r0.initial_residual - r1.initial_residual) <= 1e-12 * r0.initial_residual
        gaps = torch.ones(h.rows, dtype=torch.bool)
        for s, e in zip(begin, end):
            gaps[s:e] = False
        assert torch.equal(out["1"][1].cpu()[gaps], x0.cpu()[gaps])  # padding rows are not touched


def test_stops_before_the_launch(dev, monkeypatch):
    # a rejected diagonal, a zero right-hand side and an iteration limit of 0
    # keep their states; the other systems go on
    h, begin, end = batch("teams", np.float64)
    v = h.values.copy()
    row = int(begin[1]) + 5
    k = slice(h.row_offsets[row], h.row_offsets[row + 1])
    v[k][h.col_indices[k] == row] = -2.0
    v[np.arange(h.row_offsets[row], h.row_offsets[row + 1])[h.col_indices[k] == row]] = -2.0
    a = capi.to_device_csr(generators.CSRHost(h.rows, h.cols, h.row_offsets, h.col_indices, v), compact=True)
    b = torch.from_numpy(generators.rhs_normal(h.rows, seed=3).astype(np.float64)).to(dev)
    b[int(begin[2]):int(end[2])] = 0.0
    for most in (0, 2000):
        out = {}
        for flag in ("0", "1"):
            monkeypatch.setenv("PLAMATRIX_AMD_PERSISTENT", flag)
            x = torch.zeros_like(b)
            reps = capi.batch_pcg(a, begin, end, b, x, capi.Workspace(), relative_tolerance=1e-9, max_iterations=most)
            torch.cuda.synchronize()
            out[flag] = [(r.converged, r.status, r.bad_row) for r in reps]
            assert not bool(x[int(begin[1]):int(end[1])].any()) and not bool(x[int(begin[2]):int(end[2])].any())
        assert out["0"] == out["1"]
        assert out["1"][1][1] == 6 and out["1"][1][2] == row and out["1"][2][0]


def test_a_captured_product_keeps_its_storage(dev):
    # a graph holds an SpMM of this workspace, whose packed columns are smaller than
    # what the batch notes of its 512 systems
    small = capi.to_device_csr(diag_system(12), compact=True)
    y, z = (torch.zeros((3, 12), dtype=torch.float64, device=dev) for _ in range(2))
    v = torch.from_numpy(np.random.default_rng(1).standard_normal((3, 12))).to(dev)
    hosts = [generators.laplacian2d_csr(8, 8)] * 512
    h, begin, end = generators.block_diagonal(hosts, dtype=np.float64)
    a = capi.to_device_csr(h, compact=True)
    b = torch.ones(h.rows, dtype=torch.float64, device=dev)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        ws = capi.Workspace()
        capi.spmm(small, v, z, ws)
        side.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        capi.spmm(small, v, y, ws)
    with torch.cuda.stream(side):
        for _ in range(3):
            x = torch.zeros_like(b)
            assert all(r.converged for r in capi.batch_pcg(a, begin, end, b, x, ws, relative_tolerance=1e-8))
            y.zero_()
            graph.replay()
            side.synchronize()
            assert torch.equal(y, z)


@pytest.mark.parametrize("fault", ["refuse=0", "give_up=0", "refuse=1", "give_up=1"])
def test_falls_back_to_the_kernels(dev, monkeypatch, fault):
    # "launches": the teams of launches before the one that is turned down or gives up
    # keep their solutions, the kernels solve the other systems
    h, begin, end = batch("launches", np.float64)
    a = capi.to_device_csr(h, compact=True)
    b = torch.from_numpy(generators.rhs_normal(h.rows, seed=3).astype(np.float64)).to(dev)

    def run(ws):
        x = torch.zeros_like(b)
        reps = capi.batch_pcg(a, begin, end, b, x, ws, relative_tolerance=1e-10, max_iterations=3000)
        torch.cuda.synchronize()
        assert all(r.converged for r in reps)
        return [r.iterations for r in reps], x

    monkeypatch.setenv("PLAMATRIX_AMD_PERSISTENT", "0")
    kernels = run(capi.Workspace())
    monkeypatch.setenv("PLAMATRIX_AMD_PERSISTENT", "1")
    teams = run(capi.Workspace())
    ws = capi.Workspace()
    monkeypatch.setenv("PLAMATRIX_AMD_PERSIST_TEST", fault)
    got = run(ws)
    assert ws.solver_one_launch == -1
    one = [got[0][i] == kernels[0][i] and torch.equal(got[1][s:e], kernels[1][s:e]) for i, (s, e) in enumerate(zip(begin, end))]
    two = [got[0][i] == teams[0][i] and torch.equal(got[1][s:e], teams[1][s:e]) for i, (s, e) in enumerate(zip(begin, end))]
    assert all(p or q for p, q in zip(one, two))
    assert all(one) if fault.endswith("0") else any(p and not q for p, q in zip(one, two)) and any(q and not p for p, q in zip(one, two))
    monkeypatch.delenv("PLAMATRIX_AMD_PERSIST_TEST")
    again = run(ws)  # the pause: the kernels
    assert ws.solver_one_launch == 0 and again[0] == kernels[0] and torch.equal(again[1], kernels[1])


def test_solves_without_the_teams_storage(dev, monkeypatch):
    h, begin, end = batch("teams", np.float64)
    a = capi.to_device_csr(h, compact=True)
    b = torch.from_numpy(generators.rhs_normal(h.rows, seed=3).astype(np.float64)).to(dev)
    out = []
    for name, value in (("PLAMATRIX_AMD_PERSISTENT", "0"), ("PLAMATRIX_AMD_PERSIST_TEST", "storage=0")):
        with monkeypatch.context() as m:
            m.setenv(name, value)
            ws, x = capi.Workspace(), torch.zeros_like(b)
            reps = capi.batch_pcg(a, begin, end, b, x, ws, relative_tolerance=1e-10, max_iterations=3000)
            torch.cuda.synchronize()
            out.append(([(r.converged, r.iterations) for r in reps], x.cpu().numpy().tobytes()))
    assert out[0] == out[1] and ws.solver_one_launch == -1


def test_exchange_tags_start_again(dev, monkeypatch):
    h, begin, end = batch("launches", np.float32)
    a = capi.to_device_csr(h, compact=True)
    b = torch.from_numpy(generators.rhs_normal(h.rows, seed=3)).to(dev)
    ws, out = capi.Workspace(), []
    for test in ("", "tag=4026531830", ""):
        monkeypatch.setenv("PLAMATRIX_AMD_PERSIST_TEST", test)
        x = torch.zeros_like(b)
        reps = capi.batch_pcg(a, begin, end, b, x, ws, relative_tolerance=1e-5, max_iterations=3000)
        torch.cuda.synchronize()
        assert ws.solver_one_launch == 1
        out.append(([(r.converged, r.iterations) for r in reps], x.cpu().numpy().tobytes()))
    assert out[0] == out[1] == out[2]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_systems_past_a_team(dev, monkeypatch, dtype):
    # more rows than 64 workgroups hold (FP32 262,144, FP64 131,072), rows too long or a
    # column of another system in the last chunk of many: the kernels, bit for bit; the
    # systems beside them in teams
    lap = generators.laplacian2d_csr
    hosts = [lap(520, 510), lap(60, 60), lap(410, 330), long_rows(60, 1), lap(257, 256), lap(50, 50)]
    hosts = [generators.CSRHost(h.rows, h.cols, h.row_offsets, h.col_indices, h.values.astype(dtype)) for h in hosts]
    h, begin, end = generators.block_diagonal(hosts, dtype=dtype)
    far = h.row_offsets[int(end[4])] - 1  # the last entry of the fifth system
    h.col_indices[far] = int(begin[5]) + 3
    h.values[far] = 0.0
    a = capi.to_device_csr(h, compact=True)
    b = torch.from_numpy(generators.rhs_normal(h.rows, seed=5).astype(dtype)).to(dev)
    out = {}
    for flag in ("0", "1"):
        monkeypatch.setenv("PLAMATRIX_AMD_PERSISTENT", flag)
        ws, x = capi.Workspace(), torch.zeros_like(b)
        reps = capi.batch_pcg(a, begin, end, b, x, ws, relative_tolerance=1e-30, max_iterations=30)
        torch.cuda.synchronize()
        out[flag] = [(r.iterations, r.final_residual, x[s:e].cpu().numpy()) for r, s, e in zip(reps, begin, end)]
        assert ws.solver_one_launch == int(flag)
    for i, (p, q) in enumerate(zip(out["0"], out["1"])):
        same = p[0] == q[0] and p[1] == q[1] and np.array_equal(p[2], q[2])
        kernels = i in (0, 3, 4) or (i == 2 and dtype == np.float64)
        assert same or not kernels, i
        assert np.linalg.norm(p[2] - q[2]) <= (1e-3 if dtype == np.float32 else 1e-10) * np.linalg.norm(p[2]), i


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_many_tiny_systems_take_the_kernels(dev, monkeypatch, dtype):
    # below 1 KB of a vector and more than four for every CU; the larger ones beside them
    # get a workgroup each
    lap = generators.laplacian2d_csr
    hosts = [lap(6, 5, dtype=dtype)] * 1100 + [lap(32, 31, dtype=dtype), lap(16, 16, dtype=dtype), lap(70, 70, dtype=dtype)]
    h, begin, end = generators.block_diagonal(hosts, dtype=dtype)
    a = capi.to_device_csr(h, compact=True)
    b = torch.from_numpy(generators.rhs_normal(h.rows, seed=5).astype(dtype)).to(dev)
    out = {}
    for flag in ("0", "1"):
        monkeypatch.setenv("PLAMATRIX_AMD_PERSISTENT", flag)
        ws, x = capi.Workspace(), torch.zeros_like(b)
        reps = capi.batch_pcg(a, begin, end, b, x, ws, relative_tolerance=1e-4, max_iterations=400)
        torch.cuda.synchronize()
        assert all(r.converged for r in reps) and ws.solver_one_launch == int(flag)
        out[flag] = [r.iterations for r in reps], x.cpu().numpy()
    assert out["0"][0][:1100] == out["1"][0][:1100]
    assert np.array_equal(out["0"][1][:1100 * 64], out["1"][1][:1100 * 64])
    x0, x1 = (out[f][1][int(begin[1100]):].astype(np.float64) for f in ("0", "1"))
    assert np.linalg.norm(x0 - x1) <= 1e-1 * np.linalg.norm(x0)  # 1e-4 times a condition below 1e3
