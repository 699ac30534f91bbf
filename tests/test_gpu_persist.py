"""The persistent CG / Jacobi-PCG (plamatrix_amd/csrc/persist.hip): one launch per
solve, rows kept in registers.  It sums in the per-kernel iteration's order, so
a solve must be bitwise the one with PLAMATRIX_AMD_PERSISTENT=0: iterations,
residual and solution, at every number of rows per lane, with and without
diagonals that reach past the halos, with a short last piece, with refreshes
and at iteration limits around the launch's first decisions.
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


def matrix(kind, dims, dtype):
    if kind == "diffusion":  # unit diagonal: the unpreconditioned kernels
        return generators.diffusion3d_box_csr(*dims, seed=5, dtype=dtype)
    h = generators.laplacian2d_csr(*dims, dtype=dtype)  # diagonal 4: the Jacobi kernels
    if kind == "varied":  # a diagonal that differs from row to row
        rows = np.repeat(np.arange(h.rows), np.diff(h.row_offsets))
        on = rows == h.col_indices
        h.values[on] += np.random.default_rng(3).random(h.rows).astype(dtype)
    return h


def solve(a, b, monkeypatch, persistent, refresh, rel, most, solver=capi.pcg, x0=None):
    monkeypatch.setenv("PLAMATRIX_AMD_PERSISTENT", persistent)
    ws = capi.Workspace()
    x = torch.zeros_like(b) if x0 is None else x0.clone()
    out = []
    for _ in range(2):  # the second solve meets the first one's exchange words
        y = x.clone()
        rep = solver(a, b, y, ws, capi.policy(refresh_interval=refresh), relative_tolerance=rel, max_iterations=most)
        torch.cuda.synchronize()
        out.append((rep.converged, rep.iterations, rep.initial_residual, rep.final_residual, y.cpu().numpy().tobytes()))
    assert ws.solver_diagonals > 0 and ws.solver_form == 1
    assert out[0] == out[1]
    return out[0], ws.capacity_bytes


CASES = [
    # rows per lane 1: all neighbours in halos; the halo wider than the inner
    # diagonal; outermost diagonals past the halos; a short last piece
    ("laplace", (256, 256), np.float64, 0),
    ("varied", (2100, 33), np.float64, 20),
    ("laplace", (33, 2100), np.float32, 0),
    ("diffusion", (41, 43, 40), np.float32, 50),
    ("diffusion", (41, 43, 40), np.float64, 0),
    # 2 and 4 rows per lane, uneven chunks per wavefront
    ("laplace", (517, 601), np.float64, 0),
    ("varied", (701, 760), np.float32, 50),
    ("diffusion", (71, 70, 67), np.float32, 20),
    ("laplace", (850, 830), np.float64, 50),
    ("diffusion", (97, 89, 91), np.float32, 0),
    # 8 (FP32): x and the inner diagonals in LDS
    ("diffusion", (109, 107, 103), np.float32, 50),
    ("laplace", (1200, 1001), np.float32, 20),
]


@pytest.mark.parametrize("kind,dims,dtype,refresh", CASES)
def test_persistent_solve_is_bitwise(dev, monkeypatch, kind, dims, dtype, refresh):
    a = capi.to_device_csr(matrix(kind, dims, dtype), compact=True)
    b = torch.from_numpy(generators.rhs_normal(a.rows, seed=17).astype(dtype)).to(dev)
    ref, without = solve(a, b, monkeypatch, "0", refresh, 1e-4, 400)
    got, with_ = solve(a, b, monkeypatch, "1", refresh, 1e-4, 400)
    assert with_ > without  # the exchange words were allocated: the persistent kernel ran
    assert got == ref


@pytest.mark.parametrize("most", [0, 1, 2, 3, 50])
def test_iteration_limits(dev, monkeypatch, most):
    a = capi.to_device_csr(matrix("laplace", (300, 290), np.float64), compact=False)
    b = torch.from_numpy(generators.rhs_uniform(a.rows, seed=2)).to(dev)
    x0 = torch.from_numpy(generators.rhs_uniform(a.rows, seed=3)).to(dev)
    for solver in (capi.cg, capi.pcg):
        ref, _ = solve(a, b, monkeypatch, "0", 0, 1e-10, most, solver, x0)
        got, _ = solve(a, b, monkeypatch, "1", 0, 1e-10, most, solver, x0)
        assert got == ref and got[1] == most and not got[0]


def test_stops_at_the_start(dev, monkeypatch):
    # the first decision already converges: x must come back as it was
    a = capi.to_device_csr(matrix("laplace", (300, 290), np.float64), compact=True)
    b = torch.zeros(a.rows, dtype=torch.float64, device=dev)
    got, _ = solve(a, b, monkeypatch, "1", 0, 1e-8, 100)
    assert got[0] and got[1] == 0 and not np.frombuffer(got[4], np.uint8).any()
    # a NaN right-hand side is rejected with x untouched
    b[7] = float("nan")
    monkeypatch.setenv("PLAMATRIX_AMD_PERSISTENT", "1")
    x = torch.full_like(b, 2.0)
    with pytest.raises(capi.PlamatrixError):
        capi.pcg(a, b, x, capi.Workspace(), relative_tolerance=1e-8, max_iterations=100)
    assert bool((x == 2.0).all())


def ragged(n, seed, long_row=0, dtype=np.float64, band=0):
    """SPD matrix with 1 to 14 entries a row and, if asked, one long row; with
    `band` 1 to 9 entries a row, columns within `band` of the row."""
    import scipy.sparse as sp

    rng = np.random.default_rng(seed)
    if band:
        off = np.concatenate([[0], np.sort(rng.integers(1, band, 4))])
        i = np.concatenate([np.nonzero(rng.random(n) < 0.7)[0] for _ in off])
        i = i[(i + off[-1]) < n]
        j = i + off[rng.integers(1, 5, len(i))]
    else:
        k = rng.integers(0, 7, n)
        i = np.repeat(np.arange(n), k)
        j = rng.integers(0, n, len(i))
    if long_row:
        i = np.concatenate([i, np.full(long_row, n // 2)])
        j = np.concatenate([j, rng.permutation(n)[:long_row]])
    m = sp.csr_matrix((rng.standard_normal(len(i)), (i, j)), shape=(n, n))
    m = (m + m.T).tocsr()
    m = (m + sp.diags(np.asarray(abs(m).sum(axis=1)).ravel() * rng.uniform(1.0, 1.4, n) + 0.1)).tocsr()
    m.sort_indices()
    return generators.CSRHost(n, n, m.indptr.astype(np.int64), m.indices.astype(np.int64), m.data.astype(dtype))


SMALL = [
    (ragged(1, 1), 0), (ragged(63, 2), 4), (ragged(257, 3, dtype=np.float32), 0), (ragged(1025, 4), 20),
    (ragged(1100, 5, long_row=900), 6), (ragged(2049, 6, dtype=np.float32), 20), (ragged(4096, 7), 0),
    (ragged(3001, 8, long_row=2500, dtype=np.float32), 0),  # a chunk of more than 2,048 entries: the per-kernel solve
    (generators.laplacian2d_csr(45, 37), 0), (generators.laplacian2d_csr(64, 64, dtype=np.float32), 50),
]


@pytest.mark.parametrize("index", range(len(SMALL)))
@pytest.mark.parametrize("compact", [False, True])
def test_one_workgroup_solve_is_bitwise(dev, monkeypatch, index, compact):
    h, refresh = SMALL[index]
    a = capi.to_device_csr(h, compact=compact)
    b = torch.from_numpy(generators.rhs_normal(h.rows, seed=19).astype(h.values.dtype)).to(dev)
    rel = 1e-10 if h.values.dtype == np.float64 else 1e-5
    for solver in (capi.pcg, capi.cg):
        for most in (0, 1, 3, 4000):
            out = {}
            for flag in ("0", "1"):
                monkeypatch.setenv("PLAMATRIX_AMD_PERSISTENT", flag)
                ws = capi.Workspace()
                x = torch.full_like(b, 0.25)
                rep = solver(a, b, x, ws, capi.policy(refresh_interval=refresh), relative_tolerance=rel,
                             max_iterations=most)
                torch.cuda.synchronize()
                assert ws.solver_form == 2
                out[flag] = (rep.converged, rep.iterations, rep.initial_residual, rep.final_residual,
                             x.cpu().numpy().tobytes())
            assert out["0"] == out["1"], (solver.__name__, most)


def test_one_workgroup_errors(dev, monkeypatch):
    # a rejected diagonal, an indefinite matrix (restart, hand-over, breakdown):
    # the per-kernel solve's errors
    h = generators.laplacian2d_csr(30, 30)
    rows = np.repeat(np.arange(h.rows), np.diff(h.row_offsets))
    b = torch.from_numpy(generators.rhs_normal(h.rows, seed=23).astype(np.float64)).to(dev)
    for row, value in ((100, -1.0), (None, 1.5)):
        v = h.values.copy()
        on = (rows == h.col_indices) & ((rows == row) if row is not None else True)
        v[on] = value
        a = capi.to_device_csr(generators.CSRHost(h.rows, h.cols, h.row_offsets, h.col_indices, v), compact=True)
        out = {}
        for flag in ("0", "1"):
            monkeypatch.setenv("PLAMATRIX_AMD_PERSISTENT", flag)
            x = torch.zeros_like(b)
            try:
                rep = capi.pcg(a, b, x, capi.Workspace(), relative_tolerance=1e-9, max_iterations=500)
                out[flag] = ("ok", rep.iterations, rep.final_residual, x.cpu().numpy().tobytes())
            except capi.PlamatrixError as e:
                out[flag] = (e.kind, str(e))
        assert out["0"] == out["1"]
        if row is not None:
            assert "diagonal" in out["1"][1] and f"row {row}" in out["1"][1]


WIDE = [
    ("stencil", (67, 62), np.float64, 0),      # 4,154 rows, 64-row chunks not a multiple of four
    ("stencil", (23, 21, 19), np.float32, 50),  # 9,177 rows
    ("stencil", (39, 40, 41), np.float64, 0),   # 63,960 rows: the last size below the diagonal layout
    ("banded", 5003, np.float64, 20),
    ("banded", 70001, np.float32, 0),           # more than 64 workgroups, no few diagonals
    ("banded", 262144, np.float64, 6),          # the largest
    ("ragged", 30011, np.float32, 0),           # most entries in other pieces: the per-kernel solve
    ("long", 6007, np.float64, 6),              # a row past the kept entries: likewise
]


@pytest.mark.parametrize("kind,size,dtype,refresh", WIDE)
def test_wide_csr_solve_is_bitwise(dev, monkeypatch, kind, size, dtype, refresh):
    if kind == "stencil":
        h = generators.laplacian2d_csr(*size, dtype=dtype) if len(size) == 2 else \
            generators.diffusion3d_box_csr(*size, seed=3, dtype=dtype)
    else:
        h = ragged(size, 11, 700 if kind == "long" else 0, dtype, 300 if kind == "banded" else 0)
    rel = 1e-10 if dtype == np.float64 else 1e-5
    b = torch.from_numpy(generators.rhs_normal(h.rows, seed=29).astype(dtype)).to(dev)
    for solver, compact, most in ((capi.pcg, True, 600), (capi.cg, False, 600), (capi.pcg, False, 1), (capi.cg, True, 0)):
        a = capi.to_device_csr(h, compact=compact)
        out, storage = {}, {}
        for flag in ("0", "1"):
            monkeypatch.setenv("PLAMATRIX_AMD_PERSISTENT", flag)
            ws = capi.Workspace()
            for _ in range(2):  # the second solve meets the first one's exchange words
                x = torch.full_like(b, 0.5)
                rep = solver(a, b, x, ws, capi.policy(refresh_interval=refresh), relative_tolerance=rel,
                             max_iterations=most)
                torch.cuda.synchronize()
                got = (rep.converged, rep.iterations, rep.initial_residual, rep.final_residual, x.cpu().numpy().tobytes())
                assert out.setdefault(flag, got) == got
            storage[flag] = ws.capacity_bytes
        # the exchange words tell which kernel ran
        assert (storage["1"] > storage["0"]) == (kind in ("stencil", "banded"))
        assert out["0"] == out["1"], (solver.__name__, compact, most)


def test_wide_csr_restart_hands_over(dev, monkeypatch):
    # an indefinite matrix: restart, hand-over at the chunk schedule's
    # iteration, the three-kernel form's breakdown
    h = generators.laplacian2d_csr(90, 80)
    rows = np.repeat(np.arange(h.rows), np.diff(h.row_offsets))
    for shift in (3.9, 3.0, 0.05):
        v = h.values - shift * (rows == h.col_indices)
        a = capi.to_device_csr(generators.CSRHost(h.rows, h.cols, h.row_offsets, h.col_indices, v), compact=True)
        b = torch.from_numpy(generators.rhs_normal(h.rows, seed=31).astype(np.float64)).to(dev)
        out = {}
        for flag in ("0", "1"):
            monkeypatch.setenv("PLAMATRIX_AMD_PERSISTENT", flag)
            x = torch.zeros_like(b)
            try:
                rep = capi.cg(a, b, x, capi.Workspace(), relative_tolerance=1e-9, max_iterations=400)
                out[flag] = ("ok", rep.iterations, rep.final_residual)
            except capi.PlamatrixError as e:
                out[flag] = (e.kind, str(e))
            torch.cuda.synchronize()
            out[flag] += (x.cpu().numpy().tobytes(),)
        assert out["0"] == out["1"], shift


FACTORED = [
    ("diffusion", (41, 43, 40), np.float32, 0),   # far outermost diagonals, a short last piece
    ("diffusion", (11, 13, 480), np.float32, 20),  # every neighbour in the halos
    ("diffusion", (45, 41, 40), np.float64, 50),
    ("diffusion", (71, 70, 67), np.float32, 20),  # two rows per lane
    ("laplace", (260, 300), np.float64, 0),       # five diagonals
    ("laplace", (2500, 31), np.float32, 20),
]


@pytest.mark.parametrize("kind,dims,dtype,refresh", FACTORED)
def test_factored_solve_is_bitwise(dev, monkeypatch, kind, dims, dtype, refresh):
    a = capi.to_device_csr(matrix(kind, dims, dtype), compact=True)
    net = capi.FsaiNet(seed=0)
    p = capi.fsai_initial_parameters(2)
    p[-70:-1] += 0.03 * np.random.default_rng(4).standard_normal(69).astype(np.float32)
    net.parameters = p
    graph = capi.FsaiGraph(a)
    capi.fsai_forward(net, graph)
    b = torch.from_numpy(generators.rhs_normal(a.rows, seed=37).astype(dtype)).to(dev)
    for most in (0, 1, 300):
        out, storage = {}, {}
        for flag in ("0", "1"):
            monkeypatch.setenv("PLAMATRIX_AMD_PERSISTENT", flag)
            ws = capi.Workspace()
            for _ in range(2):  # the second solve meets the first one's exchange words
                x = torch.full_like(b, 0.5)
                rep = capi.pcg_factored(a, b, x, graph, ws, pol=capi.policy(refresh_interval=refresh),
                                        relative_tolerance=1e-4, max_iterations=most)
                torch.cuda.synchronize()
                got = (rep.converged, rep.iterations, rep.initial_residual, rep.final_residual, x.cpu().numpy().tobytes())
                assert out.setdefault(flag, got) == got
            assert ws.solver_form in (4, 5)
            storage[flag] = ws.capacity_bytes
        assert storage["1"] > storage["0"]  # the exchange words: the persistent kernel ran
        assert out["0"] == out["1"], most


def form_solve(form, dev):
    """A solver of a fixed system of that one-launch form: f(ws, most) -> report and x."""
    if form == "csr":
        h = generators.laplacian2d_csr(90, 80)
    elif form == "small":
        h = generators.laplacian2d_csr(45, 37)
    else:
        h = matrix(*{"dia": ("laplace", (300, 290), np.float64), "wide": ("laplace", (1000, 70), np.float64), "factored": ("diffusion", (41, 43, 40), np.float32)}[form])
    a = capi.to_device_csr(h, compact=True)
    b = torch.from_numpy(generators.rhs_normal(a.rows, seed=41).astype(h.values.dtype)).to(dev)
    graph = None
    if form == "factored":
        net = capi.FsaiNet(seed=0)
        net.parameters = capi.fsai_initial_parameters(2)
        graph = capi.FsaiGraph(a)
        capi.fsai_forward(net, graph)

    def run(ws, most=300):
        x = torch.full_like(b, 0.5)
        kw = dict(relative_tolerance=1e-5, max_iterations=most)
        pol = capi.policy(refresh_interval=20)
        rep = capi.pcg(a, b, x, ws, pol, **kw) if graph is None else capi.pcg_factored(a, b, x, graph, ws, pol=pol, **kw)
        torch.cuda.synchronize()
        return rep.converged, rep.iterations, rep.initial_residual, rep.final_residual, x.cpu().numpy().tobytes()

    return run


@pytest.mark.parametrize("form", ["dia", "csr", "factored"])
@pytest.mark.parametrize("fault", ["refuse=0", "give_up=0"])
def test_falls_back_to_the_kernels(dev, monkeypatch, form, fault):
    # a launch that is turned down or gives up leaves x alone and the kernels run the
    # solve; the workspace stays with them for 64 solves, then tries again
    run = form_solve(form, dev)
    monkeypatch.setenv("PLAMATRIX_AMD_PERSISTENT", "0")
    ref = run(capi.Workspace())
    monkeypatch.setenv("PLAMATRIX_AMD_PERSISTENT", "1")
    ws = capi.Workspace()
    assert run(ws) == ref and ws.solver_one_launch == 1
    monkeypatch.setenv("PLAMATRIX_AMD_PERSIST_TEST", fault)
    assert run(ws) == ref and ws.solver_one_launch == -1
    monkeypatch.delenv("PLAMATRIX_AMD_PERSIST_TEST")
    for k in range(63):
        assert run(ws, 300 if k == 0 else 1)[1] >= 1 and ws.solver_one_launch == 0
    assert run(ws) == ref and ws.solver_one_launch == 1


@pytest.mark.parametrize("form", ["dia", "csr", "factored"])
def test_a_launch_too_large_keeps_other_shapes(dev, monkeypatch, form):
    run, other = form_solve(form, dev), form_solve("dia" if form == "csr" else "csr", dev)
    ws, fresh = capi.Workspace(), capi.Workspace()
    ref = run(fresh), other(fresh)
    monkeypatch.setenv("PLAMATRIX_AMD_PERSIST_TEST", "too_large=0")
    assert run(ws) == ref[0] and ws.solver_one_launch == -1
    monkeypatch.delenv("PLAMATRIX_AMD_PERSIST_TEST")
    assert other(ws) == ref[1] and ws.solver_one_launch == 1
    assert run(ws) == ref[0] and ws.solver_one_launch == 1


@pytest.mark.parametrize("form", ["dia", "csr", "factored"])
def test_solves_without_the_exchange_storage(dev, monkeypatch, form):
    run = form_solve(form, dev)
    ref = run(capi.Workspace())
    ws = capi.Workspace()
    monkeypatch.setenv("PLAMATRIX_AMD_PERSIST_TEST", "storage=0")
    assert run(ws) == ref and ws.solver_one_launch == -1
    monkeypatch.delenv("PLAMATRIX_AMD_PERSIST_TEST")
    assert run(ws) == ref and ws.solver_one_launch == 1


def test_large_solves_reserve_six_vectors(dev):
    # past the sizes of the one-launch CSR solve, more diagonals than the layout takes
    n, offsets = 262144 + 64, range(-8, 9)
    i = np.arange(n)
    valid = np.stack([(i + o >= 0) & (i + o < n) for o in offsets], axis=1)
    cols = (i[:, None] + np.array(offsets))[valid]
    values = np.where(cols == np.repeat(i, valid.sum(axis=1)), 17.0, -1.0)
    ro = np.concatenate([[0], np.cumsum(valid.sum(axis=1))])
    a = capi.to_device_csr(generators.CSRHost(n, n, ro, cols, values), compact=True)
    b = torch.ones(n, dtype=torch.float64, device=dev)
    ws = capi.Workspace()
    rep = capi.pcg(a, b, torch.zeros_like(b), ws, relative_tolerance=1e-8, max_iterations=100)
    assert rep.converged and ws.solver_form == 2 and ws.solver_one_launch == 0
    assert ws.capacity_bytes < 6 * 8 * n * 9 / 8 + (2 << 20)  # storage grows by an eighth; partials and state


@pytest.mark.parametrize("form", ["dia", "csr", "small", "factored"])
@pytest.mark.parametrize("test", ["segment=2", "segment=6", "segment=6,tag=4026531830"])
def test_a_solve_of_several_launches(dev, monkeypatch, form, test):
    # a launch continues the one before it: x, vectors, partials, history and tags; the
    # last exchange tags used are just below 0xf0000000, where the words are cleared
    run = form_solve(form, dev)
    monkeypatch.setenv("PLAMATRIX_AMD_PERSISTENT", "0")
    ref = [run(capi.Workspace(), most) for most in (300, 5, 12)]
    monkeypatch.setenv("PLAMATRIX_AMD_PERSISTENT", "1")
    ws = capi.Workspace()
    assert run(ws) == ref[0] and ref[0][1] > 12  # the storage is in place
    monkeypatch.setenv("PLAMATRIX_AMD_PERSIST_TEST", test)
    for most, want in zip((300, 5, 12), ref):
        assert run(ws, most) == want and ws.solver_one_launch == 1


@pytest.mark.parametrize("form", ["dia", "csr", "factored"])
@pytest.mark.parametrize("fault", ["refuse=2", "give_up=2"])
def test_falls_back_after_a_launch(dev, monkeypatch, form, fault):
    # two launches of the solve have ended: x is still the caller's
    run = form_solve(form, dev)
    monkeypatch.setenv("PLAMATRIX_AMD_PERSISTENT", "0")
    ref = run(capi.Workspace())
    monkeypatch.setenv("PLAMATRIX_AMD_PERSISTENT", "1")
    monkeypatch.setenv("PLAMATRIX_AMD_PERSIST_TEST", "segment=4," + fault)
    ws = capi.Workspace()
    assert run(ws) == ref and ws.solver_one_launch == -1


@pytest.mark.parametrize("dims", [(45, 37), (90, 80), (300, 290)])
def test_hand_over_after_several_launches(dev, monkeypatch, dims):
    # an indefinite matrix in the one-workgroup, CSR and diagonal-layout forms
    h = generators.laplacian2d_csr(*dims)
    rows = np.repeat(np.arange(h.rows), np.diff(h.row_offsets))
    for shift in (3.9, 0.05, 0.01):
        v = h.values - shift * (rows == h.col_indices)
        a = capi.to_device_csr(generators.CSRHost(h.rows, h.cols, h.row_offsets, h.col_indices, v), compact=True)
        b = torch.from_numpy(generators.rhs_normal(h.rows, seed=31).astype(np.float64)).to(dev)
        out = []
        for persistent, test in (("0", ""), ("1", "segment=6")):
            monkeypatch.setenv("PLAMATRIX_AMD_PERSISTENT", persistent)
            monkeypatch.setenv("PLAMATRIX_AMD_PERSIST_TEST", test)
            x = torch.zeros_like(b)
            try:
                rep = capi.cg(a, b, x, capi.Workspace(), relative_tolerance=1e-9, max_iterations=400)
                got = ("ok", rep.iterations, rep.final_residual)
            except capi.PlamatrixError as e:
                got = (e.kind, str(e))
            torch.cuda.synchronize()
            out.append(got + (x.cpu().numpy().tobytes(),))
        assert out[0] == out[1], shift


def scattered(n, k, dtype):
    """SPD, 2 k + 1 entries a row on average, their columns anywhere."""
    import scipy.sparse as sp

    rng = np.random.default_rng(n + k)
    i = np.repeat(np.arange(n), k)
    m = sp.csr_matrix((-rng.random(len(i)) - 0.1, (i, (i + 1 + rng.integers(0, n - 1, len(i))) % n)), shape=(n, n))
    m = m + m.T
    m = (m + sp.diags(np.asarray(abs(m).sum(axis=1)).ravel() + 0.1)).tocsr()
    m.sort_indices()
    return generators.CSRHost(n, n, m.indptr.astype(np.int64), m.indices.astype(np.int64), m.data.astype(dtype))


# (matrix, whether one launch takes it): FP64 over 2,048 rows in one workgroup up to four
# entries a row, above that with a row per lane if the columns are near
BESIDE = [
    (scattered(2048, 3, np.float64), 1), (scattered(2049, 3, np.float64), 0), (scattered(2049, 1, np.float64), 1),
    (scattered(4096, 1, np.float64), 1), (scattered(4096, 3, np.float32), 1), (generators.laplacian2d_csr(2049, 1), 1),
    (generators.laplacian2d_csr(46, 45), 1), (generators.laplacian2d_csr(64, 64), 1),
]


@pytest.mark.parametrize("index", range(len(BESIDE)))
def test_one_workgroup_sizes(dev, monkeypatch, index):
    h, one = BESIDE[index]
    b = torch.from_numpy(generators.rhs_normal(h.rows, seed=43).astype(h.values.dtype)).to(dev)
    rel = 1e-10 if h.values.dtype == np.float64 else 1e-5
    for compact, solver in ((True, capi.pcg), (False, capi.cg)):
        a = capi.to_device_csr(h, compact=compact)
        out = {}
        for flag in ("0", "1"):
            monkeypatch.setenv("PLAMATRIX_AMD_PERSISTENT", flag)
            ws, x = capi.Workspace(), torch.full_like(b, 0.25)
            rep = solver(a, b, x, ws, capi.policy(refresh_interval=20), relative_tolerance=rel, max_iterations=500)
            torch.cuda.synchronize()
            assert ws.solver_one_launch == (one if flag == "1" else 0)
            out[flag] = rep.converged, rep.iterations, rep.final_residual, x.cpu().numpy().tobytes()
        assert out["0"] == out["1"]


@pytest.mark.parametrize("forms", [("dia", "csr"), ("dia", "dia"), ("factored", "dia"), ("csr", "factored"), ("small", "dia"), ("dia", "wide")])
def test_two_solves_at_once(dev, forms):
    # two threads, each with its stream and workspace: launches of both may be queued
    # together, and neither waits for the other's workgroups ("dia" and "wide": one kernel
    # with different amounts of LDS)
    import threading

    runs = [form_solve(form, dev) for form in forms]
    refs = [run(capi.Workspace()) for run in runs]
    torch.cuda.synchronize()
    got = [[], []]

    def work(k):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            ws = capi.Workspace()
            for _ in range(6):
                out = runs[k](ws)
                got[k].append((out == refs[k], ws.solver_one_launch))
            stream.synchronize()

    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert got == [[(True, 1)] * 6] * 2
