"""COO -> CSR by row buckets against the LSD sort (the asynchronous call), bit for
bit: sizes around a bucket's and a tile's edges, and shapes that leave the buckets."""
import ctypes

import numpy as np
import pytest
import torch

from plamatrix_amd import capi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    capi.lib()
    return torch.device("cuda:0")


def triplets(rows, cols, count, kind, dtype, seed):
    rng = np.random.default_rng(seed)
    r = rng.integers(0, rows, count)
    c = rng.integers(0, cols, count)
    if kind == "stencil":  # near the diagonal, most keys repeated
        c = np.clip(r * cols // rows + rng.integers(-2, 3, count), 0, cols - 1)
    elif kind == "arrow":  # half of the triplets in one row: its bucket overflows
        r[rng.random(count) < 0.5] = rows // 3
    elif kind == "one":  # one entry
        r[:], c[:] = rows - 1, cols - 1
    elif kind == "sorted":
        order = np.lexsort((c, r))
        r, c = r[order], c[order]
    v = rng.standard_normal(count).astype(dtype)
    return r, c, v


CASES = [
    (1, 1, 1, "uniform"), (1, 1, 5000, "uniform"), (3, 2, 64, "uniform"), (40, 7, 65, "one"),
    (8192, 8192, 1025, "uniform"), (8193, 8192, 3000, "uniform"), (500, 500, 8192, "stencil"), (600, 600, 4608, "stencil"), (600, 600, 4609, "uniform"),
    (5000, 5000, 8193, "stencil"), (2025, 2025, 10900, "stencil"), (5000, 900, 40000, "sorted"),
    (70000, 70000, 262145, "stencil"), (300, 300, 300000, "uniform"), (100000, 100000, 50000, "uniform"),
    (3, 1 << 29, 9000, "uniform"), (3, 1 << 33, 9000, "uniform"), (20000, 20000, 100000, "arrow"),
    (30000, 30000, 60000, "one"), (5000000, 50, 300000, "uniform"), (190000, 190000, 1100000, "stencil"),
]


@pytest.mark.parametrize("index", range(len(CASES)))
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_buckets_are_the_lsd_sort(dev, index, dtype):
    rows, cols, count, kind = CASES[index]
    r, c, v = triplets(rows, cols, count, kind, dtype, index)
    r, c, v = (torch.from_numpy(t).to(dev) for t in (r, c, v))
    ws = capi.Workspace()
    for _ in range(2):  # the second conversion meets the first one's tables
        a = capi.coo_to_csr(rows, cols, r, c, v, ws)
    out = capi.DeviceCSR(rows, cols, torch.empty_like(a.row_offsets), torch.empty_like(a.col_indices),
                         torch.empty_like(a.values))
    capi.coo_to_csr_async(rows, cols, r, c, v, out, ws)
    torch.cuda.synchronize()
    ws.check_status()
    assert torch.equal(a.row_offsets, out.row_offsets)
    assert torch.equal(a.col_indices, out.col_indices)
    assert a.values.cpu().numpy().tobytes() == out.values.cpu().numpy().tobytes()


@pytest.mark.parametrize("count", [500, 20000])
def test_errors_name_the_first_offset(dev, count):
    r, c, v = triplets(900, 900, count, "stencil", np.float64, 3)
    bad = r.copy()
    bad[[count - 1, 77]] = 900, -1
    ws = capi.Workspace()
    up = lambda *t: [torch.from_numpy(x).to(dev) for x in t]
    with pytest.raises(Exception, match="out of range at source offset 77"):
        capi.coo_to_csr(900, 900, *up(bad, c, v), ws)
    w = v.copy()
    w[[count - 1, 91]] = np.inf, np.nan
    with pytest.raises(Exception, match="non-finite value at source offset 91"):
        capi.coo_to_csr(900, 900, *up(r, c, w), ws)
    # a sum that overflows is met by the fold
    r[:2], c[:2], v[:2] = 5, 5, 1.7e308
    with pytest.raises(Exception, match="non-finite value at source offset 1"):
        capi.coo_to_csr(900, 900, *up(r, c, v), ws)
    assert capi.coo_to_csr(900, 900, *up(r, c, np.ones(count)), ws).values.sum().item() == count


@pytest.mark.parametrize("kind", ["stencil", "arrow"])
@pytest.mark.parametrize("capture", [False, True])
def test_finish_without_reading_the_nnz(dev, kind, capture):
    """A caller that knows the nnz may finish right away, also into a graph."""
    rows, count = 20000, 100000
    r, c, v = triplets(rows, rows, count, kind, np.float64, 8)
    r, c, v = (torch.from_numpy(t).to(dev) for t in (r, c, v))
    want = capi.coo_to_csr(rows, rows, r, c, v, capi.Workspace())
    ws = capi.Workspace()
    got = [torch.zeros_like(t) for t in (want.row_offsets, want.col_indices, want.values)]
    i64, p = ctypes.c_int64, lambda t: ctypes.c_void_p(t.data_ptr())
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        stream = capi.current_stream()
        capi.check(capi.lib().pm_coo_to_csr_prepare(i64(rows), i64(rows), i64(count), p(r), p(c), p(v),
                                                    ctypes.c_int32(capi.dtype_code(v)),
                                                    ctypes.c_int32(capi.PM_COO_CHECK_FINITE), ws.handle, stream))
        finish = lambda: capi.check(capi.lib().pm_coo_to_csr_finish(
            p(got[0]), p(got[1]), p(got[2]), i64(want.nnz), ws.handle, stream))
        if not capture:
            finish()
    side.synchronize()
    if capture:
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            stream = capi.current_stream()
            finish()
        for _ in range(3):
            for t in got:
                t.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(got[0], want.row_offsets) and torch.equal(got[1], want.col_indices)
            assert torch.equal(got[2], want.values)
    else:
        assert torch.equal(got[0], want.row_offsets) and torch.equal(got[1], want.col_indices)
        assert torch.equal(got[2], want.values)


def distinct(rows, count, kind, seed):
    """Triplets of distinct places: as many of any kind have the same nnz.  "even":
    buckets alike; "uneven": one of several times the mean; "over": one that outgrows
    its workgroup."""
    rng = np.random.default_rng(seed)
    heavy = {"even": 0, "uneven": 3000, "over": 20000}[kind]
    low = rng.permutation(128 * rows)[:heavy]
    rest = 128 * rows + rng.permutation((rows - 128) * 64)[:count - heavy] * (rows // 64)
    key = np.concatenate([low, rest])[rng.permutation(count)]
    return key // rows, key % rows, rng.standard_normal(count)


@pytest.mark.parametrize("read_nnz", [False, True])
def test_replayed_finish_meets_new_triplets(dev, read_nnz):
    """A captured finish folds whatever was prepared before its replay."""
    rows, count = 20000, 60000
    sets = {kind: [torch.from_numpy(t).to(dev) for t in distinct(rows, count, kind, seed)]
            for seed, kind in enumerate(("even", "uneven", "over"))}
    want = {kind: capi.coo_to_csr(rows, rows, *t, capi.Workspace()) for kind, t in sets.items()}
    ws = capi.Workspace()
    r, c, v = (t.clone() for t in sets["even"])
    ro = torch.zeros(rows + 1, dtype=torch.int64, device=dev)
    ci, vals = torch.zeros_like(c), torch.zeros_like(v)
    i64, p = ctypes.c_int64, lambda t: ctypes.c_void_p(t.data_ptr())

    def prepare(kind):
        for to, t in zip((r, c, v), sets[kind]):
            to.copy_(t)
        capi.check(capi.lib().pm_coo_to_csr_prepare(i64(rows), i64(rows), i64(count), p(r), p(c), p(v),
                                                    ctypes.c_int32(capi.dtype_code(v)), ctypes.c_int32(0), ws.handle,
                                                    capi.current_stream()))
        if read_nnz:
            nnz = i64()
            capi.check(capi.lib().pm_coo_to_csr_nnz(ws.handle, ctypes.byref(nnz)))
            assert nnz.value == count

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        prepare("even")
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        capi.check(capi.lib().pm_coo_to_csr_finish(p(ro), p(ci), p(vals), i64(count), ws.handle, capi.current_stream()))
    with torch.cuda.stream(side):
        for k, kind in enumerate(("even", "uneven", "over", "even")):
            if k > 0:
                prepare(kind)
            for t in (ro, ci, vals):
                t.zero_()
            graph.replay()
            side.synchronize()
            ws.check_status()
            assert torch.equal(ro, want[kind].row_offsets) and torch.equal(ci, want[kind].col_indices), kind
            assert torch.equal(vals, want[kind].values), kind


@pytest.mark.parametrize("kind", ["stencil", "arrow"])
def test_finish_does_not_wait(dev, kind):
    """Without a read of the nnz, prepare and finish are stream-ordered: both return
    while the stream is still busy with what came before them."""
    rows, count = 20000, 100000
    r, c, v = (torch.from_numpy(t).to(dev) for t in triplets(rows, rows, count, kind, np.float64, 8))
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    i64, p = ctypes.c_int64, lambda t: ctypes.c_void_p(t.data_ptr())
    with torch.cuda.stream(side):
        ws = capi.Workspace()
        want = capi.coo_to_csr(rows, rows, r, c, v, ws)  # the storage is in place
        got = [torch.zeros_like(t) for t in (want.row_offsets, want.col_indices, want.values)]
        side.synchronize()
        for _ in range(2):  # by buckets first, then by the sort
            for t in got:
                t.zero_()
            torch.cuda._sleep(100_000_000)
            capi.check(capi.lib().pm_coo_to_csr_prepare(i64(rows), i64(rows), i64(count), p(r), p(c), p(v),
                                                        ctypes.c_int32(capi.dtype_code(v)), ctypes.c_int32(0), ws.handle,
                                                        capi.current_stream()))
            capi.check(capi.lib().pm_coo_to_csr_finish(p(got[0]), p(got[1]), p(got[2]), i64(want.nnz), ws.handle,
                                                       capi.current_stream()))
            assert not side.query()
            side.synchronize()
            ws.check_status()
            assert torch.equal(got[0], want.row_offsets) and torch.equal(got[1], want.col_indices)
            assert torch.equal(got[2], want.values)


def test_buckets_leave_a_captured_conversion_alone(dev):
    """A captured asynchronous conversion keeps its storage when the workspace then
    converts by buckets, with more tables than the slack of that storage."""
    rows, count = 5_000_000, 1000
    r, c, v = (torch.from_numpy(t).to(dev) for t in triplets(rows, 50, count, "uniform", np.float64, 4))
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        want = capi.coo_to_csr(rows, 50, r, c, v, capi.Workspace())
        out = capi.DeviceCSR(rows, 50, torch.empty_like(want.row_offsets), torch.empty_like(want.col_indices),
                             torch.empty_like(want.values))
        ws = capi.Workspace()
        capi.coo_to_csr_async(rows, 50, r, c, v, out, ws)
        side.synchronize()
        ws.check_status()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        capi.coo_to_csr_async(rows, 50, r, c, v, out, ws)
    with torch.cuda.stream(side):
        graph.replay()
        side.synchronize()
        ws.check_status()
        for _ in range(3):
            capi.coo_to_csr(rows, 50, r, c, v, ws)
            for t in (out.row_offsets, out.col_indices, out.values):
                t.zero_()
            graph.replay()
            side.synchronize()
            assert torch.equal(out.row_offsets, want.row_offsets) and torch.equal(out.values, want.values)
            assert torch.equal(out.col_indices, want.col_indices)
