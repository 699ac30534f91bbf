"""Schur assembly and block PCG where the staged kernels meet their edges: primaries
and secondaries with one residual more or less than a stage, a batch or a segment
pair holds, and long-row solves with the direction formed inside the SpMV."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from plamatrix_amd import capi, generators  # noqa: E402
from test_gpu_schur import device_batch, oracle_equations  # noqa: E402


@pytest.fixture(scope="module")
def dev():
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    capi.lib()
    return torch.device("cuda:0")


def counted(counts, ec, seed):
    """Primary p sees counts[p] different secondaries, residuals in random order."""
    rng = np.random.default_rng(seed)
    p = np.repeat(np.arange(len(counts)), counts)
    e = np.concatenate([rng.permutation(ec)[:c] for c in counts])
    order = rng.permutation(len(p))
    n = len(p)
    res = rng.standard_normal((n, 2))
    return generators.LMInstance(len(counts), ec, 6, 3, p[order].astype(np.int64), e[order].astype(np.int64),
                                 rng.standard_normal((n, 12)), rng.standard_normal((n, 6)), res,
                                 generators.huber_weights(res, 1.0), 1.0, 1e-3)


# stages of 64 residuals per primary (8 at a time), 682 products of a primary's rhs,
# 256 residuals of 64 secondaries, 4 back-substituted blocks, segments of 16 terms in pairs
@pytest.mark.parametrize("counts,ec", [([1], 1), ([15, 1, 17], 40), ([63, 64, 65, 7, 8, 129], 130),
                                       ([681, 682, 683, 690], 700), ([1, 1500, 31, 1366], 1500), ([130] * 9, 130)])
def test_stage_edges(dev, oracle, counts, ec):
    inst = counted(counts, ec, len(counts))
    sw, ws = capi.SchurWorkspace(), capi.Workspace()
    pc = len(counts)
    weights = torch.from_numpy(inst.weights).to(dev)
    ne = capi.assemble_normal_equations(sw, pc, ec, 6, 3, **device_batch(inst, dev), weights=weights)
    got, eq = capi.normal_equations_arrays(ne), oracle_equations(oracle, inst, inst.weights)
    ref = eq.export()
    for key in ("primary_diagonal", "eliminated_diagonal", "primary_gradient", "eliminated_gradient", "cross_values"):
        assert np.array_equal(got[key].view(np.uint64), ref[key].view(np.uint64)), key
    dp = torch.zeros(pc * 6, dtype=torch.float64, device=dev)
    de = torch.zeros(ec * 3, dtype=torch.float64, device=dev)
    rep = capi.schur_solve(sw, ne, inst.damping, dp, de, ws, max_iterations=1000, relative_tolerance=1e-12,
                           absolute_tolerance=0.0)
    assert rep.converged
    a, rhs_ptr, _ = capi.schur_system(sw)
    B, cinv, rhs, _ = eq.prologue(inst.damping)
    assert np.array_equal(capi.device_array(rhs_ptr, pc * 6).view(np.uint64), rhs.view(np.uint64))
    # The segments sum in another order than the oracle.  An entry is the damped B
    # plus, per shared secondary, a 3-term product of W C^-1 (itself 3 terms) and W,
    # both sides with the same W and C^-1: each computes it within gamma_n of the sum
    # of the terms' sizes, |B| + sum |W| |C^-1| |W|^T, n = 3 max(counts) + 8 roundings.
    # That sum is far above the value itself where B and the products cancel (a
    # secondary seen once leaves S at the damping's size).
    wide = np.zeros((pc, 6, ec, 3))
    wide[ref["cross_primary"], :, ref["cross_eliminated"], :] = np.abs(ref["cross_values"]).reshape(-1, 6, 3)
    wide = wide.reshape(pc * 6, ec, 3)
    size = np.einsum("aei,eij->aej", wide, np.abs(cinv).reshape(ec, 3, 3)).reshape(pc * 6, -1) @ wide.reshape(pc * 6, -1).T
    gamma = (3 * max(counts) + 8) * 2.0 ** -53
    values, mine = eq.csr_values(inst.damping).values, capi.device_array(a.values, a.nnz)
    assert np.max(np.abs(mine - values)) <= 2 * gamma * 1.01 * (np.max(size) + np.max(np.abs(B)))


def ring(blocks, reach, seed, dtype):
    """Block ring of 6 x 6 blocks, 2 reach + 1 blocks a row, diagonally dominant."""
    rng = np.random.default_rng(seed)
    import scipy.sparse as sp

    n = blocks * 6
    m = sp.lil_matrix((n, n))
    for b in range(blocks):
        for d in range(1, reach + 1):
            c = (b + d) % blocks
            v = rng.standard_normal((6, 6))
            m[b * 6:b * 6 + 6, c * 6:c * 6 + 6] = v
            m[c * 6:c * 6 + 6, b * 6:b * 6 + 6] = v.T
    m = sp.csr_matrix(m)
    m = sp.csr_matrix(m + sp.diags(1.0 + np.asarray(abs(m).sum(axis=1)).ravel() * (1.0 + rng.random(n))))
    m.sort_indices()
    return generators.CSRHost(n, n, m.indptr.astype(np.int64), m.indices.astype(np.int64), m.data.astype(dtype))


@pytest.mark.parametrize("blocks,reach,dtype,refresh", [(8, 3, np.float64, 0), (61, 9, np.float64, 6),
                                                        (60, 29, np.float32, 0), (333, 7, np.float64, 0)])
@pytest.mark.parametrize("compact", [False, True])
def test_direction_in_the_long_row_spmv_is_bitwise(dev, monkeypatch, blocks, reach, dtype, refresh, compact):
    h = ring(blocks, reach, blocks, dtype)
    assert h.values.size >= 32 * h.rows
    a = capi.to_device_csr(h, compact=compact)
    rng = np.random.default_rng(2)
    b = torch.from_numpy(rng.standard_normal(h.rows).astype(dtype)).to(dev)
    import scipy.sparse as sp

    m = sp.csr_matrix((h.values.astype(np.float64), h.col_indices, h.row_offsets), shape=(h.rows, h.rows))
    inv = np.stack([np.linalg.inv(m[k:k + 6, k:k + 6].toarray()) for k in range(0, h.rows, 6)])
    inv = torch.from_numpy(inv.astype(dtype).reshape(-1)).to(dev)
    out = []
    for fuse in ("0", None):
        if fuse is None:
            monkeypatch.delenv("PLAMATRIX_AMD_FUSE_DIRECTION", raising=False)
        else:
            monkeypatch.setenv("PLAMATRIX_AMD_FUSE_DIRECTION", fuse)
        x = torch.zeros_like(b)
        rep = capi.block_pcg(a, b, x, inv, 6, capi.Workspace(), capi.policy(refresh_interval=refresh),
                             relative_tolerance=1e-10 if dtype == np.float64 else 1e-5, max_iterations=500)
        assert rep.converged
        out.append((rep.iterations, rep.final_residual, x.cpu().numpy().tobytes()))
    assert out[0] == out[1]
