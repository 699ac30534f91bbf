"""The training step's partial-sum reductions (k_reduce_parts, k_loss in
plamatrix_amd/csrc/learned.hip) where their splits can go wrong: fewer 32-row
strips than reduction groups (one strip, one row past a strip), strip counts off
the group size, one probe and all eight.  Loss and gradient against the float64 oracle.

Bounds.  The sums themselves are FP32 over n terms in 16 groups, 1e-6 of the
result.  Beside them an activation that sits on a BF16 rounding boundary may land
one step (2^-8) away from the oracle's; on n rows that moves one row's squared
residual, 1 / n of the loss, by up to 2 * 2^-8, and the gradient by up to 2^-7 of
that row's part, 1 / sqrt(n) of its norm.  Two such rows are allowed.  A partial
that is dropped or counted twice costs at least 1 / 16 of a sum.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from oracle import fsai  # noqa: E402
from plamatrix_amd import capi, generators  # noqa: E402


@pytest.mark.parametrize("dims,probes", [((2, 2, 2), 8), ((4, 4, 2), 1), ((11, 3, 1), 3), ((9, 8, 8), 8), ((7, 11, 13), 5)])
def test_loss_and_gradient_sums(dims, probes):
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    h = generators.diffusion3d_box_csr(*dims, seed=9)
    p = capi.fsai_initial_parameters(1)
    rng = np.random.default_rng(1)
    p[fsai.OFF_WOFF:fsai.OFF_BOFF] = 0.05 * rng.standard_normal(fsai.HID)
    p[fsai.OFF_WDIAG:fsai.OFF_BDIAG] = 0.05 * rng.standard_normal(fsai.HID)
    p[fsai.OFF_ALPHA] = -0.4
    net = capi.FsaiNet(seed=0)
    net.parameters = p
    graph = capi.FsaiGraph(capi.to_device_csr(h, compact=True))
    loss, grad = capi.fsai_loss_grad(net, graph, probes=probes, seed=13)
    ref_loss, ref = fsai.loss_and_grad(h.row_offsets, h.col_indices, h.values, p, probes, 13)
    assert abs(loss - ref_loss) <= (1e-6 + 2 * 2.0 ** -7 / h.rows) * ref_loss
    assert np.linalg.norm(grad - ref) <= (2e-3 + 2 * 2.0 ** -7 / np.sqrt(h.rows)) * np.linalg.norm(ref)
    again = capi.fsai_loss_grad(net, graph, probes=probes, seed=13)
    assert again[0] == loss and np.array_equal(again[1], grad)
