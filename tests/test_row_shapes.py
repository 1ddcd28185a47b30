"""Packed projection and per-Gaussian row kernels at the edges of their launch
shapes: workgroups of 256 and of 4,096 rows (ProjectionEWA3DGSPacked.cu:39-290
compacts the same rows), one thread per Gaussian below four features and one
per feature from there (rendering.py:170-213, 782)."""

import pytest
import torch

from tests._util import DEV

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,cams", [(1, 1), (255, 1), (257, 2), (131072, 1), (131073, 1),
                                    (43691, 3), (43690, 3)])
def test_packed_rows_equal_the_dense_projection(n, cams):
    """Every packed row is the dense projection's row of the same camera and
    Gaussian, bit for bit and in (camera, Gaussian) order."""
    from gsplat_amd import fully_fused_projection
    g = torch.Generator().manual_seed(n + cams)
    means = (torch.rand(n, 3, generator=g) * 4 - 2).to(DEV)
    quats = torch.randn(n, 4, generator=g).to(DEV)
    scales = (torch.randn(n, 3, generator=g) * 0.5 - 3).exp().to(DEV)
    opac = torch.rand(n, generator=g).to(DEV)
    vm = torch.eye(4).repeat(cams, 1, 1)
    vm[:, 2, 3] = 3.0 + torch.arange(cams)
    K = torch.tensor([[200.0, 0, 100], [0, 200, 80], [0, 0, 1]]).repeat(cams, 1, 1)
    args = (means, None, quats, scales, vm.to(DEV), K.to(DEV), 200, 160)
    radii, m2, dep, con, _ = fully_fused_projection(*args, opacities=opac)
    b, c, i, indptr, r_p, m2_p, dep_p, con_p, _ = fully_fused_projection(
        *args, packed=True, opacities=opac)
    want = torch.nonzero((radii > 0).all(-1))
    assert torch.equal(torch.stack([c, i], -1), want) and int(b.abs().sum()) == 0
    counts = torch.bincount(want[:, 0], minlength=cams).cumsum(0)
    assert indptr.tolist() == [0] + counts.tolist()
    for packed, dense in ((r_p, radii), (m2_p, m2), (dep_p, dep), (con_p, con)):
        assert torch.equal(packed, dense[want[:, 0], want[:, 1]])


@pytest.mark.parametrize("F", [1, 2, 3, 4, 5, 32, 33])
@pytest.mark.parametrize("B,C,N", [(1, 1, 257), (2, 3, 100)])
def test_row_gather_and_scatter(F, B, C, N):
    from gsplat_amd.cuda import _ops
    g = torch.Generator().manual_seed(F)
    keep = torch.rand(B, C, N, generator=g) < 0.6
    row_of = torch.where(keep, keep.reshape(-1).cumsum(0).reshape(B, C, N) - 1, -1)
    row_of = row_of.to(torch.int32).to(DEV)
    nnz = int(keep.sum())
    src = torch.randn(B, N, F, generator=g).to(DEV)
    out = _ops.rows_gather(src, row_of, C, nnz)
    at = torch.nonzero(keep).to(DEV)
    assert torch.equal(out, src[at[:, 0], at[:, 2]])
    v = torch.randn(nnz, F, generator=g).to(DEV)
    want = torch.zeros(B, N, F, device=DEV)
    for c in range(C):  # in camera order, as the kernels sum
        m = row_of[:, c] >= 0
        want[m] += v[row_of[:, c][m].long()]
    assert torch.equal(_ops.rows_scatter_sum(v, row_of, B, C, N), want)
