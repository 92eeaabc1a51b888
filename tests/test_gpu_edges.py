"""Device kernels at the sizes where a tile, a block or a dispatch rule ends
(marked ``gpu``), against the CPU oracle."""
import numpy as np
import pytest

from oracle import fem, mg
from tests.conftest import rel
from tests.test_gpu_parity import _problem, say

pytestmark = pytest.mark.gpu


# coarsest matrices of 12, 32, 60, 64, 66, 96, 130 and 266 DOFs: less than one
# pivot block, one, less than one 64x64 tile, one, two pivot blocks in the
# last tile, an odd number of pivot blocks, and several tiles
@pytest.mark.parametrize("dims,ndpn", [((4, 2, None), 2), ((14, 6, None), 1), ((10, 8, None), 2),
                                       ((14, 14, None), 1), ((20, 4, None), 2),
                                       ((22, 14, None), 1), ((24, 8, None), 2),
                                       ((36, 12, None), 2)])
def test_coarsest_inverse_sizes(gpu, dims, ndpn):
    """Two-grid V-cycle: the first PCG iterate is the oracle's, whose coarsest
    solve is a sparse direct one (rounding times the condition, as in the
    V-cycle parity test)."""
    import torch
    from topoptlab_amd.fem import StiffnessOperator
    say("coarsest inverse", dims, ndpn)
    KE, edof, ndof, fixed, free, x = _problem(dims, ndpn)
    K = fem.apply_bc(fem.assemble_K(KE, edof, fem.simp(x), ndof), free).tocsr()
    b = np.random.default_rng(3).standard_normal(len(free))
    h = mg.Hierarchy(K, *dims, ndpn, fixed, 2)
    op = StiffnessOperator(*dims, KE=KE, fixed=fixed, device=gpu)
    op.set_density(x)
    op.setup_mg(nlevels=2, precision="fp64")
    ref, _, _ = mg.pcg(K, b, h.vcycle, maxiter=1)
    got, _ = op.solve(op.full(torch.as_tensor(b, device=gpu)), maxiter=1, raise_on_fail=False)
    assert rel(got[op._free_t].cpu().numpy(), ref) < 1e-8
    op.close()


# the tiled 3D operators: tiles produce 15x15 nodes and walk node planes in z;
# grids of 1, 15, 16, 17 and 31 nodes per tile direction, one and many planes,
# a partial last tile, more (column, plane) units than workgroups
TILED = [(14, 14, 3), (15, 15, 2), (16, 14, 1), (30, 15, 5), (31, 30, 4), (29, 44, 9), (8, 46, 33),
         (61, 7, 70), (90, 75, 40)]


@pytest.mark.parametrize("dims", TILED)
@pytest.mark.parametrize("ndpn", [3, 1])
def test_tiled_operator(gpu, dims, ndpn):
    """K u on the tiles against the assembled matrix (FP64 1e-13, FP32 inputs
    and sums 1e-5: 24 terms per element, 8 elements, 6e-8 each)."""
    import torch
    from topoptlab_amd.fem import StiffnessOperator
    say("tiled operator", dims, ndpn)
    KE, edof, ndof, fixed, free, x = _problem(dims, ndpn)
    K = fem.apply_bc(fem.assemble_K(KE, edof, fem.simp(x), ndof), free).tocsr()
    u = np.random.default_rng(1).standard_normal(len(free))
    op = StiffnessOperator(*dims, KE=KE, fixed=fixed, device=gpu)
    op.set_density(x)
    y = K @ u
    uf = op.full(torch.as_tensor(u, device=gpu))
    assert rel(op.matvec_full(uf)[op._free_t].cpu().numpy(), y) < 1e-13
    assert rel(op.matvec_full(uf, "fp32")[op._free_t].cpu().numpy(), y) < 1e-5
    # the product inside PCG carries the search-direction update and the dot
    # product: three diagonal-preconditioned iterates
    d = K.diagonal()
    ref, _, _ = mg.pcg(K, y, lambda r: r / d, rtol=0.0, maxiter=3)
    got, _ = op.solve(op.full(torch.as_tensor(y, device=gpu)), rtol=0.0, maxiter=3,
                      preconditioner="jacobi", raise_on_fail=False)
    assert rel(got[op._free_t].cpu().numpy(), ref) < 1e-11
    op.close()


@pytest.mark.parametrize("dims,nlevels", [((28, 28, 4), 3), ((32, 28, 8), 3), ((60, 32, 4), 3),
                                          ((64, 60, 8), 3), ((16, 8, 24), 4)])
@pytest.mark.parametrize("ndpn", [3, 1])
def test_level1_from_densities(gpu, dims, nlevels, ndpn):
    """Level-1 residual and smoothing sweep applied from the child densities:
    the first PCG iterate of the FP64 cycle equals the oracle's, whose level-1
    matrix is P^T K P (densities over nine decades)."""
    import torch
    from topoptlab_amd.fem import StiffnessOperator
    say("level 1 from densities", dims, nlevels, ndpn)
    KE, edof, ndof, fixed, free, _ = _problem(dims, ndpn)
    x = 10.0 ** np.random.default_rng(2).uniform(-3, 0, edof.shape[0])
    K = fem.apply_bc(fem.assemble_K(KE, edof, fem.simp(x), ndof), free).tocsr()
    b = np.random.default_rng(3).standard_normal(len(free))
    h = mg.Hierarchy(K, *dims, ndpn, fixed, nlevels)
    op = StiffnessOperator(*dims, KE=KE, fixed=fixed, device=gpu)
    op.set_density(x)
    for prec, tol in (("fp64", 1e-8), ("fp32", 2e-3)):
        op.setup_mg(nlevels=nlevels, precision=prec)
        ref, _, _ = mg.pcg(K, b, h.vcycle, maxiter=1)
        got, _ = op.solve(op.full(torch.as_tensor(b, device=gpu)), maxiter=1, raise_on_fail=False)
        assert rel(got[op._free_t].cpu().numpy(), ref) < tol, prec
    op.close()
