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
