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


@pytest.mark.parametrize("dims,ndpn", [((5, 4, 3), 3), ((17, 31, 4), 1)])
def test_tiled_operator_keeps_translation_stiffness(gpu, dims, ndpn):
    """An element matrix whose translations cost 4e-14 of its largest entry is
    still taken as reflection-symmetric (to 1e-13); K times a translation is
    then 8 t per element of a node (rounding of the 8 n terms: below 1e-16 of
    the largest entry, 1 % of it)."""
    import torch
    from topoptlab_amd.fem import StiffnessOperator
    KE, edof, ndof, _, _, x = _problem(dims, ndpn)
    t = 5e-15 * np.abs(KE).max()
    op = StiffnessOperator(*dims, KE=KE + 8 * t * np.eye(len(KE)), fixed=[], device=gpu)
    op.set_density(x)
    want = np.zeros(ndof)
    np.add.at(want, edof.ravel(), np.repeat(8 * t * fem.simp(x), edof.shape[1]))
    got = op.matvec_full(torch.ones(ndof, dtype=torch.float64, device=gpu)).cpu().numpy()
    assert np.abs(got - want).max() < 0.03 * want.max()
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


# small 3D levels (up to 16,384 nodes): the correction added inside the first
# sweep; workgroups of 16 nodes over node lines of 2 to 33 nodes, node counts
# that 16 does not divide, one of 9,801
@pytest.mark.parametrize("dims,ndpn,nlevels,gamma,nu", [
    ((16, 8, 24), 3, 4, 2, 2), ((8, 128, 8), 3, 4, 1, 1), ((48, 24, 24), 1, 4, 2, 1),
    ((40, 8, 16), 1, 4, 1, 2), ((128, 128, 32), 1, 4, 1, 1)])
def test_small_stencil_levels(gpu, dims, ndpn, nlevels, gamma, nu):
    """First PCG iterate of the FP64 and FP32 cycles against the oracle's
    (rounding times the condition, as in the V-cycle parity test); with an
    element matrix of no symmetry pattern level 1 is a stencil too."""
    import torch
    from topoptlab_amd.fem import StiffnessOperator
    say("small stencil levels", dims, ndpn, nlevels, gamma, nu)
    KE, edof, ndof, fixed, free, x = _problem(dims, ndpn)
    b = np.random.default_rng(3).standard_normal(len(free))
    s = np.random.default_rng(4).uniform(0.9, 1.1, KE.shape[0])
    for ke in (KE, s[:, None] * KE * s):
        K = fem.apply_bc(fem.assemble_K(ke, edof, fem.simp(x), ndof), free).tocsr()
        h = mg.Hierarchy(K, *dims, ndpn, fixed, nlevels, nu1=nu, nu2=nu)
        ref, _, _ = mg.pcg(K, b, lambda r: h.vcycle(r, 0, gamma, 1), maxiter=1)
        op = StiffnessOperator(*dims, KE=ke, fixed=fixed, device=gpu)
        op.set_density(x)
        for prec, tol in (("fp64", 1e-8), ("fp32", 2e-3)):
            op.setup_mg(nlevels=nlevels, precision=prec, gamma=gamma, gamma_from=1, nu1=nu, nu2=nu)
            got, _ = op.solve(op.full(torch.as_tensor(b, device=gpu)), maxiter=1,
                              raise_on_fail=False)
            assert rel(got[op._free_t].cpu().numpy(), ref) < tol, prec
        op.close()


# convolution layers: result channels and nodes in tiles of 16, source channels
# in 1, 2, 4, 8 or 16 groups of 4; one channel, partial and several tiles, one
# node, more node tiles than workgroups
@pytest.mark.parametrize("stride,shape,cin,cout", [(1, (1, 1, 1), 1, 1), (1, (3, 5, 7), 4, 17),
                                                   (2, (3, 5, 7), 5, 16), (1, (2, 3, 17), 9, 33),
                                                   (2, (9, 5, 5), 17, 5), (1, (1, 4, 16), 33, 64),
                                                   (1, (29, 31, 33), 3, 6)])
def test_conv_tiles(gpu, stride, shape, cin, cout):
    """Forward, data gradient (accumulated) and weight gradient against the
    oracle: fp32 sums of up to 64 x 27 products, 1e-5."""
    import ctypes as C
    import torch
    from oracle import nn
    from topoptlab_amd._lib import check, lib
    say("conv tiles", stride, shape, cin, cout)
    rng = np.random.default_rng(cin + cout)
    a = rng.standard_normal((cin,) + shape).astype(np.float32)
    w = (rng.standard_normal((cout, cin, 27)) * 0.2).astype(np.float16)
    b = rng.standard_normal(cout).astype(np.float32)
    y_ref = nn.conv3d(a.astype(np.float64), w.astype(np.float64), b.astype(np.float64), stride, False)
    gy = rng.standard_normal(y_ref.shape).astype(np.float32)
    ga_ref, gw_ref, gb_ref = nn.conv3d_backward(a.astype(np.float64), w.astype(np.float64),
                                                gy.astype(np.float64), stride, None)
    t = lambda v: torch.as_tensor(np.ascontiguousarray(v), device=gpu)
    p = lambda v: C.c_void_p(v.data_ptr())
    s = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    da, dw, db, dgy = t(a), t(w), t(b), t(gy)
    y = torch.empty(y_ref.shape, dtype=torch.float32, device=gpu)
    check(lib().tl_nn_conv3d(cin, cout, *shape, stride, 0, p(da), p(dw), p(db), p(y), s))
    assert rel(y.cpu().numpy(), y_ref) < 1e-5
    ga = torch.ones((cin,) + shape, dtype=torch.float32, device=gpu)
    check(lib().tl_nn_conv3d_bwd_data(cin, cout, *shape, stride, p(dgy), p(dw), p(ga), 1, s))
    assert rel(ga.cpu().numpy() - 1.0, ga_ref) < 1e-5
    gw = torch.empty((cout, cin, 27), dtype=torch.float32, device=gpu)
    gb = torch.empty(cout, dtype=torch.float32, device=gpu)
    check(lib().tl_nn_conv3d_bwd_weight(cin, cout, *shape, stride, p(da), p(dgy), p(gw), p(gb), s))
    assert rel(gw.cpu().numpy(), gw_ref) < 1e-5 and rel(gb.cpu().numpy(), gb_ref) < 1e-5


# the data gradient's waves share a node tile below 512 tiles (768 with more than
# 16 source channels): 497 and 525 tiles of 5 channels, 525 and 792 of 20; one
# source channel forward (first) and in the gradient from 4,096 tiles (65,536
# nodes) on, 9 result channels in groups of 8
@pytest.mark.parametrize("stride,shape,cin,cout", [(1, (19, 19, 22), 3, 5), (1, (20, 20, 21), 3, 5),
                                                   (1, (20, 20, 21), 3, 20), (1, (22, 24, 24), 3, 20),
                                                   (1, (37, 41, 45), 1, 9), (1, (37, 41, 45), 9, 1),
                                                   (2, (37, 41, 45), 2, 1)])
def test_conv_split_rules(gpu, stride, shape, cin, cout):
    """The same against the same bounds on both sides of the rules."""
    test_conv_tiles(gpu, stride, shape, cin, cout)


@pytest.mark.parametrize("stride,shape,cin,cout", [(1, (3, 4, 18), 5, 20), (2, (5, 5, 9), 9, 33)])
def test_conv_skips_taps_without_source(gpu, stride, shape, cin, cout):
    """Infinite and NaN weights (overflowed fp16) reach the nodes whose tap has
    a source node and no others, forward and in the data gradient: the values
    of a loop that skips the other taps, finite ones to the 1e-5 above."""
    import ctypes as C
    import torch
    from oracle import nn
    from topoptlab_amd._lib import check, lib
    say("conv special weights", stride, shape, cin, cout)
    rng = np.random.default_rng(cin)
    a = rng.standard_normal((cin,) + shape).astype(np.float32)
    w = (rng.standard_normal((cout, cin, 27)) * 0.2).astype(np.float16)
    b = np.zeros(cout, np.float32)
    w[1, 2, 0], w[2, 0, 26], w[18, 4, 3], w[0, 1, 13] = np.inf, -np.inf, np.nan, np.inf
    oshape = nn.out_shape(shape, stride)
    gy = rng.standard_normal((cout,) + oshape).astype(np.float32)
    y_ref, ga_ref = np.zeros((cout,) + oshape), np.zeros(a.shape)
    with np.errstate(invalid="ignore"):
        for t, off in enumerate(nn.OFFS):
            # outputs o whose source stride o + off lies in the grid
            o = [np.array([i for i in range(m) if 0 <= stride * i + d < n], dtype=int)
                 for m, n, d in zip(oshape, shape, off)]
            to = (slice(None),) + np.ix_(*o)
            ti = (slice(None),) + np.ix_(*[stride * i + d for i, d in zip(o, off)])
            wt = w[:, :, t].astype(np.float64)
            for co in range(cout):
                for ci in range(cin):
                    y_ref[co][to[1:]] += wt[co, ci] * a[ci][ti[1:]]
                    ga_ref[ci][ti[1:]] += wt[co, ci] * gy[co][to[1:]]
    t = lambda v: torch.as_tensor(np.ascontiguousarray(v), device=gpu)
    p = lambda v: C.c_void_p(v.data_ptr())
    s = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    da, dw, db, dgy = t(a), t(w), t(b), t(gy)
    y, ga = torch.empty(y_ref.shape, device=gpu), torch.empty(a.shape, device=gpu)
    check(lib().tl_nn_conv3d(cin, cout, *shape, stride, 0, p(da), p(dw), p(db), p(y), s))
    check(lib().tl_nn_conv3d_bwd_data(cin, cout, *shape, stride, p(dgy), p(dw), p(ga), 0, s))
    for got, ref in ((y.cpu().numpy(), y_ref), (ga.cpu().numpy(), ga_ref)):
        fin = np.isfinite(ref)
        assert fin.any() and not fin.all()
        assert np.array_equal(np.isnan(got), np.isnan(ref))
        assert np.array_equal(got[np.isinf(ref)], ref[np.isinf(ref)])
        assert np.isfinite(got[fin]).all() and rel(got[fin], ref[fin]) < 1e-5


# one workgroup up to 8,192 elements (256 threads to 2,048, else 1,024), three
# steps per pass beyond; partial rows, blocks and grids
@pytest.mark.parametrize("n", [2, 255, 257, 2048, 2049, 8191, 8192, 8193, 131073])
@pytest.mark.parametrize("l2", [1e9, 1e3, 1.0])  # 40 to 50 steps, 20 to 30, 10
def test_oc_sizes(gpu, n, l2):
    """Design bit for bit the oracle's, element flags included."""
    import torch
    from topoptlab_amd.optimizer import oc_top88
    say("oc sizes", n, l2)
    rng = np.random.default_rng(n)
    x = 0.05 + 0.9 * rng.random(n)
    dc = -10.0 ** rng.uniform(-4, 1, n)
    dv = 0.5 + rng.random(n)
    fl = rng.choice([0, 0, 0, 1, 2], n)
    g = 0.01 * n
    ref, gt = fem.oc_top88(x, 0.3, dc, dv, g, el_flags=fl, l2=l2)
    t = lambda a: torch.as_tensor(a, device=gpu)
    got, ggt = oc_top88(t(x), 0.3, t(dc), t(dv), g, el_flags=t(fl), l2=l2)
    assert np.array_equal(got.cpu().numpy(), ref)
    assert abs(ggt - gt) <= 1e-12 * np.abs(dv * (ref - x)).sum() + 1e-15


@pytest.mark.parametrize("n", [5, 8192, 8193, 40000])
@pytest.mark.parametrize("e,ends", [(676, True), (675, True), (674, False), (668, False)])
def test_oc_step_limit(gpu, n, e, ends):
    """With l1 = 0 and a constraint that is never exceeded, l2 = 2^-e halves to 0
    in 1075 - e steps: 400 are done, one more is refused, whatever the size."""
    import torch
    from topoptlab_amd.optimizer import oc_top88
    say("oc step limit", n, e)
    x = torch.full((n,), 0.5, dtype=torch.float64, device=gpu)
    dv = torch.ones_like(x)
    if ends:
        got, _ = oc_top88(x, 0.3, -dv, dv, -1e9, l2=2.0 ** -e)
        assert torch.equal(got, torch.full_like(x, 0.7))
    else:
        with pytest.raises(ValueError, match="400 steps"):
            oc_top88(x, 0.3, -dv, dv, -1e9, l2=2.0 ** -e)


# one block, partial blocks, more elements than 1,024 blocks hold at once
@pytest.mark.parametrize("it,n", [(0, 2), (5, 255), (0, 257), (5, 131072), (0, 300001)])
def test_mma_sizes(gpu, it, n):
    """MMA step against the oracle, inputs and tolerances of its parity test."""
    from tests.test_gpu_parity import test_mma_update_matches_oracle as check
    check(gpu, it, n)


def test_mma_threads(gpu):
    """Two host threads on streams of their own, designs of different sizes:
    each step's design and asymptotes are the ones of the step done alone."""
    import threading
    import torch
    from topoptlab_amd.optimizer import mma_defaultkws, mma_update
    say("mma threads")
    probs = []
    for n in (3001, 40000):
        rng = np.random.default_rng(n)
        t = lambda a: torch.as_tensor(a, device=gpu)
        probs.append((t(0.05 + 0.9 * rng.random(n)), t(-10.0 ** rng.uniform(-4, 1, n)),
                      torch.full((n,), 1.0 / n, dtype=torch.float64, device=gpu)))

    def step(x, dc, dv):
        kw = mma_defaultkws(x.numel(), 1, device=gpu)
        return [mma_update(x, None, None, dc, 0.01, dv, kw, iter=0), kw["low"], kw["upp"]]

    want = [step(*p) for p in probs]
    torch.cuda.synchronize()
    got, errs = [[], []], []

    def work(i):
        try:
            with torch.cuda.stream(torch.cuda.Stream(device=gpu)):
                for _ in range(8):
                    got[i].append(step(*probs[i]))
                torch.cuda.current_stream().synchronize()
        except Exception as e:  # shown by the assertion below
            errs.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    assert not errs, errs
    for i in range(2):
        assert len(got[i]) == 8
        for res in got[i]:
            assert all(torch.equal(a, b) for a, b in zip(res, want[i]))


# cycles whose first sweep, correction and scalars are formed inside the
# operators: 2D node lines (up to 63 nodes in y) and tiles (from 64 on), one
# node line of many workgroups; tiled 3D operators with 16, 17 and 31 nodes
SEEDED = [((32, 60, None), 2, 3), ((12, 64, None), 2, 3), ((36, 68, None), 1, 3),
          ((260, 8, None), 2, 3), ((16, 16, 8), 3, 3), ((32, 28, 8), 1, 3)]


@pytest.mark.parametrize("dims,ndpn,nlevels", SEEDED)
def test_seeded_cycle_iterates(gpu, dims, ndpn, nlevels):
    """PCG iterates 1 and 3 of the FP64 cycle against the oracle's (bounds of
    the V-cycle parity test: rounding times the condition)."""
    import torch
    from topoptlab_amd.fem import StiffnessOperator
    say("seeded cycle", dims, ndpn)
    KE, edof, ndof, fixed, free, x = _problem(dims, ndpn)
    K = fem.apply_bc(fem.assemble_K(KE, edof, fem.simp(x), ndof), free).tocsr()
    b = np.random.default_rng(3).standard_normal(len(free))
    h = mg.Hierarchy(K, *dims, ndpn, fixed, nlevels)
    op = StiffnessOperator(*dims, KE=KE, fixed=fixed, device=gpu)
    op.set_density(x)
    op.setup_mg(nlevels=nlevels, precision="fp64")
    for k, tol in ((1, 1e-8), (3, 1e-7)):
        ref, _, _ = mg.pcg(K, b, h.vcycle, rtol=1e-10, maxiter=k)
        got, _ = op.solve(op.full(torch.as_tensor(b, device=gpu)), rtol=1e-10, maxiter=k,
                          raise_on_fail=False)
        assert rel(got[op._free_t].cpu().numpy(), ref) < tol, k
    op.close()


# besides, more 2D tiles than the 1,024 partials that a consumer folds itself
# (1,256 and 2,512), and the FP32 cycles
@pytest.mark.parametrize("dims,ndpn,nlevels", SEEDED + [((1248, 240, None), 1, 5),
                                                        ((1248, 480, None), 2, 5)])
def test_solve_ends_alike_within_a_chunk(gpu, dims, ndpn, nlevels):
    """r.r is folded by the next iteration's residual, or at the end of a
    chunk: whatever the chunk length, the solve stops at the same iteration
    with the same bits, also when repeated on one handle."""
    import torch
    from topoptlab_amd.fem import StiffnessOperator
    say("chunk lengths", dims, ndpn)
    KE, edof, ndof, fixed, free, x = _problem(dims, ndpn)
    f = torch.zeros(ndof, dtype=torch.float64, device=gpu)
    f[torch.as_tensor(free, device=gpu)] = torch.as_tensor(
        np.random.default_rng(3).standard_normal(len(free)), device=gpu)
    op = StiffnessOperator(*dims, KE=KE, fixed=fixed, device=gpu)
    op.set_density(x)
    for prec in ("fp64", "fp32"):
        op.setup_mg(nlevels=nlevels, precision=prec)
        want, inf = op.solve(f, rtol=1e-6, check_every=1)
        assert inf["relres_recursive"] < 1e-6
        for every in (3, 64, 1):
            got, i2 = op.solve(f, rtol=1e-6, check_every=every)
            assert i2["iterations"] == inf["iterations"], (prec, every)
            assert torch.equal(got, want), (prec, every)
        # started from the solution: ended before its first iteration
        again, i3 = op.solve(f, u0=want, rtol=1e-2, check_every=8)
        assert i3["iterations"] == 0 and torch.equal(again, want)
    op.close()


def _no_pattern(KE):
    s = np.random.default_rng(4).uniform(0.9, 1.1, len(KE))
    return s[:, None] * KE * s


# node lines: 1,090 of them, more than a consumer folds partials of; with the
# unit-cell matrix and with one that matches no pattern
@pytest.mark.parametrize("dims,ndpn", [((16400, 16, None), 1), ((16400, 16, None), 2),
                                       ((833, 320, None), 2), ((40, 7, None), 2)])
@pytest.mark.parametrize("pattern", [True, False])
def test_node_lines(gpu, dims, ndpn, pattern):
    """K u (FP64 1e-13, FP32 1e-5) and three diagonal-preconditioned PCG iterates
    (1e-11), whose product carries the search-direction update and the dot
    product, against the assembled matrix."""
    import torch
    from topoptlab_amd.fem import StiffnessOperator
    say("node lines", dims, ndpn, pattern)
    KE, edof, ndof, fixed, free, x = _problem(dims, ndpn)
    KE = KE if pattern else _no_pattern(KE)
    K = fem.apply_bc(fem.assemble_K(KE, edof, fem.simp(x), ndof), free).tocsr()
    u = np.random.default_rng(1).standard_normal(len(free))
    op = StiffnessOperator(*dims, KE=KE, fixed=fixed, device=gpu)
    op.set_density(x)
    y = K @ u
    uf = op.full(torch.as_tensor(u, device=gpu))
    assert rel(op.matvec_full(uf)[op._free_t].cpu().numpy(), y) < 1e-13
    assert rel(op.matvec_full(uf, "fp32")[op._free_t].cpu().numpy(), y) < 1e-5
    d = K.diagonal()
    ref, _, _ = mg.pcg(K, y, lambda r: r / d, rtol=0.0, maxiter=3)
    got, _ = op.solve(op.full(torch.as_tensor(y, device=gpu)), rtol=0.0, maxiter=3,
                      preconditioner="jacobi", raise_on_fail=False)
    assert rel(got[op._free_t].cpu().numpy(), ref) < 1e-11
    op.close()


# cycles on node lines with a matrix of no pattern: 1,045 lines, more than fold
# r.r themselves; up to 320 nodes in y the first sweep is formed inside the
# operators, beyond it is stored
@pytest.mark.parametrize("dims,ndpn,nlevels", [((832, 320, None), 1, 6), ((40, 316, None), 2, 3),
                                               ((40, 324, None), 2, 3), ((40, 324, None), 1, 3)])
def test_node_line_cycles(gpu, dims, ndpn, nlevels):
    """PCG iterates 1 and 3 of the FP64 cycle against the oracle's (bounds of
    test_seeded_cycle_iterates); a solve stops at the same iteration with the
    same bits whatever the chunk length, and in a lockstep batch."""
    import torch
    from topoptlab_amd.batch import batch_solve
    from topoptlab_amd.fem import StiffnessOperator
    say("node line cycles", dims, ndpn)
    KE, edof, ndof, fixed, free, x = _problem(dims, ndpn)
    KE = _no_pattern(KE)
    K = fem.apply_bc(fem.assemble_K(KE, edof, fem.simp(x), ndof), free).tocsr()
    b = np.random.default_rng(3).standard_normal(len(free))
    h = mg.Hierarchy(K, *dims, ndpn, fixed, nlevels)
    op = StiffnessOperator(*dims, KE=KE, fixed=fixed, device=gpu)
    op.set_density(x)
    f = op.full(torch.as_tensor(b, device=gpu))
    op.setup_mg(nlevels=nlevels, precision="fp64")
    for k, tol in ((1, 1e-8), (3, 1e-7)):
        ref, _, _ = mg.pcg(K, b, h.vcycle, rtol=1e-10, maxiter=k)
        got, _ = op.solve(f, rtol=1e-10, maxiter=k, raise_on_fail=False)
        assert rel(got[op._free_t].cpu().numpy(), ref) < tol, k
    for prec in ("fp64", "fp32"):
        op.setup_mg(nlevels=nlevels, precision=prec)
        want, inf = op.solve(f, rtol=1e-6, check_every=1)
        for every in (3, 64):
            got, i2 = op.solve(f, rtol=1e-6, check_every=every)
            assert i2["iterations"] == inf["iterations"] and torch.equal(got, want), (prec, every)
        got, _ = batch_solve([op], [f], rtol=1e-6)
        assert torch.equal(got[0], want), prec
    op.close()


def test_stored_and_formed_sweeps_in_one_batch(gpu):
    """A lockstep batch of systems whose first sweep is stored (node lines of 325
    nodes) and formed inside (tiles, short lines): each the single solve's bits."""
    import torch
    from topoptlab_amd.batch import batch_solve
    from topoptlab_amd.fem import StiffnessOperator
    say("mixed sweeps")
    ops, fs, want = [], [], []
    for dims, pattern in (((40, 324, None), False), ((64, 72, None), True), ((64, 40, None), False),
                          ((36, 324, None), False)):
        KE, _, ndof, fixed, free, x = _problem(dims, 2)
        op = StiffnessOperator(*dims, KE=KE if pattern else _no_pattern(KE), fixed=fixed, device=gpu)
        op.set_density(x)
        op.setup_mg(nlevels=3, precision="fp32")
        ops.append(op)
        fs.append(op.full(torch.as_tensor(np.random.default_rng(3).standard_normal(len(free)),
                                          device=gpu)))
        want.append(op.solve(fs[-1], rtol=1e-6)[0])
    for graphs in (True, False):
        got, _ = batch_solve(ops, fs, rtol=1e-6, use_graphs=graphs)
        assert all(torch.equal(a, b) for a, b in zip(got, want)), graphs
    for op in ops:
        op.close()


@pytest.mark.parametrize("decades,bound", [(0, 1.8e-16), (9, 2.5e-16)])
def test_tiled_product_error(gpu, decades, bound):
    """FP64 K u on white noise against the caller's matrix in extended precision.
    The product's group values are the means of its entries: 1.4e-16 and 2.1e-16
    in a host model of the kernel's sums, 2.2e-16 and 2.9e-16 with single ones."""
    import torch
    from topoptlab_amd.fem import StiffnessOperator
    say("tiled product error", decades)
    dims = (31, 22, 17)
    KE, edof, ndof, _, _, _ = _problem(dims, 3)
    rng = np.random.default_rng(5)
    x = 10.0 ** (-decades / 3.0 * rng.random(edof.shape[0]))
    u = rng.standard_normal(ndof)
    op = StiffnessOperator(*dims, KE=KE, fixed=[], device=gpu)
    op.set_density(x)
    got = op.matvec_full(torch.as_tensor(u, device=gpu)).cpu().numpy()
    ld = np.longdouble
    s = ld(1e-9) + (ld(1) - ld(1e-9)) * x.astype(ld) ** 3
    f = s[:, None] * np.stack([(u[edof].astype(ld) * k).sum(axis=1) for k in KE.astype(ld)], axis=1)
    ref = np.zeros(ndof, dtype=ld)
    np.add.at(ref, edof.ravel(), f.ravel())
    err = float(np.sqrt(((got - ref) ** 2).sum() / (ref ** 2).sum()))
    print(f"  {err:.2e}", flush=True)
    assert err < bound
    op.close()
