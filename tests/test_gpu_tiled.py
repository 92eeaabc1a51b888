"""The tiled 3D operators alone, called below the C ABI (marked ``gpu``):
FP32 kernels at FP32 rounding, the level-1 operator, and the split of the
tile columns that the sizes of test_gpu_edges.py do not reach.  The reference
is a matrix-free product in torch at 64 bits."""
import ctypes as C

import numpy as np
import pytest

from tests.test_gpu_parity import say
from topoptlab_amd import elements

TN = 15  # nodes produced per tile side
# local nodes of an H8 element: offsets (dx, dy, dz) (elements/trilinear_hexahedron.py)
LOC = [(1 if k & 3 in (1, 2) else 0, 1 if k & 3 in (0, 1) else 0, k >> 2) for k in range(8)]
EVEN = (480, 480, 16)


def even_split(dims, slots):
    """The launcher's rule: true where the (column, plane) units go evenly over
    the workgroups, false where every column has the same z ranges."""
    nx, ny, nz = (n + 1 for n in dims)
    ncol = -(-nx // TN) * -(-ny // TN)
    nseg = min(slots // ncol, nz)
    return nseg < 1 or -(-nz // nseg) + 1 > -(-ncol * nz // slots) + 2


def test_even_split_sizes():
    """The fine grid of EVEN is split evenly whatever the kernel's occupancy (1
    to 8 workgroups on each of 256 CUs), its level 1 for 1 or 2."""
    assert all(even_split(EVEN, 256 * k) for k in range(1, 9))
    assert all(even_split([n // 2 for n in EVEN], 256 * k) for k in (1, 2))
    assert not even_split((90, 75, 40), 512)


def _k(KE, s, u):
    """Sum of the element products; s [nz][nx][ny] scales, u node values
    [nz+1][nx+1][ny+1][ndpn]."""
    import torch
    ez, ex, ey = s.shape
    ndpn = u.shape[-1]
    at = lambda a, o: a[o[2]:o[2] + ez, o[0]:o[0] + ex, o[1]:o[1] + ey]
    f = torch.cat([at(u, o) for o in LOC], dim=-1).reshape(-1, 8 * ndpn) @ KE.T
    f = f.reshape(ez, ex, ey, 8, ndpn) * s[..., None, None]
    y = torch.zeros_like(u)
    for k, o in enumerate(LOC):
        at(y, o).add_(f[..., k, :])
    return y


def _up(c):
    """Trilinear prolongation of node values."""
    import torch
    for ax in range(3):
        n = c.shape[ax]
        mid = 0.5 * (c.narrow(ax, 0, n - 1) + c.narrow(ax, 1, n - 1))
        shape = list(c.shape)
        shape[ax] = 2 * n - 1
        f = torch.empty(shape, dtype=c.dtype, device=c.device)
        sl = lambda a, b: tuple([slice(None)] * ax + [slice(a, None, b)])
        f[sl(0, 2)], f[sl(1, 2)] = c, mid
        c = f
    return c


def _down(f):
    """Its transpose."""
    for ax in range(3):
        n = (f.shape[ax] - 1) // 2
        sl = lambda a, b: tuple([slice(None)] * ax + [slice(a, None, b)])
        even, odd = f[sl(0, 2)].clone(), f[sl(1, 2)]
        even.narrow(ax, 0, n).add_(odd, alpha=0.5)
        even.narrow(ax, 1, n).add_(odd, alpha=0.5)
        f = even
    return f


class _Case:
    def __init__(self, gpu, dims, ndpn, decades):
        import torch
        from topoptlab_amd.fem import StiffnessOperator
        self.dims, self.ndpn, self.gpu = dims, ndpn, gpu
        nelx, nely, nelz = dims
        self.shape = (nelz + 1, nelx + 1, nely + 1, ndpn)
        KE = elements.lk_linear_elast_3d() if ndpn == 3 else elements.lk_poisson_3d()
        ids = np.arange(np.prod(self.shape)).reshape(self.shape)
        self.op = StiffnessOperator(*dims, KE=KE, fixed=ids[:, 0].ravel(), device=gpu)
        gen = torch.Generator(device=gpu).manual_seed(7)
        self.rand = lambda *s: torch.randn(*s, generator=gen, dtype=torch.float64, device=gpu)
        # scale eps + (1 - eps) x^3 over that many decades
        x = 10.0 ** (-decades / 3.0 * torch.rand(self.op.nel, generator=gen, dtype=torch.float64,
                                                 device=gpu))
        self.op.set_density(x)
        self.s = (1e-9 + (1.0 - 1e-9) * x ** 3).reshape(nelz, nelx, nely)
        self.KE = torch.as_tensor(np.asarray(KE), dtype=torch.float64, device=gpu)

    def fix(self, v):
        """Node values with the clamped x = 0 face at 0."""
        v[:, 0] = 0.0
        return v

    def field(self, shape, kind):
        """White noise, or a nearly constant field; exact in FP32."""
        import torch
        v = self.rand(*shape)
        if kind == "smooth":
            z = torch.linspace(0, 1, shape[0], dtype=torch.float64, device=self.gpu)
            v = 1.0 + 0.1 * torch.sin(z)[:, None, None, None] + 0.0 * v
        return self.fix(v.float().double())

    def product(self, v):
        return self.fix(_k(self.KE, self.s, v))

    def level1(self, v):
        return self.fix(_down(_k(self.KE, self.s, _up(v))))

    def level1_shape(self):
        return tuple(n // 2 + 1 for n in (self.dims[2], self.dims[0], self.dims[1])) + (self.ndpn,)

    def coarse_apply(self, f64, mode, v, xc, b):
        """Level-1 kernel: b - A1 v (mode 0), or the sweep v' + omega D^-1 (b - A1
        v') with v' = v + P xc on the free DOFs (mode 1)."""
        import torch
        from topoptlab_amd._lib import check, lib
        fn = lib()._ZN2tl16sym_coarse_applyEP10tl_problembiPKvS3_S3_PvPKi
        fn.restype, fn.argtypes = C.c_int, [C.c_void_p, C.c_bool, C.c_int] + [C.c_void_p] * 5
        dt = torch.float64 if f64 else torch.float32
        v, xc, b = (None if t is None else t.to(dt).contiguous() for t in (v, xc, b))
        y = torch.empty_like(v)
        self.op._sync_stream()
        check(fn(self.op._h, f64, mode, v.data_ptr(), None if xc is None else xc.data_ptr(),
                 b.data_ptr(), y.data_ptr(), None), "level 1")
        return y.double()

    def coarse_residual(self, f64, v, b):
        return self.coarse_apply(f64, 0, v, None, b)

    def fine_residual(self, f64, v, b):
        """b - K v by the V-cycle's kernel (b in FP64); v None: from the first
        sweep omega D^-1 b, formed inside."""
        import torch
        from topoptlab_amd._lib import check, lib
        fn = lib()._ZN2tl13fine_apply_exEP10tl_problemPKvPviiS3_bS3_dS3_S4_PKdPdiPKib
        p = C.c_void_p
        fn.restype = C.c_int
        fn.argtypes = [p, p, p, C.c_int, C.c_int, p, C.c_bool, p, C.c_double, p, p, p, p, C.c_int, p,
                       C.c_bool]
        dt = torch.float64 if f64 else torch.float32
        y = torch.empty(self.shape, dtype=dt, device=self.gpu)
        v = None if v is None else v.to(dt).contiguous()
        self.op._sync_stream()
        check(fn(self.op._h, None if v is None else v.data_ptr(), y.data_ptr(), 0 if f64 else 1, 2,
                 b.data_ptr(), True, None, 0.0, None, None, None, None, 0, None, False), "residual")
        return y.double()

    def first_sweep(self, b):
        d = self.op.full(self.op.diagonal()).reshape(self.shape)
        return self.fix((0.6 / d * b).nan_to_num(0.0, 0.0, 0.0))


def _rel(a, b):
    return float((a - b).norm() / b.norm())


@pytest.mark.gpu
@pytest.mark.parametrize("dims,nlevels", [((28, 28, 4), 3), ((64, 60, 8), 3), ((16, 8, 24), 4)])
@pytest.mark.parametrize("ndpn", [3, 1])
def test_level1_arithmetic(gpu, dims, nlevels, ndpn):
    """Level-1 residual of the FP32 cycles: FP64 sums rounded once, so no entry
    is further off than 2^-24 of itself (6e-8), on rough and on nearly constant
    fields; FP64: 1e-13 of the terms summed."""
    say("level-1 arithmetic", dims, ndpn)
    c = _Case(gpu, dims, ndpn, 9)
    c.op.setup_mg(nlevels=nlevels, precision="fp32")
    for kind in ("rough", "smooth"):
        v = c.field(c.level1_shape(), kind)
        a = c.level1(v)
        for b in (0.0 * a, a.float().double() + c.field(v.shape, "rough") * a.std()):
            assert _rel(c.coarse_residual(False, v, b), b - a) < 6e-8, kind
    v = c.field(c.level1_shape(), "rough")
    assert _rel(c.coarse_residual(True, v, 0.0 * v), -c.level1(v)) < 1e-13
    c.op.close()


@pytest.mark.gpu
@pytest.mark.parametrize("dims", [(14, 14, 4), (16, 14, 2), (30, 28, 6), (8, 46, 34), (62, 8, 70)])
@pytest.mark.parametrize("ndpn", [3, 1])
def test_fine_residual_fp32(gpu, dims, ndpn):
    """FP32 residual on the tiles, from a stored vector and from the first sweep
    formed inside: 2e-6 of the terms (24 products of 8 elements, 6e-8 each,
    adding up at random)."""
    say("FP32 tiles", dims, ndpn)
    c = _Case(gpu, dims, ndpn, 3)
    c.op.setup_mg(nlevels=2, precision="fp32")
    b = c.fix(c.rand(*c.shape))
    for v in (c.field(c.shape, "rough"), None):
        k = c.product(c.first_sweep(b) if v is None else v)
        err = c.fine_residual(False, v, b) - (b - k)
        assert float(err.norm()) < 2e-6 * float(b.norm() + k.norm())
    c.op.close()


@pytest.mark.gpu
@pytest.mark.parametrize("ndpn", [3, 1])
def test_even_split(gpu, ndpn):
    """A grid whose (column, plane) units go evenly over the workgroups, which
    then walk several tile columns and start some above the first plane:
    products (1e-13), the product inside PCG (1e-11 after two iterates), the
    residual of the first sweep formed inside (1e-13; FP32 2e-6), the level-1
    residual (1e-13; FP32 6e-8) and its sweep with the coarse correction (1e-13
    of the terms)."""
    import torch
    say("even split", ndpn)
    c = _Case(gpu, EVEN, ndpn, 3)
    op = c.op
    v = c.field(c.shape, "rough")
    y = c.product(v)
    got = op.matvec_full(v.reshape(-1)).reshape(c.shape)
    assert _rel(got, y) < 1e-13
    say("even split: pcg", ndpn)
    d = op.full(op.diagonal()).reshape(c.shape)
    inv = c.fix((1.0 / d).nan_to_num(0.0, 0.0, 0.0))
    x, r, p, rho = torch.zeros_like(y), y.clone(), None, None
    for _ in range(2):
        z = inv * r
        new = (r * z).sum()
        p = z if p is None else z + (new / rho) * p
        rho = new
        q = c.product(p)
        a = rho / (p * q).sum()
        x, r = x + a * p, r - a * q
    got, _ = op.solve(y.reshape(-1), rtol=0.0, maxiter=2, preconditioner="jacobi",
                      raise_on_fail=False)
    assert _rel(got.reshape(c.shape), x) < 1e-11
    say("even split: cycles", ndpn)
    op.setup_mg(nlevels=5, precision="fp64")
    w = c.field(c.level1_shape(), "rough")
    a = c.level1(w)
    assert _rel(c.coarse_residual(True, w, 0.0 * w), -a) < 1e-13
    assert _rel(c.coarse_residual(False, w, 0.0 * w), -a) < 6e-8
    for f64, tol in ((True, 1e-13), (False, 2e-6)):
        for u in (v, None):
            k = c.product(c.first_sweep(y) if u is None else u)
            err = c.fine_residual(f64, u, y) - (y - k)
            assert float(err.norm()) < tol * float(y.norm() + k.norm())
    say("even split: corrected sweep", ndpn)
    xc = c.rand(*(n // 4 + 1 for n in (EVEN[2], EVEN[0], EVEN[1])), ndpn)
    zero = 0.0 * w
    omd = c.coarse_apply(True, 1, zero, None, zero + 1.0)  # omega D^-1
    wc = c.fix(w + _up(xc))
    corr = omd * (a - c.level1(wc))
    got = c.coarse_apply(True, 1, w, xc, a)
    assert float((got - c.fix(wc + corr)).norm()) < 1e-13 * float(wc.norm() + corr.norm())
    op.close()
