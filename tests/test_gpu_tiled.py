"""The tiled 3D operators alone, called below the C ABI (marked ``gpu``).  The
reference is a matrix-free product in torch at 64 bits."""
import ctypes as C

import numpy as np
import pytest

from tests.test_gpu_parity import say
from topoptlab_amd import elements

# local nodes of an H8 element: offsets (dx, dy, dz) (elements/trilinear_hexahedron.py)
LOC = [(1 if k & 3 in (1, 2) else 0, 1 if k & 3 in (0, 1) else 0, k >> 2) for k in range(8)]


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
