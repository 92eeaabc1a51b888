"""Tables of the reflection-symmetric H8 forms (csrc/sym_pattern.hpp): the
element matrix and the coarse Galerkin matrix rebuilt from the table entries
and a few group values equal the dense ones, and the transforms written as the
kernels write them (csrc/tl_sym.hip) give K u."""
import re
from pathlib import Path

import numpy as np
import pytest

from oracle import mg
from topoptlab_amd import elements
from topoptlab_amd.csrc import gen_ke_pattern as gen

HDR = (Path(gen.__file__).parent / "sym_pattern.hpp").read_text()
CASES = [("elast", 3, lambda: elements.lk_linear_elast_3d(E=2.5, nu=0.37)),
         ("poisson", 1, lambda: elements.lk_poisson_3d(k=0.7))]


def table(name):
    body = re.search(r"%s\[\d+\] = \{(.*?)\};" % name, HDR, re.S).group(1)
    return np.array([int(v) for v in body.replace("\n", " ").split(",") if v.strip()])


def rebuilt(tag, name, B):
    tab, first = table(f"kTab{tag}_{name}"), table(f"kFirst{tag}_{name}")
    kv = B.ravel()[first]
    return (np.sign(tab) * kv[np.maximum(np.abs(tab) - 1, 0)]).reshape(B.shape), kv


def hadamard(n):
    h = np.array([[gen.sign(m, gen.corner(k)) for k in range(8)] for m in range(8)])
    return np.kron(h, np.eye(n))


@pytest.mark.parametrize("name,n,KE", CASES)
def test_element_matrix(name, n, KE):
    K = np.asarray(KE())
    B, _ = gen.sym_matrices(K)
    R, _ = rebuilt("Sym", name, B)
    H = hadamard(n)
    assert np.abs(H.T @ R @ H - K).max() < 1e-14 * np.abs(K).max() * 8
    if n == 3:
        assert np.count_nonzero(R) == 45
    # couples only within a parity class (the loops visit nothing else)
    cls = np.array([m ^ (1 << c) if n == 3 else m for m in range(8) for c in range(n)])
    assert np.all((R == 0) | (cls[:, None] == cls[None, :]))


@pytest.mark.parametrize("name,n,KE", CASES)
def test_coarse_galerkin_matrix(name, n, KE):
    K = np.asarray(KE())
    _, Bm = gen.sym_matrices(K)
    R, _ = rebuilt("SymC", name, Bm)
    H = hadamard(n)
    cls = np.array([m ^ (1 << c) if n == 3 else m for m in range(8) for c in range(n)])
    rng = np.random.default_rng(1)
    s = 10.0 ** rng.uniform(-9, 0, 8)  # child scales, child (cz 2 + cx) 2 + cy
    t = np.array([sum(gen.sign(m, (c >> 1 & 1, c & 1, c >> 2)) * s[c] for c in range(8))
                  for m in range(8)])
    A = sum(t[m] * H.T @ R[m] @ H for m in range(8))
    for m in range(8):
        assert np.all((R[m] == 0) | ((cls[:, None] ^ cls[None, :]) == m))
    # the oracle's prolongator on one coarse element (2x2x2 fine elements)
    P = mg.prolongator(2, 2, 2, n).toarray()
    edof = elements.create_edofMat_3d(2, 2, 2, n)[0]
    Kf = np.zeros((27 * n, 27 * n))
    for e in range(8):
        ez, ex, ey = e // 4, e // 2 % 2, e % 2
        Kf[np.ix_(edof[e], edof[e])] += s[(ez * 2 + ex) * 2 + ey] * K
    ec = elements.create_edofMat_3d(1, 1, 1, n)[0][0]
    ref = (P.T @ Kf @ P)[np.ix_(ec, ec)]
    assert np.abs(A - ref).max() < 1e-13 * np.abs(ref).max()
