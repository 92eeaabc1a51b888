"""Generate ke_pattern.hpp: sign/group patterns of unit-cell element matrices.

For isotropic materials on unit Q4/H8 cells in the reference node order
(topoptlab/elements/bilinear_quadrilateral.py:209-212,
trilinear_hexahedron.py:252-259) the element matrix has only a handful of
distinct magnitudes, and which entries share a magnitude (and with which
relative sign) does not depend on the material constants.  The pattern is
computed at two Poisson ratios and must agree.  Each table entry is
(+-)(group+1); ``first`` lists the position of each group's first entry, from
which the run time reads the group value out of the caller's KE (and checks
every entry against the pattern before the fast path is used).

For H8 elements the tables of the reflection-symmetric form follow
(sym_pattern.hpp): in the basis of the 8 sign patterns (-1)^(m.corner) per
component, m = mx + 2 my + 4 mz, KE = H^T B H with H the 8-point Hadamard
transform of each component and B = H KE H^T / 64, whose rows and columns
couple only within one parity class (45 instead of 576 nonzeros for
elasticity).  The Galerkin matrix of a coarse element with child scales s_c is
sum_m t_m H^T B_m H with t the Hadamard transform of the child scales and
B_m = H (1/8 sum_c (-1)^(m.c) G_c) H^T / 64 (279 nonzeros together).

Usage: python topoptlab_amd/csrc/gen_ke_pattern.py  (rewrites ke_pattern.hpp
and sym_pattern.hpp)
"""
from __future__ import annotations

import sys
from pathlib import Path

import numpy as np

HERE = Path(__file__).resolve().parent
sys.path.insert(0, str(HERE.parents[1]))

from topoptlab_amd import elements  # noqa: E402


def pattern(K, tol=1e-12):
    a = K.ravel()
    reps, first, out = [], [], []
    for i, v in enumerate(a):
        for g, r in enumerate(reps):
            if abs(abs(v) - abs(r)) <= tol * max(1.0, abs(r)):
                out.append((g + 1) * (1 if np.sign(v) == np.sign(r) else -1))
                break
        else:
            reps.append(v)
            first.append(i)
            out.append(len(reps))
    return out, first


def corner(k):
    """Offset (dx, dy, dz) of local node k of an H8 element."""
    dx, dy = [(0, 1), (1, 1), (1, 0), (0, 0)][k & 3]
    return dx, dy, k >> 2


def sign(m, c):
    return -1.0 if ((m & 1) * c[0] + (m >> 1 & 1) * c[1] + (m >> 2) * c[2]) % 2 else 1.0


def sym_matrices(KE):
    """B of one element, and B_0 .. B_7 of a coarse element."""
    n = KE.shape[0] // 8
    h8 = np.array([[sign(m, corner(k)) for k in range(8)] for m in range(8)])
    H = np.kron(h8, np.eye(n))
    bits = lambda c: (c >> 1 & 1, c & 1, c >> 2)  # child (cz 2 + cx) 2 + cy -> (x, y, z)
    G = []
    for ch in range(8):
        W = np.zeros((8, 8))
        for i in range(8):
            q = [0.5 * (a + b) for a, b in zip(bits(ch), corner(i))]
            for j in range(8):
                W[i, j] = np.prod([v if d else 1.0 - v for v, d in zip(q, corner(j))])
        Q = np.kron(W, np.eye(n))
        G.append(Q.T @ KE @ Q)
    Bm = [H @ (sum(sign(m, bits(c)) * G[c] for c in range(8)) / 8.0) @ H.T / 64.0 for m in range(8)]
    return H @ KE @ H.T / 64.0, np.stack(Bm)


def sym_groups(a1, a2, tol=1e-12):
    """0 or (+-)(group+1) per entry of two equally patterned arrays."""
    reps, first, out = [], [], []
    top = max(abs(a1).max(), abs(a2).max())
    for i, (u, v) in enumerate(zip(a1.ravel(), a2.ravel())):
        if abs(u) <= tol * top and abs(v) <= tol * top:
            out.append(0)
            continue
        for g, (p, q) in enumerate(reps):
            for sg in (1, -1):
                if abs(u - sg * p) <= tol * top and abs(v - sg * q) <= tol * top:
                    out.append(sg * (g + 1))
                    break
            else:
                continue
            break
        else:
            reps.append((u, v))
            first.append(i)
            out.append(len(reps))
    return out, first


def write_sym():
    lines = ["// Generated by gen_ke_pattern.py -- do not edit.",
             "// Reflection-symmetric H8 element matrices: 0 or (+-)(group+1) of the",
             "// entry (row, column) of B (kSym*) and of B_m (kSymC*, m slowest); kFirst*",
             "// holds the position of each group's first entry.",
             "#pragma once", "", "namespace tl {", ""]
    for name, f in (("elast", lambda nu: elements.lk_linear_elast_3d(nu=nu)),
                    ("poisson", lambda nu: elements.lk_poisson_3d(k=1.0 + nu))):
        pair = [sym_matrices(np.asarray(f(nu))) for nu in (0.3, 0.17)]
        for tag, k in (("Sym", 0), ("SymC", 1)):
            pat, first = sym_groups(pair[0][k], pair[1][k])
            nd = pair[0][0].shape[0]
            lines.append(f"constexpr int kGroups{tag}_{name} = {len(first)};")
            lines.append(f"constexpr signed char kTab{tag}_{name}[{len(pat)}] = {{")
            for r in range(len(pat) // nd):
                lines.append("    " + ", ".join(str(v) for v in pat[r * nd:(r + 1) * nd]) + ",")
            lines.append("};")
            lines.append(f"constexpr int kFirst{tag}_{name}[{len(first)}] = {{"
                         + ", ".join(map(str, first)) + "};")
            lines.append("")
    lines.append("}  // namespace tl")
    (HERE / "sym_pattern.hpp").write_text("\n".join(lines) + "\n")
    print("wrote", HERE / "sym_pattern.hpp")


CASES = {
    "h8_elast": lambda nu: elements.lk_linear_elast_3d(nu=nu),
    "q4_elast": lambda nu: elements.lk_linear_elast_2d(nu=nu),
    "q4_poisson": lambda nu: elements.lk_poisson_2d(k=1.0 + nu),
    "h8_poisson": lambda nu: elements.lk_poisson_3d(k=1.0 + nu),
}


def main():
    lines = ["// Generated by gen_ke_pattern.py -- do not edit.",
             "// Entry = (+-)(group+1) of the row-major element matrix; kFirst* holds",
             "// the position of each group's first entry.",
             "#pragma once", "", "namespace tl {", ""]
    for name, f in CASES.items():
        p1, f1 = pattern(f(0.3))
        p2, f2 = pattern(f(0.17))
        if p1 != p2 or f1 != f2:
            raise SystemExit(f"pattern of {name} depends on the material constants")
        n = int(round(len(p1) ** 0.5))
        lines.append(f"constexpr int kGroups_{name} = {len(f1)};")
        lines.append(f"__host__ __device__ constexpr int kPat_{name}(int i) {{")
        lines.append(f"  constexpr signed char t[{n * n}] = {{")
        for r in range(n):
            lines.append("      " + ", ".join(str(v) for v in p1[r * n:(r + 1) * n]) + ",")
        lines.append("  };")
        lines.append("  return t[i];")
        lines.append("}")
        lines.append(f"constexpr int kFirst_{name}[{len(f1)}] = {{" + ", ".join(map(str, f1)) + "};")
        lines.append("")
    lines.append("}  // namespace tl")
    (HERE / "ke_pattern.hpp").write_text("\n".join(lines) + "\n")
    print("wrote", HERE / "ke_pattern.hpp")
    write_sym()


if __name__ == "__main__":
    main()
