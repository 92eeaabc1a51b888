"""CPU restatement of the device's 32x32 pivot-block inverse (gj_invert_pivot
in topoptlab_amd/csrc/tl_mg.hip), lane by lane: 2 x 2 blocks in the FP64
matrix-core output layout (lane l holds rows l/16 + 4i of column l%16), the
pivot row and column moved by a row broadcast and two lane-row swaps."""
import numpy as np
import pytest

L = np.arange(64)
J, G = L & 15, L >> 4


def to_c(M):
    return np.stack([M[G + 4 * i, J] for i in range(4)])


def from_c(v):
    M = np.full((16, 16), np.nan)
    for i in range(4):
        M[G + 4 * i, J] = v[i]
    return M


def row_bcast(v, n):  # lane n of each row of 16
    return v[(L & ~15) + n]


def group_bcast(v, g):
    lo, hi = v[:32], v[32:]  # permlane32_swap(v, v)
    y = np.concatenate([hi, hi] if g & 2 else [lo, lo])
    r = y.reshape(4, 16)  # permlane16_swap(y, y)
    return (np.stack([r[1], r[1], r[3], r[3]]) if g & 1
            else np.stack([r[0], r[0], r[2], r[2]])).reshape(-1)


def invert32(P):
    v = np.stack([np.stack([to_c(P[16 * r:16 * r + 16, 16 * c:16 * c + 16]) for c in range(2)])
                  for r in range(2)])
    for T in range(32):
        bt, t = T >> 4, T & 15
        gt, it = t & 3, t >> 2
        row = [group_bcast(v[bt, b, it], gt) for b in range(2)]
        c = np.stack([[row_bcast(v[b, bt, i], t) for i in range(4)] for b in range(2)])
        p = 1.0 / row_bcast(row[bt], t)
        f = [p * r for r in row]
        v[:, bt, :, J == t] = 0.0
        f[bt] = np.where(J == t, p, f[bt])
        c[bt, it] = np.where(G == gt, -1.0, c[bt, it])
        v[bt, :, it] = np.where(G == gt, 0.0, v[bt, :, it])
        for a in range(2):
            for b in range(2):
                v[a, b] -= c[a] * f[b]
    return np.block([[from_c(v[r, c]) for c in range(2)] for r in range(2)])


@pytest.mark.parametrize("seed,spread", [(0, 0), (1, 4), (2, 9)])
def test_pivot_block_inverse(seed, spread):
    rng = np.random.default_rng(seed)
    Q, _ = np.linalg.qr(rng.standard_normal((32, 32)))
    P = (Q * 10.0 ** rng.uniform(-spread, 0, 32)) @ Q.T
    P = 0.5 * (P + P.T)
    R = invert32(P)
    # residual of a backward-stable inverse: eps * n * condition
    assert np.abs(R @ P - np.eye(32)).max() < 2.3e-16 * 32 * np.linalg.cond(P)
