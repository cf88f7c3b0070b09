"""The steps of the FP32 Hex8 block pass (four lanes per element: hex8_quad,
quad_grad, quad_force in akantu2_amd/csrc/akx_fast.hip), restated lane by lane
in numpy, against the direct contraction with the dN/dxi table of the 2 x 2 x 2
Gauss rule: gradients, det J signs, nodal forces, and the neo-Hookean force on
the current configuration against F S.  FP64 on both sides: 1e-12."""
import os
import re

import numpy as np
import pytest

SRC = os.path.join(os.path.dirname(__file__), "..", "akantu2_amd", "csrc", "akx_fast.hip")
G = 1.0 / np.sqrt(3.0)
R, KS, KD = (1.0 - G) / (1.0 + G), 1307 / 2048, 1307 / 2048 * G
W = 1.0 / (2 * (1 + R) ** 2 * (4 * KS * (1 + R)) ** 2)
SIGNS = np.array([(-1, -1, -1), (1, -1, -1), (1, 1, -1), (-1, 1, -1),
                  (-1, -1, 1), (1, -1, 1), (1, 1, 1), (-1, 1, 1)], float)
LANES = np.arange(4)  # bit 0 y, bit 1 z


def corners(b):
    """Element corners (x-, x+) of lane b: the pair 2 b, 2 b + 1, turned at y+."""
    pair = (2 * b, 2 * b + 1)
    return pair[::-1] if b & 1 else pair


def x1(v):
    return v[LANES ^ 1]


def x2(v):
    return v[LANES ^ 2]


def quad_grad(v0, v1):
    d, s = v1 - v0, KS * (v0 + v1)
    dp, sp = x2(d), x2(s)
    dzd, izd = d - dp, d + R * dp
    dzs, izs = s - sp, s + R * sp
    ip = x1(izd)
    return (izd + R * ip, izs - x1(izs), KD * (izd - ip), dzs + R * x1(dzs),
            KD * (dzd + R * x1(dzd)))


def quad_force(m, p):
    X = p[0] + m[0]
    Se, E = p[1] + m[1], KD * (p[1] - m[1])
    Sz, Z = p[2] + m[2], KD * (p[2] - m[2])
    da = (X + E) + x1(R * X - E)
    db = Z + R * x1(Z)
    d = (da + db) + x2(R * da - db)
    sa = Se - x1(Se)
    sb = Sz + R * x1(Sz)
    s = (sa + sb) + x2(R * sa - sb)
    return KS * s - d, KS * s + d


def dn_table():
    d = np.zeros((8, 3, 8))
    for q in range(8):
        c = [(G if (q >> a) & 1 else -G) for a in range(3)]
        for n in range(8):
            for m in range(3):
                d[q, m, n] = 0.125 * SIGNS[n, m] * np.prod(
                    [1.0 + SIGNS[n, o] * c[o] for o in range(3) if o != m])
    return d


@pytest.mark.parametrize("seed", [1, 2, 3])
def test_quad_steps_equal_direct_contraction(seed):
    rng = np.random.default_rng(seed)
    D = dn_table()
    X = SIGNS * 0.5 + rng.uniform(-0.15, 0.15, (8, 3)) + rng.uniform(-50, 50, 3)
    U = rng.uniform(-1e-1, 1e-1, (8, 3))
    lam, mu = 0.7, 0.4
    J = np.einsum("qmn,nc->qmc", D, X)
    H = np.einsum("qmn,nc->qmc", D, U)
    Ji, det = np.linalg.inv(J), np.linalg.det(J)
    g = np.einsum("qma,qbm->qab", H, Ji)
    F = g + np.eye(3)
    Ci = np.linalg.inv(np.einsum("qki,qkj->qij", F, F))
    jdet = np.linalg.det(F)
    S = mu * np.eye(3) + (lam * np.log(jdet) - mu)[:, None, None] * Ci
    P = np.einsum("qik,qkj->qij", F, S)
    f = np.einsum("q,qkj,qjm,qmn->nk", det, P, Ji, D)

    v0 = np.array([corners(b)[0] for b in LANES])
    v1 = np.array([corners(b)[1] for b in LANES])
    assert (SIGNS[v0, 0] < 0).all() and (SIGNS[v1, 0] > 0).all()
    for a in (1, 2):
        assert np.array_equal(SIGNS[v0, a] > 0, (LANES >> (a - 1)) & 1)
        assert np.array_equal(SIGNS[v1, a] > 0, (LANES >> (a - 1)) & 1)
    gx = [quad_grad(X[v0, c] - X[0, c], X[v1, c] - X[0, c]) for c in range(3)]
    gu = [quad_grad(U[v0, c] - U[0, c], U[v1, c] - U[0, c]) for c in range(3)]
    w = np.where((LANES == 1) | (LANES == 2), -W, W)
    Q = []
    for ix in (0, 1):
        s = 1 if ix else -1
        Jl, Hl = (np.array([[t[c][0], t[c][1] + s * t[c][2], t[c][3] + s * t[c][4]]
                            for c in range(3)]).transpose(2, 1, 0) for t in (gx, gu))
        q = ix + 2 * LANES
        gl = np.einsum("lma,lbm->lab", Hl, np.linalg.inv(Jl))
        assert np.abs(gl - g[q]).max() <= 1e-12 * np.abs(g).max()
        K = np.linalg.inv(Jl) * np.linalg.det(Jl)[:, None, None]
        Qp = w[:, None, None] * np.einsum("lkj,ljm->lkm", P[q], K)
        # the neo-Hookean form: tau adj(J + H) / det F, b - I without b
        jm1 = np.trace(gl, axis1=1, axis2=2) + sum(
            gl[:, i, i] * gl[:, j, j] - gl[:, i, j] * gl[:, j, i]
            for i, j in ((0, 1), (0, 2), (1, 2))) + np.linalg.det(gl)
        bi = gl + gl.transpose(0, 2, 1) + np.einsum("lik,ljk->lij", gl, gl)
        tau = mu * bi + (lam * np.log1p(jm1))[:, None, None] * np.eye(3)
        jc = Jl + Hl
        Kc = np.linalg.inv(jc) * np.linalg.det(jc)[:, None, None]
        Qn = (w / (1 + jm1))[:, None, None] * np.einsum("lkj,ljm->lkm", tau, Kc)
        assert np.abs(Qn - Qp).max() <= 1e-12 * np.abs(Qp).max()
        Q.append(Qn)
    got = np.zeros((8, 3))
    for k in range(3):
        f0, f1 = quad_force([Q[0][:, k, m] for m in range(3)], [Q[1][:, k, m] for m in range(3)])
        got[v0, k], got[v1, k] = f0, f1
    assert np.abs(got - f).max() <= 1e-12 * np.abs(f).max()


def test_kernel_constants():
    src = open(SRC).read()
    for name, value in (("HEX_R", R), ("HEX_KS", KS), ("HEX_KD", KD)):
        got = float(re.search(name + r" = ([0-9.eE+-]+)f;", src).group(1))
        assert got == pytest.approx(value, rel=1e-15)
        # FP32 holds them well: their rounding is the same in every step
        assert abs(float(np.float32(value)) / value - 1) <= 5e-9
