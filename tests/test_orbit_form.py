"""The orbit form of the symmetric perturbed averages (CPU).

The average T over the configurations is linear in the perturbation v = (R1, Y1),
so where the rotated perturbations S_j^T v span r dimensions, S_j^T v = sum_k C_jk
S_p(k)^T v, the symmetric average is sum_j S_j sum_k C_jk T(S_p(k)^T v) / N_sym: r
averages instead of one over N N_sym images (tdscha_amd/csrc/orbit.hip).  Checked on
the C oracle for the 48 point-group images of the reference's SnTe data (Raman-like
and vector-like members, d4 on and off), and that a perturbation of no symmetry
spans all of them."""
import numpy as np
import pytest

from oracle import c_oracle as CO
from tests.systems import load_snte, random_perturbation
from tests.test_rotation_form import dense_syms


def relation(R1, Y1, S, tol=1e-10):
    W = np.array([np.concatenate([s.T @ R1, (s.T @ Y1 @ s).ravel()]) for s in S])
    W /= np.linalg.norm(W[0])
    V, piv = W.copy(), []
    while True:
        p = int(np.argmax(np.linalg.norm(V, axis=1)))
        if np.linalg.norm(V[p]) < tol or len(piv) == len(S):
            break
        piv.append(p)
        q = V[p] / np.linalg.norm(V[p])
        for _ in range(2):
            V -= np.outer(V @ q, q)
    return piv, np.linalg.lstsq(W[piv].T, W.T, rcond=None)[0].T


@pytest.mark.parametrize("d4", [0, 1])
@pytest.mark.parametrize("axis, most", [(None, 1), (0, 6), (1, 6)])
def test_orbit_average_equals_image_average(axis, most, d4):
    d = load_snte()
    ms, n = d["syms_gamma"], d["X"].shape[1]
    S = dense_syms(ms.symmetries, ms.degenerate_space, n)
    R1, Y1 = random_perturbation(n, seed=3)
    # project on the invariant perturbations, or on the sector of one degenerate mode
    deg = [b for b in ms.degenerate_space if len(b) > 1]
    chi = np.ones(len(S)) if axis is None else S[:, deg[axis][0], deg[axis][0]]
    R1 = np.einsum("j,jab,b->a", chi, S, R1)
    Y1 = np.einsum("j,jab,bc,jdc->ad", chi, S, Y1, S, optimize=True)
    piv, C = relation(R1, Y1, S)
    assert 1 <= len(piv) <= most
    args = (d["X"], d["Y"], d["w"], d["rho"])
    ident = [np.eye(len(b))[None] for b in ms.degenerate_space]
    T = [CO.oracle_perturb_averages(*args, S[p].T @ R1, S[p].T @ Y1 @ S[p], float(d["T"]), d4,
                                    ident, ms.degenerate_space, ms.sym_block_id) for p in piv]
    f = sum(s @ sum(c * t[0] for c, t in zip(cj, T)) for s, cj in zip(S, C)) / len(S)
    v = sum(s @ sum(c * t[1] for c, t in zip(cj, T)) @ s.T for s, cj in zip(S, C)) / len(S)
    fo, vo = CO.oracle_perturb_averages(*args, R1, Y1, float(d["T"]), d4, ms.symmetries,
                                        ms.degenerate_space, ms.sym_block_id)
    # 1e-8: the group's own tables hold to about 1e-9 on these relaxed positions
    assert np.linalg.norm(f - fo) <= 1e-8 * np.linalg.norm(fo)
    assert np.linalg.norm(v - vo) <= 1e-8 * np.linalg.norm(vo)


def test_no_symmetry_spans_every_image():
    d = load_snte()
    ms, n = d["syms_gamma"], d["X"].shape[1]
    R1, Y1 = random_perturbation(n, seed=4)
    S = dense_syms(ms.symmetries, ms.degenerate_space, n)
    assert len(relation(R1, Y1, S)[0]) > 6
