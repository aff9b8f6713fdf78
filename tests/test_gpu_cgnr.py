"""The iterative NFFT inverse where coils stop at different steps: one with no data,
one far below the stop test, one or two that meet it on the way, the others never; and
of volumes."""
import numpy as np
import pytest

from helpers import rand_img, rand_traj, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("C,maxit", [(4, 1), (4, 2), (11, 3), (33, 6)])
def test_coils_stop_apart(cgs, ora, C, maxit):
    """FP32 vectors, FP64 scalars: a few steps stay within 1e-5 of the FP64 oracle."""
    rng = np.random.default_rng(40 + C)
    N, M = (32, 32), 1500   # the oracle's damping mask is defined for equal sides
    k = rand_traj(rng, 2, M)
    w = rng.uniform(0.2, 1.0, M).astype(np.float32)
    O = ora.NFFT(N, M, 2.0, 3)
    O.kspace(k)
    y = np.stack([O.trafo(rand_img(rng, N)) for _ in range(C)], axis=1).astype(np.complex64)
    y[:, 0] = 0
    y[:, 1] *= 1e-4
    y[:, 2] *= 0.045         # stops after one step
    if C > 4:
        y[:, C - 1] *= 0.07  # after two or three
    eps = 1e-3 * float(np.sum(w * np.abs(y[:, 3].astype(np.complex128)) ** 2))
    y = np.asfortranarray(y)
    P = cgs.Plan(N, M, 2.0, 3, ncoils=C)
    P.kspace(k)
    P.weights(w)
    g = np.asarray(P.nfft_inverse_ref(y, maxit=maxit, eps=eps)).reshape(N + (C,), order="F")
    its = []
    for c in range(C):
        o, it, _ = O.itrafo(y[:, c], w, maxit=maxit, eps=eps)
        its.append(it)
        assert rel(g[..., c], o) <= 1e-5, (c, it)
    print(f"C={C} maxit={maxit}: steps {its[:4]} .. {its[-1]}")
    assert not g[..., 0].any()
    assert its[:2] == [0, 0] and its[3] == maxit
    assert maxit == 1 or any(0 < i < maxit for i in its)


@pytest.mark.parametrize("C", [3, 10])
def test_volume(cgs, ora, C):
    """24^3 on 36-point lines: the damping ball's third axis, with several rows in a block
    of the transform (3 coils) and one (10).  As above, 1e-5."""
    rng = np.random.default_rng(60 + C)
    N, M = (24, 24, 24), 4000
    k = rand_traj(rng, 3, M)
    w = rng.uniform(0.2, 1.0, M).astype(np.float32)
    y = rand_img(rng, (M, C))
    O = ora.NFFT(N, M, 1.5, 3)
    O.kspace(k)
    P = cgs.Plan(N, M, 1.5, 3, ncoils=C)
    P.kspace(k)
    P.weights(w)
    g = np.asarray(P.nfft_inverse_ref(y, maxit=3, eps=0.0)).reshape(N + (C,), order="F")
    for c in range(C):
        o, it, _ = O.itrafo(y[:, c], w, maxit=3, eps=0.0)
        assert it == 3 and rel(g[..., c], o) <= 1e-5
    i = np.indices(N) - 12
    assert not g[(i * i).sum(0) > 144].any()
