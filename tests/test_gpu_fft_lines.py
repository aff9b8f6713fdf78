"""Every line length of the register FFT passes (36 to 648 points) against the
FP64 oracle, with coil counts that leave lanes of a 16-line block idle, put
several rows into a block, and let a block's rows lie in two frames."""
import numpy as np
import pytest

from helpers import rand_img, rand_traj, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,sigma,C", [
    ((24, 32), 1.5, 1), ((36, 48), 1.5, 3), ((54, 64), 1.5, 8), ((32, 54), 2.0, 5), ((64, 72), 2.0, 2),
    ((72, 64), 2.0, 16), ((96, 72), 2.0, 12), ((72, 96), 2.0, 17), ((108, 162), 2.0, 7), ((162, 108), 1.5, 9),
    ((128, 144), 2.0, 4), ((144, 128), 2.0, 24), ((192, 216), 2.0, 6), ((216, 192), 2.0, 20), ((324, 288), 1.5, 10),
    ((256, 288), 2.0, 3), ((288, 256), 2.0, 18), ((324, 216), 2.0, 1), ((192, 324), 2.0, 33),
    # one and two coils, either side of where few rows leave k_fft_pt for k_fft
    ((96, 1024), 2.0, 1), ((96, 1152), 2.0, 1), ((72, 54), 2.0, 1), ((256, 96), 2.0, 1), ((162, 54), 1.5, 1),
    ((128, 384), 2.0, 2), ((128, 432), 2.0, 2), ((192, 96), 2.0, 2), ((216, 36), 2.0, 2), ((256, 768), 2.0, 2),
])
def test_lines_match_oracle(cgs, ora, N, sigma, C):
    """E and E^H W: FP32 transforms of at most 648 x 576 points, errors of a few
    1e-7; the Toeplitz operator (lines of 2 N points) to the window's accuracy."""
    rng = np.random.default_rng(N[0] * 1000 + N[1] + C)
    M = 400
    k = rand_traj(rng, 2, M)
    w = rng.uniform(0.2, 1.0, M).astype(np.float32)
    S = rand_img(rng, N + (C,))
    x, y = rand_img(rng, N), rand_img(rng, (M, C))
    P = cgs.Plan(N, M, sigma, 3, ncoils=C)
    P.kspace(k)
    P.weights(w)
    P.sensitivities(S)
    O = ora.NFFT(N, M, sigma, 3)
    O.kspace(k)
    e1, e2 = rel(P.E(x), O.E(S, x)), rel(P.EH(y), O.EH_true(S, w, y))
    # (the spectrum's set-up transforms four times the side, at most 4096 points)
    e3 = rel(P.normal(x, lam=0.5, toeplitz=True), P.normal(x, lam=0.5)) if 4 * max(N) <= 4096 else 0.0
    print(f"{N} sigma={sigma} C={C}: E {e1:.2e}, E^H W {e2:.2e}, Toeplitz {e3:.2e}")
    assert e1 <= 1e-5 and e2 <= 1e-5
    assert e3 <= (2e-5 if sigma == 2.0 else 2e-4)


@pytest.mark.parametrize("N,C", [((24, 36, 32), 3), ((32, 24, 36), 10), ((36, 32, 24), 17), ((24, 32, 36), 1)])
def test_volume_lines_match_oracle(cgs, ora, N, C):
    """Volumes of three different sides (a row's place on the other two axes): errors as
    in the plane."""
    rng = np.random.default_rng(N[0] * 1000 + N[1] + C)
    M = 500
    k = rand_traj(rng, 3, M)
    w = rng.uniform(0.2, 1.0, M).astype(np.float32)
    S = rand_img(rng, N + (C,))
    x, y = rand_img(rng, N), rand_img(rng, (M, C))
    P = cgs.Plan(N, M, 1.5, 3, ncoils=C)
    P.kspace(k)
    P.weights(w)
    P.sensitivities(S)
    O = ora.NFFT(N, M, 1.5, 3)
    O.kspace(k)
    e1, e2 = rel(P.E(x), O.E(S, x)), rel(P.EH(y), O.EH_true(S, w, y))
    e3 = rel(P.normal(x, lam=0.5, toeplitz=True), P.normal(x, lam=0.5))
    print(f"{N} C={C}: E {e1:.2e}, E^H W {e2:.2e}, Toeplitz {e3:.2e}")
    assert e1 <= 1e-5 and e2 <= 1e-5 and e3 <= 2e-4


@pytest.mark.parametrize("N,C", [((32, 18), 3), ((48, 54), 1), ((36, 18), 10)])
@pytest.mark.parametrize("toeplitz", [False, True])
def test_rows_of_two_frames(cgs, N, C, toeplitz):
    """Frames that stop at different iterations (weights of another scale against the
    same lam), with blocks that hold rows of two frames, so that for some iterations a
    block has a finished and a live one: each frame equals its own solve of as many
    iterations."""
    rng = np.random.default_rng(N[0] + C)
    off = np.array([0, 300, 900, 1100], dtype=np.int64)
    k = rand_traj(rng, 2, int(off[-1]))
    w = rng.uniform(0.2, 1.0, int(off[-1])).astype(np.float32)
    w[:off[1]] *= 1e-4
    w[off[2]:] *= 1e-4
    S = rand_img(rng, N + (C,))
    x = rand_img(rng, N + (3,))
    P = cgs.Plan(N, int(off[-1]), 2.0, 3, ncoils=C, frame_offsets=off)
    P.kspace(k)
    P.weights(w)
    P.sensitivities(S)
    y = P.E(x)
    xb, rb = P.solve(y, maxit=12, tol=0.2, lam=0.5, toeplitz=toeplitz)
    its = [int(i) for i in rb["iters"]]
    print(f"{N} C={C} toeplitz={toeplitz}: iterations {its}")
    assert its[0] < its[1] and its[2] < its[1] < 12
    for f in range(3):
        Mf = int(off[f + 1] - off[f])
        P1 = cgs.Plan(N, Mf, 2.0, 3, ncoils=C)
        P1.kspace(k[:, off[f]:off[f + 1]])
        P1.weights(w[off[f]:off[f + 1]])
        P1.sensitivities(S)
        yf = y[C * off[f]:C * off[f + 1]].reshape((Mf, C), order="F")
        x1, _ = P1.solve(yf, maxit=its[f], tol=0.0, lam=0.5, toeplitz=toeplitz)
        assert rel(xb[..., f], x1) <= 1e-5


@pytest.mark.parametrize("graph", [0, 3])
def test_toeplitz_runs_of_frames(cgs, graph):
    """25 frames of 192^2 x 16 coils: the Toeplitz passes go over them in two runs
    (13 and 12 frames); frames at the ends of both runs equal their own solves."""
    N, C, F, Mf = (192, 192), 16, 25, 250
    rng = np.random.default_rng(192)
    off = np.arange(F + 1, dtype=np.int64) * Mf
    k = rand_traj(rng, 2, F * Mf)
    w = rng.uniform(0.2, 1.0, F * Mf).astype(np.float32)
    S = rand_img(rng, N + (C,))
    P = cgs.Plan(N, F * Mf, 2.0, 3, ncoils=C, frame_offsets=off)
    P.kspace(k)
    P.weights(w)
    P.sensitivities(S)
    y = P.E(rand_img(rng, N + (F,)))
    xb, rb = P.solve(y, maxit=6, tol=0.0, lam=0.5, toeplitz=True, graph_iters=graph)
    P1 = cgs.Plan(N, Mf, 2.0, 3, ncoils=C)
    P1.sensitivities(S)
    for f in (0, 12, 13, 24):
        P1.kspace(k[:, off[f]:off[f + 1]])
        P1.weights(w[off[f]:off[f + 1]])
        yf = y[C * off[f]:C * off[f + 1]].reshape((Mf, C), order="F")
        x1, _ = P1.solve(yf, maxit=6, tol=0.0, lam=0.5, toeplitz=True)
        assert rel(xb[..., f], x1) <= 1e-5
