"""The matrix-core scatters at the edges of its tiles, coil groups and visit
lists, against the FP64 oracle's adjoint: coil counts around the 8- and 16-coil
groups (odd ones without 16-byte loads), every window width, grids whose sides
are not multiples of the 8-cell tile, lists shared by 1 to 8 waves, split over
work items, shorter than one staged batch, and empty."""
import numpy as np
import pytest

from helpers import rand_img, rand_traj, rel

pytestmark = pytest.mark.gpu


def _samples(rng, kind):
    if kind == "few":
        return rand_traj(rng, 2, 5)
    spread = rng.uniform(-0.5, 0.5, size=(2, 700))
    if kind == "spread":
        return np.asfortranarray(spread.astype(np.float32))
    # dense: thousands of visits to the tiles around one point, hundreds around another
    c = 0.03 * rng.standard_normal((2, 3000)) + np.array([[0.0], [0.11]])
    c2 = 0.01 * rng.standard_normal((2, 300)) + np.array([[-0.3], [0.49]])
    k = np.concatenate([spread, c, np.clip(c2, -0.5, 0.4999)], axis=1)
    return np.asfortranarray(k.astype(np.float32))


@pytest.mark.parametrize("C,m,N,kind", [
    (1, 3, (32, 32), "dense"), (2, 1, (18, 27 * 2), "spread"), (7, 3, (24, 18), "dense"), (8, 4, (32, 32), "dense"),
    (9, 2, (18, 24), "dense"), (15, 3, (32, 18), "few"), (16, 3, (32, 32), "dense"), (17, 4, (18, 18), "spread"),
    (32, 3, (48, 32), "dense"), (33, 3, (24, 24), "spread"), (5, 2, (16, 16), "few"),
])
def test_scatter_matches_oracle(cgs, ora, C, m, N, kind):
    """FP32 products and sums over at most a few thousand visits: well within 1e-5."""
    rng = np.random.default_rng(1000 * C + 10 * m + len(kind))
    k = _samples(rng, kind)
    M = k.shape[1]
    w = rng.uniform(0.2, 1.0, M).astype(np.float32)
    S = rand_img(rng, N + (C,))
    y = rand_img(rng, (M, C))
    P = cgs.Plan(N, M, 2.0, m, ncoils=C)
    P.kspace(k)
    P.weights(w)
    P.sensitivities(S)
    O = ora.NFFT(N, M, 2.0, m)
    O.kspace(k)
    a = P.nfft_adjoint(y).reshape(N + (C,), order="F")
    e1 = max(rel(a[..., c], O.adjoint(y[:, c])) for c in range(C))
    e2 = rel(P.EH(y), O.EH_true(S, w, y))
    print(f"C={C} m={m} N={N} {kind}: adjoint {e1:.2e}, E^H W {e2:.2e}")
    assert e1 <= 1e-5 and e2 <= 1e-5


@pytest.mark.parametrize("C,m,N,kind", [
    (1, 3, (16, 16, 16), "dense"), (8, 2, (18, 16, 12), "dense"), (7, 4, (16, 12, 16), "few"),
    (9, 3, (12, 18, 16), "dense"), (16, 1, (16, 16, 18), "spread"), (17, 3, (16, 16, 16), "spread"),
])
def test_scatter_3d_matches_oracle(cgs, ora, C, m, N, kind):
    """3D: partial tiles on every axis, items split over blocks, batches with few or no
    visits of a plane.  FP32 sums as above."""
    rng = np.random.default_rng(7000 + 100 * C + m)
    M = {"few": 3, "spread": 1500, "dense": 6000}[kind]
    k = rng.uniform(-0.5, 0.5, size=(3, M))
    if kind == "dense":
        k[:, 1000:] *= 0.08
    k = np.asfortranarray(k.astype(np.float32))
    w = rng.uniform(0.2, 1.0, M).astype(np.float32)
    S = rand_img(rng, N + (C,))
    y = rand_img(rng, (M, C))
    P = cgs.Plan(N, M, 2.0 if m == 4 else 1.5, m, ncoils=C)
    P.kspace(k)
    P.weights(w)
    P.sensitivities(S)
    O = ora.NFFT(N, M, 2.0 if m == 4 else 1.5, m)
    O.kspace(k)
    a = P.nfft_adjoint(y).reshape(N + (C,), order="F")
    e1 = max(rel(a[..., c], O.adjoint(y[:, c])) for c in range(C))
    e2 = rel(P.EH(y), O.EH_true(S, w, y))
    print(f"3D C={C} m={m} N={N} {kind}: adjoint {e1:.2e}, E^H W {e2:.2e}")
    assert e1 <= 1e-5 and e2 <= 1e-5
