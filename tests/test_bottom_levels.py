"""One-workgroup kernel for the small multigrid levels (k_mg_bottom): its threads' columns on the CPU, and on the GPU V cycles
with it against the same V cycles with one launch per step, which are the same arithmetic: equal bits."""
import os

import numpy as np
import pytest

import ow3d
from ow3d import problems

NT = 256


def _inner(nxg, nyg, d3):
    return (nxg - 3) // 2 * (nyg - 4 if d3 else 1) if nxg > 4 and (not d3 or nyg > 4) else 0


def _fits(nxg, nyg, d3):
    edge = 2 * ((nxg - 1) // 2) + 2 * ((nyg - 1) // 2) if d3 else 2
    ghosts = 2 * nxg + 2 * (nyg - 2) if d3 else 2
    return -(-_inner(nxg, nyg, d3) // 64) * 64 + -(-edge // 32) * 64 <= NT and ghosts <= NT // 2 and nxg * nyg <= 2 * NT


@pytest.mark.parametrize("d3", [True, False])
def test_threads_cover_each_column_of_a_colour_once(d3):
    fitting = 0
    for nxg in range(4, 400):
        for nyg in (range(4, 70) if d3 else [1]):
            if not _fits(nxg, nyg, d3):
                continue
            fitting += 1
            ni, hw, g = _inner(nxg, nyg, d3), max((nxg - 3) // 2, 1), 1 if d3 else 0
            nip = -(-ni // 64) * 64
            bx, by = ((nxg - 1) // 2, (nyg - 1) // 2) if d3 else (0, 1)
            for c in (0, 1):
                cols = []
                for th in range(NT):
                    if th < nip:
                        r = th // hw if d3 else 0
                        j = 2 + r if d3 else 0
                        i = 2 + (1 if (j & 1) != c else 0) + 2 * (th - r * hw)
                        on = th < ni and i <= nxg - 3
                    else:
                        if (th - nip) & 32:   # the second lane of a column
                            continue
                        l = ((th - nip) >> 6) * 32 + ((th - nip) & 31)
                        if d3 and l < 2 * bx:
                            first = l < bx
                            j = 1 if first else nyg - 2
                            i = 1 + (1 if ((1 + j) & 1) != c else 0) + 2 * (l if first else l - bx)
                            on = i <= nxg - 2 and (first or nyg > 3)
                        else:
                            q = l - 2 * bx
                            first = q < by
                            i = 1 if first else nxg - 2
                            j = g + (1 if ((i + g) & 1) != c else 0) + 2 * (q if first else q - by)
                            on = q < 2 * by and j <= (nyg - 2 if d3 else 0) and (first or nxg > 3) and not (d3 and j in (1, nyg - 2))
                    if on:
                        cols.append((i, j))
                want = [(i, j) for j in (range(1, nyg - 1) if d3 else [0]) for i in range(1, nxg - 1) if (i + j) & 1 == c]
                assert sorted(cols) == want or sorted(cols) == sorted(want)
    assert fitting > 100


@pytest.mark.gpu
@pytest.mark.parametrize("mg", [0, 1, 2])
@pytest.mark.parametrize("nx,ny,nz,kw", [
    (33, 33, 9, {}),                                          # 17^2 below: the largest square level that fits
    (65, 33, 9, dict(nu1=2, nu2=3, maxit=2)),                 # several sweeps and cycles
    (41, 25, 13, {}),                                         # deepest columns, coarsened in sigma
    (33, 17, 12, {}),                                         # odd column depth, not coarsened in sigma
    (17, 9, 4, dict(alpha=2, beta=2, gamma=2)),               # shallowest
    (25, 41, 7, dict(alpha=2, beta=2, gamma=2)), (33, 33, 13, {}),
    (97, 161, 8, {}),                                         # dense solve of 432 points: a launch of its own
    (65, 65, 9, dict(mg_maxgrids=4)),                         # and of 1210
    (257, 1, 9, {}), (129, 1, 12, dict(nu1=2)), (33, 1, 6, dict(alpha=2, beta=2, gamma=2)),   # x-z
])
def test_same_bits_as_one_launch_per_step(nx, ny, nz, mg, kw):
    lx = 2 * np.pi * (nx - 1) / 24
    ly = 2 * np.pi * (ny - 1) / 24 if ny > 1 else 1.0
    bath = problems.gaussian_shoal(nx, ny, lx, ly)
    cfg = dict(nx=nx, ny=ny, nz=nz, lx=lx, ly=ly, mg_precision=mg, **kw)
    T = ow3d.Tank(cfg, **bath)
    os.environ["OW3D_MG_BOTTOM"] = "0"
    try:
        W = ow3d.Tank(cfg, **bath)
    finally:
        del os.environ["OW3D_MG_BOTTOM"]
    rng = np.random.default_rng(nx * ny + nz)
    for scale in (1.0, 1e-3):   # the second application reuses every buffer of the first
        r = scale * rng.standard_normal(T.shape3)
        want = W.precond_apply(r)
        assert np.abs(want).max() > 0
        assert np.array_equal(T.precond_apply(r), want)
    T.close()
    W.close()
