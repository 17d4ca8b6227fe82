"""Zebra sweep kernels (k_mg_sweep, k_mg_sweep_tiled): the arithmetic of their tiles on the CPU for every level size,
and V cycles on the GPU against the oracle where tiles, walls and column depths can go wrong."""
import numpy as np
import pytest

import ow3d
from ow3d import problems
from conftest import oracle_params

TILES = [(18, 8, False), (36, 8, True), (18, 8, True), (66, 1, False)]   # k_mg_sweep, k_mg_sweep_tiled FP32 / FP64, x-z


def _begin(n, t, nt):
    return 1 + n * t // nt


def _colour(lo, hi, fixed, col):
    """Indices lo .. hi of colour col beside the fixed index, as the kernels enumerate them."""
    return list(range(lo + (1 if ((lo + fixed) & 1) != col else 0), hi + 1, 2))


@pytest.mark.parametrize("TX,TY,tiled", TILES)
@pytest.mark.parametrize("nx", [2, 3, 4, 5, 17, 18, 19, 33, 35, 36, 37, 38, 65, 67, 73, 129, 257, 513])
def test_tiles_cover_each_column_once_and_fit_their_lists(TX, TY, tiled, nx):
    d3 = TY > 1
    for ny in ([2, 3, 8, 9, 10, 17, 33, 129] if d3 else [1]):
        nxg, nyg = nx + 2, ny + 2 if d3 else 1
        gx, gy = -(-nx // TX), -(-ny // TY) if d3 else 1
        RX, RY = TX // 2 + 1, TY + 2 if d3 else 1
        NT = -(-RX * RY // 64) * 64
        WX, WY = TX + 4, TY + 4 if d3 else 1
        BX, BY = (TX // 2 + 1, TY // 2 + 1) if d3 else (0, 1)
        seen = [np.zeros((nyg, nxg), int) for _ in range(2)]
        for bx in range(gx):
            i0, ie = _begin(nx, bx, gx), _begin(nx, bx + 1, gx)
            assert 2 <= ie - i0 <= TX
            for by in range(gy):
                j0, je = (_begin(ny, by, gy), _begin(ny, by + 1, gy)) if d3 else (0, 1)
                assert not d3 or 2 <= je - j0 <= TY
                lox, loy = max(i0 - 2, 0), max(j0 - 2, 0) if d3 else 0
                wcols, wrows = min(ie + 2, nxg) - lox, min(je + 2, nyg) - loy if d3 else 1
                assert wcols <= WX and wrows <= WY
                for row in range(wrows):   # one thread per window column of a colour
                    assert max(len(_colour(lox, lox + wcols - 1, loy + row, c)) for c in (0, 1)) <= WX // 2
                for col in (0, 1):
                    ilo, ihi = (max(i0 - 1, 1), min(ie, nxg - 2)) if col == 0 else (i0, ie - 1)
                    jlo, jhi = (0, 0) if not d3 else ((max(j0 - 1, 1), min(je, nyg - 2)) if col == 0 else (j0, je - 1))
                    cols = []
                    assert jhi - jlo + 1 <= RY
                    for j in range(jlo, jhi + 1):      # away from the walls
                        row = _colour(ilo, ihi, j, col)
                        assert len(row) <= RX
                        cols += [(i, j) for i in row if 2 <= i <= nxg - 3 and (not d3 or 2 <= j <= nyg - 3)]
                    if d3:
                        for j in [1] + ([nyg - 2] if nyg > 3 else []):
                            row = _colour(ilo, ihi, j, col)
                            assert len(row) <= BX
                            cols += [(i, j) for i in row if jlo <= j <= jhi]
                    for i in [1] + ([nxg - 2] if nxg > 3 else []):
                        row = _colour(jlo, jhi, i, col)
                        assert len(row) <= BY
                        cols += [(i, j) for j in row if ilo <= i <= ihi and not (d3 and j in (1, nyg - 2))]
                    assert len(cols) == len(set(cols))
                    want = [(i, j) for j in range(jlo, jhi + 1) for i in range(ilo, ihi + 1) if (i + j) & 1 == col]
                    assert sorted(cols) == sorted(want)
                    for i, j in cols:
                        # every neighbour a column reads is staged: in the window, and a ghost column within the ring
                        for a, b in [(i - 1, j), (i + 1, j)] + ([(i, j - 1), (i, j + 1)] if d3 else []):
                            assert lox <= a < lox + wcols and loy <= b < loy + wrows
                            assert i0 - 1 <= a <= ie or 1 <= a <= nxg - 2
                            assert not d3 or j0 - 1 <= b <= je or 1 <= b <= nyg - 2
                        if i0 <= i < ie and j0 <= j < je:
                            seen[col][j, i] += 1
                if not tiled:
                    assert 2 * (BX + BY) <= 32 and (WX // 2) * WY <= NT + 64
        inner = (slice(1, -1) if d3 else slice(0, 1), slice(1, -1))
        assert (seen[0] + seen[1])[inner].min() == 1 and (seen[0] + seen[1]).sum() == nx * ny


# the tolerances of the other V-cycle comparisons with the oracle: FP64 rounding through the levels' solves, FP32
# rounding of a few hundred operations
TOL = {0: 1e-10, 1: 1e-4}


@pytest.mark.gpu
@pytest.mark.parametrize("mg", [0, 1])
@pytest.mark.parametrize("nx,ny,nz,kw", [
    (17, 17, 9, {}),                              # one tile: every wall in it
    (37, 19, 5, dict(alpha=2, beta=2, gamma=2, mg_maxgrids=2)),   # one column more than a tile, shallow
    (41, 73, 13, {}),                             # deepest columns
    (97, 161, 8, dict(nu1=2, nu2=2, maxit=2)),    # odd column depth, several sweeps and cycles
    (129, 1, 9, {}), (67, 1, 12, dict(nu1=2, mg_maxgrids=2)),    # x-z
    (385, 257, 12, dict(mg_maxgrids=6)),          # finest level above the record limit: the tiled kernel
])
def test_v_cycle_matches_the_oracle(oracle_mod, nx, ny, nz, mg, kw):
    lx = 2 * np.pi * (nx - 1) / 24
    ly = 2 * np.pi * (ny - 1) / 24 if ny > 1 else 1.0
    bath = problems.gaussian_shoal(nx, ny, lx, ly)
    cfg = dict(nx=nx, ny=ny, nz=nz, lx=lx, ly=ly, mg_maxgrids=5)
    cfg.update(kw)
    p = oracle_params(nx, ny, nz, **{k: v for k, v in cfg.items() if k not in ("nx", "ny", "nz")})
    O = oracle_mod.OracleTank(p, bath["h"], bath["hx"], bath["hy"], bath["hxx"], bath["hyy"])
    T = ow3d.Tank(dict(cfg, mg_precision=mg), **bath)
    r = np.random.default_rng(nx * ny + nz).standard_normal(T.shape3)
    want = O.precond(r)
    for scale in (1.0, -3.0):   # the second application reuses every buffer of the first
        got = T.precond_apply(scale * r)
        assert np.max(np.abs(got - scale * want)) <= TOL[mg] * abs(scale) * np.max(np.abs(want))
    T.close()
    O.close()
