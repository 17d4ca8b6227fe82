"""Column matvec with each column split over two waves (k_matvec3s, both summation orders) against the oracle where its 16 x 8
tiles, odd column depths and stencil widths can go wrong."""
import numpy as np
import pytest

import ow3d
from ow3d import problems
from conftest import oracle_params


@pytest.mark.gpu
@pytest.mark.parametrize("nx,ny,nz,half", [
    (14, 14, 9, 3),      # 16 x 16 columns with the ghosts: whole tiles
    (15, 15, 9, 3),      # one column and one row more: tiles of a single column
    (33, 9, 8, 4),       # odd column depth, one window in y
    (7, 31, 6, 3),       # one window in x
    (47, 23, 4, 2), (18, 40, 13, 4), (9, 9, 5, 1),
])
def test_both_orders_match_the_oracle(oracle_mod, nx, ny, nz, half):
    lx, ly = 2 * np.pi * (nx - 1) / 24, 2 * np.pi * (ny - 1) / 24
    bath = problems.gaussian_shoal(nx, ny, lx, ly)
    cfg = dict(nx=nx, ny=ny, nz=nz, lx=lx, ly=ly, alpha=half, beta=half, gamma=half, precond=0, mg_maxgrids=1)
    p = oracle_params(nx, ny, nz, **{k: v for k, v in cfg.items() if k not in ("nx", "ny", "nz")})
    O = oracle_mod.OracleTank(p, bath["h"], bath["hx"], bath["hy"], bath["hxx"], bath["hyy"])
    T = ow3d.Tank(cfg, **bath)
    rng = np.random.default_rng(nx + 100 * ny + nz)
    X, Y = np.meshgrid(*problems.coords(nx, ny, lx, ly))
    E = 0.02 * np.cos(X) * np.sin(Y + 1)
    P = 0.1 * rng.standard_normal(E.shape)
    O.surface(E, P)
    T.set_surface(E, P)
    phi = rng.standard_normal(T.shape3)
    want = O.matvec(phi)
    got = {}
    for variant in (0, 1, 3):
        T.tune(variant, 0)
        got[variant] = T.laplace_apply(phi)
        # a row is a sum of some 60 products: the bound of the other comparisons with the oracle
        assert np.linalg.norm(got[variant] - want) <= 1e-12 * np.linalg.norm(want)
    assert np.array_equal(got[0], got[1])
    T.close()
    O.close()
