"""V cycles of hierarchies whose small levels run in the one-workgroup kernel (k_mg_bottom), each checked to do so, against
the oracle: every column depth, sigma-coarsened and partly coarsened levels, a dense solve of its own, x-z."""
import os

import numpy as np
import pytest

import ow3d
from ow3d import problems
from conftest import oracle_params

CASES = [
    (33, 33, 9, {}),                                          # last level coarsened in every direction
    (33, 33, 13, {}), (13, 13, 9, {}), (33, 17, 13, dict(nu1=3, nu2=2, maxit=2)),   # one coarsened in sigma alone
    (5, 25, 9, dict(alpha=1, beta=1, gamma=1, nu1=3)),        # in y alone, three columns wide below
    (17, 17, 4, dict(alpha=2, beta=2, gamma=2)),
    (33, 33, 5, dict(alpha=2, beta=2, gamma=2)), (33, 17, 6, {}), (25, 41, 7, {}),
    (33, 9, 10, {}), (65, 1, 11, {}), (33, 17, 12, {}),       # the other column depths
    (97, 17, 6, {}),                                          # levels of an even number of columns
    (97, 161, 8, {}),                                         # dense solve of 432 points: a launch of its own
    (257, 1, 9, {}), (129, 1, 12, dict(nu1=2)), (65, 1, 13, {}), (33, 1, 6, dict(alpha=2, beta=2, gamma=2)),   # x-z
]


def tank(nx, ny, nz, mg, kw, bottom=True):
    lx = 2 * np.pi * (nx - 1) / 24
    ly = 2 * np.pi * (ny - 1) / 24 if ny > 1 else 1.0
    bath = problems.gaussian_shoal(nx, ny, lx, ly)
    cfg = dict(nx=nx, ny=ny, nz=nz, lx=lx, ly=ly, mg_precision=mg, **kw)
    if not bottom:
        os.environ["OW3D_MG_BOTTOM"] = "0"
    try:
        T = ow3d.Tank(cfg, **bath)
    finally:
        if not bottom:
            del os.environ["OW3D_MG_BOTTOM"]
    assert T.mg_bottom_level() >= 1 if bottom else T.mg_bottom_level() == -1
    return T, cfg, bath


# the tolerances of the other V-cycle comparisons with the oracle: FP64 rounding through the levels' solves, FP32
# rounding of a few hundred operations
TOL = {0: 1e-10, 1: 1e-4}


@pytest.mark.gpu
@pytest.mark.parametrize("mg", [0, 1])
@pytest.mark.parametrize("nx,ny,nz,kw", CASES)
def test_v_cycle_matches_the_oracle(oracle_mod, nx, ny, nz, mg, kw):
    T, cfg, bath = tank(nx, ny, nz, mg, kw)
    p = oracle_params(nx, ny, nz, **{k: v for k, v in cfg.items() if k not in ("nx", "ny", "nz", "mg_precision")})
    O = oracle_mod.OracleTank(p, bath["h"], bath["hx"], bath["hy"], bath["hxx"], bath["hyy"])
    r = np.random.default_rng(nx * ny + nz).standard_normal(T.shape3)
    want = O.precond(r)
    for scale in (1.0, -3.0):   # the second application reuses every buffer of the first
        assert np.max(np.abs(T.precond_apply(scale * r) - scale * want)) <= TOL[mg] * abs(scale) * np.max(np.abs(want))
    T.close()
    O.close()


def smooth(shape, rng):
    """A residual whose V cycle lives on the coarse levels: a few long waves."""
    j, i, k = np.meshgrid(*[np.arange(n) for n in shape], indexing="ij")
    r = np.zeros(shape)
    for q in range(4):
        a = rng.uniform(0, 0.5, 3)
        a[q % 3] *= 0.1
        r += rng.standard_normal() * np.cos(a[0] * j + rng.uniform(0, 6)) * np.cos(a[1] * i + rng.uniform(0, 6)) * np.cos(a[2] * k + 1)
    return r


@pytest.mark.gpu
@pytest.mark.parametrize("mg", [0, 1, 2])
@pytest.mark.parametrize("nx,ny,nz,kw", CASES + [(25, 49, 13, dict(nu1=2, nu2=1)), (49, 33, 11, {}), (13, 13, 13, {})])
def test_same_bits_as_one_launch_per_step(nx, ny, nz, mg, kw):
    T, _, _ = tank(nx, ny, nz, mg, kw)
    W, _, _ = tank(nx, ny, nz, mg, kw, bottom=False)
    rng = np.random.default_rng(nx * ny + nz)
    # one rounding of a coarse level reaches the finest in one vector of several only
    for n in range(24):
        r = smooth(T.shape3, rng) * (1.0 + (n % 2) * 0.1 * rng.standard_normal(T.shape3))
        want = W.precond_apply(r)
        assert np.abs(want).max() > 0
        assert np.array_equal(T.precond_apply(r), want), n
    T.close()
    W.close()
