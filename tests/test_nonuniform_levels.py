"""V cycles on grids whose x rows differ by rounding (coordinates ((i - g) / (n - 1)) lx of some thousand columns): the level
operators then take every column's own stencil rows instead of one set for all, in tiles beside a wall and away from one."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

import ow3d
from ow3d import problems
from conftest import ROOT, oracle_params

# finest levels with column records (k_mg_sweep; several tiles without a wall): x-z, 3D, odd column depth; and one above
# the record limit (k_mg_sweep_tiled)
GRIDS = [(4097, 1, 9), (3073, 17, 9), (3073, 17, 8), (3073, 65, 9)]
STEP = 2 * np.pi / 24

HARNESS = r"""
#include "ow3d_grid.hpp"
using namespace ow3d;
extern "C" int finest_uniform(int nx, int ny, int nz, double lx, double ly) {
    Grid g;
    g.nx = nx; g.ny = ny; g.nz = nz; g.gx = 1; g.gy = ny > 1 ? 1 : 0;
    g.a = 3; g.b = ny > 1 ? 3 : 0; g.c = 3;
    g.alloc();
    fine_coords(g, lx, ly, 1.0, 1);
    grid_stencils(g);
    std::vector<Grid> lev;
    std::string err;
    if (!mg_levels(g, 20, lev, err)) return -1;
    const Grid &f = lev.back();
    double c[6];
    return uniform_rows(f.sx, f.nxg, c) && (ny == 1 || uniform_rows(f.sy, f.nyg, c + 3));
}
"""


def test_the_finest_levels_are_not_uniform(tmp_path):
    src, so = tmp_path / "uniform.cpp", tmp_path / "libuniform.so"
    src.write_text(HARNESS)
    subprocess.run(["g++", "-std=c++17", "-O2", "-shared", "-fPIC", "-I",
                    os.path.join(ROOT, "oceanwave3d-fortran90_amd", "csrc"), "-o", str(so), str(src)], check=True)
    f = ctypes.CDLL(str(so)).finest_uniform
    f.argtypes = [ctypes.c_int] * 3 + [ctypes.c_double] * 2
    for nx, ny, nz in GRIDS:
        assert f(nx, ny, nz, STEP * (nx - 1), STEP * (ny - 1)) == 0
    for nx, ny, nz in [(513, 513, 9), (257, 1, 9)]:
        assert f(nx, ny, nz, STEP * (nx - 1), STEP * (ny - 1)) == 1


# the tolerances of the other V-cycle comparisons with the oracle: FP64 rounding through the levels' solves, FP32
# rounding of a few hundred operations
TOL = {0: 1e-10, 1: 1e-4}


@pytest.mark.gpu
@pytest.mark.parametrize("mg", [0, 1])
@pytest.mark.parametrize("nx,ny,nz", GRIDS)
def test_v_cycle_matches_the_oracle(oracle_mod, nx, ny, nz, mg):
    lx, ly = STEP * (nx - 1), STEP * (ny - 1) if ny > 1 else 1.0
    bath = problems.gaussian_shoal(nx, ny, lx, ly)
    cfg = dict(nx=nx, ny=ny, nz=nz, lx=lx, ly=ly)
    p = oracle_params(nx, ny, nz, lx=lx, ly=ly)
    O = oracle_mod.OracleTank(p, bath["h"], bath["hx"], bath["hy"], bath["hxx"], bath["hyy"])
    T = ow3d.Tank(dict(cfg, mg_precision=mg), **bath)
    rng = np.random.default_rng(nx + ny + nz)
    r = rng.standard_normal(T.shape3)
    want = O.precond(r)
    got = T.precond_apply(r)
    T.precond_apply(rng.standard_normal(T.shape3))   # leaves other values in the compute units' LDS
    assert np.array_equal(T.precond_apply(r), got)
    assert np.max(np.abs(got - want)) <= TOL[mg] * np.max(np.abs(want))
    T.close()
    O.close()
