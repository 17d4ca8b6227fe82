"""ow3d_estimate_bytes follows the switches that ow3d_create reads (OW3D_MG_BOTTOM, OW3D_MG_FUSED_RB) and counts the buffers of
the one-workgroup kernel."""
import os

import pytest

import ow3d
from ow3d import problems

SWITCHES = [("OW3D_MG_BOTTOM", "0"), ("OW3D_MG_BOTTOM", "400"), ("OW3D_MG_FUSED_RB", "0")]


def _with(env, f):
    if env:
        os.environ[env[0]] = env[1]
    try:
        return f()
    finally:
        if env:
            del os.environ[env[0]]


def test_unfused_sweeps_need_the_finest_right_hand_side():
    # two levels, no one-workgroup kernel: fused FP64 sweeps read the residual itself as the finest right-hand side
    cfg = dict(nx=33, ny=33, nz=9, mg_maxgrids=2, mg_precision=0)
    plain, unfused = (_with(e, lambda: ow3d.estimate_bytes(cfg)) for e in (None, SWITCHES[2]))
    assert unfused - plain == 8 * 35 * 35 * 10


@pytest.mark.parametrize("mg", [0, 1])
def test_launches_for_every_level_need_their_residuals(mg):
    # x-z: every level below the finest is in the one-workgroup kernel and keeps no residual in HBM
    cfg = dict(nx=129, ny=1, nz=9, mg_precision=mg)
    plain, launches = (_with(e, lambda: ow3d.estimate_bytes(cfg)) for e in (None, SWITCHES[0]))
    assert plain != launches


@pytest.mark.gpu
@pytest.mark.parametrize("mg", [0, 1, 2])
@pytest.mark.parametrize("nx,ny,nz", [(129, 1, 9), (33, 33, 9), (97, 161, 8)])   # the last with a dense solve of its own
def test_estimate_changes_with_the_allocation(nx, ny, nz, mg):
    bath = problems.gaussian_shoal(nx, ny, 5.0, 5.0)
    cfg = dict(nx=nx, ny=ny, nz=nz, lx=5.0, ly=5.0, mg_precision=mg)
    got, est, levels = [], [], 0
    for env in [None] + SWITCHES:
        T = _with(env, lambda: ow3d.Tank(cfg, **bath))
        got.append(T.device_bytes())
        est.append(_with(env, lambda: ow3d.estimate_bytes(cfg)))
        levels = T.mg_levels
        T.close()
    # everything but the switched buffers cancels; the tables' size is a bound, 16 values a level above it at most in x-z
    for g, e in zip(got[1:], est[1:]):
        assert abs((e - est[0]) - (g - got[0])) <= 128 * levels
