"""ow3d_laplace_apply_device promises to take a result buffer of any 8-byte alignment: the same bits as the host entry point at
an address that is not 16-byte aligned, and nothing written beside it."""
import numpy as np
import pytest
import torch

import ow3d
from ow3d import problems


@pytest.mark.gpu
@pytest.mark.parametrize("nx,ny,nz,half", [
    (33, 17, 9, 3), (33, 17, 8, 3),     # even (results stored in pairs) and odd column depth
    (18, 40, 13, 4), (47, 23, 5, 1),
    (65, 1, 9, 3),                      # x-z
])
def test_result_at_any_8_byte_alignment(nx, ny, nz, half):
    lx, ly = 2 * np.pi * (nx - 1) / 24, 2 * np.pi * (ny - 1) / 24 if ny > 1 else 1.0
    T = ow3d.Tank(dict(nx=nx, ny=ny, nz=nz, lx=lx, ly=ly, alpha=half, beta=half, gamma=half, precond=0),
                  **problems.gaussian_shoal(nx, ny, lx, ly))
    rng = np.random.default_rng(nx + ny)
    T.set_surface(0.02 * rng.standard_normal(T.shape2), np.zeros(T.shape2))
    phi = rng.standard_normal(T.shape3)
    d_phi = torch.from_numpy(phi).cuda()
    for variant in (0, 1, 2, 3) if ny > 1 else (0,):
        T.tune(variant, 0)
        want = T.laplace_apply(phi).ravel()
        for off in (0, 1, 2, 3):
            buf = torch.full((T.n + 8,), 7.5, dtype=torch.float64, device="cuda")
            assert buf.data_ptr() % 16 == 0
            torch.cuda.synchronize()
            T.laplace_apply_device(d_phi.data_ptr(), buf.data_ptr() + 8 * off)
            torch.cuda.synchronize()   # (the whole device: the matvec ran on the handle's stream)
            got = buf.cpu().numpy()
            assert (got[off:off + T.n] == want).all()
            assert (got[:off] == 7.5).all() and (got[off + T.n:] == 7.5).all()
    T.close()
