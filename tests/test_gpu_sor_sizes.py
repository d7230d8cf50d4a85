"""The Poisson solve on grids whose sides are not multiples of the SOR kernels'
blocks (256 slots of a colour, planes taken in pairs l, l + 2): every sweep
bit for bit the oracle's, with the sweeps cut off at relax_max, where the
reference leaves the potential as it is."""
import numpy as np
import pytest

from cumc3d_amd import ic
from cumc3d_amd.config import collapsar
from cumc3d_amd.solver import make_solver
from oracle import oracle as O


@pytest.mark.gpu
@pytest.mark.parametrize("nr,nth,nphi", [(16, 8, 1), (33, 17, 1), (21, 13, 2), (20, 9, 3), (19, 12, 5), (40, 30, 6),
                                         (17, 31, 7)])
def test_sor_sizes_bit_exact(nr, nth, nphi):
    cfg = collapsar(nr, nth, nphi, n_dim=2 if nphi == 1 else 3).with_(relax_max=37)
    if nphi in (2,):                                     # periodic needs three cells on an active axis
        cfg = cfg.with_(boundary_flag=(1, 1, 3, 3, 1, 1))
    st = ic.collapsar(cfg)
    s, o = make_solver(cfg, st), O.Oracle(cfg, st)
    assert np.array_equal(s.run(1), o.run(1))
    got, want = s.gravity(), o.gravity()
    box = (slice(2, cfg.nz + 4), slice(2, cfg.ny + 4), slice(2, cfg.nx + 4))
    assert got["iterations"] == want["iterations"] and got["m_bh"] == want["m_bh"]
    assert np.array_equal(got["phi"][box], want["phi"][box], equal_nan=True)
