"""PPM sweeps that share slopes and edges between neighbours: along x between
the lanes of a wave (61 interfaces a wave, rows of nx + 4 cells end to end),
along y and z from one cell of a march to the next.  Rows shorter and longer
than a wave, rows that end at its first and last whole lanes, one-cell axes."""
import numpy as np
import pytest

from cumc3d_amd import ic
from cumc3d_amd.config import Config
from cumc3d_amd.solver import make_solver
from oracle import oracle as O
from test_gpu_selector import forcing_params

FIELDS = ("rho", "vx", "vy", "vz", "p", "bx", "by", "bz", "eps", "bcx", "bcy", "bcz")
SIZES = [(3, 3, 3), (57, 5, 4), (58, 5, 4), (59, 7, 3), (61, 4, 5), (62, 3, 7), (121, 5, 3), (5, 66, 4), (4, 5, 67),
         (127, 6, 1), (245, 1, 1)]


def setup(size, precision, riemann="hlld"):
    nx, ny, nz = size
    dim = 1 if ny == 1 else (2 if nz == 1 else 3)
    flags = (0, 0, 1, 1, 2, 2) if dim == 3 else (0, 0, 0, 0, 0, 0)
    cfg = Config(nx=nx, ny=ny, nz=nz, n_dim=dim, cfl=0.3, boundary_flag=flags, riemann=riemann, recon="ppm",
                 precision=precision)
    return cfg, ic.orszag_tang(cfg)


@pytest.mark.gpu
@pytest.mark.parametrize("riemann", ["hlld", "hll"])
@pytest.mark.parametrize("size", SIZES)
def test_fp64_matches_oracle(size, riemann):
    cfg, st = setup(size, "fp64", riemann)
    s, o = make_solver(cfg, st), O.Oracle(cfg, st)
    assert np.array_equal(s.run(3), o.run(3))
    got = s.state()
    for f in FIELDS:
        a, b = got[f][2:-2, 2:-2, 2:-2], o.get(f)[2:-2, 2:-2, 2:-2]
        assert np.array_equal(a, b, equal_nan=True), f"{f}: {np.count_nonzero(a != b)} differ"


@pytest.mark.gpu
@pytest.mark.parametrize("size", [s for s in SIZES if s[2] > 1])
def test_fp32_matches_cellwise_ppm(size):
    """The selector's sweep takes each cell's faces from its whole stencil; with
    every cell of class PPM it computes the same values in the same precision.
    Three steps of a few rounding errors (6e-8) each: 1e-5 of the largest."""
    cfg, st = setup(size, "fp32")
    plain, sel = make_solver(cfg, st, hlld_bn_mode="field"), make_solver(cfg, st, hlld_bn_mode="field")
    sel.selector_init(capacity=1024)
    sel.selector_params(forcing_params(1))
    sel.selector_enable(True)
    assert np.allclose(plain.run(3), sel.run(3), rtol=1e-5, atol=0)
    a, b = plain.state(), sel.state()
    for group in (("rho",), ("p",), ("eps",), ("vx", "vy", "vz"), ("bx", "by", "bz")):
        scale = max(np.max(np.abs(b[f][3:-3, 3:-3, 3:-3])) for f in group)
        for f in group:
            assert np.max(np.abs(a[f] - b[f])[3:-3, 3:-3, 3:-3]) <= 1e-5 * scale, f
