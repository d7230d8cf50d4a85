"""1D and 2D runs: the stages of a whole step leave the outer ghost layers of the
axes without a sweep to its last stage.  Every ghosted array after whole steps
has the bits it has after the same steps stage by stage, where each stage fills
every layer, and steps past the end of a run change nothing."""
import numpy as np
import pytest

from cumc3d_amd import ic
from cumc3d_amd.config import Config
from cumc3d_amd.solver import make_solver

CASES = [((70, 1, 1), (1, 1, 0, 0, 0, 0)), ((33, 20, 1), (0, 0, 0, 0, 0, 0)), ((20, 33, 1), (1, 1, 0, 0, 1, 1))]


def solver(size, flags, precision):
    cfg = Config(nx=size[0], ny=size[1], nz=size[2], n_dim=1 if size[1] == 1 else 2, cfl=0.3, boundary_flag=flags,
                 riemann="hlld", recon="ppm", precision=precision)
    return make_solver(cfg, ic.orszag_tang(cfg), hlld_bn_mode="field" if precision == "fp32" else "carry")


def same(a, b):
    for f in a:
        assert np.array_equal(a[f], b[f], equal_nan=True), f"{f}: {np.count_nonzero(a[f] != b[f])} differ"


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("size,flags", CASES)
def test_whole_steps_equal_stages(size, flags, precision):
    s, o, r = (solver(size, flags, precision) for _ in range(3))
    dts = []
    for _ in range(2):
        dts.append(s.finddt())
        s.rungekutta(dts[-1])
        assert o.finddt() == dts[-1]
        for k in (1, 2, 3):
            o.stage(k, dts[-1])
    same(s.state(), o.state())
    assert np.array_equal(r.run(2), dts)
    same(r.state(), o.state())
    # whole steps, then a stage
    dt = s.finddt()
    assert dt == o.finddt()
    s.stage(1, dt)
    o.stage(1, dt)
    same(s.state(), o.state())


@pytest.mark.gpu
@pytest.mark.parametrize("size,flags", CASES)
def test_steps_past_the_end_keep_every_layer(size, flags):
    s, o = solver(size, flags, "fp64"), solver(size, flags, "fp64")
    o.run(3)
    s.run(8, total_time=o.t, sync_each_step=False)
    assert s.t == o.t
    same(s.state(), o.state())
