"""Physical-space pass over phi lengths: the wave form at every length it is
instantiated for, at the largest M of the 3/2 rule and past it (workgroup
form), with theta counts that leave row pairs over, against the C oracle.

The nonlinear terms of one timestep are compared per field, relative to the
field's norm, at dt = 1e-4 (they are those of the predicted state, whose wall
values carry the solves' roundoff of about 1e-17 / dt).  Bounds: FP64 1e-11
(that of the other parity tests); FP32 5e-6,
from 6e-8 per operation through two Legendre sums and two transforms (about
25 roundings each on the longest path, growing with its square root) and the
factor 2-3 by which the products' terms exceed their sum."""
import numpy as np
import pytest

import oracle_lib
from lsd import make_config, seeded_state, MIXED_F32, PLAIN_F64
from lsd.gpu import Context

pytestmark = pytest.mark.gpu

SHORT = (36, 48, 54, 64, 72, 96, 108, 128, 144, 162, 192, 216, 256, 288, 324, 384, 432, 486, 512)
LONG = (576, 648, 768, 864, 972, 1024)


def compare(cfg, bound):
    st = seeded_state(cfg, 11, 1e-3)
    g = Context(cfg)
    o = oracle_lib.Oracle(cfg)
    g.set_state(st)
    o.set_state(st)
    assert g.step(1).evaluations == o.step(1).evaluations
    # an adaptive run starts at dt = 8e-11, where the solves' wall roundoff
    # (which grows as 1/dt) is all that N - N_oracle shows: only its CFL limit,
    # formed on the initial state, is compared
    for k in range(6, 12) if cfg.dt > 0 else ():
        a, b = g.get_coll(k), o.get_coll(k)
        den = np.sqrt((b[0] ** 2).sum() + (b[1] ** 2).sum())
        num = np.sqrt(((a[0] - b[0]) ** 2).sum() + ((a[1] - b[1]) ** 2).sum())
        assert num <= bound * den, (k, num / den)
    if cfg.dt < 0:
        c, d = g.get_dt()[1], o.get_dt()[1]
        assert abs(c - d) <= bound * abs(d), (c, d)
    g.close()


def config(Ph, M, precision, Th, **kw):
    # dterr: few theta points under-resolve the large L; one corrector is taken
    # as it comes
    base = dict(L=M, M=M, N=8, dterr=1e30, Th=Th, Ph=Ph, comp=1, dt=1e-4, precision=precision, Ra_comp=2.0e4)
    base.update(kw)
    return make_config(**base)


@pytest.mark.parametrize("Ph", SHORT)
@pytest.mark.parametrize("precision,bound", [(PLAIN_F64, 1e-11), (MIXED_F32, 5e-6)])
def test_lengths(Ph, precision, bound):
    M = Ph // 3 // 2 * 2
    # 3 and 11 row pairs: one partial workgroup, and whole ones with a rest
    # or a single partial one, by the row pairs a workgroup takes
    compare(config(Ph, M, precision, 6), bound)
    compare(config(Ph, M - 2, precision, 22, comp=0), bound)


@pytest.mark.parametrize("Ph", LONG)
def test_long_lengths(Ph):
    # (an even count of theta pairs: the analysis of odd ones ends at L = 256)
    compare(config(Ph, Ph // 3 // 2 * 2, MIXED_F32, 12), 5e-6)
    compare(config(Ph, 64, MIXED_F32, 6, mag=0), 5e-6)


@pytest.mark.parametrize("Ph,M", [(36, 14), (48, 20), (128, 48), (192, 80), (512, 180), (512, 220), (24, 8), (32, 10)])
@pytest.mark.parametrize("precision,bound", [(PLAIN_F64, 1e-11), (MIXED_F32, 5e-6)])
def test_workgroup_form(Ph, M, precision, bound):
    """M past the 3/2 rule, and lengths that the wave form does not take."""
    compare(config(Ph, M, precision, 10), bound)


@pytest.mark.parametrize("Ph", (48, 96, 162, 512))
@pytest.mark.parametrize("precision,bound", [(PLAIN_F64, 1e-11), (MIXED_F32, 5e-6)])
@pytest.mark.parametrize("mag", (0, 1))
def test_cfl(Ph, precision, bound, mag):
    compare(config(Ph, Ph // 3 // 2 * 2, precision, 14, dt=-1e-6, mag=mag), bound)
