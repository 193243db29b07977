"""Mixed-form solves at radial resolutions without a compiled column length:
columns padded with identity rows to a multiple of 16, at the smallest and
largest N, at whole multiples of 16 and one row to either side, with partial
blocks of harmonics, against the plain form's LDS-column solves.

States after steps: both forms solve in FP64 and differ in the FP32 nonlinear
terms N, of which dt N enters the state.  dt |N| < |x| here, so the states differ
by less than one FP32 rounding, 2^-24 = 6e-8, a step; a wrong row of the predictor
shows at the order of its value.  The corrector's changes are smaller than that
bound in most fields: they are compared by themselves, on equal N."""
import numpy as np
import pytest

from lsd import make_config, seeded_state, MIXED_F32, PLAIN_F64
from lsd.gpu import Context
from lsd.initial import harmonics

pytestmark = pytest.mark.gpu


def run(cfg, state):
    g = Context(cfg)
    g.set_state(state)
    ev = g.step(2).evaluations
    out = [g.get_coll(k) for k in range(6)]
    v = g.variants()["solve"]
    g.close()
    return out, ev, v


SIZES = [7, 15, 16, 17, 31, 40, 49, 63, 79, 80, 81, 95, 97, 111, 112, 113, 127, 128]


@pytest.mark.parametrize("N", SIZES)
@pytest.mark.parametrize("kw", [{}, {"rot": 1, "Nic": 8, "vel_bc": 2}], ids=["shell", "inner core"])
def test_padded_columns(N, kw):
    N = max(N, kw.get("Nic", 0))  # an inner core has at most N rows
    def cfg(p):
        return make_config(L=40, M=36, N=N, comp=1, Ra_comp=2.0e4, dt=1e-7, precision=p, **kw)
    st = seeded_state(cfg(PLAIN_F64), 7, 1e-3)
    a, ea, va = run(cfg(MIXED_F32), st)
    b, eb, _ = run(cfg(PLAIN_F64), st)
    assert va == 2 and ea == eb
    for k in range(6):
        den = np.sqrt((b[k][0] ** 2).sum() + (b[k][1] ** 2).sum())
        num = np.sqrt(((a[k][0] - b[k][0]) ** 2).sum() + ((a[k][1] - b[k][1]) ** 2).sum())
        assert num <= 2 * 2.0 ** -24 * den, (k, num / den)


@pytest.mark.parametrize("N", SIZES)
@pytest.mark.parametrize("kw", [{}, {"rot": 1, "Nic": 8, "vel_bc": 2}], ids=["shell", "inner core"])
def test_padded_increments(N, kw):
    """The predictor's and the corrector's own changes of the state.  The phases
    transform in FP64 in both forms, so their N agree to about 1e-13, and the
    changes may differ by the solves' rounding alone: 1e-6 of the change (the
    operators' entries reach 1e5 times those of the change's smooth part) and a
    few roundings of the state that it is the difference of.  l = 0, whose
    conduction profile is most of C and xi, is compared by itself."""
    N = max(N, kw.get("Nic", 0))

    def phases(p):
        cfg = make_config(L=40, M=36, N=N, comp=1, Ra_comp=2.0e4, dt=1e-5, precision=p, **kw)
        g = Context(cfg)
        g.set_state(seeded_state(cfg, 7, 1e-1))
        states = []

        def keep():
            states.append([np.array(g.get_coll(k)) for k in range(6)])

        keep()
        g.transform()
        g.nonlinear()
        g.predictor()
        keep()
        for _ in range(2):
            g.transform()
            g.nonlinear()
            g.corrector()
            keep()
        v = g.variants()["solve"]
        g.close()
        return cfg, states, v

    cfg, a, va = phases(MIXED_F32)
    _, b, _ = phases(PLAIN_F64)
    assert va == 2
    l = harmonics(cfg.L, cfg.M, cfg.Mp)[0]
    for k in range(6):
        for name, part in (("l = 0", l == 0), ("l > 0", l > 0)):
            for s in range(1, 4):
                da = a[s][k][:, part] - a[s - 1][k][:, part]
                db = b[s][k][:, part] - b[s - 1][k][:, part]
                x = np.sqrt((b[s][k][:, part] ** 2).sum())
                d = np.sqrt((db ** 2).sum())
                err = np.sqrt(((da - db) ** 2).sum())
                assert err <= 1e-6 * d + 8 * 2.0 ** -53 * x, (k, name, s, err, d, x)
                # a change to compare, far above those roundings
                assert d >= 1e3 * 2.0 ** -53 * x or name == "l = 0", (k, s, d, x)
