"""Line runs (whole steps of a 1D propagation in one launch) against the FP64 oracle.

Lengths at the edges of the plans: single-thread lines (8, 12, 20), lines within a wave (48, 64,
320, 512), lines over several waves (768, 1280) and the longest of each family (2560, 3072, 4096).
Steps are taken as uneven run_steps calls and single steps, so runs begin and end at every kind of
boundary; a long run crosses the limit of one launch. Bars as for the axis passes: FP64 1e-10,
FP32-mixed 1e-4, FP32 state 2e-6; records 1e-9 / 1e-4 / 1e-5 of each column's largest value. Fluxes
are compared in FP64 only: a current is a difference of neighbouring values, so the rounding of an
FP32 state is a fraction of |psi|^2 at the border and not of the current (on any path).
"""
import numpy as np
import pytest

from oracle import oracle as O
from qsf_amd import qsf_types as T

pytestmark = pytest.mark.gpu

PSI_TOL = {T.FP64: 1e-10, T.FP32_MIXED: 1e-4, T.FP32_STATE: 2e-6}
REC_TOL = {T.FP64: 1e-9, T.FP32_MIXED: 1e-4, T.FP32_STATE: 1e-5}


@pytest.fixture(scope="module")
def ctx():
    from qsf_amd import hip
    c = hip.Context(0)
    yield c
    c.close()


def rel(a, b):
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300)


def packet(n, dx):
    x = -0.5 * dx * (n - 1) + dx * np.arange(n)
    w = 0.2 * n * dx
    psi = np.exp(-np.abs(x)) + 0.5 * np.exp(-(x / w) ** 2 + 0.3j * x)
    return psi / np.sqrt(np.sum(np.abs(psi) ** 2) * dx)


def both(ctx, n, prec, mode, order, gauge, outputs, borders, takes, max_steps=0, accuracy=0.0):
    from qsf_amd import hip
    dx = 0.1
    desc = [T.grid_desc(1, n, dx, precision=p, potential=T.POT_COULOMB, Ncharge=1, Echarge=-1, Nsoft=1.0,
                        absorber=T.ABS_COS18, nCAP=max(2, n // 10), absorber_tau=0.05) for p in (prec, T.FP64)]
    pd = T.prop_desc(mode, order, 0.05, gauge=gauge, outputs=outputs, borders=borders, max_steps=max_steps,
                     state_accuracy=accuracy)
    f = [T.field_desc(T.AXIS_X, 0.08 if mode == T.MODE_RE else 0.0, 0.3, 2)]
    out = []
    for mod, d in ((hip, desc[0]), (O, desc[1])):
        g = mod.GridSet(ctx, d) if mod is hip else mod.GridSet(d)
        g[0].set_psi(packet(n, dx))
        p = mod.Propagator(g, pd, f)
        p.start()
        for k in takes:
            if mod is hip and k > 1:
                p.run_steps(k)
                continue
            for _ in range(k):
                if p.should_continue():
                    p.step()
        out.append((g[0].psi(), p.records(), p.step_count))
    return out


def check(got, want, prec, n):
    assert got[2] == want[2], f"n={n} steps"
    assert rel(got[0], want[0]) < PSI_TOL[prec], f"n={n}"
    a, b = got[1], want[1]
    assert a.shape == b.shape
    for c in range(a.shape[1] if prec == T.FP64 else T.REC_FLUX0):
        if np.isnan(b[:, c]).all():
            assert np.isnan(a[:, c]).all(), f"n={n} column {c}"
            continue
        assert np.abs(a[:, c] - b[:, c]).max() <= REC_TOL[prec] * max(np.abs(b[:, c]).max(), 1e-6), f"n={n} column {c}"


@pytest.mark.parametrize("prec", [T.FP64, T.FP32_MIXED, T.FP32_STATE])
@pytest.mark.parametrize("n", [8, 12, 20, 48, 64, 320, 512, 768, 1280, 2560, 3072, 4096])
def test_line_pulse(ctx, n, prec):
    print(f"[case] line pulse n={n} prec={prec}", flush=True)
    box = max(2, n // 3)
    for gauge, order, outputs in ((T.GAUGE_LENGTH, 1, T.OUT_NORM | T.OUT_EPOT | T.OUT_EKIN | T.OUT_ETOT | T.OUT_FLUX),
                                  (T.GAUGE_VELOCITY, 2, T.OUT_NORM | T.OUT_FLUX),
                                  (T.GAUGE_LENGTH, 2, T.OUT_NORM | T.OUT_EPOT)):
        borders = [(T.BORDER_BOX, box), (T.BORDER_BOX, 1)] if outputs & T.OUT_FLUX else []
        got, want = both(ctx, n, prec, T.MODE_RE, order, gauge, outputs, borders, (3, 1, 5))
        check(got, want, prec, n)


@pytest.mark.parametrize("prec", [T.FP64, T.FP32_STATE])
@pytest.mark.parametrize("n", [20, 64, 768, 4096])
def test_line_ground_state(ctx, n, prec):
    print(f"[case] line ground n={n} prec={prec}", flush=True)
    out = T.OUT_NORM | T.OUT_EPOT | T.OUT_EKIN | T.OUT_ETOT | T.OUT_EDIFF | T.OUT_NORMALIZE
    got, want = both(ctx, n, prec, T.MODE_IM, 1, T.GAUGE_VELOCITY, out, [], (4, 1, 20), max_steps=17)
    assert want[2] == 17
    check(got, want, prec, n)


def test_line_ground_state_stops_inside_a_run(ctx):
    # the accuracy is met between two steps' differences (far from either), inside one launch
    out = T.OUT_NORM | T.OUT_EPOT | T.OUT_EKIN | T.OUT_ETOT | T.OUT_EDIFF | T.OUT_NORMALIZE
    free = both(ctx, 256, T.FP64, T.MODE_IM, 1, T.GAUGE_VELOCITY, out, [], (60,), max_steps=60)[1][1]
    dif = np.abs(free[:, T.REC_EDIFF])
    acc = float(np.sqrt(dif[40] * dif[41]))
    got, want = both(ctx, 256, T.FP64, T.MODE_IM, 1, T.GAUGE_VELOCITY, out, [], (10, 200), max_steps=400, accuracy=acc)
    assert 10 < want[2] < 60
    check(got, want, T.FP64, 256)


def test_line_run_longer_than_one_launch(ctx):
    got, want = both(ctx, 128, T.FP64, T.MODE_RE, 1, T.GAUGE_VELOCITY, T.OUT_NORM | T.OUT_FLUX, [(T.BORDER_BOX, 40)],
                     (300,))
    check(got, want, T.FP64, 128)


def test_line_and_member_calls_agree(ctx):
    # rows of line runs, then of member calls, in one record
    from qsf_amd import hip
    dx, n = 0.1, 512
    d = T.grid_desc(1, n, dx, potential=T.POT_COULOMB, Ncharge=1, Echarge=-1, Nsoft=1.0)
    pd = T.prop_desc(T.MODE_RE, 1, 0.05, gauge=T.GAUGE_VELOCITY, outputs=T.OUT_NORM | T.OUT_EPOT | T.OUT_FLUX,
                     borders=[(T.BORDER_BOX, 100)])
    f = [T.field_desc(T.AXIS_X, 0.08, 0.3, 2)]
    res = []
    for switch in (False, True):
        g = hip.GridSet(ctx, d)
        g[0].set_psi(packet(n, dx))
        p = hip.Propagator(g, pd, f)
        p.start()
        p.run_steps(4)
        if switch:
            ctx.check(hip.load().qsf_prop_set_exec(p.h, 1), "set_exec")
        p.run_steps(4)
        res.append((g[0].psi(), p.records(), p.flux_integral()))
        p.close()
        g.close()
    assert rel(res[1][0], res[0][0]) < 1e-12
    assert np.allclose(np.nan_to_num(res[1][1]), np.nan_to_num(res[0][1]), rtol=1e-11, atol=1e-14)
    assert np.allclose(res[1][2], res[0][2], rtol=1e-10)
