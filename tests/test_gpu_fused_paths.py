"""The fused paths beside the plain real-time step, against the FP64 oracle.

* Regions of a plane: several substeps of one pass (orders up to 4 fit one pass, 5 takes two) and the
  untransformed region's step as one pending factor, in both gauges.
* Imaginary time of planes and cubes (fused passes, normalisation and stop on the device): partial
  tiles, unequal sides, one and two substeps, with and without the kinetic energy, and a stop inside
  a run of steps.
* CoulombInteraction over both coordinates of a plane with unequal sides (a table factor in FP64).
* Real-time step boundaries in every form of the row pass, the mixed plan, large reads.

Bars as for the axis passes: psi 1e-10 FP64, 1e-4 FP32-mixed, 2e-6 FP32 state; records 1e-9 / 1e-4 /
1e-5 of each column's largest value (fluxes in FP64 only, where they are a difference of
neighbouring values of a rounded state).
"""
import numpy as np
import pytest

from oracle import oracle as O
from qsf_amd import qsf_types as T

pytestmark = pytest.mark.gpu

PSI_TOL = {T.FP64: 1e-10, T.FP32_MIXED: 1e-4, T.FP32_STATE: 2e-6}
REC_TOL = {T.FP64: 1e-9, T.FP32_MIXED: 1e-4, T.FP32_STATE: 1e-5}
GROUND = T.OUT_NORM | T.OUT_EPOT | T.OUT_EKIN | T.OUT_ETOT | T.OUT_EDIFF | T.OUT_NORMALIZE


@pytest.fixture(scope="module")
def ctx():
    from qsf_amd import hip
    c = hip.Context(0)
    yield c
    c.close()


def rel(a, b):
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300)


def state(shape, dx):
    """A smooth packet that reaches the edges."""
    psi = np.ones(())
    for k, n in enumerate(shape):
        x = -0.5 * dx * (n - 1) + dx * np.arange(n)
        f = np.exp(-np.abs(x - 0.2)) + 0.4 * np.exp(-(x / (0.3 * n * dx)) ** 2 + 0.2j * (k + 1) * x)
        psi = np.multiply.outer(psi, f)
    psi = psi.ravel()
    return psi / np.sqrt(np.sum(np.abs(psi) ** 2) * dx ** len(shape))


def both(ctx, shape, prec, pd, fields, takes, dx=0.3, **desc):
    from qsf_amd import hip
    out = []
    for mod, p in ((hip, prec), (O, T.FP64)):
        d = T.grid_desc(len(shape), list(shape), dx, precision=p, **desc)
        g = mod.GridSet(ctx, d) if mod is hip else mod.GridSet(d)
        psi = state(shape, dx)
        for r in range(len(g)):
            g[r].set_psi(psi if r == 0 else np.zeros_like(psi))
        prop = mod.Propagator(g, pd, fields)
        prop.start()
        for k in takes:
            if mod is hip and k > 1:
                prop.run_steps(k)
                continue
            for _ in range(k):
                if prop.should_continue():
                    prop.step()
        out.append(([g[r].psi() for r in range(len(g))], prop.records(), prop.step_count))
    return out


def check(got, want, prec):
    assert got[2] == want[2]
    for r, (a, b) in enumerate(zip(got[0], want[0])):
        assert rel(a, b) < PSI_TOL[prec], f"region {r}"
    a, b = got[1], want[1]
    assert a.shape == b.shape
    for c in range(a.shape[1] if prec == T.FP64 else T.REC_FLUX0):
        if np.isnan(b[:, c]).all():
            assert np.isnan(a[:, c]).all(), f"column {c}"
            continue
        assert np.abs(a[:, c] - b[:, c]).max() <= REC_TOL[prec] * max(np.abs(b[:, c]).max(), 1e-6), f"column {c}"


@pytest.mark.parametrize("prec", [T.FP64, T.FP32_MIXED])
@pytest.mark.parametrize("gauge", [T.GAUGE_VELOCITY, T.GAUGE_LENGTH])
@pytest.mark.parametrize("order", [1, 3, 4, 5])
def test_regions(ctx, order, gauge, prec):
    print(f"[case] regions order={order} gauge={gauge} prec={prec}", flush=True)
    pd = T.prop_desc(T.MODE_RE, order, 0.04, gauge=gauge, outputs=T.OUT_NORM | T.OUT_EPOT | T.OUT_FLUX,
                     borders=[(b, 0) for b in T.ZOA_FLUX_2D])
    got, want = both(ctx, (96, 96), prec, pd, [T.field_desc(T.AXIS_XY, 0.1, 0.3, 2)], (3, 1, 2), potential=T.POT_EBERLY,
                     Ncharge=2, Echarge=-1, Nsoft=0.5, Esoft=0.33, absorber=T.ABS_CAP, nCAP=12, multigrid=1)
    check(got, want, prec)


SHAPES = [(40, 40), (96, 48), (256, 256), (20, 20, 20), (64, 64, 64)]


@pytest.mark.parametrize("prec", [T.FP64, T.FP32_MIXED, T.FP32_STATE])
@pytest.mark.parametrize("shape", SHAPES, ids=["x".join(map(str, s)) for s in SHAPES])
def test_ground_state(ctx, shape, prec):
    print(f"[case] ground {shape} prec={prec}", flush=True)
    model = dict(potential=T.POT_EBERLY if len(shape) == 2 and shape[0] == shape[1] else
                 T.POT_ECKHARDT_SACHA if len(shape) == 3 else T.POT_NONE, Ncharge=2, Echarge=-1, Nsoft=0.5, Esoft=1.0)
    f = [T.field_desc([0, T.AXIS_X, T.AXIS_XY, T.AXIS_XYZ][len(shape)], 0.0, 0.3, 1)]
    for order, outputs in ((1, GROUND), (2, GROUND), (1, T.OUT_NORM | T.OUT_EPOT | T.OUT_NORMALIZE)):
        pd = T.prop_desc(T.MODE_IM, order, 0.05, max_steps=11, outputs=outputs)
        got, want = both(ctx, shape, prec, pd, f, (3, 1, 20), **model)
        assert want[2] == 11
        check(got, want, prec)


@pytest.mark.parametrize("shape", [(64, 64), (32, 32, 32)], ids=["plane", "cube"])
def test_ground_state_stops_inside_a_run(ctx, shape):
    f = [T.field_desc(T.AXIS_XYZ, 0.0, 0.3, 1)]
    model = dict(potential=T.POT_EBERLY, Ncharge=2, Echarge=-1, Nsoft=0.5, Esoft=1.0)
    free = both(ctx, shape, T.FP64, T.prop_desc(T.MODE_IM, 1, 0.05, max_steps=40, outputs=GROUND), f, (40,), **model)
    dif = np.abs(free[1][1][:, T.REC_EDIFF])
    acc = float(np.sqrt(dif[21] * dif[22]))   # between two steps' differences, far from either
    pd = T.prop_desc(T.MODE_IM, 1, 0.05, max_steps=200, state_accuracy=acc, outputs=GROUND)
    got, want = both(ctx, shape, T.FP64, pd, f, (200,), **model)
    assert 10 < want[2] < 40
    check(got, want, T.FP64)


@pytest.mark.parametrize("shape", [(40, 96), (128, 64)], ids=["40x96", "128x64"])
def test_coulomb_plane_with_unequal_sides(ctx, shape):
    f = [T.field_desc(T.AXIS_XY, 0.1, 0.3, 2)]
    for gauge, order in ((T.GAUGE_LENGTH, 1), (T.GAUGE_VELOCITY, 2)):
        pd = T.prop_desc(T.MODE_RE, order, 0.05, gauge=gauge, outputs=T.OUT_NORM | T.OUT_EPOT | T.OUT_EKIN | T.OUT_FLUX,
                         borders=[(T.BORDER_BOX, 12)])
        got, want = both(ctx, shape, T.FP64, pd, f, (4, 1, 3), potential=T.POT_COULOMB, Ncharge=1, Echarge=-1, Nsoft=0.7,
                         absorber=T.ABS_CAP, nCAP=6)
        check(got, want, T.FP64)


BOUNDARY_SHAPES = [(80, 80), (160, 160), (64, 64), (80, 80, 80), (64, 64, 64)]


@pytest.mark.parametrize("prec", [T.FP64, T.FP32_MIXED, T.FP32_STATE])
@pytest.mark.parametrize("gauge", [T.GAUGE_VELOCITY, T.GAUGE_LENGTH])
@pytest.mark.parametrize("shape", BOUNDARY_SHAPES, ids=["x".join(map(str, s)) for s in BOUNDARY_SHAPES])
def test_real_time_with_and_without_energies(ctx, shape, gauge, prec):
    """One and two interaction terms along the line, the two halves equal (velocity gauge) or sharing
    their interaction term (length gauge), the boundary state formed (energies) or not; lengths with
    eight elements a thread and with the mixed plan."""
    print(f"[case] boundary {shape} gauge={gauge} prec={prec}", flush=True)
    f = [T.field_desc([0, T.AXIS_X, T.AXIS_XY, T.AXIS_XYZ][len(shape)], 0.1, 0.3, 2)]
    for outputs in (T.OUT_NORM | T.OUT_FLUX, T.OUT_NORM | T.OUT_EPOT | T.OUT_EKIN | T.OUT_FLUX):
        pd = T.prop_desc(T.MODE_RE, 1, 0.04, gauge=gauge, outputs=outputs, borders=[(T.BORDER_BOX, 16)])
        got, want = both(ctx, shape, prec, pd, f, (3, 1), potential=T.POT_ECKHARDT_SACHA if len(shape) == 3 else T.POT_EBERLY,
                         Ncharge=2, Echarge=-1, Nsoft=0.5, Esoft=1.0, absorber=T.ABS_CAP, nCAP=8)
        check(got, want, prec)


MIXED_SHAPES = [(80, 20), (20, 80), (160, 48), (24, 320), (320, 12), (640, 40), (1280, 10), (16, 1280), (2560, 8), (8, 2560)]


@pytest.mark.parametrize("shape", MIXED_SHAPES, ids=["x".join(map(str, s)) for s in MIXED_SHAPES])
def test_mixed_plan_partial_tiles(ctx, shape):
    """The mixed plan of the 5*2^k lengths beside short axes: tiles with idle lines and columns."""
    print(f"[case] mixed {shape}", flush=True)
    f = [T.field_desc(T.AXIS_XY, 0.1, 0.3, 2)]
    pd = T.prop_desc(T.MODE_RE, 1, 0.04, gauge=T.GAUGE_LENGTH, outputs=T.OUT_NORM | T.OUT_EPOT | T.OUT_EKIN)
    for prec in (T.FP64, T.FP32_STATE):
        got, want = both(ctx, shape, prec, pd, f, (3, 1), potential=T.POT_COULOMB, Ncharge=1, Echarge=-1, Nsoft=0.7)
        check(got, want, prec)


@pytest.mark.parametrize("prec", [T.FP64, T.FP32_MIXED, T.FP32_STATE])
@pytest.mark.parametrize("shape", [(1024, 1024), (160, 160, 48), (2048, 1280)], ids=["least", "remainder", "ring"])
def test_large_states_come_whole(ctx, shape, prec):
    """States read through the pinned slots: whole chunks, a last part of one, more than the ring holds."""
    from qsf_amd import hip
    print(f"[case] download {shape} prec={prec}", flush=True)
    gs = hip.GridSet(ctx, T.grid_desc(len(shape), list(shape), 0.2, precision=prec))
    rng = np.random.default_rng(3)
    a = rng.normal(size=gs[0].m) + 1j * rng.normal(size=gs[0].m)
    gs[0].set_psi(a)
    want = a if prec == T.FP64 else a.astype(np.complex64).astype(np.complex128)
    for _ in range(2):
        assert np.array_equal(gs[0].psi(), want)
