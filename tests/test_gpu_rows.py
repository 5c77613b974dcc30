"""Record rows reduced for several boundaries together against rows reduced one at a time.

Steps taken by one run_steps call leave their sums and flux stencils in slots (at most 32 at a time)
that one set of launches reduces; steps taken one by one are reduced by the single-boundary kernels.
Both sum in the same order, so states, rows and flux integrals have the same bits. Grids: a plane
whose run fills the slots more than twice, a cube whose boundary needs the second reduction level
(8192 blocks and more), lengths with partial tiles, and a set of regions.
"""
import numpy as np
import pytest

from qsf_amd import qsf_types as T

pytestmark = pytest.mark.gpu

CASES = [
    ("plane 96", 2, 96, 70, T.FP64, T.GAUGE_VELOCITY, 1, 0, 0),
    ("plane 160 FP32", 2, 160, 34, T.FP32_MIXED, T.GAUGE_LENGTH, 2, 30, 0),
    ("cube 128", 3, 128, 5, T.FP64, T.GAUGE_LENGTH, 1, 40, 0),
    ("cube 24 FP32 state", 3, 24, 40, T.FP32_STATE, T.GAUGE_VELOCITY, 2, 8, 0),
    ("regions 128", 2, 128, 35, T.FP64, T.GAUGE_VELOCITY, 2, 0, 1),
]


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_rows_together_and_one_at_a_time(case):
    from qsf_amd import hip
    name, dim, n, steps, prec, gauge, order, box, multi = case
    print(f"[case] rows {name}", flush=True)
    borders = [(T.BORDER_BOX, box)] if box else [(b, 0) for b in T.ZOA_FLUX_2D]
    d = T.grid_desc(dim, n, 0.3, precision=prec, potential=T.POT_EBERLY, Ncharge=2, Echarge=-1, Nsoft=0.5, Esoft=0.33,
                    absorber=T.ABS_CAP, nCAP=8, multigrid=multi)
    pd = T.prop_desc(T.MODE_RE, order, 0.02, gauge=gauge, outputs=T.OUT_NORM | T.OUT_EPOT | T.OUT_EKIN | T.OUT_FLUX,
                     borders=borders)
    f = [T.field_desc([0, T.AXIS_X, T.AXIS_XY, T.AXIS_XYZ][dim], 0.1, 0.3, 2)]
    rng = np.random.default_rng(7)
    psi = (rng.normal(size=n ** dim) + 1j * rng.normal(size=n ** dim)) * 0.01
    ctx = hip.Context(0)
    got = []
    for together in (True, False):
        g = hip.GridSet(ctx, d)
        g[0].set_psi(psi)
        p = hip.Propagator(g, pd, f)
        p.start()
        if together:
            p.run_steps(steps)
        else:
            for _ in range(steps):
                p.step()
        got.append((p.records(), p.flux_integral(), [x.psi() for x in g.grids]))
        p.close()
        g.close()
    ctx.close()
    assert np.array_equal(got[0][0], got[1][0], equal_nan=True)
    assert got[0][0].shape[0] == steps + 1
    assert np.array_equal(got[0][1], got[1][1])
    for a, b in zip(got[0][2], got[1][2]):
        assert np.array_equal(a, b)
