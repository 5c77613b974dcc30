"""The work this library is used for, as cases that can be timed and checked.

A case is one stretch of a propagation on the device: a program holds a grid set with its start
state, makes a propagator for a pulse (or for imaginary time), runs a number of steps and takes the
state of every region, the record rows and the flux time integrals back to the host. Batches are
whole: made, run over their pulse and read. States and outputs are in the grid's own type (complex64
and float32 for the grids whose state is FP32).
"""
import math

import numpy as np
import torch

from qsf_amd import hip
from qsf_amd import qsf_types as T

PRECISION = {"fp64": T.FP64, "fp32": T.FP32_MIXED, "fp32_state": T.FP32_STATE}
POTENTIAL = {"coulomb": T.POT_COULOMB, "eberly": T.POT_EBERLY, "eckhardt": T.POT_ECKHARDT_SACHA}
AXES = {1: T.AXIS_X, 2: T.AXIS_XY, 3: T.AXIS_XYZ}
ENERGIES = T.OUT_NORM | T.OUT_EPOT | T.OUT_EKIN | T.OUT_ETOT


# ------------------------------------------------------------------------------------- the cases
def _pulse(name, dim, n, steps, precision="fp64", potential="eberly", gauge="velocity", order=1, dt=0.05,
           energies=False, box=0, regions=False):
    """Real time: norm and fluxes at every step (through a box of half side `box` nodes, or the
    seven 2D ionisation families where `box` is 0)."""
    return dict(name=name, kind="pulse", dim=dim, n=n, steps=steps, precision=precision, potential=potential,
                gauge=gauge, order=order, dt=dt, energies=energies, box=box, regions=regions)


def _ground(name, dim, n, steps, precision="fp64", potential="eberly", dt=0.05):
    """Imaginary time: normalised at every step, with all energies and their difference."""
    return dict(name=name, kind="ground", dim=dim, n=n, steps=steps, precision=precision, potential=potential,
                dt=dt)


def _batch(name, sides, precision="fp32", dt=0.02, omega=1.2):
    """Uneven 2D solves advanced together over a one-cycle pulse each."""
    return dict(name=name, kind="batch", sides=sides, precision=precision, dt=dt, omega=omega)


def listed():
    return [
        # one electron on a line under an 800 nm pulse, energies and the flux through |x| = 150 at
        # every step: the smallest ordinary solve, most of a served stream
        _pulse("line_4096", 1, 4096, 1000, potential="coulomb", gauge="length", energies=True, box=1500),
        # the same kind of solve as a server runs it, in FP32 and on a length that is no power of two
        _pulse("line_1536_fp32", 1, 1536, 1000, precision="fp32", potential="coulomb", box=600),
        # its ground state by imaginary time: the stage before every pulse
        _ground("line_2560_ground", 1, 2560, 300, potential="coulomb"),
        # a small two-electron plane, where a step is a few short launches
        _pulse("plane_256", 2, 256, 1000, dt=0.02),
        # the ground state of an ordinary plane
        _ground("plane_768_ground", 2, 768, 150),
        # one electron in a plane: the Coulomb factor does not separate into axes
        _pulse("plane_640_coulomb", 2, 640, 400, potential="coulomb", box=200),
        # the two-electron workload with its ionisation regions, second-order splitting
        _pulse("regions_2048", 2, 2048, 250, order=2, dt=0.02, regions=True),
        # the same on a smaller plane in FP32
        _pulse("regions_1024_fp32", 2, 1024, 100, precision="fp32", order=2, dt=0.02, regions=True),
        # three electrons, length gauge: the largest single solve
        _pulse("cube_512", 3, 512, 150, potential="eckhardt", gauge="length", box=224),
        # the cube that is served, in FP32
        _pulse("cube_256_fp32", 3, 256, 500, precision="fp32", potential="eckhardt", gauge="length", box=100),
        # an FP32 state under FP64 arithmetic, velocity gauge, with energies
        _pulse("cube_320_state", 3, 320, 150, precision="fp32_state", potential="eckhardt", energies=True, box=120),
        # an intensity scan: uneven planes as one batch, replayed as a graph
        _batch("batch_12_fp32", "512,768,1024,512,1536,1024,768,512,1024,1536,768,512"),
    ]


LINES = [512, 640, 768, 1024, 1280, 1536, 2048, 2560, 3072, 4096]
PLANES = [128, 160, 192, 256, 320, 384, 512, 640, 768, 1024, 1280, 1536, 2048]
CUBES = [64, 80, 96, 128, 160, 192, 256, 320, 384]


def _log_pick(rng, sizes):
    """One of `sizes`, evenly over the logarithm of the range."""
    at = math.exp(rng.uniform(math.log(sizes[0] * 0.9), math.log(sizes[-1] * 1.1)))
    return min(sizes, key=lambda s: abs(math.log(s / at)))


def draw(rng):
    kind = rng.choice(["line", "line", "plane", "plane", "plane_ground", "coulomb", "regions", "cube", "cube", "batch"])
    any_precision = rng.choice(["fp64", "fp64", "fp32", "fp32_state"])
    gauge = rng.choice(["velocity", "length"])
    if kind == "line":
        n, steps = _log_pick(rng, LINES), rng.randint(200, 1200)
        if rng.random() < 0.3:
            c = _ground("", 1, n, steps // 4, precision=any_precision, potential="coulomb")
        else:
            c = _pulse("", 1, n, steps, precision=any_precision, potential="coulomb", gauge=gauge,
                       energies=rng.random() < 0.5, box=n // 2 - n // 8)
    elif kind == "batch":
        sides = [_log_pick(rng, PLANES[3:11]) for _ in range(rng.randint(4, 8))]
        c = _batch("", ",".join(map(str, sides)), precision=any_precision, omega=rng.uniform(1.0, 2.0))
    else:
        n = _log_pick(rng, CUBES if kind == "cube" else PLANES[3:] if kind == "regions" else PLANES)
        dim = 3 if kind == "cube" else 2
        steps = max(20, min(1000, int(rng.uniform(0.5, 1.0) * 8e8 / n ** dim)))
        if kind == "plane_ground":
            c = _ground("", 2, n, max(10, steps // 4), precision=any_precision)
        elif kind == "coulomb":
            c = _pulse("", 2, n, steps // 2, precision=any_precision, potential="coulomb", gauge=gauge, box=n // 3)
        elif kind == "regions":
            c = _pulse("", 2, n, min(100, steps // 4), precision=rng.choice(["fp64", "fp32"]), order=rng.choice([1, 2]),
                       dt=0.02, regions=True)
        elif kind == "cube":
            c = _pulse("", 3, n, steps, precision=any_precision, potential=rng.choice(["eckhardt", "eberly"]),
                       gauge=gauge, order=rng.choice([1, 1, 2]), energies=rng.random() < 0.3, box=n // 2 - n // 8)
        else:
            c = _pulse("", 2, n, steps, precision=any_precision, gauge=gauge, order=rng.choice([1, 2]), dt=0.02,
                       energies=rng.random() < 0.3, box=0 if n >= 128 and gauge == "velocity" else n // 3)
    del c["name"]
    return c


# ------------------------------------------------------------------------- what a program has in hand
def _dx(dim):
    return {1: 0.1, 2: 0.2, 3: 0.3}[dim]


def _ncap(dim, n):
    return max(8, n // 16) if dim == 3 else int(round(0.1 * n))


def _grid(dim, n, precision, potential, dt, regions=False):
    two = dict(Ncharge=2, Nsoft=0.5, Esoft=0.33) if dim == 2 else dict(Ncharge=1 if dim == 1 else 3, Nsoft=1.0, Esoft=1.0)
    return T.grid_desc(dim, n, _dx(dim), precision=PRECISION[precision], potential=POTENTIAL[potential], Echarge=-1,
                       absorber=T.ABS_CAP if dim == 3 else T.ABS_COS18, nCAP=_ncap(dim, n), absorber_tau=dt,
                       multigrid=int(regions), **two)


def _borders(dim, box):
    return [(T.BORDER_BOX, box)] if box or dim != 2 else [(b, 0) for b in T.ZOA_FLUX_2D]


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _start_state(dim, n, seed, ionised=True):
    """A state in the middle of a pulse: two bound-like packets (products of displaced and kicked
    orbitals) and, where `ionised`, a broad packet that reaches the borders and the absorbers; unit
    norm. Axes are torch vectors, the products are formed on the device."""
    rng = np.random.default_rng([seed, dim, n])
    dx = _dx(dim)
    x = torch.from_numpy(-0.5 * dx * (n - 1) + dx * np.arange(n)).to(_device())
    psi = None
    for weight in (1.0, 0.4, 2.5 if ionised else 0.0):
        term = None
        for _ in range(dim):
            x0, soft, k = rng.uniform(-1.5, 1.5), rng.uniform(0.3, 2.0), rng.uniform(-0.4, 0.4)
            f = torch.exp(-torch.sqrt((x - x0) ** 2 + soft)) if weight in (1.0, 0.4) else \
                torch.exp(-0.5 * ((x - 10 * x0) / (0.35 * n * dx)) ** 2)
            f = f * torch.exp(1j * k * x)
            f = f / torch.linalg.vector_norm(f)
            term = f if term is None else term.unsqueeze(-1) * f
        psi = weight * term if psi is None else psi.add_(weight * term)
    psi /= torch.sqrt(torch.sum(torch.view_as_real(psi) ** 2) * dx ** dim)
    return psi


def _fields(case, seed):
    rng = np.random.default_rng([seed, 77])
    strength, phase = float(rng.uniform(0.05, 0.12)), float(rng.uniform(0.0, 0.5))
    if case["kind"] == "ground":
        return [T.field_desc(AXES[case["dim"]], 0.0, 0.057, 1)]
    return [T.field_desc(AXES[case["dim"]], strength, 0.057, 4, phase_in_pi=phase)]


def _batch_members(case, seed):
    rng = np.random.default_rng([seed, 78])
    sides = [int(s) for s in case["sides"].split(",")]
    fields = [T.field_desc(T.AXIS_XY, float(rng.uniform(0.05, 0.15)), case["omega"], 1,
                           phase_in_pi=float(rng.uniform(0, 2))) for _ in sides]
    return sides, fields


def _prop(case):
    if case["kind"] == "ground":
        return T.prop_desc(T.MODE_IM, 1, case["dt"], max_steps=case["steps"] + 2, state_accuracy=0.0,
                           outputs=ENERGIES | T.OUT_NORMALIZE | T.OUT_EDIFF)
    if case["kind"] == "batch":
        return T.prop_desc(T.MODE_RE, 1, case["dt"], gauge=T.GAUGE_VELOCITY, outputs=T.OUT_NORM | T.OUT_FLUX,
                           borders=_borders(2, 0))
    gauge = T.GAUGE_LENGTH if case["gauge"] == "length" else T.GAUGE_VELOCITY
    return T.prop_desc(T.MODE_RE, case["order"], case["dt"], gauge=gauge,
                       outputs=T.OUT_FLUX | (ENERGIES if case["energies"] else T.OUT_NORM),
                       borders=_borders(case["dim"], case["box"]))


class _State:
    def __init__(self):
        self.ctx = hip.Context(0)

    def __del__(self):
        self.ctx.close()


def prepare(case, seed):
    s = _State()
    s.case, s.pd = case, _prop(case)
    s.single = case["precision"] != "fp64"
    if case["kind"] == "batch":
        # the descriptors, start states and tuned kernels; the batch itself belongs to one run
        sides, s.fields = _batch_members(case, seed)
        s.descs = [_grid(2, n, case["precision"], "eberly", case["dt"]) for n in sides]
        packets = {n: _start_state(2, n, seed).cpu().numpy().ravel() for n in set(sides)}
        s.psi = [packets[n] for n in sides]
        for n in sorted(set(sides)):
            gs = hip.GridSet(s.ctx, _grid(2, n, case["precision"], "eberly", case["dt"]))
            gs[0].set_psi(packets[n])
            gs[0].autotune(5)
            gs.close()
        return s
    s.fields = _fields(case, seed)
    s.gs = hip.GridSet(s.ctx, _grid(case["dim"], case["n"], case["precision"], case["potential"], case["dt"],
                                    case.get("regions", False)))
    s.guess = _start_state(case["dim"], case["n"], seed, case["kind"] == "pulse").cpu().numpy()
    s.gs[0].set_psi(s.guess)
    if case["kind"] != "ground":
        s.guess = None   # a pulse goes on from the state on the device
    for g in s.gs.grids:
        g.autotune(5)
    if s.pd.nborders:   # the border plan of the grid, made once
        s.gs[0].flux(_borders(case["dim"], case["box"]))
    s.ctx.synchronize()
    return s


def _own(s, a):
    """An output in the grid's own type."""
    if not s.single:
        return a
    return a.astype(np.complex64 if a.dtype == np.complex128 else np.float32)


def run(s):
    if s.case["kind"] == "batch":
        b = hip.Batch(s.ctx, s.descs, s.fields, s.pd)
        for k, psi in enumerate(s.psi):
            b.set_psi(k, psi)
        b.run_all(use_graph=True)
        out = {"psi": [_own(s, b.psi(k)) for k in range(b.n)], "records": [_own(s, b.records(k)) for k in range(b.n)],
               "flux_integral": [_own(s, b.flux_integral(k)) for k in range(b.n)]}
        b.close()
        return out
    if s.guess is not None:   # imaginary time begins at its guess again
        s.gs[0].set_psi(s.guess)
    p = hip.Propagator(s.gs, s.pd, s.fields)
    p.start()
    p.run_steps(s.case["steps"])
    out = {"records": _own(s, p.records()), "psi": [_own(s, g.psi()) for g in s.gs.grids]}
    if s.pd.nborders:
        out["flux_integral"] = _own(s, p.flux_integral())
    p.close()
    return out


def _batch_total(case):
    return int(2 * math.pi / case["omega"] / case["dt"] + 1) + 2


def work(case):
    """Each step reads and writes the state once (a line stays on the chip: it is read and written
    once a pass); the transforms of each substep and the phase products."""
    if case["kind"] == "batch":
        points, steps, dim = sum(int(n) ** 2 for n in case["sides"].split(",")), _batch_total(case), 2
        log2m = math.log2(points / len(case["sides"].split(",")))
        sub = 1
    else:
        dim, steps = case["dim"], case["steps"]
        points = case["n"] ** dim
        log2m, sub = math.log2(points), case.get("order", 1)
        points *= 4 if case.get("regions") else 1
    width = 16 if case["precision"] == "fp64" else 8
    sweeps = 1 if dim == 1 else steps
    return {"bytes": 2.0 * width * points * sweeps, "flops": points * float(steps) * sub * (10.0 * log2m + 24.0)}


# --------------------------------------------------------------- the same propagation in 64 bits
def _field_at(f, t):
    """The carrier times its sin^2 envelope, zero outside the pulse."""
    if t > 2 * math.pi * f.ncycles / f.omega or t < 0:
        return 0.0
    return f.field * math.sin(f.omega * t + f.phase_in_pi * math.pi) * math.sin(f.omega / (2 * f.ncycles) * t) ** 2


class _Vector:
    """A(t) as the running right-hand sum over the times at which the coupling is evaluated."""

    def __init__(self, field):
        self.field, self.a, self.last = field, 0.0, 0.0

    def at(self, t):
        self.a += (self.last - t) * _field_at(self.field, t)
        self.last = t
        return self.a


def _border_points(dim, n, borders):
    """Linear indices of the border points and their unit vectors per family."""
    half = n // 2

    def in2(i, lo, hi):
        return ((i >= lo) & (i < hi)) | ((i >= -hi) & (i < -lo))

    def pt2(i, at):
        return np.where((i == at - 1) | (i == -at), np.sign(i), 0).astype(float)

    def seg(i, j, at, lo, hi):
        return np.where((i >= lo) & (i < hi) & (j == at - 1), np.sign(j), 0).astype(float)

    def seg22(i, j, at, lo, hi):
        return np.where(in2(i, lo, hi), pt2(j, at), 0.0)

    def duo(i, j, at, lo, hi):
        return [seg22(j, i, at, lo, hi), seg22(i, j, at, lo, hi)]

    ns, sd, cap = 25, 14, 40   # the node distances of the ionisation regions

    def family(kind, size, ix):
        if kind == T.BORDER_BOX:
            if dim == 1:
                return [pt2(ix[0], size)]
            if dim == 2:
                return duo(ix[0], ix[1], size, 0, size)
            return [np.where(in2(ix[(a + 1) % 3], 0, size) & in2(ix[(a + 2) % 3], 0, size), pt2(ix[a], size), 0.0)
                    for a in range(3)]
        i, j = ix
        return {
            T.BORDER_N2S: lambda: duo(i, j, ns, 0, sd),
            T.BORDER_S2CAP: lambda: duo(i, j, cap, 0, sd),
            T.BORDER_D2CAP: lambda: duo(i, j, cap, sd, cap),
            T.BORDER_N2D_SYM: lambda: [seg(j + 1, i, sd, sd, ns + 1) - seg(-j, -i - 1, sd, sd, ns + 1),
                                       seg(i + 1, j, sd, sd, ns + 1) - seg(-i, -j - 1, sd, sd, ns + 1)],
            T.BORDER_N2D_ASYM: lambda: [-seg(j + 1, -i - 1, sd, sd, ns + 1) + seg(-j, i, sd, sd, ns + 1),
                                        -seg(i + 1, -j - 1, sd, sd, ns + 1) + seg(-i, j, sd, sd, ns + 1)],
            T.BORDER_S2D_SYM: lambda: [seg(j, i, sd, ns, cap) - seg(-j - 1, -i - 1, sd, ns, cap),
                                       seg(i, j, sd, ns, cap) - seg(-i - 1, -j - 1, sd, ns, cap)],
            T.BORDER_S2D_ASYM: lambda: [-seg(j, -i - 1, sd, ns, cap) + seg(-j - 1, i, sd, ns, cap),
                                        -seg(i, -j - 1, sd, ns, cap) + seg(-i - 1, j, sd, ns, cap)],
        }[kind]()

    at = sorted({p for kind, size in borders for s in ((size,) if kind == T.BORDER_BOX else (ns, sd, cap))
                 for p in (s - 1, -s)})
    found = []
    for a in range(dim):
        for p in at:
            if 0 <= p + half < n:
                ax = [np.array([p + half]) if d == a else np.arange(n) for d in range(dim)]
                lin = ax[0]
                for d in range(1, dim):
                    lin = lin[..., None] * n + ax[d]
                found.append(lin.ravel())
    lin = np.unique(np.concatenate(found))
    ix = [lin // n ** (dim - 1 - d) % n - half for d in range(dim)]
    vec = np.zeros((len(borders), dim, len(lin)))
    for b, (kind, size) in enumerate(borders):
        v = np.stack(family(kind, size, ix))
        size_of = np.sqrt((v ** 2).sum(0))
        vec[b] = np.where(size_of > 0.001, v / np.where(size_of > 0, size_of, 1), v)
    keep = np.abs(vec).sum((0, 1)) > 0
    return lin[keep], vec[:, :, keep]


class _Reference:
    """One solve as plain torch in 64 bits: the regions of a plane, or one grid."""

    def __init__(self, desc, dt, imaginary=False, borders=()):
        self.dim, self.n, self.dx, self.dt, self.im = desc.dim, int(desc.n[0]), desc.dx[0], dt, imaginary
        self.dev, self.desc = _device(), desc
        n, dx, dim = self.n, self.dx, self.dim
        i = np.arange(n)
        self.x = -0.5 * dx * (n - 1) + dx * i
        self.p = 2 * math.pi / n / dx * np.where(i < n // 2, i, i - n)
        self.node = desc.nCAP + np.where(i < n // 2, -i, i - n + 1)
        self.free = [()] if not desc.multigrid else [(), (0,), (1,), (0, 1)]
        self.borders = list(borders)
        if self.borders:
            lin, vec = _border_points(dim, n, self.borders)
            self.lin, self.vec = torch.from_numpy(lin).to(self.dev), torch.from_numpy(vec).to(self.dev)

    def t(self, a):
        return torch.from_numpy(np.ascontiguousarray(a)).to(self.dev)

    def along(self, v, a):
        return v.reshape([-1 if d == a else 1 for d in range(self.dim)])

    def mask1(self):
        d = self.desc
        k = np.maximum(self.node, 0)
        if d.absorber == T.ABS_COS18:
            return np.where(k > 0, np.sin(0.5 * math.pi * (d.nCAP - k) / d.nCAP) ** 0.125, 1.0)
        return np.exp(-(k.astype(float) ** 4) * (3.0 / d.nCAP) ** 4)

    def potential(self, free):
        """V over the bounded axes of a region."""
        d, dim = self.desc, self.dim
        x = [self.along(self.t(self.x), a) for a in range(dim)]
        bound = [a for a in range(dim) if a not in free]
        ne, ee = d.Ncharge * d.Echarge, d.Echarge ** 2
        v = torch.zeros([1] * dim, dtype=torch.float64, device=self.dev)
        if d.potential == T.POT_COULOMB:
            return v + ne / torch.sqrt(sum(x[a] ** 2 for a in bound) + d.Nsoft) if bound else v
        for a in bound:
            v = v + ne / torch.sqrt(x[a] ** 2 + d.Nsoft)
        for k, a in enumerate(bound):
            for b in bound[k + 1:]:
                mixed = x[a] * x[b] if d.potential == T.POT_ECKHARDT_SACHA else 0.0
                v = v + ee / torch.sqrt((x[a] - x[b]) ** 2 + mixed + d.Esoft)
        return v

    def turn(self, h, delta):
        return torch.exp(-delta * h) if self.im else torch.exp(-1j * delta * h)

    def x_half(self, r, delta, c):
        """The X factor of region r (a full array; kept by the caller where it does not change)."""
        h = self.potential(self.free[r])
        for a in range(self.dim):
            if c:
                h = h + c * self.along(self.t(self.x), a)
        f = self.turn(h, delta)
        if not self.desc.multigrid and self.desc.absorber != T.ABS_NONE:
            d, k = self.desc, np.maximum(self.node, 0).astype(float)
            if d.absorber == T.ABS_CAP:
                one = np.exp(-delta * k ** 4 * (3.0 / d.nCAP) ** 4)
            else:
                one = self.mask1() ** (delta / d.absorber_tau)
            for a in range(self.dim):
                f = f * self.along(self.t(one), a)
        return f

    def kinetic(self, psi, r, delta, c):
        axes = [a for a in range(self.dim) if r == 0 or a not in self.free[r]]
        if axes:
            psi = torch.fft.fftn(psi, dim=axes)
        for a in range(self.dim):
            psi = psi * self.along(self.turn(self.t(0.5 * self.p ** 2 + self.p * c), delta), a)
        return torch.fft.ifftn(psi, dim=axes) if axes else psi

    def row(self, psi, step, time, a, want):
        vol = self.dx ** self.dim
        out = [float(step), time] + [math.nan] * 5
        dens = torch.view_as_real(psi).square().sum(-1)
        out[2] = float(dens.sum()) * vol
        if want:
            out[3] = float((dens * self.potential(())).sum()) * vol
            mom = torch.view_as_real(torch.fft.fftn(psi)).square().sum(-1)
            k2 = sum(self.along(self.t(0.5 * self.p ** 2), d) for d in range(self.dim))
            out[4] = float((mom * k2).sum()) * vol / self.n ** self.dim
            out[5] = out[3] + out[4]
        if self.borders:
            flat, m = psi.reshape(-1), self.n ** self.dim
            mid = flat[self.lin]
            total = torch.zeros(len(self.borders), dtype=torch.float64, device=self.dev)
            for d in range(self.dim):
                step_d = self.n ** (self.dim - 1 - d)
                inside = (self.lin - step_d > 0) & (self.lin + step_d < m)
                up, down = (self.lin + step_d).clamp(max=m - 1), (self.lin - step_d).clamp(min=0)
                j = torch.where(inside, (mid.conj() * (flat[up] - flat[down])).imag / (2 * self.dx), 0.0)
                j = j + a * torch.view_as_real(mid).square().sum(-1)
                total += (self.vec[:, d] * j).sum(-1)
            out += [float(v) * vol / self.dx for v in total]
        return out

    def transfer(self, psi):
        """The edges of each region moved to the regions that free one axis more, then the masks."""
        n, cap = self.n, self.desc.nCAP
        i = np.arange(n)
        m1 = self.mask1()
        edge = self.t(np.where((i < cap) | (i >= n - cap), 1.0 - m1, 0.0))
        corr = self.t(1 - 0.5 * (1.0 - m1))
        for src, dst, a in ((0, 1, 0), (0, 2, 1), (1, 3, 1), (2, 3, 0)):
            part = psi[src] * self.along(edge, a)
            if src == 0:
                part = part * self.along(corr, 1 - a)
            psi[dst] = psi[dst] + torch.fft.fft(part, dim=a)
        one = self.t(m1)
        for r, axes in ((0, (0, 1)), (1, (1,)), (2, (0,))):
            for a in axes:
                psi[r] = psi[r] * self.along(one, a)


def _exact_pulse(desc, dt, order, gauge, field, psi0, steps, borders, energies):
    ref = _Reference(desc, dt, borders=borders)
    psi = [psi0] + [torch.zeros_like(psi0) for _ in ref.free[1:]]
    length = gauge == "length"
    vec, timer, rows = _Vector(field), 0.0, []
    d = dt / order
    still = None if length else [ref.x_half(r, d / 2, 0.0) for r in range(len(psi))]
    rows.append(ref.row(psi[0], 0, 0.0, 0.0, energies))
    for k in range(steps):
        start = timer
        for c in range(1, order):   # the shorter chains only advance the coupling
            timer = start
            for _ in range(c):
                if not length:
                    vec.at(timer)
                timer += dt / c
        timer = start
        # X half steps of neighbouring substeps join into one, at one time
        for sub in range(order):
            if length:
                f = _field_at(field, timer)
                weight = d / 2 if sub == 0 else d
                psi = [q * ref.x_half(r, weight, f) for r, q in enumerate(psi)]
                timer += weight
                psi = [ref.kinetic(q, r, d, 0.0) for r, q in enumerate(psi)]
            else:
                a = vec.at(timer)
                for r in range(len(psi)):
                    psi[r] = psi[r] * (still[r] if sub == 0 else still[r] * still[r])
                    psi[r] = ref.kinetic(psi[r], r, d, a)
                timer += d
        if length:
            f = _field_at(field, timer)
            psi = [q * ref.x_half(r, d / 2, f) for r, q in enumerate(psi)]
            timer += d / 2
        else:
            psi = [q * s for q, s in zip(psi, still)]
        rows.append(ref.row(psi[0], k + 1, timer, 0.0 if length else vec.a, energies))
        if desc.multigrid:
            ref.transfer(psi)
    return psi, np.array(rows)


def exact(case, seed):
    if case["kind"] == "batch":
        sides, fields = _batch_members(case, seed)
        out = {"psi": [], "records": [], "flux_integral": []}
        for n, f in zip(sides, fields):
            desc = _grid(2, n, case["precision"], "eberly", case["dt"])
            psi, rows = _exact_pulse(desc, case["dt"], 1, "velocity", f, _start_state(2, n, seed), _batch_total(case),
                                     _borders(2, 0), False)
            out["psi"].append(psi[0].cpu().numpy().ravel())
            out["records"].append(np.concatenate([rows[:, :3], rows[:, 7:]], axis=1))
            out["flux_integral"].append(rows[1:-1, 7:].sum(0) * case["dt"])
        return out
    desc = _grid(case["dim"], case["n"], case["precision"], case["potential"], case["dt"], case.get("regions", False))
    psi = _start_state(case["dim"], case["n"], seed, case["kind"] == "pulse")
    if case["kind"] == "pulse":
        borders = _borders(case["dim"], case["box"])
        psi, rows = _exact_pulse(desc, case["dt"], case["order"], case["gauge"], _fields(case, seed)[0], psi,
                                 case["steps"], borders, case["energies"])
        return {"records": rows, "psi": [q.cpu().numpy().ravel() for q in psi],
                "flux_integral": rows[:, 7:].sum(0) * case["dt"]}
    ref = _Reference(desc, case["dt"], imaginary=True)
    half, rows, last, timer = ref.x_half(0, case["dt"] / 2, 0.0), [], 0.0, 0.0
    for k in range(case["steps"] + 1):
        if k:
            psi = ref.kinetic(psi * half, 0, case["dt"], 0.0) * half
            timer += case["dt"]
        psi = psi / math.sqrt(float(torch.view_as_real(psi).square().sum()) * ref.dx ** ref.dim)
        row = ref.row(psi, k, timer, 0.0, True)
        row[6], last = row[5] - last, row[5]
        rows.append(row)
    return {"records": np.array(rows), "psi": [psi.cpu().numpy().ravel()]}
