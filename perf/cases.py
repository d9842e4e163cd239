"""Timed workloads of the library: what a user's program has it do, through
the public entry points of ``komegafoulingmodel_amd``.

Each case is a dict of plain values; ``kind`` says which path it takes:

flow       plain lattice-Boltzmann steps (k-omega off) on a flat or fouled channel
turbulent  k-omega steps on a flat channel or one with a thin deposit
thermal    k-omega steps with a temperature call each, then one Nusselt record
ensemble   several channels of uneven size stepped together
gradient   an objective run with checkpoints and its adjoint (wall-shape gradient)
removal    wall shear and re-entrainment of deposited particles on the tracer's arrays

Walls: "flat" (solid edge rows), "thin" (a deposit well below one node, as at
the beginning of fouling) and "fouled" (the seeded Gaussian layers of the named
workloads).  The k-omega kinds keep to flat and thin walls: on curved walls the
reference's near-wall rows are ill-conditioned and amplify the last bit of any
arithmetic a thousandfold within a few steps.

A field is returned in the precision of the run it comes from (float32 for
FP32 and 16-bit populations, float64 for FP64 ones), populations as the FP64
restart file holds them.
"""
import math

import numpy as np
import torch

from komegafoulingmodel_amd import channel, lib

BULK = 0.05      # bulk velocity of the turbulent channels
SPIN_UP = 32     # k-omega steps a program has behind it before the measured ones
SAVE = lib.OPTION_SAVE_MACRO_FIELDS
BYTES = {"f32": 4, "f32x": 4, "f16": 2, "bf16": 2, "f64": 8}
# particle re-entrainment: sizes, and their constants in lattice units
SIZES = 4
DRAG, LIFT, MASS = [300.0, 500.0, 700.0, 900.0], [200.0, 100.0, 50.0, 20.0], [1.0, 2.0, 3.0, 4.0]


def listed():
    return [
        # a parameter study on a tiny, oddly sized channel at the reference's
        # cadence (macros every step, wall shear every 3): launches and latency
        dict(name="tiny_257x61", kind="flow", nX=257, nY=61, walls="flat", storage="f32",
             steps=24, cadence=True, tuned=False),
        # the plane Poiseuille configuration (1024 x 128), between two outputs
        dict(name="poiseuille_1024x128", kind="flow", nX=1024, nY=128, walls="flat",
             storage="f32", steps=2048, cadence=False, tuned=True),
        # production cadence on a ragged fouled channel near the shipped size
        dict(name="production_2001x203", kind="flow", nX=2001, nY=203, walls="fouled",
             storage="f32", steps=300, cadence=True, tuned=False),
        # the headline shape: 8192 x 1024 with fouling on both walls
        dict(name="fouled_8192x1024", kind="flow", nX=8192, nY=1024, walls="fouled",
             storage="f32", steps=1000, cadence=False, tuned=True),
        # 16-bit populations
        dict(name="fouled_4096x512_f16", kind="flow", nX=4096, nY=512, walls="fouled",
             storage="f16", steps=2000, cadence=False, tuned=True),
        # the shipped run's size (nX 2000, nY 204) with k-omega on
        dict(name="turbulent_2000x204", kind="turbulent", nX=2000, nY=204, walls="thin",
             storage="f32", Re=10800.0, steps=48),
        # the k-omega configuration's grid (4096 x 512, Re 10,000)
        dict(name="turbulent_4096x512", kind="turbulent", nX=4096, nY=512, walls="flat",
             storage="f32", Re=10000.0, steps=64),
        # FP64 populations on an odd size
        dict(name="turbulent_1001x131_f64", kind="turbulent", nX=1001, nY=131, walls="flat",
             storage="f64", Re=5000.0, steps=32),
        # LB + k-omega + temperature each step, and a Nusselt record
        dict(name="thermal_2048x256", kind="thermal", nX=2048, nY=256, walls="flat",
             storage="f32", Re=10000.0, steps=24),
        # uneven channels advanced together, k-omega on
        dict(name="ensemble_6_turbulent", kind="ensemble", members=6, maxX=2048, maxY=256,
             komega=True, storage="f32", steps=16),
        # wall-shape gradient on the sensitivity grid, exact k-omega adjoint
        dict(name="gradient_2048x256", kind="gradient", nX=2048, nY=256, komega=True,
             frozen=False, storage="f32", steps=128, window=32, interval=16),
        # a tracer step's particle re-entrainment over 16M deposited particles
        dict(name="removal_16M", kind="removal", nX=4096, nY=256, particles=1 << 24),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["flow", "flow", "flow", "turbulent", "turbulent", "turbulent", "thermal",
                       "ensemble", "gradient", "removal"])
    if kind == "flow":
        nX, nY = _log(rng, 130, 4096), _log(rng, 40, 512)
        cadence = rng.random() < 0.4
        steps = max(24, min(2000, int(2.0e9 / (nX * nY))))
        if cadence:
            steps = 3 * min(100, steps // 3)
        return dict(kind=kind, nX=nX, nY=nY, walls=rng.choice(["flat", "fouled"]),
                    storage=rng.choice(["f32", "f32", "f16", "bf16", "f64"]), steps=steps,
                    cadence=cadence, tuned=rng.random() < 0.5)
    if kind in ("turbulent", "thermal"):
        nX, nY = _log(rng, 256, 3000), _log(rng, 48, 400)
        walls = rng.choice(["flat", "thin"])
        steps = rng.randrange(8, 57)
        storage = rng.choice(["f32", "f32", "f64"])
        Re = round(rng.uniform(2000.0, 20000.0), 1)
        return dict(kind=kind, nX=nX, nY=nY, walls=walls, storage=storage, Re=Re,
                    steps=steps if kind == "turbulent" else max(8, steps // 2))
    if kind == "ensemble":
        return dict(kind=kind, members=rng.randrange(2, 9), maxX=_log(rng, 512, 2048),
                    maxY=_log(rng, 64, 256), komega=rng.random() < 0.5, storage="f32",
                    steps=rng.randrange(8, 65))
    if kind == "gradient":
        komega = rng.random() < 0.6
        steps = rng.randrange(32, 129)
        return dict(kind=kind, nX=_log(rng, 256, 2048), nY=_log(rng, 64, 256), komega=komega,
                    frozen=komega and rng.random() < 0.5, storage="f32", steps=steps,
                    window=rng.randrange(8, steps), interval=rng.randrange(4, 25))
    return dict(kind=kind, nX=_log(rng, 512, 4096), nY=_log(rng, 64, 256),
                particles=_log(rng, 1 << 14, 1 << 24))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------


def _thin(nX, rng):
    """A deposit of at most 0.2 nodes."""
    h = channel.gaussian_fouling(nX, rng, amp=(0.0, 1.0))
    top = float(np.max(h(np.arange(nX, dtype=np.float64))))
    return lambda x: 0.2 / top * h(x)


def _turbulent(nX, nY, walls, Re, seed):
    """A plane channel with k-omega on, as the ensemble of channels has them."""
    H = nY - 2.0
    nu = BULK * H / Re
    rng = np.random.Generator(np.random.PCG64(seed))
    hb, ht = (_thin(nX, rng), _thin(nX, rng)) if walls == "thin" else ((lambda x: 0.0 * x),) * 2
    C0, BL = channel.wall_points(nX, lambda x: 0.5 + hb(x), lambda x: nY - 1.5 - ht(x))
    k0 = 1.5 * (0.05 * BULK) ** 2
    return channel.Workload("turbulent", nX, nY, C0, BL, pipe_radius=H / 2.0,
                            tau0=1.0 / (3.0 * nu + 0.5), nu=nu,
                            Fval=channel.turbulent_forcing(H, nu, Re), komega=True, k_ini=k0,
                            omega_ini=math.sqrt(k0) / (0.09 ** 0.25 * 0.07 * H), Re=Re, noise=0.01,
                            u_init=BULK, seed=seed)


def _flow(nX, nY, walls, seed):
    if walls == "flat":
        return channel.flat_channel(nX, nY, seed=seed)
    return channel.fouled_channel(nX, nY, seed=seed, amp=(0.0, 8.0 * nY / 1024.0))


def _lattice(w, storage, tuned=False):
    """The workload's lattice with its seeded state, ready to step."""
    L = lib.Lattice(w.nX, w.nY, storage=storage, komega=w.komega)
    L.set_params(w.tau0, w.Fval, w.nu)
    # near-flat walls: the nearest link lies within a few columns
    gp = dict(w.geom_params(), wall_d_search_rad=10 if w.komega else 1)
    L.build_geometry(w.C0, w.BL, **gp)
    if tuned:
        L.autotune(20)
    rho, ux, uy = w.initial_velocity(L.geometry("nType"))
    L.init_state(rho, ux, uy)
    if w.komega:
        L.init_komega(w.k_ini, w.omega_ini, w.Re)
    return L


def _members(case, seed):
    """Sizes of an ensemble: uneven, up to maxX x maxY, from the case alone."""
    out = []
    for i in range(case["members"]):
        nX = max(192, case["maxX"] * (8 - 3 * i % 7) // 8 // 64 * 64)
        nY = max(48, case["maxY"] * (8 - 5 * i % 6) // 8)
        if case["komega"]:
            out.append(_turbulent(nX, nY, "thin" if i % 2 else "flat", 4000.0 + 2000.0 * i, seed + i))
        else:
            out.append(_flow(nX, nY, "fouled", seed + i))
    return out


def prepare(case, seed):
    kind, seed = case["kind"], int(seed) % (1 << 31)
    s = dict(case=case, dtype=np.float64 if case.get("storage") == "f64" else np.float32)
    if kind == "flow":
        s["L"] = _lattice(_flow(case["nX"], case["nY"], case["walls"], seed), case["storage"],
                          case["tuned"])
    elif kind in ("turbulent", "thermal"):
        w = _turbulent(case["nX"], case["nY"], case["walls"], case["Re"], seed)
        L = s["L"] = _lattice(w, case["storage"])
        if kind == "thermal":
            L.thermal_init(alpha_fluid=w.nu / 0.708, alpha_foul=0.1 * w.nu / 0.708, pr_turb=0.9,
                           t_in=2.0, t_initial=0.5)
            L.nusselt_init(height=2 * int(w.pipe_radius), wavy_start=case["nX"] // 8,
                           wavy_period=case["nX"] // 8, wavy_periods=5, k_soot=0.057, k_air=0.042)
        L.step(SPIN_UP)
    elif kind == "ensemble":
        s["members"] = [_lattice(w, case["storage"]) for w in _members(case, seed)]
        if case["komega"]:
            for L in s["members"]:
                L.step(SPIN_UP)
        s["E"] = lib.Ensemble(s["members"])
    elif kind == "gradient":
        from komegafoulingmodel_amd import sensitivity

        nY = case["nY"]
        H = nY - 2.0
        P = sensitivity.WallShapeProblem(nX=case["nX"], nY=nY, H=H, amp=0.0, n_ctrl=16,
                                         nu=0.005, Re=BULK * H / 0.005, seed=seed,
                                         storage=case["storage"], komega=case["komega"])
        C0, BL = P.points(0.05 * P.initial_theta())
        w = channel.Workload("gradient", P.nX, nY, C0, BL, pipe_radius=H / 2.0, tau0=P.tau0,
                             nu=P.nu, Fval=P.Fval, komega=P.komega, k_ini=P.k_ini,
                             omega_ini=P.omega_ini, Re=P.Re, noise=0.01, u_init=P.Ub, seed=seed)
        s["L"] = _lattice(w, case["storage"])
        s["dydth"] = P.dy_dtheta(C0)
    else:
        L = s["L"] = _lattice(_flow(case["nX"], case["nY"], "fouled", seed), "f32")
        L.step(60, SAVE)
        L.wall_shear()
        tau, b = L.download("tau_bl"), L.geometry("bounds")
        links = np.r_[np.arange(b[0], b[0] + b[1]), np.arange(b[2], b[2] + b[3])]
        n, g = case["particles"], torch.Generator(device="cuda").manual_seed(seed)
        a = np.abs(tau[tau != 0.0])
        # most particles stay, as on a wall in steady fouling; a few per cent
        # leave, a few have left or settled for good before
        s["crit"] = np.quantile(a, [0.99, 0.98, 0.995, 0.99, 0.9975, 0.995, 1.0, 0.9975])
        ints = lambda lo, hi, dt: torch.randint(lo, hi, (n,), device="cuda", generator=g).to(dt)  # noqa: E731
        # the tracer keeps them sorted by location, so in link order
        flag = torch.sort(ints(0, len(links), torch.int64)).values
        flag = torch.from_numpy(links.astype(np.int32)).cuda()[flag]
        u = torch.rand(n, device="cuda", generator=g)
        flag = torch.where(u < 0.02, -1, torch.where(u < 0.04, -2, flag)).to(torch.int32)
        s["P"] = dict(pos=torch.zeros(2 * n, dtype=torch.float64, device="cuda"),
                      num_rep=ints(1, 1000, torch.int32), type=ints(0, SIZES, torch.int16),
                      dep_flag=flag, dep_timer=ints(20000, 30000, torch.int16),
                      loc=torch.zeros(n, dtype=torch.int32, device="cuda"),
                      timer=torch.zeros(n, dtype=torch.int32, device="cuda"))
        s["dep"] = torch.zeros(SIZES * L._nBL, dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------


def _fields(L, dt, names):
    """rho, the velocity (both components) and the named fields."""
    D = L.D
    u = np.empty((2, D), dt)
    u[0], u[1] = L.download("ux"), L.download("uy")
    out = {n: L.download(n).astype(dt, copy=False) for n in names}
    return dict(out, u=u, rho=L.download("rho").astype(dt, copy=False))


def run(s):
    case, dt = s["case"], s["dtype"]
    kind, L = case["kind"], s.get("L")
    if kind == "flow":
        if not case["cadence"]:
            L.step(case["steps"] - 1)
            L.step(1, SAVE)
            return _fields(L, dt, ())
        for _ in range(case["steps"] // 3):
            L.step(3, SAVE)
            L.wall_shear()
        out = _fields(L, dt, ("tau_node", "tau_bl"))
        out["f"] = L.download("f")  # the restart file's populations
        return out
    if kind == "turbulent":
        L.step(case["steps"])
        return _fields(L, dt, ("k", "omega"))
    if kind == "thermal":
        for _ in range(case["steps"]):
            L.step(1)
            L.thermal_step(1)
        out = _fields(L, dt, ("T", "k", "omega"))
        nu = L.nusselt()
        return dict(out, nu=nu["nu"].astype(dt), mean=nu["mean"].astype(dt))
    if kind == "ensemble":
        s["E"].step(case["steps"] - 1)
        s["E"].step(1, SAVE)
        return [_fields(m, dt, ("k", "omega") if case["komega"] else ()) for m in s["members"]]
    if kind == "gradient":
        J = L.objective_run(case["steps"], case["interval"], case["window"],
                            frozen_turbulence=case["frozen"])
        dy, dq = L.adjoint()
        return dict(J=np.array([J], dt), dy=dy.astype(dt), dq=dq.astype(dt),
                    dtheta=(s["dydth"].T @ dy).astype(dt))
    P = s["P"]
    L.wall_shear()
    L.shear_removal({k: v.data_ptr() for k, v in P.items()}, s["dep"].data_ptr(), 0,
                    case["particles"], tau_crit=s["crit"], drag_coeff=DRAG, lift_coeff=LIFT,
                    mass=MASS, loc_stride=case["nX"], timer_start=1000)
    return dict({k: P[k] for k in ("pos", "dep_flag", "dep_timer", "loc", "timer")}, dep=s["dep"])


# ---------------------------------------------------------------------------
# compulsory work
# ---------------------------------------------------------------------------


def _step_bytes(storage, komega, save):
    """State a step reads and writes per node: populations, the node type; with
    k-omega k, omega and the strain in FP64 (read and written), the eddy
    viscosity (written) and the wall distance (read); the macros when saved."""
    b = BYTES[storage]
    n = 18 * b + 2
    if komega:
        n += 8 * (2 * 2 + 2 * 3 + 1 + 1)
    if save:
        n += 3 * max(b, 4)
    return n


def work(case):
    kind = case["kind"]
    if kind == "removal":
        return {"bytes": 10.0 * case["particles"], "flops": 4.0 * case["particles"]}
    if kind == "ensemble":
        nodes = sum(w.nX * (w.nY - 2) for w in _members(case, 0))
    else:
        nodes = case["nX"] * (case["nY"] - 2)
    komega = case.get("komega", kind in ("turbulent", "thermal"))
    per = _step_bytes(case["storage"], komega, komega or case.get("cadence", False))
    # flops of a node: collision 130, k-omega rows and one solver iteration 400
    flops = 530.0 if komega else 130.0
    if kind == "thermal":
        per, flops = per + 8 * 3 + 8, flops + 150.0  # T read and written, nu_t, u
    if kind == "gradient":
        # forward, recompute and adjoint step (adjoint populations and state read, written)
        per, flops = 3 * per, 3 * flops
    return {"bytes": float(per) * nodes * case["steps"], "flops": flops * nodes * case["steps"]}


# ---------------------------------------------------------------------------
# the same in 64 bits, in plain torch, for flat walls
# ---------------------------------------------------------------------------

CX, CY = (0, 1, -1, 0, 0, 1, -1, 1, -1), (0, 0, 0, 1, -1, 1, -1, -1, 1)
REV = (0, 2, 1, 4, 3, 6, 5, 8, 7)
W1 = {0: 2.0 / 3.0, 1: 1.0 / 6.0, -1: 1.0 / 6.0}


class _Flat:
    """A flat channel in FP64: arrays [nY - 2, nX] of the fluid rows."""

    def __init__(self, w):
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.w = w
        self.nX, self.n, self.XF = w.nX, w.nY - 2, w.XF

        def rows(a):
            a = torch.from_numpy(np.ascontiguousarray(a.reshape(w.nY, self.XF)[1:-1, :w.nX]))
            return a.to(dev, torch.float64)

        nType = np.zeros(w.D, np.int16)
        nType.reshape(w.nY, -1)[[0, -1]] = 1
        rho, ux, uy = (rows(a) for a in w.initial_velocity(nType))
        self.g = torch.stack([self.geq(i, rho, ux, uy) for i in range(9)])
        one = torch.ones_like(rho)
        y = torch.arange(self.n, device=dev, dtype=torch.float64)[:, None] + 0.5
        self.yw = torch.minimum(y, float(self.n) - y) * one
        # wall spacings: 1, half a node towards a wall
        up, dn = one.clone(), one.clone()
        up[-1] = dn[0] = 0.5
        self.ax, self.ay = self.weights(one, one, 2), self.weights(up, dn, 2)
        self.tx, self.ty = self.weights(one, one, 2), self.weights(up, dn, 0)
        self.wall = torch.zeros_like(rho, dtype=torch.bool)
        self.wall[0] = self.wall[-1] = True
        if w.komega:
            self.k, self.o = w.k_ini * one, w.omega_ini * one
            self.S = [0.0 * one] * 3

    @staticmethod
    def weights(dp, dm, test):
        dc = dp + dm
        d1 = [dm / (dp * dc), -dp / (dm * dc), (dp - dm) / (dp * dm)]
        two = d1[test].abs() > 10.0
        d1 = [torch.where(two, c, d) for c, d in zip((1.0 / dc, -1.0 / dc, 0.0 * dc), d1)]
        return d1 + [2.0 / (dp * dc), 2.0 / (dm * dc), -2.0 / (dp * dm)]

    @staticmethod
    def geq(i, rho, ux, uy):
        """feq - w of direction i."""
        px = -ux * ux if CX[i] == 0 else 0.5 * (CX[i] * ux + ux * ux)
        py = -uy * uy if CY[i] == 0 else 0.5 * (CY[i] * uy + uy * uy)
        a, b = W1[CX[i]], W1[CY[i]]
        return (rho - 1.0) * a * b + rho * (a * py + b * px + px * py)

    @staticmethod
    def nbs(a):
        """E, W, N, S neighbours; zero on the solid rows."""
        z = torch.zeros_like(a[:1])
        return (torch.roll(a, -1, 1), torch.roll(a, 1, 1), torch.cat([a[1:], z]),
                torch.cat([z, a[:-1]]))

    def grad(self, a):
        e, w, n, s = self.nbs(a)
        ax, ay = self.ax, self.ay
        return ax[0] * e + ax[1] * w + ax[2] * a, ay[0] * n + ay[1] * s + ay[2] * a

    def lb(self):
        w, g = self.w, self.g
        rho = 1.0 + g.sum(0)
        ux = sum(CX[i] * g[i] for i in range(9)) / rho
        uy = sum(CY[i] * g[i] for i in range(9)) / rho
        eq = [self.geq(i, rho, ux, uy) for i in range(9)]
        omega = w.tau0
        if w.komega:
            self.k = torch.where(self.k < 0, 1e-16 + 0 * self.k, self.k)
            self.o = self.o.abs()
            k, o, yw, S = self.k, self.o, self.yw, self.S
            arg = torch.maximum(2.0 * k.sqrt() / (0.09 * o * yw), 500.0 * w.nu / (yw * yw * o))
            F2 = torch.tanh(arg * arg) * (2.0 * (S[0] ** 2 + 2.0 * S[1] ** 2 + S[2] ** 2)).sqrt()
            self.nut = (0.31 * k / torch.maximum(0.31 * o, F2)).clamp(1e-16, 10.0)
            omega = 1.0 / (3.0 * (self.nut + w.nu) + 0.5)
            ne = [g[i] - eq[i] for i in range(9)]
            c = -1.5 * w.tau0 / rho
            self.S = [c * sum(CX[i] ** 2 * ne[i] for i in range(9)),
                      c * sum(CX[i] * CY[i] * ne[i] for i in range(9)),
                      c * sum(CY[i] ** 2 * ne[i] for i in range(9))]
        self.rho, self.ux, self.uy = rho, ux + 0.5 * w.Fval, uy
        new = torch.empty_like(g)
        for i in range(9):
            out = g[i] + omega * (eq[i] - g[i]) + self.geq(i, rho, ux + w.Fval, uy) - eq[i]
            moved = torch.roll(out, CX[i], 1)
            if CY[i] == 0:
                new[i] = moved
            elif CY[i] > 0:  # the last fluid row bounces back into its own slot
                new[i, 1:], new[REV[i], -1] = moved[:-1], out[-1]
            else:
                new[i, :-1], new[REV[i], 0] = moved[1:], out[0]
        self.g = new

    def solve(self, A, b, x):
        """The five-point system with diagonal 1 to the FP64 floor (BiCGStab)."""
        def mul(v):
            return v + sum(a * q for a, q in zip(A, self.nbs(v)))

        r = b - mul(x)
        rh, rho, al, om = r, 1.0, 1.0, 1.0
        v = p = torch.zeros_like(r)
        goal = 1e-13 * float(b.norm())
        for _ in range(60):
            if float(r.norm()) <= goal:
                break
            new = (rh * r).sum()
            beta = new / rho * (al / om)
            rho = new
            p = r + beta * (p - om * v)
            v = mul(p)
            al = rho / (rh * v).sum()
            q = r - al * v
            t = mul(q)
            om = (t * q).sum() / (t * t).sum().clamp_min(1e-300)
            x = x + al * p + om * q
            r = q - om * t
        return x

    def komega(self):
        w, k, o, yw, nt, S = self.w, self.k, self.o, self.yw, self.nut, self.S
        ax, ay, nu = self.ax, self.ay, w.nu
        okx, oky = self.grad(k)
        oox, ooy = self.grad(o)
        mx, my = 1.712 / o * okx, 1.712 / o * oky
        cd = (self.rho * (mx * oox + my * ooy)).clamp_min(1e-10)
        arg = torch.minimum(torch.maximum(k.sqrt() / (0.09 * o * yw), 500.0 * nu / (yw * yw * o)),
                            3.424 * k / (cd * yw * yw))
        F1 = torch.tanh(arg ** 4)
        Dk = nu + (0.85 * F1 + (1.0 - F1)) * nt
        Do = nu + (0.5 * F1 + 0.856 * (1.0 - F1)) * nt
        dkx, dky = self.grad(Dk)
        dox, doy = self.grad(Do)
        tr = S[0] + S[2]
        Pk = 2.0 * nt * (S[0] ** 2 + S[2] ** 2 + 2.0 * S[1] ** 2) - 2.0 / 3.0 * k * self.rho * tr
        Pk = torch.minimum(Pk, 0.9 * k * o).clamp_min(0.0)
        gam = (F1 * (5.0 / 9.0) + (1.0 - F1) * 0.44) / nt
        wall = torch.minimum(((6.0 * nu / 0.075 / yw ** 2) ** 2
                              + (k.sqrt() / (0.5477225575 * 0.41 * yw)) ** 2).sqrt(),
                             torch.full_like(o, 1000.0))

        def rows(jx, jy, d, sink, dt):
            c = 1.0 + dt * (jx * ax[2] + jy * ay[2] - d * (ax[5] + ay[5])) + sink
            return [dt * (jx * ax[0] - d * ax[3]) / c, dt * (jx * ax[1] - d * ax[4]) / c,
                    dt * (jy * ay[0] - d * ay[3]) / c, dt * (jy * ay[1] - d * ay[4]) / c], c

        Ak, ck = rows(self.ux - dkx, self.uy - dky, Dk, 0.09 * o, 1.0)
        free = (~self.wall).to(o.dtype)
        Ao, co = rows(self.ux - dox - mx, self.uy - doy - my, Do, 0.09 * o * free, free)
        bo = torch.where(self.wall, wall, o + gam * Pk) / co
        self.k = self.solve(Ak, (k + Pk) / ck, k)
        self.o = self.solve(Ao, bo, o)

    def temperature(self, T, alpha, prt, tin):
        tx, ty, at = self.tx, self.ty, self.nut / prt
        e, w, n, s = self.nbs(self.nut / prt)
        jx = self.ux - (tx[0] * e + tx[1] * w + tx[2] * at / prt)
        jy = self.uy - (ty[0] * n + ty[1] * s + ty[2] * at / prt)
        al = alpha + at
        src = T.clamp(0.0, tin)
        c = 1.0 + jx * tx[2] + jy * ty[2] - al * (tx[5] + ty[5])
        E, W = jx * tx[0] - al * tx[3], jx * tx[1] - al * tx[4]
        N, S = jy * ty[0] - al * ty[3], jy * ty[1] - al * ty[4]
        src[:, 0] -= tin * W[:, 0]
        c[:, -1] += E[:, -1]
        E[:, -1] = 0.0
        W[:, 0] = 0.0
        return self.solve([a / c for a in (E, W, N, S)], src / c, T)

    def out(self, a, solid=0.0):
        """A field in the library's layout: solid rows and padding hold `solid`."""
        full = np.full((self.n + 2, self.XF), solid)
        full[1:-1, :self.nX] = a.cpu().numpy()
        return full.reshape(-1)

    def fields(self):
        return dict(rho=self.out(self.rho), u=np.stack([self.out(self.ux), self.out(self.uy)]))


def exact(case, seed):
    kind, seed = case["kind"], int(seed) % (1 << 31)
    if case.get("walls") != "flat" or case.get("nX", 0) * case.get("nY", 0) > 2200000:
        return None
    if kind == "flow":
        if case["steps"] * max(2.0e5, case["nX"] * case["nY"]) > 1.2e9:
            return None
        F = _Flat(_flow(case["nX"], case["nY"], "flat", seed))
        for _ in range(case["steps"]):
            F.lb()
        out = F.fields()
        if case["cadence"]:
            weight = [W1[CX[i]] * W1[CY[i]] for i in range(9)]
            f = np.concatenate([F.out(F.g[i] + weight[i]) for i in range(9)])
            out.update(f=f, tau_node=None, tau_bl=None)
        return out
    if kind not in ("turbulent", "thermal"):
        return None
    w = _turbulent(case["nX"], case["nY"], "flat", case["Re"], seed)
    F = _Flat(w)
    for _ in range(SPIN_UP):
        F.lb()
        F.komega()
    T = torch.full_like(F.k, 0.5)
    for _ in range(case["steps"]):
        F.lb()
        F.komega()
        if kind == "thermal":
            T = F.temperature(T, w.nu / 0.708, 0.9, 2.0)
    out = dict(F.fields(), k=F.out(F.k), omega=F.out(F.o))
    return out if kind == "turbulent" else dict(out, T=F.out(T), nu=None, mean=None)
