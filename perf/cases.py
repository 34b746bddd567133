"""The work that users have this time-stepper do, as cases that can be timed.

Every case runs through diablo_amd.gpu, the Python face of the C-ABI: RK3
time steps of a resident state (FP64 and mixed precision, with a fixed and
with a COURANT time step, with and without the subgrid model), an ensemble's
step, SAVE_STATS, POISSON_P_CHAN, the transforms of host arrays, and the
Fortran bridge's default time step, which carries the host's arrays to the
GPU and back.  `exact` states the same operations in plain torch at 64 bits.
"""
import math

import numpy as np
import torch

from diablo_amd import case as decks
from diablo_amd import gpu

# even transform lengths 2^a 3^b: those with plans fixed at compile time (64,
# 96, 128, 192, 256, 384) and those without
LENGTHS = (32, 36, 48, 54, 64, 72, 96, 108, 128, 144, 162, 192, 216, 256, 288, 324, 384)
STATE = ("CU1", "CU2", "CU3", "CP", "CF1", "CF2", "CF3", "CTH0", "CFTH0")
IDS = {"CU1": gpu.CU1, "CU2": gpu.CU2, "CU3": gpu.CU3, "CP": gpu.CP, "CF1": gpu.CF1, "CF2": gpu.CF2,
       "CF3": gpu.CF3, "CTH0": gpu.CTH0, "CFTH0": gpu.CFTH0}


def listed():
    return [
        # the smallest run in use (the 200-step channel of the decks): launches count
        dict(name="step_64", kind="step", deck="channel", nx=64, ny=65, nz=64, precision="fp64"),
        # the flagship run: a resolved channel at Re = 395, as in the benchmark
        dict(name="step_384", kind="step", deck="channel", nx=384, ny=257, nz=384, precision="fp64"),
        # the same run in mixed precision
        dict(name="step_384_mixed", kind="step", deck="channel", nx=384, ny=257, nz=384, precision="mixed"),
        # the Kelvin-Helmholtz layer between free-slip walls, buoyancy on
        dict(name="step_kh256_mixed", kind="step", deck="kh", nx=256, ny=193, nz=256, precision="mixed"),
        # VARIABLE_DT with UPDATE_DT = 1 on a grid without power-of-two lengths
        dict(name="step_cfl_162", kind="step_cfl", deck="channel", nx=162, ny=101, nz=108, precision="fp64"),
        # large-eddy simulation at the flagship size, the model in every substep
        dict(name="les_384", kind="les", deck="channel", nx=384, ny=257, nz=384, precision="fp64"),
        # large-eddy simulation on the coarse grid it is usually run on
        dict(name="les_96", kind="les", deck="channel", nx=96, ny=81, nz=108, precision="fp64"),
        # 64 independent layers on grids of their own, advanced together
        dict(name="ensemble_64", kind="ensemble", members=64, precision="mixed"),
        # SAVE_STATS of a resident run every SAVE_STATS_INT steps
        dict(name="stats_256", kind="stats", deck="kh", nx=256, ny=193, nz=256, precision="fp64"),
        # the pressure of a new flow or of one read without it
        dict(name="poisson_192", kind="poisson", deck="channel", nx=192, ny=129, nz=192, precision="fp64"),
        # FFT_XZ_TO_FOURIER and FFT_XZ_TO_PHYSICAL of a host array, as user hooks call them
        dict(name="transforms_192", kind="transforms", deck="channel", nx=192, ny=129, nz=192, precision="fp64"),
        # the Fortran bridge's default time step: the COMMON arrays go to the GPU and come back
        dict(name="bridge_step_192", kind="bridge", deck="channel", nx=192, ny=129, nz=192, precision="fp64"),
    ]


def draw(rng):
    kind = rng.choice(("step", "step", "step", "step", "step_cfl", "les", "les", "ensemble", "stats", "poisson",
                       "transforms", "bridge"))
    if kind == "ensemble":
        return dict(kind=kind, members=rng.randint(3, 40), precision=rng.choice(("mixed", "mixed", "fp64")))
    big = kind in ("step", "les", "step_cfl", "stats")

    def length():
        x = math.exp(rng.uniform(math.log(32), math.log(384 if big else 192)))
        return min(LENGTHS, key=lambda n: abs(math.log(n / x)))

    ny = round(math.exp(rng.uniform(math.log(21), math.log(257 if big else 129))))
    precision = rng.choice(("fp64", "fp64", "mixed", "mixed", "mixed_f64state")) if kind == "step" else "fp64"
    return dict(kind=kind, deck=rng.choice(("channel", "kh")), nx=length(), ny=ny, nz=length(), precision=precision)


def config(c):
    """The run parameters of a case: the repository's decks at the case's size,
    with the velocity fluctuations of a developed flow (0.14 rms)."""
    if c["deck"] == "kh":
        return decks.kh_case(c["nx"], c["ny"], c["nz"], re=1000.0, ri=0.1, dt=2.0e-3, kick=0.5)
    re, dt = (395.0, 5.0e-4) if c["nx"] >= 256 else (180.0, 1.0e-3)
    return decks.channel_case(c["nx"], c["ny"], c["nz"], re=re, dt=dt, kick=0.5, streak=0.1)


def member_configs(c, seed):
    return decks.ensemble_cases(c["members"], seed=2024 + seed % 1000, kick=0.5)


class Fields(dict):
    """The state as it lies on the GPU after the pass, by field name.  A run
    that stays resident reads a field back only where it looks at it, and so
    does this: a value is fetched when it is asked for.  A DGPU_MIXED run's
    state is FP32 on the device, and its values are handed out as that; its
    pressure holds the velocity's FP32 round-off divided by the substep, which
    leaves it 8 to 10 bits, and it is handed out with 8."""

    def __init__(self, owner, names, more=None):
        super().__init__({k: None for k in names})
        self.owner, self.more = owner, more or {}  # the owner lives as long as its fields are looked at
        self.flat = hasattr(owner, "members")
        self.channels = owner.members if self.flat else [owner]
        super().update(self.more)

    def __getitem__(self, k):
        if k in self.more:
            return self.more[k]
        got = [g.get_field(IDS[k]) for g in self.channels]
        a = np.concatenate([a.ravel() for a in got]) if self.flat else got[0]
        if self.channels[0].precision == "mixed":
            a = a.astype(np.float32)
            return torch.from_numpy(a).to(torch.bfloat16) if k == "CP" else a
        return a

    def items(self):
        return [(k, self[k]) for k in self]

    def values(self):
        return [self[k] for k in self]


def prepare(c, seed):
    if c["kind"] == "ensemble":
        cfgs = member_configs(c, seed)
        ens = gpu.GpuEnsemble(cfgs, precision=c["precision"])
        for n, (m, cfg) in enumerate(zip(ens.members, cfgs)):
            load(m, Case(cfg).initial(seed * 64 + n))
            m.synchronize()
        return dict(case=c, ens=ens)
    cfg = config(c)
    if c["kind"] == "transforms":
        g = torch.Generator(device="cuda").manual_seed(seed)
        a = np.zeros(cfg.field_shape())
        a[:, :cfg.nz, :cfg.nx] = torch.randn(cfg.ny + 2, cfg.nz, cfg.nx, dtype=torch.float64, device="cuda",
                                             generator=g).cpu().numpy()
        return dict(case=c, chan=gpu.GpuChannel(cfg), a=a)
    first = Case(cfg).initial(seed)
    chan = gpu.GpuChannel(cfg, precision=c["precision"])
    if c["kind"] == "bridge":
        return dict(case=c, chan=chan, arrays={k: Case(cfg).fortran(v) for k, v in first.items()})
    load(chan, first)
    if c["kind"] == "les":
        chan.set_les(True, True)
    return dict(case=c, chan=chan)


def load(chan, fields):
    for k, v in fields.items():
        chan.set_field(IDS[k], Case(chan.cfg).fortran(v))


def run(s):
    kind = s["case"]["kind"]
    if kind == "ensemble":
        s["ens"].step(1)
        return Fields(s["ens"], STATE)
    g = s["chan"]
    if kind in ("step", "les"):
        g.step(1)
        return Fields(g, STATE)
    if kind == "step_cfl":
        g.step(1, courant_cfl=0.5)
        return Fields(g, STATE, {"DELTA_T": g.delta_t})
    if kind == "stats":
        profiles, ubulk = g.stats_chan()
        return dict(profiles, ubulk=ubulk)
    if kind == "poisson":
        g.poisson_p_chan()
        return Fields(g, ("CP",))
    if kind == "transforms":
        g.fft_xz_to_fourier(s["a"], 0, g.cfg.ny + 1)
        g.fft_xz_to_physical(s["a"], 0, g.cfg.ny + 1)
        return s["a"]
    g.load_state(s["arrays"])
    g.step(1)
    s["arrays"] = g.state()
    return s["arrays"]


def work(c):
    if c["kind"] == "ensemble":
        parts = [work_of("step", cfg, 8 if c["precision"] == "fp64" else 4) for cfg in member_configs(c, 0)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    return work_of(c["kind"], config(c), 4 if c["precision"] == "mixed" else 8)


def work_of(kind, cfg, size):
    modes = (cfg.nkx + 1) * (cfg.tnkz + 1) * (cfg.ny + 2)
    points = cfg.nx * cfg.nz * (cfg.ny + 2)
    transform = 2.5 * points * math.log2(cfg.nx * cfg.nz)  # of one real field
    if kind == "stats":
        return dict(bytes=2.0 * 8 * 5 * modes, flops=60.0 * modes)
    if kind == "poisson":
        return dict(bytes=2.0 * 8 * 5 * modes, flops=15 * transform + 80.0 * modes + 12 * points)
    if kind == "transforms":
        return dict(bytes=4.0 * 8 * points, flops=2 * transform)
    # a time step reads CU1-3, CTH and CP and writes them and CF1-3, CFTH; per
    # substep 4 fields go to physical space and 11 products come back, and four
    # CN systems and the Poisson equation are solved (8 + 6 flops a row and real part)
    transforms, phys, spec = 15, 60, 250
    if kind == "les":  # the strain, the stress, the scalar's eddy flux and the physical solves
        transforms, phys = transforms + 6 + 7 + 4 + 12, phys + 220
    w = dict(bytes=2.0 * size * (5 + 9) * modes, flops=3.0 * (transforms * transform + phys * points + spec * modes))
    if kind == "bridge":  # the host's nine arrays each way
        w["bytes"] = 2.0 * 9 * 8 * (cfg.nx + 2) * (cfg.nz + 2) * (cfg.ny + 2)
    return w


# --------------------------------------------------------------------------
# The path in plain torch, 64 bits: kept modes as [J = 0..NY+1][K][I] complex,
# physical fields as [J][z][x].
# --------------------------------------------------------------------------

def exact(c, seed):
    if c["kind"] == "ensemble":
        parts = []
        for n, cfg in enumerate(member_configs(c, seed)):
            e = Case(cfg)
            f = e.initial(seed * 64 + n)
            for k in range(3):
                e.substep(f, k, cfg.delta_t)
            parts.append({k: e.fortran(v).ravel() for k, v in f.items()})
        return {k: np.concatenate([p[k] for p in parts]) for k in STATE}
    e = Case(config(c))
    if c["kind"] == "transforms":
        g = torch.Generator(device="cuda").manual_seed(seed)
        x = torch.randn(e.ny + 2, e.nz, e.nx, dtype=torch.float64, device="cuda", generator=g)
        a = np.zeros((e.ny + 2, e.nz + 2, e.nx + 2))
        a[:, :e.nz, :e.nx] = e.phys(e.four(x)).cpu().numpy()
        return a
    f = e.initial(seed)
    if c["kind"] == "stats":
        return e.stats(f)
    if c["kind"] == "poisson":
        return {"CP": e.fortran(e.poisson(f))}
    dt = e.cfg.delta_t
    for k in range(3):
        cfl = e.substep(f, k, dt, les=c["kind"] == "les")
    out = {k: e.fortran(v) for k, v in f.items()}
    if c["kind"] == "step_cfl":
        out["DELTA_T"] = cfl(0.5)
    return out


class Case:
    def __init__(self, cfg):
        self.cfg, self.nx, self.ny, self.nz = cfg, cfg.nx, cfg.ny, cfg.nz
        self.mk, self.nkz = cfg.nx // 3 + 1, cfg.nz // 3
        self.mz = 2 * self.nkz + 1
        ny = cfg.ny
        gy = np.zeros(ny + 2)
        gy[1:] = decks.grid_gy(cfg)
        gyf, dy, dyf = np.zeros(ny + 2), np.zeros(ny + 2), np.zeros(ny + 2)
        gyf[1:ny + 1] = 0.5 * (gy[1:ny + 1] + gy[2:ny + 2])
        gyf[0], gyf[ny + 1] = 2 * gyf[1] - gyf[2], 2 * gyf[ny] - gyf[ny - 1]
        dy[1:] = gyf[1:] - gyf[:-1]
        dyf[1:ny + 1] = gy[2:ny + 2] - gy[1:ny + 1]
        dyf[ny + 1] = dyf[ny]
        self.gyf = gyf
        self.dy, self.dyf = dy, dyf
        self.DY, self.DYF, self.GYF = (self.dev(v)[:, None, None] for v in (dy, dyf, gyf))
        slot = np.arange(self.mz)
        kz = np.where(slot <= self.nkz, slot, slot - self.mz)
        self.zslot = self.dev(kz % self.nz)
        self.kx = self.dev(np.arange(self.mk) * (2 * math.pi) / cfg.lx)[None, None, :]
        self.kz = self.dev(kz * (2 * math.pi) / cfg.lz)[None, :, None]
        self.ikx, self.ikz = 1j * self.kx, 1j * self.kz
        self.k2 = self.kx ** 2 + self.kz ** 2

    @staticmethod
    def dev(a):
        return torch.from_numpy(np.ascontiguousarray(a)).cuda()

    # -- transforms and layout --
    def four(self, x):
        y = torch.fft.rfft(x, dim=2, norm="forward")[:, :, :self.mk]
        return torch.fft.fft(y, dim=1, norm="forward")[:, self.zslot, :]

    def phys(self, f):
        y = torch.zeros(f.shape[0], self.nz, self.nx // 2 + 1, dtype=torch.complex128, device="cuda")
        y[:, self.zslot, :self.mk] = f
        return torch.fft.irfft(torch.fft.ifft(y, dim=1, norm="forward"), n=self.nx, dim=2, norm="forward")

    def fortran(self, f):
        a = np.zeros((self.ny + 2, self.nz + 2, self.nx // 2 + 1), dtype=np.complex128)
        a[:, :self.mz, :self.mk] = f.cpu().numpy()
        return a.view(np.float64)

    # -- the start: the decks' profiles with noise, wall conditions, no divergence --
    def initial(self, seed):
        cfg, ny = self.cfg, self.ny
        rand = torch.Generator(device="cuda").manual_seed(seed)

        def noise(scale):
            return scale * (torch.rand(ny + 2, self.nz, self.nx, dtype=torch.float64, device="cuda", generator=rand) - 0.5)

        y = self.GYF
        if cfg.ic == "kh":
            u, th, env = torch.tanh(y), torch.tanh(y), 1.0
        else:
            env = y * (2.0 - y)
            z = torch.arange(self.nz, dtype=torch.float64, device="cuda")[None, :, None] / self.nz
            u, th = env * (1.0 + cfg.streak * torch.sin(4 * math.pi * z)), y / cfg.ly
        f = {"CU1": self.four(u + env * noise(cfg.kick)), "CU2": self.four(env * noise(cfg.kick)),
             "CU3": self.four(env * noise(cfg.kick)), "CTH0": self.four(th + env * noise(cfg.kick)),
             "CP": self.four(noise(cfg.kick)) / (1.0 + self.k2)}
        f["CTH0"][0], f["CTH0"][ny + 1] = 0.0, 0.0
        f["CP"][0], f["CP"][ny + 1] = 0.0, 0.0
        for k in ("CF1", "CF2", "CF3", "CFTH0"):
            f[k] = torch.zeros_like(f["CP"])
        self.walls(f)
        self.project(f)
        return {k: f[k] for k in STATE}

    def walls(self, f):
        """APPLY_BC_VEL with all wall values zero."""
        cfg, ny = self.cfg, self.ny
        for k, lo, hi in (("CU1", cfg.u_bc_ymin, cfg.u_bc_ymax), ("CU3", cfg.w_bc_ymin, cfg.w_bc_ymax)):
            a = f[k]
            a[:2] = a[2] if lo else 0.0
            a[ny:] = a[ny - 1] if hi else 0.0
        v = f["CU2"]
        v[:2] = -v[2]
        v[ny + 1, 0, 0] = -v[ny, 0, 0]

    @staticmethod
    def thomas(L, D, U, V, lo, hi):
        """Rows lo..hi of a tridiagonal system; V becomes the solution."""
        B = [None] * len(V)
        B[lo] = D[lo]
        for j in range(lo + 1, hi + 1):
            m = -L[j] / B[j - 1]
            B[j] = D[j] + m * U[j - 1]
            V[j] += m * V[j - 1]
        V[hi] = V[hi] / B[hi]
        for j in range(hi - 1, lo - 1, -1):
            V[j] = (V[j] - U[j] * V[j + 1]) / B[j]

    def pressure(self, rhs):
        """The Poisson equation of REM_DIV_CHAN and POISSON_P_CHAN, rows 1..NY;
        the pressure's gauge is PHI(0,0) = 0 on row 1."""
        ny, dy, dyf = self.ny, self.dy, self.dyf
        k2 = self.k2[0]
        L, D, U = [None] * (ny + 1), [None] * (ny + 1), [None] * (ny + 1)
        for j in range(2, ny):
            a, b = 1.0 / (dy[j] * dyf[j]), 1.0 / (dy[j + 1] * dyf[j])
            L[j], D[j], U[j] = torch.full_like(k2, a), -k2 - a - b, torch.full_like(k2, b)
        one = torch.ones_like(k2)
        D[1], U[1], L[ny], D[ny], U[ny] = one, -one, one, -one, 0 * one
        U[1][0, 0] = 0.0
        rhs[1], rhs[ny] = 0.0, 0.0
        self.thomas(L, D, U, rhs, 1, ny)
        return rhs

    def project(self, f):
        """REM_DIV_CHAN; returns PHI."""
        ny = self.ny
        div = torch.zeros_like(f["CP"])
        J = slice(1, ny + 1)
        div[J] = self.ikx * f["CU1"][J] + (f["CU2"][2:] - f["CU2"][J]) / self.DYF[J] + self.ikz * f["CU3"][J]
        phi = self.pressure(div)
        f["CU1"][J] -= self.ikx * phi[J]
        f["CU3"][J] -= self.ikz * phi[J]
        f["CU2"][2:ny + 1] -= (phi[2:ny + 1] - phi[1:ny]) / self.DY[2:ny + 1]
        return phi

    def solve(self, V, system, c, nut, t2, mean):
        """One Crank-Nicolson system over J; `nut` is the eddy viscosity in
        physical space or None, `mean` picks where a wall's value goes."""
        cfg, ny, dy, dyf = self.cfg, self.ny, self.dy, self.dyf
        th = system == "TH"
        first = 1 if th and cfg.th_bc_ymin[0] else 2
        L, D, U = [0.0] * (ny + 2), [1.0] * (ny + 2), [0.0] * (ny + 2)
        for j in range(first, ny + 1):
            if system == "U2":
                a, b = c / (dyf[j - 1] * dy[j]), c / (dyf[j] * dy[j])
                if nut is not None:
                    a = a + t2 * 0.5 * (nut[j] + nut[j - 1]) / (dyf[j - 1] * dy[j])
                    b = b + t2 * 0.5 * (nut[j] + nut[j + 1]) / (dyf[j] * dy[j])
            else:
                a, b = c / (dy[j] * dyf[j]), c / (dy[j + 1] * dyf[j])
                if nut is not None:
                    a, b = a + t2 * nut[j] / (dy[j] * dyf[j]), b + t2 * nut[j + 1] / (dy[j + 1] * dyf[j])
            L[j], D[j], U[j] = -a, 1.0 + a + b, -b
        V[0], V[ny + 1] = 0.0, 0.0

        def fixed(j, value):
            L[j], D[j], U[j], V[j] = 0.0, 1.0, 0.0, value * mean
        lo, hi, clo, chi = {
            "U1": (cfg.u_bc_ymin, cfg.u_bc_ymax, 0.0, 0.0), "U2": (0, 0, 0.0, 0.0),
            "U3": (cfg.w_bc_ymin, cfg.w_bc_ymax, 0.0, 0.0),
            "TH": (cfg.th_bc_ymin[0], cfg.th_bc_ymax[0], cfg.th_bc_ymin_c1[0], cfg.th_bc_ymax_c1[0])}[system]
        fixed(0, 0.0)
        fixed(ny + 1, 0.0)
        if system == "U2":
            for j in (1, 2, ny):
                fixed(j, 0.0)
        else:
            if lo:
                L[1], D[1], U[1], V[1] = 0.0, -1.0, 1.0, dy[2] * clo * mean
            else:
                fixed(1, clo)
            if hi:
                L[ny], D[ny], U[ny], V[ny] = -1.0, 1.0, 0.0, dy[ny] * chi * mean
            else:
                fixed(ny, chi)
        if nut is None:
            L, D, U = (torch.tensor([float(x) for x in v], dtype=torch.float64, device="cuda") for v in (L, D, U))
        self.thomas(L, D, U, V, 0, ny + 1)
        return V, (first - 1 if system != "U2" else 1)

    def smagorinsky(self, f, F):
        """les_chan: the SGS force into F, NU_T and the physical U1, U3."""
        cfg, ny, DY, DYF, P = self.cfg, self.ny, self.DY, self.DYF, self.phys
        self.walls(f)
        u, v, w = f["CU1"], f["CU2"], f["CU3"]
        J, G = slice(1, ny + 1), slice(1, ny + 2)
        z = lambda: torch.zeros_like(u)  # noqa: E731
        s11, s22, s33, s13, s12, s23 = z(), z(), z(), z(), z(), z()
        s11[J], s33[J] = self.ikx * u[J], self.ikz * w[J]
        s22[J] = (v[2:] - v[J]) / DYF[J]
        s13[J] = 0.5 * (self.ikz * u[J] + self.ikx * w[J])
        s12[G] = 0.5 * ((u[G] - u[:-1]) / DY[G] + self.ikx * v[G])
        s23[G] = 0.5 * (self.ikz * v[G] + (w[G] - w[:-1]) / DY[G])
        s11, s22, s33, s13, s12, s23 = (P(s) for s in (s11, s22, s33, s13, s12, s23))
        U, W = P(u), P(w)
        dU, dW = (torch.zeros(ny + 2, 1, 1, dtype=torch.float64, device="cuda") for _ in range(2))
        dU[G] = 0.5 * (u[G, :1, :1].real - u[:-1, :1, :1].real) / DY[G]
        dW[G] = 0.5 * (w[G, :1, :1].real - w[:-1, :1, :1].real) / DY[G]
        R = slice(2, ny + 1)
        up = slice(3, ny + 2)
        S = torch.sqrt(2 * s11[R] ** 2 + 4 * (0.5 * (s12[up] + s12[R]) - dU[R] - dU[up]) ** 2 + 4 * s13[R] ** 2
                       + 2 * s22[R] ** 2 + 4 * (0.5 * (s23[up] + s23[R]) - dW[R] - dW[up]) ** 2 + 2 * s33[R] ** 2)
        E, dn = slice(2, ny + 2), slice(1, ny + 1)

        def at_gy(s):
            return (s[E] * DYF[dn] + s[dn] * DYF[E]) / (2 * DY[E])
        T = torch.zeros_like(U)
        T[E] = torch.sqrt(2 * at_gy(s11) ** 2 + 4 * (s12[E] - dU[E]) ** 2 + 4 * at_gy(s13) ** 2 + 2 * at_gy(s22) ** 2
                          + 4 * (s23[E] - dW[E]) ** 2 + 2 * at_gy(s33) ** 2)
        s11[R], s13[R], s33[R] = S * s11[R], S * s13[R], S * s33[R]
        s12[E] = T[E] * (s12[E] - 0.5 * (U[E] - U[dn]) / DY[E])
        s23[E] = T[E] * (s23[E] - 0.5 * (W[E] - W[dn]) / DY[E])
        width = 2 * (cfg.lx / self.nx) * (cfg.lz / self.nz)
        dF, dG = -2 * 0.13 ** 2 * (width * DYF) ** (2 / 3), -2 * 0.13 ** 2 * (width * DY) ** (2 / 3)
        nut = -0.5 * dG * T
        nut[:3], nut[ny:] = 0.0, 0.0
        t11, t13, t33 = (dF * self.four(s) for s in (s11, s13, s33))
        t12, t23 = (dG * self.four(s) for s in (s12, s23))
        A, Ap = slice(2, ny), slice(3, ny + 1)
        F["CF1"][A] -= self.ikx * t11[A] + (t12[Ap] - t12[A]) / DYF[A] + self.ikz * t13[A]
        F["CF3"][A] -= self.ikx * t13[A] + (t23[Ap] - t23[A]) / DYF[A] + self.ikz * t33[A]
        F["CF2"][R] -= self.ikx * t12[R] + self.ikz * t23[R]
        for X, ik in ((U, self.ikx), (W, self.ikz)):
            g = torch.zeros_like(U)
            g[R] = nut[R] * (X[R] - X[1:ny]) / DY[R]
            F["CF2"][R] += ik * self.four(g)[R]
        return nut

    def walls_phys(self, U, V, W):
        """APPLY_BC_VEL_PHYS with all wall values zero."""
        cfg, ny = self.cfg, self.ny
        for a, lo, hi in ((U, cfg.u_bc_ymin, cfg.u_bc_ymax), (W, cfg.w_bc_ymin, cfg.w_bc_ymax)):
            a[:2] = a[2] if lo else 0.0
            a[ny:] = a[ny - 1] if hi else 0.0
        V[:2] = -V[2]
        V[ny + 1] = -V[ny]

    def substep(self, f, k, dt, les=False):
        """RK_CHAN_1; f is updated in place.  Returns COURANT's DELTA_T as a
        function of CFL, from the velocity before the projection."""
        cfg, ny, DY, DYF, P, Q = self.cfg, self.ny, self.DY, self.DYF, self.phys, self.four
        nu, ikx, ikz = cfg.nu, self.ikx, self.ikz
        h = dt * (8 / 15, 2 / 15, 5 / 15)[k]
        t1, t3, t5 = nu * h / 2, (0.0, -17 / 8, -5 / 4)[k] * h, (1.0, 25 / 8, 9 / 4)[k] * h
        first = 1 if cfg.th_bc_ymin[0] else 2
        R, dn, up, T = slice(2, ny + 1), slice(1, ny), slice(3, ny + 2), slice(first, ny + 1)
        Tdn, Tup = slice(first - 1, ny), slice(first + 1, ny + 2)
        rhs = {}
        for u, c, q in (("CU1", "CF1", R), ("CU2", "CF2", R), ("CU3", "CF3", R), ("CTH0", "CFTH0", T)):
            rhs[u] = f[u].clone()
            if k:
                rhs[u][q] += t3 * f[c][q]
        p = f["CP"]
        rhs["CU1"][R] -= h * ikx * p[R]
        rhs["CU3"][R] -= h * ikz * p[R]
        rhs["CU2"][R] -= h * (p[R] - p[dn]) / DY[R]
        if cfg.f_type == 1:
            rhs["CU1"][R, 0, 0] -= h * cfg.px0
        F = {c: torch.zeros_like(p) for c in ("CF1", "CF2", "CF3", "CFTH0")}
        for u, c, q, d in (("CU1", "CF1", R, nu), ("CU2", "CF2", R, nu), ("CU3", "CF3", R, nu),
                           ("CTH0", "CFTH0", T, nu / cfg.pr[0])):
            F[c][q] = -d * self.k2 * f[u][q]
        th = f["CTH0"]
        b = cfg.ri[0] * cfg.grav_y * (th[R] * DYF[dn] + th[dn] * DYF[R]) / (2 * DY[R])
        b[:, 0, 0] = 0.0
        F["CF2"][R] += b
        nut = self.smagorinsky(f, F) if les else None
        U, V, W, H = P(f["CU1"]), P(f["CU2"]), P(f["CU3"]), P(th)
        if les:
            self.walls_phys(U, V, W)
            for ik in (ikx, ikz):
                g = P(ik * th)
                g[0], g[1:] = 0.0, nut[1:] * g[1:]
                F["CFTH0"][T] += ik * Q(g)[T]

        def flux(x, q, a, b_, sel):  # d/dy of U2 times x at GYF rows
            return Q((x[b_] * V[b_] + x[q] * V[b_] - x[q] * V[q] - x[a] * V[q]) / (2 * DYF[q]))
        g = Q(U[R] * W[R])
        F["CF1"][R] -= ikz * g + ikx * Q(U[R] * U[R]) + flux(U, R, dn, up, R)
        F["CF3"][R] -= ikx * g + ikz * Q(W[R] * W[R]) + flux(W, R, dn, up, R)
        gu, gw = ((DYF[R] * x[R] + DYF[dn] * x[dn]) / (2 * DY[R]) * V[R] for x in (U, W))
        vv = (0.25 * (V[R] + V[up]) ** 2 - 0.25 * (V[R] + V[dn]) ** 2) / DY[R]
        F["CF2"][R] -= ikx * Q(gu) + ikz * Q(gw) + Q(vv)
        F["CFTH0"][T] -= ikx * Q(H[T] * U[T]) + ikz * Q(H[T] * W[T]) + flux(H, T, Tdn, Tup, T)
        for c in F:
            q = T if c == "CFTH0" else R
            f[c][q] = F[c][q]
        found = {}
        mean = torch.zeros(self.mz, self.mk, dtype=torch.complex128, device="cuda")
        mean[0, 0] = 1.0
        for system, u, c, q, a, b_, x in (("TH", "CTH0", "CFTH0", T, Tdn, Tup, H), ("U2", "CU2", "CF2", R, dn, up, V),
                                          ("U1", "CU1", "CF1", R, dn, up, U), ("U3", "CU3", "CF3", R, dn, up, W)):
            r, cm = rhs[u], (t1 / cfg.pr[0] if system == "TH" else t1)
            r[q] += t5 * F[c][q]
            y = x if les else f[u]
            if les:
                r = P(r)
            n_up = n_dn = 0.0
            if les:
                n_up, n_dn = (0.5 * (nut[q] + nut[b_]), 0.5 * (nut[q] + nut[a])) if system == "U2" else (nut[b_], nut[q])
            du, dd = (DYF[q], DYF[a]) if system == "U2" else (DY[b_], DY[q])
            r[q] += ((cm + h / 2 * n_up) * (y[b_] - y[q]) / du - (cm + h / 2 * n_dn) * (y[q] - y[a]) / dd) / (
                DY[q] if system == "U2" else DYF[q])
            r, lo = self.solve(r, system, cm, nut, h / 2, torch.ones_like(r[0]) if les else mean)
            if les:
                x[lo:] = r[lo:]
                found[u] = Q(x)
            else:
                found[u] = torch.cat([f[u][:lo], r[lo:]])
        f.update(found)
        speed = [P(f[u])[1:ny + 1].abs().amax(dim=(1, 2)).cpu().numpy() for u in ("CU1", "CU2", "CU3")] if k == 2 else None
        phi = self.project(f)
        f["CP"][R] += phi[R] / h

        def courant(cfl):
            dx, dz = cfg.lx / self.nx, cfg.lz / self.nz
            with np.errstate(divide="ignore"):
                limits = [cfl * dx / speed[0].max(), (cfl * self.dy[1:ny + 1] / speed[1]).min(), cfl * dz / speed[2].max()]
            return float(min([999.0, 0.5 * min(dx, self.dy[1]) ** 2 / nu] + limits))
        return courant

    def poisson(self, f):
        """POISSON_P_CHAN."""
        ny, DYF, GYF, P = self.ny, self.DYF, self.GYF, self.phys
        R, dn, up = slice(2, ny + 1), slice(1, ny), slice(3, ny + 2)
        u, v, w, th = f["CU1"], f["CU2"], f["CU3"], f["CTH0"]
        vc = 0.5 * (v[R] + v[up])
        s = sum(self.four(P(x) ** 2) for x in (self.ikx * u[R], (v[up] - v[R]) / DYF[R], self.ikz * w[R]))
        for a, b in (((u[up] - u[dn]) / (2 * DYF[R]), self.ikx * vc), ((w[up] - w[dn]) / (2 * DYF[R]), self.ikz * vc),
                     (self.ikz * u[R], self.ikx * w[R])):
            s = s + self.four(2 * P(a) * P(b))
        b = self.cfg.ri[0] * (th[up] - th[dn]) / (GYF[up] - GYF[dn])
        b[:, 0, 0] = 0.0
        rhs = torch.zeros_like(u)
        rhs[R] = -(s + b)
        p = self.pressure(rhs)
        out = f["CP"].clone()
        out[1:ny + 1] = p[1:ny + 1]
        return out

    def stats(self, f):
        """SAVE_STATS_CHAN's profiles from sums over the physical points."""
        ny, DY, DYF, GYF, P = self.ny, self.DY, self.DYF, self.GYF, self.phys
        J, dn, up = slice(1, ny + 1), slice(0, ny), slice(2, ny + 2)
        u, v, w, th = (f[k] for k in ("CU1", "CU2", "CU3", "CTH0"))
        mean = {k: f[k][:, :1, :1].real for k in ("CU1", "CU2", "CU3", "CTH0", "CP")}
        U, V, W, H = (P(f[k]) for k in ("CU1", "CU2", "CU3", "CTH0"))
        a, b, c, d = U - mean["CU1"], V - mean["CU2"], W - mean["CU3"], H - mean["CTH0"]
        avg = lambda x: x.mean(dim=(1, 2)).cpu().numpy()  # noqa: E731
        one = lambda x: x[:, 0, 0].cpu().numpy()  # noqa: E731

        def gy(x):
            return (DYF[dn] * x[J] + DYF[J] * x[dn]) / (2 * DY[J])
        vc = 0.5 * (v[up] + v[J])
        vort = ((w[up] - w[dn]) / (2 * DYF[J]) - self.ikz * vc, self.ikz * u[J] - self.ikx * w[J],
                self.ikx * vc - (u[up] - u[dn]) / (2 * DYF[J]))
        out = {"ume": one(mean["CU1"][J]), "vme": one(mean["CU2"][J]), "wme": one(mean["CU3"][J]),
               "urms": np.sqrt(avg(a[J] ** 2)), "vrms": np.sqrt(avg(0.5 * (b[J] ** 2 + b[up] ** 2))),
               "wrms": np.sqrt(avg(c[J] ** 2)), "uv": avg(gy(a) * b[J]), "uw": avg(a[J] * c[J]), "wv": avg(gy(c) * b[J]),
               "cp": one(mean["CP"][J]), "thme": one(mean["CTH0"][J]), "thrms": np.sqrt(avg(d[J] ** 2)),
               "thv": avg(d[J] * 0.5 * (b[J] + b[up])),
               "shear": avg(((U[up] - U[dn]) / (2 * DYF[J])) ** 2 + ((W[up] - W[dn]) / (2 * DYF[J])) ** 2)}
        for k, x in zip(("omega_x", "omega_y", "omega_z"), vort):
            out[k] = np.sqrt(avg(P(x) ** 2))
        for k, m in (("dudy", "CU1"), ("dwdy", "CU3"), ("dthdy", "CTH0")):
            out[k] = one((mean[m][J] - mean[m][dn]) / (GYF[J] - GYF[dn]))
        out["pe_diss"] = avg(P(self.ikx * th[J]) ** 2 + P((th[up] - th[dn]) / (GYF[up] - GYF[dn])) ** 2
                             + P(self.ikz * th[J]) ** 2)
        m = out["ume"]
        out["ubulk"] = float((0.5 * (m[1:] + m[:-1]) * self.dy[2:ny + 1]).sum() / self.cfg.ly)
        return out
