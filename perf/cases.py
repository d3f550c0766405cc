"""Performance cases of the nsPipe time step and the calls around it.

Each case is one call, or one short run of calls, that a user's program makes through the public entry
points (the `nsp` binding of libnsp.so) with its fields on the GPU: time steps from a given state, the
nonlinear term of caller fields, ensembles, monitoring output and remeshing.  Grids and physical
parameters are those of the benchmark and the tests, or generic ones between them.  `exact` restates the
reference's method (grid, tables, banded solves, influence matrix, dealiased products) in plain
numpy and torch at 64 bits, without the library.
"""
import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nspipe-gpu_amd"))
import nsp  # noqa: E402

PREC = {"fp64": nsp.FP64, "mixed": nsp.MIXED, "refined": nsp.MIXED_REFINED}
# kernel forms saved from an autotuner run on the headline grid, as a program keeps them between runs
SAVED = {
    "fp64": {"theta_inv": {"alg": 0, "tl": 16, "nthr": 512, "pad": 0, "ord": 1},
             "theta_fwd": {"alg": 1, "tl": 8, "nthr": 256, "pad": 0, "ord": 1},
             "z_alg": 4, "z_nthr": 512, "z_pad": 1, "z_pf": 0, "s_ord": 1, "nl_chunks": 1},
    "mixed": {"theta_inv": {"alg": 0, "tl": 16, "nthr": 512, "pad": 0, "ord": 1},
              "theta_fwd": {"alg": 1, "tl": 16, "nthr": 256, "pad": 0, "ord": 1},
              "z_alg": 4, "z_nthr": 512, "z_pad": 1, "z_pf": 0, "s_ord": 1, "nl_chunks": 1},
}
NT_PLANS = (64, 96, 128, 192, 384, 768)        # azimuthal sizes with compiled transform plans
NZ_PLANS = (65, 385, 513, 1025, 1537, 3073)    # axial sizes with compiled transform plans
N_HEADLINE = 96 * 384 * 1537
IW, STEN = 3, 7


# ------------------------------------------------------------------------------------------- the cases
def _step(name, nr, nt, nz, form, steps, tuned=False, re=5300.0, lz=2 * math.pi, dt=0.002):
    return {"name": name, "do": "step", "nr": nr, "nt": nt, "nz": nz, "form": form, "steps": steps, "tuned": tuned,
            "re": re, "lz": lz, "dt": dt}


def listed():
    return [
        # the smallest grid of the tests: one step is launches and latency only (runtime-radix transforms)
        _step("step tiny", 16, 8, 9, "fp64", 1, re=500.0, dt=0.01),
        # Re 2000 pipe of length 4 pi R, the small FP64 run (transition studies, regression runs)
        _step("step small fp64", 32, 64, 65, "fp64", 10, re=2000.0, lz=4 * math.pi, dt=0.005),
        # odd, ragged sizes without compiled transform plans
        _step("step ragged fp64", 45, 80, 161, "fp64", 2, re=3000.0, dt=0.002),
        # Re 5300 turbulent pipe, the ordinary run: FP64, and refined mixed for long runs
        _step("step medium fp64", 64, 192, 385, "fp64", 4),
        _step("step medium refined", 64, 192, 385, "refined", 4),
        # Re 11700 pipe of length 10 pi R with saved kernel forms: the benchmark's headline run, both forms
        _step("step headline fp64", 96, 384, 1537, "fp64", 2, True, re=11700.0, lz=10 * math.pi, dt=0.001),
        _step("step headline mixed", 96, 384, 1537, "mixed", 3, True, re=11700.0, lz=10 * math.pi, dt=0.001),
        # the planes of the Re 19000 pipe (768 x 3073) on fewer levels, default kernel forms
        _step("step wide mixed", 24, 768, 3073, "mixed", 1, re=19000.0, lz=4 * math.pi, dt=0.0005),
        # predictability ensemble at Re 2000, L = 50R: members of two sizes in one launch per stage
        {"name": "ensemble mixed", "do": "ensemble", "nr": 48, "nt": 96, "nz": 513, "nr2": 64, "nt2": 128, "nz2": 1025,
         "members": 3, "form": "mixed", "steps": 2, "tuned": True, "re": 2000.0, "lz": 50.0, "dt": 0.005},
        # the nonlinear term of a caller's own fields (a drop-in for the reference's nonlinear())
        {"name": "nonlinear fp64", "do": "nonlinear", "nr": 64, "nt": 128, "nz": 1025, "form": "fp64", "tuned": False,
         "re": 5300.0, "lz": 50.0, "dt": 0.002},
        # monitoring between output intervals: diagnostics, cross sections, mean profile, a physical field
        {"name": "monitor fp64", "do": "monitor", "nr": 48, "nt": 96, "nz": 513, "form": "fp64", "tuned": False,
         "re": 2000.0, "lz": 50.0, "dt": 0.005},
        # a state moved to a finer grid before a run at higher resolution
        {"name": "remesh fp64", "do": "remesh", "nr": 48, "nt": 96, "nz": 513, "nr2": 64, "nt2": 192, "nz2": 1025,
         "form": "fp64", "tuned": False, "re": 2000.0, "lz": 50.0, "dt": 0.005},
    ]


def _smooth(n):
    for p in (2, 3, 5):
        while n % p == 0:
            n //= p
    return n == 1


def _logint(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _plan_grid(rng, most, nt_max=768):
    while True:
        nt = rng.choice([n for n in NT_PLANS if n <= nt_max])
        nz = rng.choice(NZ_PLANS)
        if nt * nz * 9 <= most:
            return _logint(rng, 9, min(96, most // (nt * nz))), nt, nz


def _free_grid(rng):
    while True:
        nt, nz = 2 * _logint(rng, 4, 72), 2 * _logint(rng, 4, 160) + 1
        if _smooth(3 * nt // 2) and _smooth(3 * (nz - 1) // 2):
            return _logint(rng, 9, 64), nt, nz


def draw(rng):
    do = rng.choice(["step"] * 6 + ["ensemble", "nonlinear", "monitor", "remesh"])
    par = {"re": float(_logint(rng, 500, 19000)), "lz": rng.choice([2, 4, 10]) * math.pi, "dt": rng.choice([0.001, 0.002])}
    if do == "step":
        form = rng.choice(["fp64", "fp64", "mixed", "refined"])
        tuned = rng.random() < 0.4
        if form == "fp64" and not tuned and rng.random() < 0.4:
            nr, nt, nz = _free_grid(rng)
        else:
            nr, nt, nz = _plan_grid(rng, N_HEADLINE // (1 if form == "mixed" else 2), 384 if tuned else 768)
        return {"do": do, "nr": nr, "nt": nt, "nz": nz, "form": form, "tuned": tuned,
                "steps": 1 if nr * nt * nz > 2_000_000 else rng.randint(1, 4), **par}
    if do == "ensemble":
        nr, nt, nz = _plan_grid(rng, 2_500_000, 384)
        nr2, nt2, nz2 = _plan_grid(rng, 5_000_000, 384)
        return {"do": do, "nr": nr, "nt": nt, "nz": nz, "nr2": nr2, "nt2": nt2, "nz2": nz2, "members": rng.randint(2, 5),
                "form": rng.choice(["fp64", "mixed"]), "tuned": rng.random() < 0.5, "steps": 1, **par}
    if do == "nonlinear":
        form = rng.choice(["fp64", "mixed"])
        nr, nt, nz = _plan_grid(rng, 16_000_000) if form == "mixed" or rng.random() < 0.6 else _free_grid(rng)
        return {"do": do, "nr": nr, "nt": nt, "nz": nz, "form": form, "tuned": False, **par}
    nr, nt, nz = _plan_grid(rng, 4_000_000, 384) if rng.random() < 0.5 else _free_grid(rng)
    case = {"do": do, "nr": nr, "nt": nt, "nz": nz, "form": "fp64", "tuned": False, **par}
    if do == "remesh":
        nr2, nt2, nz2 = _plan_grid(rng, 8_000_000, 384) if rng.random() < 0.5 else _free_grid(rng)
        case.update(nr2=nr2, nt2=nt2, nz2=nz2)
    return case


def _grid(case, which=""):
    return case["nr" + which], case["nt" + which], case["nz" + which]


def _members(case):
    return [_grid(case)] * case["members"] + [_grid(case, "2")] * case["members"]


# ------------------------------------------------------------------------------------ inputs and passes
def _initial(shape, lz, r, seed):
    """Poiseuille flow plus divergence-free, no-slip noise with a k^(-5/3) envelope over two thirds of the
    modes (rms 0.075): a turbulent-like field.  The same values for the library and for `exact`."""
    nr, nt, nz = shape
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    gen = torch.Generator(device=dev).manual_seed(seed)
    m = torch.fft.fftfreq(nt, 1.0 / nt, dtype=torch.float64, device=dev)[:, None]
    kz = (2 * math.pi / lz) * torch.arange(nz, dtype=torch.float64, device=dev)[None, :]
    on = (m.abs() <= nt / 3) & (kz > 0) & (kz <= kz[0, -1] * 2 / 3)
    env = torch.where(on, (kz * kz + m * m).clamp_min(1e-30) ** (-5.0 / 6.0), 0.0)
    a, b = (env * torch.randn(nt, nz, dtype=torch.complex128, device=dev, generator=gen) for _ in range(2))
    r = torch.as_tensor(r, dtype=torch.float64, device=dev)[:, None, None]
    q = m.abs()[None]
    w = (1 - r * r) ** 2
    s = torch.where(q > 0, r ** (q - 1), r) * w  # regular at the axis
    z = torch.where(q > 0, -4 * r ** q * (1 - r * r), 2 * w - 4 * r * r * (1 - r * r)) / kz.clamp_min(1e-30)[None]
    u = [s * a, s * torch.where(m == 0, b, 1j * torch.sign(m) * a), z * (1j * a)]
    dr = torch.as_tensor(np.gradient(r.flatten().cpu().numpy()), device=dev)
    e = sum((4 * r[:, 0, 0] * dr * v.abs().square().sum((1, 2))).sum() for v in u)
    u = [v * (0.075 / math.sqrt(float(e))) for v in u]
    u[2][:, 0, 0] += (1 - r * r)[:, 0, 0]
    return [v.contiguous() for v in u]


def _ptrs(fields):
    return [f.data_ptr() for f in fields]


def _pipe(case, which=""):
    nr, nt, nz = _grid(case, which)
    p = nsp.Pipe(nr, nt, nz, case["lz"], case["re"], case["dt"], precision=PREC[case["form"]])
    if case["tuned"]:
        p.set_tuning(SAVED["fp64" if case["form"] == "fp64" else "mixed"])
    return p


def prepare(case, seed):
    s = {"case": case}
    if case["do"] == "ensemble":
        grids = _members(case)
        s["ens"] = nsp.Ensemble([dict(nr=g[0], nt=g[1], nz=g[2], lz=case["lz"], re=case["re"], dt=case["dt"],
                                      precision=PREC[case["form"]]) for g in grids])
        pipes = s["ens"].members
        if case["tuned"]:
            for p in pipes:
                p.set_tuning(SAVED[case["form"]])
    else:
        grids, pipes = [_grid(case)], [_pipe(case)]
    s["pipes"] = pipes
    s["in"] = [_initial(g, case["lz"], p.tables()["r"], seed * 100 + j) for j, (g, p) in enumerate(zip(grids, pipes))]
    s["out"] = [[torch.empty_like(f) for f in u] for u in s["in"]]
    if case["do"] in ("monitor", "remesh"):
        torch.cuda.synchronize()
        pipes[0].set_state_device(*_ptrs(s["in"][0]))
    if case["do"] == "monitor":
        s["phys"] = torch.empty(pipes[0].physical_shape, dtype=torch.float64, device="cuda")
    if case["do"] == "remesh":
        s["fine"] = _pipe(case, "2")
        s["out"] = [[torch.empty(s["fine"].shape, dtype=torch.complex128, device="cuda") for _ in range(3)]]
    torch.cuda.synchronize()
    return s


def _kept(case, pipe, fields):
    """A field as the program keeps it: the mixed forms carry single precision, so it is kept in complex64
    (converted on the pipe's own stream, which orders it against the pipe's next call)."""
    if case["form"] == "fp64":
        return fields
    with torch.cuda.stream(torch.cuda.ExternalStream(pipe.stream())):
        return [f.to(torch.complex64) for f in fields]


def run(s):
    case, pipes = s["case"], s["pipes"]
    if case["do"] in ("step", "ensemble"):
        for p, u in zip(pipes, s["in"]):
            p.set_state_device(*_ptrs(u))
        n_it, _, flags = (s["ens"] if "ens" in s else pipes[0]).step(case["steps"])
        for p, u in zip(pipes, s["out"]):
            p.get_state_device(*_ptrs(u))
        return {"fields": [_kept(case, p, u) for p, u in zip(pipes, s["out"])], "n_it": n_it, "flags": flags}
    if case["do"] == "nonlinear":
        st = nsp.lib().nsp_nonlinear(pipes[0].h, *_ptrs(s["in"][0]), *_ptrs(s["out"][0]), nsp.DEVICE)
        if st:
            raise nsp.NspError(nsp.lib().nsp_last_error().decode())
        return {"fields": [_kept(case, pipes[0], s["out"][0])]}
    if case["do"] == "remesh":
        nsp.remesh(s["fine"], pipes[0])
        s["fine"].get_state_device(*_ptrs(s["out"][0]))
        return {"fields": s["out"]}
    p = pipes[0]
    q, u2 = p.cross_sections()
    if nsp.lib().nsp_physical_field(p.h, 2, s["phys"].data_ptr(), nsp.DEVICE):
        raise nsp.NspError(nsp.lib().nsp_last_error().decode())
    return {"diag": p.diagnostics(), "q": q, "u2": u2, "profile": p.mean_profile(), "phys": s["phys"]}


def _transform_flops(g, inverse_t, inverse_z, forward):
    nr, nt, nz = g
    ntp, nzf = 3 * nt // 2, 3 * (nz - 1)
    theta, z = 5.0 * ntp * math.log2(ntp) * nz, 2.5 * nzf * math.log2(nzf) * ntp
    return nr * ((inverse_t + forward) * theta + (inverse_z + forward) * z)


def work(case):
    """Per step the state is read and written once (it does not fit on the chip) and twice evaluated (predictor
    and one corrector: 12 inverse and 3 forward transforms and about 500 operations of the solves per value)."""
    n = [math.prod(_grid(case))]
    if case["do"] in ("step", "ensemble"):
        grids = _members(case) if case["do"] == "ensemble" else [_grid(case)]
        k, total = case["steps"], sum(math.prod(g) for g in grids)
        return {"bytes": 96.0 * total * k, "flops": k * 2 * (sum(_transform_flops(g, 9, 12, 3) for g in grids) + 500.0 * total)}
    if case["do"] == "nonlinear":
        return {"bytes": 96.0 * n[0], "flops": _transform_flops(_grid(case), 9, 12, 3) + 60.0 * n[0]}
    if case["do"] == "remesh":
        fine = math.prod(_grid(case, "2"))
        return {"bytes": 48.0 * (n[0] + fine), "flops": 72.0 * fine}
    nr, nt, nz = _grid(case)
    phys = nr * (3 * nt // 2) * (3 * nz - 1)
    return {"bytes": 48.0 * n[0] + 8.0 * phys, "flops": _transform_flops(_grid(case), 3, 3, 0) + 100.0 * n[0] + 12.0 * phys}


# -------------------------------------------------------------------------- the method at 64 bits
def _fd_weights(x, x0, order):
    """Fornberg's weights at x0 of the derivatives 0..order from the points x: [order + 1][len(x)]."""
    n = len(x)
    c = np.zeros((n, order + 1))
    c[0, 0], c1, c4 = 1.0, 1.0, x[0] - x0
    for i in range(1, n):
        top, c2, c5, c4 = min(i, order), 1.0, c4, x[i] - x0
        for j in range(i):
            c3 = x[i] - x[j]
            c2 *= c3
            if j == i - 1:
                for k in range(top, 0, -1):
                    c[i, k] = c1 * (k * c[i - 1, k - 1] - c5 * c[i - 1, k]) / c2
                c[i, 0] = -c1 * c5 * c[i - 1, 0] / c2
            for k in range(top, 0, -1):
                c[j, k] = (c4 * c[j, k] - k * c[j, k - 1]) / c3
            c[j, 0] = c4 * c[j, 0] / c3
        c1 = c2
    return c.T


def _radii(nr):
    n = nr + int(math.sqrt(nr))
    r = 0.5 * (1 + np.cos(math.pi * (nr - 1 - np.arange(nr)) / n))
    for _ in range(10):
        d = 1.5 * r[0] - 0.5 * r[1]
        r = r * (1 + d) - d
    return r


@functools.lru_cache(maxsize=4)
def _tables(nr):
    """r, the first and second derivative matrices of functions even [0] and odd [1] in r, and the weights of
    2 int f r dr (Taylor expansions over the neighbouring cells)."""
    r = _radii(nr)
    x = np.concatenate([-r[IW - 1::-1], r])
    edge = np.concatenate([[0.0], r, [r[-1]]])
    D, D2, rdr = np.zeros((2, nr, nr)), np.zeros((2, nr, nr)), np.zeros(nr)
    for i in range(nr):
        pts = np.arange(i, min(i + 2 * IW, nr + IW - 1) + 1)
        c = _fd_weights(x[pts], r[i], len(pts) - 1)
        for j, p in enumerate(pts):
            col, mirror = (p - IW, False) if p >= IW else (IW - 1 - p, True)
            for par in range(2):
                sign = -1.0 if mirror and par else 1.0
                D[par, i, col] += sign * c[1, j]
                D2[par, i, col] += sign * c[2, j]
            for k in range(len(pts)):
                cell = ((edge[i + 2] - r[i]) ** (k + 1) - (edge[i] - r[i]) ** (k + 1)) / math.factorial(k + 1)
                rdr[col] += cell * r[i] * c[k, j]
    return r, D, D2, rdr


class _Method:
    """The reference's operators and solves on one grid, vectorised over the modes."""

    def __init__(self, shape, case):
        self.nr, self.nt, self.nz = shape
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.re, self.dt, self.c = case["re"], case["dt"], 0.51
        r, D, D2, rdr = _tables(self.nr)
        t = lambda v: torch.as_tensor(v, dtype=torch.float64, device=self.dev)  # noqa: E731
        self.r, self.rdr, self.D = t(r), t(rdr), t(D)
        Lu = D2 + D / r[None, :, None]
        Lp = Lu.copy()
        Lu[:, -1], Lu[:, -1, -1] = 0.0, 1.0  # Dirichlet wall row
        Lp[:, -1] = D[:, -1]                 # Neumann wall row
        self.Lu, self.Lp = t(Lu), t(Lp)
        self.band = {"u": Lu, "p": Lp}
        self.m = torch.fft.fftfreq(self.nt, 1.0 / self.nt, dtype=torch.float64, device=self.dev)[:, None].expand(self.nt, self.nz)
        self.kz = (2 * math.pi / case["lz"]) * torch.arange(self.nz, dtype=torch.float64, device=self.dev).expand(self.nt, self.nz)
        self.rr = self.r[:, None, None]

    def apply(self, T, f, flag):
        """T[parity] along r; the parity of a field is that of |m|, swapped where flag is 1 (u_r, u_theta)."""
        out = torch.empty_like(f)
        for odd in range(2):
            rows = f[:, odd::2].reshape(self.nr, -1)
            y = T[abs(odd - flag)] @ torch.view_as_real(rows).reshape(self.nr, -1)
            out[:, odd::2] = torch.view_as_complex(y.reshape(self.nr, -1, 2)).reshape(out[:, odd::2].shape)
        return out

    def nonlinear(self, u):
        nr, nt, nz, half = self.nr, self.nt, self.nz, self.nt // 2
        ntp, nzf = 3 * nt // 2, 3 * (nz - 1)
        dr = [self.apply(self.D, u[0], 1), self.apply(self.D, u[1], 1), self.apply(self.D, u[2], 0)]
        out = [torch.zeros_like(f) for f in u]
        for i in range(nr):
            rad = float(self.r[i])
            lev = [f[i] for f in u]
            spec = torch.stack(lev + [d[i] for d in dr] + [1j * self.m * f / rad for f in lev] + [1j * self.kz * f for f in lev])
            pad = torch.zeros(12, ntp, nz, dtype=torch.complex128, device=self.dev)
            pad[:, :half], pad[:, ntp - half:] = spec[:, :half], spec[:, half:]
            row = torch.fft.ifft(pad, dim=1, norm="forward")
            row[:, :, 0].imag = 0.0
            f = torch.fft.irfft(row, n=nzf, dim=2, norm="forward")
            ur, ut, uz = f[0], f[1], f[2]
            v = [ur * f[3 + c] + ut * f[6 + c] + uz * f[9 + c] for c in range(3)]
            v[0] -= ut * ut / rad
            v[1] += ur * ut / rad
            w = torch.fft.fft(torch.fft.rfft(-torch.stack(v), dim=2)[:, :, :nz], dim=1) / (float(ntp) * nzf)
            for c in range(3):
                out[c][i] = torch.cat([w[c, :half], w[c, ntp - half:]])
                out[c][i, half] = 0
                out[c][i, :, nz - 1] = 0
        wall = (self.D[0, -1] * u[2][:, 0, 0].real).sum()
        out[2][:, 0, 0] -= (2.0 / self.re) * wall
        return out

    def diag(self, kind):
        d = -self.kz ** 2 - (self.m / self.rr) ** 2
        return d if kind > 1 else d - 1 / self.rr ** 2 - (2.0 if kind == 0 else -2.0) * self.m / self.rr ** 2

    def laplace(self, f, kind):
        return self.apply(self.Lu, f, 1 if kind < 2 else 0) + self.diag(kind) * f

    @functools.lru_cache(maxsize=None)
    def factors(self, kind):
        """Banded LU rows, kind 0 u+, 1 u-, 2 uz (Helmholtz), 3 pressure; vectorised over the modes."""
        nr, vel, a = self.nr, kind < 3, self.c / self.re
        T = self.band["u" if vel else "p"]
        odd = self.m.abs() % 2
        flag = 1 if kind < 2 else 0
        dg = self.diag(kind)
        lower, upper = [], []
        for i in range(nr):
            cols = range(max(0, i - IW), min(nr, i + IW + 1))
            row = {}
            for j in cols:
                e = odd * float(T[1 - flag, i, j]) + (1 - odd) * float(T[flag, i, j])
                if i < nr - 1:
                    if j == i:
                        e = e + dg[i]
                    if vel:
                        e = -a * e + (1.0 / self.dt if j == i else 0.0)
                elif kind == 3:  # the mean pressure is fixed at the wall
                    e[0, 0] = 1.0 if j == i else 0.0
                row[j] = e
            mult = {}
            for j in cols:
                if j < i:
                    mult[j] = row[j] / upper[j][j]
                    for k in upper[j]:
                        if k > j:
                            row[k] = row[k] - mult[j] * upper[j][k]
            lower.append(mult)
            upper.append({j: row[j] for j in cols if j >= i})
        return lower, upper

    def solve(self, kind, rhs):
        lower, upper = self.factors(kind)
        x = rhs.clone()
        for i in range(self.nr):
            for j, l in lower[i].items():
                x[i] -= l * x[j]
        for i in range(self.nr - 1, -1, -1):
            for j, w in upper[i].items():
                if j > i:
                    x[i] -= w * x[j]
            x[i] /= upper[i][i]
        return x

    def divergence(self, u):
        return self.apply(self.D, u[0], 1) + u[0] / self.rr + 1j * self.m * u[1] / self.rr + 1j * self.kz * u[2]

    def gradient(self, p):
        return [self.apply(self.D, p, 0), 1j * self.m * p / self.rr, 1j * self.kz * p]

    @staticmethod
    def pm(u):
        return [u[0] + 1j * u[1], u[0] - 1j * u[1], u[2]]

    @staticmethod
    def rt(v):
        return [0.5 * (v[0] + v[1]), -0.5j * (v[0] - v[1]), v[2]]

    @functools.lru_cache(maxsize=None)
    def influence(self):
        """Homogeneous solutions with unit wall values (u+, u-, uz, pressure gradient) and the inverse of
        their wall conditions: column of the wall divergence."""
        unit = torch.zeros(self.nr, self.nt, self.nz, dtype=torch.complex128, device=self.dev)
        unit[-1] = 1.0
        zero = torch.zeros_like(unit)
        h = [[self.solve(0, unit), zero, zero], [zero, self.solve(1, unit), zero], [zero, zero, 1j * self.solve(2, unit)],
             self.pm(self.gradient(self.solve(3, -unit)))]
        M = torch.stack([torch.stack([g[c][-1] for g in h], -1) for c in range(3)]
                        + [torch.stack([self.divergence(self.rt(g))[-1] for g in h], -1)], -2)
        M[0, 0] = torch.eye(4, dtype=M.dtype, device=self.dev)
        # rows 0..2 are c_j h_j + c_3 p_j = 0: eliminate them by hand
        d = [M[..., j, j] for j in range(3)]
        c3 = 1.0 / (M[..., 3, 3] - sum(M[..., 3, j] * M[..., j, 3] / d[j] for j in range(3)))
        coef = [-c3 * M[..., j, 3] / d[j] for j in range(3)] + [c3]
        for v in coef:
            v[0, 0] = 0.0  # the mean flow has no wall divergence to correct
        return h, coef

    @functools.lru_cache(maxsize=None)
    def flux_profile(self):
        one = torch.ones(self.nr, self.nt, self.nz, dtype=torch.complex128, device=self.dev)
        one[-1] = 0.0
        uc = self.solve(2, one)[:, 0, 0].real.clone()
        return uc, (self.rdr * uc).sum()

    def advance(self, rhs):
        """One sweep: pressure, velocity solves, wall correction, flux (rhs in the +/- form)."""
        f = self.rt(rhs)
        dv = self.divergence(f)
        dv[-1] = 0
        v = self.pm([a - b for a, b in zip(f, self.gradient(self.solve(3, dv)))])
        for a in v:
            a[-1] = 0
        v = [self.solve(k, v[k]) for k in range(3)]
        h, coef = self.influence()
        wall = self.divergence(self.rt(v))[-1]
        v = [v[c] + sum(-wall * coef[j] * h[j][c] for j in range(4)) for c in range(3)]
        u = self.rt(v)
        u[0][:, 0, 0] = 0
        u[1][:, 0, 0].imag = 0
        u[2][:, 0, 0].imag = 0
        uc, qc = self.flux_profile()
        u[2][:, 0, 0] += (0.5 - (self.rdr * u[2][:, 0, 0].real).sum()) / qc * uc
        return u

    def step(self, u):
        N = self.pm(self.nonlinear(u))
        w = self.pm(u)
        E = [w[k] / self.dt + (1 - self.c) * (self.laplace(w[k], k) / self.re + N[k]) for k in range(3)]
        it, err, new = 0, math.inf, self.advance([e + self.c * n for e, n in zip(E, N)])
        while it < 10 and err > 5e-8:
            old = new
            new = self.advance([e + self.c * n for e, n in zip(E, self.pm(self.nonlinear(old)))])
            err = float(max((a - b).abs().square().max() for a, b in zip(old, new)) / max(a.abs().square().max() for a in old))
            it += 1
        return new, it

    def physical(self, f):
        half, ntp, nzf = self.nt // 2, 3 * self.nt // 2, 3 * (self.nz - 1)
        out = torch.zeros(self.nr, ntp, nzf + 2, dtype=torch.float64, device=self.dev)
        for i in range(self.nr):
            pad = torch.zeros(ntp, self.nz, dtype=torch.complex128, device=self.dev)
            pad[:half], pad[ntp - half:] = f[i, :half], f[i, half:]
            row = torch.fft.ifft(pad, dim=0, norm="forward")
            row[:, 0].imag = 0.0
            out[i, :, :nzf] = torch.fft.irfft(row, n=nzf, dim=1, norm="forward")
        return out

    def monitor(self, u):
        phys = [self.physical(f) for f in u]
        nzf = 3 * (self.nz - 1)
        q, u2 = ((self.rdr[:, None] * f.mean(1)[:, :nzf]).sum(0) for f in (phys[0] ** 2 + phys[1] ** 2, phys[2] ** 2))
        prof = u[2][:, 0, 0].real.clone()
        x = self.r[:IW + 1].cpu().numpy()
        dr0 = torch.as_tensor(_fd_weights(x, 0.0, 0)[0], device=self.dev)
        w = torch.full((self.nz,), 2.0, dtype=torch.float64, device=self.dev)
        w[0] = 1.0
        ke = 0.5 * sum(((f.abs().square() * w).sum((1, 2)) * self.rdr).sum() for f in u)
        diag = {"u_cl": float((dr0 * prof[:IW + 1]).sum()), "u_tau": math.sqrt(abs(float((self.D[0, -1] * prof).sum())) / self.re),
                "ke": float(ke), "div_l2": None, "wall_max": None, "wall_div_max": None, "flux": float((self.rdr * prof).sum())}
        # q: the periodic three-point rule sums to the plain mean over theta
        return {"diag": diag, "q": q, "u2": u2, "profile": prof, "phys": phys[2]}


def _remesh(u, coarse, fine):
    """6-point Lagrange interpolation through the axis; modes cut or padded; the mean mode's imaginary parts and
    radial velocity dropped.  A mirrored point at stencil position j is added to column 2 - j."""
    ro, rn = _radii(coarse[0]), _radii(fine[0])
    x = np.concatenate([-ro[IW - 1::-1], ro])
    R = np.zeros((2, fine[0], coarse[0]))
    R[:, -1, -1] = 1.0
    for i in range(fine[0] - 1):
        a = int(np.argmax(x >= rn[i])) - IW
        pts = np.arange(a, min(len(x) - 1, a + 2 * IW - 1) + 1)
        for j, (p, c) in enumerate(zip(pts, _fd_weights(x[pts], rn[i], 0)[0])):
            if p < IW:
                R[0, i, IW - 1 - j] += c
                R[1, i, IW - 1 - j] -= c
            else:
                R[:, i, p - IW] += c
    nt, nz = min(coarse[1], fine[1]) // 2, min(coarse[2], fine[2])
    out = []
    for c, f in enumerate(u):
        g = torch.zeros(*fine, dtype=torch.complex128, device=f.device)
        for m in range(-nt, nt):
            w = torch.as_tensor(R[abs(abs(m) % 2 - (1 if c < 2 else 0))], device=f.device)
            src = f[:, m % coarse[1], :nz].contiguous()
            y = w @ torch.view_as_real(src).reshape(coarse[0], -1)
            g[:, m % fine[1], :nz] = torch.view_as_complex(y.reshape(fine[0], nz, 2))
        g[:, 0, 0] = g[:, 0, 0].real if c else 0
        out.append(g)
    return out


def exact(case, seed):
    if case["do"] == "ensemble":
        grids = _members(case)
    else:
        grids = [_grid(case)]
    fields, n_it = [], []
    for j, g in enumerate(grids):
        u = _initial(g, case["lz"], _radii(g[0]), seed * 100 + j)
        if case["do"] == "remesh":
            return {"fields": [_remesh(u, g, _grid(case, "2"))]}
        M = _Method(g, case)
        if case["do"] == "monitor":
            return M.monitor(u)
        if case["do"] == "nonlinear":
            u = M.nonlinear(u)
        else:
            for _ in range(case["steps"]):
                u, it = M.step(u)
                n_it.append(it)
        fields.append(u)
        M.factors.cache_clear(), M.influence.cache_clear(), M.flux_profile.cache_clear()
    return {"fields": fields, "n_it": None, "flags": None}
