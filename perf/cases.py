"""The work a user of this package has it do, as cases that can be timed: each case is a plain
dict, `prepare` makes what the user's program has in hand before the call, `run` is one pass
through public entry points, `work` what such a pass cannot do without, and `exact` the same
results from plain torch/numpy in 64 bits (no code of this package).

Kinds:
  atom      one atom's response through the drop-in C API (TDSE_DLL.call1DTDSE): host arrays in
            and out, as 1DTDSE/PythonTDSE.py calls it
  batch     propagate_batch: a few (r, z) points of a beam on one grid, called directly
  plan      BatchPlan.replay: a whole beam on one grid, prepared once and replayed
  uneven    BatchPlan.replay over instances of different grids, durations and wavelengths
  gradient  TDSEDipole and harmonic_yield, forward and backward
  farm      farm.run: a CUPRAD field cube (SI, float32) to the merged outputs
  far       Hankel_long on sources in device memory, results on the host
  grid      hankel.gridded: the matrix-core contractions, device tensors in and out
  plane     HankelTransform: one plane, host arrays in and out
"""
import math

import numpy as np
import torch

from mma_amd import adjoint, farm, hankel, tdse, workloads as W
from mma_amd.ctdse import TDSE_DLL, inputs_def, outputs_def

A, E_GUESS = W.SOFT_COULOMB_A["Ar"], W.SOFT_COULOMB_E["Ar"]
X_INT = 2.0
ROWS = tdse.OUTPUT_ROWS


def listed():
    return [
        # one plane of an XUV field looked at on a screen: the smallest call, all launch and copy
        dict(name="plane", kind="plane", no=64, nr=200, nrho=301, near=True),
        # the reference's own entry point at its default grid and a 10-cycle 800 nm pulse
        dict(name="atom", kind="atom", num_r=16000, dx=0.1, dt=0.25, cycles=10),
        # a radial scan of one plane of the beam: fewer instances than the chip has room for
        dict(name="batch-48", kind="batch", n=48, num_r=16000, dx=0.1, dt=0.25, cycles=5),
        # the same on an odd, smaller grid, with more instances than compute units
        dict(name="batch-300-odd", kind="batch", n=300, num_r=6001, dx=0.1, dt=0.25, cycles=4),
        # the focused beam at full duration, 64 radii x 32 planes
        dict(name="plan-2048", kind="plan", n=2048, num_r=16000, dx=0.1, dt=0.25, cycles=10),
        # members of the uneven workload (Nx 4001-32001, 6-20 cycles, 800-1800 nm)
        dict(name="uneven-384", kind="uneven", n=384, nr_lo=2000, nr_hi=16000, cyc_lo=6, cyc_hi=20),
        # a gradient of the harmonic yield on the gradient workload's grid
        dict(name="gradient-512", kind="gradient", n=512, num_r=8000, dx=0.1, dt=0.1, nt=3000, cycles=2),
        # the task farm on a coarsened field cube, the field refined threefold
        dict(name="farm", kind="farm", nz=8, nr=16, num_r=8000, dx=0.1, dt=0.25, dt_field=0.6, cycles=4),
        # the far field in the default precision: a window of harmonics, and the whole plateau
        dict(name="far-small", kind="far", nz=64, no=300, nr=256, nrho=512, contraction="fp64", cumulative=False,
             c64=False),
        dict(name="far-large", kind="far", nz=256, no=768, nr=512, nrho=1024, contraction="fp64", cumulative=False,
             c64=False),
        # the build-up of the far field along the cell (cumulative outputs)
        dict(name="far-cumulative", kind="far", nz=40, no=200, nr=250, nrho=256, contraction="fp64", cumulative=True,
             c64=False),
        # the whole plateau on the matrix cores, sources in single precision
        dict(name="grid-bf16x3", kind="grid", nz=256, no=2048, nr=512, nrho=1024, contraction="bf16x3-mfma", c64=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["plane", "atom", "batch", "batch", "plan", "uneven", "gradient", "farm", "far", "far", "grid"])
    if kind == "plane":
        return dict(kind=kind, no=_log(rng, 8, 400), nr=_log(rng, 40, 1500), nrho=_log(rng, 20, 1000),
                    near=rng.random() < 0.8)
    if kind == "atom":
        return dict(kind=kind, num_r=_log(rng, 1500, 32000), dx=rng.choice([0.1, 0.2]), dt=0.25,
                    cycles=rng.randint(2, 10))
    if kind in ("batch", "plan"):
        c = dict(kind=kind, n=_log(rng, 1, 1500), num_r=_log(rng, 1500, 32000), dx=rng.choice([0.1, 0.2]), dt=0.25,
                 cycles=rng.randint(1, 8))
        while _pt_steps(c) > 1.4e11:
            c["n"] = c["n"] // 2
        return c
    if kind == "uneven":
        lo = _log(rng, 1000, 6000)
        return dict(kind=kind, n=_log(rng, 20, 300), nr_lo=lo, nr_hi=rng.randint(lo + 500, 16000), cyc_lo=rng.randint(3, 6),
                    cyc_hi=rng.randint(8, 20))
    if kind == "gradient":
        return dict(kind=kind, n=_log(rng, 2, 600), num_r=_log(rng, 1500, 16000), dx=0.1, dt=rng.choice([0.1, 0.25]),
                    nt=_log(rng, 1000, 2500), cycles=1)
    if kind == "farm":
        return dict(kind=kind, nz=rng.randint(2, 10), nr=rng.randint(3, 24), num_r=_log(rng, 2000, 16000), dx=0.1,
                    dt=0.25, dt_field=rng.choice([0.3, 0.6, 1.1]), cycles=rng.randint(1, 4))
    if kind == "far":
        cumulative = rng.random() < 0.3
        nz = rng.randint(4, 40) if cumulative else _log(rng, 8, 256)
        return dict(kind=kind, nz=nz, no=_log(rng, 16, 300 if cumulative else 800), nr=_log(rng, 64, 700),
                    nrho=_log(rng, 32, 300 if cumulative else 1024),
                    contraction=rng.choice(["fp64", "fp64", "fp64", "fp64-grid", "fp32-mfma", "fp16x3-mfma"]),
                    cumulative=cumulative, c64=rng.random() < 0.4)
    return dict(kind=kind, nz=_log(rng, 16, 256), no=_log(rng, 64, 2048), nr=_log(rng, 100, 512),
                nrho=_log(rng, 100, 1024),
                contraction=rng.choice(["fp64-grid", "fp32-mfma", "bf16x3-mfma", "bf16x6-mfma", "fp16x3-mfma"]),
                c64=rng.random() < 0.5)


# -- inputs -----------------------------------------------------------------------------------

def _n_e(c):
    return int(math.ceil(c["cycles"] * 2.0 * math.pi / W.omega_au(800e-9) / c["dt"])) + 1


def _beam(c, seed, n):
    """n sin^2 pulses of a focused beam: amplitude falling with the radius, a phase of each point."""
    rng = np.random.default_rng(seed)
    t = np.arange(_n_e(c)) * c["dt"]
    w = W.omega_au(800e-9)
    amp = W.field_au(1.5e14 * rng.uniform(0.8, 1.2)) * np.exp(-np.linspace(0.0, 2.0, n) ** 2)
    phase = rng.uniform(-1.5, 1.5, n)
    env = np.sin(math.pi * t / (c["cycles"] * 2.0 * math.pi / w)) ** 2
    return t, amp[:, None] * env[None, :] * np.sin(w * t[None, :] + phase[:, None])


def _geometry(c):
    return tdse.Geometry(c["num_r"], c["dx"], c["dt"], A, E_GUESS, 1e-12, X_INT)


def _uneven(c, seed):
    """Members of the workload's own draw (grids and durations), their intensities from the seed."""
    members = W.uneven_batch(n_inst=c["n"], nr_range=(c["nr_lo"], c["nr_hi"]), cycles=(c["cyc_lo"], c["cyc_hi"]))
    fields, steps = W.stack_fields([m["field"] for m in members])
    fields *= np.random.default_rng(seed).uniform(0.7, 1.0, (c["n"], 1))
    return [m["num_r"] for m in members], fields, steps


def _cube(c, seed):
    """A CUPRAD-like field (z, t, r) in SI units, float32, with its grids."""
    rng = np.random.default_rng(seed)
    w = W.omega_au(800e-9)
    T = c["cycles"] * 2.0 * math.pi / w
    t = np.arange(int(math.ceil(T / c["dt_field"])) + 1) * c["dt_field"]
    z, r = np.linspace(0, 1e-3, c["nz"]), np.linspace(0, 150e-6, c["nr"])
    amp = W.field_au(1.2e14) * np.exp(-(r[None, :] / 100e-6) ** 2) * (1 - 0.1 * rng.uniform(0.5, 1.0, (c["nz"], 1)))
    wave = np.where(t <= T, np.sin(math.pi * t / T) ** 2, 0.0) * np.sin(w * t + rng.uniform(-0.5, 0.5))
    return (farm.EFIELDAU * amp[:, None, :] * wave[None, :, None]).astype(np.float32), t * farm.TIMEAU, r, z


def _sources(c, seed):
    return W.hankel_workload(nz=c["nz"], no=c["no"], nr=c["nr"], nrho=c["nrho"], seed=seed, complex64=c["c64"])


def _weights(z):
    w = np.zeros(len(z))
    w[:-1] += 0.5 * np.diff(z)
    w[1:] += 0.5 * np.diff(z)
    return np.stack([w, np.eye(len(z))[0], np.eye(len(z))[-1]])


def _plane(c, seed):
    rng = np.random.default_rng(seed)
    r = np.linspace(0, 1.5e-4, c["nr"])
    o = W.OMEGA0_SI * np.linspace(11, 61, c["no"])
    F = (rng.standard_normal((c["no"], c["nr"])) + 1j * rng.standard_normal((c["no"], c["nr"]))) * np.exp(-(r / 6e-5) ** 2)
    pre = np.exp(1j * rng.uniform(0, 6, (c["nr"], c["no"])))
    return o, r, F, pre, np.linspace(0, 7e-3, c["nrho"])


def prepare(case, seed):
    c, s = case, {"case": case}
    kind = c["kind"]
    if kind == "atom":
        t, f = _beam(c, seed, 1)
        dll = TDSE_DLL()
        inputs = inputs_def()
        inputs.init_default_inputs(Eguess=E_GUESS, num_r=c["num_r"], dx=c["dx"], dt=c["dt"], trg_a=A, CV=1e-12, x_int=X_INT)
        inputs.init_time_and_field(dll, t=t, E=f[0])
        dll.init_GS(inputs)
        s.update(dll=dll, inputs=inputs)
    elif kind in ("batch", "plan"):
        s["geo"] = _geometry(c)
        s["fields"] = torch.tensor(tdse.pad_fields(_beam(c, seed, c["n"])[1]), device="cuda")
        if kind == "plan":
            s["plan"] = tdse.BatchPlan(s["geo"], s["fields"])
    elif kind == "uneven":
        num_r, fields, steps = _uneven(c, seed)
        s["geo"] = tdse.Geometry.create_many(num_r, 0.1, 0.25, A, E_GUESS, W.UNEVEN_CV, X_INT)
        s["fields"] = torch.tensor(fields, device="cuda")
        s["out"] = torch.zeros((c["n"], 5, max(steps)), dtype=torch.float64, device="cuda")
        s["plan"] = tdse.BatchPlan(s["geo"], s["fields"], n_steps=steps, out=s["out"])
    elif kind == "gradient":
        s["geo"] = _geometry(c)
        s["E"], s["n_steps"], s["window"] = _gradient_inputs(c, seed)
    elif kind == "farm":
        s["cube"] = _cube(c, seed)
    elif kind in ("far", "grid"):
        s["src"] = _sources(c, seed)
        if kind == "grid":
            zall, r, o = s["src"][:3]
            f, _ = hankel.get_propagation_pre_factor_function(zall[:-1], r, o, "Ar", W.hankel_pressure(), "Henke", True,
                                                              "NIST", True)
            s["pre"], s["w"] = f.tables.pre, _weights(zall[:-1])
    else:
        s["plane"] = _plane(c, seed)
    return s


def _gradient_inputs(c, seed):
    rng = np.random.default_rng(seed)
    t = np.arange(c["nt"]) * c["dt"]
    w = W.omega_au(800e-9)
    T = min(c["cycles"] * 2.0 * math.pi / w, t[-1])
    amp = W.field_au(1.5e14 * rng.uniform(0.8, 1.2)) * np.exp(-np.linspace(0.0, 1.5, c["n"]) ** 2)
    f = amp[:, None] * (np.where(t <= T, np.sin(math.pi * t / T) ** 2, 0.0) * np.sin(w * t + rng.uniform(-0.5, 0.5)))
    E = torch.tensor(np.concatenate([f, np.zeros((c["n"], 3))], axis=1), device="cuda")
    n = E.shape[1] - 1
    return E, n, adjoint.harmonic_window(n, c["dt"], n * c["dt"], w, 11, 31).cuda()


def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "atom":
        out = outputs_def()
        s["dll"].call1DTDSE(s["inputs"], out)
        res = {k: getattr(out, "get_" + k)() for k in ("sourceterm", "PopTot", "PopInt", "expval", "Efield", "Fsourceterm",
                                                       "FEfield")}
        out.delete(s["dll"])
        return res
    if kind == "batch":
        return dict(zip(ROWS, tdse.propagate_batch(s["geo"], s["fields"]).unbind(1)))
    if kind in ("plan", "uneven"):
        return dict(zip(ROWS, s["plan"].replay().unbind(1)))
    if kind == "gradient":
        E = s["E"].clone().requires_grad_(True)
        src = adjoint.TDSEDipole.apply(E, s["geo"], s["n_steps"])
        adjoint.harmonic_yield(src, c["dt"], s["window"]).sum().backward()
        return {"sourceterm": src.detach(), "grad": E.grad}
    if kind == "farm":
        f, t, r, z = s["cube"]
        return farm.run(f, t, r, z, 1, c["nz"], 1, c["nr"], c["num_r"], c["dx"], c["dt"], A, E_GUESS, 1e-12, X_INT)
    if kind == "far":
        z, r, o, rho, src, distance = s["src"]
        target = hankel.FSources_provider(z, r, o, FSource=src)
        res = hankel.Hankel_long(target, distance, rho, "Ar", W.hankel_pressure(), "Henke", True, "NIST", True,
                                 store_cumulative_result=c["cumulative"], contraction=c["contraction"])
        out = {"FF": res.FF_integrated, "entry": res.entry_plane_transform, "exit": res.exit_plane_transform}
        if c["cumulative"]:
            out["cumulative"] = res.cumulative_field
        return out
    if kind == "grid":
        z, r, o, rho, src, distance = s["src"]
        return hankel.gridded(src, z[:-1], o, r, rho, distance, s["w"], pre=s["pre"], kind=c["contraction"])
    o, r, F, pre, rho = s["plane"]
    return hankel.HankelTransform(o, r, F, 0.98, rho, near_field_factor=c["near"], pre_factor=pre)


# -- the least a pass can do ------------------------------------------------------------------

def _pt_steps(c):
    return float(c["n"]) * (c["num_r"] + 1) * (_n_e(c) + 2)


def work(case):
    """TDSE: fields in, five series out, and 68 flop per grid point and step (right-hand side,
    the two recurrences of the solve, the phase, the observables).  Far field: sources in,
    fields out, one complex multiply-add per source element, and the product with J0 sampled at
    its band limit (rho q / pi points), which every screen radius and frequency needs."""
    c = case
    kind = c["kind"]
    if kind in ("atom", "batch", "plan"):
        c = dict(c, n=c.get("n", 1))
        return {"bytes": c["n"] * 6.0 * 8 * (_n_e(c) + 2), "flops": 68.0 * _pt_steps(c)}
    if kind == "uneven":
        nr, ne = 2.0 * (c["nr_lo"] + c["nr_hi"]) / 2, (c["cyc_lo"] + c["cyc_hi"]) / 2 * 2 * math.pi / W.omega_au(1300e-9) / 0.25
        return {"bytes": c["n"] * 6.0 * 8 * ne, "flops": 68.0 * c["n"] * nr * ne}
    if kind == "gradient":
        # the backward sweep solves for the adjoint state and for the state it needs
        return {"bytes": c["n"] * 3.0 * 8 * c["nt"], "flops": 3 * 68.0 * c["n"] * (c["num_r"] + 1) * (c["nt"] + 2)}
    if kind == "farm":
        k1 = 1 + math.floor(c["dt_field"] / c["dt"]) if math.floor(c["dt_field"] / c["dt"]) != 1 else 1
        nt = c["cycles"] * 2 * math.pi / W.omega_au(800e-9) / c["dt_field"]
        n = c["nz"] * c["nr"]
        return {"bytes": n * 8.0 * (nt / 2 + 8 * k1 * nt), "flops": 68.0 * n * (c["num_r"] + 1) * k1 * nt}
    if kind == "plane":
        el = float(c["no"]) * c["nr"]
        return {"bytes": 16.0 * (2 * el + c["no"] * c["nrho"]), "flops": 4.0 * el * c["nrho"]}
    items = float(c["nz"]) * c["no"] * c["nr"]
    n_out = c["nz"] + 2 if c.get("cumulative") else 3
    n_q = 61 * W.OMEGA0_SI / W.C_LIGHT * 200e-6 * 7e-3 / math.pi
    return {"bytes": (8.0 if c["c64"] else 16.0) * items + 16.0 * n_out * c["nrho"] * c["no"],
            "flops": 8.0 * items + 4.0 * n_out * c["nrho"] * c["no"] * n_q}


# -- the same results from plain torch in 64 bits -----------------------------------------------

BLOCK, REACH = 512, 168  # the step's matrix decays by ~0.75 a point: nothing is left after REACH points


class _Stepper:
    """Crank-Nicolson with Numerov's M2 and the potential indexed by column (prop.c:138-204):
    U = (M2 + iH)^-1 (M2 - iH) as a band, by dense solves of overlapping windows."""

    def __init__(self, num_r, dx, dt):
        n = self.n = num_r + 1
        self.x = (np.arange(n) - 0.5 * num_r) * dx
        V = -1.0 / np.sqrt(A * A + self.x ** 2)
        self.dpot = torch.tensor(self.x * (A * A + self.x ** 2) ** -1.5, device="cuda")
        self.nb = -(-n // BLOCK)
        size, pad = BLOCK + 4 * REACH, 2 * REACH
        Vp, on = np.zeros(self.nb * BLOCK + 2 * pad), np.zeros(self.nb * BLOCK + 2 * pad, dtype=bool)
        Vp[pad:pad + n], on[pad:pad + n] = V, True
        U = np.empty((self.nb, BLOCK, BLOCK + 2 * REACH), dtype=np.complex128)
        i = np.arange(size)
        for b in range(self.nb):
            v, m = Vp[b * BLOCK:b * BLOCK + size], on[b * BLOCK:b * BLOCK + size]
            M2, H = np.zeros((size, size)), np.zeros((size, size))
            M2[i, i], M2[i[1:], i[:-1]], M2[i[:-1], i[1:]] = 10 / 12, 1 / 12, 1 / 12
            H[i, i], H[i[1:], i[:-1]], H[i[:-1], i[1:]] = (1 / dx ** 2, -0.5 / dx ** 2, -0.5 / dx ** 2)
            S = 0.5 * dt * (H + M2 * v[None, :])
            off = ~(m[:, None] & m[None, :])
            M2[off], S[off] = 0.0, 0.0
            M2[i[~m], i[~m]] = 1.0
            X = np.linalg.solve(M2 + 1j * S, M2 - 1j * S)
            U[b] = X[pad:pad + BLOCK, REACH:size - REACH]
        self.U = torch.tensor(U, device="cuda")
        self.Ut = self.U.transpose(1, 2).contiguous()  # (nb, window, BLOCK)
        self.Uc = self.U.conj().resolve_conj().contiguous()
        self.xp = self._pad(torch.tensor(self.x, device="cuda"))
        self.dp = self._pad(self.dpot)
        self.dt = dt

    def _pad(self, v):
        out = torch.zeros(self.nb * BLOCK, dtype=v.dtype, device="cuda")
        out[:self.n] = v
        return out

    def windows(self, psi):
        p = torch.nn.functional.pad(torch.view_as_real(psi).permute(2, 0, 1), (REACH, REACH))
        w = p.unfold(2, BLOCK + 2 * REACH, BLOCK)  # (2, inst, nb, window)
        return torch.complex(w[0], w[1]).transpose(0, 1).contiguous()

    def apply(self, psi, Ut):
        return torch.bmm(self.windows(psi), Ut).transpose(0, 1).reshape(psi.shape[0], -1)

    def adjoint(self, y):
        w = torch.bmm(y.reshape(y.shape[0], self.nb, BLOCK).transpose(0, 1).contiguous(), self.Uc).transpose(0, 1)
        out = w[:, :, REACH:REACH + BLOCK].clone()
        out[:, :-1, BLOCK - REACH:] += w[:, 1:, :REACH]
        out[:, 1:, :REACH] += w[:, :-1, REACH + BLOCK:]
        return out.reshape(y.shape[0], -1)

    def phase(self, F):
        return torch.exp(1j * self.dt * F[:, None] * self.xp[None, :])

    def ground_state(self):
        """The lowest state of the Numerov pencil H + M2 V = E M2 around the atom."""
        keep = np.abs(self.x) <= 70.0
        x = self.x[keep]
        dx, m = x[1] - x[0], len(x)
        i = np.arange(m)
        M2, H = np.zeros((m, m)), np.zeros((m, m))
        M2[i, i], M2[i[1:], i[:-1]], M2[i[:-1], i[1:]] = 10 / 12, 1 / 12, 1 / 12
        H[i, i], H[i[1:], i[:-1]], H[i[:-1], i[1:]] = 1 / dx ** 2, -0.5 / dx ** 2, -0.5 / dx ** 2
        H = H - M2 / np.sqrt(A * A + x ** 2)[None, :]
        e, v = E_GUESS, np.ones(m)
        for _ in range(4):
            w = np.linalg.solve(H - e * M2, M2 @ v)
            e, v = e + (v @ v) / (v @ w), w / np.linalg.norm(w)
        full = np.zeros(self.n)
        full[keep] = v * np.sign(v[m // 2])
        return full


def _gate(E):
    """True after the first k with E_k E_{k+1} <= 0: up to it the field is taken as 0 (prop.c:125-134)."""
    hit = E[:, :-1] * E[:, 1:] <= 0
    first = np.where(hit.any(axis=1), hit.argmax(axis=1), E.shape[1])
    return np.arange(E.shape[1])[None, :] > first[:, None]


def _cn(num_r, dx, dt, fields, n_steps, gobs=None):
    """The five series of every row of `fields`; with gobs(sourceterm) -> dL/dsourceterm also
    dL/dfield by the discrete adjoint, its states rebuilt by inverse steps (U^-1 = conj U)."""
    S = _Stepper(num_r, dx, dt)
    open_ = torch.tensor(_gate(np.asarray(fields)), device="cuda")
    F = torch.tensor(np.asarray(fields), device="cuda") * open_
    n = F.shape[0]
    psi0 = S._pad(torch.tensor(S.ground_state(), device="cuda"))
    psi = psi0[None, :].expand(n, -1).to(torch.complex128).contiguous()
    lo = int(np.searchsorted(S.x, -X_INT)) - 1
    hi = int(np.searchsorted(S.x, X_INT))
    out = torch.zeros((n, 5, n_steps), dtype=torch.float64, device="cuda")
    out[:, 1, 0] = 1.0
    out[:, 2, 0] = (psi0[lo:hi + 1] ** 2).sum()
    for k in range(n_steps - 1):
        psi = S.apply(psi, S.Ut) * S.phase(F[:, k])
        p = psi.real ** 2 + psi.imag ** 2
        out[:, 0, k + 1] = F[:, k] - p @ S.dp
        ov = torch.view_as_real(psi).permute(2, 0, 1) @ psi0
        out[:, 1, k + 1] = ov[0] ** 2 + ov[1] ** 2
        out[:, 2, k + 1] = p[:, lo:hi + 1].sum(1)
        out[:, 3, k + 1] = p @ S.xp
        out[:, 4, k + 1] = F[:, k]
    if gobs is None:
        return out
    gs = gobs(out[:, 0])
    dE = torch.zeros_like(F)
    lam = torch.zeros_like(psi)
    back = S.Ut.conj().resolve_conj().contiguous()
    for k in range(n_steps - 1, 0, -1):
        lam = lam - 2.0 * gs[:, k, None] * S.dp * psi
        dE[:, k - 1] = gs[:, k] - dt * ((lam.conj() * psi).imag @ S.xp)
        u = S.phase(-F[:, k - 1])
        lam, psi = S.adjoint(u * lam), S.apply(u * psi, back)
    return out, dE * open_


def _prefactor(z, o, pressure):
    """The z-tabulated branch of get_propagation_pre_factor_function (Hankel_transform.py:146-239)
    for argon, absorption from the Henke tables, dispersion from NIST's."""
    with np.load(hankel.TABLES, allow_pickle=False) as t:
        tab = {k: t[k] for k in t.files if k.startswith("Ar_")}
    hbar, ialpha, c, q, m = 1.0545718e-34, 137.035999139, 299792458.0, 1.602176565e-19, 9.10938356e-31
    a0 = hbar * ialpha / (c * m)
    au = o * (m * a0 ** 2 / hbar)  # omega in atomic units
    lam = 2.0 * np.pi * hbar / (au * m * c / ialpha ** 2)
    ev = au / (q / (m / ialpha ** 2 * c * c))
    scale = 2.7e25 * a0 / ialpha ** 2 * lam ** 2 / (2.0 * np.pi)
    f1 = np.interp(ev, tab["Ar_NIST/Energy_f1"], tab["Ar_NIST/f1"]) * scale
    beta = np.interp(ev, tab["Ar_Henke/Energy_f2"], tab["Ar_Henke/f2"]) * scale
    zp, pv = pressure["zgrid"], pressure["value"]

    def cum(y):
        return np.interp(z, zp, np.concatenate([[0.0], np.cumsum(0.5 * np.diff(zp) * (y[1:] + y[:-1]))]))

    # (1/v_IR - 1/v_XUV) = p f1 / c for n_IR = 1
    P = cum(pv)
    absw = P[:, None] * (beta * o / c)[None, :]
    pre = np.interp(z, zp, pv)[:, None] * np.exp(1j * P[:, None] * (f1 * o / c)[None, :] + absw - absw[-1])
    return pre, np.exp(absw[-1] - absw)


def _j0(x):
    """J0 to 64-bit rounding: below 25 the mean of cos(x sin t) over 64 angles (the first alias is
    J_64), above it Hankel's expansion, whose terms fall below 1e-16 there."""
    out = torch.empty_like(x)
    low = x < 25.0
    s = x[low]
    acc = torch.ones_like(s)  # the angle 0
    for k in range(1, 17):
        acc += torch.cos(s * math.sin(2 * math.pi * k / 64)) * (1.0 if k == 16 else 2.0)
    out[low] = acc / 32.0
    b = x[~low]
    y, P, Q, a = 1.0 / b, torch.zeros_like(b), torch.zeros_like(b), [1.0]
    for k in range(1, 24):
        a.append(-a[-1] * (2 * k - 1) ** 2 / (8.0 * k))
    for k in range(11, -1, -1):
        sign = -1.0 if k % 2 else 1.0
        P, Q = P * y * y + sign * a[2 * k], Q * y * y + sign * a[2 * k + 1]
    c, s = torch.cos(b), torch.sin(b)
    out[~low] = (P * (c + s) - Q * y * (s - c)) / torch.sqrt(math.pi * b)
    return out


def _screen(src, z, o, r, rho, distance, pre, near=True):
    """Every plane's transform (plane, rho, omega): the trapezoid over r of r J0 pre F e^{-iKr^2/2D}."""
    dev = dict(dtype=torch.float64, device="cuda")
    r_, rho_ = torch.tensor(r, **dev), torch.tensor(rho, **dev)
    w = np.zeros(len(r))
    w[:-1] += 0.5 * np.diff(r)
    w[1:] += 0.5 * np.diff(r)
    w_ = torch.tensor(w * r, **dev)
    K = torch.tensor(o / 299792458.0, **dev)
    out = torch.empty((len(z), len(rho), len(o)), dtype=torch.complex128, device="cuda")
    step = max(1, int(1e8 // (len(r) * len(rho))))
    for k in range(len(z)):
        D = distance - z[k]
        for a in range(0, len(o), step):
            kk = K[a:a + step]
            u = src[k, a:a + step].to(torch.complex128) * w_
            if near:
                u = u * torch.exp(-1j * kk[:, None] * r_ ** 2 / (2.0 * D))
            u = torch.view_as_real(u * pre[k, a:a + step]).contiguous()
            J = _j0(kk[:, None, None] * (rho_[:, None] * r_[None, :]) / D)
            out[k, :, a:a + step] = torch.view_as_complex(torch.bmm(J, u)).T
    return out


def exact(case, seed):
    c = case
    kind = c["kind"]
    if kind in ("atom", "batch", "plan"):
        if c.get("n", 1) * _pt_steps(dict(c, n=1)) > 1.2e10:
            return None
        f = tdse.pad_fields(_beam(c, seed, c.get("n", 1))[1])
        n = f.shape[1] - 1
        rows = _cn(c["num_r"], c["dx"], c["dt"], f, n)
        if kind != "atom":
            return dict(zip(ROWS, rows.unbind(1)))
        rows = rows[0].cpu().numpy()
        spec = {k: np.fft.rfft(rows[i]).conj() * c["dt"] / math.sqrt(2 * math.pi) for k, i in (("Fsourceterm", 0), ("FEfield", 4))}
        return {"sourceterm": rows[0], "PopTot": rows[1], "PopInt": rows[2], "expval": rows[3], "Efield": rows[4], **spec}
    if kind == "gradient":
        if c["n"] * (c["num_r"] + 1.0) * c["nt"] > 6e9:
            return None
        E, n, window = _gradient_inputs(c, seed)

        def gobs(s):
            s = s.detach().clone().requires_grad_(True)
            X = torch.fft.rfft(s, dim=-1)
            ((X.real ** 2 + X.imag ** 2) * (c["dt"] ** 2 / (2 * math.pi)) * window).sum().backward()
            return s.grad

        rows, dE = _cn(c["num_r"], c["dx"], c["dt"], E.cpu().numpy(), n, gobs)
        return {"sourceterm": rows[:, 0].contiguous(), "grad": dE}
    if kind in ("far", "grid"):
        if float(c["nz"]) * c["no"] * c["nr"] * c["nrho"] > 6e9:
            return None
        zall, r, o, rho, src, distance = _sources(c, seed)
        z = zall[:-1]
        pre, renorm = _prefactor(z, o, W.hankel_pressure())
        planes = _screen(src, z, o, r, rho, distance, torch.tensor(pre, device="cuda")[:, :, None])
        w = torch.tensor(_weights(z), device="cuda")
        if kind == "grid":
            return torch.stack([(planes * v[:, None, None]).sum(0) for v in w])
        out = {"FF": (planes * w[0][:, None, None]).sum(0), "entry": planes[0], "exit": planes[-1]}
        if c["cumulative"]:
            dz = torch.tensor(np.diff(z), device="cuda")[:, None, None]
            out["cumulative"] = torch.tensor(renorm[:-1], device="cuda")[:, None, :] * torch.cumsum(
                0.5 * dz * (planes[:-1] + planes[1:]), dim=0)
        return {k: v.cpu().numpy() for k, v in out.items()}
    if kind == "plane":
        o, r, F, pre, rho = _plane(c, seed)
        res = _screen(torch.tensor(F, device="cuda")[None], [0.0], o, r, rho, 0.98,
                      torch.tensor(np.ascontiguousarray(pre.T), device="cuda")[None], c["near"])
        return res[0].T.cpu().numpy()
    return None
