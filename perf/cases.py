"""Performance cases of the fused collide-and-stream-pull step and of what a
run does with it: advancing a domain, monitoring it, writing its fields.

Every case goes through ``metalbm_amd.Algorithm``.  ``prepare`` creates a
handle and its initial state from the seed, ``run`` advances it (``iterate``)
and returns the populations as the handle holds them on the device (shifted
and scaled as stored), together with whatever else the pass computes.
``exact`` is the same pass in 64-bit torch.

Sizes are those of this repository's benchmark, smoke run and tests, and
ragged ones between them.  The forcing is weak enough for a handle to be
advanced by tens of thousands of steps.
"""
import math

import numpy as np
import torch

from metalbm_amd import (Algorithm, AlphaMode, CollisionType, Config, EquilibriumType, ForceType,
                         ForcingSchemeType, LatticeType, Precision)

DEV = "cuda" if torch.cuda.is_available() else "cpu"

# Velocity sets in the order of the population index (the data format).
_C = {
    "D2Q9": [(0, 0), (-1, 1), (-1, 0), (-1, -1), (1, -1), (1, 0), (1, 1), (0, -1), (0, 1)],
    "D3Q19": [(0, 0, 0), (-1, 0, 0), (-1, -1, 0), (-1, 1, 0), (-1, 0, -1), (-1, 0, 1), (1, 0, 0),
              (1, 1, 0), (1, -1, 0), (1, 0, 1), (1, 0, -1), (0, -1, 0), (0, 0, -1), (0, -1, -1),
              (0, -1, 1), (0, 1, 0), (0, 0, 1), (0, 1, 1), (0, 1, -1)],
    "D3Q27": [(0, 0, 0), (-1, 0, 0), (-1, -1, 0), (-1, 1, 0), (-1, 0, -1), (-1, 0, 1),
              (-1, -1, -1), (-1, -1, 1), (-1, 1, -1), (-1, 1, 1), (1, 0, 0), (1, 1, 0),
              (1, -1, 0), (1, 0, 1), (1, 0, -1), (1, 1, 1), (1, 1, -1), (1, -1, 1), (1, -1, -1),
              (0, -1, 0), (0, 0, -1), (0, -1, -1), (0, -1, 1), (0, 1, 0), (0, 0, 1), (0, 1, 1),
              (0, 1, -1)],
}
_WEIGHT = {  # by the number of nonzero components
    "D2Q9": (4 / 9, 1 / 9, 1 / 36), "D3Q19": (1 / 3, 1 / 18, 1 / 36),
    "D3Q27": (8 / 27, 2 / 27, 1 / 54, 1 / 216)}


def _lattice(name):
    c = _C[name]
    return c, [_WEIGHT[name][sum(1 for v in ci if v)] for ci in c]


# Storage / compute / shifted of each precision.
_PRECISION = {"f64": ("F64", "F64", False),   # the reference-order parity build
              "f32": ("F32", "F32", True),    # the production build
              "f16": ("F16", "F32", True),    # half storage, single compute
              "f64s": ("F64", "F32", True)}   # double storage of single compute
_BYTES = {"f64": 8, "f32": 4, "f16": 2, "f64s": 8}


def _case(name, lattice, n, precision, steps, **more):
    c = dict(name=name, kind="step", lattice=lattice, nx=n[0], ny=n[1],
             nz=n[2] if len(n) > 2 else 1, precision=precision, steps=steps, collision="BGK",
             alpha="NEWTON", scheme="Guo", force="Kolmogorov", equilibrium="TruncationMa3",
             tau=0.6, push=1e-5, init="noise", amp=1e-3, store=False)
    c.update(more)
    return c


def listed():
    return [
        # The smoke run: the smallest domain, ten steps; latency and launches.
        _case("smoke-32", "D2Q9", (32, 32), "f64", 10),
        # The parity configuration (D2Q9 128^2, FP64, Guo + Kolmogorov): a
        # study of a small flow, a hundred steps between looks at it.
        _case("d2q9-128-f64", "D2Q9", (128, 128), "f64", 100),
        # Forced two-dimensional turbulence (EDM with the spectral force that
        # is rebuilt from the stored fields), fields stored every tenth step.
        _case("d2q9-turb-2048", "D2Q9", (2048, 2048), "f32", 10,
              scheme="ExactDifferenceMethod", force="Turbulent2D", push=5e-4, store=True),
        # The headline: D3Q19 256^3, FP32, Guo + constant force.
        _case("d3q19-256-f32", "D3Q19", (256, 256, 256), "f32", 20, tau=0.55, force="Constant",
              push=1e-6),
        # The same step in FP64 on a ragged box of odd extents.
        _case("d3q19-ragged-f64", "D3Q19", (171, 150, 133), "f64", 12, tau=0.55, push=1e-6),
        # The largest: D3Q27 Taylor-Green 384^3 with FP16 storage.
        _case("d3q27-384-f16", "D3Q27", (384, 384, 384), "f16", 10, tau=0.51, scheme="None_",
              force="None_", init="taylor_green", amp=0.05),
        # D3Q27 FP32 with the exact equilibrium on an odd box.
        _case("d3q27-odd-f32", "D3Q27", (193, 161, 130), "f32", 10, tau=0.55,
              equilibrium="Exact", push=1e-6),
        # Entropic D2Q9 2048^2 at high Reynolds number, the default solver
        # (the reference Newton).
        _case("d2q9-elbm-newton", "D2Q9", (2048, 2048), "f32", 5, collision="ELBM", tau=0.50003),
        # The same with the learned alpha.
        _case("d2q9-elbm-learned", "D2Q9", (2048, 2048), "f32", 10, collision="ELBM",
              tau=0.50003, alpha="LEARNED"),
        # Entropic decaying turbulence, D3Q27 256^3, plain Newton at the
        # residual tolerance.
        _case("d3q27-elbm-256", "D3Q27", (256, 256, 256), "f32", 2, collision="ELBM",
              tau=0.50006, alpha="NEWTON_RESIDUAL", scheme="None_", force="None_",
              init="spectral", amp=0.1 / 3 ** 0.5),
        # Monitoring a run: some steps, then mass, energy, enstrophy, the
        # vorticity and both spectra.
        _case("monitor-192-f64", "D3Q19", (192, 192, 192), "f64", 5, kind="monitor", tau=0.55,
              push=1e-6, store=True),
        # Output: some steps, then the fields on the host.
        _case("fields-out-f64", "D3Q19", (96, 80, 72), "f64", 10, kind="fields", push=1e-6,
              store=True),
    ]


def _spread(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    scheme = rng.choice(["Guo", "ExactDifferenceMethod", "ShanChen", "None_"])
    tau = round(rng.uniform(0.53, 0.95), 4)
    amp = round(10 ** rng.uniform(-3, -1.7), 6)
    family = rng.choice(["2d-small", "2d-large", "2d-turb", "3d-q19", "3d-q19", "3d-q27",
                         "3d-q27", "2d-elbm", "2d-elbm", "3d-elbm", "monitor", "fields"])
    if family in ("2d-small", "2d-large"):
        lo, hi = (24, 320) if family == "2d-small" else (320, 2048)
        n = (_spread(rng, lo, hi), _spread(rng, lo, hi))
        c = _case("", "D2Q9", n, rng.choice(["f64", "f64", "f32", "f16"]), _spread(rng, 5, 100),
                  scheme=scheme, tau=tau, amp=amp,
                  equilibrium=rng.choice(["TruncationMa3", "TruncationMa3", "Exact"]))
    elif family == "2d-turb":
        n = (_spread(rng, 256, 2048), _spread(rng, 256, 2048))
        c = _case("", "D2Q9", n, "f32", _spread(rng, 2, 20), scheme="ExactDifferenceMethod",
                  force="Turbulent2D", push=5e-4, tau=tau, store=True)
    elif family == "3d-q19":
        n = tuple(_spread(rng, 24, 288) for _ in range(3))
        c = _case("", "D3Q19", n, rng.choice(["f32", "f32", "f64", "f16", "f64s"]),
                  _spread(rng, 3, 20), scheme=scheme, tau=tau, amp=amp)
    elif family == "3d-q27":
        n = tuple(_spread(rng, 24, 256) for _ in range(3))
        c = _case("", "D3Q27", n, rng.choice(["f32", "f32", "f16", "f64"]), _spread(rng, 3, 16),
                  scheme=scheme, tau=tau, amp=amp,
                  equilibrium=rng.choice(["TruncationMa3", "TruncationMa3", "Exact"]))
    elif family == "2d-elbm":
        n = (_spread(rng, 192, 2048), _spread(rng, 192, 2048))
        c = _case("", "D2Q9", n, "f32", _spread(rng, 2, 10), collision="ELBM", tau=0.50003,
                  alpha=rng.choice(["NEWTON", "NEWTON_RESIDUAL", "WARM_RESIDUAL", "LEARNED"]))
    elif family == "3d-elbm":
        n = tuple(_spread(rng, 48, 224) for _ in range(3))
        c = _case("", rng.choice(["D3Q27", "D3Q27", "D3Q19"]), n, "f32", 2, collision="ELBM",
                  tau=0.50006, scheme="None_", force="None_", init="spectral",
                  amp=round(rng.uniform(0.02, 0.06), 4),
                  alpha=rng.choice(["NEWTON", "NEWTON_RESIDUAL", "WARM_RESIDUAL"]))
    elif family == "monitor":
        n = tuple(_spread(rng, 40, 200) for _ in range(3))
        c = _case("", rng.choice(["D3Q19", "D3Q27"]), n, "f64", _spread(rng, 1, 8),
                  kind="monitor", tau=tau, amp=amp, store=True)
    else:
        n = tuple(_spread(rng, 24, 96) for _ in range(3))
        c = _case("", rng.choice(["D3Q19", "D3Q27"]), n, "f64", _spread(rng, 1, 20),
                  kind="fields", scheme=scheme, tau=tau, amp=amp, store=True)
    del c["name"]
    cells = c["nx"] * c["ny"] * c["nz"]
    # the forcing bounds the velocity that a long run reaches
    if c["collision"] == "ELBM":
        c["push"] = 1e-5 * min(1.0, cells / 2048.0 ** 2)
    elif c["force"] == "Kolmogorov":
        nu, k = (c["tau"] - 0.5) / 3.0, 8.0 * math.pi / c["ny"]
        c["push"] = 0.01 * nu * k * k
    return c


# -- the pass -------------------------------------------------------------------

def _seeded(case, seed):
    """Initial amplitude of the Taylor-Green state, which takes no seed."""
    return case["amp"] * (0.8 + 0.4 * ((seed * 2654435761) % 1000003) / 1000003.0)


def _wavelength(case):
    return case["ny"] / 4.0


def _kmax(case):
    small = min(case[d] for d in (("nx", "ny", "nz") if case["lattice"] != "D2Q9" else ("nx", "ny")))
    return min(16, (small - 1) // 2)


def _config(case):
    storage, compute, shifted = _PRECISION[case["precision"]]
    push = case["push"]
    amplitude = (push, push, push) if case["force"] == "Turbulent2D" else (push, 0.0, 0.0)
    return Config(
        lattice=LatticeType[case["lattice"]], collision=CollisionType[case["collision"]],
        forcing_scheme=ForcingSchemeType[case["scheme"]], force=ForceType[case["force"]],
        equilibrium=EquilibriumType[case["equilibrium"]], nx=case["nx"], ny=case["ny"],
        nz=case["nz"], tau=case["tau"], amplitude=amplitude,
        wavelength=(_wavelength(case), 1.0, 1.0), storage=Precision[storage],
        compute=Precision[compute], shifted=shifted, alpha_mode=AlphaMode[case["alpha"]],
        force_kmin=5, force_kmax=7, removal_amplitude=(1e-6,) * 3, removal_kmin=1, removal_kmax=2)


def prepare(case, seed):
    a = Algorithm(_config(case))
    if case["init"] == "noise":
        a.init_noise(1.0, case["amp"], seed)
    elif case["init"] == "taylor_green":
        a.init_taylor_green(1.0, _seeded(case, seed))
    else:
        a.init_spectral(1.0, case["amp"], _kmax(case), 4.0, seed)
    if case["alpha"] == "LEARNED":
        params, mean, scale, out_scale = _network(case, seed)
        a.set_mlp_params(params)
        a.set_normalization(mean, scale, 2.0, out_scale)
    return {"case": case, "handle": a}


class _OnDevice:
    """The handle's populations for torch, without a copy; keeps the handle."""

    def __init__(self, handle):
        ptr, elem = handle.device_populations()
        self.handle = handle
        self.__cuda_array_interface__ = {
            "shape": (handle.Q, handle.N), "typestr": "<f%d" % elem, "data": (ptr, False),
            "version": 2}


def run(state):
    a, case = state["handle"], state["case"]
    a.iterate(case["steps"], store=case["store"])
    out = {"populations": torch.as_tensor(_OnDevice(a), device="cuda")}
    if case["kind"] == "monitor":
        out["mass"], out["energy"], out["enstrophy"] = a.reduce()
        _, out["spectral_enstrophy"] = a.vorticity("physical", field=False)
        out["energy_spectrum"], out["forcing_spectrum"] = a.spectra("physical")
    elif case["kind"] == "fields":
        out["rho"], out["u"], _, out["force"] = a.store_fields()
    return out


def work(case):
    """One pass: the populations (and the entropic alpha) read and written
    once, the operations of every step; spectra and fields on top."""
    c, _ = _lattice(case["lattice"])
    q, d = len(c), len(c[0])
    cells = case["nx"] * case["ny"] * case["nz"]
    nbytes = 2 * q * cells * _BYTES[case["precision"]]
    # moments (1 + d) and relaxation (2), polynomial (8), source (7 Guo, 10 EDM)
    per = 11 + d + {"Guo": 7, "ExactDifferenceMethod": 10}.get(case["scheme"], 0)
    if case["collision"] == "ELBM":
        nbytes += 2 * cells * 4
        per += 24  # deviation and bound (4), one logarithm (15), Newton sums (5)
    flops = case["steps"] * cells * q * per
    if case["store"] and case["kind"] != "step":
        nbytes += cells * (2 + 2 * d) * 8
    if case["kind"] == "monitor":
        nbytes += cells * (1 + 2 * d) * 8
        flops += 3 * d * 2.5 * cells * math.log2(cells)
    return {"bytes": nbytes, "flops": flops}


# -- the same pass in 64-bit torch ------------------------------------------------

def _shape(case):
    return tuple(case[d] for d in ("nx", "ny", "nz"))[:len(_C[case["lattice"]][0])]


def _i64(v):
    v &= (1 << 64) - 1
    return v - (1 << 64) if v >> 63 else v


def _splitmix(seed, k):
    """SplitMix64 outputs k (an int64 tensor) of the stream `seed`, as the
    uniform numbers (z >> 11) 2^-53."""
    def shift(z, s):
        return (z >> s) & ((1 << (64 - s)) - 1)
    z = (k + 1) * _i64(0x9E3779B97F4A7C15) + _i64(seed)
    z = (z ^ shift(z, 30)) * _i64(0xBF58476D1CE4E5B9)
    z = (z ^ shift(z, 27)) * _i64(0x94D049BB133111EB)
    z = z ^ shift(z, 31)
    return shift(z, 11).double() * 2.0 ** -53


def _initial_velocity(case, seed):
    shape, d = _shape(case), len(_shape(case))
    n = math.prod(shape)
    if case["init"] == "noise":
        k = torch.arange(n * d, dtype=torch.int64, device=DEV)
        return (case["amp"] * (2.0 * _splitmix(seed, k) - 1.0)).reshape(n, d).t().reshape(d, *shape)
    if case["init"] == "taylor_green":
        x = torch.meshgrid(*[torch.arange(m, dtype=torch.float64, device=DEV) * (2 * math.pi / m)
                             for m in shape], indexing="ij")
        cz = torch.cos(x[2]) if d == 3 else 1.0
        u = torch.zeros(d, *shape, dtype=torch.float64, device=DEV)
        u[0] = _seeded(case, seed) * torch.sin(x[0]) * torch.cos(x[1]) * cz
        u[1] = -_seeded(case, seed) * torch.cos(x[0]) * torch.sin(x[1]) * cz
        return u
    # solenoidal random phases (the specification of init_spectral)
    K = _kmax(case)
    r = np.arange(-K, K + 1)
    k = np.stack(np.meshgrid(*[r] * d, indexing="ij"), -1).reshape(-1, d)
    s = np.floor(np.sqrt((k * k).sum(1)) + 0.5).astype(int)
    active = (s >= 1) & (s <= K)
    lead = k[np.arange(len(k)), (k != 0).argmax(1)]
    half = active & (lead > 0)
    count = np.bincount(s[active], minlength=K + 1)
    energy = np.array([0.0] + [e ** 4 * math.exp(-2 * (e / 4.0) ** 2) for e in range(1, K + 1)])
    kh, sh = k[half].astype(float), s[half]
    m = len(kh)
    t = 2 * math.pi * _splitmix(seed, torch.arange(3 * m, dtype=torch.int64)).numpy().reshape(m, 3)
    amp = np.sqrt(energy[sh] / count[sh])
    if d == 3:
        axis = np.abs(kh).argmin(1)
        e1 = np.cross(kh, np.eye(3)[axis])
        e1 /= np.linalg.norm(e1, axis=1, keepdims=True)
        e2 = np.cross(kh, e1)
        e2 /= np.linalg.norm(e2, axis=1, keepdims=True)
        uh = amp[:, None] * ((np.cos(t[:, 2]) * np.exp(1j * t[:, 0]))[:, None] * e1
                             + (np.sin(t[:, 2]) * np.exp(1j * t[:, 1]))[:, None] * e2)
    else:
        e1 = np.stack([-kh[:, 1], kh[:, 0]], 1) / np.linalg.norm(kh, axis=1, keepdims=True)
        uh = (amp * np.exp(1j * t[:, 0]))[:, None] * e1
    uh = torch.from_numpy(uh).to(DEV)
    at = [torch.from_numpy(k[half][:, i] % shape[i]).to(DEV) for i in range(d)]
    gamma = case["amp"] * math.sqrt(d / energy.sum())
    u = torch.empty(d, *shape, dtype=torch.float64, device=DEV)
    for c in range(d):
        full = torch.zeros(*shape, dtype=torch.complex128, device=DEV)
        full[tuple(at)] = uh[:, c]
        u[c] = 2.0 * gamma * n * torch.fft.ifftn(full).real
    return u


class _Equilibrium:
    def __init__(self, case, rho, u):
        self.c, self.w = _lattice(case["lattice"])
        self.rho, self.u = rho, u
        self.exact = case["equilibrium"] == "Exact"
        if self.exact:
            s = torch.sqrt(1 + 3 * u * u)
            self.a, self.b = 2 - s, (2 * u + s) / (1 - u)
        else:
            self.u2 = (u * u).sum(0)

    def __call__(self, i):
        c, w = self.c[i], self.w[i]
        if self.exact:
            p = self.rho * w
            for d, cd in enumerate(c):
                p = p * self.a[d]
                if cd:
                    p = p * self.b[d] if cd > 0 else p / self.b[d]
            return p
        cu, u2 = _dot(c, self.u), self.u2
        if cu is None:
            return self.rho * w * (1 + u2 * (1.125 * u2 - 1.5))
        return self.rho * w * (1 + u2 * (1.125 * u2 - 1.5)
                               + cu * ((3 - 4.5 * u2) + cu * ((4.5 - 6.75 * u2)
                                                              + cu * (4.5 + 3.375 * cu))))


def _dot(c, v):
    s = None
    for d, cd in enumerate(c):
        if cd:
            t = v[d] if cd > 0 else -v[d]
            s = t if s is None else s + t
    return s


def _alpha(p, n, w, stored):
    """The entropic alpha of cells with populations p[q, cells] and
    non-equilibrium parts n: the deviation test, the bound, Newton."""
    alpha = torch.full_like(stored, 2.0)
    small = ((n.abs() / p) <= 1e-3).all(0)
    ratio = torch.where(n > 0, p.abs() / n, torch.full_like(p, math.inf))
    amax = ratio.min(0).values.clamp(max=2.5)
    capped = ~small & (amax < 2.0)
    alpha[capped] = 0.95 * amax[capped]
    left = torch.nonzero(~small & ~capped).reshape(-1)
    solved = left
    x, f, m, a_max = stored[left], p[:, left], n[:, left], amax[left]
    wc = w[:, None]
    h0 = (f * torch.log(f / wc)).sum(0)
    for _ in range(50):
        if not left.numel():
            break
        fm = f - x * m
        lg = torch.log(fm / wc)
        step = (h0 - (fm * lg).sum(0)) / (m * (1 + lg)).sum(0)
        done = step.abs() <= 1e-8
        good = done & (x > 1) & (x < a_max)
        alpha[left[good]] = x[good]
        on = ~done & ~step.isnan()
        left, x, f, m, a_max, h0 = (left[on], (x - step)[on], f[:, on], m[:, on], a_max[on], h0[on])
    return alpha, solved


class _Run:
    """The domain in 64 bits: f[q, *shape] and the entropic alpha field."""

    def __init__(self, case, seed):
        self.case, self.shape = case, _shape(case)
        self.d = len(self.shape)
        self.c, self.w = _lattice(case["lattice"])
        self.w_t = torch.tensor(self.w, dtype=torch.float64, device=DEV)
        u = _initial_velocity(case, seed)
        rho = torch.ones(self.shape, dtype=torch.float64, device=DEV)
        e = _Equilibrium(case, rho, u)
        self.f = torch.stack([e(i) for i in range(len(self.c))])
        self.alpha = torch.full(self.shape, 2.0, dtype=torch.float64, device=DEV)
        self.fields = (rho, u)
        self.samples = []
        self.injection = self._shell_force() if case["force"] == "Turbulent2D" else None

    def _half_k(self):
        k = [torch.fft.fftfreq(m, 1.0 / m, device=DEV, dtype=torch.float64) for m in self.shape]
        k[-1] = torch.arange(self.shape[-1] // 2 + 1, device=DEV, dtype=torch.float64)
        return torch.meshgrid(*k, indexing="ij")

    def _shell_force(self):
        kx, ky = self._half_k()
        k2 = kx * kx + ky * ky
        psi = self.case["push"] * ((k2 >= 25) & (k2 <= 49)).double()
        return torch.stack([torch.fft.irfftn(1j * ky * psi, s=self.shape),
                            torch.fft.irfftn(-1j * kx * psi, s=self.shape)])

    def force(self):
        case = self.case
        if case["force"] == "Constant":
            return [case["push"]] + [0.0] * (self.d - 1)
        if case["force"] == "Kolmogorov":
            y = torch.arange(case["ny"], dtype=torch.float64, device=DEV)
            fx = case["push"] * torch.sin(2 * math.pi * y / _wavelength(case))
            fx = fx.reshape((1, -1) + (1,) * (self.d - 2)).expand(self.shape)
            return [fx] + [0.0] * (self.d - 1)
        if case["force"] == "Turbulent2D":
            kx, ky = self._half_k()
            k2 = kx * kx + ky * ky
            keep = ((k2 >= 1) & (k2 <= 4)).double()
            rho, u = self.fields
            return [self.injection[d] - 1e-6 * torch.fft.irfftn(torch.fft.rfftn(rho * u[d]) * keep,
                                                               s=self.shape) for d in range(2)]
        return [0.0] * self.d

    def step(self, F, log=False):
        case, q = self.case, len(self.c)
        dims = tuple(range(self.d))
        p = torch.empty_like(self.f)
        for i, c in enumerate(self.c):
            p[i] = torch.roll(self.f[i], c, dims)
        rho = p.sum(0)
        u = torch.stack([sum(p[i] * c[d] for i, c in enumerate(self.c) if c[d])
                         for d in range(self.d)]) / rho
        e = _Equilibrium(case, rho, u)
        scheme, tau = case["scheme"], case["tau"]
        forced = case["force"] != "None_"
        e2 = None
        if scheme == "ExactDifferenceMethod" and forced:
            e2 = _Equilibrium(case, rho, torch.stack([u[d] + F[d] / rho for d in range(self.d)]))
        if case["collision"] == "ELBM":
            n = torch.stack([p[i] - e(i) for i in range(q)])
            flat_p, flat_n, flat_a = p.reshape(q, -1), n.reshape(q, -1), self.alpha.reshape(-1)
            for at in range(0, flat_a.numel(), 1 << 21):
                part = slice(at, at + (1 << 21))
                a, solved = _alpha(flat_p[:, part], flat_n[:, part], self.w_t, flat_a[part])
                flat_a[part] = a
                if log:
                    self.samples.append((flat_n[:, part][:, solved]
                                         / rho.reshape(-1)[part][solved], a[solved]))
            rate = self.alpha / (2 * tau)
        else:
            n, rate = None, 1 / tau
        g = 1 - 1 / (2 * tau)
        for i, c in enumerate(self.c):
            fe = p[i] - n[i] if n is not None else e(i)
            r = p[i] - rate * (p[i] - fe)
            if scheme == "Guo" and forced:
                cu = _dot(c, u)
                s = 0.0
                for d in range(self.d):
                    s = s + ((c[d] - u[d]) + (c[d] * 3 * cu if c[d] else 0.0)) * F[d]
                r = r + g * self.w[i] * 3 * s
            elif e2 is not None:
                r = r + e2(i) - fe
            self.f[i] = r
        if scheme == "None_":
            uh = u
        else:
            uh = torch.stack([u[d] + 0.5 * F[d] / rho for d in range(self.d)])
        return rho, uh


def exact(case, seed):
    with torch.no_grad():
        r = _Run(case, seed)
        F = r.force()
        for _ in range(case["steps"]):
            rho, uh = r.step(F)
        q, n = len(r.c), math.prod(r.shape)
        pops = r.f.reshape(q, n)
        if _PRECISION[case["precision"]][2]:
            for i, w in enumerate(r.w):
                pops[i] -= w
                if case["precision"] == "f16":  # the power of two at most 1 / w
                    pops[i] *= 2.0 ** math.floor(math.log2(1 / w) + 1e-9)
        out = {"populations": pops}
        if case["kind"] == "monitor":
            out["mass"] = float(rho.sum())
            out["energy"] = float((0.5 * rho * (uh * uh).sum(0)).sum() / n)
            out.update(_monitor(r, uh, F))
        elif case["kind"] == "fields":
            out["rho"], out["u"] = rho.reshape(n).cpu().numpy(), uh.reshape(r.d, n).cpu().numpy()
            out["force"] = torch.stack([torch.zeros_like(rho) + F[d] for d in range(r.d)]
                                       ).reshape(r.d, n).cpu().numpy()
        return out


def _monitor(r, uh, F):
    """Enstrophy by central differences and spectrally, shell spectra of the
    velocity and of the force (the physical scaling)."""
    n, d, shape = math.prod(r.shape), r.d, r.shape

    def diff(v, axis):
        return 0.5 * (torch.roll(v, -1, axis) - torch.roll(v, 1, axis))
    pairs = [(2, 1), (0, 2), (1, 0)]  # curl component: (v, derivative axis) - swapped
    w2 = sum((diff(uh[a], b) - diff(uh[b], a)) ** 2 for a, b in pairs)
    k = r._half_k()
    last = k[-1]
    kd = [torch.where(torch.tensor(m % 2 == 0, device=DEV) & (kk.abs() == m // 2),
                      torch.zeros_like(kk), kk) * (2 * math.pi / m) for kk, m in zip(k, shape)]
    uhat = [torch.fft.rfftn(uh[c]) for c in range(d)]
    ens = sum((torch.fft.irfftn(1j * (kd[b] * uhat[a] - kd[a] * uhat[b]), s=shape) ** 2).sum()
              for a, b in pairs)
    k2 = sum(kk * kk for kk in k)
    shell = torch.floor(torch.sqrt(k2) + 0.5).long()
    weight = torch.where((last == 0) | ((last == shape[-1] // 2) & (shape[-1] % 2 == 0)), 0.5, 1.0)
    ns = max(shape) // 2
    keep = shell < ns

    def spectrum(hats):
        e = sum(h.real ** 2 + h.imag ** 2 for h in hats) * weight
        out = torch.zeros(ns, dtype=torch.float64, device=DEV)
        out.index_add_(0, shell[keep], e[keep])
        return (out / float(n) ** 2).cpu().numpy()
    forces = [torch.zeros(shape, dtype=torch.float64, device=DEV) + F[c] for c in range(d)]
    return {"enstrophy": float(0.5 * w2.sum() / n), "spectral_enstrophy": float(0.5 * ens / n),
            "energy_spectrum": spectrum(uhat),
            "forcing_spectrum": spectrum([torch.fft.rfftn(v) for v in forces])}


def _network(case, seed):
    """The alpha predictor a learned run has in hand: trained here on the
    solves of a small domain of the same flow, in the library's parameter
    layout (9-32-32-1 over the normalised non-equilibrium moments)."""
    small = dict(case, nx=96, ny=96)
    r = _Run(small, seed)
    F = r.force()
    with torch.no_grad():
        for _ in range(6):
            r.step(F, log=True)
    basis = []
    for k in range(9):
        phi = [lambda v: 1, lambda v: v, lambda v: v * v]
        basis.append([phi[k // 3](c[0]) * phi[k % 3](c[1]) for c in r.c])
    basis = torch.tensor(basis, dtype=torch.float64, device=DEV)
    x = torch.cat([basis @ n for n, _ in r.samples], 1).t()
    y = torch.cat([a for _, a in r.samples]) - 2.0
    sd = x.std(0, unbiased=False)
    mean, scale = x.mean(0), 1.0 / torch.clamp(sd, min=1e-3 * float(sd.max()) + 1e-300)
    out_scale = max(float(y.square().mean().sqrt()), 1e-12)
    z, t = ((x - mean) * scale).float(), (y / out_scale).float()
    gen = torch.Generator().manual_seed(seed)
    sizes = [(32, 9), (32, 32), (1, 32)]
    params = []
    for o, i in sizes:
        lim = math.sqrt(6.0 / i)
        params += [((2 * torch.rand(o, i, generator=gen) - 1) * lim).to(DEV).requires_grad_(),
                   torch.zeros(o, device=DEV, requires_grad=True)]
    adam = torch.optim.Adam(params, lr=4e-3)
    iters = 400
    for it in range(iters):
        adam.param_groups[0]["lr"] = 4e-3 * (1 - it / iters) + 1e-5
        at = torch.randint(len(z), (4096,), generator=gen).to(DEV)
        h = z[at]
        for k in range(3):
            h = torch.nn.functional.linear(h, params[2 * k], params[2 * k + 1])
            if k < 2:
                h = torch.relu(h)
        loss = (h.reshape(-1) - t[at]).square().mean()
        adam.zero_grad()
        loss.backward()
        adam.step()
    flat = torch.cat([p.detach().reshape(-1) for p in params]).cpu().numpy()
    return (flat, mean.float().cpu().numpy(), scale.float().cpu().numpy(), out_scale)
