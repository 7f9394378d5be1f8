"""What the engine's performance is measured on: the calls its users' programs make, over the range they make them in.

A case is one call (or the few calls that belong together) through pgmhip's public entry points:

  md      one molecular-dynamics step as an OpenMM-like program takes it: float4 positions and the fixed-point force
          buffer in HBM, pgm_launch_device + pgm_finish_device, the mu4 guess from the four steps before
  eval    one evaluation for a program that keeps FP64 positions and forces in HBM (pgm_compute_device_f64), same guess
  host    one evaluation from host arrays with the strain derivative (pgm_compute): barostats, single points, tools
  frames  frames of a trajectory that are far apart, scored one after another from host float arrays
          (pgm_compute_f32 + pgm_forces): a list build and a solve from alpha E each
  fit     one step of a parameter fit: new parameters, energies and forces, and the gradients of a loss by the
          adjoint; several snapshots packed in one batch, or one system through the torch layer (PgmModel)

Mixed-precision results carry FP32 accuracy (energies, forces and gradients a few 1e-6 from the exact ones), and a
program that runs in mixed precision holds them in FP32: those outputs are FP32 tensors here, the FP64 path's are FP64.
`exact` evaluates the same model in FP64 with plain torch operations.
"""

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pgm-md_amd"))

from pgmhip import adjoint, engine, systems  # noqa: E402

LIQUID = 33.43  # water molecules per nm^3 at 1 g/cm^3
FIXED_SCALE = 2.0**32
STEP_NM = 0.002  # how far the mean atom moves from one step to the next


# ------------------------------------------------------------------------------------------------ the cases


def listed():
    base = {"density": LIQUID, "species": 1, "order": 6, "cutoff": 0.9, "precision": "mixed", "tune": True, "gvdw": False}

    def case(name, kind, nmol, grid, tol, **kw):
        kx, ky, kz = (grid,) * 3 if isinstance(grid, int) else grid
        return dict(base, name=name, kind=kind, nmol=nmol, kx=kx, ky=ky, kz=kz, tol=tol, **kw)

    return [
        # the smallest systems a user runs: launches and round trips count; default pair-pass settings
        case("md_1.5k", "md", 512, 32, 1e-6, tune=False),
        case("host_1.5k_fp64", "host", 512, 32, 1e-6, precision="double", tune=False),
        # a solute-sized box of mixed species, every molecule with radii and polarizabilities of one of five kinds
        case("md_8.6k_species", "md", 2851, 48, 1e-5, species=5),
        # a mid-sized box with the van der Waals term in the same pass, grid with factors 5 and 7
        case("md_24k_gvdw", "md", 8000, 70, 1e-4, gvdw=True),
        # a skewed, ragged box, FP64 with strain: a barostat's or a minimiser's call
        case("host_30k_fp64", "host", 10007, (75, 80, 72), 1e-5, precision="double", skew=0.2),
        # trajectory frames far apart: every one builds its list and solves from alpha E
        case("frames_12k", "frames", 4019, 63, 1e-5),
        # 98,304 atoms at liquid density, the box the reference publishes an MD rate for
        case("md_98k", "md", 32768, 112, 1e-4),
        # the 96,000-atom workload of bench.py (three times liquid density), both precisions
        case("eval_96k", "eval", 32000, 72, 1e-4, density=100.0),
        case("eval_96k_fp64", "eval", 32000, 72, 1e-4, density=100.0, precision="double"),
        # the largest box on one GPU: 999,000 atoms
        case("eval_999k", "eval", 333000, 216, 1e-5),
        # parameter fits: one system through the torch layer in FP64, and the 64-snapshot batch in mixed precision
        case("fit_1.5k_fp64", "fit", 512, 32, 1e-8, precision="double", snaps=1),
        case("fit_64", "fit", 2048, 0, 1e-8, snaps=64),
    ]


SMOOTH = sorted(
    v for v in (2**a * 3**b * 5**c * 7**d for a in range(8) for b in range(5) for c in range(3) for d in range(2)) if v <= 128
)


def draw(rng):
    kind = rng.choice(["md", "md", "eval", "host", "frames", "fit"])
    precision = "double" if kind == "host" else rng.choice(["mixed", "mixed", "double"]) if kind in ("eval", "fit") else "mixed"
    most = {"md": 33000, "eval": 33000 if precision == "mixed" else 16000, "host": 12000, "frames": 12000, "fit": 2048}[kind]
    nmol = int(round(math.exp(rng.uniform(math.log(512), math.log(most)))))
    if kind == "eval" and rng.random() < 0.3:
        density = rng.uniform(60.0, 100.0)
        nmol = max(nmol, 3000)
    else:
        density = LIQUID * rng.uniform(0.9, 1.1)
    edge = (nmol / density) ** (1.0 / 3.0)
    cutoff = round(rng.uniform(0.8, min(1.0, 0.44 * edge)), 3)
    spacing = rng.uniform(0.075, 0.1)
    near = [v for v in SMOOTH if edge / spacing <= v <= 1.15 * edge / spacing + 4] or [SMOOTH[-1]]
    kx, ky, kz = (rng.choice(near) for _ in range(3))
    case = {"kind": kind, "nmol": nmol, "kx": kx, "ky": ky, "kz": kz, "density": density, "cutoff": cutoff,
            "tol": rng.choice([1e-4, 1e-5, 1e-6]), "species": rng.choice([1, 1, 2, 5]),
            "order": rng.choice([6, 6, 6, 5, 8, 4]), "precision": precision, "tune": rng.random() < 0.7,
            "gvdw": kind == "md" and rng.random() < 0.25}  # fmt: skip
    if kind == "host" and rng.random() < 0.5 and nmol >= 2000:
        case["skew"] = round(rng.uniform(0.05, 0.25), 3)
    if kind == "fit":
        case["tol"] = 1e-8
        case["snaps"] = rng.choice([1, rng.randint(2, 8), rng.randint(9, 40)])
        if case["snaps"] > 1:
            case["kx"] = case["ky"] = case["kz"] = 0
    return case


# ------------------------------------------------------------------------------------------------ inputs


def water(case, seed, nmol=None, grid=None):
    """A seeded water box: jittered lattice sites, random orientations; species > 1: every molecule takes the radii
    and polarizabilities of one of that many kinds (the ranges of the package's ring liquid)."""
    nmol = nmol or case["nmol"]
    edge = (nmol / case["density"]) ** (1.0 / 3.0)
    grid = grid or (case["kx"], case["ky"], case["kz"])
    st = systems.base_settings(grid=grid, tol=case["tol"], cutoff=case["cutoff"], order=case["order"])
    nside = math.ceil(nmol ** (1.0 / 3.0) - 1e-9)
    sy = systems.water_box(nmol, edge, nside, seed, 0.02, "water", st)
    if case["species"] > 1:
        rng = np.random.default_rng([seed, 7])
        kind = rng.integers(0, case["species"], nmol)
        radius = np.stack([rng.uniform(0.065, 0.09, case["species"])] + 2 * [rng.uniform(0.05, 0.065, case["species"])], 1)
        alpha = np.stack([rng.uniform(0.7e-3, 1.2e-3, case["species"])] + 2 * [rng.uniform(0.3e-3, 0.6e-3, case["species"])], 1)
        sy.radius, sy.alpha = radius[kind].reshape(-1), alpha[kind].reshape(-1)
    if case.get("skew"):
        t = case["skew"]  # a reduced triclinic box of the same volume; the molecules move with their oxygen
        box = np.array([[edge, 0, 0], [t * edge, edge, 0], [-t * edge, 0.5 * t * edge, edge]])
        o = sy.pos[::3].repeat(3, 0)
        sy.pos = sy.pos - o + (o / edge) @ box
        sy.box = box
    return sy


def velocities(sy, seed):
    v = np.random.default_rng([seed, 11]).normal(0.0, 1.0, sy.pos.shape)
    return v / np.sqrt((v * v).sum(1)).mean()


def gvdw_parameters(sy):
    """Gaussian repulsion and dispersion on O, dispersion on H, intramolecular pairs skipped."""
    n = sy.n
    o = np.arange(0, n, 3)
    sa, sc, b = np.zeros(n), np.zeros(n), np.full(n, 0.9453)
    sa[o] = math.sqrt(422.0 * 4.184)
    sc[o] = math.sqrt(594.825035 * 4.184e-6)
    sc[o + 1] = sc[o + 2] = 0.3 * sc[o]
    return sa, sc, b, np.concatenate([o, o, o + 1]), np.concatenate([o + 1, o + 2, o + 2])


def history(sy, seed):
    """The converged dipoles of the four steps before (most recent first), as a running simulation has them."""
    e = engine.Engine.for_system(sy, precision="double", tol=1e-10, predictor=0, peek=0.0, max_iter=500)
    v, sets = velocities(sy, seed), []
    for k in range(4):
        e.compute(sy.pos - (k + 1) * STEP_NM * v, sy.box, forces=False)
        sets.append(e.induced_dipoles())
    return np.stack(sets)


def snapshots(case, seed):
    """The systems of a fit: uneven snapshots of 256 to nmol molecules on grids of 0.08 nm, or one system."""
    if case["snaps"] == 1:
        return [water(case, seed)]
    rng = np.random.default_rng([case["nmol"], case["snaps"]])  # the same sizes for every seed
    out = []
    for k, m in enumerate(rng.integers(256, case["nmol"] + 1, case["snaps"])):
        m = max(int(m), math.ceil((2.0 * case["cutoff"] + 0.1) ** 3 * case["density"]))
        K = systems.smooth_grid((m / case["density"]) ** (1.0 / 3.0))
        out.append(water(case, 1000 * seed + k, m, (K, K, K)))
    return out


def scaled(sy, f):
    return sy.q * f[0], sy.radius * f[1], sy.alpha * f[2], sy.cov_strength * f[3]


def fit_factors(seed):
    return 1.0 + 0.01 * np.random.default_rng([seed, 12]).standard_normal((2, 4))


def fit_targets(systems_, seed):
    """The reference forces of a fit (single system: the loss pulls the forces towards them) and the cotangent of a
    batch, in the caller's order."""
    n = sum(s.n for s in systems_)
    return np.random.default_rng([seed, 13]).normal(0.0, 1.0, (n, 3))


# ------------------------------------------------------------------------------------------------ prepare and run


def prepare(case, seed):
    dev = torch.device("cuda:0")
    s = {"case": case, "stream": torch.cuda.current_stream().cuda_stream}
    kind, precision = case["kind"], case["precision"]
    if kind == "fit":
        return prepare_fit(case, seed, s, dev)
    sy = water(case, seed)
    s["sy"], s["box"] = sy, sy.box
    e = s["engine"] = engine.Engine.for_system(sy, precision=precision)
    if case["gvdw"]:
        e.set_gvdw(0, case["cutoff"], *gvdw_parameters(sy))
    if kind == "frames":
        s["frames"] = [water(case, 100 * seed + k + 1).pos.astype(np.float32) for k in range(2)]
        e.compute_f32(sy.pos, sy.box)
        if case["tune"]:
            e.autotune(3)
        return s
    e.set_history(history(sy, seed))
    e.freeze_history(True)  # every pass is the same step
    if kind == "host":
        s["pos"] = sy.pos
        e.compute(sy.pos, sy.box)
    elif kind == "eval":
        s["pos"] = torch.from_numpy(sy.pos).to(dev)
        s["forces"] = torch.zeros((sy.n, 3), dtype=torch.float64, device=dev)
        e.compute_device_f64(s["pos"].data_ptr(), sy.box, True, s["forces"].data_ptr(), s["stream"])
    else:
        s["pos"] = torch.zeros((sy.n, 4), dtype=torch.float32, device=dev)
        s["pos"][:, :3] = torch.from_numpy(sy.pos).to(dev)
        s["fixed"] = torch.zeros((3, sy.n), dtype=torch.int64, device=dev)
        e.launch_device(s["pos"].data_ptr(), sy.box, True, s["fixed"].data_ptr(), sy.n, FIXED_SCALE, s["stream"])
        e.finish_device()
    if case["tune"]:
        e.autotune(3)
    return s


def prepare_fit(case, seed, s, dev):
    sys_ = snapshots(case, seed)
    fac = fit_factors(seed)
    s["target"] = torch.from_numpy(fit_targets(sys_, seed)).to(dev)
    keys = ("cutoff", "beta", "order", "max_iter", "ke", "skin", "polarizable")
    st = sys_[0].settings
    e = s["engine"] = engine.Engine(
        precision=case["precision"], grid=tuple(st["grid"]), tol=case["tol"], predictor=0, peek=0.0, **{k: st[k] for k in keys}
    )
    n = len(s["target"])
    off = np.concatenate([[0], np.cumsum([y.n for y in sys_])]).astype(np.int32)
    cat = lambda key: np.concatenate([getattr(y, key) for y in sys_])  # noqa: E731
    q, radius, alpha = cat("q"), cat("radius"), cat("alpha")
    cov_a = np.concatenate([y.cov_atom + off[k] for k, y in enumerate(sys_)])
    cov_p = np.concatenate([y.cov_partner + off[k] for k, y in enumerate(sys_)])
    strength = cat("cov_strength")
    s["pos"] = torch.from_numpy(cat("pos")).to(dev)
    if case["snaps"] == 1:
        # the types: O and H of every species (all entries of a covalent type share a strength)
        key = np.stack([q, radius, alpha], 1)
        vals, types = np.unique(key, axis=0, return_inverse=True)
        s["model"] = adjoint.PgmModel(e, types.reshape(-1), cov_a, cov_p, np.zeros(len(cov_a), np.int64), sys_[0].box)
        s["params"] = [
            [torch.tensor(v, dtype=torch.float64, device=dev) for v in (vals[:, 0] * f[0], vals[:, 1] * f[1], vals[:, 2] * f[2], strength[:1] * f[3])]
            for f in fac
        ]
        return s
    s["boxes"] = np.stack([y.box for y in sys_])
    s["cov"] = (cov_a, cov_p, strength * fac[0, 3])
    s["params"] = (q * fac[0, 0], radius * fac[0, 1], alpha * fac[0, 2])
    s["forces"] = torch.zeros((n, 3), dtype=torch.float64, device=dev)
    s["g"] = 1e-3 * s["target"]
    s["grads"] = [torch.empty(m, dtype=torch.float64, device=dev) for m in (n, n, n, len(cov_a))]
    e.set_atoms(*s["params"])
    e.set_covalent(*s["cov"])
    e.set_batch(off, np.array([y.settings["grid"] for y in sys_], np.int32))
    if case["tune"]:
        e.compute_batch_device(s["pos"].data_ptr(), s["boxes"], True, None, s["stream"])
        e.autotune(3)
    return s


def energies(terms, precision):
    v = np.array([list(t.values()) for t in (terms if isinstance(terms, list) else [terms])])
    return v.astype(np.float32) if precision == "mixed" else v


def run(s):
    case, e, stream = s["case"], s["engine"], s["stream"]
    kind, precision = case["kind"], case["precision"]
    real = torch.float32 if precision == "mixed" else torch.float64
    if kind == "md":
        n = s["sy"].n
        while True:  # a step whose pair list or solve fell short is taken again
            s["fixed"].zero_()
            e.launch_device(s["pos"].data_ptr(), s["box"], True, s["fixed"].data_ptr(), n, FIXED_SCALE, stream)
            terms, valid = e.finish_device()
            if valid:
                break
        forces = (s["fixed"].to(torch.float64) * (1.0 / FIXED_SCALE)).to(real)
        return {"terms": energies(terms, precision), "forces": forces.t()}
    if kind == "eval":
        s["forces"].zero_()
        terms = e.compute_device_f64(s["pos"].data_ptr(), s["box"], True, s["forces"].data_ptr(), stream)
        return {"terms": energies(terms, precision), "forces": s["forces"].to(real)}
    if kind == "host":
        terms, forces, strain = e.compute(s["pos"], s["box"], strain=True)
        return {"terms": energies(terms, precision), "forces": forces, "strain": strain}
    if kind == "frames":
        out = []
        for frame in s["frames"]:
            e.reset_history()
            terms, forces = e.compute_f32(frame, s["box"])
            out.append({"terms": energies(terms, precision), "forces": forces.astype(np.float32)})
        return out
    if case["snaps"] == 1:
        out = []
        for params in s["params"]:  # two steps of an optimiser
            params = [p.detach().requires_grad_() for p in params]
            e.reset_history()
            energy, forces = s["model"](*params, s["pos"])
            loss = ((forces - s["target"]) ** 2).mean() + 1e-3 * energy
            loss.backward()
            out.append({"energy": energy.reshape(1).to(real), "forces": forces.to(real), "grads": [p.grad.to(real) for p in params]})
        return out
    e.set_atoms(*s["params"])
    e.set_covalent(*s["cov"])
    e.reset_history()
    s["forces"].zero_()
    terms = e.compute_batch_device(s["pos"].data_ptr(), s["boxes"], True, s["forces"].data_ptr(), stream)
    e.backward_batch_device(
        s["pos"].data_ptr(), s["boxes"], s["g"].data_ptr(), None, *[t.data_ptr() for t in s["grads"]], stream
    )
    return {"terms": energies(terms, precision), "forces": s["forces"].to(real), "grads": [t.to(real) for t in s["grads"]]}


# ------------------------------------------------------------------------------------------------ work


def work(case):
    """Compulsory bytes (positions, parameters and history in, energies, forces and gradients out, each once) and the
    algorithmic operations: per half pair geometry 26, kernels 44, dual field 76, CG product 62, final body 152; per atom
    splines and spread 2,050, field gather 1,300, final gather 3,950; 5 K log2 K + 8 Kc per PME solve."""
    fit = case["kind"] == "fit"
    its = {1e-4: 3, 1e-5: 4, 1e-6: 6, 1e-8: 14}[case["tol"]] + (6 if case["kind"] == "frames" else 0)
    sizes = [(case["nmol"], (case["kx"], case["ky"], case["kz"]))]
    if fit and case["snaps"] > 1:
        rng = np.random.default_rng([case["nmol"], case["snaps"]])
        sizes = []
        for m in rng.integers(256, case["nmol"] + 1, case["snaps"]):
            m = max(int(m), math.ceil((2.0 * case["cutoff"] + 0.1) ** 3 * case["density"]))
            sizes.append((m, (systems.smooth_grid((m / case["density"]) ** (1.0 / 3.0)),) * 3))
    flops = nbytes = 0.0
    for nmol, K in sizes:
        n = 3.0 * nmol
        pairs = n * 3.0 * case["density"] * 4.0 / 3.0 * math.pi * case["cutoff"] ** 3 / 2.0
        kt = K[0] * K[1] * K[2]
        fft = 5.0 * kt * math.log2(kt) + 8.0 * K[0] * K[1] * (K[2] // 2 + 1)
        f = pairs * (312 + 62 * its) + n * (12100 + 3050 * its) + (its + 3) * fft
        b = n * (24 + 24 + 24 + (96 if case["kind"] in ("md", "eval", "host") else 0))
        if fit:
            f += its * (62 * pairs + 3050 * n + fft) + 2 * (178 * pairs + 3950 * n + fft)
            b += n * 48
        times = 2 if case["kind"] == "frames" or (fit and case["snaps"] == 1) else 1
        flops += times * f
        nbytes += times * b
    return {"bytes": nbytes, "flops": flops}


# ------------------------------------------------------------------------------------------------ the exact results


class Exact:
    """The pGM energy of one system in FP64 with plain torch operations: Gaussian charges and dipoles, smooth PME on the
    system's own grid, covalent dipoles, GVDW; derivatives by autograd, the induced dipoles by the engine's CG."""

    def __init__(self, sy, pos, dev="cuda:0", gvdw=None):
        t = lambda a: torch.as_tensor(np.asarray(a), device=dev, dtype=torch.float64)  # noqa: E731
        self.dev, self.st, self.n = dev, sy.settings, sy.n
        self.pos, self.box = t(pos).reshape(-1, 3), t(sy.box)
        self.q, self.R, self.alpha, self.c = t(sy.q), t(sy.radius), t(sy.alpha), t(sy.cov_strength)
        self.ca = torch.as_tensor(sy.cov_atom, device=dev, dtype=torch.int64)
        self.cp = torch.as_tensor(sy.cov_partner, device=dev, dtype=torch.int64)
        self.beta, self.ke = self.st["beta"], self.st["ke"]
        self.cself = 4.0 * self.beta**3 / (3.0 * math.sqrt(math.pi))
        self.i, self.j, self.shift = self.half_list()
        self.mod = [t(self.moduli(K, self.st["order"])) for K in self.st["grid"]]
        self.gvdw = None
        if gvdw is not None:
            sa, sc, b, si, sj = gvdw
            lo, hi = torch.as_tensor(np.minimum(si, sj), device=dev), torch.as_tensor(np.maximum(si, sj), device=dev)
            a, b_ = torch.minimum(self.i, self.j), torch.maximum(self.i, self.j)
            keep = ~torch.isin(a * self.n + b_, lo.long() * self.n + hi.long())
            self.gvdw = (t(sa), t(sc), t(b), keep)

    def image(self, x):
        """The shift (whole box vectors) of the minimum image: c first, then b, then a."""
        H = self.box
        s = torch.zeros_like(x)
        for a in (2, 1, 0):
            k = torch.round((x + s)[..., a] / H[a, a])
            s = s - k[..., None] * H[a]
        return s

    def half_list(self):
        rc2, rows = self.st["cutoff"] ** 2, max(1, 60_000_000 // self.n)
        ii, jj, ss = [], [], []
        for r0 in range(0, self.n, rows):
            x = self.pos[r0 : r0 + rows, None, :] - self.pos[None, :, :]
            s = self.image(x)
            d = x + s
            near = (d * d).sum(-1) < rc2
            near &= torch.arange(self.n, device=self.dev)[None, :] > torch.arange(r0, min(self.n, r0 + rows), device=self.dev)[:, None]
            a, b = near.nonzero(as_tuple=True)
            ii.append(a + r0)
            jj.append(b)
            ss.append(torch.round(s[a, b] @ torch.linalg.inv(self.box)))
        return torch.cat(ii), torch.cat(jj), torch.cat(ss)

    @staticmethod
    def moduli(K, p):
        m = np.zeros(p + 1)
        m[0] = 1.0
        for k in range(2, p + 1):
            m = np.array([(j * (m[j] if j < k - 1 else 0.0) + (k - j) * (m[j - 1] if j > 0 else 0.0)) / (k - 1) if j < k else 0.0
                          for j in range(p + 1)])  # fmt: skip
        k = np.arange(min(p - 1, K))
        b = np.abs((m[k + 1][None, :] * np.exp(2j * np.pi * np.arange(K)[:, None] * k[None, :] / K)).sum(1)) ** 2
        for x in np.nonzero(b < 1e-7)[0]:
            b[x] = 0.5 * (b[x - 1] + b[(x + 1) % K])
        return b

    def kernels(self, r, R, count):
        """G_0 .. G_{count-1} of the pairs: the damped erfc forms Bc_n(beta) - Bc_n(a)."""
        a = 1.0 / torch.sqrt(2.0 * R[self.i] ** 2 + 2.0 * R[self.j] ** 2)
        out = []
        for w in (torch.as_tensor(self.beta, device=self.dev, dtype=torch.float64), a):
            g = 2.0 / math.sqrt(math.pi) * w * torch.exp(-((w * r) ** 2))
            B = [torch.erfc(w * r) / r]
            for k in range(1, count):
                B.append(((2 * k - 1) * B[-1] + (2.0 * w * w) ** (k - 1) * g) / (r * r))
            out.append(B)
        return [u - v for u, v in zip(*out)]

    def splines(self, frac, K, p):
        w = frac * K
        base = torch.floor(w.detach())
        fr = w - base
        m, dm = [torch.ones_like(fr)], None
        for k in range(2, p + 1):
            z = torch.zeros_like(fr)
            hi, lo = m + [z], [z] + m
            if k == p:
                dm = [h - g for h, g in zip(hi, lo)]
            m = [((fr + j) * hi[j] + (k - fr - j) * lo[j]) / (k - 1) for j in range(k)]
        index = (base.long()[:, None] - torch.arange(p, device=self.dev)) % K
        return torch.stack(m, 1), torch.stack(dm, 1), index

    def reciprocal(self, pos, box, q, d):
        recip = torch.linalg.inv(box)
        volume = torch.linalg.det(box)
        K, p = self.st["grid"], self.st["order"]
        frac = pos @ recip
        frac = frac - torch.floor(frac.detach())
        (t1, u1, g1), (t2, u2, g2), (t3, u3, g3) = (self.splines(frac[:, a], K[a], p) for a in range(3))
        e = d @ recip * torch.tensor(K, device=self.dev, dtype=torch.float64)
        q = q[:, None]
        xy = ((q * t1 + e[:, :1] * u1)[:, :, None] * t2[:, None, :] + e[:, 1:2, None] * t1[:, :, None] * u2[:, None, :])
        val = xy[..., None] * t3[:, None, None, :] + (e[:, 2:3, None] * t1[:, :, None] * t2[:, None, :])[..., None] * u3[:, None, None, :]
        at = (g1[:, :, None, None] * K[1] + g2[:, None, :, None]) * K[2] + g3[:, None, None, :]
        grid = torch.zeros(K[0] * K[1] * K[2], dtype=torch.float64, device=self.dev).index_add(0, at.reshape(-1), val.reshape(-1))
        F = torch.fft.rfftn(grid.reshape(tuple(K)))
        f = [torch.fft.fftfreq(K[a], 1.0 / K[a], device=self.dev, dtype=torch.float64) for a in (0, 1)]
        f = [torch.where(v == -K[a] / 2, -v, v) for a, v in enumerate(f)]
        f3 = torch.arange(K[2] // 2 + 1, device=self.dev, dtype=torch.float64)
        m = torch.stack(torch.meshgrid(f[0], f[1], f3, indexing="ij"), -1) @ recip.t()
        m2 = (m * m).sum(-1)
        zero = torch.zeros_like(m2, dtype=torch.bool)
        zero[0, 0, 0] = True
        m2 = torch.where(zero, torch.ones_like(m2), m2)
        b = self.mod[0][:, None, None] * self.mod[1][None, :, None] * self.mod[2][None, None, : K[2] // 2 + 1]
        infl = torch.where(zero, torch.zeros_like(m2), torch.exp(-((math.pi / self.beta) ** 2) * m2) / (math.pi * volume * m2) / b)
        w = torch.full((K[2] // 2 + 1,), 2.0, dtype=torch.float64, device=self.dev)
        w[0] = 1.0
        if K[2] % 2 == 0:
            w[-1] = 1.0
        return 0.5 * (infl * w * (F.real**2 + F.imag**2)).sum()

    def displacements(self, pos, box):
        return pos[self.i] - pos[self.j] + self.shift @ box

    def permanent(self, pos, box, c):
        x = pos[self.cp] - pos[self.ca]
        with torch.no_grad():
            s = torch.round(self.image(x) @ torch.linalg.inv(self.box))
        x = x + s @ box
        u = x / torch.linalg.vector_norm(x, dim=1, keepdim=True)
        return torch.zeros_like(pos).index_add(0, self.ca, c[:, None] * u)

    def terms(self, pos, box, mu, q, R, alpha, c):
        """direct, reciprocal, self, background, polarization, gvdw [kJ/mol]."""
        d = self.permanent(pos, box, c) + mu
        x = self.displacements(pos, box)
        r = torch.linalg.vector_norm(x, dim=1)
        G = self.kernels(r, R, 3)
        qi, qj, di, dj = q[self.i], q[self.j], d[self.i], d[self.j]
        dix, djx = (di * x).sum(1), (dj * x).sum(1)
        direct = (qi * qj * G[0] + (qi * djx - qj * dix + (di * dj).sum(1)) * G[1] - dix * djx * G[2]).sum()
        rec = self.reciprocal(pos, box, q, d)
        self_ = -self.beta / math.sqrt(math.pi) * (q * q).sum() - 0.5 * self.cself * (d * d).sum()
        back = -math.pi * q.sum() ** 2 / (2.0 * torch.linalg.det(box) * self.beta**2)
        pol = ((mu * mu).sum(1) / (2.0 * alpha)).sum()
        vdw = torch.zeros((), dtype=torch.float64, device=self.dev)
        if self.gvdw is not None:
            sa, sc, b, keep = self.gvdw
            i, j, r = self.i[keep], self.j[keep], r[keep]
            w = 1.0 / torch.sqrt(2.0 * R[i] ** 2 + 2.0 * R[j] ** 2)
            y = w * r
            s, ex = y * y, torch.exp(-y * y)
            A = torch.erf(y) - 2.0 * y / math.sqrt(math.pi) * (1.0 + 2.0 / 3.0 * s) * ex
            g = 4.0 / (3.0 * math.sqrt(math.pi)) * s * y * ex
            vdw = (sa[i] * sa[j] * torch.exp(-0.5 * (b[i] + b[j]) * s) - sc[i] * sc[j] * w**6 * (A * A + 0.5 * g * g) / s**3).sum()
        return torch.stack([self.ke * direct, self.ke * rec, self.ke * self_, self.ke * back, self.ke * pol, vdw])

    def field(self, q, d):
        """-dE/dd of the direct, reciprocal and self energies of the charges and dipoles given, per ke."""
        i, j, x, (G1, G2) = self.i, self.j, self.x, self.g12
        di, dj = d[i], d[j]
        dix, djx = (di * x).sum(1, keepdim=True), (dj * x).sum(1, keepdim=True)
        f = torch.zeros_like(d)
        f.index_add_(0, i, (q[j][:, None] * G1 + djx * G2) * x - dj * G1)
        f.index_add_(0, j, (-q[i][:, None] * G1 + dix * G2) * x - di * G1)
        with torch.enable_grad():
            dd = d.detach().requires_grad_()
            (g,) = torch.autograd.grad(self.reciprocal(self.pos, self.box, q, dd), dd)
        return f - g + self.cself * d

    def induce(self, tol, peek, guess=None):
        with torch.no_grad():
            self.x = self.displacements(self.pos, self.box)
            G = self.kernels(torch.linalg.vector_norm(self.x, dim=1), self.R, 3)
            self.g12 = (G[1][:, None], G[2][:, None])
            zero, al = torch.zeros_like(self.q), self.alpha[:, None]
            b = self.field(self.q, self.permanent(self.pos, self.box, self.c))
            mu = self.solve(b, tol, peek, al * b if guess is None else guess, zero, al)
            del self.x, self.g12
        return mu

    def solve(self, b, tol, peek, x, zero, al):
        A = lambda v: v / al - self.field(zero, v)  # noqa: E731
        norm = (al * b).abs().mean()
        r = b - A(x)
        z = al * r
        p, rz = z, (r * z).sum()
        for _ in range(500):
            if (al * r).abs().max() / norm <= tol:
                break
            ap = A(p)
            step = rz / (p * ap).sum()
            x = x + step * p
            new = r - step * ap
            z = al * new
            top, r = (z * (new - r)).sum(), new
            p, rz = z + top / rz * p, (r * z).sum()
        return x + peek * al * r

    def results(self, mu, strain=False):
        pos = self.pos.clone().requires_grad_()
        eps = torch.zeros((3, 3), dtype=torch.float64, device=self.dev, requires_grad=True)
        h = torch.eye(3, dtype=torch.float64, device=self.dev) + eps
        t = self.terms(pos @ h.t(), self.box @ h.t(), mu, self.q, self.R, self.alpha, self.c)
        f, s = torch.autograd.grad(t.sum(), (pos, eps))
        return t.detach(), -f, s

    def gradients(self, mu, g, wE):
        """dL/d(q, R, alpha, c) of a loss with dL/dF = g and dL/dE = wE."""
        leaf = lambda v: v.detach().clone().requires_grad_()  # noqa: E731
        pos, m, q, R, al, c = (leaf(v) for v in (self.pos, mu, self.q, self.R, self.alpha, self.c))
        E = self.terms(pos, self.box, m, q, R, al, c).sum()
        er, em = torch.autograd.grad(E, (pos, m), create_graph=True)
        (b,) = torch.autograd.grad((er * g).sum() / self.ke, m, retain_graph=True)
        with torch.no_grad():
            self.x = self.displacements(self.pos, self.box)
            G = self.kernels(torch.linalg.vector_norm(self.x, dim=1), self.R, 3)
            self.g12 = (G[1][:, None], G[2][:, None])
            a = self.alpha[:, None]
            lam = self.solve(b, 1e-12, 0.0, a * b, torch.zeros_like(self.q), a)
            del self.x, self.g12
        return torch.autograd.grad(wE * E - (er * g).sum() + (em * lam).sum(), (q, R, al, c))


def exact(case, seed):
    kind = case["kind"]
    if kind == "fit":
        return exact_fit(case, seed)
    if case["nmol"] > 34000:
        return None
    sy = water(case, seed)
    gv = gvdw_parameters(sy) if case["gvdw"] else None
    tol, peek = case["tol"], sy.settings["peek"]
    if kind == "frames":
        out = []
        for k in range(2):
            x = Exact(sy, water(case, 100 * seed + k + 1).pos.astype(np.float32).astype(np.float64))
            t, f, _ = x.results(x.induce(tol, peek))
            out.append({"terms": t.reshape(1, -1), "forces": f})
        return out
    v = velocities(sy, seed)
    sets = []
    for k in range(4):
        x = Exact(sy, sy.pos - (k + 1) * STEP_NM * v)
        sets.append(x.induce(1e-10, 0.0))
        del x
    guess = 4.0 * sets[0] - 6.0 * sets[1] + 4.0 * sets[2] - sets[3]
    x = Exact(sy, sy.pos.astype(np.float32).astype(np.float64) if kind == "md" else sy.pos, gvdw=gv)
    t, f, s = x.results(x.induce(tol, peek, guess))
    out = {"terms": t.reshape(1, -1), "forces": f}
    if kind == "host":
        out["strain"] = s
    return out


def exact_fit(case, seed):
    sys_ = snapshots(case, seed)
    fac, target = fit_factors(seed), torch.from_numpy(fit_targets(sys_, seed)).to("cuda:0")
    if case["snaps"] == 1:
        out = []
        sy = sys_[0]
        _, types = np.unique(np.stack([sy.q, sy.radius, sy.alpha], 1), axis=0, return_inverse=True)
        types = torch.from_numpy(types.reshape(-1)).to("cuda:0")
        for f in fac:
            x = Exact(sy, sy.pos)
            x.q, x.R, x.alpha, x.c = x.q * f[0], x.R * f[1], x.alpha * f[2], x.c * f[3]
            mu = x.induce(1e-12, 0.0)
            t, forces, _ = x.results(mu)
            g = x.gradients(mu, 2.0 * (forces - target) / forces.numel(), 1e-3)
            per = [torch.zeros(int(types.max()) + 1, dtype=torch.float64, device="cuda:0").index_add(0, types, v) for v in g[:3]]
            out.append({"energy": t.sum().reshape(1), "forces": forces, "grads": per + [g[3].sum().reshape(1)]})
        return out
    terms, forces, grads, at = [], [], [[], [], [], []], 0
    for sy in sys_:
        sy.q, sy.radius, sy.alpha, sy.cov_strength = scaled(sy, fac[0])
        x = Exact(sy, sy.pos)
        mu = x.induce(1e-12, 0.0)
        t, f, _ = x.results(mu)
        terms.append(t)
        forces.append(f)
        for k, v in enumerate(x.gradients(mu, 1e-3 * target[at : at + sy.n], 0.0)):
            grads[k].append(v)
        at += sy.n
    return {"terms": torch.stack(terms), "forces": torch.cat(forces), "grads": [torch.cat(v) for v in grads]}
