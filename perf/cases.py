"""Performance cases of the reaction-diffusion and mass-effect solvers.

Each case is one call a user's program makes: a diffusion solve, a forward solve, a gradient
evaluation of one tumor or of an ensemble, a Hessian product, an elasticity solve, an advection step,
a smoothing of an input map, a mass-effect forward.  `exact` restates the same mathematics with
torch's FFTs in 64 bits.
"""
import ctypes
import math

import numpy as np
import torch

from glia_amd import _lib, adv, elasticity, mass_effect, rd

DEV = "cuda"
TWO_PI = 2.0 * math.pi

# grid lengths the engine plans (x and y; the z lengths leave out 48 and 80)
LENGTHS_XY = (32, 48, 64, 80, 96, 128, 160, 192, 256)
LENGTHS_Z = (32, 64, 96, 128, 160, 192, 256)

# CG iterations a pass is priced with: means over the synthetic brains (diffusion solves of half a
# step at dt = 0.02; elasticity solves to 1e-3)
DIFFUSION_ITERATIONS = 5.5
ELASTICITY_ITERATIONS = 48


def listed():
    """The cases; the grids and options are those of the benchmark, the tests and the input flow."""
    return [
        # one Crank-Nicolson solve on the smallest grid: launches and latency only
        dict(name="diffusion_32", kind="diffusion", n0=32, n1=32, n2=32),
        # the forward solve of the first benchmark configuration: 64^3, 50 steps
        dict(name="forward_64", kind="forward", n0=64, n1=64, n2=64, nt=50, members=1),
        # one tumor's gradient on the reference's test grid, the inner call of an inversion
        dict(name="gradient_64", kind="gradient", n0=64, n1=64, n2=64, nt=20, members=1, mode=2, slots=0, half=False),
        # an ensemble at 128^3 (the inversion and batching configurations), few steps of the 50
        dict(name="gradient_128x16", kind="gradient", n0=128, n1=128, n2=128, nt=4, members=16, mode=2, slots=0,
             half=False),
        # kappa/rho inversion (c0 fixed, half-step states kept) on a cropped, anisotropic grid
        dict(name="gradient_160x96x192x2", kind="gradient", n0=160, n1=96, n2=192, nt=5, members=2, mode=1, slots=0,
             half=True),
        # the headline ensemble, 8 members at 256^3
        dict(name="gradient_256x8", kind="gradient", n0=256, n1=256, n2=256, nt=2, members=8, mode=2, slots=0,
             half=False),
        # one tumor at imaging resolution under checkpointing (states recomputed)
        dict(name="gradient_256_checkpointed", kind="gradient", n0=256, n1=256, n2=256, nt=5, members=1, mode=0, slots=2,
             half=False),
        # Gauss-Newton: Hessian products of two members at 128^3
        dict(name="hessian_128x2", kind="hessian", n0=128, n1=128, n2=128, nt=4, members=2),
        # the displacement solve of the mass-effect grid, vectors resident on the GPU
        dict(name="elasticity_160", kind="elasticity", n0=160, n1=160, n2=160),
        # the advection of a mass-effect step's six fields at imaging resolution
        dict(name="advection_256x6", kind="advection", n0=256, n1=256, n2=256, fields=6),
        # smoothing of an atlas map (sigma of one cell), the input flow's device work
        dict(name="smoothing_192", kind="smoothing", n0=192, n1=192, n2=192, width=1.0),
        # the mass-effect forward (model 4) on its benchmark grid, three of its 41 steps
        dict(name="masseffect_160", kind="masseffect", n0=160, n1=160, n2=160, nt=2),
    ]


def _cost(case):
    """Relative cost of a case: grid points times steps, members or sweeps."""
    ng = case["n0"] * case["n1"] * case["n2"]
    k = case["kind"]
    if k == "gradient":
        extra = 2.0 if case["slots"] else 1.0
        return ng * case["members"] * (case["nt"] + 0.5) * 5.0 * extra
    if k == "hessian":
        return ng * case["members"] * (case["nt"] + 0.5) * 5.0
    if k == "forward":
        return ng * case["members"] * case["nt"] * 2.0
    if k == "elasticity":
        return ng * 48.0
    if k == "masseffect":
        return ng * 55.0 * (case["nt"] + 2)
    if k == "advection":
        return ng * (4.0 + case["fields"])
    return float(ng)


def draw(rng):
    """One more case of the ranges the listed ones stand for."""
    limit = max(_cost(c) for c in listed())
    while True:
        kind = rng.choice(["diffusion", "forward", "gradient", "gradient", "gradient", "hessian", "elasticity",
                           "advection", "smoothing", "masseffect"])
        if rng.random() < 0.4:
            n = rng.choice([v for v in LENGTHS_Z])
            shape = (n, n, n)
        else:
            shape = (rng.choice(LENGTHS_XY), rng.choice(LENGTHS_XY), rng.choice(LENGTHS_Z))
        case = dict(kind=kind, n0=shape[0], n1=shape[1], n2=shape[2])
        if kind in ("forward", "gradient", "hessian"):
            case["nt"] = int(round(math.exp(rng.uniform(math.log(2), math.log(50)))))
            case["members"] = int(round(math.exp(rng.uniform(0.0, math.log(16)))))
        if kind == "gradient":
            case["mode"] = rng.choice([0, 1, 2])
            case["slots"] = rng.choice([0, 0, 0, 2, 3])
            case["half"] = case["slots"] == 0 and rng.random() < 0.3
        if kind == "hessian":
            case["members"] = min(case["members"], 4)
        if kind == "advection":
            case["fields"] = rng.randint(1, 8)
        if kind == "smoothing":
            case["width"] = rng.choice([0.5, 1.0, 1.5, 2.0])
        if kind == "masseffect":
            case["nt"] = rng.choice([1, 2, 3])
        if kind in ("elasticity", "masseffect") and max(shape) > 3 * min(shape):
            continue  # a brain's bounding box, not a slab
        if _cost(case) <= 0.9 * limit and (kind != "gradient" or case["nt"] * case["members"] <= 100):
            return case


# ---------------------------------------------------------------------------------------------
# inputs: synthetic brains and tumors, made on the GPU from the seed alone
# ---------------------------------------------------------------------------------------------
def _shape(case):
    return (case["n0"], case["n1"], case["n2"])


def _rng(case, seed, member=0):
    return np.random.default_rng([int(seed), int(member), case["n0"], case["n1"], case["n2"]])


def _coords(shape):
    ax = [torch.arange(m, device=DEV, dtype=torch.float64) for m in shape]
    return ax[0][:, None, None], ax[1][None, :, None], ax[2][None, None, :]


def _ball(shape, centre, radii):
    x, y, z = _coords(shape)
    return ((x - centre[0]) / radii[0]) ** 2 + ((y - centre[1]) / radii[1]) ** 2 + ((z - centre[2]) / radii[2]) ** 2


def _blur(f, cells):
    """Periodic Gaussian blur with a width in cells."""
    w = [2 * math.pi * torch.fft.fftfreq(m, device=DEV, dtype=torch.float64) for m in f.shape[:2]]
    w.append(2 * math.pi * torch.fft.rfftfreq(f.shape[2], device=DEV, dtype=torch.float64))
    w2 = w[0][:, None, None] ** 2 + w[1][None, :, None] ** 2 + w[2][None, None, :] ** 2
    return torch.fft.irfftn(torch.fft.rfftn(f) * torch.exp(-0.5 * cells ** 2 * w2), s=f.shape)


def _brain(shape, rng):
    """White matter, gray matter, CSF and ventricle probabilities of nested ellipsoids (FP32)."""
    N = np.array(shape, dtype=np.float64)
    centre = N / 2 + rng.uniform(-0.02, 0.02, 3) * N
    rb = np.array([0.36, 0.30, 0.34]) * N * rng.uniform(0.95, 1.05, 3)
    brain = _ball(shape, centre, rb) <= 1
    inner = _ball(shape, centre, 0.9 * rb) <= 1
    white = _ball(shape, centre + rng.uniform(-0.02, 0.02, 3) * N, rb * rng.uniform(0.55, 0.65, 3)) <= 1
    off, rv = np.array([0.06, 0.0, 0.0]) * N, rb * np.array([0.16, 0.10, 0.12]) * rng.uniform(0.9, 1.1, 3)
    vent = (_ball(shape, centre + off, rv) <= 1) | (_ball(shape, centre - off, rv) <= 1)
    maps = [white & ~vent, inner & ~white & ~vent, brain & ~inner, vent]
    maps = [_blur(m.double(), 2.0).clamp_(min=0.0) for m in maps]
    total = maps[0] + maps[1] + maps[2] + maps[3]
    inside = (_blur(brain.double(), 2.0) > 0.5) & (total > 1e-6)
    wm, gm, csf, vt = [torch.where(inside, m / total.clamp(min=1e-6), torch.zeros_like(m)).float() for m in maps]
    return dict(wm=wm, gm=gm, csf=csf, vt=vt, centre=centre, radii=rb)


def _white_voxels(wm, count, rng):
    """Coordinates of distinct voxels with wm > 0.5."""
    cand = torch.nonzero(wm > 0.5).cpu().numpy()
    pick = rng.choice(cand.shape[0], size=count, replace=False)
    return cand[pick].astype(np.float64) * (TWO_PI / np.array(wm.shape, dtype=np.float64))


def _tumor(shape, brain, rng, cells=0.08):
    """A smooth tumor concentration in [0, 0.8] around a point of the white matter."""
    N = np.array(shape, dtype=np.float64)
    at = brain["centre"] + rng.uniform(-0.12, 0.12, 3) * N
    r2 = _ball(shape, at, cells * N * rng.uniform(0.8, 1.2, 3))
    return 0.8 * torch.exp(-0.5 * r2) * (brain["wm"].double() + brain["gm"].double())


def _rd_member(case, seed, m):
    """One member of an ensemble: tissue, basis, parameters, data and a fixed c(0)."""
    rng = _rng(case, seed, m)
    shape = _shape(case)
    b = _brain(shape, rng)
    nb = 64 if min(shape) >= 64 else 16
    centres = _white_voxels(b["wm"], nb, rng)
    p = np.zeros(nb)
    p[rng.choice(nb, size=8, replace=False)] = rng.uniform(0.1, 1.0, 8)
    tumor = _tumor(shape, b, rng)
    b.update(centers=centres, sigma=TWO_PI / 32 if min(shape) < 64 else TWO_PI / 64, p=p,
             direction=rng.standard_normal(nb), kappa=rng.uniform(0.01, 0.1), rho=rng.uniform(4.0, 15.0),
             c0=tumor.float(), d1=(_tumor(shape, b, rng, 0.14) > 0.3).float())
    return b


RATIOS = dict(k_gm_wm=0.2, r_gm_wm=0.2)
DT = 0.02


def _rd_solver(case, members):
    s = rd.RDSolver(_shape(case), nmembers=len(members), dt=DT, nt=case.get("nt", 1),
                    checkpoint_slots=case.get("slots", 0), adjoint_store=case.get("half", False), **RATIOS)
    for m, b in enumerate(members):
        torch.cuda.synchronize()  # the maps were made on torch's stream
        s.set_tissue(m, b["wm"], b["gm"], b["csf"], b["vt"])
        s.set_coefficients(m, b["kappa"], b["rho"])
        s.set_field(m, "c0", b["c0"])
    s.ctx_dt = DT / 2  # as every evaluation after the first finds it
    s.precFactor()
    return s


def _vector_case(case, seed):
    """Inputs of the elasticity and advection cases: tissue, a tumor, and vector fields."""
    rng = _rng(case, seed)
    shape = _shape(case)
    b = _brain(shape, rng)
    b["bg"] = (1.0 - (b["wm"] + b["gm"] + b["csf"] + b["vt"])).clamp(0.0, 1.0)
    b["c"] = _tumor(shape, b, rng).float()
    return b, rng


def _velocity(shape, rng):
    """Smooth velocities of a few sinusoids around a mean drift (the reference's advection test)."""
    x, y, z = [TWO_PI * c / m for c, m in zip(_coords(shape), shape)]
    v = []
    for _ in range(3):
        a, f, ph = rng.uniform(0.1, 1.0), rng.integers(1, 5, 3), rng.uniform(0, TWO_PI, 3)
        v.append((1.0 + a * torch.sin(int(f[0]) * x + ph[0]) * torch.cos(int(f[1]) * y + ph[1])
                  * torch.sin(int(f[2]) * z + ph[2])).float())
    return v


ADV_DT = 0.02
ADV_MODES = (1, 1, 2, 2, 1, 2, 1, 1)
ME = dict(dt=0.025, k=0.01, rho=8.0, k_gm_wm=0.0, r_gm_wm=0.0, forcing=6e4)


def prepare(case, seed):
    kind, shape = case["kind"], _shape(case)
    st = dict(case=case)
    if kind in ("forward", "gradient", "hessian", "diffusion"):
        members = [_rd_member(case, seed, m) for m in range(case.get("members", 1))]
        s = _rd_solver(case, members)
        st["solver"] = s
        if kind in ("gradient", "hessian"):
            for m, b in enumerate(members):
                if not (kind == "gradient" and case["mode"] == 1):
                    s.set_basis(m, b["centers"], b["sigma"])
                s.set_data(m, b["d1"], None, -0.99)
            st["x"] = [np.concatenate([b["p"] if s.np[m] else [], [b["kappa"], b["rho"]]])
                       for m, b in enumerate(members)]
        if kind == "hessian":
            s.objective_and_gradient(st["x"], 0)
            st["v"] = [np.concatenate([b["direction"], [0.0, 0.0]]) for b in members]
        if kind in ("forward", "diffusion"):
            st["c0"] = [b["c0"] for b in members]
            st["out"] = [torch.empty(shape, device=DEV) for _ in members]
    elif kind == "elasticity":
        b, rng = _vector_case(case, seed)
        st["stream"] = torch.cuda.Stream()
        s = elasticity.ElasticitySolver(shape, stream=st["stream"].cuda_stream)
        f = [b[k].cpu().numpy() for k in ("c", "wm", "gm", "csf", "vt", "bg")]
        s.set_material(*f)
        st.update(solver=s, f=_elastic_force(b["c"]), u=torch.zeros((3,) + shape, device=DEV))
    elif kind == "advection":
        b, rng = _vector_case(case, seed)
        st["stream"] = torch.cuda.Stream()
        st["solver"] = adv.SemiLagrangianSolver(shape, stream=st["stream"].cuda_stream)
        st["v"] = _velocity(shape, rng)
        st["fields"] = _adv_fields(case, b)
        st["out"] = [torch.empty(shape, device=DEV) for _ in st["fields"]]
    elif kind == "smoothing":
        b, _ = _vector_case(case, seed)
        st["solver"] = rd.RDSolver(shape)
        st["f"], st["out"] = b["gm"], torch.empty(shape, device=DEV)
    elif kind == "masseffect":
        b, _ = _vector_case(case, seed)
        s = mass_effect.MassEffectSolver(shape, ME["dt"], case["nt"], k=ME["k"], rho=ME["rho"], k_gm_wm=ME["k_gm_wm"],
                                         r_gm_wm=ME["r_gm_wm"])
        s.set_tissue(*[b[k].cpu().numpy() for k in ("wm", "gm", "csf", "vt")])
        st.update(solver=s, inputs=[b[k] for k in ("c", "wm", "gm", "vt", "csf")], bg=b["bg"])
        p = _lib.MeParams()
        s.L.glia_me_params_init(ctypes.byref(p))
        p.forcing_factor = ME["forcing"]
        st["params"] = p
    torch.cuda.synchronize()
    return st


def _elastic_force(c):
    """A force along the tumor's gradient."""
    h = [TWO_PI / m for m in c.shape]
    return (-1e2 * torch.stack(torch.gradient(c.double(), spacing=h))).float().contiguous()


def _adv_fields(case, b):
    names = ("gm", "wm", "vt", "csf", "c", "bg", "wm", "gm")
    return [b[k] for k in names[:case["fields"]]]


def run(state):
    case, s = state["case"], state["solver"]
    kind = case["kind"]
    if kind == "diffusion":
        s.set_field(0, "work", state["c0"][0])
        s.diffusion_solve("work", DT / 2)
        return s.get_field(0, "work", out=state["out"][0])
    if kind == "forward":
        for m, c0 in enumerate(state["c0"]):
            s.set_field(m, "c0", c0)
        s.solve_state(0)
        return [s.get_field(m, "ct", out=o) for m, o in enumerate(state["out"])]
    if kind == "gradient":
        J, dJ = s.objective_and_gradient(state["x"], case["mode"])
        return dict(J=J, dJ=dJ)
    if kind == "hessian":
        return s.hessian(state["v"])
    if kind == "elasticity":
        with torch.cuda.stream(state["stream"]):
            state["u"].zero_()
        s.solve_device(state["f"], state["u"])
        return state["u"]
    if kind == "advection":
        with torch.cuda.stream(state["stream"]):
            s.set_velocity(*state["v"])
            s.advect(state["fields"], ADV_MODES[:case["fields"]], ADV_DT, out=state["out"])
        return state["out"]
    if kind == "smoothing":
        s.set_field(0, "work", state["f"])
        s.smooth_field(0, "work", case["width"] * TWO_PI / case["n0"])
        return s.get_field(0, "work", out=state["out"])
    # masseffect: the tumor's state is advanced in place, as a simulation does
    f = [t.clone() for t in state["inputs"]]
    u = torch.zeros((3,) + _shape(case), device=DEV)
    v = torch.zeros_like(u)
    torch.cuda.synchronize()  # the solver's stream is its own
    up = (ctypes.c_void_p * 3)(*[u[d].data_ptr() for d in range(3)])
    vp = (ctypes.c_void_p * 3)(*[v[d].data_ptr() for d in range(3)])
    info = _lib.MeInfo()
    rc = s.L.glia_me_solve_state(s.h, ctypes.byref(state["params"]), *[t.data_ptr() for t in f], None,
                                 state["bg"].data_ptr(), up, vp, ctypes.byref(info))
    if rc != 0:
        raise rd.GliaError(rc, s.L.glia_me_last_error(s.h).decode())
    return f + [u, v]


def work(case):
    """Bytes: a CG iteration of a diffusion solve reads and writes x, r and p, reads k, and passes two
    spectra each way through memory between the two halves of the transform (15 fields); a solve's
    set-up costs as much.  The elasticity iteration: five vectors of three components updated, three
    coefficient fields, and ten spectra each way (three of u, seven of the products), three more
    each way for the preconditioner.  Pointwise steps: inputs and outputs once."""
    ng = case["n0"] * case["n1"] * case["n2"]
    R = 4.0 * ng
    lg = math.log2(ng)
    m = DIFFUSION_ITERATIONS + 1
    cn = (15 * R * m, m * (8 * 2.5 * ng * lg + 40 * ng))
    el = (ELASTICITY_ITERATIONS * (30 + 3 + 52) * R, ELASTICITY_ITERATIONS * (26 * 2.5 * ng * lg + 100 * ng))
    kind = case["kind"]
    if kind == "diffusion":
        b, f = cn[0] + 2 * R, cn[1] + 5 * ng * lg
    elif kind == "forward":
        nt, nm = case["nt"], case["members"]
        b, f = nm * nt * (2 * cn[0] + 5 * R), nm * nt * (2 * cn[1] + 5 * ng * lg)
    elif kind == "gradient":
        nt, nm = case["nt"], case["members"]
        solves = nt * (4 if case["half"] else 5)
        if case["slots"]:
            solves += nt * 2
        b, f = nm * (solves * cn[0] + nt * 20 * R), nm * (solves * cn[1] + nt * 30 * ng * lg)
    elif kind == "hessian":
        nt, nm = case["nt"], case["members"]
        b, f = nm * (5 * nt * cn[0] + nt * 14 * R), nm * (5 * nt * cn[1] + nt * 20 * ng * lg)
    elif kind == "elasticity":
        b, f = el
    elif kind == "advection":
        k = case["fields"]
        b, f = (3 + 2 + 2 * k) * R, (k + 4) * 150.0 * ng + 4 * 2.5 * ng * lg
    elif kind == "smoothing":
        b, f = 2 * R, 3 * 2 * (24 * case["width"] + 1) * ng
    else:
        steps = case["nt"] + 1
        b = (steps + 1) * el[0] + steps * (cn[0] + 50 * R)
        f = (steps + 1) * el[1] + steps * (cn[1] + 1500.0 * ng)
    return {"bytes": b, "flops": f}


def tolerance(case):
    """FP32 fields with FP64 reductions.  The CG solves stop at 1e-6 (diffusion) and 1e-3 (elasticity) of
    a norm, so a different rounding moves the last iterate within that; measured against 64 bits."""
    return {"rel": {"diffusion": 2e-6, "forward": 2e-5, "gradient": 2e-5, "hessian": 2e-5, "elasticity": 5e-6,
                    "advection": 5e-7, "smoothing": 2e-7, "masseffect": 2e-5}[case["kind"]]}


# ---------------------------------------------------------------------------------------------
# the same in 64 bits with torch's FFTs
# ---------------------------------------------------------------------------------------------
class _Spectral:
    """Wave numbers (the Nyquist mode zeroed), gradient and divergence on a periodic grid."""

    def __init__(self, shape):
        self.shape = shape
        w = [torch.fft.fftfreq(m, 1.0 / m, device=DEV, dtype=torch.float64) for m in shape[:2]]
        w.append(torch.fft.rfftfreq(shape[2], 1.0 / shape[2], device=DEV, dtype=torch.float64))
        for a, m in zip(w, shape):
            a[a.abs() == m // 2] = 0.0
        self.w = (w[0][:, None, None], w[1][None, :, None], w[2][None, None, :])
        self.w2 = self.w[0] ** 2 + self.w[1] ** 2 + self.w[2] ** 2

    def r2c(self, f):
        return torch.fft.rfftn(f)

    def c2r(self, F):
        return torch.fft.irfftn(F, s=self.shape)

    def grad(self, f):
        F = self.r2c(f)
        return [self.c2r(1j * w * F) for w in self.w]

    def div_hat(self, g):
        out = 1j * self.w[0] * self.r2c(g[0])
        out += 1j * self.w[1] * self.r2c(g[1])
        out += 1j * self.w[2] * self.r2c(g[2])
        return out

    def div(self, g):
        return self.c2r(self.div_hat(g))

    def smooth(self, f, sigma):
        """Periodic Gaussian of two images per axis, normalized by its discrete sum."""
        F = self.r2c(f)
        for a, m in enumerate(self.shape):
            x = torch.arange(m, device=DEV, dtype=torch.float64) * (TWO_PI / m)
            g = torch.exp(-x ** 2 / (2 * sigma ** 2)) + torch.exp(-(x - TWO_PI) ** 2 / (2 * sigma ** 2))
            G = torch.fft.rfft(g / g.sum()) if a == 2 else torch.fft.fft(g / g.sum())
            F = F * G.reshape([-1 if d == a else 1 for d in range(3)])
        return self.c2r(F)


def _cg(A, B, b, x, rtol, maxit):
    """Preconditioned CG from x, stopped on the preconditioned residual relative to ||B b||."""
    dot = lambda a, c: float((a * c).sum())  # noqa: E731
    r = b - A(x)
    z = B(r)
    ttol = rtol * math.sqrt(dot(B(b), B(b)))
    beta, p = dot(z, r), None
    if math.sqrt(dot(z, z)) <= ttol:
        return x
    old = 1.0
    for _ in range(maxit):
        p = z if p is None else z + (beta / old) * p
        w = A(p)
        a = beta / dot(p, w)
        x = x + a * p
        r = r - a * w
        z = B(r)
        if math.sqrt(dot(z, z)) <= ttol:
            break
        old, beta = beta, dot(z, r)
        if beta == 0:
            break
    return x


class _Diffusion:
    def __init__(self, sp, k, kbar, prec_dt):
        self.sp, self.k = sp, k
        self.P = 1.0 / (1.0 + 0.25 * prec_dt * kbar * sp.w2)

    def D(self, f):
        return self.sp.div([self.k * g for g in self.sp.grad(f)])

    def solve(self, c, tau):
        A = lambda v: v - 0.5 * tau * self.D(v)  # noqa: E731
        B = lambda v: self.sp.c2r(self.P * self.sp.r2c(v))  # noqa: E731
        return _cg(A, B, c + 0.5 * tau * self.D(c), c, 1e-6, 5000)


class _Member:
    """One member in 64 bits: coefficients, basis, forward, adjoint."""

    def __init__(self, shape, b, dt, nt):
        self.sp, self.b, self.dt, self.nt = _Spectral(shape), b, dt, nt
        self.h3 = TWO_PI ** 3 / float(np.prod(shape))
        wm, gm, vt = b["wm"].double(), b["gm"].double(), b["vt"].double()
        self.mask = (((b["wm"] > 0.1) | (b["gm"] > 0.1)) & (b["vt"] < 0.8)).double()
        self.mk, self.mr = wm + RATIOS["k_gm_wm"] * gm, wm + RATIOS["r_gm_wm"] * gm
        k = b["kappa"] * self.mk
        self.diff = _Diffusion(self.sp, k, float(k.sum() / self.mask.sum()), dt / 2)
        self.e = torch.exp(b["rho"] * self.mr * dt)

    def basis(self, i):
        shape, sigma = self.sp.shape, self.b["sigma"]
        x, y, z = [c * (TWO_PI / m) for c, m in zip(_coords(shape), shape)]
        ctr = self.b["centers"][i]
        r2 = (x - ctr[0]) ** 2 + (y - ctr[1]) ** 2 + (z - ctr[2]) ** 2
        g = self.sp.smooth(self.mask * torch.exp(-r2 / (2 * sigma ** 2)), TWO_PI / shape[0])
        return torch.where(torch.sqrt(r2) / sigma <= 5, g, torch.zeros_like(g))

    def phi(self, p):
        out, top = torch.zeros_like(self.mask), 0.0
        for i in np.flatnonzero(p):
            g = self.basis(i)
            out += float(p[i]) * g
            top = max(top, float(g.max()))
        return out / (top if top else 1.0)

    def phi_t(self, v):
        s, top = np.zeros(len(self.b["centers"])), 0.0
        for i in range(len(s)):
            g = self.basis(i)
            s[i] = float((g * v).sum())
            top = max(top, float(g.max()))
        return s / top

    def forward(self, c):
        hist, half, e = [c], [], self.e
        for _ in range(self.nt):
            c = self.diff.solve(c, self.dt / 2)
            half.append(c)
            c = self.diff.solve(c * e / (c * e + 1.0 - c), self.dt / 2)
            hist.append(c)
        return hist, half

    def adjoint(self, a, half, visit=None):
        for i in reversed(range(self.nt)):
            a = self.diff.solve(a, self.dt / 2)
            a = a * self.e / (half[i] * self.e + 1.0 - half[i]) ** 2
            a = self.diff.solve(a, self.dt / 2)
            if visit:
                visit(i, a)
        return a

    def gradient(self, mode):
        b = self.b
        c0 = b["c0"].double() if mode == 1 else self.phi(b["p"])
        hist, half = self.forward(c0)
        t = hist[-1] - b["d1"].double()
        gk, gr = [0.0], [0.0]

        def quad(i, a):
            w = 0.5 if i in (0, self.nt) else 1.0
            gc, ga = self.sp.grad(hist[i]), self.sp.grad(a)
            gk[0] += w * float((self.mk * (gc[0] * ga[0] + gc[1] * ga[1] + gc[2] * ga[2])).sum())
            gr[0] += w * float((self.mr * (hist[i] ** 2 - hist[i]) * a).sum())

        quad(self.nt, -t)
        a0 = self.adjoint(-t, half, quad)
        J = 0.5 * self.h3 * float((t * t).sum())
        gp = [] if mode == 1 else -self.h3 * self.phi_t(a0)
        return J, np.concatenate([gp, [self.h3 * self.dt * gk[0], 0.0 if mode == 0 else self.h3 * self.dt * gr[0]]])

    def hessian(self):
        hist, half = self.forward(self.phi(self.b["p"]))
        c = self.phi(self.b["direction"])
        for i in range(self.nt):
            c = self.diff.solve(c, self.dt / 2)
            c = c * self.e / (hist[i] * self.e + 1.0 - hist[i]) ** 2
            c = self.diff.solve(c, self.dt / 2)
        return np.concatenate([-self.h3 * self.phi_t(self.adjoint(-c, half)), [0.0, 0.0]])


def _interpolate(f, q):
    """Cubic Lagrange interpolation of f at x + q (grid units), periodic."""
    shape = f.shape
    x = _coords(shape)
    idx, wgt = [], []
    for a in range(3):
        base = torch.floor(q[a])
        t = q[a] - base
        wgt.append([-t * (t - 1) * (t - 2) / 6, (t + 1) * (t - 1) * (t - 2) / 2, -(t + 1) * t * (t - 2) / 2,
                    (t + 1) * t * (t - 1) / 6])
        idx.append([torch.remainder(x[a] + base + (k - 1), shape[a]).long() for k in range(4)])
    out, flat = torch.zeros(shape, device=DEV, dtype=torch.float64), f.reshape(-1)
    for i in range(4):
        for j in range(4):
            row = (idx[0][i] * shape[1] + idx[1][j]) * shape[2]
            acc = torch.zeros_like(out)
            for k in range(4):
                acc += wgt[2][k] * flat[row + idx[2][k]]
            out += wgt[0][i] * wgt[1][j] * acc
    return out


def _advect(sp, fields, modes, v, dt):
    s = [dt * m / TWO_PI for m in sp.shape]
    q1 = [-s[a] * v[a] for a in range(3)]
    q = [-0.5 * s[a] * (v[a] + _interpolate(v[a], q1)) for a in range(3)]
    dv = sp.div(v)
    dvi = _interpolate(dv, q)
    out = []
    for f, mode in zip(fields, modes):
        ci = _interpolate(f, q)
        if mode == 1:
            src = -ci * dvi
            ci = ci + 0.5 * dt * (src - (ci + dt * src) * dv)
        out.append(ci)
    return out


class _Elastic:
    """div(mu (grad u + grad u^T)) + grad(lam div u) - s u, and its constant-coefficient inverse."""

    def __init__(self, sp, c, wm, gm, csf, vt, bg):
        self.sp = sp
        mu = lambda E, nu: E / (2 * (1 + nu))  # noqa: E731
        la = lambda E, nu: nu * E / ((1 + nu) * (1 - 2 * nu))  # noqa: E731

        def mix(fn):
            a = fn(15000, 0.45) * bg + fn(2100, 0.4) * (wm + gm) + fn(100, 0.1) * (vt + csf)
            return a.clamp(min=0.0) + fn(8000, 0.45) * c.clamp(min=0.0)

        self.mu, self.lam = mix(mu), mix(la)
        low = torch.full_like(c, 1e-2)
        # thresholds on the FP32 fields a caller passes
        self.s = torch.where(c.float() >= 0.005, low, torch.full_like(c, 1e2))
        self.s = torch.where(bg.float() > 0.95, torch.full_like(c, 1e6), self.s)
        self.avg = [float(a.mean()) for a in (self.mu, self.lam, self.s)]

    def A(self, u):
        sp, w = self.sp, self.sp.w
        U = [sp.r2c(u[d]) for d in range(3)]
        L = sp.r2c(self.lam * sp.c2r(1j * (w[0] * U[0] + w[1] * U[1] + w[2] * U[2])))
        out = [1j * w[i] * L for i in range(3)]
        for i in range(3):
            for j in range(i, 3):
                S = sp.r2c(self.mu * sp.c2r(1j * (w[j] * U[i] + w[i] * U[j])))
                out[i] = out[i] + 1j * w[j] * S
                if i != j:
                    out[j] = out[j] + 1j * w[i] * S
        return torch.stack([sp.c2r(out[i]) - self.s * u[i] for i in range(3)])

    def B(self, f):
        sp, w, (mu, lam, scr) = self.sp, self.sp.w, self.avg
        F = [sp.r2c(f[d]) for d in range(3)]
        s1 = -scr - mu * sp.w2
        s2 = lam + mu
        c = s2 / (1.0 - sp.w2 * s2 / s1) / s1 ** 2
        wf = w[0] * F[0] + w[1] * F[1] + w[2] * F[2]
        return torch.stack([sp.c2r(F[d] / s1 + c * w[d] * wf) for d in range(3)])

    def solve(self, f, u):
        return _cg(self.A, self.B, f, u, 1e-3, 100)


def _mass_effect(case, b):
    sp = _Spectral(_shape(case))
    c, wm, gm, vt, csf, bg = [b[k].double() for k in ("c", "wm", "gm", "vt", "csf", "bg")]
    dt, sigma = ME["dt"], TWO_PI / case["n0"]
    mask = ((b["wm"] > 0.1) | (b["gm"] > 0.1)) & (b["vt"] < 0.8)
    kbar = float((ME["k"] * (wm + ME["k_gm_wm"] * gm)).sum() / mask.sum())
    wm, gm = wm * (1 - c), gm * (1 - c)

    def force():
        s = sp.smooth(c, sigma)
        return torch.stack([ME["forcing"] * g * torch.tanh(s) for g in sp.grad(s)])

    u = torch.zeros((3,) + sp.shape, device=DEV, dtype=torch.float64)
    v = torch.zeros_like(u)
    old = _Elastic(sp, c, wm, gm, csf, vt, bg).solve(force(), torch.zeros_like(u))
    for _ in range(case["nt"] + 1):
        if dt * float(torch.sqrt((v * v).sum(0)).max()) * case["n0"] / TWO_PI >= 14.0:
            break
        base = bg + vt + csf
        rho = ME["rho"] * (1 - base - (1 - ME["r_gm_wm"]) * gm).clamp(min=0.0)
        k = ME["k"] * (1 - base - (1 - ME["k_gm_wm"]) * gm).clamp(min=0.0)
        gm, wm, vt, csf, c = _advect(sp, (gm, wm, vt, csf, c), (1, 1, 2, 2, 1), v, dt)
        c = _Diffusion(sp, k, kbar, dt).solve(c, dt)
        e = torch.exp(rho * dt)
        c = c * e / (c * e + 1 - c)
        u = _Elastic(sp, c, wm, gm, csf, vt, bg).solve(force(), u)
        v = torch.stack([sp.smooth(a, sigma) for a in (u - old) / dt])
        old = u
    return [c, wm, gm, vt, csf, u, v]


def exact(case, seed):
    kind, shape = case["kind"], _shape(case)
    if kind in ("forward", "gradient", "hessian", "diffusion"):
        if _cost(case) > 2.0 * _cost(listed()[5]):
            return None
        J, out = [], []
        for i in range(case.get("members", 1)):
            m = _Member(shape, _rd_member(case, seed, i), DT, case.get("nt", 1))
            if kind == "diffusion":
                return m.diff.solve(m.b["c0"].double(), DT / 2)
            if kind == "forward":
                out.append(m.forward(m.b["c0"].double())[0][-1])
            elif kind == "hessian":
                out.append(m.hessian())
            else:
                j, g = m.gradient(case["mode"])
                J.append(j)
                out.append(g)
        return dict(J=np.array(J), dJ=out) if kind == "gradient" else out
    b, rng = _vector_case(case, seed)
    sp = _Spectral(shape)
    if kind == "elasticity":
        e = _Elastic(sp, *[b[k].double() for k in ("c", "wm", "gm", "csf", "vt", "bg")])
        f = _elastic_force(b["c"]).double()
        return e.solve(f, torch.zeros_like(f))
    if kind == "advection":
        v = _velocity(shape, rng)
        return _advect(sp, [f.double() for f in _adv_fields(case, b)], ADV_MODES[:case["fields"]],
                       [a.double() for a in v], ADV_DT)
    if kind == "smoothing":
        return sp.smooth(b["gm"].double(), case["width"] * TWO_PI / case["n0"])
    return _mass_effect(case, b)
