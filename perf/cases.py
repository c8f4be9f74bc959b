"""Performance cases of the registration path, through the C ABI of claire_amd.

Fields live on the GPU (torch tensors whose addresses go through the ABI), the
problem object is claire_amd.Claire on the default stream.  A case is a plain
dict; its "kind" names the call that is timed:

  grad       spectral gradient of an image (clr_grad)
  precond    inverse regularization operator, the Krylov preconditioner
             (clr_apply_inv_reg)
  warp       an image resampled at arbitrary points (clr_interp_points)
  transport  a new velocity and the forward solve: all time steps of the
             warped template (clr_set_velocity, clr_solve_state)
  det        a new velocity and det(grad y) (clr_set_velocity,
             clr_det_def_grad)
  objective  the objective at a new velocity, a line-search trial
             (clr_evaluate_objective)
  step       objective and reduced gradient at a new velocity, the end of a
             Newton step (clr_evaluate_objective, clr_evaluate_gradient)
  matvec     Gauss-Newton Hessian matvec, the inner loop of the Krylov solver
             (clr_hessian_matvec)
  solve      a whole Gauss-Newton-Krylov registration (clr_solve_gn)
"""
import ctypes
import math

import torch

import claire_amd
from claire_amd import Claire, GNOptions, GNReport

SIZES = (16, 32, 48, 64, 96, 128, 150, 192, 256, 512)
TWO_PI = 2.0 * math.pi
BETA = {"h1": (1e-2, 1e-4, 0.0), "h2": (1e-3, 1e-1, 0.0), "h1sn": (1e-2, 1e-4, 0.0), "h2sn": (1e-3, 0.0, 0.0)}


def _case(kind, n, nt=4, cfl=2.0, norm="h1sn", precision="fp32", model="compressible", rk_order=2, pde="transport",
          solver="sl"):
    n1, n2, n3 = n
    return {"kind": kind, "n1": n1, "n2": n2, "n3": n3, "nt": nt, "cfl": cfl, "norm": norm, "precision": precision,
            "model": model, "rk_order": rk_order, "pde": pde, "solver": solver}


def listed():
    return [
        # the smallest call: one operator on a coarse grid, all launch latency
        dict(_case("grad", (32, 32, 32)), name="grad_32"),
        # preconditioner of a Krylov iteration on brain images of 128x150x128
        dict(_case("precond", (128, 150, 128), norm="h2"), name="precond_128x150x128"),
        # resampling an image along a deformation map, all three sizes unequal
        dict(_case("warp", (192, 150, 256), cfl=6.0), name="warp_192x150x256"),
        # forward warp by a large deformation, fourth-order characteristic
        dict(_case("transport", (128, 128, 128), cfl=9.0, rk_order=4), name="transport_128_rk4_cfl9"),
        # regularity check of a deformation on a batch-sized grid
        dict(_case("det", (96, 96, 96)), name="det_96"),
        # a line-search trial on a clinical-sized grid
        dict(_case("objective", (192, 192, 192)), name="objective_192"),
        # gradient evaluation after a Newton step, H1 regularization
        dict(_case("step", (128, 128, 128), norm="h1"), name="step_128_h1"),
        # Krylov matvec of the small registrations that are run in batches
        dict(_case("matvec", (64, 64, 64), norm="h1"), name="matvec_64_h1"),
        # the headline benchmark: Hessian matvec at 256^3
        dict(_case("matvec", (256, 256, 256)), name="matvec_256"),
        # incompressible registration, mixed precision storage, odd sizes
        dict(_case("matvec", (256, 192, 150), norm="h1", precision="mixed", model="stokes"),
             name="matvec_256x192x150_stokes_mixed"),
        # the largest single registration: 512^3, eight time steps
        dict(_case("matvec", (512, 512, 512), nt=8, cfl=3.0), name="matvec_512"),
        # a whole small registration, 64^3, from v = 0
        dict(_case("solve", (64, 64, 64)), name="solve_64"),
    ]


def draw(rng):
    kind = rng.choice(("grad", "precond", "warp", "transport", "det", "objective", "step", "matvec", "matvec", "matvec",
                       "solve"))
    sizes = [s for s in SIZES if (32 <= s <= 96 if kind == "solve" else s <= 256)]
    base = math.exp(rng.uniform(math.log(sizes[0]), math.log(sizes[-1] * 1.2)))
    near = min(range(len(sizes)), key=lambda i: abs(math.log(sizes[i] / base)))
    if rng.random() < 0.4:
        n = (sizes[near],) * 3
    else:  # ragged: each axis up to two sizes away
        n = tuple(sizes[min(max(near + rng.randint(-2, 1), 0), len(sizes) - 1)] for _ in range(3))
    if kind == "solve":
        return _case(kind, n)
    cfl = round(math.exp(rng.uniform(math.log(0.5), math.log(9.0))), 2)
    solver, pde, rk_order = "sl", "transport", 2
    if kind in ("transport", "objective", "step", "matvec"):
        if rng.random() < 0.15:  # explicit integrator: conditionally stable
            solver, cfl = "rk2", min(cfl, 0.5)
        elif kind in ("transport", "objective") and rng.random() < 0.2:
            pde = "continuity"
    if rng.random() < 0.25:
        rk_order = 4
    precision = "mixed" if kind == "matvec" and rng.random() < 0.3 else "fp32"
    model = "compressible"
    if kind in ("matvec", "step") and rng.random() < 0.25:
        model = "stokes"
    # fourth derivatives of single-precision fields amplify rounding by |k|^4:
    # the second-order norms are drawn where they are inverted
    norms = ("h1", "h2", "h1sn", "h2sn") if kind == "precond" else ("h1", "h1sn")
    return _case(kind, n, rng.choice((2, 4, 4, 8)), cfl, rng.choice(norms), precision, model, rk_order, pde, solver)


# --- inputs -----------------------------------------------------------------
def _shape(case):
    return case["n1"], case["n2"], case["n3"]


def _generator(seed, stream):
    g = torch.Generator(device="cpu")
    g.manual_seed(1000003 * int(seed) + stream)
    return g


def _smooth_field(shape, g, kmax):
    """Band-limited field: white noise of |w| <= kmax decayed by 1/(1+|w|^2)."""
    m = 2 * kmax + 1
    f = torch.fft.fftn(torch.randn((m, m, m), generator=g, dtype=torch.float64))
    w = torch.fft.fftfreq(m, 1.0 / m, dtype=torch.float64)
    f = f / (1.0 + w[:, None, None] ** 2 + w[None, :, None] ** 2 + w[None, None, :] ** 2)
    half = torch.zeros((shape[0], shape[1], shape[2] // 2 + 1), dtype=torch.complex64, device="cuda")
    rows = [torch.round(w).to(torch.int64) % n for n in shape[:2]]
    block = f[:, :, : kmax + 1].to(torch.complex64).cuda()
    half[rows[0].cuda()[:, None], rows[1].cuda()[None, :], : kmax + 1] = block
    return torch.fft.irfftn(half, s=shape)


def _velocity(case, seed, stream, cfl, kmax=8):
    """Random smooth velocity of CFL number max sum_i |v_i|/h_i / nt = cfl."""
    shape = _shape(case)
    g = _generator(seed, stream)
    k = min(kmax, min(shape) // 4)
    v = torch.empty((3,) + shape, dtype=torch.float32, device="cuda")
    for a in range(3):
        v[a] = _smooth_field(shape, g, k)
    top = torch.zeros(shape, dtype=torch.float32, device="cuda")
    for a in range(3):
        top += v[a].abs() * (shape[a] / TWO_PI)
    v *= cfl * case["nt"] / float(top.max())
    return v


def _image(case, seed, stream, count=24):
    """Sum of periodic Gaussian blobs of 2 to 8 cells, intensities in [0, 1]."""
    shape = _shape(case)
    g = _generator(seed, stream)
    centre, width, height = (torch.rand((count, 3), generator=g, dtype=torch.float64) * TWO_PI,
                             2.0 + 6.0 * torch.rand((count,), generator=g, dtype=torch.float64),
                             torch.rand((count,), generator=g, dtype=torch.float64))
    rows = []
    for a, n in enumerate(shape):
        h = TWO_PI / n
        x = torch.arange(n, dtype=torch.float64) * h
        d = torch.remainder(x[None, :] - centre[:, a : a + 1] + math.pi, TWO_PI) - math.pi
        rows.append(torch.exp(-0.5 * (d / (width[:, None] * h)) ** 2))
    rows[0] = rows[0] * height[:, None]
    r = [x.to(torch.float32).cuda() for x in rows]
    f = torch.zeros(shape, dtype=torch.float32, device="cuda")
    for b in range(count):
        f += r[0][b][:, None, None] * (r[1][b][:, None] * r[2][b][None, :])[None]
    return f


def _grid(shape, dtype):
    return [torch.arange(n, dtype=dtype, device="cuda").mul_(TWO_PI / n).reshape([-1 if a == i else 1 for i in range(3)])
            for a, n in enumerate(shape)]


def _points(case, seed):
    """Foot points of a smooth deformation of up to about cfl cells, over 2 pi."""
    shape = _shape(case)
    u = _velocity(dict(case, nt=1), seed, 5, case["cfl"])
    x = _grid(shape, torch.float32)
    return torch.stack([(x[a] - u[a]) / TWO_PI for a in range(3)], dim=-1).contiguous()


def _pair(case, seed):
    """Smooth template (sin^2 x1 + sin^2 x2 + sin^2 x3)/3 with random phases,
    and the same image seen through a smooth displacement."""
    shape = _shape(case)
    g = _generator(seed, 7)
    p = torch.rand(6, generator=g, dtype=torch.float64).tolist()
    x = [c + p[a] for a, c in enumerate(_grid(shape, torch.float64))]
    s = 0.2 + 0.1 * p[3]
    y = [x[0] + s * torch.sin(x[2]) * torch.cos(x[1]), x[1] + s * torch.sin(x[0]) * torch.cos(x[2] + p[4]),
         x[2] + s * torch.sin(x[1] + p[5]) * torch.cos(x[0])]
    f = [torch.broadcast_to((torch.sin(z[0]) ** 2 + torch.sin(z[1]) ** 2 + torch.sin(z[2]) ** 2) / 3.0, shape) for z in (x, y)]
    return [z.to(torch.float32).contiguous() for z in f]


def _inputs(case, seed):
    """The arrays a program has in hand, by name."""
    kind = case["kind"]
    if kind == "grad":
        return {"f": _image(case, seed, 1)}
    if kind == "precond":
        return {"f": _velocity(case, seed, 2, case["cfl"])}
    if kind == "warp":
        return {"f": _image(case, seed, 1), "X": _points(case, seed)}
    if kind == "solve":
        mT, mR = _pair(case, seed)
        return {"mT": mT, "mR": mR}
    d = {"v": _velocity(case, seed, 2, case["cfl"]), "mT": _image(case, seed, 1)}
    if kind in ("objective", "step"):
        d["mR"] = _image(case, seed, 4)
    if kind == "matvec":
        d["vt"] = _velocity(case, seed, 3, 1.0)
    return d


# --- the calls ----------------------------------------------------------------
class State:
    pass


def _call(name, *args):
    lib = claire_amd.lib()
    rc = getattr(lib, name)(*args)
    if rc != 0:
        raise RuntimeError("%s: %s" % (name, lib.clr_last_error().decode()))


def _p(t):
    return ctypes.c_void_p(t.data_ptr())


def prepare(case, seed):
    s = State()
    shape = _shape(case)
    kind = s.kind = case["kind"]
    s.inputs = d = _inputs(case, seed)
    s.problem = c = Claire(shape, nt=case["nt"], regnorm=case["norm"], beta=BETA[case["norm"]],
                           precision=case["precision"], rk_order=case["rk_order"], model=case["model"], pde=case["pde"],
                           pde_solver=case["solver"])
    s.ctx = c.ctx
    if "mT" in d:
        _call("clr_set_template_image", s.ctx, _p(d["mT"]))
    if "mR" in d:
        _call("clr_set_reference_image", s.ctx, _p(d["mR"]))
    scalar = kind in ("warp", "det")
    series = kind == "transport"
    out = (case["nt"] + 1,) + shape if series else shape if scalar else (3,) + shape
    s.out = torch.zeros(out, dtype=torch.float32, device="cuda")
    if kind == "matvec":
        _call("clr_set_velocity", s.ctx, _p(d["v"]))
        _call("clr_prepare_hessian", s.ctx)
    if kind == "solve":
        s.options = GNOptions()
        _call("clr_gn_options_default", ctypes.byref(s.options))
        s.options.maxit = 10
    return s


def run(s):
    d, ctx, out, kind = s.inputs, s.ctx, s.out, s.kind
    if kind == "grad":
        _call("clr_grad", ctx, _p(d["f"]), _p(out))
        return out
    if kind == "precond":
        _call("clr_apply_inv_reg", ctx, _p(d["f"]), _p(out), ctypes.c_int(0))
        return out
    if kind == "warp":
        _call("clr_interp_points", ctx, _p(d["f"]), _p(d["X"]), _p(out))
        return out
    if kind == "transport":
        _call("clr_set_velocity", ctx, _p(d["v"]))
        _call("clr_solve_state", ctx, _p(out))
        return out
    if kind == "det":
        stats = (ctypes.c_double * 3)()
        _call("clr_set_velocity", ctx, _p(d["v"]))
        _call("clr_det_def_grad", ctx, ctypes.c_int(0), _p(out), stats)
        return [out, list(stats)]
    if kind in ("objective", "step"):
        J, D, R = ctypes.c_double(), ctypes.c_double(), ctypes.c_double()
        _call("clr_evaluate_objective", ctx, _p(d["v"]), ctypes.byref(J), ctypes.byref(D), ctypes.byref(R))
        if kind == "objective":
            return [J.value, D.value, R.value]
        _call("clr_evaluate_gradient", ctx, None, _p(out))
        return [J.value, D.value, R.value, out]
    if kind == "matvec":
        _call("clr_hessian_matvec", ctx, _p(out), _p(d["vt"]), ctypes.c_int(1))
        return out
    report = GNReport()
    out.zero_()  # the initial guess v = 0
    _call("clr_solve_gn", ctx, _p(out), ctypes.byref(s.options), ctypes.byref(report), None, ctypes.c_int(0))
    return [out, report.iterations, report.pcg_iterations, report.J, report.D, report.gnorm / report.gnorm0]


# --- what a pass cannot do without ----------------------------------------------
def work(case):
    n1, n2, n3 = _shape(case)
    nl, nt, kind = float(n1 * n2 * n3), case["nt"], case["kind"]
    fft = 2.5 * math.log2(nl)  # real transform, per point
    gather = 160.0  # tricubic weights and 64 terms
    foot = 6 * gather * (1 if case["rk_order"] == 2 else 3)  # two trajectories
    sl = case["solver"] == "sl"
    state = nt * gather + foot if sl else nt * 8 * fft
    adjoint = nt * gather if sl else nt * 8 * fft
    if kind == "grad":
        return {"bytes": 16 * nl, "flops": 4 * fft * nl}
    if kind == "precond":
        return {"bytes": 24 * nl, "flops": 6 * fft * nl}
    if kind == "warp":
        return {"bytes": 20 * nl, "flops": gather * nl}
    if kind == "transport":  # v and the template in, nt + 1 images out
        return {"bytes": (12 + 4 + 4 * (nt + 1)) * nl, "flops": state * nl}
    if kind == "det":
        return {"bytes": 16 * nl, "flops": (foot + (nt + 1) * gather + 4 * fft) * nl}
    if kind == "objective":  # v and both images in
        return {"bytes": 20 * nl, "flops": (state + 6 * fft) * nl}
    if kind == "step":
        return {"bytes": 32 * nl, "flops": (state + adjoint + 4 * (nt + 1) * fft + 6 * fft) * nl}
    if kind == "matvec":  # v~ in, Hv~ out, foot points, coefficient, gradients of the state
        grads = (6 if case["precision"] == "mixed" else 12) * (nt + 1)
        return {"bytes": (24 + 24 + 4 + grads) * nl, "flops": ((nt + 2) * gather + adjoint + 6 * fft + 30 * nt) * nl}
    # a registration takes about three Newton steps of two matvecs here
    return {"bytes": 20 * nl, "flops": 6 * (2 * nt + 3) * gather * nl + 4 * state * nl}


# --- the same in 64 bits ------------------------------------------------------
class _Ref:
    """The discretization in float64: tricubic Lagrange semi-Lagrangian steps
    and Fourier derivatives whose Nyquist index counts as zero."""

    def __init__(self, case):
        self.case, self.shape, self.nt = case, _shape(case), case["nt"]
        self.nl = self.shape[0] * self.shape[1] * self.shape[2]
        self.ht = 1.0 / self.nt
        self.hd = TWO_PI ** 3 / self.nl
        self.norm, self.beta = case["norm"], BETA[case["norm"]]
        w = [torch.fft.fftfreq(n, 1.0 / n, dtype=torch.float64) for n in self.shape[:2]]
        w.append(torch.arange(self.shape[2] // 2 + 1, dtype=torch.float64))
        self.full, self.w = [], []
        for a, n in enumerate(self.shape):
            k = w[a].clone()
            k[n // 2] = n // 2
            z = k.clone()
            z[n // 2] = 0.0
            at = [-1 if a == i else 1 for i in range(3)]
            self.full.append(k.cuda().reshape(at))
            self.w.append(z.cuda().reshape(at))
        self.k2 = sum(z * z for z in self.w)

    def back(self, f):
        return torch.fft.irfftn(f, s=self.shape)

    def grad(self, f):
        s = torch.fft.rfftn(f)
        return [self.back(1j * z * s) for z in self.w]

    def div(self, v):
        return self.back(sum(1j * z * torch.fft.rfftn(c) for z, c in zip(self.w, v)))

    def multiply(self, v, m):
        return [self.back(m * torch.fft.rfftn(c)) for c in v]

    def symbol(self):
        b0, b1 = self.beta[:2]
        if self.norm in ("h1", "h1sn"):
            return b0 * (self.k2 + (b1 if self.norm == "h1" else 0.0))
        return b0 * (self.k2 ** 2 + (b1 if self.norm == "h2" else 0.0))

    def regularize(self, v):
        return self.multiply(v, self.symbol() * (1.0 if self.norm == "h2" else self.hd))

    def inverse(self, v):
        m = self.symbol()
        if self.norm in ("h1sn", "h2sn"):
            m = torch.where(self.k2 == 0, torch.full_like(m, self.beta[0]), m)
        return self.multiply(v, 1.0 / m)

    def functional(self, v):
        if self.norm in ("h1", "h1sn"):
            r = sum(float((g * g).sum()) for c in v for g in self.grad(c))
            if self.norm == "h1":
                r += self.beta[1] * sum(float((c * c).sum()) for c in v)
            return 0.5 * self.hd * self.beta[0] * r
        m = -self.k2 + (math.sqrt(self.beta[1]) if self.norm == "h2" else 0.0)
        return 0.5 * self.hd * self.beta[0] * sum(float((c * c).sum()) for c in self.multiply(v, m))

    def stencil(self, X):
        """Nodes and weights of the points X (three arrays over 2 pi)."""
        out = []
        for a, n in enumerate(self.shape):
            u = X[a] * n
            i = torch.floor(u)
            t = u - i + 1.0
            i = i.to(torch.int64) - 1
            w = [-(t - 1) * (t - 2) * (t - 3) / 6, t * (t - 2) * (t - 3) / 2, -t * (t - 1) * (t - 3) / 2,
                 t * (t - 1) * (t - 2) / 6]
            out.append([(torch.remainder(i + k, n), w[k]) for k in range(4)])
        return out

    def interp(self, fields, st):
        n1, n2, n3 = self.shape
        flat = [f.reshape(-1) for f in fields]
        out = [torch.zeros(self.shape, dtype=torch.float64, device="cuda") for _ in fields]
        for i, wi in st[0]:
            for j, wj in st[1]:
                row, wij = (i * n2 + j) * n3, wi * wj
                for k, wk in st[2]:
                    at, w = row + k, wij * wk
                    for f, o in zip(flat, out):
                        o += w * f[at]
        return out

    def points(self, v, sigma):
        x = _grid(self.shape, torch.float64)
        h = sigma * self.ht

        def at(step, u):
            return self.stencil([(x[a] - step * u[a]) / TWO_PI for a in range(3)])

        if self.case["rk_order"] == 2:
            vx = self.interp(v, at(h, v))
            return at(h / 2, [p + q for p, q in zip(vx, v)])
        k2 = self.interp(v, at(h / 2, v))
        k3 = self.interp(v, at(h / 2, k2))
        k4 = self.interp(v, at(h, k3))
        return at(h / 6, [a + 2 * b + 2 * c + d for a, b, c, d in zip(v, k2, k3, k4)])

    def coefficient(self, div, st, alpha):
        dx = alpha * self.interp([div], st)[0]
        return 1.0 + 0.5 * self.ht * (dx + alpha * (1.0 + self.ht * dx) * div)

    def forward(self, m, v):
        """m at all time steps, and the state trajectory where there is one."""
        series = [m]
        if self.case["solver"] == "rk2" and self.case["pde"] == "transport":
            for _ in range(self.nt):
                r0 = -sum(g * c for g, c in zip(self.grad(series[-1]), v))
                r1 = -sum(g * c for g, c in zip(self.grad(series[-1] + self.ht * r0), v))
                series.append(series[-1] + 0.5 * self.ht * (r0 + r1))
            return series, None
        st = self.points(v, 1.0)
        c = self.coefficient(self.div(v), st, -1.0) if self.case["pde"] == "continuity" else 1.0
        for _ in range(self.nt):
            series.append(c * self.interp([series[-1]], st)[0])
        return series, st

    def body_force(self, lam, grads, v):
        """hd * integral of lambda grad m, lambda transported backward from lam."""
        nt, ht = self.nt, self.ht
        rk2 = self.case["solver"] == "rk2"
        if not rk2:
            st = self.points(v, -1.0)
            c = 1.0 if self.case["model"] == "stokes" else self.coefficient(self.div(v), st, 1.0)
        b = [0.0, 0.0, 0.0]
        for j in range(nt + 1):
            weight = self.hd * (0.5 * ht if j in (0, nt) else ht)
            b = [b[a] + weight * lam * grads[nt - j][a] for a in range(3)]
            if j == nt:
                break
            if rk2:
                r0 = self.div([lam * c for c in v])
                r1 = self.div([(lam + ht * r0) * c for c in v])
                lam = lam + 0.5 * ht * (r0 + r1)
            else:
                lam = c * self.interp([lam], st)[0]
        if self.case["model"] == "stokes":
            k2 = sum(z * z for z in self.full)
            m = torch.where(k2 == 0, torch.full_like(k2, -1.0), -1.0 / torch.where(k2 == 0, torch.ones_like(k2), k2))
            s = [torch.fft.rfftn(c) for c in b]
            along = m * sum(z * c for z, c in zip(self.w, s))
            b = [c + self.back(z * along) for c, z in zip(b, self.w)]
        return b

    def matvec(self, v, mT, vt):
        series, st = self.forward(mT, v)
        grads = [self.grad(m) for m in series]
        mt = torch.zeros_like(mT)
        if st is None:
            for j in range(self.nt):
                r0 = -sum(g * c for g, c in zip(self.grad(mt), v)) - sum(g * c for g, c in zip(grads[j], vt))
                r1 = (-sum(g * c for g, c in zip(self.grad(mt + self.ht * r0), v))
                      - sum(g * c for g, c in zip(grads[j + 1], vt)))
                mt = mt + 0.5 * self.ht * (r0 + r1)
        else:
            vx = self.interp(vt, st)
            for j in range(self.nt):
                x = self.interp([mt] + grads[j], st)
                mt = x[0] - 0.5 * self.ht * (sum(g * c for g, c in zip(x[1:], vx)) +
                                             sum(g * c for g, c in zip(grads[j + 1], vt)))
        b = self.body_force(-mt, grads, v)
        return torch.stack([p + q for p, q in zip(self.regularize(vt), b)])


def exact(case, seed):
    kind = case["kind"]
    # a registration has no closed value; the largest grids take too long
    if kind == "solve" or case["n1"] * case["n2"] * case["n3"] > 1.1 * 256 ** 3:
        return None
    d = {k: x.double() for k, x in _inputs(case, seed).items()}
    ref = _Ref(case)
    if kind == "grad":
        return torch.stack(ref.grad(d["f"]))
    if kind == "precond":
        return torch.stack(ref.inverse(list(d["f"])))
    if kind == "warp":
        return ref.interp([d["f"]], ref.stencil([d["X"][..., a] for a in range(3)]))[0]
    v = list(d["v"])
    if kind == "transport":
        return torch.stack(ref.forward(d["mT"], v)[0])
    if kind == "det":
        st = ref.points(v, 1.0)
        c, J = ref.coefficient(ref.div(v), st, 1.0), torch.ones(_shape(case), dtype=torch.float64, device="cuda")
        for _ in range(case["nt"]):
            J = c * ref.interp([J], st)[0]
        return [J, [float(J.min()), float(J.max()), float(J.mean())]]
    if kind == "matvec":
        return ref.matvec(v, d["mT"], list(d["vt"]))
    series = ref.forward(d["mT"], v)[0]
    D = 0.5 * ref.hd * float(((d["mR"] - series[-1]) ** 2).sum())
    R = ref.functional(v)
    if kind == "objective":
        return [D + R, D, R]
    b = ref.body_force(d["mR"] - series[-1], [ref.grad(m) for m in series], v)
    return [D + R, D, R, torch.stack([p + q for p, q in zip(ref.regularize(v), b)])]
