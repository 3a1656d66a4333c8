"""What a user of the framework has it do, as timed cases.

A case names a site (the physical set-up), a grid and what is called on it:

  advance    the time loop: pfhip_advance_richards over whole time steps
             (Newton-Krylov solves with the multigrid preconditioner), in
             the plain form (FP64, the reference's SPGMR) or the mixed form
             (FP32 V-cycle inside flexible GMRES)
  ensemble   the time loop of many small hillslopes advanced together
  residual   NlFunctionEval
  jacobian   RichardsJacobianEval (all seven couplings) and a Matvec with it
  precond    the preconditioner module: set-up from a PC matrix, then one
             V-cycle for each of three right-hand sides
  output     what an output step evaluates: saturation, relative
             permeability, face velocities, storage and water-balance fluxes
  nvector    the N_Vector operations a KINSOL that keeps its own Krylov loop
             calls: one modified Gram-Schmidt step and the stop-test norms

Sites (grid spacings, soils and forcing of parflow_amd/decks.py):

  box        homogeneous column box, dx = 1 m, dz = 0.5 m, infiltration
  basin      heterogeneous aquifer, dx = 10 m, dz = 1 m, infiltration
  valley     tilted V with kinematic overland flow on top, dx = 10 m,
             dz = 0.5 m, rain

Every input is made on the GPU from the seed alone.  exact() restates each
path in plain torch FP64.
"""
import ctypes as C
import math

import torch
import torch.nn.functional as F

from parflow_amd import api, decks
from parflow_amd.problem import BC_DIR_EQUIL, BC_FLUX, BC_OVERLAND, SolverOptions

PORO, SS, SRES, SSAT = 0.4, 1e-4, 0.2, 1.0
MANN, OV_EPS = 5.52e-6, 1e-5
SITES = {
    # dx (= dy), dz, dt, top flux (rain or infiltration, m/h), ResidualTol and
    # StepTol: the reference's defaults, or the residual alone at a tolerance
    # that closes the water balance
    "box": (1.0, 0.5, 0.1, -0.01, 1e-12, 1e-30),
    "basin": (10.0, 1.0, 0.5, -0.005, 1e-7, 1e-7),
    "valley": (10.0, 0.5, 0.05, -0.05, 1e-10, 1e-30),
}
RIGHT_HAND_SIDES = 3      # V-cycles per preconditioner set-up
BASIS = 4                 # Krylov vectors of the N_Vector case
ENSEMBLE_STEPS = 2


# ---------------------------------------------------------------- the cases
def _advance(name, site, nx, ny, nz, form, precond="PFMG", sweeps=1, krylov_dim=25, steps=1):
    return dict(name=name, kind="advance", site=site, nx=nx, ny=ny, nz=nz, form=form,
                precond=precond, sweeps=sweeps, krylov_dim=krylov_dim, steps=steps)


def listed():
    return [
        # the smallest run a user makes: a homogeneous 32^3 box, the
        # reference's algorithm throughout; launches and host round trips
        _advance("box 32^3 plain", "box", 32, 32, 32, "plain", steps=4),
        # a study site whose extents are odd, with the default preconditioner
        _advance("basin 131x97x25 plain", "basin", 131, 97, 25, "plain", precond="MGSemi",
                 krylov_dim=10, steps=2),
        # the drop-in form on a heterogeneous aquifer of 4.2M cells, and the
        # mixed form on the same
        _advance("basin 256x256x64 plain", "basin", 256, 256, 64, "plain", steps=2),
        _advance("basin 256x256x64 mixed", "basin", 256, 256, 64, "mixed", steps=2),
        # the benchmark's workload: 16.8M cells, mixed, two sweeps
        _advance("basin 512x512x64 mixed", "basin", 512, 512, 64, "mixed", sweeps=2,
                 krylov_dim=30, steps=2),
        # a catchment with overland flow under rain
        _advance("valley 512x512x32 mixed", "valley", 512, 512, 32, "mixed", sweeps=2,
                 krylov_dim=30, steps=2),
        # many small hillslopes at once (a parameter study)
        dict(name="ensemble of 64", kind="ensemble", members=64),
        # the modules a C driver calls by themselves, at ragged and even sizes
        dict(name="residual 301x203x47", kind="residual", site="basin", nx=301, ny=203, nz=47),
        dict(name="jacobian 256x256x64", kind="jacobian", site="basin", nx=256, ny=256, nz=64),
        dict(name="precond 512x512x64 fp32", kind="precond", site="basin", nx=512, ny=512, nz=64,
             precision=32, precond="PFMG", sweeps=2),
        dict(name="output 512x512x32", kind="output", site="valley", nx=512, ny=512, nz=32),
        # the vector operations of a small problem under a foreign KINSOL
        dict(name="nvector 64x64x40", kind="nvector", site="basin", nx=64, ny=64, nz=40),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["advance"] * 6 + ["ensemble", "residual", "jacobian", "precond", "output",
                                         "nvector"])
    if kind == "ensemble":
        return dict(kind=kind, members=_log_int(rng, 8, 64))
    site = rng.choice(["box", "basin", "basin", "valley"])
    case = dict(kind=kind, site=site, nx=_log_int(rng, 24, 512), ny=_log_int(rng, 24, 512),
                nz=_log_int(rng, 12, 64))
    if kind == "advance":
        form = rng.choice(["plain", "mixed"])
        while form == "plain" and case["nx"] * case["ny"] * case["nz"] > 4200000:
            case["nx"], case["ny"] = _log_int(rng, 24, 512), _log_int(rng, 24, 512)
        case.update(form=form, precond=rng.choice(["PFMG", "PFMG", "MGSemi"]),
                    sweeps=rng.choice([1, 2]), krylov_dim=rng.choice([10, 25, 30]), steps=1)
    if kind == "precond":
        case.update(precision=rng.choice([32, 64]), precond=rng.choice(["PFMG", "MGSemi"]),
                    sweeps=rng.choice([1, 2]))
    return case


# ------------------------------------------------------------------- inputs
def _zeros(*shape):
    return torch.zeros(shape, dtype=torch.float64, device="cuda")


def _rough(gen, shape):
    """A zero-mean field of about unit variance, correlated over some eight
    cells: white noise on a coarse lattice, interpolated, plus fine noise."""
    coarse = [max(2, (n + 7) // 8 + 1) for n in shape]
    c = torch.randn(coarse, generator=gen, dtype=torch.float64, device="cuda")
    up = F.interpolate(c[None, None], size=list(shape), mode="trilinear",
                       align_corners=True)[0, 0]
    fine = torch.randn(shape, generator=gen, dtype=torch.float64, device="cuda")
    return 1.3 * up + 0.5 * fine


def _ghosted(a, edge):
    """a with one ghost layer: zero, or repeating the edge value."""
    if edge:
        return F.pad(a[None, None], (1,) * 6, mode="replicate")[0, 0].contiguous()
    return F.pad(a, (1,) * 6).contiguous()


def _inner(g):
    return g[1:-1, 1:-1, 1:-1]


class Site:
    """The fields of one problem on the GPU and, on request, the framework's
    problem handle over them."""

    def __init__(self, case, seed):
        self.nx, self.ny, self.nz = nx, ny, nz = case["nx"], case["ny"], case["nz"]
        self.site = case["site"]
        self.dx, self.dz, self.dt, self.top, *self.tols = SITES[self.site]
        self.overland = self.site == "valley"
        gen = torch.Generator(device="cuda")
        gen.manual_seed(int(seed))
        self.gen = gen
        shape = (nz, ny, nx)
        ones = torch.ones(shape, dtype=torch.float64, device="cuda")
        if self.site == "basin":
            # ln K: mean ln 0.1 m/h; alpha lognormal; n uniform in [1.5, 3]
            self.K = torch.exp(math.log(0.1) + _rough(gen, shape))
            self.alpha = torch.exp(0.3 * torch.randn(shape, generator=gen, dtype=torch.float64,
                                                     device="cuda"))
            self.n = 1.5 + 1.5 * torch.rand(shape, generator=gen, dtype=torch.float64,
                                            device="cuda")
        else:
            # one soil, its conductivity drawn (m/h)
            u = torch.rand(1, generator=gen, dtype=torch.float64, device="cuda")
            self.K = ones * (1.0 if self.site == "box" else 0.01) * (0.8 + 0.4 * u)
            self.alpha, self.n = 2.0 * ones, 2.0 * ones
        self.poro, self.ss = PORO * ones, SS * ones
        depth = nz * self.dz
        z = (torch.arange(nz, dtype=torch.float64, device="cuda") + 0.5) * self.dz
        if self.overland:
            # two slopes towards a channel that falls along y
            x = (torch.arange(nx, dtype=torch.float64, device="cuda") + 0.5) / nx
            noise = torch.randn((2, ny, nx), generator=gen, dtype=torch.float64, device="cuda")
            slope = torch.where(x < 0.5, -1.0, 1.0) * (0.01 + 0.04 * (2.0 * x - 1.0).abs())
            self.slope_x = slope.expand(ny, nx) + 0.002 * noise[0]
            self.slope_y = 0.005 + 0.002 * noise[1]
        # hydrostatic above and below a level water table (m of head)
        self.bottom = min(decks.WATER_TABLE, 0.5 * depth)
        self.p0 = (self.bottom - z)[:, None, None].expand(shape).contiguous()
        self.handle = None

    def randn(self, *shape):
        return torch.randn(shape, generator=self.gen, dtype=torch.float64, device="cuda")

    def later(self):
        """A pressure some way into a run: p0 with local variation, and under
        rain a surface that is wet in places."""
        p = self.p0 + 0.05 * self.randn(self.nz, self.ny, self.nx)
        if self.overland:
            p[-1] = 0.02 * self.randn(self.ny, self.nx) - 0.01
        return p

    def make(self):
        """The framework's problem over these fields."""
        d = api.ProblemDescC()
        d.nx, d.ny, d.nz = self.nx, self.ny, self.nz
        d.dx = d.dy = self.dx
        d.dz = self.dz
        d.rho = d.mu = d.gravity = 1.0
        self.keep = {"kx": _ghosted(self.K, False)}
        for name, a in (("poro", self.poro), ("ss", self.ss), ("alpha", self.alpha),
                        ("nvg", self.n)):
            self.keep[name] = _ghosted(a, True)
        for name, t in self.keep.items():
            setattr(d, name, t.data_ptr())
        d.ky = d.kz = d.kx
        d.sres_value, d.ssat_value = SRES, SSAT
        for f in range(6):
            _bc(d.bc[f], BC_FLUX, 0.0)
        _bc(d.bc[4], BC_DIR_EQUIL, 0.0, self.bottom)
        _bc(d.bc[5], BC_OVERLAND if self.overland else BC_FLUX, self.top)
        if self.overland:
            self.keep["slope_x"] = F.pad(self.slope_x, (1,) * 4).contiguous()
            self.keep["slope_y"] = F.pad(self.slope_y, (1,) * 4).contiguous()
            self.keep["mann"] = F.pad(torch.full_like(self.slope_x, MANN), (1,) * 4).contiguous()
            for name in ("slope_x", "slope_y", "mann"):
                setattr(d, name, self.keep[name].data_ptr())
        d.ov_eps = OV_EPS
        d.base_unit = self.dt
        torch.cuda.synchronize()
        h = C.c_void_p()
        api.check(api.lib().pfhip_problem_create(C.byref(d), C.byref(h)), "pfhip_problem_create")
        self.handle = self.h = h
        api.check(api.lib().pfhip_bc_pressure(h, self.dt, None), "bc_pressure")
        return self

    def vector(self, a=None):
        """A ghosted vector of the problem, zero on its ghost layer."""
        if a is None:
            return _zeros(self.nz + 2, self.ny + 2, self.nx + 2)
        return _ghosted(a, False)

    def __del__(self):
        if self.handle is not None and api is not None:     # None at the interpreter's end
            api.lib().pfhip_problem_destroy(self.handle)


def _bc(b, kind, value, z_ref=0.0):
    b.type, b.n_intervals, b.repeat, b.z_ref = kind, 1, -1, z_ref
    b.lengths[0], b.values[0] = 1, value


class Array:
    """A torch tensor under the name the api's device arrays have."""

    def __init__(self, t):
        self.t, self.ptr, self.value = t, C.c_void_p(t.data_ptr()), t.data_ptr()


def _p(t):
    return C.c_void_p(t.data_ptr())


def _options(case, tols):
    return SolverOptions(residual_tol=tols[0], step_tol=tols[1],
                         krylov_dim=case["krylov_dim"], precond=case["precond"],
                         num_pre_relax=case["sweeps"], num_post_relax=case["sweeps"])


def prepare(case, seed):
    kind = case["kind"]
    if kind == "ensemble":
        return _prepare_ensemble(case, seed)
    st = {"kind": kind, "site": Site(case, seed).make()}
    s = st["site"]
    if kind == "advance":
        mixed = case["form"] == "mixed"
        st["solver"] = api.GPUSolver(s, _options(case, s.tols), precision=32 if mixed else 64,
                                     krylov=1 if mixed else 0)
        st["start"] = s.vector(s.p0)
        st["p"], st["s"] = Array(s.vector()), Array(s.vector())
        st["steps"] = case["steps"]
    elif kind == "residual":
        st["p"], st["p_old"], st["s_old"] = (s.vector(s.later()), s.vector(s.p0),
                                             s.vector(_closure(s, s.p0)[0]))
        st["F"] = s.vector()
    elif kind == "jacobian":
        st["p"], st["x"], st["y"] = s.vector(s.later()), s.vector(_direction(s)), s.vector()
        st["J"] = [s.vector() for _ in range(7)]
    elif kind == "precond":
        st["A"] = [s.vector(a) for a in _jacobian(s, s.later(), True)]
        st["b"] = [s.vector(_direction(s)) for _ in range(RIGHT_HAND_SIDES)]
        st["x"] = [s.vector() for _ in range(RIGHT_HAND_SIDES)]
        pre, post, sym = _sweeps(case)
        st["mg"] = api.GPUMultigrid(s, pre, post, sym, precision=case["precision"])
        C_, E, N, U = st["A"]
        zero = s.vector()
        st["zero"] = zero
        st["table"] = (C.c_void_p * 7)(*[t.data_ptr() for t in (C_, zero, E, zero, N, zero, U)])
    elif kind == "output":
        st["p"], st["p_old"] = s.vector(s.later()), s.vector(s.p0)
        st["s"], st["kr"] = s.vector(), s.vector()
        st["v"] = [_zeros(s.nz, s.ny, s.nx + 1), _zeros(s.nz, s.ny + 1, s.nx),
                   _zeros(s.nz + 1, s.ny, s.nx)]
    else:
        st["V"] = [s.vector(v) for v in _basis(s)]
        st["w"], st["u"], st["f"] = (s.vector(_direction(s)), s.vector(s.p0),
                                     s.vector(_direction(s)))
        st["one"] = s.vector(torch.ones_like(s.p0))
        st["out"], st["step"], st["scaled"] = s.vector(), s.vector(), s.vector()
    torch.cuda.synchronize()
    return st


def _sweeps(case):
    """(pre, post, symmetric) as the solver keys give them."""
    return SolverOptions(precond=case["precond"], num_pre_relax=case["sweeps"],
                         num_post_relax=case["sweeps"]).mg_params()


def _direction(s):
    """A Krylov direction: rough, with long waves."""
    return _rough(s.gen, (s.nz, s.ny, s.nx))


def _basis(s):
    """BASIS orthogonal unit vectors: fields on disjoint sets of cells."""
    out = []
    cells = torch.arange(s.nz * s.ny * s.nx, device="cuda").reshape(s.nz, s.ny, s.nx)
    for q in range(BASIS):
        v = torch.where(cells % BASIS == q, _direction(s), 0.0)
        out.append(v / v.norm())
    return out


def _prepare_ensemble(case, seed):
    # the decks' hillslopes, each with its water table moved by up to 0.2 m
    shift = torch.rand(case["members"], generator=torch.Generator().manual_seed(int(seed)),
                       dtype=torch.float64) * 0.4 - 0.2
    members = []
    for m in range(case["members"]):
        prob, opts, p0, dt = decks.c4_member(m)
        opts.residual_tol, opts.step_tol = 1e-12, 1e-30
        p0[1:-1, 1:-1, 1:-1] += float(shift[m])
        members.append((prob, opts, p0, dt))
    ens = api.GPUEnsemble([(prob, opts) for prob, opts, _, _ in members])
    # every member's vectors in one allocation, 256-byte aligned
    offsets, total = [], 0
    for _, _, p0, _ in members:
        offsets.append(total)
        total += (p0.size + 31) // 32 * 32
    start, p, s = _zeros(total), _zeros(total), _zeros(total)
    for o, (_, _, p0, _) in zip(offsets, members):
        start[o:o + p0.size] = torch.from_numpy(p0.ravel()).cuda()
    st = {"kind": "ensemble", "ensemble": ens, "start": start, "p": p, "s": s,
          "dt": [dt for _, _, _, dt in members]}
    st["dps"] = [Array(p[o:]) for o in offsets]
    st["dss"] = [Array(s[o:]) for o in offsets]
    torch.cuda.synchronize()
    return st


# ------------------------------------------------------------------- a pass
def run(st):
    kind, lib = st["kind"], api.lib()
    if kind == "ensemble":
        st["p"].copy_(st["start"])
        st["ensemble"].advance_device(st["dps"], st["dss"], 0.0, st["dt"], ENSEMBLE_STEPS)
        return st["p"], st["s"]
    s = st["site"]
    h = s.h
    if kind == "advance":
        st["p"].t.copy_(st["start"])
        st["solver"].advance_device(st["p"], st["s"], 0.0, s.dt, st["steps"])
        return st["p"].t, st["s"].t
    if kind == "residual":
        api.check(lib.pfhip_nl_function_eval(h, _p(st["p"]), _p(st["F"]), _p(st["p_old"]),
                                             _p(st["s_old"]), s.dt, None), "nl_function_eval")
        return st["F"]
    if kind == "jacobian":
        J = (C.c_void_p * 7)(*[t.data_ptr() for t in st["J"]])
        api.check(lib.pfhip_richards_jacobian_eval(h, _p(st["p"]), s.dt, 0, J, None),
                  "jacobian_eval")
        api.check(lib.pfhip_matvec(h, J, 0, _p(st["x"]), _p(st["y"]), None), "matvec")
        return st["J"] + [st["y"]]
    if kind == "precond":
        api.check(lib.pfhip_mg_setup(st["mg"].h, st["table"], None), "mg_setup")
        for b, x in zip(st["b"], st["x"]):
            api.check(lib.pfhip_mg_apply(st["mg"].h, _p(b), _p(x), None), "mg_apply")
        return st["x"]
    if kind == "output":
        return _run_output(lib, st, s, h)
    return _run_nvector(lib, st, h)


def _run_output(lib, st, s, h):
    p, sat = _p(st["p"]), _p(st["s"])
    api.check(lib.pfhip_saturation(h, p, sat, 0, None), "saturation")
    api.check(lib.pfhip_phase_rel_perm(h, p, _p(st["kr"]), 0, None), "phase_rel_perm")
    api.check(lib.pfhip_face_velocity(h, p, _p(st["p_old"]), s.dt, *[_p(v) for v in st["v"]],
                                      None), "face_velocity")
    sub, surf, flux = C.c_double(), C.c_double(), (C.c_double * 4)()
    api.check(lib.pfhip_water_balance_storage(h, p, sat, C.byref(sub), C.byref(surf), None),
              "water_balance_storage")
    api.check(lib.pfhip_water_balance_fluxes(h, p, _p(st["p_old"]), s.dt, flux, None),
              "water_balance_fluxes")
    return {"saturation": st["s"], "rel_perm": st["kr"], "velocity": st["v"],
            "storage": [sub.value, surf.value], "fluxes": list(flux)}


def _run_nvector(lib, st, h):
    # modified Gram-Schmidt of w against the basis, and its normalisation
    r, w, src = C.c_double(), _p(st["out"]), _p(st["w"])
    coefficients = []
    for v in st["V"]:
        api.check(lib.pfhip_vec_dot(h, _p(v), src, C.byref(r), None), "dot")
        coefficients.append(r.value)
        api.check(lib.pfhip_vec_linear_sum(h, 1.0, src, -r.value, _p(v), w, None), "linear_sum")
        src = w
    api.check(lib.pfhip_vec_dot(h, w, w, C.byref(r), None), "dot")
    coefficients.append(math.sqrt(r.value))
    api.check(lib.pfhip_vec_scale(h, 1.0 / coefficients[-1], w, w, None), "scale")
    # KINScSteplength: max |w / (1 + |u|)|; KINScFNorm and the weighted norm of f
    t, norms = _p(st["step"]), []
    api.check(lib.pfhip_vec_abs(h, _p(st["u"]), t, None), "abs")
    api.check(lib.pfhip_vec_add_const(h, t, 1.0, t, None), "add_const")
    api.check(lib.pfhip_vec_div(h, w, t, t, None), "div")
    api.check(lib.pfhip_vec_max_norm(h, t, C.byref(r), None), "max_norm")
    norms.append(r.value)
    api.check(lib.pfhip_vec_prod(h, _p(st["one"]), _p(st["f"]), _p(st["scaled"]), None), "prod")
    api.check(lib.pfhip_vec_max_norm(h, _p(st["scaled"]), C.byref(r), None), "max_norm")
    norms.append(r.value)
    api.check(lib.pfhip_vec_wl2_norm(h, _p(st["f"]), _p(st["one"]), C.byref(r), None), "wl2_norm")
    norms.append(r.value)
    return {"w": st["out"], "step": st["step"], "scaled": st["scaled"],
            "coefficients": coefficients, "norms": norms}


# --------------------------------------------------------------------- work
def work(case):
    """Bytes and operations of one pass, each array moved once per use the
    algorithm makes of it.  A time step is counted with the Newton and Krylov
    iterations that the sites take, rounded down."""
    kind = case["kind"]
    if kind == "ensemble":
        # a member has about 23 thousand cells on average
        n, steps, sweeps, w = 23000.0 * case["members"], ENSEMBLE_STEPS, 2, 4
    else:
        n = float(case["nx"]) * case["ny"] * case["nz"]
    if kind in ("advance", "ensemble"):
        if kind == "advance":
            steps, sweeps = case["steps"], case["sweeps"]
            w = 4 if case["form"] == "mixed" else 8
        newton, krylov = (6, 8) if case.get("site") == "basin" else (3, 3)
        # V-cycle over a hierarchy of twice the points: four couplings and b
        # read on the way down and up, x written and read, the transfers
        vcycle, vflops = 2 * 16 * w + 16, 2 * (2 * sweeps * 2 + 2) * 14
        per = newton * ((72 + 24) + (48 + 4 * w) + 24 * w) + krylov * (vcycle + 80 + 8 * 6)
        flops = newton * (2 * 300 + 500) + krylov * (vflops + 300 + 16)
        return {"bytes": n * steps * (per + 40), "flops": n * steps * flops}
    if kind == "residual":
        return {"bytes": n * 72, "flops": n * 300}
    if kind == "jacobian":
        return {"bytes": n * (48 + 56 + 56 + 16), "flops": n * 520}
    if kind == "precond":
        w = case["precision"] // 8
        vcycle = 2 * 16 * w + 16
        return {"bytes": n * (32 + 24 * w + RIGHT_HAND_SIDES * vcycle),
                "flops": n * (60 + RIGHT_HAND_SIDES * 2 * (4 * case["sweeps"] + 2) * 14)}
    if kind == "output":
        return {"bytes": n * (8 * 5 + 16 + 24 + 16), "flops": n * 250}
    return {"bytes": n * 8 * (BASIS * 4 + 2 + 2 + 4 + 4 + 2), "flops": n * (BASIS * 4 + 12)}


# ------------------------------------------------- the same in plain torch
def _powers(s, p):
    """(alpha h), 1 + (alpha h)^n and m of the van Genuchten curves; 1 where
    the cell is saturated (the caller masks those)."""
    ah = torch.where(p < 0, s.alpha * p.abs(), 1.0)
    return ah, 1.0 + ah ** s.n, 1.0 - 1.0 / s.n


def _closure(s, p):
    """Saturation and relative permeability."""
    ah, op, m = _powers(s, p)
    dry = p < 0
    sat = torch.where(dry, (SSAT - SRES) * op ** -m + SRES, SSAT)
    kr = torch.where(dry, (1.0 - ah ** (s.n - 1.0) * op ** -m) ** 2 * op ** (-m / 2.0), 1.0)
    return sat, kr


def _derivatives(s, p):
    """dS/dp and dkr/dp."""
    ah, op, m = _powers(s, p)
    n, al, dry = s.n, s.alpha, p < 0
    an = ah ** (n - 1.0)
    ds = torch.where(dry, m * n * al * an * (SSAT - SRES) * op ** (-m - 1.0), 0.0)
    co = 1.0 - an * op ** -m
    dk = (2.0 * co * op ** (-m / 2.0) *
          ((n - 1.0) * an / ah * al * op ** -m - an * m * op ** (-m - 1.0) * n * al * an) +
          co * co * (m / 2.0) * op ** (-m / 2.0 - 1.0) * n * al * an)
    return ds, torch.where(dry, dk, 0.0)


def _kr_at(s, value):
    """kr of the bottom cells' soil at a pressure."""
    if value >= 0.0:
        return torch.ones_like(s.alpha[0])
    ah, n = s.alpha[0] * abs(value), s.n[0]
    op, m = 1.0 + ah ** n, 1.0 - 1.0 / n
    return (1.0 - ah ** (n - 1.0) * op ** -m) ** 2 * op ** (-m / 2.0)


def _pair(a, ax):
    """The cells below and above every interior face along an axis."""
    n = a.shape[ax]
    return a.narrow(ax, 0, n - 1), a.narrow(ax, 1, n - 1)


def _face_terms(s, ax, p):
    """Along axis ax (0 z, 1 y, 2 x) of every interior face: driving
    difference per length, and conductance per area."""
    lo, hi = _pair(p, ax)
    ka, kb = _pair(s.K, ax)
    d = s.dz if ax == 0 else s.dx
    drive = (lo - hi) / d
    if ax == 0:
        drive = drive - 1.0
    return drive, 2.0 * ka * kb / (ka + kb), d


def _area(s, ax):
    return s.dx * s.dx if ax == 0 else s.dx * s.dz


def _velocities(s, p, kr):
    """Darcy velocities of the interior faces, z, y, x."""
    out = []
    for ax in range(3):
        drive, cond, _ = _face_terms(s, ax, p)
        ka, kb = _pair(kr, ax)
        out.append(cond * drive * torch.where(drive >= 0, ka, kb))
    return out


def _bottom_velocity(s, p, kr):
    value = s.bottom           # hydrostatic pressure at the bottom face
    drive = (value - p[0]) / s.dz - 0.5
    return torch.where(drive >= 0, _kr_at(s, value), kr[0]) * s.K[0] * 2.0 * drive


def _overland(s, p):
    """Kinematic fluxes through the surface faces: qx (ny, nx + 1) and qy
    (ny + 1, nx), the outer faces included."""
    top = p[-1].clamp(min=0.0)
    mag = torch.sqrt(s.slope_x ** 2 + s.slope_y ** 2).clamp(min=OV_EPS)
    den = torch.sqrt(mag) * MANN
    out = []
    for ax, slope in ((1, s.slope_x), (0, s.slope_y)):
        ahead = torch.cat([top.narrow(ax, 1, top.shape[ax] - 1),
                           torch.zeros_like(top.narrow(ax, 0, 1))], ax)
        q = -(slope / den) * torch.where(slope <= 0, top, ahead) ** (5.0 / 3.0)
        edge = -(slope / den) * top ** (5.0 / 3.0)
        first = torch.where(slope > 0, edge, 0.0).narrow(ax, 0, 1)
        out.append(torch.cat([first, q], ax))
    return out


def _surface_inflow(s, p, p_old):
    """What the overland top adds to F beside its flux: the change of the
    ponded water and the divergence of the surface fluxes, m^3."""
    qx, qy = _overland(s, p)
    a = s.dx * s.dx
    div = (qx[:, 1:] - qx[:, :-1] + qy[1:] - qy[:-1]) / s.dx
    return a * (p[-1].clamp(min=0.0) - p_old[-1].clamp(min=0.0)) + s.dt * a * div


def _residual(s, p, p_old, sat_old):
    sat, kr = _closure(s, p)
    vol = s.dx * s.dx * s.dz
    f = (sat - sat_old) * s.poro * vol + s.ss * vol * (p * sat - p_old * sat_old)
    for ax, v in enumerate(_velocities(s, p, kr)):
        q = s.dt * _area(s, ax) * v
        n = f.shape[ax]
        f.narrow(ax, 0, n - 1).add_(q)
        f.narrow(ax, 1, n - 1).sub_(q)
    f[0] -= s.dt * s.dx * s.dx * _bottom_velocity(s, p, kr)
    if s.overland:
        f[-1] += _surface_inflow(s, p, p_old)
    f[-1] += s.dt * s.dx * s.dx * s.top
    return f


def _jacobian(s, p, symmetric):
    """The Jacobian's couplings: C, E, N, U of the symmetric part, or C, W,
    E, S, N, L, U.  Without the surface couplings of an overland top."""
    sat, kr = _closure(s, p)
    ds, dk = _derivatives(s, p)
    vol = s.dx * s.dx * s.dz
    c = ds * s.poro * vol + s.ss * vol * (ds * p + sat)
    up, low = [], []
    for ax in range(3):
        drive, cond, d = _face_terms(s, ax, p)
        ka, kb = _pair(kr, ax)
        da, db = _pair(dk, ax)
        x = s.dt * _area(s, ax) * cond
        fwd = drive >= 0
        sym = -x / d * torch.where(fwd, ka, kb)
        t1 = sym - x * drive * torch.where(fwd, da, 0.0)
        t2 = sym + x * drive * torch.where(fwd, 0.0, db)
        n = c.shape[ax]
        c.narrow(ax, 0, n - 1).sub_(t1)
        c.narrow(ax, 1, n - 1).sub_(t2)
        u, l_ = torch.zeros_like(c), torch.zeros_like(c)
        u.narrow(ax, 0, n - 1).copy_(sym if symmetric else t2)
        l_.narrow(ax, 1, n - 1).copy_(t1)
        up.append(u)
        low.append(l_)
    value = s.bottom
    drive = (value - p[0]) / s.dz - 0.5
    g = 2.0 * s.dt * s.dx * s.dx * s.K[0]
    c[0] -= g * torch.where(drive >= 0, -_kr_at(s, value) / s.dz,
                            drive * dk[0] - kr[0] / s.dz)
    if symmetric:
        return [c, up[2], up[1], up[0]]
    return [c, low[2], up[2], low[1], up[1], low[0], up[0]]


def _neighbours(up, x):
    """Sum of the off-diagonal terms of a symmetric-stored operator (up: the
    couplings to the upper neighbour along z, y, x)."""
    out = torch.zeros_like(x)
    for ax in range(3):
        n = x.shape[ax]
        if n < 2:
            continue
        u = up[ax].narrow(ax, 0, n - 1)
        out.narrow(ax, 0, n - 1).addcmul_(u, x.narrow(ax, 1, n - 1))
        out.narrow(ax, 1, n - 1).addcmul_(u, x.narrow(ax, 0, n - 1))
    return out


def _shift(a, ax, by):
    """a moved by one cell along ax, zero entering."""
    z, n = torch.zeros_like(a), a.shape[ax]
    if by > 0:
        z.narrow(ax, 1, n - 1).copy_(a.narrow(ax, 0, n - 1))
    else:
        z.narrow(ax, 0, n - 1).copy_(a.narrow(ax, 1, n - 1))
    return z


class Levels:
    """The semicoarsened hierarchy of a symmetric-stored operator: the
    direction of the smallest spacing is halved, coarse points are the even
    ones, weights are induced by the operator at the odd points and the
    off-direction couplings are collapsed."""

    def __init__(self, s, A, pre, post, symmetric):
        self.pre, self.post, self.symmetric = pre, post, symmetric
        c, up = A[0], [A[3], A[2], A[1]]
        n, d = [s.nx, s.ny, s.nz], [s.dx, s.dx, s.dz]
        self.levels = []
        while True:
            ax = None
            best = sum(d)
            for q in range(3):
                if n[q] >= 2 and d[q] < best:
                    best, ax = d[q], 2 - q
            idx = sum(torch.meshgrid(*[torch.arange(m, device="cuda") for m in c.shape],
                                     indexing="ij"))
            self.levels.append({"c": c, "up": up, "ax": ax, "red": idx % 2 == 1})
            if ax is None or len(self.levels) == 100:
                break
            d[2 - ax] *= 2
            n[2 - ax] = (n[2 - ax] + 1) // 2
            c, up = self._coarsen(self.levels[-1])

    @staticmethod
    def _coarsen(lv):
        c, up, ax = lv["c"], lv["up"], lv["ax"]
        off = [q for q in range(3) if q != ax]
        lateral = c.clone()
        for q in off:
            lateral += up[q] + _shift(up[q], q, 1)
        below = _shift(up[ax], ax, 1)
        safe = torch.where(lateral != 0, lateral, 1.0)
        w1 = torch.where(lateral != 0, -below / safe, 0.0)
        w2 = torch.where(lateral != 0, -up[ax] / safe, 0.0)
        odd = torch.arange(c.shape[ax], device="cuda") % 2 == 1
        odd = odd.reshape([-1 if q == ax else 1 for q in range(3)])
        lv["w1"], lv["w2"] = torch.where(odd, w1, 0.0), torch.where(odd, w2, 0.0)

        def even(a):
            return a.index_select(ax, torch.arange(0, a.shape[ax], 2, device="cuda"))

        cc = even(lateral + below * _shift(lv["w2"], ax, 1) + up[ax] * _shift(lv["w1"], ax, -1))
        coarse = [None] * 3
        for q in off:
            u = up[q] + 0.5 * _shift(up[q], ax, 1) + 0.5 * _shift(up[q], ax, -1)
            coarse[q] = even(u)
            cc = cc - coarse[q] - _shift(coarse[q], q, 1)
        u = even(_shift(up[ax], ax, -1) * _shift(lv["w1"], ax, -1))
        u.narrow(ax, u.shape[ax] - 1, 1).zero_()
        coarse[ax] = u
        return cc, coarse

    @staticmethod
    def _smooth(lv, x, b, zero, sweeps, symmetric):
        count, red = (1 if symmetric else 2), True
        if zero:
            count += 1
            x = torch.zeros_like(b)
            if count // 2 > sweeps and not symmetric:
                return x
            x = torch.where(lv["red"], b / lv["c"], x)
            red = False
        while count // 2 <= sweeps:
            new = (b - _neighbours(lv["up"], x)) / lv["c"]
            x = torch.where(lv["red"] == red, new, x)
            red = not red
            count += 1
        return x

    def cycle(self, b, l=0):
        lv = self.levels[l]
        if l == len(self.levels) - 1:
            return self._smooth(lv, None, b, True, 1, self.symmetric)
        ax = lv["ax"]
        x = self._smooth(lv, None, b, True, self.pre, self.symmetric)
        r = b - lv["c"] * x - _neighbours(lv["up"], x)
        r = r + (_shift(lv["w2"] * r, ax, 1) + _shift(lv["w1"] * r, ax, -1))
        at = torch.arange(0, r.shape[ax], 2, device="cuda")
        e = self.cycle(r.index_select(ax, at), l + 1)
        full = torch.zeros_like(x).index_copy_(ax, at, e)
        full += lv["w1"] * _shift(full, ax, 1) + lv["w2"] * _shift(full, ax, -1)
        return self._smooth(lv, x + full, b, False, self.post, self.symmetric)


def _step(s, p_old):
    """One time step solved to round-off: Newton with GMRES on difference
    quotients, preconditioned by a V-cycle."""
    sat_old, _ = _closure(s, p_old)
    p = p_old.clone()
    f = _residual(s, p, p_old, sat_old)
    for _ in range(40):
        A = _jacobian(s, p, True)
        if s.overland:
            # the ponded cells' storage and outflow on the diagonal
            wet = p[-1].clamp(min=0.0)
            mag = torch.sqrt(s.slope_x ** 2 + s.slope_y ** 2).clamp(min=OV_EPS)
            slow = (s.slope_x.abs() + s.slope_y.abs()) / (torch.sqrt(mag) * MANN)
            A[0][-1] += torch.where(wet > 0, s.dx * s.dx + s.dt * s.dx * (5.0 / 3.0) * slow *
                                    wet ** (2.0 / 3.0), 0.0)
            A[1][-1].zero_()
            A[2][-1].zero_()
        M = Levels(s, A, 2, 2, 0)

        def product(v):
            size = 1e-7 * (1.0 + p.norm()) / v.norm()
            return (_residual(s, p + size * v, p_old, sat_old) - f) / size

        d = _gmres(product, M.cycle, -f, 1e-6, 30)
        norm, lam = f.norm(), 1.0
        while True:
            trial = p + lam * d
            ft = _residual(s, trial, p_old, sat_old)
            if ft.norm() < norm or lam < 1e-3:
                break
            lam *= 0.5
        if not ft.norm() < norm:
            break
        small = (lam * d).abs().max() < 1e-14 * (1.0 + p.abs().max())
        p, f = trial, ft
        if small:
            break
    return p


def _gmres(product, precondition, b, tol, most):
    beta = b.norm()
    if beta == 0:
        return torch.zeros_like(b)
    V, Z, H = [b / beta], [], torch.zeros((most + 1, most), dtype=torch.float64)
    for k in range(most):
        Z.append(precondition(V[k]))
        w = product(Z[k])
        for i in range(k + 1):
            H[i, k] = (w * V[i]).sum().item()
            w = w - H[i, k].item() * V[i]
        H[k + 1, k] = w.norm().item()
        e = torch.zeros((k + 2, 1), dtype=torch.float64)
        e[0] = beta.item()
        y = torch.linalg.lstsq(H[:k + 2, :k + 1], e).solution
        if (H[:k + 2, :k + 1] @ y - e).norm() <= tol * beta.item() or H[k + 1, k] == 0:
            break
        V.append(w / H[k + 1, k].item())
    return sum(z * y[i].item() for i, z in enumerate(Z))


def exact(case, seed):
    kind = case["kind"]
    if kind == "ensemble":
        return None            # a solve of its own for every member
    s = Site(case, seed)
    if kind == "advance":
        p = s.p0
        for _ in range(case["steps"]):
            p = _step(s, p)
        return s.vector(p), s.vector(_closure(s, p)[0])
    if kind == "residual":
        p = s.later()
        return s.vector(_residual(s, p, s.p0, _closure(s, s.p0)[0]))
    if kind == "jacobian":
        p, x = s.later(), _direction(s)
        if s.overland:
            return None        # the surface couplings are not restated here
        J = _jacobian(s, p, False)
        y = J[0] * x
        for q, (ax, by) in enumerate(((2, 1), (2, -1), (1, 1), (1, -1), (0, 1), (0, -1))):
            y = y + J[q + 1] * _shift(x, ax, by)
        return [s.vector(a) for a in J] + [s.vector(y)]
    if kind == "precond":
        A = _jacobian(s, s.later(), True)
        M = Levels(s, A, *_sweeps(case))
        return [s.vector(M.cycle(_direction(s))) for _ in range(RIGHT_HAND_SIDES)]
    if kind == "output":
        return _exact_output(s)
    return _exact_nvector(s)


def _exact_output(s):
    p, p_old = s.later(), s.p0
    sat, kr = _closure(s, p)
    vz, vy, vx = _velocities(s, p, kr)
    a, side, vol = s.dx * s.dx, s.dx * s.dz, s.dx * s.dx * s.dz
    vx, vy = F.pad(vx, (1, 1)), F.pad(vy, (0, 0, 1, 1))
    top = torch.full_like(p[-1], s.top)
    fluxes = [0.0, 0.0, 0.0, 0.0]
    if s.overland:
        qx, qy = _overland(s, p)
        top = top + _surface_inflow(s, p, p_old) / s.dt / a
        fluxes[1] = -s.dt * a * s.top * s.nx * s.ny
        fluxes[2] = s.dt * s.dx * float((qx[:, -1] - qx[:, 0]).sum() + (qy[-1] - qy[0]).sum())
    else:
        fluxes[0] = -s.dt * a * s.top * s.nx * s.ny
    bottom = _bottom_velocity(s, p, kr)
    fluxes[0] += s.dt * a * float(bottom.sum())
    vz = torch.cat([bottom[None], vz, top[None]])
    stored = s.poro * sat * vol + torch.where(p < 0, 0.0, p * sat * s.ss * vol)
    return {"saturation": s.vector(sat), "rel_perm": s.vector(kr), "velocity": [vx, vy, vz],
            "storage": [float(stored.sum()), float((p[-1] * a).clamp(min=0.0).sum())],
            "fluxes": fluxes}


def _exact_nvector(s):
    V = _basis(s)
    w, f = _direction(s), _direction(s)
    coefficients = []
    for v in V:
        coefficients.append(float((v * w).sum()))
        w = w - coefficients[-1] * v
    coefficients.append(float(w.norm()))
    w = w / coefficients[-1]
    step = w / (1.0 + s.p0.abs())
    return {"w": s.vector(w), "step": s.vector(step), "scaled": s.vector(f),
            "coefficients": coefficients,
            "norms": [float(step.abs().max()), float(f.abs().max()), float(f.norm())]}
