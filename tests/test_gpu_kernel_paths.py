"""GPU tests of single kernels and dispatch branches at the sizes where they
can go wrong: tile edges, remainders, the smallest grids.  Bars are the
rounding of the summed terms, as in the parity tests."""
import ctypes as C
import dataclasses

import numpy as np
import pytest

from oracle import oracle as O
import cases

pytestmark = pytest.mark.gpu


def _api():
    from parflow_amd import api
    return api


def _field(prob, rng, ghost=1e9):
    a = np.full(prob.shape, ghost)
    a[1:-1, 1:-1, 1:-1] = rng.normal(size=(prob.nz, prob.ny, prob.nx))
    return a


def _form(prob, form):
    """prob with independent kx, ky and kz ("aniso"), or with uniform van
    Genuchten parameters and kr from a table ("table")."""
    if form == "aniso":
        rng = np.random.default_rng(51)
        ky, kz = (np.exp(rng.normal(np.log(0.1), 1.0, (prob.nz, prob.ny, prob.nx)))
                  for _ in range(2))
        return dataclasses.replace(prob, ky=ky, kz=kz)
    if form == "table":
        return dataclasses.replace(prob, alpha=1.3, nvg=2.3, vg_table=(40, -6.0, "Spline"))
    return prob


@pytest.mark.parametrize("shape", [(1, 1, 2), (5, 3, 2), (65, 33, 40)])
def test_reduction_results_reach_the_host(gpu, shape):
    """Sums, maxima and mixed results of two problems in turn: each call
    returns its own values (fewer blocks than threads, and more rows than
    blocks)."""
    api = _api()
    probs = [cases.hetero(*shape, seed=1), cases.hetero(7, 4, 3, seed=2)]
    gps = [api.GPUProblem(p) for p in probs]
    rng = np.random.default_rng(7)
    r, a, b = C.c_double(), C.c_double(), C.c_double()
    lib = api.lib()
    for rep in range(3):
        for prob, gp in zip(probs, gps):
            x, y = _field(prob, rng), _field(prob, rng)
            X, Y = prob.interior(x), prob.interior(y)
            dx, dy = gp.vec(x), gp.vec(y)
            api.check(lib.pfhip_vec_dot(gp.h, dx.ptr, dy.ptr, C.byref(r), None), "dot")
            assert abs(r.value - np.sum(X * Y)) <= 1e-13 * np.sum(np.abs(X * Y))
            api.check(lib.pfhip_vec_max_norm(gp.h, dx.ptr, C.byref(r), None), "max")
            assert r.value == np.max(np.abs(X))
            api.check(lib.pfhip_vec_min(gp.h, dy.ptr, C.byref(r), None), "min")
            assert r.value == np.min(Y)
            lib.pfhip_vec_dot_scsteplength.argtypes = [C.c_void_p] * 6
            api.check(lib.pfhip_vec_dot_scsteplength(gp.h, dx.ptr, dy.ptr, C.byref(a),
                                                     C.byref(b), None), "dot_scsteplength")
            assert abs(a.value - np.sum(Y * Y)) <= 1e-13 * np.sum(Y * Y)
            assert abs(b.value - np.max(np.abs(Y) / (1 + np.abs(X)))) <= 1e-15 * b.value


def test_shared_pinned_memory_is_coherent(gpu):
    """The ensemble's result slots and staging ring, which kernels and the host
    use without a copy or a synchronisation between them, are allocated
    coherent, whatever the runtime's default is."""
    class Results(C.Structure):
        _fields_ = [("host", C.c_void_p), ("flag", C.c_void_p), ("seq", C.c_ulonglong),
                    ("ticket", C.c_void_p)]

    class Stage(C.Structure):
        _fields_ = [("host", C.c_void_p), ("dev", C.c_void_p), ("off", C.c_long),
                    ("cap", C.c_long)]
    api = _api()
    lib = api.lib()                    # and the HIP runtime it is linked to
    r, st, flags = Results(), Stage(), C.c_uint()
    api.check(lib.pfhip_ens_results_create(C.byref(r), C.c_long(64)), "results")
    api.check(lib.pfhip_ens_stage_create(C.byref(st), C.c_long(1 << 16)), "stage")
    for p in (r.host, st.host):
        assert lib.hipHostGetFlags(C.byref(flags), C.c_void_p(p)) == 0
        assert flags.value & 0x40000000          # hipHostMallocCoherent
    lib.pfhip_ens_results_destroy(C.byref(r))
    lib.pfhip_ens_stage_destroy(C.byref(st))


@pytest.mark.parametrize("shape", [(1, 1, 1), (64, 8, 16), (65, 9, 17), (130, 3, 33)])
@pytest.mark.parametrize("overland,dirs", [(False, True), (True, False)])
@pytest.mark.parametrize("form", ["iso", "aniso", "table"])
def test_face_velocity_tiles(gpu, shape, overland, dirs, form):
    """Face velocities over grids that fill, exceed and fall short of the
    kernel's 64 x 8 x 16 tiles, with one permeability, three, and kr from a
    lookup table, against the oracle."""
    api = _api()
    prob = _form(cases.hetero(*shape, seed=4, overland=overland, dir_sides=dirs), form)
    gp, op = api.GPUProblem(prob), O.OracleProblem(prob)
    p, p_old = cases.random_pressure(prob, seed=5), cases.random_pressure(prob, seed=6)
    t = 0.1
    got = gp.face_velocity(p, p_old, 0.1, t)
    want = O.face_velocity(op, p, p_old, 0.1, t)
    scale = max(np.max(np.abs(b)) for b in want)
    for a, b in zip(got, want):
        assert np.max(np.abs(a - b)) <= 1e-12 * scale


@pytest.mark.parametrize("iso", [True, False])
def test_face_velocity_infinities_and_zeros(gpu, iso):
    """Interior face velocities of saturated cells (kr = 1) with infinite and
    overflowing pressures, differences and permeabilities and with zero ones:
    NaN, the infinities and the sign of a zero as the oracle's divisions leave
    them, finite values to the rounding of their dozen operations (z faces:
    of the two heads they subtract)."""
    api = _api()
    prob = cases.hetero(70, 17, 20, seed=41)
    rng = np.random.default_rng(42)
    K = []
    for q in range(1 if iso else 3):
        k = np.exp(rng.normal(np.log(0.1), 1.0, (prob.nz, prob.ny, prob.nx)))
        k.ravel()[rng.choice(k.size, 900, replace=False)] = np.resize(
            [0.0, 1e200, 1.7e308, np.inf, 1e-200], 900)
        K.append(k)
    prob = dataclasses.replace(prob, kx=K[0], ky=K[-1] if iso else K[1], kz=K[-1])
    p = prob.zeros()
    inner = rng.uniform(0.0, 50.0, (prob.nz, prob.ny, prob.nx))
    inner.ravel()[rng.choice(inner.size, 1500, replace=False)] = np.resize(
        [np.inf, 1.7e308, 0.0, -0.0, 1e-310, 1e160], 1500)
    p[1:-1, 1:-1, 1:-1] = inner
    got = api.GPUProblem(prob).face_velocity(p, p, 0.1, 0.1)
    want = O.face_velocity(O.OracleProblem(prob), p, p, 0.1, 0.1)
    seen = np.zeros(3, dtype=int)
    for ax, (a, b) in enumerate(zip(got, want)):
        face = [slice(None)] * 3
        face[2 - ax] = slice(1, -1)
        a, b = a[tuple(face)], b[tuple(face)]
        assert np.array_equal(np.isnan(a), np.isnan(b))
        assert np.array_equal(np.isinf(a), np.isinf(b))
        signed = np.isinf(b) | (b == 0)
        assert np.array_equal(np.signbit(a[signed]), np.signbit(b[signed]))
        assert np.all(a[b == 0] == 0)
        fin = np.isfinite(b) & (b != 0)
        with np.errstate(all="ignore"):
            if ax < 2:
                bar = 4e-15 * np.abs(b)
            else:
                k = K[-1]
                h = 2 * k[:-1] * k[1:] / (k[:-1] + k[1:])
                bar = 4e-15 * h * (inner[:-1] / prob.dz + inner[1:] / prob.dz + 1)
            assert np.all(np.abs(a - b)[fin] <= np.maximum(bar, 1e-300)[fin])
        seen += [np.sum(np.isnan(b)), np.sum(np.isinf(b)), np.sum((b == 0) & np.signbit(b))]
    assert np.all(seen > 0)


@pytest.mark.parametrize("shape", [(1, 1, 1), (2, 2, 2), (70, 9, 5)])
@pytest.mark.parametrize("with_src", [False, True])
def test_water_balance_fluxes_shell(gpu, shape, with_src):
    """The step's volumes from the shell cells alone (and all cells of a
    source field), against the face velocities summed over the domain."""
    api = _api()
    prob = cases.hetero(*shape, seed=8, dir_sides=True)
    src = cases.hetero_src(prob, 9) if with_src else None
    gp = api.GPUProblem(prob, src=src)
    p = cases.random_pressure(prob, seed=10)
    dt, t = 0.1, 0.1
    f = gp.water_balance_fluxes(p, p, dt, t)
    vx, vy, vz = O.face_velocity(O.OracleProblem(prob), p, p, dt, t)
    ax, ay, az = prob.dy * prob.dz, prob.dx * prob.dz, prob.dx * prob.dy
    terms = [ax * vx[:, :, 0], -ax * vx[:, :, -1], ay * vy[:, 0], -ay * vy[:, -1],
             az * vz[0], -az * vz[-1]]
    want = dt * sum(float(np.sum(a)) for a in terms)
    scale = dt * sum(float(np.sum(np.abs(a))) for a in terms)
    assert abs(f[0] - want) <= 1e-12 * scale
    vol = prob.dx * prob.dy * prob.dz * dt
    if with_src:
        want = vol * float(np.sum(prob.interior(src)))
        assert abs(f[3] - want) <= 1e-12 * vol * float(np.sum(np.abs(src)))
    else:
        assert f[3] == 0.0


@pytest.mark.parametrize("shape,form", [
    ((1, 1, 1), "iso"), ((64, 8, 2), "iso"), ((65, 9, 3), "iso"), ((200, 130, 9), "iso"),
    ((513, 130, 13), "iso"), ((513, 130, 35), "iso"), ((513, 262, 18), "iso"),
    ((65, 9, 3), "aniso"), ((130, 20, 37), "aniso"), ((513, 130, 13), "aniso"),
    ((65, 9, 5), "table")])
def test_residual_and_jacobian_plane_chunks(gpu, shape, form):
    """F and both Jacobians where the tiles march 2 planes (grids below 513 x
    130), 4, 8 and 16 (513 x 130 x 13 and 35, 513 x 262 x 18) and the last
    chunk is cut short, against the oracle."""
    api = _api()
    prob = _form(cases.hetero(*shape, seed=11, dir_sides=True), form)
    gp, op = api.GPUProblem(prob), O.OracleProblem(prob)
    p, p_old = cases.random_pressure(prob, seed=12), cases.random_pressure(prob, seed=13)
    s_old = O.saturation(op, p_old, 0)
    I = prob.interior
    a = I(gp.nl_function_eval(p, p_old, s_old, 0.1, 0.1))
    b = I(O.nl_function_eval(op, p, p_old, s_old, 0.1, 0.1))
    assert np.max(np.abs(a - b)) <= 1e-12 * np.max(np.abs(b))
    for symm in (0, 1):
        A = gp.richards_jacobian_eval(p, 0.1, 0.1, symm)
        B = O.jacobian_eval(op, p, 0.1, 0.1, symm)
        scale = np.max(np.abs(I(B[0])))
        for q in ((0, 2, 4, 6) if symm else range(7)):
            assert np.max(np.abs(I(A[q]) - I(B[q]))) <= 1e-11 * scale, (symm, q)


@pytest.mark.parametrize("shape", [(2, 1, 1), (1, 1, 9), (3, 5, 7), (16, 9, 14), (1, 64, 64), (33, 8, 8)])
@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("sweeps", [(1, 1, 1), (1, 1, 0), (2, 2, 0), (0, 1, 0), (2, 0, 1)])
def test_multigrid_bottom_levels(gpu, shape, precision, sweeps):
    """V-cycles whose levels all run in the one-workgroup bottom but the
    first: single points, odd extents, one point per row (more pairs than
    threads keep a level on the grid), against the oracle."""
    api = _api()
    pre, post, sym = sweeps
    prob = cases.hetero(*shape, seed=21)
    gp = api.GPUProblem(prob)
    A = cases.full_operator(prob, 22, symmetric=True)
    b = np.zeros(prob.shape)
    prob.interior(b)[...] = np.random.default_rng(23).normal(size=prob.interior(b).shape)
    mg = api.GPUMultigrid(gp, pre, post, sym, precision=precision)
    mg.setup(A)
    got = prob.interior(mg.apply(b))
    om = O.MG(prob, pre, post, sym)
    om.setup(A)
    want = prob.interior(om.apply(b))
    tol = 1e-11 if precision == 64 else 2e-5
    assert np.max(np.abs(got - want)) <= tol * np.max(np.abs(want))


@pytest.mark.parametrize("shape", [(32, 32, 32), (45, 33, 20), (7, 5, 60), (96, 80, 6), (130, 3, 40)])
@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("sweeps", [(1, 1, 0), (2, 2, 0), (1, 1, 1), (1, 2, 0)])
def test_multigrid_block_launches_bitwise(gpu, shape, precision, sweeps, monkeypatch):
    """Levels visited by one block launch each against the separate launches:
    the same bits, in the V-cycles that launch directly and that replay a
    graph; odd extents, single-column tiles and blocks cut by the boundary.
    The separate side restricts along z point by point: the marching form of
    that kernel rounds one product together with the sum it enters."""
    api = _api()
    monkeypatch.setenv("PFHIP_MG_RRZ", "0")
    prob = cases.hetero(*shape, seed=31)
    gp = api.GPUProblem(prob)
    A = cases.full_operator(prob, 32, symmetric=True)
    bs = []
    for q in range(3):
        b = np.zeros(prob.shape)
        prob.interior(b)[...] = np.random.default_rng(33 + q).normal(size=prob.interior(b).shape)
        bs.append(b)
    out = {}
    for blocks in ("0", "300000"):
        monkeypatch.setenv("PFHIP_MG_BLOCK", blocks)
        mg = api.GPUMultigrid(gp, *sweeps, precision=precision)
        mg.setup(A)
        out[blocks] = [mg.apply(b) for b in bs]
    for a, b in zip(out["0"], out["300000"]):
        assert np.array_equal(prob.interior(a), prob.interior(b))


def test_ensemble_vector_blocks(gpu):
    """Members whose cells a block of the ensemble's vector kernel steps
    through differently (rows longer than a block, single rows, a remainder of
    one cell, several blocks) against the same members advanced alone, at the
    tolerances and the bar of the 512-member comparison."""
    from parflow_amd.decks import c4_member
    api = _api()
    members = []
    for m, (nx, ny, nz) in enumerate([(300, 3, 20), (5, 41, 5), (3, 1, 24), (37, 28, 25)]):
        prob, opts, _, dt = c4_member(m)
        prob = dataclasses.replace(prob, nx=nx, ny=ny, nz=nz)
        opts = dataclasses.replace(opts, residual_tol=1e-12, step_tol=1e-30)
        p0 = prob.zeros()
        z = prob.z0 + (np.arange(nz) + 0.5) * prob.dz
        p0[1:-1, 1:-1, 1:-1] = (0.5 * nz * prob.dz - z)[:, None, None]
        members.append((prob, opts, p0, dt))
    ens = api.GPUEnsemble([(p, o) for p, o, _, _ in members])
    dps = [ens.problems[i].vec(m[2]) for i, m in enumerate(members)]
    dss = [ens.problems[i].vec() for i in range(len(members))]
    lg = ens.advance_device(dps, dss, 0.0, [m[3] for m in members], 2)
    assert np.all(lg["steps"] == 2)
    for i, (prob, _, p0, dt) in enumerate(members):
        pg, sg, l1 = ens.solvers[i].advance(p0, 0.0, dt, 2, history=False)
        got, want = prob.interior(ens.problems[i].get(dps[i])), prob.interior(pg)
        e = np.max(np.abs(got - want) / np.maximum(np.abs(want), 1e-3))
        assert e < 1e-10, (i, e)
        assert np.all(np.abs(lg["newton"][i] - l1["newton"]) <= 1), i


@pytest.mark.parametrize("sweeps", [(1, 1), (2, 1), (0, 1), (1, 0)])
def test_ensemble_phase_conversions(gpu, sweeps, monkeypatch):
    """The ensemble's phase launches with the FP64 vectors converted by level
    0's first and last half-sweep, or by passes of their own where there is no
    such half-sweep, against every level inside one workgroup: the same bits.
    Odd extents, so the last pair of a row has one point."""
    from parflow_amd.decks import c4_member
    api = _api()
    members = []
    for m, (nx, ny, nz) in enumerate([(33, 20, 25), (45, 31, 30), (8, 9, 24)]):
        prob, opts, _, dt = c4_member(m)
        prob = dataclasses.replace(prob, nx=nx, ny=ny, nz=nz)
        opts = dataclasses.replace(opts, num_pre_relax=sweeps[0], num_post_relax=sweeps[1])
        p0 = prob.zeros()
        z = prob.z0 + (np.arange(nz) + 0.5) * prob.dz
        p0[1:-1, 1:-1, 1:-1] = (0.5 * nz * prob.dz - z)[:, None, None]
        members.append((prob, opts, p0, dt))
    out = []
    for small in (None, "100000000"):
        if small:
            monkeypatch.setenv("PFHIP_ENS_MG_SMALL", small)
        ens = api.GPUEnsemble([(p, o) for p, o, _, _ in members])
        dps = [ens.problems[i].vec(m[2]) for i, m in enumerate(members)]
        dss = [ens.problems[i].vec() for i in range(len(members))]
        lg = ens.advance_device(dps, dss, 0.0, [m[3] for m in members], 1)
        assert np.all(lg["steps"] == 1)
        out.append(([ens.problems[i].get(d) for i, d in enumerate(dps)], lg))
    for a, b in zip(out[0][0], out[1][0]):
        assert np.array_equal(a, b)
    assert np.array_equal(out[0][1]["gmres"], out[1][1]["gmres"])


@pytest.mark.parametrize("precision", [32, 64])
def test_ensemble_bottoms_that_do_not_fit_lds(gpu, precision, monkeypatch):
    """Members whose hierarchies are cut off at a level that the LDS bottom
    cannot take (1500 pairs of points; 12,000 points) beside one that it
    takes: the same bits as with every level in one workgroup in global
    memory, and the members' own solutions (at the deck's tolerances the two
    paths differ by up to 5e-8)."""
    from parflow_amd.decks import c4_member
    api = _api()
    members = []
    for m, (nx, ny, nz, levels) in enumerate([(12, 10, 20, 100), (30, 20, 20, 3), (40, 30, 20, 2),
                                              (9, 30, 21, 100)]):
        prob, opts, _, dt = c4_member(m)
        prob = dataclasses.replace(prob, nx=nx, ny=ny, nz=nz)
        opts = dataclasses.replace(opts, max_levels=levels)
        p0 = prob.zeros()
        z = prob.z0 + (np.arange(nz) + 0.5) * prob.dz
        p0[1:-1, 1:-1, 1:-1] = (0.5 * nz * prob.dz - z)[:, None, None]
        members.append((prob, opts, p0, dt))
    out = []
    for small in (None, "100000000"):
        if small:
            monkeypatch.setenv("PFHIP_ENS_MG_SMALL", small)
        ens = api.GPUEnsemble([(p, o) for p, o, _, _ in members], precision=precision)
        dps = [ens.problems[i].vec(m[2]) for i, m in enumerate(members)]
        dss = [ens.problems[i].vec() for i in range(len(members))]
        lg = ens.advance_device(dps, dss, 0.0, [m[3] for m in members], 2)
        assert np.all(lg["steps"] == 2)
        out.append(([ens.problems[i].get(d) for i, d in enumerate(dps)], lg))
    for a, b in zip(out[0][0], out[1][0]):
        assert np.array_equal(a, b)
    assert np.array_equal(out[0][1]["gmres"], out[1][1]["gmres"])
    for i, (prob, _, p0, dt) in enumerate(members):
        pg, _, l1 = ens.solvers[i].advance(p0, 0.0, dt, 2, history=False)
        got, want = prob.interior(out[0][0][i]), prob.interior(pg)
        assert np.max(np.abs(got - want) / np.maximum(np.abs(want), 1e-3)) < 1e-6, i
        assert np.all(np.abs(out[0][1]["newton"][i] - l1["newton"]) <= 1), i
