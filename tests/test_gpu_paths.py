"""Kernels that are chosen by a rule on the mesh, each at the sizes where its
split can go wrong: tiles and blocks with a remainder, tables that overflow,
both sides of a rule's line.  Against the oracle at the parity bars
(reconstruction 1e-12, residual 1e-11, relative L2 per variable), or against
the kernels that the rule leaves (another order of FP64 sums: a few hundred
roundings of 1.1e-16, held to 1e-12 of the largest value; cotangents behind a
march to 1e-10)."""
import ctypes
import dataclasses

import numpy as np
import pytest

from oracle.oracle import Oracle
from shuffle import shuffled_structs
from ucns3d_amd.case import HEX, HYBRID, PRISM, TET, Case, CaseSpec, reduced
from ucns3d_amd.native import UCNS_FP64, UCNS_KERNELS_REGISTER, UCNS_MIXED
from ucns3d_amd.solver import Solver, UcnsError

pytestmark = pytest.mark.gpu


def close(a, b, tol):
    a, b = np.asarray(a), np.asarray(b)
    assert np.isfinite(a).all()
    d = np.abs(a - b).max()
    assert d <= tol * np.abs(b).max(), (d, np.abs(b).max())


def rel_l2(a, b):
    """relative L2 per variable, the momenta against the whole momentum"""
    a, b = a.reshape(-1, 5), b.reshape(-1, 5)
    num, den = np.sqrt(((a - b) ** 2).sum(0)), np.sqrt((b ** 2).sum(0))
    den[1:4] = np.sqrt((den[1:4] ** 2).sum())
    return num / den


# cell counts that are no multiple of a tile (8 cells) or of a block (32)
REMAINDERS = {
    "hex-muscl-125": CaseSpec("r-muscl", HEX, 5, "muscl", jitter=0.1, seed=3),
    "hex-weno4-729": CaseSpec("r-hex4", HEX, 9, "weno4", jitter=0.1, seed=3),
    "hex-weno4-char-729": CaseSpec("r-hex4c", HEX, 9, "weno4", jitter=0.1, seed=3, wenwrt=2),
    "tet-weno4-char-750": CaseSpec("r-tet4c", TET, 5, "weno4", jitter=0.1, seed=3, wenwrt=2),
    "prism-weno3-686": CaseSpec("r-prism3", PRISM, 7, "weno3", jitter=0.1, seed=3),
    "tet-cweno5-2058": CaseSpec("r-tet5", TET, 7, "weno5", jitter=0.1, seed=3, ees=5),
}


@pytest.mark.parametrize("name", list(REMAINDERS))
def test_remainders_against_the_oracle(name):
    case = Case(REMAINDERS[name])
    assert case.ncell == int(name.split("-")[-1]) and case.ncell % 8 and case.ncell % 32
    u = case.init_state()
    orc = Oracle(case)
    r_ref, cnt = orc.residual(u)
    print(f"[remainder] {name}", flush=True)
    s = Solver(case, UCNS_FP64)
    s.set_state(u)
    err = rel_l2(s.residual(), r_ref)
    st = s.stats()
    s.close()
    print("  residual", err)
    assert (st["n_reduced_last"], st["n_firstorder_last"]) == (cnt[0], cnt[1])
    assert np.all(err <= 1e-11), err


# tiles whose distinct members exceed the table in LDS (512 rows; 768 with 7
# stencils of 39 members): 8 cells far apart, in the caller's order
OVERFLOW = {
    "hex-weno4": CaseSpec("o-hex4", HEX, 11, "weno4", jitter=0.1, seed=5),
    "tet-weno4-char": CaseSpec("o-tet4c", TET, 7, "weno4", jitter=0.1, seed=5, wenwrt=2),
    "prism-weno3": CaseSpec("o-prism3", PRISM, 9, "weno3", jitter=0.1, seed=5),
}


@pytest.mark.parametrize("name", list(OVERFLOW))
def test_tiles_past_the_member_table(name):
    case = Case(OVERFLOW[name])
    u = case.init_state() * (1 + 1e-3 * np.random.default_rng(2).uniform(-1, 1, (case.ncell, 5)))
    sh = np.random.default_rng(4).permutation(case.ncell).astype(np.int64)
    keep, st = shuffled_structs(case, sh)
    w = np.random.default_rng(6).standard_normal(u.shape)
    print(f"[member table] {name} ncell={case.ncell}", flush=True)
    a = Solver(case, UCNS_FP64)
    b = Solver(case, UCNS_FP64, structs=st)
    a.set_state(u)
    b.set_state(u[sh])
    close(b.reconstruct(), a.reconstruct()[sh], 1e-12)
    if case.spec.wenwrt == 1:  # the products do not cover characteristic variables
        close(b.residual_vjp(w[sh])[0], a.residual_vjp(w)[0][sh], 1e-10)
    a.close()
    b.close()


# marches on one-point faces: fluxes and update in one kernel up to 32,768
# cells; a timed context keeps the two kernels
@pytest.mark.parametrize("n", [3, 5, 31, 33])
def test_march_on_one_point_faces(n):
    case = Case(CaseSpec("f-muscl", HEX, n, "muscl", jitter=0.1, seed=3))
    u = case.init_state()
    out = []
    for timed in (False, True):
        print(f"[one-point march] ncell={case.ncell} timed={timed}", flush=True)
        s = Solver(case, UCNS_FP64)
        if timed:
            s.reset_stats()
        s.set_state(u)
        t = s.rk3_steps(3, cfl=0.5)
        out.append((s.get_state(), t))
        s.close()
    (a, ta), (b, tb) = out
    close(a, b, 1e-12)
    assert abs(ta - tb) <= 1e-12 * tb


# the last value of a state, with one block per 1,024 values and with more
# values than the 256 blocks take in one trip
@pytest.mark.parametrize("n", [3, 38])
def test_non_finite_last_value(n):
    case = Case(CaseSpec("nf-muscl", HEX, n, "muscl", seed=3))
    u = case.init_state()
    print(f"[non-finite last value] ncell={case.ncell}", flush=True)
    s = Solver(case, UCNS_FP64)
    s.set_state(u)
    s.rk3_steps(0, dt_fixed=1e-3)
    u[-1, 4] = np.inf
    s.set_state(u)
    with pytest.raises(UcnsError, match="non-finite"):
        s.rk3_steps(0, dt_fixed=1e-3)
    s.close()


@pytest.mark.parametrize("spec", [CaseSpec("geo-prism", PRISM, 3, "weno3", jitter=0.1, seed=13), reduced("c4", 3)],
                         ids=["prisms", "channel"])
def test_geometry_product_on_the_row_stream_of_6_stencils(spec):
    case = Case(spec)
    w = np.random.default_rng(3).standard_normal((case.ncell, 5))
    out = []
    for kw in ({}, {"kernels": UCNS_KERNELS_REGISTER}):
        s = Solver(case, UCNS_FP64, **kw)
        if spec.mach > 0:
            fs = spec.freestream()
            s.set_boundary(1, fs, fs)
        s.set_state(case.init_state())
        print(f"[geometry product] {spec.name} ncell={case.ncell} {kw}", flush=True)
        a, bc, g, _ = s.rk3_adjoint_geometry(2, w, 1e-3)
        out.append((a, bc, g))
        s.close()
    (a0, b0, g0), (a1, b1, g1) = out
    close(a0, a1, 1e-10)
    for k in g1:
        close(g0[k], g1[k], 1e-10)


# states without a sound speed: the components of the fluxes that are NaN in
# the reference's HLLC (its side that sign(S_M) does not pick enters with a
# factor 0) are NaN here, and a march from them is reported.  Only states whose
# pressure is exact: on tetrahedra a flow without pressure holds roundings of
# either sign in its place
NO_SOUND = {
    "at-rest-tet-weno4": CaseSpec("np-tet4", TET, 4, "weno4", jitter=0.1, seed=5),
    "at-rest-hex-weno4": CaseSpec("np-hex4", HEX, 9, "weno4", seed=5),
    "at-rest-hex-muscl": CaseSpec("np-muscl", HEX, 5, "muscl", jitter=0.1, seed=5),
    "moving-hex-weno4": CaseSpec("np-hex4", HEX, 9, "weno4", seed=5),
    "moving-hex-muscl": CaseSpec("np-muscl", HEX, 5, "muscl", jitter=0.1, seed=5),
}


@pytest.mark.parametrize("name", list(NO_SOUND))
def test_states_without_a_sound_speed(name):
    case = Case(NO_SOUND[name])
    u = np.zeros((case.ncell, 5))
    u[:, 0] = 1.0
    if name.startswith("moving"):  # no pressure anywhere
        u[:, 1], u[:, 4] = 1.0, 0.5
    else:  # one cell of negative pressure
        u[:, 4] = 2.5
        u[case.ncell // 2, 4] = -1.0
    r_ref, _ = Oracle(case).residual(u)
    assert not np.isfinite(r_ref).all()
    print(f"[no sound speed] {name} ncell={case.ncell}", flush=True)
    s = Solver(case, UCNS_FP64)
    s.set_state(u)
    r = s.residual()
    assert np.array_equal(np.isfinite(r), np.isfinite(r_ref))
    with pytest.raises(UcnsError, match="non-finite"):
        s.rk3_steps(1, dt_fixed=1e-3)
    s.close()


# triangles of a mesh with quadrilaterals leave slots of the face-point array
# without a point; nothing may depend on what the caller left there
UNUSED = {
    "channel-weno3": reduced("c4", 3),
    "channel-weno3-char": dataclasses.replace(reduced("c4", 3), wenwrt=2),
    "hybrid-weno3": CaseSpec("u-hybrid", HYBRID, 6, "weno3", jitter=0.1, seed=3),
    "blast-cweno5": reduced("c5", 10),
}


@pytest.mark.parametrize("precision", [UCNS_FP64, UCNS_MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("name", list(UNUSED))
def test_slots_without_a_face_point(name, precision):
    spec = UNUSED[name]
    case = Case(spec)
    u = case.init_state()
    w = np.random.default_rng(3).standard_normal(u.shape)
    q = case.array("qpoints").reshape(case.ncell, case.nface_max, -1, 3)
    nv = (case.array("face_nodes").reshape(case.ncell, -1, 4) >= 0).sum(2)
    nq = np.where(nv == 4, case.qp_quad, np.where(nv == 3, case.qp_tri, 0))
    unused = np.arange(q.shape[2]) >= nq[:, :, None]
    assert (unused & (nq > 0)[:, :, None]).any()
    out = []
    for fill in (0.0, np.nan):
        q[unused] = fill
        print(f"[unused slots] {name} ncell={case.ncell} precision={precision} fill={fill}", flush=True)
        s = Solver(case, precision)
        fs = spec.freestream() if spec.mach > 0 else np.array([1.0, 0.0, 0.0, 0.0, 2.5])
        s.set_boundary(1 if spec.mach > 0 else 0, fs, fs)
        s.set_state(u)
        r = s.residual()
        out.append((r, None if spec.wenwrt == 2 or spec.ees == 5 else s.residual_vjp(w)[0]))
        s.close()
    assert np.isfinite(out[0][0]).all() and np.array_equal(out[0][0], out[1][0])
    if out[0][1] is not None:  # sums of atomics: another order on every run
        close(out[1][1], out[0][1], 1e-12)


# iweno 1 with the linear polynomial of the central stencil: one stencil, so a
# weight of 1 whatever the indicator, and the limiter only where CHECKSOL asks
@pytest.mark.parametrize("precision,tol", [(UCNS_FP64, 1e-11), (UCNS_MIXED, 1e-5)], ids=["fp64", "mixed"])
def test_linear_weno(precision, tol):
    case = Case(CaseSpec("l-weno", HEX, 5, "muscl", jitter=0.1, seed=3))
    mesh, scheme, pre = structs = case.structs(precision)
    scheme.iweno = 1
    ind = np.tile(np.eye(3), (case.ncell, 1, 1))
    full = (np.arange(case.ncell) % 3 > 0).astype(np.int32)
    pre.indicator = ind.ctypes.data_as(ctypes.POINTER(ctypes.c_double))
    pre.full = full.ctypes.data_as(ctypes.POINTER(ctypes.c_int32))
    u = case.init_state()
    orc = Oracle(case)
    orc.m, orc.s, orc.p = structs
    r_ref, cnt = orc.residual(u)
    print(f"[linear WENO] ncell={case.ncell} precision={precision}", flush=True)
    s = Solver(case, precision, structs=structs)
    s.set_state(u)
    err = rel_l2(s.residual(), r_ref)
    st = s.stats()
    s.close()
    print("  residual", err, "MUSCL cells", cnt[0])
    assert 0 < cnt[0] < case.ncell
    assert (st["n_reduced_last"], st["n_firstorder_last"]) == (cnt[0], cnt[1])
    assert np.all(err <= tol), err


# The geometry product forms the stencil coefficients again: it neither stores
# nor keeps the row stream's, so a march keeps as many stages as on the register
# kernels, and holds no more device memory
def test_geometry_product_keeps_no_coefficients():
    import torch
    spec = reduced("c4", 9)
    case = Case(spec)
    steps, fs = 3, spec.freestream()
    nv = (case.array("face_nodes").reshape(case.ncell, -1, 4) >= 0).sum(2)
    face_values = case.ncell * int((nv > 0).sum(1).max()) * max(case.qp_quad, case.qp_tri) * 5 * 8
    gib = 1.01 * 3 * steps * face_values / 2.0 ** 30  # every stage's, and nothing beside them
    w = np.random.default_rng(3).standard_normal((case.ncell, 5))
    u = case.init_state()

    def context(**kw):
        s = Solver(case, UCNS_FP64, adj_keep_gib=gib, **kw)
        s.set_boundary(1, fs, fs)
        s.set_state(u)
        s.reset_stats()
        return s

    out = []
    for kw in ({"kernels": UCNS_KERNELS_REGISTER}, {}):
        print(f"[geometry product, kept stages] ncell={case.ncell} {kw}", flush=True)
        s = context(**kw)
        free = torch.cuda.mem_get_info()[0]
        g = s.rk3_adjoint_geometry(steps, w, 1e-3)[0]
        out.append((g, s.stats()["n_recon_adj"], free - torch.cuda.mem_get_info()[0]))
        s.close()
    (g_reg, again_reg, mem_reg), (g_row, again_row, mem_row) = out
    print("  stages reconstructed again", again_reg, again_row, "bytes held", mem_reg, mem_row)
    assert again_reg == 0 and again_row == 0
    assert mem_row <= mem_reg + (8 << 20)  # allocations come in 2 MiB pieces
    close(g_row, g_reg, 1e-10)


# products that store and geometry products in turn, in one context whose budget
# holds only some stages of the first kind
def test_geometry_and_ordinary_adjoints_in_turn():
    spec = reduced("c4", 6)
    case = Case(spec)
    fs = spec.freestream()
    w = np.random.default_rng(3).standard_normal((case.ncell, 5))
    u = case.init_state()

    def call(s, kind):
        s.set_state(u)
        return (s.rk3_adjoint_geometry(2, w, 1e-3) if kind == "geometry" else s.rk3_adjoint(2, w, dt_fixed=1e-3))[0]

    def context(gib):
        s = Solver(case, UCNS_FP64, adj_keep_gib=gib)
        s.set_boundary(1, fs, fs)
        return s

    ref = {}
    for kind in ("geometry", "ordinary"):
        s = context(0.0)
        ref[kind] = call(s, kind)
        s.close()
    for order in (("ordinary", "geometry", "ordinary"), ("geometry", "ordinary", "geometry", "geometry")):
        for gib in (0.02, 0.05, 1.0):
            print(f"[adjoints in turn] ncell={case.ncell} {order} {gib} GiB", flush=True)
            s = context(gib)
            for kind in order:
                close(call(s, kind), ref[kind], 1e-10)
            s.close()


# The rule for the block kernels in conserved variables: at most 512 tiles (768 in
# mixed precision), and no tile past the member table.  A context on them builds
# the member tables (three allocations) at its upload, one on the row stream with
# its first adjoint
@pytest.mark.parametrize("precision,n,shuffled,block", [
    (UCNS_FP64, 15, False, True), (UCNS_FP64, 15, True, False), (UCNS_FP64, 16, False, True),
    (UCNS_FP64, 17, False, False), (UCNS_MIXED, 17, False, True), (UCNS_MIXED, 17, True, False),
    (UCNS_MIXED, 19, False, False)])
def test_rule_of_the_block_kernels(precision, n, shuffled, block):
    case = Case(CaseSpec("b-hex4", HEX, n, "weno4", jitter=0.1, seed=5))
    u = case.init_state()
    w = np.random.default_rng(6).standard_normal(u.shape)
    sh = np.random.default_rng(4).permutation(case.ncell) if shuffled else np.arange(case.ncell)
    keep, st = shuffled_structs(case, sh.astype(np.int64), precision)
    print(f"[block rule] ncell={case.ncell} precision={precision} shuffled={shuffled}", flush=True)
    s = Solver(case, precision, structs=st)
    s.set_state(u[sh])
    made = 0
    while True:  # one allocation more on every try, until the set-up succeeds
        s.debug_fail_alloc(made + 1)
        try:
            s.residual_vjp(w[sh])
            break
        except UcnsError as e:
            assert "injected" in str(e)
            made += 1
    s.close()
    # 7 work arrays, the 3 of the stored forward, 5 of the tables' index by cell
    assert made == (15 if block else 18), made


# MUSCL in mixed precision: a step against the FP64 oracle (1e-5), on one-point
# faces with fluxes and update in one kernel (32,768 cells are the most it takes)
# and on meshes it does not take
@pytest.mark.parametrize("spec", [CaseSpec("mm-125", HEX, 5, "muscl", jitter=0.1, seed=3),
                                  CaseSpec("mm-32768", HEX, 32, "muscl", jitter=0.1, seed=3),
                                  CaseSpec("mm-35937", HEX, 33, "muscl", jitter=0.1, seed=3),
                                  CaseSpec("mm-prism", PRISM, 7, "muscl", jitter=0.1, seed=3)], ids=lambda s: s.name)
def test_muscl_in_mixed_precision(spec):
    case = Case(spec)
    u = case.init_state()
    print(f"[mixed MUSCL] {spec.name} ncell={case.ncell}", flush=True)
    s = Solver(case, UCNS_MIXED)
    s.set_state(u)
    s.rk3_steps(1, cfl=0.5)
    err = rel_l2(s.get_state(), Oracle(case).rk3(u, 1, cfl=0.5)[0])
    s.close()
    print("  rel L2", err)
    assert np.all(err <= 1e-5), err


# The one-kernel march forms a face's flux in both of its cells: the two must hold
# the same bits, so a periodic march conserves to the rounding of its updates (of
# the order 1e-16 a cell and stage; FP32 fluxes that differed would leave 1e-9)
@pytest.mark.parametrize("precision", [UCNS_FP64, UCNS_MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("n", [5, 32])
def test_one_point_march_conserves(n, precision):
    case = Case(CaseSpec("cons-muscl", HEX, n, "muscl", jitter=0.1, seed=3))
    u = case.init_state()
    vol = np.ctypeslib.as_array(case.structs()[0].totvolume, shape=(case.ncell,))[:, None]
    print(f"[conservation] ncell={case.ncell} precision={precision}", flush=True)
    s = Solver(case, precision)
    s.set_state(u)
    s.rk3_steps(3, cfl=0.5)
    gap = np.abs((vol * (s.get_state() - u)).sum(0)) / np.abs(vol * u).sum(0).max()
    s.close()
    print("  gap", gap)
    assert np.all(gap <= 1e-13), gap


# the largest mesh of the one-kernel march, against the two kernels
def test_largest_march_on_one_point_faces():
    case = Case(CaseSpec("f-muscl-32", HEX, 32, "muscl", jitter=0.1, seed=3))
    assert case.ncell == 32768
    u = case.init_state()
    out = []
    for timed in (False, True):
        print(f"[one-point march] ncell={case.ncell} timed={timed}", flush=True)
        s = Solver(case, UCNS_FP64)
        if timed:
            s.reset_stats()
        s.set_state(u)
        t = s.rk3_steps(3, cfl=0.5)
        out.append((s.get_state(), t, s.stats()["n_flux"]))
        s.close()
    (a, ta, na), (b, tb, nb) = out
    assert (na, nb) == (0, 9)
    close(a, b, 1e-12)
    assert abs(ta - tb) <= 1e-12 * tb


# per-face boundary states in the one-kernel march
@pytest.mark.parametrize("precision,tol", [(UCNS_FP64, 1e-12), (UCNS_MIXED, 1e-5)], ids=["fp64", "mixed"])
def test_jet_inflow_on_one_point_faces(precision, tol):
    from oracle import oracle
    from test_boundary import face_centres
    from test_gpu_boundary import P0, prim2cons
    case = Case(CaseSpec("jet-muscl", HEX, 9, "muscl", jitter=0.1, seed=9, bc=(1, 2, 4, 4, 3, 3)))
    outer = prim2cons(1.0, 0.5, 0.0, 0.0, P0)
    jet = prim2cons(1.4, 2.0, 0.2, -0.1, 0.9 * P0)
    inside = np.linalg.norm(face_centres(case)[..., 1:] - 0.5 * case.spec.length, axis=-1) < 0.3 * case.spec.length
    states = np.where(inside[..., None], jet, outer)
    u = case.init_state()
    print(f"[one-point jet] ncell={case.ncell} precision={precision}", flush=True)
    oracle.set_boundary(1, outer, outer)
    oracle.set_boundary_faces(states, None)
    try:
        ref = Oracle(case).rk3(u, 1, cfl=0.4)[0]
    finally:
        oracle.set_boundary_faces(None, None)
    uniform = Oracle(case).rk3(u, 1, cfl=0.4)[0]
    s = Solver(case, precision)
    s.set_boundary(1, outer, outer)
    s.set_boundary_faces(states, None)
    s.set_state(u)
    s.rk3_steps(1, cfl=0.4)
    err = rel_l2(s.get_state(), ref)
    s.close()
    print("  rel L2", err)
    assert np.all(err <= tol), err
    assert rel_l2(uniform, ref).max() > 1e-4  # the jet is seen
