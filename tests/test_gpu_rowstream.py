"""The row-stream kernels of WENO-4 on meshes past the block kernels' lines (512
tiles, 768 in mixed precision) whose last tile is partial: 9,261 hexahedra (5
cells in it) and 13,182 tetrahedra (6), with open sides, in a calm state and in
one with cells that fall to MUSCL and to first order.

Reconstruction and residual against the oracle at the parity bars (relative L2
per variable 1e-11; mixed precision 1e-5 after a step), the products against the
register kernels: in FP64 another order of sums (1e-10 of the largest value), in
mixed precision products of the same FP32 forward values (a hundred FP32
roundings, 1e-5)."""
import numpy as np
import pytest

from oracle import oracle
from oracle.oracle import Oracle
from ucns3d_amd.case import HEX, TET, Case, CaseSpec
from ucns3d_amd.native import UCNS_FP64, UCNS_KERNELS_REGISTER, UCNS_MIXED
from ucns3d_amd.solver import Solver

from test_gpu_boundary import P0, prim2cons
from test_gpu_parity import valid_uleft_mask
from test_gpu_paths import close, rel_l2

pytestmark = pytest.mark.gpu

MESHES = {
    "hex-9261": (CaseSpec("rs-hex", HEX, 21, "weno4", jitter=0.1, seed=3, bc=(1, 2, 4, 4, 3, 3)),
                 prim2cons(1.0, 0.5, 0.0, 0.0, P0)),
    "tet-13182": (CaseSpec("rs-tet", TET, 13, "weno4", jitter=0.1, seed=4, bc=(6,) * 6),
                  prim2cons(1.0, 0.3, 0.1, 0.0, P0)),
}
_cache = {}


def get(name):
    if name not in _cache:
        spec, fs = MESHES[name]
        case = Case(spec)
        assert case.ncell % 8 in (5, 6) and case.ncell > 8 * 768
        calm = case.init_state() * (1 + 1e-3 * np.random.default_rng(2).uniform(-1, 1, (case.ncell, 5)))
        # a staircase of factors 40 through a cell and one of its neighbours: the
        # cell's limited value still leaves its average by more than 0.95
        rough = calm.copy()
        m = case.structs()[0]
        nb = np.ctypeslib.as_array(m.ineigh, shape=(case.ncell * case.nface_max,)).reshape(case.ncell, -1)
        code = np.ctypeslib.as_array(m.bcode, shape=(case.ncell * case.nface_max,)).reshape(case.ncell, -1)
        for c in np.r_[np.random.default_rng(8).choice(case.ncell, 8, replace=False), case.ncell - 1]:
            f = int(np.flatnonzero(code[c, :4] == 0)[0])
            rough[c] *= 40.0
            rough[nb[c, f] - m.index_base] *= 1600.0
        _cache[name] = (case, Oracle(case), fs, {"calm": calm, "rough": rough})
    return _cache[name]


def solver(name, precision, **kw):
    case, _, fs, _ = get(name)
    s = Solver(case, precision, **kw)
    s.set_boundary(1, fs, fs)
    oracle.set_boundary(1, fs, fs)
    return s


@pytest.mark.parametrize("state", ["calm", "rough"])
@pytest.mark.parametrize("name", list(MESHES))
def test_residual_fp64(name, state):
    case, orc, _, states = get(name)
    u = states[state]
    print(f"[row stream residual] {name} {state} ncell={case.ncell}", flush=True)
    s = solver(name, UCNS_FP64)
    s.set_state(u)
    err = rel_l2(s.residual(), orc.residual(u)[0])
    ul, (ul_ref, cnt) = s.reconstruct(), orc.reconstruct(u)
    st = s.stats()
    s.close()
    print("  rel L2", err, "MUSCL, first order", cnt)
    assert (st["n_reduced_last"], st["n_firstorder_last"]) == (cnt[0], cnt[1])
    assert 0 < cnt[0] < case.ncell and (cnt[1] > 0) == (state == "rough")
    assert np.all(err <= 1e-11), err
    m = valid_uleft_mask(case)
    assert np.abs(ul[m] - ul_ref[m]).max() <= 1e-12 * np.abs(ul_ref[m]).max()


@pytest.mark.parametrize("state", ["calm", "rough"])
@pytest.mark.parametrize("name", list(MESHES))
def test_mixed_step(name, state):
    case, orc, _, states = get(name)
    u = states[state]
    print(f"[row stream mixed] {name} {state} ncell={case.ncell}", flush=True)
    s = solver(name, UCNS_MIXED)
    s.set_state(u)
    s.rk3_steps(1, cfl=0.2)
    err = rel_l2(s.get_state(), orc.rk3(u, 1, cfl=0.2)[0])
    s.close()
    print("  rel L2", err)
    assert np.all(err <= 1e-5), err


@pytest.mark.parametrize("precision,tol", [(UCNS_FP64, 1e-10), (UCNS_MIXED, 1e-5)], ids=["fp64", "mixed"])
@pytest.mark.parametrize("name", list(MESHES))
def test_products_agree_with_the_register_kernels(name, precision, tol):
    case, _, _, states = get(name)
    u = states["calm"]
    w = np.random.default_rng(6).standard_normal(u.shape)
    out = []
    for kw in ({}, {"kernels": UCNS_KERNELS_REGISTER}):
        print(f"[row stream products] {name} precision={precision} {kw}", flush=True)
        s = solver(name, precision, **kw)
        s.set_state(u)
        dt = 0.5 * s.compute_dt(0.5)
        v, vb = s.residual_vjp(w)
        a, ab, _ = s.rk3_adjoint(2, w, dt_fixed=dt)
        out.append((v, vb, a, ab))
        s.close()
    for x, y in zip(*out):
        close(x, y, tol)
