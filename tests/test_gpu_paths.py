"""Kernels that are chosen by a rule on the mesh, each at the sizes where its
split can go wrong: against the oracle, or against the kernels that the rule
leaves (another summation order in FP64: differences of a few hundred roundings
of 1.1e-16, held to 1e-12 of the largest value; products behind a march 1e-10)."""
import numpy as np
import pytest

from ucns3d_amd.case import PRISM, Case, CaseSpec, reduced
from ucns3d_amd.native import UCNS_FP64, UCNS_KERNELS_REGISTER
from ucns3d_amd.solver import Solver

pytestmark = pytest.mark.gpu


def close(a, b, tol):
    a, b = np.asarray(a), np.asarray(b)
    assert np.isfinite(a).all()
    d = np.abs(a - b).max()
    assert d <= tol * np.abs(b).max(), (d, np.abs(b).max())


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
