"""bench.py names the reconstruction kernel that the library's rules pick: both
sides of every line of the dispatch (ucns_upload_prestore, launch_recon_t)."""
import dataclasses

import pytest

import bench
from ucns3d_amd.case import HEX, PRISM, TET, Case, CaseSpec, reduced

W4 = CaseSpec("n-hex4", HEX, 9, "weno4", jitter=0.1, seed=3)
NAMES = [
    (CaseSpec("n-muscl", HEX, 4, "muscl"), "k_recon_muscl<double>", "k_recon_muscl<float>"),
    (W4, "k_recon_block<double,19,39,7>", "k_recon_block<float,19,39,7>"),
    (dataclasses.replace(W4, n=16), "k_recon_block<double,19,39,7>", "k_recon_block<float,19,39,7>"),
    (dataclasses.replace(W4, n=17), "k_recon_s64<19,39,7,7>", "k_recon_block<float,19,39,7>"),
    (dataclasses.replace(W4, n=19), "k_recon_s64<19,39,7,7>", "k_recon_s32<19,39,7,7>"),
    (CaseSpec("n-tet4", TET, 5, "weno4"), "k_recon_block<double,19,39,5>", "k_recon_block<float,19,39,5>"),
    (CaseSpec("n-prism4", PRISM, 10, "weno4"), "k_recon_w64<19,39,7>", "k_recon_w32<19,39,7>"),
    (CaseSpec("n-tet3", TET, 5, "weno3"), "k_recon_s64<9,19,3,5>", "k_recon_s32<9,19,3,5>"),
    (CaseSpec("n-hex3", HEX, 9, "weno3"), "k_recon_s64<9,19,3,7>", "k_recon_s32<9,19,3,7>"),
    (reduced("c4", 3), "k_recon_s64<9,19,3,6>", "k_recon_s32<9,19,3,6>"),
    (dataclasses.replace(reduced("c4", 3), ees=5), "k_recon_cw64<9,19,3>", "k_recon_cw32<9,19,3>"),
    (dataclasses.replace(W4, ees=5), "k_recon_cw64<19,39,7>", "k_recon_cw32<19,39,7>"),
    (dataclasses.replace(W4, wenwrt=2, n=17), "k_recon_block<double,19,39,7>", "k_recon_block<float,19,39,7>"),
    (CaseSpec("n-tet5", TET, 6, "weno5"), "k_recon<double,34,69,7>", "k_recon<float,34,69,7>"),
    (CaseSpec("n-tet5c", TET, 6, "weno5", ees=5), "k_recon_cweno5<double,4>", "k_recon_cweno5<float,4>"),
    (CaseSpec("n-tet5ch", TET, 6, "weno5", wenwrt=2), "k_recon<double,34,69,7,true>", "k_recon<float,34,69,7,true>"),
]


@pytest.mark.parametrize("spec,fp64,mixed", NAMES, ids=[f"{s.name}-{s.n}-{s.ees}-{s.wenwrt}" for s, _, _ in NAMES])
def test_reconstruction_kernel_names(spec, fp64, mixed):
    case = Case(spec)
    assert bench.recon_kernel_name(case, 0) == fp64
    assert bench.recon_kernel_name(case, 1) == mixed
