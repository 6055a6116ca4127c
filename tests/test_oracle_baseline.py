"""The CPU baseline's AVX-512 kernel (bench.py's cpu_baseline on AVX-512
hosts; not the oracle) against the FP64 oracle with the exact Ewald closed
form: it must compute the same physics to float accuracy, or the baseline
it reports would not be a step of the same workload."""
import numpy as np
import pytest

from gmxapi_amd import systems as S
from oracle import oracle as O
from tests.helpers import oracle_for, rms


def _baseline(s):
    o = O.Oracle("bench_f32", "ewald", rlist=s.rlist, rcoulomb=s.rcoulomb)
    o.setup(s.box, s.x, s.types, s.charges, O.nblib_nbfp(s.c6, s.c12, "f32"), s.ntypes, s.excl_off, s.excl_idx)
    if not o.simd_available():
        pytest.skip("no AVX-512 on this host")
    return o


@pytest.mark.parametrize("s", [S.config(0), S.hetero_chains(1200, 2.3, ntypes=5, seed=3, rc=0.9, rlist=1.0)],
                         ids=["water9000", "chains1200"])
def test_simd_baseline_matches_fp64(s):
    o = _baseline(s)
    r = o.compute_simd(s.x, 4)
    r64 = oracle_for(s, "f64", ewald_exact=True).compute(s.x)
    assert rms(r["f"] - r64["f"]) / rms(r64["f"]) < 5e-6
    scale = abs(r64["Vvdw"]) + abs(r64["Vc"])
    assert abs(r["Vvdw"] - r64["Vvdw"]) < 1e-5 * scale
    assert abs(r["Vc"] - r64["Vc"]) < 1e-5 * scale
    # the thread count changes the summation order only
    r1 = o.compute_simd(s.x, 1)
    assert rms(r1["f"] - r["f"]) / rms(r64["f"]) < 1e-6


def test_simd_baseline_declines_other_flavours():
    s = S.small_water_box(216, seed=11)
    o = O.Oracle("bench_f32", "rf", rlist=s.rlist, rcoulomb=s.rcoulomb)
    o.setup(s.box, s.x, s.types, s.charges, O.nblib_nbfp(s.c6, s.c12, "f32"), s.ntypes, s.excl_off, s.excl_idx)
    assert not o.simd_available()
    assert o.compute_simd(s.x, 2) is None
