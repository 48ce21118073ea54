"""GPU: the ladder's y pass and threshold in one kernel (plane_fft.hpp).

Every length it is built for, where its pieces meet edges: one radix after the
eight (N = 32, 48, 64) or two (96, 128), row blocks that do not fill the
workgroup (48, 96), two to four fields, groups of one radius, of three (a
remainder at the end) and of the whole ladder.  Crossings are folded into the
state in radius order whatever the group, so the grids are the same bits; the
first group size is also held to the oracle's outcome.
"""
import numpy as np
import pytest

from meraxes_amd import params as P
from meraxes_amd import synth

from test_gpu_hii import check_parity, run_pair
from test_gpu_ladder_radii import run_with

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,spin,uvb,ftype", [(32, 1, 1, 0), (48, 0, 1, 2), (48, 1, 0, 0), (64, 0, 0, 0), (96, 1, 1, 2),
                                              (96, 0, 1, 0), (128, 1, 1, 0), (128, 0, 0, 2)])
def test_planes_for_any_group_of_radii(ctx, N, spin, uvb, ftype):
    print(f"plane N={N} spin={spin} uvb={uvb} filter={ftype}", flush=True)
    d, s, w = synth.snapshot_inputs(N, 40 + N)
    xe = None
    if spin:
        xe = synth.to_padded(np.random.default_rng(7).uniform(0.0, 0.2, (N, N, N)).astype(np.float32))
    p = P.hii_params(N, 100.0 * N / 64, 8.5, filter_type=ftype, efficiency=100.0, uvb_flag=uvb, include_spin_temp=spin)
    g, o = run_pair(ctx, p, d, s, w, xe=xe)
    check_parity(g, o, N, f"N={N}", eff=100.0, neutral_vs_fp64=True)
    for K in (1, 3):
        r = run_with(K, p, d, s, w, xe)
        for k in ("xH", "r_bubble", "z_at_ionization", "J_21", "J_21_at_ionization"):
            assert np.array_equal(r[k], g[k]), (K, k)
        assert r["volume_weighted_global_xH"] == g["volume_weighted_global_xH"]
    assert len(np.unique(g["r_bubble"])) > 2
