"""GPU: the inverse row transforms (row_fft.hpp) at every row length they are built for.

The C2R round trip ends in k_c2r_z, the bubble finder's ladder in
k_c2r_threshold; both bring rows back with row_fft.hpp, whose row blocks and
first / last stages differ from length to length: an odd count of first-stage
butterflies (N = 48), results that meet in LDS (N = 128, 1024), three-wave
workgroups (N = 320).  The transform is compared with float64 at eps log2(N^3),
the error bound of a float Stockham transform's rms; the bubble finder with the
oracle, with three to five fields.
"""
import numpy as np
import pytest

from meraxes_amd import params as P
from meraxes_amd import reion, synth
from oracle import oracle as O

from test_gpu_hii import check_parity, run_pair
from test_gpu_recomb import close, nrec_field

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [32, 48, 64, 96, 128, 160, 192, 320, 384])
def test_c2r_rows_against_float64(ctx, N):
    print(f"c2r N={N}", flush=True)
    rng = np.random.default_rng(N)
    f = rng.normal(0, 1, (N, N, N)).astype(np.float32)
    H = np.fft.rfftn(f.astype(np.float64)).astype(np.complex64)
    got = reion.fft_c2r_3d(ctx, H)
    want = np.fft.irfftn(H.astype(np.complex128), s=(N, N, N), axes=(0, 1, 2)) * float(N) ** 3
    e = np.sqrt(((got[:, :, :N] - want) ** 2).sum() / (want ** 2).sum())
    print(f"  rel L2 {e:.2e}", flush=True)
    assert e <= 6e-8 * np.log2(float(N) ** 3)
    assert (got[:, :, N:] == 0).all()


@pytest.mark.parametrize("N,spin,rec,ftype", [(32, 0, 0, 0), (48, 1, 0, 2), (48, 0, 1, 0), (96, 1, 1, 0),
                                              (96, 0, 0, 1), (128, 1, 1, 0), (192, 0, 0, 1)])
def test_ladder_rows_against_the_oracle(ctx, N, spin, rec, ftype):
    print(f"ladder N={N} spin={spin} rec={rec} filter={ftype}", flush=True)
    d, s, w = synth.snapshot_inputs(N, 60 + N)
    xe = None
    if spin:
        xe = synth.to_padded(np.random.default_rng(3).uniform(0.0, 0.2, (N, N, N)).astype(np.float32))
    p = P.hii_params(N, 100.0 * N / 64, 8.5, filter_type=ftype, efficiency=100.0, uvb_flag=1, include_spin_temp=spin,
                     include_recombinations=rec, prev_redshift=8.8)
    if not rec:
        g, o = run_pair(ctx, p, d, s, w, xe=xe)
        check_parity(g, o, N, f"N={N}", eff=100.0, neutral_vs_fp64=True)
        return
    nrec, g12 = nrec_field(N, 5, 0.05), np.zeros((N, N, N), np.float32)
    o = O.find_hii_bubbles(p, d, s, w, x_e=xe, want_ratio=True, N_rec=nrec.copy(), Gamma12=g12.copy())
    g = reion.find_hii_bubbles(ctx, p, d, s, w, x_e=xe, N_rec=nrec.copy(), Gamma12=g12.copy())
    flips = check_parity(g, o, N, f"N={N}", eff=100.0, neutral_vs_fp64=True)
    crossed = ~flips & (o["Gamma12"] != 0)
    assert crossed.sum() > 50
    close(g["Gamma12"], o["Gamma12"], "Gamma12", crossed)
    close(g["N_rec"][:, :, :N], o["N_rec"][:, :, :N], "N_rec", ~flips)


@pytest.mark.parametrize("N,spin,ftype", [(32, 0, 0), (96, 1, 2), (256, 0, 1), (256, 1, 0)])
def test_ladder_without_the_uvb_leaves_the_sfr_out(ctx, N, spin, ftype):
    """The weighted SFR only feeds J_21: without the UVB the ladder transforms one field less
    (two or three, also where rows of 256^3 go through registers), every other grid the same.
    The cells are dealt to lanes by the number of fields there, so the globals' double sums are
    formed in another order: some 30 roundings of 2^-53 along each path of the reduction."""
    print(f"N={N} spin={spin} filter={ftype}", flush=True)
    d, s, w = synth.snapshot_inputs(N, 80 + N)
    xe = None
    if spin:
        xe = synth.to_padded(np.random.default_rng(5).uniform(0.0, 0.2, (N, N, N)).astype(np.float32))
    r = [reion.find_hii_bubbles(ctx, P.hii_params(N, 0.8 * N, 8.0, filter_type=ftype, efficiency=30.0, uvb_flag=u,
                                                  include_spin_temp=spin), d, s, w, x_e=xe) for u in (1, 0)]
    for k in ("xH", "r_bubble", "z_at_ionization"):
        assert np.array_equal(r[0][k], r[1][k]), k
    for k in ("volume_weighted_global_xH", "mass_weighted_global_xH", "n_radii"):
        assert abs(r[0][k] - r[1][k]) <= 30 * 2.0**-53 * abs(r[1][k]), k
    assert (r[0]["r_bubble"] > 0).any()
