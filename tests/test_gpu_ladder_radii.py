"""The bubble ladder's multi-radius x pass is the single-radius one, bit for bit.

With tabulated windows (top-hat, Gaussian) the inverse x pass covers several
radii per launch (MRX_LADDER_RADII, read when a context is created; by default
as many as fit a fixed number of bytes, two at least).  Each radius's spectra
are those of the one-radius pass, so every output grid and global must be
identical for 1, 3 (groups that do not divide the ladder) and 4 radii per pass,
from 64^3 to the full 512^3.

The spin temperature's sharp-k shells that share a transform are grouped in the
same way, by the same variable.
"""
import os

import numpy as np
import pytest

from meraxes_amd import params as P
from meraxes_amd import reion, synth
from meraxes_amd._lib import Context

pytestmark = pytest.mark.gpu


def context_with(radii):
    old = os.environ.pop("MRX_LADDER_RADII", None)
    if radii is not None:
        os.environ["MRX_LADDER_RADII"] = str(radii)
    try:
        return Context(0)
    finally:
        os.environ.pop("MRX_LADDER_RADII", None)
        if old is not None:
            os.environ["MRX_LADDER_RADII"] = old


def run_with(radii, p, d, s, w, xe):
    c = context_with(radii)
    try:
        return reion.find_hii_bubbles(c, p, d, s, w, x_e=xe)
    finally:
        c.close()


@pytest.mark.parametrize("N,filt,spin", [(64, 0, 0), (64, 2, 1), (128, 0, 1), (512, 0, 1)])
def test_radii_per_pass_do_not_change_results(ctx, N, filt, spin):
    print(f"ladder radii N={N} filter={filt} spin={spin}", flush=True)
    d, s, w = synth.snapshot_inputs(N, 17)
    xe = None
    if spin:
        rng = np.random.default_rng(3)
        xe = synth.to_padded((0.02 + 0.05 * rng.random((N, N, N))).astype(np.float32))
    p = P.hii_params(N, 100.0, 8.0, filter_type=filt, uvb_flag=1, include_spin_temp=spin)
    ref = run_with(1, p, d, s, w, xe)
    for k in (3, 4):
        got = run_with(k, p, d, s, w, xe)
        for name in ("xH", "r_bubble", "J_21", "z_at_ionization", "J_21_at_ionization"):
            assert np.array_equal(got[name], ref[name]), (k, name)
        for name in ("volume_weighted_global_xH", "mass_weighted_global_xH", "volume_weighted_global_J_21"):
            assert got[name] == ref[name], (k, name)


def shells_with(radii, N, nsteps):
    """The filtered shells and T_S of one snapshot in a context of their own, and the device memory
    it took."""
    import torch

    zz = P.snapshot_redshifts()
    snap, nh = 24, 8
    d, st, w = (torch.from_numpy(a).cuda() for a in synth.snapshot_inputs(N, 23))
    hist = torch.stack([w * (1.0 - 0.05 * k) for k in range(nh)])
    fc = np.zeros(len(zz))
    fc[:snap] = np.linspace(1e-4, 5e-3, snap)
    p = P.ts_params(N, 0.78125 * N, snap, zz, fc, nh, num_filter_steps=nsteps, on_device=1)
    xe, xe_box = torch.full_like(d, 2e-3), torch.empty_like(d)
    Tk = torch.full((N, N, N), 50.0, device="cuda")
    TS = torch.empty_like(Tk)
    c = context_with(radii)
    try:
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        reion.compute_ts(c, p, d, st, w, hist, xe, Tk, x_e_box=xe_box, TS_box=TS)
        torch.cuda.synchronize()
        took = free - torch.cuda.mem_get_info()[0]
        return reion.ts_last_shells(c, N, nsteps), TS.cpu().numpy(), took
    finally:
        c.close()


@pytest.mark.parametrize("N,nsteps", [(64, 40), (96, 13), (160, 7)])
def test_shells_per_pass_do_not_change_results(ctx, N, nsteps):
    print(f"shells N={N} steps={nsteps}", flush=True)
    ref = shells_with(1, N, nsteps)
    for k in (3, None):
        got = shells_with(k, N, nsteps)
        assert np.array_equal(got[0], ref[0]), k
        assert np.array_equal(got[1], ref[1]), k


def test_memory_of_shells_one_per_pass(ctx):
    """The shells, three spectra or grids and a byte per cell: what a call is left with when the
    spectra of a group are not to be had."""
    N, nsteps = 128, 8
    cells = N**3
    took = shells_with(1, N, nsteps)[2]
    print(f"one shell per pass {took / 2**20:.0f} MiB", flush=True)
    assert took <= 4 * cells * (nsteps + 3) + cells + (32 << 20)  # and small buffers, rounding of allocations
