"""GPU: the shell tables' frequency integrals (ts_quad.hpp) against the host build.

The step's averages of X-ray ionisation and Ly-alpha flux are linear in the
tables, so they are recomputed here in float64 from the library's own filtered
shells and the host tables (mrx_ts_snapshot_tables, the same QAG and Brent on the
CPU).  The two builds round differently (sums over a wave, the device's exp, log,
pow and atan), a few 1e-16 per operation over sums of 61 terms and some 60
intervals, and Brent's last secant step carries that into the lower limit by a
factor of order ten: 1e-11 is asked.
"""
import numpy as np
import pytest

from meraxes_amd import params as P
from meraxes_amd import reion, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,snap,xe0,nsteps,spec,thresh", [(32, 1, 2e-4, 40, 1.0, 500.0), (32, 12, 0.02, 40, 1.5, 500.0),
                                                           (48, 24, 0.3, 64, 1.0, 200.0), (32, 28, 0.97, 7, 0.8, 500.0),
                                                           (64, 20, 0.99995, 40, 1.0, 500.0),
                                                           (32, 24, 2e-3, 1, 1.0, 20.0)])
def test_tables_from_the_device(ctx, N, snap, xe0, nsteps, spec, thresh):
    print(f"N={N} snapshot {snap} x_e {xe0} {nsteps} shells", flush=True)
    zz = P.snapshot_redshifts()
    d, s, w = synth.snapshot_inputs(N, 70 + snap)
    nh = snap + 1
    hist = np.stack([w * np.float32(1.0 - 0.01 * k) for k in range(nh)])

    def params():
        fc = np.zeros(len(zz))
        fc[:snap] = np.linspace(1e-4, 5e-3, snap)
        p = P.ts_params(N, 100.0 * N / 64, snap, zz, fc, nh, num_filter_steps=nsteps)
        p.spec_index_xray_gal = spec
        p.nu_xray_gal_threshold = thresh
        return p, fc

    p, fc = params()
    xe = np.full_like(d, xe0)
    Tk = np.full((N, N, N), 40.0, np.float32)
    g = reion.compute_ts(ctx, p, d, s, w, hist, xe.copy(), Tk)
    v = reion.ts_last_shells(ctx, N, nsteps).astype(np.float64)
    ph, fch = params()
    t = reion.ts_snapshot_tables(ph, g["collapse_fraction"], g["x_e_ave"])
    assert fch[snap] == fc[snap] and t.no_light == 0
    arr = lambda a: np.ctypeslib.as_array(a)  # noqa: E731
    XH = np.array([1.0e-4, 2.318e-4, 4.677e-4, 1.0e-3, 2.318e-3, 4.677e-3, 1.0e-2, 2.318e-2, 4.677e-2, 1.0e-1, 0.5, 0.9,
                   0.99, 0.999], np.float32)
    x = float(np.float32(xe0))
    if x > XH[-1] * 0.999:
        x = float(XH[-1]) * 0.999
    lo = int(np.searchsorted(XH, np.float32(x), side="right")) - 1
    fr = x - float(XH[lo])
    dxh = float(XH[lo + 1] - XH[lo])
    pv = (100.0 * N / 64 / P.HUBBLE_H / N) ** 3
    fac = 1.0 / pv * (P.UNIT_MASS_G / P.units()["unit_time_s"]) * P.UNIT_LENGTH_CM ** -3.0 / 1.989e33
    total = {}
    for name, tab in (("ion", arr(t.freq_ion)), ("lya", arr(t.freq_lya))):
        f = (tab[lo + 1][:nsteps] - tab[lo][:nsteps]) / dxh * fr + tab[lo][:nsteps]
        wgt = fac * arr(t.dt_dzpp)[:nsteps] * arr(t.dzpp)[:nsteps] * arr(t.zpp_pow)[:nsteps] * f
        total[name] = np.tensordot(wgt, v, 1) * t.const_zp_prefactor
    ion = (t.dt_dzp * total["ion"]).mean()
    e = abs(g["volume_ave_Xion"] - ion) / abs(ion)
    print(f"  <Xion> {g['volume_ave_Xion']:.6e} rel {e:.2e}", flush=True)
    assert e <= 1e-11
    zf = np.float32(t.zp)
    No = 3.0 * P.HUBBLE ** 2 * P.HUBBLE_H ** 2 / (8 * np.pi * P.GRAVITY) * P.BARYON_FRAC * P.OMEGA_M
    Nb0 = No * (1 - P.Y_HE) / 1.6726e-24 + No * P.Y_HE / (4 * 1.6726e-24)
    n_b = Nb0 * float(np.float32(1) + zf) ** 3 * (np.float32(1) + d[:, :, :N]).astype(np.float64)
    star = fac * float(np.float32(1) + zf) ** 2 * (1 + arr(t.zpp)[:nsteps]) * arr(t.sum_lyn)[:nsteps] * arr(
        t.dt_dzpp)[:nsteps] * arr(t.dzpp)[:nsteps]
    J = total["lya"] * n_b + np.tensordot(star, v, 1) * ((2.9979e10 / (4.0 * np.pi)) / (1.6726e-24 / 1.989e33))
    e = abs(g["volume_ave_J_alpha"] - J.mean()) / abs(J.mean())
    print(f"  <J_alpha> {g['volume_ave_J_alpha']:.6e} rel {e:.2e}", flush=True)
    assert e <= 1e-11
