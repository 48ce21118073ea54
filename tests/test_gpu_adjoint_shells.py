"""GPU: the shells' adjoint in groups (shared gradients, one inverse transform per state of
the working grid) at grids with factors 3 and 5 and shell counts that do not fill a group.

Central differences of the forward along random directions of the SFR and of its history,
with an efficiency so small that nothing ionises (delta_T is then smooth in them).  The
difference is cubic in the step: 0.05 of each cell's own SFR leaves about 0.05^2 of the
second logarithmic derivatives, which are of order one; 1e-2 is asked.
"""
import numpy as np
import pytest

from meraxes_amd import autograd as MA
from meraxes_amd import params as P
from meraxes_amd import synth

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("N,nsteps,ftype", [(48, 40, 1), (96, 37, 1), (160, 18, 1), (64, 40, 0), (32, 9, 1)])
def test_shell_adjoint_along_directions(ctx, N, nsteps, ftype):
    print(f"N={N} shells {nsteps} filter {ftype}", flush=True)
    L, snap, nh = 0.78125 * N, 24, 8
    zz = P.snapshot_redshifts()
    d, s, w = (torch.from_numpy(a).cuda() for a in synth.snapshot_inputs(N, 90 + N))
    hist = torch.stack([w * (1.0 - 0.05 * k) for k in range(nh)])
    fc = np.zeros(len(zz))
    fc[:snap] = np.linspace(1e-4, 5e-3, snap)
    tsp = P.ts_params(N, L, snap, zz, fc, nh, num_filter_steps=nsteps, heating_filter_type=ftype, on_device=1)
    z = float(zz[snap])
    hp = P.hii_params(N, L, z, efficiency=1e-6, include_spin_temp=1, on_device=1)
    bp = P.tb_params(N, z, include_spin_temp=1, on_device=1)
    xe = torch.full_like(d, 2e-3)
    Tk = torch.full((N, N, N), 50.0, device="cuda")
    g = torch.Generator(device="cuda").manual_seed(N)
    weight = torch.rand((N, N, N), generator=g, device="cuda", dtype=torch.float64)

    def loss(w_, h_):
        return (MA.snapshot(ctx, tsp, hp, bp, d, s, w, w_, h_, xe, Tk)[0].double() * weight).sum()

    wr, hr = w.clone().requires_grad_(True), hist.clone().requires_grad_(True)
    gw, gh = torch.autograd.grad(loss(wr, hr), (wr, hr))
    eps = 0.05
    for name, base, grad in (("sfr", w, gw), ("history", hist, gh)):
        p = torch.randint(0, 2, base.shape, generator=g, device="cuda").float() * base  # half of the cells, upwards
        a, b = (base + eps * p, base - eps * p)
        fd = float((loss(a, hist) - loss(b, hist)) if name == "sfr" else (loss(w, a) - loss(w, b))) / (2 * eps)
        an = float((grad.double() * p.double()).sum())
        print(f"  {name}: differences {fd:.6e} adjoint {an:.6e} ({abs(an - fd) / abs(fd):.1e})", flush=True)
        assert abs(an - fd) <= 1e-2 * abs(fd), name
