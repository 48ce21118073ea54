"""GPU: the shells' adjoint in groups (shared gradients, one inverse transform per state of
the working grid) at grids with factors 3 and 5 and shell counts that do not fill a group.

* Central differences of the forward along random directions of the SFR and of its history,
  with an efficiency so small that nothing ionises (delta_T is then smooth in them).  The
  difference is cubic in the step: 0.05 of each cell's own SFR leaves about 0.05^2 of the
  second logarithmic derivatives, which are of order one; 1e-2 is asked.
* The same gradients against float64 autograd of an independent restatement
  (tests/ts_torch.py), every cell.
* Groups of any size (MRX_ADJOINT_SHELLS) against shells taken one by one, and the memory
  that one by one takes.
"""
import os

import numpy as np
import pytest

import ts_torch as TT
from meraxes_amd import autograd as MA
from meraxes_amd import params as P
from meraxes_amd import reion, synth
from meraxes_amd._lib import Context
from oracle import oracle as O
from test_gpu_adjoint import rel_l2, tb_const

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(autouse=True)
def give_back():
    """The float64 graph takes tens of GB that torch's cache would keep from the tests after."""
    yield
    torch.cuda.empty_cache()


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


def fixed_case(N, nsteps, seed):
    """A snapshot whose table means are given and in which nothing ionises; weights of the loss."""
    L, snap, nh = 0.78125 * N, 24, 8
    zz = P.snapshot_redshifts()
    d, s, w = (torch.from_numpy(a).cuda() for a in synth.snapshot_inputs(N, seed))
    hist = torch.stack([w * (1.0 - 0.05 * k) for k in range(nh)])
    fc = np.zeros(len(zz))
    fc[:snap] = np.linspace(1e-4, 5e-3, snap)
    tsp = P.ts_params(N, L, snap, zz, fc, nh, num_filter_steps=nsteps, on_device=1)
    tsp.fixed_globals, tsp.fixed_collapse_fraction, tsp.fixed_x_e_ave = 1, 5e-3, 2e-3
    z = float(zz[snap])
    hp = P.hii_params(N, L, z, efficiency=1e-6, include_spin_temp=1, on_device=1)
    bp = P.tb_params(N, z, include_spin_temp=1, on_device=1)
    xe = torch.full_like(d, 2e-3)
    Tk = torch.full((N, N, N), 50.0, device="cuda")
    weight = torch.rand((N, N, N), generator=torch.Generator(device="cuda").manual_seed(N), device="cuda")
    return dict(tsp=tsp, hp=hp, bp=bp, d=d, s=s, w=w, hist=hist, xe=xe, Tk=Tk, weight=weight, keep=(zz, fc))


@pytest.mark.parametrize("N,nsteps", [(48, 40), (96, 37), (192, 40)])
def test_shell_adjoint_in_64_bits(ctx, N, nsteps):
    """1e-4 as for the 64^3 snapshot (test_gpu_adjoint): the float32 shells' rounding and, where
    a shell's value is 0 up to rounding, the clamp's derivative."""
    print(f"N={N} shells {nsteps}", flush=True)
    c = fixed_case(N, nsteps, 70 + N)
    wr, hr = c["w"].clone().requires_grad_(True), c["hist"].clone().requires_grad_(True)
    dT = MA.snapshot(ctx, c["tsp"], c["hp"], c["bp"], c["d"], c["s"], c["w"], wr, hr, c["xe"], c["Tk"])[0]
    gw, gh = torch.autograd.grad((dT.double() * c["weight"]).sum(), (wr, hr))
    tsp, hp = c["tsp"], c["hp"]
    cst = O.ts_export(tsp)
    assert cst["nsteps"] == nsteps and not cst["no_light"] and len(cst["ops"]) > 0
    w64, h64 = c["w"].double().requires_grad_(True), c["hist"].double().requires_grad_(True)
    d64 = c["d"][:, :, :N].double()
    sh = TT.shells(cst, w64, h64, N, tsp.box_size, c["d"].device)
    xn, _, TS = TT.ts_step(cst, d64, c["xe"][:, :, :N].double(), c["Tk"].double(), sh,
                           (tsp.box_size / tsp.hubble_h / N) ** 3, tsp.unit_mass_g / tsp.unit_time_s,
                           tsp.unit_length_cm ** -3.0)
    R = P.radius_ladder(hp)[-1]
    s64 = c["s"][:, :, :N].double()
    s64 = torch.where(s64 < 1e-8, torch.zeros_like(s64), s64)
    fcoll = s64 * (R**3 / (hp.box_size / N) ** 3 / (R**3 * hp.omega_m * hp.rho_crit)) / (1.0 + d64)
    xH = 1.0 - torch.where(xn < 1e-8, torch.zeros_like(xn), torch.clamp(xn, max=0.999)) - hp.efficiency * fcoll
    zf = float(np.float32(hp.redshift))
    dT64 = tb_const(hp.redshift) * torch.clamp(xH, 0.0, 1.0) * (1.0 + d64) * (1.0 - 2.728 * (1.0 + zf) / TS)
    e_T = rel_l2(dT.detach().cpu().numpy(), dT64.detach().cpu().numpy())
    rw, rh = torch.autograd.grad((dT64 * c["weight"]).sum(), (w64, h64))
    errs = [rel_l2(g.cpu().numpy(), r.cpu().numpy()) for g, r in ((gw, rw), (gh, rh))]
    print(f"  delta_T {e_T:.1e}; gradient of the SFR {errs[0]:.1e}, of its history {errs[1]:.1e}", flush=True)
    assert e_T < 1e-5 and max(errs) < 1e-4


def adjoint_with(shells, c):
    """The gradients with `shells` shells per group (None: the default) in a context of their own,
    and the device memory that the adjoint took in it."""
    old = os.environ.pop("MRX_ADJOINT_SHELLS", None)
    if shells is not None:
        os.environ["MRX_ADJOINT_SHELLS"] = str(shells)
    try:
        one = Context(0)
    finally:
        os.environ.pop("MRX_ADJOINT_SHELLS", None)
        if old is not None:
            os.environ["MRX_ADJOINT_SHELLS"] = old
    try:
        TS, xe_box = torch.empty_like(c["Tk"]), torch.empty_like(c["d"])
        reion.compute_ts(one, c["tsp"], c["d"], c["s"], c["w"], c["hist"], c["xe"].clone(), c["Tk"].clone(),
                         x_e_box=xe_box, TS_box=TS)
        xH = reion.find_hii_bubbles(one, c["hp"], c["d"], c["s"], c["w"], x_e=xe_box)["xH"]
        adj = lambda: reion.snapshot_adjoint(one, c["tsp"], c["hp"], c["bp"], c["d"], c["s"], c["w"],  # noqa: E731
                                             c["hist"], c["xe"], c["Tk"], xH, TS, xe_box, c["weight"])
        hold = [torch.empty_like(c[k]) for k in ("d", "s", "w", "hist", "xe", "Tk")]  # torch's cache for the gradients
        del hold
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        g = adj()
        torch.cuda.synchronize()
        return g, free - torch.cuda.mem_get_info()[0]
    finally:
        one.close()


@pytest.mark.parametrize("N,nsteps", [(64, 40), (96, 11)])
def test_groups_of_shells_give_one_gradient(ctx, N, nsteps):
    """Each shell's field passes a forward and an inverse transform (3e-7 together) and up to 40
    are added in float (2.4e-6 at worst): 3e-6 between any two ways of grouping."""
    c = fixed_case(N, nsteps, 80 + N)
    ref, _ = adjoint_with(0, c)
    for k in (1, 3, 8, None):
        got, _ = adjoint_with(k, c)
        e = {n: rel_l2(got[n].cpu().numpy(), ref[n].cpu().numpy()) for n in ref}
        print(f"N={N} groups of {k}: " + ", ".join(f"{n} {v:.1e}" for n, v in e.items()), flush=True)
        assert max(e.values()) < 3e-6, k


def test_memory_of_shells_one_by_one(ctx):
    """Beside the four double grids of the shell sums, two padded grids: what is left to take when
    a group's work space is not to be had."""
    N = 128
    c = fixed_case(N, 12, 3)
    sums, grid = 4 * 8 * N**3, 4 * N * N * (N + 2)
    took = {k: adjoint_with(k, c)[1] for k in (0, 8)}
    print(f"one by one {took[0] / 2**20:.0f} MiB, groups of 8 {took[8] / 2**20:.0f} MiB", flush=True)
    slack = 16 << 20  # rounding of allocations
    assert took[0] <= sums + 2 * grid + slack
    assert took[8] >= sums + 9 * (grid + 4 * N**3) - slack
