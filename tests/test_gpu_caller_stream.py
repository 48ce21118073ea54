"""GPU: calls queued one after the other on a caller's stream, through the C ABI.

The stream is handed over once (mrx_set_stream waits, so a call that is bound again waits for
the one before it) and other work lies ahead of the calls on it, so that they return with
theirs still queued.  Each must give what it gives when it is waited for, bit for bit: the
kernels are the same and add in a fixed order.
"""
import ctypes as C

import numpy as np
import pytest

from meraxes_amd import params as P
from meraxes_amd import reion, synth

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

N, L, NH = 64, 50.0, 8


def ptr(t):
    return C.c_void_p(t.data_ptr())


def snapshot(ctx, kind, snap, seed):
    """One snapshot's parameters, inputs and forward outputs."""
    zz = P.snapshot_redshifts()
    z = float(zz[snap])
    d, s, w = (torch.from_numpy(a).cuda() for a in synth.snapshot_inputs(N, seed))
    hist = torch.stack([w * (1.0 - 0.05 * k) for k in range(NH)])
    fc = np.zeros(len(zz))
    fc[:snap] = np.linspace(1e-4, 5e-3, snap)
    tsp = P.ts_params(N, L, snap, zz, fc, NH, on_device=1,
                      max_heating_redshift=z - 1.0 if kind == "homogeneous" else 20.0)
    if kind in ("fixed", "dark"):  # the grid means given; no light where the collapse fraction is 0
        tsp.fixed_globals = 1
        tsp.fixed_collapse_fraction = 0.0 if kind == "dark" else 1e-3 * seed
        tsp.fixed_x_e_ave = 2e-3
    hp = P.hii_params(N, L, z, efficiency=8.0, include_spin_temp=1, on_device=1)
    bp = P.tb_params(N, z, include_spin_temp=1, on_device=1)
    xe0 = torch.full_like(d, 2e-3)
    Tk0 = torch.full((N, N, N), 40.0 + seed, device="cuda")
    TS, xe_box = torch.empty_like(Tk0), torch.empty_like(d)
    reion.compute_ts(ctx, tsp, d, s, w, hist, xe0.clone(), Tk0.clone(), x_e_box=xe_box, TS_box=TS)
    xH = reion.find_hii_bubbles(ctx, hp, d, s, w, x_e=xe_box)["xH"]
    gdT = torch.rand((N, N, N), generator=torch.Generator(device="cuda").manual_seed(seed), device="cuda")
    torch.cuda.synchronize()
    return dict(tsp=tsp, hp=hp, bp=bp, ins=(d, s, w, hist, xe0, Tk0, xH, TS, xe_box, gdT), keep=(zz, fc))


def adjoint(ctx, c, out):
    """The snapshot's gradients into out, queued on the context's stream."""
    ctx.check(ctx.lib.mrx_snapshot_adjoint(ctx.ptr, C.byref(c["tsp"]), C.byref(c["hp"]), C.byref(c["bp"]),
                                           *[ptr(t) for t in c["ins"]], *[ptr(t) for t in out]), "snapshot_adjoint")


@pytest.mark.parametrize("first,second", [("homogeneous", "homogeneous"), ("fixed", "fixed"), ("dark", "fixed"),
                                          ("fixed", "homogeneous"), ("homogeneous", "measured")])
def test_adjoints_queued_on_one_stream(ctx, first, second):
    print(f"{first} then {second}", flush=True)
    cases = [snapshot(ctx, first, 24, 1), snapshot(ctx, second, 22, 2)]
    st = torch.cuda.Stream()
    backlog = torch.zeros(1 << 28, device="cuda")  # 1 GiB: some 0.4 ms a pass
    alone, queued = ([[torch.full_like(t, float("nan")) for t in c["ins"][:6]] for c in cases] for _ in range(2))
    torch.cuda.synchronize()
    ctx.check(ctx.lib.mrx_set_stream(ctx.ptr, C.c_void_p(st.cuda_stream)), "set_stream")
    try:
        for c, out in zip(cases, alone):
            adjoint(ctx, c, out)
            st.synchronize()
        ahead = torch.cuda.Event()
        with torch.cuda.stream(st):
            for _ in range(100):
                backlog.add_(1.0)
            ahead.record()
        adjoint(ctx, cases[0], queued[0])
        print(f"  the first call returned {'after' if ahead.query() else 'before'} the work ahead of it", flush=True)
        adjoint(ctx, cases[1], queued[1])
        st.synchronize()
    finally:
        ctx.check(ctx.lib.mrx_set_stream(ctx.ptr, None), "set_stream")
    for kind, a, q in zip((first, second), alone, queued):
        for name, x, y in zip(("deltax", "stars", "sfr", "history", "x_e_prev", "T_K"), a, q):
            assert torch.isfinite(x).all(), (kind, name)
            assert torch.equal(x, y), (kind, name)
    assert not torch.equal(alone[0][0], alone[1][0])  # the two snapshots do differ
