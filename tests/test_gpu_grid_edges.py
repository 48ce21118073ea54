"""GPU: the gridding's edges against the oracle, bit for bit: the smallest grid, rows that
are no multiple of 4 floats, one and nine history slots, grids that are only 4-byte aligned
(the scalar form of the initialisation), no galaxy, one galaxy, only dead ones."""
import numpy as np
import pytest

from meraxes_amd import params as P
from meraxes_amd import reion
from oracle import oracle as O

from test_gpu_grid import catalogue, dev

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("N,n,ns,spin,off,dead", [(2, 50, 3, 1, 0, 0), (6, 5, 1, 1, 0, 0), (6, 5, 9, 1, 1, 0),
                                                  (50, 100_001, 5, 1, 3, 0), (50, 100_001, 5, 0, 1, 0),
                                                  (16, 0, 4, 1, 0, 0), (16, 1, 4, 1, 0, 0), (16, 3000, 4, 1, 0, 1),
                                                  (64, 70_000, 9, 1, 0, 0)])
def test_gridding_edges(ctx, N, n, ns, spin, off, dead):
    print(f"gridding N={N} n={n} slots={ns} spin={spin} offset {off} floats dead={dead}", flush=True)
    L = 1.5 * N
    p = P.grid_params(N, L, 8.0, include_spin_temp=spin, n_store_sfr=ns, bh_mass_limit_reion=np.exp(-4.0))
    pos, type_, fesc, gross, bhm, ebhm = catalogue(max(n, 10), L, 3 + N)
    pos, type_, fesc, gross, bhm, ebhm = (np.ascontiguousarray(a[:n]) for a in (pos, type_, fesc, gross, bhm, ebhm))
    if dead:
        type_[:] = 3
    shape = (N, N, N + 2)
    hist = np.random.default_rng(2).random((ns,) + shape).astype(np.float32) if spin else None
    o = O.construct_baryon_grids(p, pos, type_, fesc, gross, bhm, ebhm, hist)

    def grid(shp, fill=None):
        t = torch.full((int(np.prod(shp)) + off,), 7.0, device="cuda")[off:].view(shp)
        if fill is not None:
            t.copy_(torch.from_numpy(fill))
        return t

    kw = dict(stars=grid(shape), weighted_sfr=grid(shape))
    if spin:
        kw.update(sfr=grid(shape), sfr_histories=grid((ns,) + shape, hist))
    g = reion.construct_baryon_grids(ctx, p, *dev(pos, type_, fesc, gross, bhm, ebhm), **kw)
    torch.cuda.synchronize()
    for k in ("stars", "weighted_sfr") + (("sfr", "sfr_histories") if spin else ()):
        a, b = g[k].cpu().numpy(), o[k]
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), (k, int((a != b).sum()))
    for k in ("n_gridded", "n_dead", "n_bh_below_limit"):
        assert g[k] == o[k], k
