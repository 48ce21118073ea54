"""The benchmark's byte accounting against the launches a call makes (CPU)."""
import pytest

import bench


@pytest.mark.parametrize("N,F,S,groups", [(64, 3, 42, 1), (128, 4, 44, 11), (192, 3, 48, 24), (512, 4, 44, 22)])
def test_kernel_bytes_add_up_to_the_path(N, F, S, groups):
    """Over the launches of one call (groups of radii, the unfiltered last step) the kernels' bytes are
    the path's but for what the path leaves out: the window tables, the spectra that the x pass of
    a group reads once instead of once per radius, and the state and crossings of the test."""
    steps = 3
    plane = N <= 128
    launches = {"r2c_z": 1, "colpass_y_fwd": 1, "colpass_x_fwd": 1, "window_table": 1, "ix_filter_k": groups,
                "ix_filter": 1, "colpass_y_inv": 1 if plane else groups + 1,
                "c2r_threshold": 1 if plane else groups + 1}
    if plane:
        launches.update(plane_threshold=groups, ladder_combine=groups)
    prof = {k: (1.0, n * steps) for k, n in launches.items()}
    radii = {k: bench.ladder_radii(k, S, prof, steps) for k in launches}
    for k in ("window_table", "ix_filter_k", "plane_threshold", "ladder_combine"):
        if k in launches:
            assert radii[k] * launches[k] == pytest.approx(S - 1)
    assert radii["c2r_threshold"] * launches["c2r_threshold"] == pytest.approx(1 if plane else S)
    assert radii["colpass_y_inv"] * launches["colpass_y_inv"] == pytest.approx(1 if plane else S)
    total = sum(n * bench.kernel_bytes(k, N, F, radii[k]) for k, n in launches.items())
    spec, Nr = 8 * N * N * (N // 2), N**3
    tables = (S - 1) * 4 * (N // 2 + 1) ** 3
    reads = (S - 1 - groups) * F * (spec + 8 * N * N)  # of the unfiltered spectra, once per group
    if plane:  # two passes over the state per group, crossings written and read, against the path's two per radius
        state = groups * 3 * Nr + (S - 1) * Nr + 2 * Nr
    else:
        state = (groups + 1) * 2 * Nr
    path = bench.path_bytes_hii(N, F, S) - S * 2 * Nr
    assert total == pytest.approx(path + tables - reads + state, rel=1e-12)
