"""Backprojection bricks of their full depths, 8 slices in mode R and up to 16
in mode A, with shadows of three and four columns and up to eight rows under a
wide arc: the first and last plane of such a brick bound the columns of all the
slices between them.  Mode R must give the oracle's bits; mode A adds the same
terms in another order (test_gpu_bp_rows).  The depths are read from the
launches on a HIP runtime without a GPU."""
import numpy as np
import pytest

from test_segment_lists import run  # noqa: F401  (fixture)

# vol, spacing, det, pitch, views, arc; slices per brick in modes R and A
CASES = {
    "four_columns": (((700, 600, 32), (0.25, 0.25, 0.5), (1850, 900), (0.15, 0.3), 2, 20.0), 8, 16),
    "three_columns": (((520, 900, 24), (0.25, 0.25, 0.4), (1000, 1100), (0.2, 0.35), 2, 24.0), 8, 12),
    "eight_rows": (((640, 500, 48), (0.25, 0.25, 0.8), (1000, 1200), (0.27, 0.2), 2, 24.0), 8, 16),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_depths(run, name):  # noqa: F811
    args, zr, za = CASES[name]
    run("""
g = G.arc_geometry(*%r)
c = context(g)
for mode, zt in ((R, %d), (A, %d)):
    assert L.kv_back_project(c.handle, buf, buf, mode) == 0
    assert H.fake_grid_z() == -(-g.nz // zt), (mode, H.fake_grid_z())
""" % (args, zr, za))


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(CASES))
def test_both_modes_against_the_oracle(name):
    import torch

    import kevernals_amd as K
    from kevernals_amd import geometry as G
    from oracle.oracle import Oracle

    print("case", name, flush=True)
    g = G.arc_geometry(*CASES[name][0])
    rng = np.random.Generator(np.random.PCG64(41))
    proj = rng.random(g.proj_shape, dtype=np.float32) + np.float32(0.5)
    o, ctx = Oracle(g), K.Context(0, g)
    d, out = torch.from_numpy(proj).cuda(), torch.empty(g.vol_shape, device="cuda")
    ctx.back_project(d, out, K.MODE_R)
    np.testing.assert_array_equal(out.cpu().numpy(), o.bp_r(proj))
    ctx.back_project(d, out, K.MODE_A)
    length = np.linalg.norm(g.det - g.src, axis=1).max() + g.nu * g.pu + g.nv * g.pv
    np.testing.assert_allclose(out.cpu().numpy(), o.bp_a(proj), rtol=2 * (g.nviews * 16 * 16 + 3) * 2.0**-24,
                               atol=4 * 2.0**-24 * length * 1.5)
