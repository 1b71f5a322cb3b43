"""Voxel-driven backprojections at the edges of their row and column loops.

From one to thirteen detector rows and one to six columns per voxel, detectors
of fewer than one group of either, shadows cut by the detector's edges.  Both modes against the oracle: mode R has its order of
operations and must give its bits.  Mode A adds the oracle's own terms (the
same FP32 plane crossings) in another order, at most N of them a voxel, all
positive: N + 3 roundings of 2**-24 on either side, and terms of a single
rounding of alpha (2**-24 of the ray's length) that one side may leave out.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# rows x columns of a voxel's shadow: (vol, spacing, det, pitch, views, arc)
CASES = {
    "1x1": ((66, 19, 9), (0.3, 0.3, 0.5), (24, 12), (1.5, 1.5), 3, 1.0),
    "3x2": ((65, 21, 8), (0.4, 0.4, 1.0), (120, 80), (0.4, 0.25), 3, 1.0),
    "4x3": ((64, 18, 7), (0.5, 0.5, 1.0), (190, 100), (0.3, 0.22), 3, 1.0),
    "6x4": ((50, 14, 9), (0.5, 0.8, 1.0), (210, 110), (0.22, 0.22), 3, 1.0),
    "8x6": ((30, 12, 3), (0.9, 1.2, 1.0), (200, 120), (0.25, 0.24), 3, 1.0),
    "10x2": ((40, 10, 3), (0.4, 1.5, 1.0), (75, 120), (0.4, 0.24), 3, 1.0),
    "13x2": ((40, 10, 3), (0.4, 2.0, 1.0), (75, 160), (0.4, 0.24), 3, 1.0),
    "steep": ((40, 30, 4), (0.4, 0.3, 12.0), (75, 420), (0.4, 0.3), 3, 8.0),
    # fewer rows or columns than one group (SHIFT keeps them off the axis, whose
    # rays mode R takes for parallel to the planes)
    "nv1": ((70, 9, 5), (0.5, 0.5, 1.0), (160, 1), (0.5, 0.5), 2, 0.5),
    "nu1": ((9, 40, 5), (0.5, 0.5, 1.0), (1, 90), (0.5, 0.4), 2, 0.5),
    "nu2": ((9, 40, 5), (0.5, 0.5, 1.0), (2, 90), (0.5, 0.4), 2, 0.5),
    "nu3": ((9, 40, 5), (0.5, 0.5, 1.0), (3, 90), (0.2, 0.4), 2, 0.5),
    # the middle columns' and rows' rays run inside the x and y planes' gaps
    # (crossings at -INF and +INF in mode A), several columns per voxel
    "axis": ((31, 30, 7), (0.5, 0.5, 2.0), (131, 65), (0.25, 0.25), 3, 0.0),
    "axis_wide": ((31, 31, 7), (0.5, 0.5, 2.0), (33, 33), (0.5, 0.5), 1, 0.0),
    # the first voxel's shadow begins left of the detector
    "left": ((40, 10, 3), (0.4, 1.5, 1.0), (60, 120), (0.4, 0.24), 3, 1.0),
    "left_far": ((40, 10, 9), (0.4, 1.5, 1.0), (57, 120), (0.4, 0.24), 3, 1.0),
    # mode A's deep bricks: a tall and a wide brick grid of more than one round
    "deep": ((333, 287, 33), (0.25, 0.25, 0.6), (400, 380), (0.35, 0.35), 2, 1.0),
    "deep_wide": ((450, 230, 37), (0.25, 0.25, 1.2), (500, 300), (0.4, 0.4), 2, 1.0),
    # detector smaller than the volume's shadow, and off to one side
    "cut": ((96, 64, 9), (0.5, 0.5, 1.0), (61, 37), (0.4, 0.4), 3, 1.5),
    "side": ((96, 64, 9), (0.5, 0.5, 1.0), (61, 37), (0.4, 0.4), 3, 1.5),
}


SHIFT = {"nv1": (0.13, 0.07), "nu1": (0.13, 0.07), "nu2": (0.13, 0.07), "nu3": (0.13, 0.07), "side": (21.3, -13.1)}


def geometry(name):
    from kevernals_amd import geometry as G

    return G.arc_geometry(*CASES[name], det_shift=SHIFT.get(name, (0.0, 0.0)))


@pytest.mark.parametrize("name", sorted(CASES))
def test_both_modes_against_the_oracle(name):
    import torch

    import kevernals_amd as K
    from oracle.oracle import Oracle

    print("case", name, flush=True)
    g = geometry(name)
    rng = np.random.Generator(np.random.PCG64(19))
    proj = rng.random(g.proj_shape, dtype=np.float32) + np.float32(0.5)
    o, ctx = Oracle(g), K.Context(0, g)
    out = torch.empty(g.vol_shape, device="cuda")
    ctx.back_project(torch.from_numpy(proj).cuda(), out, K.MODE_R)
    ref = o.bp_r(proj)
    assert ref.max() > 0
    np.testing.assert_array_equal(out.cpu().numpy(), ref)
    ctx.back_project(torch.from_numpy(proj).cuda(), out, K.MODE_A)
    got, ref = out.cpu().numpy(), o.bp_a(proj)
    terms = g.nviews * 16 * 16
    length = np.linalg.norm(g.det - g.src, axis=1).max() + g.nu * g.pu + g.nv * g.pv
    np.testing.assert_allclose(got, ref, rtol=2 * (terms + 3) * 2.0**-24, atol=4 * 2.0**-24 * length * 1.5)
