"""Backprojections in which many bricks lie beside the detector rows of some or
all views: volumes taller than the detector's view of them, more views than one
test of them covers, detectors off to one side, no view that meets the volume,
sources inside the volume (whose bricks are never left out).  Against the
oracle as in test_gpu_bp_rows: mode R bit for bit; mode A with one rounding per
term on either side, and terms of a rounding of alpha that a side may leave
out."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# vol, spacing, det, pitch, views, arc, det_shift
CASES = {
    "short": ((40, 90, 24), (0.5, 0.5, 2.5), (70, 30), (0.5, 0.5), 9, 25.0, (0.0, 0.0)),
    "one_row": ((33, 50, 9), (0.5, 0.5, 2.5), (60, 1), (0.5, 0.5), 7, 20.0, (0.13, 0.07)),
    "views_64": ((20, 40, 9), (0.5, 0.5, 2.0), (40, 20), (0.5, 0.5), 64, 40.0, (0.0, 0.0)),
    "views_65": ((20, 40, 9), (0.5, 0.5, 2.0), (40, 20), (0.5, 0.5), 65, 40.0, (0.0, 0.0)),
    "views_131": ((20, 40, 9), (0.5, 0.5, 2.0), (40, 20), (0.5, 0.5), 131, 60.0, (0.0, 0.0)),
    "above": ((66, 61, 18), (0.5, 0.5, 2.0), (120, 60), (0.5, 0.5), 5, 15.0, (1.3, 27.0)),
    "below": ((66, 61, 18), (0.5, 0.5, 2.0), (120, 60), (0.5, 0.5), 5, 15.0, (1.3, -27.0)),
    "none": ((66, 61, 18), (0.5, 0.5, 2.0), (120, 60), (0.5, 0.5), 5, 15.0, (0.0, 300.0)),
    "wide": ((300, 46, 33), (0.25, 0.25, 1.9), (560, 70), (0.26, 0.26), 13, 24.0, (0.0, 0.0)),
}


def geometry(name):
    from kevernals_amd import geometry as G

    *args, shift = CASES[name]
    return G.arc_geometry(*args, det_shift=shift)


def beside(g):
    """Share of (view, voxel row, slice) whose centre's shadow misses the
    detector's rows by more than the row's own height."""
    y = (np.arange(g.ny) + 0.5 - g.ny / 2) * g.sy
    z = (np.arange(g.nz) + 0.5 - g.nz / 2) * g.sz
    out = []
    for p in range(g.nviews):
        t = (g.det[p, 2] - g.src[p, 2]) / (z - g.src[p, 2])
        v = (g.src[p, 1] + t[:, None] * (y - g.src[p, 1])[None, :] - g.det[p, 1]) / g.pv
        out.append(((v < -8) | (v > g.nv + 8)).mean())
    return float(np.mean(out))


@pytest.mark.parametrize("name", sorted(CASES))
def test_both_modes_against_the_oracle(name):
    import torch

    import kevernals_amd as K
    from oracle.oracle import Oracle

    print("case", name, flush=True)
    g = geometry(name)
    assert beside(g) > 0.2
    rng = np.random.Generator(np.random.PCG64(29))
    proj = rng.random(g.proj_shape, dtype=np.float32) + np.float32(0.5)
    d = torch.from_numpy(proj).cuda()
    o, ctx = Oracle(g), K.Context(0, g)
    out = torch.full(g.vol_shape, float("nan"), device="cuda")
    ctx.back_project(d, out, K.MODE_R)
    ref = o.bp_r(proj)
    assert (ref.max() > 0) == (name != "none")
    np.testing.assert_array_equal(out.cpu().numpy(), ref)
    ctx.back_project(d, out, K.MODE_A)
    length = np.linalg.norm(g.det - g.src, axis=1).max() + g.nu * g.pu + g.nv * g.pv
    np.testing.assert_allclose(out.cpu().numpy(), o.bp_a(proj), rtol=2 * (g.nviews * 16 * 16 + 3) * 2.0**-24,
                               atol=4 * 2.0**-24 * length * 1.5)


def test_sources_inside_the_volume():
    """Planes behind the source cast no shadow: every row counts there."""
    import torch

    import kevernals_amd as K
    from kevernals_amd import geometry as G
    from oracle.oracle import Oracle

    g = G.arc_geometry((30, 90, 30), (1.0, 1.0, 2.0), (60, 33), (1.0, 1.0), 3, 40.0, sod=20.0, sid=60.0)
    proj = np.random.Generator(np.random.PCG64(31)).random(g.proj_shape, dtype=np.float32)
    out = torch.empty(g.vol_shape, device="cuda")
    K.Context(0, g).back_project(torch.from_numpy(proj).cuda(), out, K.MODE_R)
    np.testing.assert_array_equal(out.cpu().numpy(), Oracle(g).bp_r(proj))


@pytest.mark.parametrize("mode", ["R", "A"])
def test_batches_equal_single(mode):
    import torch

    import kevernals_amd as K

    mode = {"R": K.MODE_R, "A": K.MODE_A}[mode]
    gs = [geometry(n) for n in ("short", "views_65", "none", "above")]
    data = [np.random.Generator(np.random.PCG64(37 + i)).random(g.proj_shape, dtype=np.float32) + np.float32(0.2)
            for i, g in enumerate(gs)]
    b = K.Batch(gs, mode=mode)
    for i, g in enumerate(gs):
        b.set_volume(i, np.ones(g.vol_shape, np.float32))
        b.set_data(i, data[i])
    b.mlem(2)
    for i, g in enumerate(gs):
        ctx = K.Context(0, g)
        x, d = torch.ones(g.vol_shape, device="cuda"), torch.from_numpy(data[i]).cuda()
        for _ in range(2):
            ctx.mlem_iteration(x, d, 1.0, mode)
        np.testing.assert_array_equal(b.get_volume(i), x.cpu().numpy())
