"""Row-by-row forward walks against the voxel-by-voxel ones.

Mode R is compared with the oracle, the reference's own sequence of operations.
In mode A the row-by-row walks follow a detector row's segment lists; kv_trace_rays
records the voxels and weights of the general walk of single rays.  The
projection is defined by those: FP32 products added in walk order, so a
row-by-row projection must give the same bits.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def arc(vol, sp, det, pitch, views, arc_deg, **kw):
    from kevernals_amd import geometry as G

    return G.arc_geometry(vol, sp, det, pitch, views, arc_deg, **kw)


CASES = {
    # one column; a wavefront's 64 and its neighbours
    "nu1": lambda: arc((40, 33, 9), (0.5, 0.5, 2.0), (1, 37), (0.6, 0.6), 3, 15.0),
    "nu63": lambda: arc((40, 33, 9), (0.5, 0.5, 2.0), (63, 37), (0.5, 0.6), 3, 15.0),
    "nu64": lambda: arc((40, 33, 9), (0.5, 0.5, 2.0), (64, 5), (0.5, 0.6), 3, 15.0),
    "nu65": lambda: arc((40, 33, 9), (0.5, 0.5, 2.0), (65, 1), (0.5, 0.6), 3, 15.0),
    # odd sizes: the middle column's and row's rays run along the x and y planes
    "axis": lambda: arc((31, 30, 7), (0.5, 0.5, 2.0), (131, 65), (0.25, 0.5), 3, 0.0),
    # the volume entered and left through its x faces, the detector shifted
    "faces": lambda: arc((24, 90, 60), (0.5, 0.5, 2.0), (200, 90), (0.6, 0.9), 5, 20.0, det_shift=(17.3, -9.1)),
    # several x planes per segment (thin in x, thick slices)
    "thin_x": lambda: arc((300, 40, 6), (0.05, 0.5, 9.0), (140, 40), (0.2, 0.8), 3, 12.0),
    # pixels of a voxel and more: rays too far apart for one load per row
    "coarse": lambda: arc((150, 60, 12), (0.2, 0.4, 2.0), (130, 50), (0.9, 0.7), 4, 18.0),
    # steep in y, one slice, one view
    "slice": lambda: arc((70, 80, 1), (0.3, 0.3, 3.0), (97, 120), (0.4, 0.4), 1, 0.0),
    # source close to the volume: wide cone
    "cone": lambda: arc((96, 96, 40), (0.5, 0.5, 1.0), (160, 160), (1.1, 1.1), 3, 30.0, sod=60.0, sid=120.0),
    # source inside the volume
    "inside": lambda: arc((50, 40, 30), (1.0, 1.0, 2.0), (90, 33), (1.0, 1.0), 2, 10.0, sod=20.0, sid=60.0),
}


def rays_of(g, count, seed=1):
    rng = np.random.Generator(np.random.PCG64(seed))
    n = g.nrays
    ids = rng.integers(0, n, size=count)
    mid = (g.nv // 2) * g.nu + np.arange(min(g.nu, 140))  # a whole row, every lane of its wavefronts
    return np.unique(np.concatenate([ids, mid, [0, n - 1]])).astype(np.int32)


def lengths(g, rays):
    """Source-to-pixel lengths in the projector's FP32 operations."""
    f = np.float32
    p, v, u = rays // (g.nu * g.nv), rays // g.nu % g.nv, rays % g.nu
    sp = [f(g.sx), f(g.sy), f(g.sz)]
    q = [(g.det[p, 0] + (u.astype(f) + f(0.5)) * f(g.pu)) / sp[0],
         (g.det[p, 1] + (v.astype(f) + f(0.5)) * f(g.pv)) / sp[1], g.det[p, 2] / sp[2]]
    d = [(q[k] - g.src[p, k] / sp[k]) * sp[k] for k in range(3)]
    return np.sqrt((d[0] * d[0] + d[1] * d[1]) + d[2] * d[2])


@pytest.mark.parametrize("name", sorted(CASES))
def test_mode_a_rows_equal_the_voxel_walk(name):
    import torch

    import kevernals_amd as K

    print("case", name, flush=True)
    g = CASES[name]()
    ctx = K.Context(0, g)
    rng = np.random.Generator(np.random.PCG64(7))
    vols = [rng.random(g.vol_shape, dtype=np.float32) + np.float32(0.1) for _ in range(3)]
    dev = [torch.from_numpy(v).cuda() for v in vols]
    out = torch.empty(g.proj_shape, device="cuda")
    ctx.forward_project(dev[0], out, K.MODE_A)
    got = out.cpu().numpy().ravel()
    rays = rays_of(g, 200)
    L = lengths(g, rays)
    for (idx, w, n), r, ln in zip(ctx.trace_rays(rays, cap=2048, mode=K.MODE_A), rays, L):
        prod = np.concatenate([np.zeros(1, np.float32), w * vols[0].ravel()[idx]]).astype(np.float32)
        assert got[r] == ln * np.add.accumulate(prod, dtype=np.float32)[-1], (name, int(r), n)
    # several volumes in one walk: the same projections, hence the same sums
    data = torch.rand(g.proj_shape, device="cuda") + 0.5
    assert ctx.log_likelihoods(data, dev) == [ctx.log_likelihood(data, v) for v in dev]


def test_mode_a_rows_touch_only_their_voxels():
    """INF and NaN reach exactly the rays that pass through their voxel: a
    voxel read with weight zero leaves a sum as it was."""
    import torch

    import kevernals_amd as K

    g = CASES["faces"]()
    ctx = K.Context(0, g)
    vol = np.full(g.vol_shape, 0.5, np.float32)
    clean, out = (torch.empty(g.proj_shape, device="cuda") for _ in range(2))
    ctx.forward_project(torch.from_numpy(vol).cuda(), clean, K.MODE_A)
    bad = {(30, 41, 0): np.inf, (20, 50, 23): np.nan, (59, 89, 12): -np.inf, (0, 0, 11): np.nan}
    for at, x in bad.items():
        vol[at] = x
    ctx.forward_project(torch.from_numpy(vol).cuda(), out, K.MODE_A)
    got, clean = out.cpu().numpy().ravel(), clean.cpu().numpy().ravel()
    hit = np.array([np.ravel_multi_index(at, g.vol_shape) for at in bad])
    rays = np.unique(np.concatenate([rays_of(g, 4000), np.nonzero(~np.isfinite(got))[0][:500].astype(np.int32)]))
    for (idx, _, _), r in zip(ctx.trace_rays(rays, cap=1024, mode=K.MODE_A), rays):
        if np.isin(idx, hit).any():
            assert not np.isfinite(got[r])
        else:
            assert got[r] == clean[r]


CASES_R = {
    # rays in the middle columns, the volume's x faces, several views
    "wide": lambda: arc((200, 90, 20), (0.3, 0.3, 1.0), (330, 150), (0.28, 0.3), 5, 20.0),
    # plane positions that FP32 rounds: odd sizes, sources off the grid
    "offset": lambda: shifted(arc((167, 71, 13), (0.37, 0.41, 1.3), (215, 117), (0.43, 0.41), 4, 17.0)),
    # one or two slices: no z entries left in the run, or no filler
    "slices1": lambda: arc((90, 60, 1), (0.4, 0.4, 2.0), (140, 90), (0.4, 0.5), 3, 10.0),
    "slices2": lambda: arc((90, 60, 2), (0.4, 0.4, 2.0), (140, 90), (0.4, 0.5), 3, 10.0),
    "slices3": lambda: arc((90, 60, 3), (0.4, 0.4, 2.0), (140, 90), (0.4, 0.5), 3, 10.0),
    # longer runs: more rounding in the run values
    "tall": lambda: arc((140, 400, 64), (0.15, 0.15, 1.0), (260, 300), (0.14, 0.3), 3, 20.0),
}


def shifted(g):
    src = g.src.copy()
    src[:, 0] += np.float32(3.137)
    src[:, 1] -= np.float32(1.77)
    return g.scaled(src=src)


@pytest.mark.parametrize("name", sorted(CASES) + sorted(CASES_R))
def test_mode_r_rows_equal_the_oracle(name):
    """Ray sums bit for bit on a volume without equal neighbours, so that one
    voxel or weight taken differently shows."""
    import torch

    import kevernals_amd as K
    from oracle.oracle import Oracle

    print("case", name, flush=True)
    g = (CASES.get(name) or CASES_R[name])()
    rng = np.random.Generator(np.random.PCG64(11))
    vol = rng.random(g.vol_shape, dtype=np.float32) + np.float32(0.1)
    ctx = K.Context(0, g)
    out = torch.empty(g.proj_shape, device="cuda")
    ctx.forward_project(torch.from_numpy(vol).cuda(), out, K.MODE_R)
    np.testing.assert_array_equal(out.cpu().numpy(), Oracle(g).fp_r(vol))


@pytest.mark.parametrize("name", ["faces", "coarse"])
def test_mode_a_batch_rows_equal_single(name):
    """Batched iterations of reconstructions with segment lists, uneven."""
    import torch

    import kevernals_amd as K

    gs = [CASES[name](), CASES["nu65"](), CASES["cone"]()]
    rng = np.random.Generator(np.random.PCG64(3))
    data = [(rng.random(g.proj_shape, dtype=np.float32) + np.float32(0.2)) for g in gs]
    b = K.Batch(gs, mode=K.MODE_A)
    for i, g in enumerate(gs):
        b.set_volume(i, np.ones(g.vol_shape, np.float32))
        b.set_data(i, data[i])
    b.mlem([2, 1, 2], use_graph=True)
    for i, (g, n) in enumerate(zip(gs, (2, 1, 2))):
        ctx = K.Context(0, g)
        x, d = torch.ones(g.vol_shape, device="cuda"), torch.from_numpy(data[i]).cuda()
        for _ in range(n):
            ctx.mlem_iteration(x, d, 1.0, K.MODE_A)
        np.testing.assert_array_equal(b.get_volume(i), x.cpu().numpy())
