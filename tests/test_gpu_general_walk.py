"""Forward walks of contexts without segment lists (too large, or no memory for
them): voxel by voxel in tiles, several volumes interleaved, batches in every
tile layout.  The lists are given up as a context short of memory does; the
passes before and after must agree bit for bit, on geometries whose rows have
one pixel, fill no tile, or are cut by the volume's faces."""
import ctypes

import numpy as np
import pytest

from test_gpu_rows import CASES, CASES_R, arc

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

NAMES = sorted(CASES) + ["wide", "offset", "slices1", "coarse_hit"]
# pixels of several voxels, in views that all meet the volume
COARSE = ((150, 60, 12), (0.2, 0.4, 2.0), (130, 50), (0.9, 0.7), 4, 3.0)


@pytest.fixture(scope="module")
def K():
    import kevernals_amd

    assert torch.cuda.is_available(), "GPU tests need a GPU"
    return kevernals_amd


def drop_lists(obj):
    name = "_Z28kv_internal_batch_drop_listsP8kv_batch" if hasattr(obj, "mlem") else \
        "_Z22kv_internal_drop_listsP10kv_context"
    fn = getattr(obj.lib, name)
    fn.argtypes = [ctypes.c_void_p]
    assert fn(obj.handle) == 0


def geometry(name):
    if name == "coarse_hit":
        return arc(*COARSE)
    return (CASES.get(name) or CASES_R[name])()


def random(shape, seed, low=0.1):
    return np.random.Generator(np.random.PCG64(seed)).random(shape, dtype=np.float32) + np.float32(low)


@pytest.mark.parametrize("name", NAMES)
def test_passes_without_lists(K, name):
    print("case", name, flush=True)
    g = geometry(name)
    ctx = K.Context(0, g)
    vols = [torch.from_numpy(random(g.vol_shape, s)).cuda() for s in (1, 2, 3)]
    data = torch.from_numpy(random(g.proj_shape, 4, 0.5)).cuda()

    def passes():
        out = []
        for mode in (K.MODE_R, K.MODE_A):
            fp = torch.full(g.proj_shape, float("nan"), device="cuda")
            ctx.forward_project(vols[0], fp, mode)
            x = vols[1].clone()
            ctx.mlem_iteration(x, data, 0.9, mode)
            out += [fp.cpu().numpy(), x.cpu().numpy()]
        x = vols[1].clone()
        ctx.sart_iteration(x, data, 0.5)
        return out + [x.cpu().numpy()], [ctx.log_likelihoods(data, vols[:n]) for n in (1, 2, 3)]

    arrays, ll = passes()
    assert ll[2][:2] == ll[1] and ll[1][:1] == ll[0]
    drop_lists(ctx)
    plain, ll_plain = passes()
    for a, b in zip(arrays, plain):
        np.testing.assert_array_equal(a, b)
    assert ll_plain == ll


@pytest.mark.parametrize("name", ["faces", "wide", "offset", "coarse_hit"])
def test_mode_r_infinities_and_nan_reach_the_oracles_rays(K, name):
    """A ray's value is INF or NaN where the reference's is, and all others
    keep their bits: voxels taken with weight zero, or read and rejected, leave
    the sums alone.  Row by row and without lists."""
    from oracle.oracle import Oracle

    g = geometry(name)
    vol = random(g.vol_shape, 6)
    rng = np.random.Generator(np.random.PCG64(7))
    for value in (np.inf, -np.inf, np.nan):
        vol.ravel()[rng.integers(0, vol.size, 30)] = value
    ref = Oracle(g).fp_r(vol)
    assert 0 < np.count_nonzero(~np.isfinite(ref)) < ref.size // 2
    ctx = K.Context(0, g)
    for _ in range(2):
        out = torch.empty(g.proj_shape, device="cuda")
        ctx.forward_project(torch.from_numpy(vol).cuda(), out, K.MODE_R)
        np.testing.assert_array_equal(out.cpu().numpy(), ref)
        drop_lists(ctx)


@pytest.mark.parametrize("layout", [1, 2, 4, 8])
@pytest.mark.parametrize("mode", ["R", "A"])
def test_batches_without_lists(K, mode, layout):
    """One detector column, less and more than a tile, wide cones."""
    mode = {"R": K.MODE_R, "A": K.MODE_A}[mode]
    gs = [geometry(n) for n in ("nu65", "faces", "nu1", "coarse_hit", "cone")]
    iters = [2, 1, 2, 1, 2]
    data = [random(g.proj_shape, 20 + i, 0.2) for i, g in enumerate(gs)]
    b = K.Batch(gs, mode=mode)
    for i, g in enumerate(gs):
        b.set_tiles(i, layout, 8 if i % 2 else 4)
        b.set_data(i, data[i])

    def run(graph):
        for i, g in enumerate(gs):
            b.set_volume(i, np.ones(g.vol_shape, np.float32))
        b.mlem(iters, use_graph=graph)
        return [b.get_volume(i) for i in range(len(gs))]

    want = run(True)
    drop_lists(b)
    for graph in (False, True, True):
        for got, ref in zip(run(graph), want):
            np.testing.assert_array_equal(got, ref)
