"""Shift-and-add at every chunk size the kernel is built for, against the
oracle, bit for bit: shift spreads that fit 32 or 64 staged rows with 8, 4, 2
planes a chunk, and none; detector sizes that fill no tile; a last chunk that
is not full; planes in any order."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("noalloc", [False, True])
@pytest.mark.parametrize("step", [0.3, 2.0, 6.0, 14.0, 30.0, 90.0, 400.0])
def test_chunk_sizes(step, noalloc):
    """`step`: rows of the largest shift between neighbouring planes."""
    import torch

    import kevernals_amd as K
    from kevernals_amd import geometry as G
    from oracle import oracle as O

    g = G.arc_geometry((16, 16, 8), (1.0, 1.0, 1.0), (67, 133), (0.5, 0.5), 5, 20.0)
    sid = 1000.0
    planes = np.arange(-5, 6, dtype=np.float32)  # 11: no multiple of a chunk
    if step > 10:
        planes = planes[np.random.Generator(np.random.PCG64(2)).permutation(11)]
    src_y = g.src[:, 1]
    dy = float(np.abs(src_y).max()) * 1.0 / sid / step  # shift of a 1 mm step is about `step` rows
    rng = np.random.Generator(np.random.PCG64(5))
    proj = rng.standard_normal(g.proj_shape).astype(np.float32)
    ctx = K.Context(0, g)
    out = torch.full((len(planes), g.nv, g.nu), np.nan, device="cuda")
    ctx.shift_and_add(torch.from_numpy(proj).cuda(), out, src_y, planes, sid, 0.0, dy, noalloc=noalloc)
    rc, ref = O.saa(proj, src_y, planes, sid, 0.0, dy)
    assert rc == 0
    np.testing.assert_array_equal(out.cpu().numpy(), ref)
