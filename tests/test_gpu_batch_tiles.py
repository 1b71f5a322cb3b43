"""Work items of batches: detectors narrower than a round of tile stripes (whose
tiles follow each other without padding), of exactly one and of more, rows that
end in every part of a stripe, one reconstruction and many.  Bit for bit against
the same iterations one reconstruction at a time."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (nu, nv): 512 columns are one round of the row-by-row walks' stripes
DETECTORS = [(7, 70), (65, 33), (200, 17), (511, 9), (512, 21), (513, 5), (700, 16), (130, 1), (33, 129)]


@pytest.mark.parametrize("mode", ["R", "A"])
@pytest.mark.parametrize("picks", [[0], [8], list(range(9)), [4, 0, 7, 4, 2]])
def test_batch_equals_single(mode, picks):
    import torch

    import kevernals_amd as K
    from kevernals_amd import geometry as G

    mode = {"R": K.MODE_R, "A": K.MODE_A}[mode]
    gs = [G.arc_geometry((40 + 9 * i, 30 - i, 5 + i), (0.5, 0.5, 1.0), DETECTORS[i], (0.4, 0.4), 2 + i % 3, 6.0,
                         det_shift=(0.05, 0.03)) for i in picks]
    rng = np.random.Generator(np.random.PCG64(23))
    data = [rng.random(g.proj_shape, dtype=np.float32) + np.float32(0.2) for g in gs]
    iters = [1 + i % 2 for i in range(len(gs))]
    b = K.Batch(gs, mode=mode)
    for i, g in enumerate(gs):
        b.set_volume(i, np.ones(g.vol_shape, np.float32))
        b.set_data(i, data[i])
    b.mlem(iters)
    for i, (g, n) in enumerate(zip(gs, iters)):
        ctx = K.Context(0, g)
        x, d = torch.ones(g.vol_shape, device="cuda"), torch.from_numpy(data[i]).cuda()
        for _ in range(n):
            ctx.mlem_iteration(x, d, 1.0, mode)
        np.testing.assert_array_equal(b.get_volume(i), x.cpu().numpy())
