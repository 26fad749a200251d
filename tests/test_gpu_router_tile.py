"""Router logits in register tiles (kmoe_route.hip): the reference's bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# 2 x 2 and 4 x 4 tiles; rows that leave 0, 1 and 2 of a 48-row tile in
# dot_f32 order (128: two, 100: one, 96: none), ragged row and token tiles,
# 0 to 3 tokens in dot_f32 order, one and several column chunks
@pytest.mark.parametrize("E,d,S", [(33, 256, 261), (96, 512, 131), (100, 768, 130), (17, 2048, 395),
                                   (128, 512, 803), (100, 256, 801), (500, 256, 207), (60, 1024, 1606)])
def test_batch_logits_bit_exact(E, d, S):
    import torch
    from kestrel_amd.kmoe import F32, Context
    from oracle import pyoracle as orc

    w = orc.normal(E, E * d).reshape(E, d)
    x = orc.normal(S, S * d).reshape(S, d)
    x[3, 5], x[S - 1, 0], w[E - 1, 7] = np.inf, np.nan, -np.inf
    c = Context(0)
    got = c.matmul(F32, torch.from_numpy(w).cuda(), E, d, torch.from_numpy(x).cuda()).cpu().numpy()
    c.close()
    ref = orc.matmul(F32, w.view(np.uint8).ravel(), E, d, x)
    ok = ~np.isnan(ref)
    assert np.array_equal(np.isnan(got), ~ok)
    assert np.array_equal(got[ok].view(np.uint32), ref[ok].view(np.uint32))
