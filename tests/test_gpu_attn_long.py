"""Long rows of the chunked attention kernels: the cross-work-group merge."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# chunk counts around the merge's batches of 16 loads and 64 lanes (16, 17, 63,
# 64, 65, 130 chunks), host and device positions, one row and a few, query
# groups, both head dims; each call twice (the counters are zero again)
@pytest.mark.parametrize("nh,nkv,hd,S,n", [(4, 4, 128, 1, 1024), (4, 1, 64, 1, 1025), (2, 2, 128, 1, 4032),
                                           (4, 2, 128, 1, 4096), (2, 1, 64, 3, 4097), (3, 3, 128, 2, 8311),
                                           (8, 2, 128, 5, 1990)])
def test_long_rows_match_oracle(nh, nkv, hd, S, n):
    import torch
    from kestrel_amd.kmoe import Context
    from oracle import pyoracle as orc

    rng = np.random.default_rng(n)
    kc = orc.f16_store(rng.standard_normal((n, nkv * hd)) * 2)
    vc = orc.f16_store(rng.standard_normal((n, nkv * hd)))
    q = rng.standard_normal((S, nh * hd)).astype(np.float32)
    ref = orc.attention(q, kc, vc, nh, nkv, hd, n - S)
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    kd, vd, qd = d(kc.view(np.int16)), d(vc.view(np.int16)), d(q)
    pos = torch.tensor([n - S], dtype=torch.int32).cuda()
    ctx = Context(0)
    got = [ctx.attention(qd, kd, vd, nh, nkv, hd, n - S, n).cpu().numpy() for _ in range(2)]
    got += [ctx.attention(qd, kd, vd, nh, nkv, hd, 0, n, pos_dev=pos).cpu().numpy() for _ in range(2)]
    ctx.close()
    assert all(np.array_equal(g, got[0]) for g in got)
    # the bound of the other attention kernels: f32 scores and sums in another order
    assert np.abs(got[0] - ref).max() <= 1e-5 * max(1.0, np.abs(ref).max())
