"""Prompt-chunk attention on the matrix cores (kmoe_attn_rows.hip) against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _run(ctx, q, kc, vc, nh, nkv, hd, pos0, n_ctx, pos_dev=None):
    import torch

    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    return ctx.attention(d(q), d(kc.view(np.int16)), d(vc.view(np.int16)), nh, nkv, hd, pos0, n_ctx,
                         pos_dev=pos_dev).cpu().numpy()


@pytest.fixture(scope="module")
def ctx():
    from kestrel_amd.kmoe import Context

    c = Context(0)
    yield c
    c.close()


# one row tile and its edges (16, 32, 33), ragged key blocks, fewer positions
# than a block, both wave counts (8 from 257 positions on a small grid), head
# dims, query groups, heads that do not divide the XCDs
@pytest.mark.parametrize("nh,nkv,hd,S,pos0", [(4, 4, 128, 16, 0), (4, 1, 64, 16, 3), (3, 1, 128, 32, 0),
                                              (8, 2, 64, 33, 31), (2, 2, 128, 31, 226), (2, 1, 128, 40, 230),
                                              (6, 2, 64, 70, 500), (32, 4, 64, 300, 9), (16, 16, 128, 530, 17)])
def test_rows_match_oracle(ctx, nh, nkv, hd, S, pos0):
    import torch
    from oracle import pyoracle as orc

    rng = np.random.default_rng(nh + S + pos0)
    n_ctx = pos0 + S  # the cache ends with the last row's position
    kc = orc.f16_store(rng.standard_normal((n_ctx, nkv * hd)) * 2)
    vc = orc.f16_store(rng.standard_normal((n_ctx, nkv * hd)))
    q = rng.standard_normal((S, nh * hd)).astype(np.float32)
    q *= np.exp2(rng.integers(-20, 3, size=(S, 1))).astype(np.float32)  # rows of very different size
    ref = orc.attention(q, kc, vc, nh, nkv, hd, pos0)
    got = _run(ctx, q, kc, vc, nh, nkv, hd, pos0, n_ctx)
    # the bound of the other attention kernels: f32 scores and sums in another order
    assert np.abs(got - ref).max() <= 1e-5 * max(1.0, np.abs(ref).max())
    pos = torch.tensor([pos0], dtype=torch.int32).cuda()
    assert np.array_equal(got, _run(ctx, q, kc, vc, nh, nkv, hd, 0, n_ctx, pos_dev=pos))


def test_values_that_are_not_finite_stay_in_the_rows_that_see_them(ctx):
    """A cached V of inf or NaN (f16 overflow) reaches the rows at and after its
    position, in its own head dim, and no earlier row of the same tile; huge q
    rows give NaN where the oracle does."""
    from oracle import pyoracle as orc

    rng = np.random.default_rng(3)
    nh, nkv, hd, S, pos0 = 4, 2, 128, 75, 20
    n = pos0 + S
    kc = orc.f16_store(rng.standard_normal((n, nkv * hd)))
    v = rng.standard_normal((n, nkv * hd)).astype(np.float32)
    v[45, 7] = np.inf
    v[46, 7 + hd] = -np.inf
    v[70, 100] = np.nan
    v[94, 3] = np.inf
    vc = v.astype(np.float16).view(np.uint16)
    q = rng.standard_normal((S, nh * hd)).astype(np.float32)
    q[30, :hd] = np.inf
    with np.errstate(all="ignore"):
        ref = orc.attention(q, kc, vc, nh, nkv, hd, pos0)
    got = _run(ctx, q, kc, vc, nh, nkv, hd, pos0, n)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(np.isposinf(got), np.isposinf(ref)) and np.array_equal(np.isneginf(got), np.isneginf(ref))
    f = np.isfinite(ref)
    assert np.isinf(ref).any() and f.mean() > 0.9 and np.abs(got[f] - ref[f]).max() <= 1e-5 * max(1.0, np.abs(ref[f]).max())


# the cache ends inside a key block (1, 5 and 31 rows of the last one), more
# rows behind it in the same allocation: zeros there or NaN, the same bits
@pytest.mark.parametrize("nh,nkv,hd,S,pos0", [(4, 2, 128, 33, 0), (4, 2, 64, 20, 17), (2, 2, 128, 70, 281)])
def test_nothing_past_the_last_position_is_read(ctx, nh, nkv, hd, S, pos0):
    from oracle import pyoracle as orc

    rng = np.random.default_rng(S)
    n = pos0 + S
    kc, vc = (orc.f16_store(rng.standard_normal((n, nkv * hd))) for _ in range(2))
    q = rng.standard_normal((S, nh * hd)).astype(np.float32)
    got = [_run(ctx, q, np.concatenate([kc, t]), np.concatenate([vc, t]), nh, nkv, hd, pos0, n)
           for t in (np.zeros((64, nkv * hd), np.uint16), np.full((64, nkv * hd), 0x7E00, np.uint16))]
    assert np.array_equal(*(g.view(np.uint32) for g in got))
    ref = orc.attention(q, kc, vc, nh, nkv, hd, pos0)
    assert np.abs(got[1] - ref).max() <= 1e-5 * max(1.0, np.abs(ref).max())


# bits far below a row's largest: a first position that takes all but e^-20 of
# the weight and has a zero value, and a q element 2^24 above the others whose
# K is zero; what is left keeps f32's bits
@pytest.mark.parametrize("kind,hd", [("sink", 128), ("sink", 64), ("outlier", 128), ("outlier", 64)])
def test_small_weights_and_elements_keep_their_bits(ctx, kind, hd):
    rng = np.random.default_rng(hd)
    nh, nkv, S, pos0 = 4, 2, 70, 90
    n = pos0 + S
    q = rng.standard_normal((S, nh, hd)).astype(np.float32)
    k, v = (rng.standard_normal((n, nkv, hd)).astype(np.float16) for _ in range(2))
    if kind == "sink":
        q[:, :, 0] = 8.0
        k[:, :, 0] = 0.0
        k[0] = 0.0
        k[0, :, 0] = 20 * np.sqrt(hd) / 8.0
        v[0] = 0.0
    else:
        q[:, :, 3] = 2.0 ** 24
        k[:, :, 3] = 0.0
    got = _run(ctx, q.reshape(S, -1), k.view(np.uint16).reshape(n, -1), v.view(np.uint16).reshape(n, -1), nh, nkv, hd,
               pos0, n).reshape(S, nh, hd)
    for s in range(S):
        for h in range(nh):
            sc = k[:pos0 + s + 1, h // 2].astype(np.float64) @ q[s, h].astype(np.float64) / np.sqrt(hd)
            e = np.exp(sc - sc.max())
            ref = e @ v[:pos0 + s + 1, h // 2].astype(np.float64) / e.sum()
            # an f32 score is off by up to |score| 2^-23, and as much of its weight (20 at the sink)
            assert np.linalg.norm(got[s, h] - ref) <= (3e-6 if kind == "sink" else 1.5e-6) * np.linalg.norm(ref)


# a row's bits are the same for a position on the host or on the device, however
# much longer than the call's positions the cache is (either side of 256)
@pytest.mark.parametrize("nh,nkv,hd,S,pos0", [(4, 2, 128, 40, 100), (2, 2, 64, 33, 223), (4, 2, 128, 20, 400)])
def test_bits_do_not_depend_on_the_cache_length(ctx, nh, nkv, hd, S, pos0):
    import torch
    from oracle import pyoracle as orc

    rng = np.random.default_rng(S)
    kc, vc = (orc.f16_store(rng.standard_normal((2000, nkv * hd))) for _ in range(2))
    q = rng.standard_normal((S, nh * hd)).astype(np.float32)
    pos = torch.tensor([pos0], dtype=torch.int32).cuda()
    got = [_run(ctx, q, kc, vc, nh, nkv, hd, p, n, pos_dev=pd) for p, pd in ((pos0, None), (0, pos))
           for n in (pos0 + S, 2000)]
    assert all(np.array_equal(g.view(np.uint32), got[0].view(np.uint32)) for g in got)
    ref = orc.attention(q, kc, vc, nh, nkv, hd, pos0)
    assert np.abs(got[0] - ref).max() <= 1e-5 * max(1.0, np.abs(ref).max())
