"""The f32 regime on the f16 matrix cores (kmoe_f16gemm.hip): many activation
rows against Q4_K, Q6_K and Q8_0 weights, plain and in expert layers."""
import numpy as np
import pytest

from helpers import Q4_K, Q6_K, Q8_0, LayerSpec, random_blocks, rel_l2

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from kestrel_amd.kmoe import Context

    c = Context(0)
    c.profile_enable(True)
    yield c
    c.close()


def _matmul(ctx, t, w, rows, cols, x):
    import torch

    n0 = ctx.profile_read("f16_gemm")[1]
    out = ctx.matmul(t, torch.from_numpy(w).cuda(), rows, cols, torch.from_numpy(x).cuda()).cpu().numpy()
    assert ctx.profile_read("f16_gemm")[1] == n0 + 1, "another kernel ran"
    return out


def _bound(t, w64, x, cols):
    """Largest error of the sum of products: the pieces (2^-23 of each x; 2^-17
    of 2^-24 of the row's largest is more than they leave of small ones) and one fp32 rounding per 8 products of partial sums
    no larger than sum |w x| (Q4_K: of the scale and the minimum term apart, at
    most 8 times that for these blocks: |d sc q| + |dmin m| <= 7 * max |w| of
    the sub-block, its rms at least max / 4)."""
    a = np.abs(x).astype(np.float64)
    s = a @ np.abs(w64).T + 2.0 ** -17 * a.max(1, keepdims=True) * np.abs(w64).sum(1)
    return (cols / 8 + 8) * 2.0 ** -24 * s * (8 if t == Q4_K else 1)


# edges of the row blocks (128, 256), of the 32-token tiles and 64-token blocks,
# rows that end inside a 128-column stage (Q8_0), one and several superblocks,
# one and two token tiles per work-group
@pytest.mark.parametrize("t,rows,cols,S", [(Q4_K, 16390, 256, 24), (Q4_K, 4100, 512, 97), (Q4_K, 33000, 768, 64),
                                           (Q4_K, 1500, 2048, 513), (Q8_0, 3000, 64, 31), (Q8_0, 2817, 1344, 33),
                                           (Q8_0, 40001, 192, 65), (Q6_K, 22501, 256, 4), (Q6_K, 700, 768, 130),
                                           (Q6_K, 33001, 512, 95)])
def test_plain_rows(ctx, t, rows, cols, S):
    from oracle import pyoracle as orc

    w = random_blocks(t, rows, cols, seed=rows + cols)
    rng = np.random.default_rng(S)
    x = rng.standard_normal((S, cols)).astype(np.float32)
    x *= np.exp2(rng.integers(-60, 60, size=(S, 1))).astype(np.float32)  # rows of very different size
    x[1] = 0.0
    x[2, 3::7] *= np.float32(2.0 ** -20)  # and small elements beside large ones
    w64 = orc.dequant(t, w, rows * cols).reshape(rows, cols).astype(np.float64)
    ref = x.astype(np.float64) @ w64.T
    got = _matmul(ctx, t, w, rows, cols, x)
    assert np.all(np.abs(got - ref) <= _bound(t, w64, x, cols) + 1e-45)
    n = np.linalg.norm(ref, axis=1)
    assert np.all(np.linalg.norm(got - ref, axis=1) <= 1e-6 * n)


# an element 2^24 above the others whose weights are all zero: what is left of
# the sums keeps f32's bits (one and two token tiles; Q4_K's minimum term)
@pytest.mark.parametrize("t,S", [(Q4_K, 70), (Q4_K, 1100), (Q6_K, 70), (Q8_0, 70), (Q8_0, 1100)])
def test_small_elements_beside_a_large_one_keep_their_bits(ctx, t, S):
    from oracle import pyoracle as orc

    rows, cols = 8192, 512
    w = random_blocks(t, rows, cols, seed=9)
    b = w.reshape(rows, -1)
    if t == Q8_0:
        b[:, 2 + 7] = 0
    elif t == Q4_K:  # the first sub-block's minimum and the element's nibble
        b[:, 4 + 4] &= 0xC0
        b[:, 16 + 7] &= 0xF0
    else:  # q = 32
        b[:, 7] &= 0xF0
        b[:, 128 + 7] = (b[:, 128 + 7] & 0xFC) | 2
    x = np.random.default_rng(S).standard_normal((S, cols)).astype(np.float32)
    x[:, 7] = 2.0 ** 24
    w64 = orc.dequant(t, w, rows * cols).reshape(rows, cols).astype(np.float64)
    assert not w64[:, 7].any()
    ref = x[:, 8:].astype(np.float64) @ w64[:, 8:].T + x[:, :7].astype(np.float64) @ w64[:, :7].T
    got = _matmul(ctx, t, w, rows, cols, x)
    assert np.all(np.linalg.norm(got - ref, axis=1) <= 1e-6 * np.linalg.norm(ref, axis=1))


@pytest.mark.parametrize("t", [Q4_K, Q6_K, Q8_0])
def test_values_that_are_not_finite_stay_in_their_row(ctx, t):
    from oracle import pyoracle as orc

    rows, cols, S = 6000, 512, 70
    w = random_blocks(t, rows, cols, seed=3)
    rng = np.random.default_rng(4)
    x = rng.standard_normal((S, cols)).astype(np.float32)
    x[5, 100] = np.inf
    x[40, 3] = np.nan
    x[69, 500] = -np.inf
    x[7] *= np.float32(3e38 / np.abs(x[7]).max())  # the sums overflow
    got = _matmul(ctx, t, w, rows, cols, x)
    w64 = orc.dequant(t, w, rows * cols).reshape(rows, cols).astype(np.float64)
    fin = np.ones(S, bool)
    fin[[5, 40, 69, 7]] = False
    assert not np.isfinite(got[[5, 40, 69]]).any()
    assert rel_l2(got[fin], x[fin].astype(np.float64) @ w64.T) < 1e-6
    ref7 = (x[7].astype(np.float64) / 2.0 ** 20) @ w64.T
    over, under = np.abs(ref7) > 3.5e38 / 2.0 ** 20, np.abs(ref7) < 3.3e38 / 2.0 ** 20
    assert np.isinf(got[7][over]).all() and np.isfinite(got[7][under]).all()
    assert np.array_equal(np.sign(got[7][over]), np.sign(ref7[over]))


# ragged experts (Zipf: one of several hundred rows, some of none or below the
# f32 regime's 4), in both f32 regimes; gate/up and down of every type
@pytest.mark.parametrize("E,k,d,F,S,gt,dt,regime", [(9, 2, 512, 384, 701, Q4_K, Q8_0, 0),
                                                    (70, 3, 256, 512, 900, Q4_K, Q4_K, 2),
                                                    (6, 2, 256, 512, 1801, Q6_K, Q6_K, 0),
                                                    (5, 1, 512, 256, 1801, Q8_0, Q4_K, 0)])
def test_expert_layers(ctx, E, k, d, F, S, gt, dt, regime):
    import torch
    from oracle import pyoracle as orc

    spec = LayerSpec(E, k, d, F, gt, seed=E + S, down_type=dt, zipf=1.3)
    x = orc.normal(S, S * d).reshape(S, d) + np.float32(1.0)
    spec.upload(ctx, E)
    n0 = [ctx.profile_read(n)[1] for n in ("moe_gate_up_f16", "moe_down_f16")]
    ctx.set_regime(regime)
    try:
        out = ctx.moe_ffn(E, torch.from_numpy(x).cuda()).cpu().numpy()
    finally:
        ctx.set_regime(0)
    assert [ctx.profile_read(n)[1] for n in ("moe_gate_up_f16", "moe_down_f16")] == [n + 1 for n in n0]
    layer = spec.oracle_layer()
    idx = ctx.last_routing(S, k, E)[0].cpu().numpy().astype(np.uint32)
    assert np.array_equal(idx, layer.route(x)[0])
    cnt = np.bincount(idx.ravel(), minlength=E)
    ref = layer.moe_ffn(x, regime)
    big = cnt[idx].min(1) >= 4 if regime == 0 else np.ones(S, bool)  # tokens whose experts are all in the f32 regime
    assert big.sum() > S // 2
    assert rel_l2(out[big], ref[big]) < 3e-6
    assert rel_l2(out, ref) < 1e-3


def test_a_budget_without_room_for_the_pieces_keeps_the_other_kernels():
    import torch
    from kestrel_amd.kmoe import Context
    from oracle import pyoracle as orc

    rows, cols, S = 40000, 256, 600  # no partial sums: the pieces are the larger need
    w = random_blocks(Q4_K, rows, cols, seed=8)
    x = orc.normal(8, S * cols).reshape(S, cols)
    c = Context(0)
    c.profile_enable(True)
    wd, xd = torch.from_numpy(w).cuda(), torch.from_numpy(x).cuda()
    full = c.matmul(Q4_K, wd, rows, cols, xd).cpu().numpy()
    used = c.vram_usage()[0]
    c.close()
    c = Context(0)
    c.profile_enable(True)
    c.vram_set_limit(used - 1)
    tight = c.matmul(Q4_K, wd, rows, cols, xd).cpu().numpy()
    assert c.profile_read("f16_gemm")[1] == 0 and c.profile_read("f32_rows_plain")[1] == 1
    c.close()
    assert rel_l2(full, tight) < 2e-6


# the int8 regime's ragged experts: every weight type, the per-block integers
# of the kernels that ran (Q4_K, Q8_0), with blocks and activations at their
# extremes so that a stage's sums reach their largest
@pytest.mark.parametrize("E,k,d,F,S,gt,dt", [(70, 3, 256, 384, 401, Q4_K, Q8_0), (66, 2, 512, 256, 700, Q4_K, Q4_K),
                                             (5, 2, 256, 512, 90, Q6_K, Q6_K), (6, 1, 384, 256, 130, Q8_0, Q6_K)])
def test_int8_regime_expert_layers(ctx, E, k, d, F, S, gt, dt):
    import torch
    from oracle import pyoracle as orc

    spec = LayerSpec(E, k, d, F, gt, seed=E + S, down_type=dt, zipf=1.2)
    if gt == Q4_K:  # all-ones scales, minimums and nibbles
        for e in range(E):
            spec.up[e].reshape(-1, 144)[::2, 4:] = 0xFF
    x = orc.normal(S, S * d).reshape(S, d) + np.float32(1.0)
    x[::3] = np.sign(x[::3]) * 3.0
    spec.upload(ctx, S)
    xd = torch.from_numpy(x).cuda()
    ctx.set_regime(1)
    try:
        n0 = [ctx.profile_read(n)[1] for n in ("moe_gate_up_i8_f16", "moe_down_i8_f16")]
        out = ctx.moe_ffn(S, xd).cpu().numpy()
        assert [ctx.profile_read(n)[1] for n in ("moe_gate_up_i8_f16", "moe_down_i8_f16")] == [n + 1 for n in n0]
        cap_out, cap = ctx.moe_ffn_dbg(S, xd, k, F, gt, dt)
        idx, _, perm, off = (t.cpu().numpy() for t in ctx.last_routing(S, k, E))
    finally:
        ctx.set_regime(0)
    layer = spec.oracle_layer()
    assert np.array_equal(idx.astype(np.uint32), layer.route(x)[0])
    assert rel_l2(out, layer.moe_ffn(x, 1)) < 1e-3
    if Q6_K not in (gt, dt):
        assert np.array_equal(out.view(np.uint32), cap_out.cpu().numpy().view(np.uint32))
    if gt != Q4_K:
        return
    cap = {n: v.cpu().numpy() for n, v in cap.items()}
    off = off.view(np.uint32)
    q, _, bs = orc.q8k_quantize(x)
    big = int(np.argmax(np.diff(off.astype(np.int64))))
    for e in (big, int(np.argmin(np.where(np.diff(off.astype(np.int64)) > 4, np.diff(off.astype(np.int64)), 1 << 30)))):
        for p in (int(off[e]), int(off[e + 1]) - 1):
            tok = int(perm.view(np.uint32)[p]) // k
            for r in (0, F // 2 + 1, F - 1):
                row = spec.up[e].reshape(F, -1)[r]
                s, m = orc.q4k_block_acc(row, d, q.reshape(S, d)[tok], bs.reshape(S, -1)[tok])
                assert np.array_equal(cap["up_sumi"].reshape(S * k, F, -1)[p, r], s)
                assert np.array_equal(cap["up_mins"].reshape(S * k, F, -1)[p, r], m)


# small grids: the columns split over work-groups (an even and an uneven last
# part), one row tile per wave, plain and in the down product of few experts
@pytest.mark.parametrize("t,rows,cols,S", [(Q4_K, 4100, 4096, 33), (Q6_K, 4096, 4352, 9), (Q8_0, 2052, 5056, 20),
                                           (Q8_0, 2050, 4096, 17), (Q6_K, 8192, 1792, 64)])
def test_column_split_plain(ctx, t, rows, cols, S):
    from oracle import pyoracle as orc

    w = random_blocks(t, rows, cols, seed=rows + cols)
    x = np.random.default_rng(S).standard_normal((S, cols)).astype(np.float32)
    w64 = orc.dequant(t, w, rows * cols).reshape(rows, cols).astype(np.float64)
    ref = x.astype(np.float64) @ w64.T
    got = _matmul(ctx, t, w, rows, cols, x)
    assert np.all(np.abs(got - ref) <= _bound(t, w64, x, cols))
    assert rel_l2(got, ref) < 1e-6


@pytest.mark.parametrize("dt,E,S", [(Q4_K, 3, 52), (Q6_K, 3, 52), (Q8_0, 4, 71)])
def test_column_split_expert_down(ctx, dt, E, S):
    import torch
    from oracle import pyoracle as orc

    d, F, k = 512, 2304, 2
    spec = LayerSpec(E, k, d, F, Q4_K, seed=S + dt, down_type=dt, quantized=False)
    x = orc.normal(S, S * d).reshape(S, d)
    spec.upload(ctx, 2000 + dt)
    n0 = ctx.profile_read("moe_down_f16")[1]
    out = ctx.moe_ffn(2000 + dt, torch.from_numpy(x).cuda()).cpu().numpy()
    assert ctx.profile_read("moe_down_f16")[1] == n0 + 1
    layer = spec.oracle_layer()
    assert np.bincount(layer.route(x)[0].ravel(), minlength=E).min() >= 4
    assert rel_l2(out, layer.moe_ffn(x, 0)) < 3e-6


# AVX2 regime, experts of both kinds: the captured int8 rows of h are those of
# the int path's slots, though the f32 regime's slots are split into pieces
# before the capture is handed out
@pytest.mark.parametrize("dt", [Q4_K, Q6_K, Q8_0])
def test_capture_of_a_mixed_layer_keeps_the_int8_rows(ctx, dt):
    import torch
    from oracle import pyoracle as orc

    E, k, d, F, S = 70, 3, 256, 512, 900  # 21 slots of experts with 1-3 rows, two of them 8 x another's number
    spec = LayerSpec(E, k, d, F, Q4_K, seed=16, down_type=dt, zipf=0.5)
    x = orc.normal(S, S * d).reshape(S, d) + np.float32(1.0)
    spec.upload(ctx, 3000 + dt)
    n0 = ctx.profile_read("moe_down_f16")[1]
    _, cap = ctx.moe_ffn_dbg(3000 + dt, torch.from_numpy(x).cuda(), k, F, Q4_K, dt)
    assert ctx.profile_read("moe_down_f16")[1] == n0 + 1
    idx, _, perm, off = (t.cpu().numpy().astype(np.int64) for t in ctx.last_routing(S, k, E))
    hq, hd, hs = (cap[n].cpu().numpy() for n in ("hq", "hd", "hs"))
    seen = 0
    for e in np.flatnonzero((np.diff(off) > 0) & (np.diff(off) < 4)):
        p = np.arange(off[e], off[e + 1])
        h = orc.swiglu(*(orc.matmul(Q4_K, w[e], F, d, x[perm[p] // k]) for w in (spec.gate, spec.up)))
        q, sc = (orc.q8_quantize if dt == Q8_0 else orc.q8k_quantize)(h)[:2]
        # (h in another float order: 1e-6 of it, which may move an int8 value across a rounding)
        assert np.abs(hd[p] - np.asarray(sc).reshape(hd[p].shape)).max() <= 1e-5 * np.abs(sc).max()
        assert np.abs(hq[p].astype(int) - np.asarray(q).reshape(hq[p].shape)).max() <= 1
        assert np.array_equal(hs[p], hq[p].astype(np.int32).reshape(len(p), -1, 16).sum(2))
        seen += len(p)
    assert seen >= 8


# the int8 regime's products on int8 rows are exact integers joined once per
# block: the captured call gives the layer's own bits, the integers are the
# oracle's, and the down product is within the roundings of its join. Rows past
# one chain of roundings (17 superblocks), one and two token tiles.
@pytest.mark.parametrize("gt,dt,E,S,F", [(Q6_K, Q6_K, 3, 60, 4352), (Q8_0, Q6_K, 6, 130, 512), (Q4_K, Q8_0, 3, 60, 4352),
                                         (Q4_K, Q4_K, 4, 240, 4352), (Q6_K, Q8_0, 5, 33, 384)])
def test_int8_regime_down_is_the_exact_integers(ctx, gt, dt, E, S, F):
    import torch
    from oracle import pyoracle as orc

    d, k, lid = 256, 2, 4000 + 100 * gt + dt
    spec = LayerSpec(E, k, d, F, gt, seed=S + dt, down_type=dt, quantized=False)
    x = orc.normal(S, S * d).reshape(S, d)
    spec.upload(ctx, lid)
    xd = torch.from_numpy(x).cuda()
    ctx.set_regime(1)
    try:
        n0 = ctx.profile_read("moe_down_i8_f16")[1]
        out = ctx.moe_ffn(lid, xd).cpu().numpy()
        assert ctx.profile_read("moe_down_i8_f16")[1] == n0 + 1
        cap_out, cap = ctx.moe_ffn_dbg(lid, xd, k, F, gt, dt)
        idx, wsel, perm, off = (t.cpu().numpy() for t in ctx.last_routing(S, k, E))
    finally:
        ctx.set_regime(0)
    assert np.array_equal(out.view(np.uint32), cap_out.cpu().numpy().view(np.uint32))
    hq, hd, hs, si, mi = (cap[n].cpu().numpy() for n in ("hq", "hd", "hs", "down_sumi", "down_mins"))
    y, mag = np.zeros((2, S * k, d))
    size, at = {Q4_K: (144, 0), Q6_K: (210, 208), Q8_0: (34, 0)}[dt]
    assert dt != Q4_K or np.diff(off.astype(np.int64)).max() > 32  # (fewer rows: the int8 kernels)
    for e in range(E):
        b = spec.down[e].reshape(d, -1, size)
        half = lambda i: b[:, :, i:i + 2].copy().view(np.float16)[:, :, 0].astype(np.float64)
        for p in range(int(off[e]), int(off[e + 1])):
            for r in (0, 100, d - 1) if dt != Q8_0 else ():
                acc = orc.q4k_block_acc if dt == Q4_K else orc.q6k_block_acc
                s, m = acc(b[r].reshape(-1), F, hq[p], hs[p])
                assert np.array_equal(si[p, r], s) and np.array_equal(mi[p, r], m)
            if dt == Q8_0:
                q = b[:, :, 2:].copy().view(np.int8).astype(np.int64)
                assert np.array_equal(si[p], (q * hq[p].reshape(1, -1, 32)).sum(2))
            t = si[p] * half(at) * hd[p]
            if dt != Q8_0:
                u = mi[p] * (half(2) if dt == Q4_K else 32 * half(at)) * hd[p]
                if dt == Q4_K:  # the minimum term is rounded by itself
                    mag[p] += np.abs(u).sum(1)
                t = t - u
            y[p], mag[p] = t.sum(1), mag[p] + np.abs(t).sum(1)
    order = np.empty(S * k, np.int64)
    order[perm.view(np.uint32).astype(np.int64)] = np.arange(S * k)
    w = wsel.astype(np.float64).reshape(S, k, 1)
    ref, bound = ((v[order].reshape(S, k, d) * w).sum(1) for v in (y, mag))
    # roundings on one element's way: 3 in its term, chains of 8 (Q8_0: 4 and 4), of the parts and of the k slots
    n = 3 + 8 + F // 2048 + 1 + k + (F // 512 if dt == Q8_0 else 0)
    assert np.all(np.abs(out - ref) <= n * 2.0 ** -24 * bound)
    assert rel_l2(out, ref) < 1.5e-7


def _product(S, rows=8192, cols=512, seed=5):
    """A Q4_K product whose pieces are far larger than the int8 rows' workspace."""
    import torch
    from oracle import pyoracle as orc

    w = torch.from_numpy(random_blocks(Q4_K, rows, cols, seed=seed)).cuda()
    return w, rows, cols, torch.from_numpy(orc.normal(seed, S * cols).reshape(S, cols)).cuda()


def test_products_leave_the_workspace_and_the_last_routing_alone(ctx):
    import torch

    S, d = 300, 512
    spec = LayerSpec(6, 2, d, 256, Q4_K, seed=3, quantized=False)
    spec.upload(ctx, 5000)
    w, rows, cols, x = _product(S)
    gen = []
    for _ in range(2):  # (the second time nothing grows)
        ctx.moe_ffn(5000, x)
        before = [t.cpu().numpy().copy() for t in ctx.last_routing(S, 2, 6)]
        ctx.matmul(Q4_K, w, rows, cols, x)
        gen.append(ctx.workspace_generation())
    assert gen[0] == gen[1]
    assert all(np.array_equal(a, b.cpu().numpy()) for a, b in zip(before, ctx.last_routing(S, 2, 6)))


def test_scratch_of_products_gives_way_to_other_allocations():
    from kestrel_amd.kmoe import REGIME_INT8, Context

    w, rows, cols, x = _product(600)
    c = Context(0)
    c.profile_enable(True)
    try:
        c.set_regime(REGIME_INT8)  # int8 rows: no pieces
        c.matmul(Q4_K, w, rows, cols, x)
        base = c.vram_usage()[0]
        c.set_regime(0)
        full = c.matmul(Q4_K, w, rows, cols, x).cpu().numpy()
        assert c.vram_usage()[0] > base and c.profile_read("f16_gemm")[1] == 1
        E, d, F = 12, 256, 256
        room = c.vram_usage()[0] - base
        c.vram_set_limit(c.vram_usage()[0] + room // 4)
        assert room // 4 < 3 * E * F * 144 < room  # more than is free, less than with the pieces' bytes
        c.layer_create(0, E, 1, d, F, Q4_K, Q4_K, Q4_K)
        again = c.matmul(Q4_K, w, rows, cols, x).cpu().numpy()  # no room for the pieces now
        assert c.profile_read("f16_gemm")[1] == 1 and rel_l2(again, full) < 2e-6
        c.layer_destroy(0)
        assert np.array_equal(c.matmul(Q4_K, w, rows, cols, x).cpu().numpy(), full)
        c.vram_set_limit(base)  # a lower limit takes them too
        assert c.vram_usage()[0] == base
    finally:
        c.close()


def test_a_product_first_called_in_a_capture_runs_the_same_kernels():
    """Nothing before the capture but the int8 workspace: the graph holds the
    matrix-core product, its replays give the eager bits, and a larger eager
    product between replays leaves the graph's scratch alone."""
    import torch
    from kestrel_amd.kmoe import REGIME_INT8, Context

    w, rows, cols, x = _product(200)
    wl, _, _, xl = _product(900, seed=6)
    c = Context(0)
    c.profile_enable(True)
    want = c.matmul(Q4_K, w, rows, cols, x).cpu().numpy()
    want_l = c.matmul(Q4_K, wl, rows, cols, xl).cpu().numpy()
    c.close()
    c = Context(0)
    try:
        c.set_regime(REGIME_INT8)
        c.matmul(Q4_K, w, rows, cols, x)
        c.matmul(Q4_K, wl, rows, cols, xl)
        c.set_regime(0)
        out = torch.empty((200, rows), device="cuda")
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        try:
            with torch.cuda.graph(g):
                c.set_stream(torch.cuda.current_stream())
                out.copy_(c.matmul(Q4_K, w, rows, cols, x))
        finally:
            c.set_stream(torch.cuda.current_stream())
        for i in range(4):
            out.zero_()
            g.replay()
            torch.cuda.synchronize()
            assert np.array_equal(out.cpu().numpy().view(np.uint32), want.view(np.uint32)), i
            t = (wl, xl, want_l) if i % 2 == 0 else (w, x, want)
            assert np.array_equal(c.matmul(Q4_K, t[0], rows, cols, t[1]).cpu().numpy(), t[2])
        torch.cuda.synchronize()
        del g
    finally:
        c.close()


def test_products_on_two_streams_do_not_share_pieces_at_once():
    import torch
    from kestrel_amd.kmoe import Context

    rows, cols, S = 4096, 4096, 512
    w, _, _, _ = _product(1, rows, cols)
    xs = [torch.randn(S, cols, device="cuda", generator=torch.Generator("cuda").manual_seed(i)) for i in range(2)]
    c = Context(0)
    try:
        want = [c.matmul(Q4_K, w, rows, cols, x).clone() for x in xs]
        st = [torch.cuda.Stream(), torch.cuda.Stream()]
        outs = [torch.empty((8, S, rows), device="cuda") for _ in range(2)]
        torch.cuda.synchronize()
        for i in range(8):
            for j in range(2):
                c.set_stream(st[j])
                c.check(c.lib.kmoe_matmul(c.h, Q4_K, w.data_ptr(), w.numel(), rows, cols, xs[j].data_ptr(), S,
                                          outs[j][i].data_ptr()))
        torch.cuda.synchronize()
        assert all(torch.equal(outs[j][i], want[j]) for j in range(2) for i in range(8))
    finally:
        torch.cuda.synchronize()
        c.close()
