"""GPU: the long-prompt GEMM whose wavefronts own columns (csrc/kq_mm_own.hip), at the edges of its tiles: every
tile height, rows and columns that end inside one, one super-block of K and an odd number of them, one
row of an expert. Against a float64 product over the bf16-rounded dequantized weights, which is what the matrix cores
are fed: an element may be off by the rounding of the bf16 result (half an ulp of 8 significant bits: 2^-8 of it at most) and by its fp32 sum, whose K additions
err by at most 2^-24 each of what has been added up, sum |x w| at most; twice that for the matrix cores' own order."""
import numpy as np
import pytest

import util
from util import Q4K, Q6K

pytestmark = pytest.mark.gpu


def _deq(kind, t, E, O, K):
    w = util.orc_dequant(kind, *t, E * O * K // 256).reshape(E, O, K)
    return util.bf16_to_f32(util.f32_to_bf16(w)).astype(np.float64)


def _check(got_bits, x, w, what):
    want, mass = x @ w.T, np.abs(x) @ np.abs(w).T
    err = np.abs(util.bf16_to_f32(got_bits).astype(np.float64) - want)
    bound = 2.0 ** -8 * np.abs(want) + 2 * x.shape[1] * 2.0 ** -24 * mass
    assert np.all(err <= bound), (what, float((err / bound).max()))


@pytest.mark.parametrize("kind,O,K,M", [
    # the lowest row counts of the rule; columns that end inside a tile
    (Q4K, 40, 256, 129), (Q6K, 264, 768, 129), (Q4K, 2304, 768, 129),
    (Q4K, 2056, 2048, 193), (Q6K, 2056, 2304, 193), (Q4K, 2304, 256, 513), (Q6K, 2051, 768, 545), (Q6K, 72, 256, 2049),
    (Q4K, 257, 2048, 1025 + 512),
    # two sets of wavefronts with half of K each: one super-block a set and an odd number, the ends of the rule, columns and rows that
    # end inside a tile, tiles of 2, 3 and 4 row blocks
    (Q4K, 2056, 512, 129), (Q6K, 2049, 1536, 193), (Q4K, 2056, 2048, 256), (Q4K, 2056, 2048, 257), (Q4K, 600, 2048, 513), (Q6K, 2043, 2048, 545),
    (Q6K, 1032, 2048, 2048), (Q6K, 1032, 2048, 2049), (Q4K, 10880, 512, 200), (Q4K, 16384, 512, 225), (Q6K, 2304, 768, 200),
    # 64 column tiles: the tile height that fills 256 compute units, 8, 8, 7, 6 and 5 blocks of 32 rows, and what is left of it
    (Q4K, 16384, 256, 1000), (Q6K, 16384, 256, 900), (Q4K, 16384, 256, 890), (Q6K, 16384, 256, 760), (Q4K, 16380, 512, 601),
    # more than one round of tiles, in patches of eight row tiles and a rest
    (Q6K, 4100, 256, 4129)])
def test_own_columns_matmul(orn, ctx, kind, O, K, M):
    rng = np.random.default_rng(O + K + M + kind)
    t = util.make_kq(kind, rng, 1, O, K)
    w = orn.KMatrix(ctx, kind, *t, 1, O, K)
    xb = util.bf16_normal(rng, (M, K))
    dx, dy = ctx.to_device(xb), ctx.alloc((M + 1) * O * 2)
    ctx.memset(dy, 0xFF, (M + 1) * O * 2)
    orn.kq_matmul(ctx, w, dx, M, dy)
    got = dy.download(np.uint16, (M + 1, O))
    assert np.all(got[M] == 0xFFFF)
    _check(got[:M], util.bf16_to_f32(xb).astype(np.float64), _deq(kind, t, 1, O, K)[0], (kind, O, K, M))
    for b in (dx, dy): b.free()
    w.free()


TALL = (1, 31, 32, 33, 64, 65, 97, 128, 129, 161, 192, 193, 225, 256, 257, 0, 555)
LOW = (1, 31, 32, 33, 64, 65, 0, 97, 48, 20, 129, 7, 12, 260, 3)  # 53 an expert: a plan of tiles lower than the kernel's


@pytest.mark.parametrize("counts,kind,O,K", [
    # tiles of 128 x 128, while larger ones are half the compute units or fewer
    (TALL, Q4K, 264, 512), (TALL, Q6K, 131, 256), (TALL, Q6K, 512, 768), (TALL, Q4K, 1032, 2048), (LOW, Q4K, 264, 4352), (LOW, Q6K, 131, 1280),
    # ... of 256 x 256
    (TALL, Q4K, 2056, 512), (TALL, Q6K, 2051, 256), (TALL, Q6K, 2304, 768), (LOW, Q4K, 2312, 4352), (LOW, Q6K, 2307, 1280)])
def test_own_columns_experts_of_every_height(orn, ctx, counts, kind, O, K):
    """an expert of each number of 32-row blocks, one row to either side of a block's end, one without rows, one of several tiles"""
    E, pairs = len(counts), sum(counts)
    assert pairs >= (80 if counts is TALL else 48) * E and orn.gather_form(kind, E, O, K, pairs) == (1 if O > 2048 else 4)
    rng = np.random.default_rng(O + K)
    t = util.make_kq(kind, rng, E, O, K)
    w = orn.KMatrix(ctx, kind, *t, E, O, K)
    inds = rng.permutation(np.repeat(np.arange(E), counts)).astype(np.uint32)
    xb = util.bf16_normal(rng, (pairs, K))
    plan = ctx.alloc(orn.kq_gather_plan_bytes(pairs, E))
    di, dx, dy = ctx.to_device(inds), ctx.to_device(xb), ctx.alloc((pairs + 1) * O * 2)
    ctx.memset(dy, 0xFF, (pairs + 1) * O * 2)
    orn.kq_gather_matmul(ctx, w, dx, di, pairs, 1, False, plan, True, dy)
    got, x, deq = dy.download(np.uint16, (pairs + 1, O)), util.bf16_to_f32(xb).astype(np.float64), _deq(kind, t, E, O, K)
    assert np.all(got[pairs] == 0xFFFF)
    for e in range(E):
        sel = np.nonzero(inds == e)[0]
        if len(sel): _check(got[sel], x[sel], deq[e], (kind, O, K, counts[e]))
    for b in (plan, di, dx, dy): b.free()
    w.free()


@pytest.mark.parametrize("kind", [Q4K, Q6K])
@pytest.mark.parametrize("O,K,M", [(2056, 256, 300), (2051, 768, 257), (2056, 2048, 609), (2304, 512, 1400), (4104, 2048, 260)])
def test_small_tiles_give_the_full_ones_sums(orn, ctx, kind, O, K, M):
    """a matrix that by itself runs in 128 x 128 tiles, every number of row blocks and an end inside one: the same bits beside a matrix that fills
    the device, where it runs in 256 x 256 ones, no store past the last row, and float64's numbers"""
    rng = np.random.default_rng(O + K + M)
    t, big = util.make_kq(kind, rng, 1, O, K), 32768
    w = orn.Linear.kquant(ctx, kind, *t, O, K)
    wide = orn.Linear.kquant(ctx, kind, *util.make_kq(kind, rng, 1, big, K), big, K)
    assert orn.gemm_form(kind, O, K, M) == 4 and orn.gemm_form(kind, big, K, M) == 1
    xb = util.bf16_normal(rng, (M, K))
    dx, alone, beside, ybig = ctx.to_device(xb), ctx.alloc((M + 1) * O * 2), ctx.alloc((M + 1) * O * 2), ctx.alloc(M * big * 2)
    for y in (alone, beside): ctx.memset(y, 0xFF, (M + 1) * O * 2)
    ctx.linear_matmul(w, dx, M, alone)
    ctx.linear_matmul_multi([wide, w], dx, M, [ybig, beside])
    got = alone.download(np.uint16, (M + 1, O))
    assert np.array_equal(got, beside.download(np.uint16, (M + 1, O)))
    assert np.all(got[M] == 0xFFFF)
    _check(got[:M], util.bf16_to_f32(xb).astype(np.float64), _deq(kind, t, 1, O, K)[0], (kind, O, K, M))
    for b in (dx, alone, beside, ybig, w, wide): b.free()


@pytest.mark.parametrize("mats,K,M,form", [
    # a gated-delta layer's two wide projections; both kinds, columns that end inside a tile, more than one round of tiles; the ends of the rule
    ([(Q4K, 8192), (Q4K, 4096)], 2048, 200, 2), ([(Q4K, 1032), (Q6K, 2043)], 2048, 700, 2), ([(Q6K, 2048), (Q4K, 1800), (Q6K, 2041)], 2048, 2048, 2),
    ([(Q6K, 4104), (Q4K, 4100), (Q6K, 4097), (Q4K, 4096)], 512, 256, 2),
    # small tiles over all of K: both kinds, three and four matrices
    ([(Q4K, 2060), (Q6K, 2051), (Q6K, 300)], 768, 1025, 4)])
def test_matrices_of_one_form_share_a_launch(orn, ctx, mats, K, M, form):
    """each the same bits as alone, and float64's numbers; no store past the last row"""
    rng = np.random.default_rng(M + K)
    ts = [util.make_kq(kind, rng, 1, O, K) for kind, O in mats]
    ws = [orn.Linear.kquant(ctx, kind, *t, O, K) for (kind, O), t in zip(mats, ts)]
    xb = util.bf16_normal(rng, (M, K))
    dx, ys, alone = ctx.to_device(xb), [ctx.alloc((M + 1) * O * 2) for _, O in mats], ctx.alloc(M * max(O for _, O in mats) * 2)
    for (_, O), y in zip(mats, ys): ctx.memset(y, 0xFF, (M + 1) * O * 2)
    ctx.linear_matmul_multi(ws, dx, M, ys)
    x = util.bf16_to_f32(xb).astype(np.float64)
    for (kind, O), t, w, y in zip(mats, ts, ws, ys):
        assert orn.gemm_form(kind, O, K, M) == form, (kind, O)
        got = y.download(np.uint16, (M + 1, O))
        assert np.all(got[M] == 0xFFFF)
        ctx.linear_matmul(w, dx, M, alone)
        assert np.array_equal(got[:M], alone.download(np.uint16, (M, O))), (kind, O)
        _check(got[:M], x, _deq(kind, t, 1, O, K)[0], (kind, O, K, M))
    for b in [dx, alone] + ys + ws: b.free()


def test_own_columns_forms_in_one_call(orn, ctx):
    """matrices of one call whose sums are taken over K as a whole and in halves, and one that neither form takes: each the same bits as alone"""
    K, M, Os = 2048, 1100, (2304, 600, 264, 64)
    rng = np.random.default_rng(3)
    ws = [orn.Linear.kquant(ctx, kind, *util.make_kq(kind, rng, 1, O, K), O, K) for kind, O in zip((Q4K, Q6K, Q6K, Q6K), Os)]
    dx, ys = ctx.to_device(util.bf16_normal(rng, (M, K))), [ctx.alloc(M * O * 2) for O in Os]
    ctx.linear_matmul_multi(ws, dx, M, ys)
    for w, O, y in zip(ws, Os, ys):
        alone = ctx.alloc(M * O * 2)
        ctx.linear_matmul(w, dx, M, alone)
        assert np.array_equal(y.download(np.uint16, (M, O)), alone.download(np.uint16, (M, O))), O
        for b in (y, alone): b.free()
        w.free()
    dx.free()
