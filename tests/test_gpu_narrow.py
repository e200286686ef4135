"""GPU: the few-row GEMM over quantized weights (csrc/mm_narrow.h) at the edges of its row tiles and
column blocks, against a float64 product: of the weights rounded to bf16 for the k-quants (what
the kernel feeds the matrix cores), of the true weights for the affine formats (which it does not
round), and the MoE block built on it against the oracle's exact block."""
import numpy as np
import pytest

import util
from util import Q4K, Q6K

pytestmark = pytest.mark.gpu


def _weights(lin):
    if lin.mode == "kq":
        w = util.orc_dequant(lin.km.kind, lin.km.qs, lin.km.scales, lin.km.dm, lin.O * lin.K // 256)
        return util.bf16_to_f32(util.f32_to_bf16(w)).astype(np.float64).reshape(lin.O, lin.K)
    if lin.mode == "affine4":
        q = np.stack([lin.w & 15, lin.w >> 4], -1).reshape(lin.O, lin.K).astype(np.float64)
        g = 32
    else:
        q, g = lin.w.astype(np.float64), 64
    s, b = (np.repeat(util.bf16_to_f32(t).astype(np.float64), g, axis=1) for t in (lin.scales, lin.biases))
    return q * s + b


@pytest.mark.parametrize("fmt", ["q4k", "q6k", "affine4", "affine8"])
@pytest.mark.parametrize("O,K,M", [(512, 2048, 32), (200, 512, 33), (264, 768, 48), (2048, 4096, 65), (40, 1024, 130),
                                    (4096, 2048, 64), (64, 4096, 17 + 64), (8, 2048, 200),
                                    # two and four column tiles a wavefront; an odd number of columns
                                    (4096, 512, 65), (4096, 2048, 65), (4099, 2048, 130), (12288, 2048, 33),
                                    # 32-row tiles: the last product that one workgroup a compute unit covers with 16 columns
                                    # each, with 32, and the first past both; remainders of 1 and 17 rows; 64-row tiles whose
                                    # scales would leave a compute unit one workgroup
                                    (2048, 4096, 64), (2040, 4096, 113), (2048, 4096, 129), (2048, 2048, 65), (256, 2048, 512),
                                    (2048, 4096, 577),
                                    # the last rows that narrow k-quant matrices take here, and the first past them
                                    (264, 2048, 1536), (264, 2048, 1537), (256, 2048, 2560), (256, 2048, 2561),
                                    # columns owned by wavefronts: row tiles of 64 and remainders of 16, 32 and 48, two, three,
                                    # eight and sixteen blocks of K, columns past the last workgroup's
                                    (2056, 512, 193), (2184, 768, 481), (4099, 2048, 525), (2064, 4096, 449), (8192, 2048, 940)])
def test_few_row_matmul_vs_float64(orn, ctx, fmt, O, K, M):
    rng = np.random.default_rng(O + K + M)
    lin = (util.HostLinear.kq(rng, Q4K if fmt == "q4k" else Q6K, O, K) if fmt[0] == "q" else
           getattr(util.HostLinear, fmt)(rng, O, K))
    dl = lin.dev(orn, ctx)
    xb = util.bf16_normal(rng, (M, K))
    dx, dy = ctx.to_device(xb), ctx.alloc(M * O * 2)
    ctx.memset(dy, 0xFF, M * O * 2)
    ctx.linear_matmul(dl, dx, M, dy)
    got = util.bf16_to_f32(dy.download(np.uint16, (M, O))).astype(np.float64)
    want = util.bf16_to_f32(xb).astype(np.float64) @ _weights(lin).T
    scale = np.sqrt(np.mean(want ** 2))
    # one rounding of the output, and fp32 sums in another order
    assert np.all(np.abs(got - want) <= 2.0 ** -8 * np.abs(want) + 2e-5 * scale), float(np.abs(got - want).max() / scale)
    for b in (dx, dy): b.free()
    dl.free()


@pytest.mark.parametrize("fmt", ["q4k", "affine4", "affine8"])
@pytest.mark.parametrize("O,dense,K,M", [(512, (32, 32), 2048, 32), (4096, (1, 40), 2048, 51), (2056, (32,), 2048, 193),
                                         (4096, (32, 17), 2048, 500), (264, (16, 1), 4096, 77), (512, (32, 32), 1024, 40),
                                         (4096, (32, 32), 2048, 1300),
                                         # a dense matrix beside them that does not ride: too large (192 rows and fewer, more, long prompts)
                                         (512, (4096,), 2048, 192), (512, (512, 40), 2048, 300), (264, (48, 32), 2048, 2100)])
def test_dense_matrices_ride_along_with_a_few_row_gemm(orn, ctx, fmt, O, dense, K, M):
    """linear_matmul_multi of two quantized matrices and one or two dense ones at prompt widths: one launch where K and the dense ones'
    size allow (in the form with K split over wavefronts and in the one with columns owned; rows and columns ragged), and
    every output is the matrix's own launch bit for bit, past every output nothing is written"""
    rng = np.random.default_rng(O + K + M)
    make = {"q4k": lambda o: util.HostLinear.kq(rng, Q4K, o, K), "affine4": lambda o: util.HostLinear.affine4(rng, o, K),
            "affine8": lambda o: util.HostLinear.affine8(rng, o, K)}[fmt]
    hls = [make(O), make(256)] + [util.HostLinear.dense(rng, o, K) for o in dense]
    Os = [O, 256] + list(dense)
    lins = [h.dev(orn, ctx) for h in hls]
    dx = ctx.to_device(util.bf16_normal(rng, (M, K)))
    ys = [ctx.alloc((M + 1) * o * 2) for o in Os]
    for y, o in zip(ys, Os): ctx.memset(y, 0x5A, (M + 1) * o * 2)
    ctx.linear_matmul_multi(lins, dx, M, ys)
    y1 = ctx.alloc(M * max(Os) * 2)
    for lin, y, o in zip(lins, ys, Os):
        ctx.linear_matmul(lin, dx, M, y1)
        got = y.download(np.uint16, (M + 1, o))
        assert np.array_equal(got[:M], y1.download(np.uint16, (M, o))), o
        assert np.all(got[M] == 0x5A5A), o
    for b in [dx, y1] + ys: b.free()
    for l in lins: l.free()


@pytest.mark.parametrize("fmt", ["kq", "affine4"])
@pytest.mark.parametrize("T", [32, 100, 150, 300])
def test_few_row_moe_block_vs_exact(orn, ctx, fmt, T):
    """16-, 32- and 64-row expert tiles (4 to 38 rows an expert on average), the shared expert among
    them. A router tie may fall the other way than in the oracle's exact block: such a row differs by an
    expert, so the bound is on the rows' median and 93 % of them. (The operator keeps affine experts exact;
    their GEMMs are a layer's, below.)"""
    rng = np.random.default_rng(T)
    moe = util.HostMoe(rng, H=1024, E=64, I=512, top_k=8, gate_kind=util.AFFINE4 if fmt == "affine4" else Q4K)
    xb = util.bf16_normal(rng, (T, 1024))
    want = util.bf16_to_f32(util.orc_moe_block(moe, xb, T)[0]).astype(np.float64)
    w = moe.dev(orn, ctx)
    dx, out = ctx.to_device(xb), ctx.alloc(T * 1024 * 2)
    outs = []
    for fill in (0xFF, 0x00):
        ctx.memset(out, fill, T * 1024 * 2)
        ctx.moe_block(w, dx, T, out)
        outs.append(out.download(np.uint16, (T, 1024)))
    assert np.array_equal(outs[0], outs[1])
    got = util.bf16_to_f32(outs[0]).astype(np.float64)
    rel = np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)
    bound = 0.004 if fmt == "affine4" else 0.01
    assert np.median(rel) < bound and (rel < 0.03).mean() >= 0.93, (float(np.median(rel)), float(np.sort(rel)[-5]))
    for b in (dx, out): b.free()
    moe.free()


@pytest.mark.parametrize("E,T", [(128, 40), (512, 33), (1024, 32)])
def test_few_row_moe_block_of_other_expert_counts(orn, ctx, E, T):
    """The other layouts of the router's tail, against the oracle's exact block as above."""
    rng = np.random.default_rng(E)
    moe = util.HostMoe(rng, H=512, E=E, I=512, top_k=8)
    xb = util.bf16_normal(rng, (T, 512))
    want = util.bf16_to_f32(util.orc_moe_block(moe, xb, T)[0]).astype(np.float64)
    w = moe.dev(orn, ctx)
    dx, out = ctx.to_device(xb), ctx.alloc(T * 512 * 2)
    ctx.moe_block(w, dx, T, out)
    got = util.bf16_to_f32(out.download(np.uint16, (T, 512))).astype(np.float64)
    rel = np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)
    assert np.median(rel) < 0.01 and (rel < 0.03).mean() >= 0.93, np.sort(rel)[-5:]
    for b in (dx, out): b.free()
    moe.free()


@pytest.mark.parametrize("T", [32, 100, 150, 300])
def test_few_row_moe_block_of_a_layer_over_affine_experts(orn, ctx, T):
    """ornith_add_rms_moe_block from gemm_rows rows on: the affine experts as GEMMs behind the layer's norm,
    against the oracle's exact block on the normed rows, with the bound of the test above; with GEMMs
    switched off its bits."""
    rng = np.random.default_rng(T)
    H = 1024
    moe = util.HostMoe(rng, H=H, E=64, I=512, top_k=8, gate_kind=util.AFFINE4)
    res, y, wn = (util.bf16_normal(rng, s) for s in ((T, H), (T, H), (H,)))
    wh, wnormed = util.orc_add_rms_norm(res, y, wn)
    want16 = util.orc_moe_block(moe, wnormed, T)[0]
    want = util.bf16_to_f32(want16).astype(np.float64)
    w = moe.dev(orn, ctx)
    bufs = [ctx.to_device(a) for a in (res, y, wn)] + [ctx.alloc(T * H * 2) for _ in range(3)]
    dres, dy, dwn, dh, dn, out = bufs
    try:
        got = {}
        for rows in (32, 0):
            orn.set_option("gemm_rows", rows)
            ctx.memset(out, 0xFF, T * H * 2)
            orn.add_rms_moe_block(ctx, w, dres, dy, dwn, 1e-6, T, dh, dn, out)
            assert np.array_equal(dh.download(np.uint16, (T, H)), wh) and np.array_equal(dn.download(np.uint16, (T, H)), wnormed)
            got[rows] = out.download(np.uint16, (T, H))
    finally:
        orn.set_option("gemm_rows", 32)
    assert np.array_equal(got[0], want16) and not np.array_equal(got[32], want16)
    rel = np.linalg.norm(util.bf16_to_f32(got[32]).astype(np.float64) - want, axis=1) / np.linalg.norm(want, axis=1)
    assert np.median(rel) < 0.004 and (rel < 0.03).mean() >= 0.93, (float(np.median(rel)), float(np.sort(rel)[-5]))
    for b in bufs: b.free()
    moe.free()


def _deq(kind, t, E, O, K):
    w = util.orc_dequant(kind, *t, E * O * K // 256)
    return util.bf16_to_f32(util.f32_to_bf16(w)).astype(np.float64).reshape(E, O, K)


@pytest.mark.parametrize("kind,E,O,K,T,k", [
    # 16-, 32- and 64-row tiles; columns below, at and past a workgroup's 128; K of two, three, eight and sixteen blocks
    (Q4K, 8, 200, 512, 20, 2), (Q6K, 8, 200, 512, 20, 2), (Q6K, 16, 8, 768, 90, 3), (Q4K, 16, 136, 768, 200, 2),
    (Q4K, 8, 128, 2048, 60, 3), (Q6K, 8, 264, 2048, 90, 4), (Q4K, 4, 64, 4096, 33, 4), (Q6K, 4, 129, 4096, 33, 4),
    # the most rows an expert that these kernels take (79), and past the 48 from which other matrices go elsewhere
    (Q4K, 8, 200, 1024, 316, 2), (Q6K, 16, 136, 512, 200, 4)])
@pytest.mark.parametrize("skew", [False, True])
def test_few_row_gathered_matmul_vs_float64(orn, ctx, kind, E, O, K, T, k, skew):
    """The expert form whose wavefronts own columns, over every pair of a token list: one rounding of the output, and
    fp32 sums in another order (as above). skew: half of the picks fall on expert 1, which then has several tiles."""
    rng = np.random.default_rng(E * O + K + T)
    t = (util.make_q4k if kind == Q4K else util.make_q6k)(rng, E, O, K)
    inds = np.stack([rng.permutation(E)[:k] for _ in range(T)]).astype(np.uint32)
    if skew:
        inds[: T // 2 * 2 : 2, 0] = 1
    pairs = T * k
    assert pairs < 80 * E
    wt = _deq(kind, t, E, O, K)
    w = orn.KMatrix(ctx, kind, *t, E, O, K)
    plan = ctx.alloc(orn.kq_gather_plan_bytes(pairs, E))
    di = ctx.to_device(inds.reshape(-1))
    for is_up in (True, False):
        rows = T if is_up else pairs
        xb = util.bf16_normal(rng, (rows, K))
        dx, dy = ctx.to_device(xb), ctx.alloc((pairs + 1) * O * 2)
        ctx.memset(dy, 0xFF, (pairs + 1) * O * 2)
        orn.kq_gather_matmul(ctx, w, dx, di, pairs, k, is_up, plan, is_up, dy)
        out = dy.download(np.uint16, (pairs + 1, O))
        assert np.all(out[pairs] == 0xFFFF)
        got = util.bf16_to_f32(out[:pairs]).astype(np.float64)
        x = util.bf16_to_f32(xb).astype(np.float64)
        want = np.stack([wt[inds[p // k, p % k]] @ x[p // k if is_up else p] for p in range(pairs)])
        scale = np.sqrt(np.mean(want ** 2))
        assert np.all(np.abs(got - want) <= 2.0 ** -8 * np.abs(want) + 2e-5 * scale), float(np.abs(got - want).max() / scale)
        for b in (dx, dy): b.free()
    for b in (di, plan, w): b.free()


@pytest.mark.parametrize("fmt,T", [("kq", 70), ("kq", 200), ("affine4", 40), ("affine4", 150)])
def test_few_row_moe_block_whose_shared_expert_has_another_format(orn, ctx, fmt, T):
    """Launches of two formats (Q4_K and Q6_K, 4-bit and 8-bit affine), at K = 2048 (where the 4-bit scales lie turned by
    the row), against the oracle's exact block on the normed rows, with the bounds of the tests above."""
    rng = np.random.default_rng(T)
    H, I = 2048, 512
    moe = util.HostMoe(rng, H=H, E=64, I=I, top_k=8, gate_kind=util.AFFINE4 if fmt == "affine4" else Q4K)
    other = (lambda o, k, kind: util.HostLinear.kq(rng, kind, o, k)) if fmt == "kq" else (lambda o, k, _: util.HostLinear.affine8(rng, o, k))
    moe.sh_gate, moe.sh_up, moe.sh_down = other(I, H, Q6K), other(I, H, Q6K), other(H, I, Q4K)
    res, y, wn = (util.bf16_normal(rng, s) for s in ((T, H), (T, H), (H,)))
    _, normed = util.orc_add_rms_norm(res, y, wn)
    want = util.bf16_to_f32(util.orc_moe_block(moe, normed, T)[0]).astype(np.float64)
    w = moe.dev(orn, ctx)
    bufs = [ctx.to_device(a) for a in (res, y, wn)] + [ctx.alloc(T * H * 2) for _ in range(3)]
    dres, dy, dwn, dh, dn, out = bufs
    orn.add_rms_moe_block(ctx, w, dres, dy, dwn, 1e-6, T, dh, dn, out)
    got = util.bf16_to_f32(out.download(np.uint16, (T, H))).astype(np.float64)
    rel = np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)
    bound = 0.004 if fmt == "affine4" else 0.01
    assert np.median(rel) < bound and (rel < 0.03).mean() >= 0.93, (float(np.median(rel)), float(np.sort(rel)[-5]))
    for b in bufs: b.free()
    moe.free()
