"""GPU parity of the 4-bit affine (group 32) format against the oracle, bit for bit: Linear
mat-vec at decode widths, the gathered form over stacked experts, the table lookup, and a
small model whose affine modules (embed_tokens, shared_expert_gate) are in that format through
both generation loops."""
import numpy as np
import pytest

import synth
import util
from util import oracle, p

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("O,K", [(512, 2048), (7, 32), (2048, 4096), (33, 96), (1, 2048)])
def test_affine4_linear_bit_exact(orn, ctx, O, K):
    rng = np.random.default_rng(O + K)
    lin = util.HostLinear.affine4(rng, O, K)
    dl = lin.dev(orn, ctx)
    for M in (1, 2, 4, 5):
        xb = util.bf16_normal(rng, (M, K))
        want = np.empty((M, O), np.uint16)
        oracle().orc_affine4_gather_qmv(p(lin.w), p(lin.scales), p(lin.biases), 1, O, K, p(xb), None, None, M, p(want))
        dx, dy = ctx.to_device(xb), ctx.alloc(M * O * 2)
        ctx.linear_matmul(dl, dx, M, dy)
        assert np.array_equal(dy.download(np.uint16, (M, O)), want), M
        dx.free(); dy.free()
    dl.free()


def test_affine4_gather_and_lookup_bit_exact(orn, ctx):
    rng = np.random.default_rng(3)
    E, O, K, T, k = 16, 256, 512, 3, 4
    lin = util.HostLinear.affine4(rng, E * O, K)
    xb = util.bf16_normal(rng, (T, K))
    lhs = np.repeat(np.arange(T, dtype=np.uint32), k)
    rhs = np.concatenate([rng.permutation(E)[:k] for _ in range(T)]).astype(np.uint32)
    want = np.empty((T * k, O), np.uint16)
    oracle().orc_affine4_gather_qmv(p(lin.w), p(lin.scales), p(lin.biases), E, O, K, p(xb), p(lhs), p(rhs), T * k, p(want))
    d = [ctx.to_device(a) for a in (lin.w, lin.scales, lin.biases, xb, lhs, rhs)]
    dy = ctx.alloc(T * k * O * 2)
    ctx.affine4_gather_qmv(d[0], d[1], d[2], E, O, K, d[3], T, d[4], d[5], T * k, dy)
    assert np.array_equal(dy.download(np.uint16, (T * k, O)), want)
    # the lookup: rows of the same tensors seen as a [E*O, K] table
    table = orn.Linear(orn.LinearStruct(orn.LIN_AFFINE4, E * O, K, orn.KMatrixStruct(), d[0].ptr, d[1].ptr, d[2].ptr), [])
    ids = np.array([0, E * O - 1, 77], np.uint32)
    wout = np.empty((3, K), np.uint16)
    oracle().orc_embedding4(p(lin.w), p(lin.scales), p(lin.biases), K, p(ids), 3, p(wout))
    di, do = ctx.to_device(ids), ctx.alloc(3 * K * 2)
    ctx.embedding(table, di, 3, do)
    assert np.array_equal(do.download(np.uint16, (3, K)), wout)
    for b in d + [dy, di, do]: b.free()


def test_model_with_4bit_affine_modules_matches_oracle(orn, ctx):
    s = synth.SynthModel(dict(synth.TINY, vocab_size=256), seed=31, affine="affine4")
    ws = s.upload(orn, ctx)
    model = orn.TextModel(ctx, ws, s.text_config(orn))
    prompt = np.random.default_rng(1).integers(0, 256, 9).astype(np.uint32)
    caches = model.make_cache(48, 3)
    head = orn.MtpHead(model, ws, 48)
    try:
        ar = orn.generate_step(model, caches, prompt, 14, prefill_step=4)
        caches.reset()
        spec, st = orn.generate_step_mtp(model, head, None, caches, prompt, 2, 14, prefill_step=4)
        o = synth.OracleRun(s, 48)
        want = o.generate(prompt, 14, prefill_step=4)
        o.close()
        assert ar == want and spec == ar
    finally:
        head.close(); caches.close(); model.close(); ws.close()


@pytest.mark.parametrize("T", [1, 2, 4, 9, 150])
def test_moe_block_with_4bit_affine_experts_bit_exact(orn, ctx, T):
    """The published artifact's block: routed and shared experts 4-bit affine group 32, router and
    shared gate 8-bit. Expert ids, scores and output by bits against the oracle. 150 rows: a
    prompt chunk wider than the operator path's 64 rows, taken in blocks."""
    rng = np.random.default_rng(40 + T)
    moe = util.HostMoe(rng, H=1024, E=64, I=256, top_k=8, gate_kind=util.AFFINE4)
    xb = util.bf16_normal(rng, (T, 1024))
    want, winds, wscores, _ = util.orc_moe_block(moe, xb, T)
    w = moe.dev(orn, ctx)
    dx = ctx.to_device(xb)
    out, inds, scores = ctx.alloc(T * 1024 * 2), ctx.alloc(T * 8 * 4), ctx.alloc(T * 8 * 2)
    try:
        # the two fused expert launches (the default), then one launch per operator
        for fuse in (1, 0):
            orn.set_option("fuse_moe", fuse)
            for b in (out, inds, scores): b.zero()
            ctx.moe_block(w, dx, T, out, inds, scores)
            assert np.array_equal(inds.download(np.uint32, (T, 8)), winds), fuse
            assert np.array_equal(scores.download(np.uint16, (T, 8)), wscores), fuse
            assert np.array_equal(out.download(np.uint16, (T, 1024)), want), fuse
    finally:
        orn.set_option("fuse_moe", 1)
        for b in (dx, out, inds, scores): b.free()
        moe.free()


def test_model_in_the_published_artifacts_format_matches_oracle(orn, ctx):
    """Every projection, the routed and shared experts, embed_tokens and lm_head 4-bit affine
    group 32 (routers 8-bit), as the published mlx artifact stores them: both loops, with and
    without a pruned draft head, token for token against the oracle."""
    s = synth.SynthModel(dict(synth.TINY, vocab_size=256), seed=33, affine="affine4", trunk="affine4")
    ws = s.upload(orn, ctx)
    model = orn.TextModel(ctx, ws, s.text_config(orn))
    prompt = np.random.default_rng(2).integers(0, 256, 9).astype(np.uint32)
    caches = model.make_cache(48, 3)
    head = orn.MtpHead(model, ws, 48)
    fr_ids = synth.zipf_frspec_ids(256, 96, seed=3)
    fr = orn.FrSpec(model, ids=fr_ids)
    try:
        ar = orn.generate_step(model, caches, prompt, 14, prefill_step=4)
        o = synth.OracleRun(s, 48)
        want = o.generate(prompt, 14, prefill_step=4)
        o.close()
        assert ar == want
        for frs, frh in ((None, None), (fr, synth.prune_head(s.lm_head, fr_ids))):
            caches.reset()
            head.set_offset(0)
            spec, st = orn.generate_step_mtp(model, head, frs, caches, prompt, 2, 14, prefill_step=4)
            o = synth.OracleRun(s, 48)
            wspec, wst = o.mtp_generate(prompt, 2, 14, fr_ids if frs else None, frh, prefill_step=4)
            o.close()
            assert spec == ar == wspec
            assert (st.cycles, st.drafted, st.accepted) == (wst.cycles, wst.drafted, wst.accepted)
    finally:
        fr.close(); head.close(); caches.close(); model.close(); ws.close()


@pytest.mark.parametrize("gemm_rows,T", [(32, 32), (32, 100), (1, 1), (1, 3), (2, 70), (5, 9)])
def test_affine_block_with_index_outputs_at_every_gemm_rows(orn, ctx, gemm_rows, T):
    """Ids, scores and output of a block over affine experts are the oracle's bits at every setting of gemm_rows,
    from one row on (70 and 100 rows: two blocks), and not asking for the ids changes nothing."""
    rng = np.random.default_rng(60 + T)
    moe = util.HostMoe(rng, H=512, E=64, I=512, top_k=8, gate_kind=util.AFFINE4)
    xb = util.bf16_normal(rng, (T, 512))
    want, winds, wscores, _ = util.orc_moe_block(moe, xb, T)
    w = moe.dev(orn, ctx)
    dx = ctx.to_device(xb)
    out, inds, scores = ctx.alloc(T * 512 * 2), ctx.alloc(T * 8 * 4), ctx.alloc(T * 8 * 2)
    try:
        orn.set_option("gemm_rows", gemm_rows)
        for fuse in (1, 0):
            orn.set_option("fuse_moe", fuse)
            for outs in ((inds, scores), (None, None), (inds, None), (None, scores)):
                for b in (out, inds, scores): b.zero()
                ctx.moe_block(w, dx, T, out, *outs)
                assert np.array_equal(out.download(np.uint16, (T, 512)), want), (fuse, outs)
                if outs[0]: assert np.array_equal(inds.download(np.uint32, (T, 8)), winds), fuse
                if outs[1]: assert np.array_equal(scores.download(np.uint16, (T, 8)), wscores), fuse
    finally:
        orn.set_option("gemm_rows", 32)
        orn.set_option("fuse_moe", 1)
        for b in (dx, out, inds, scores): b.free()
        moe.free()


def test_misaligned_norm_operands_are_refused(orn, ctx):
    """Rows off a 16-byte boundary: an error from the host, with the norm in the head of the launch as with the
    norm in front, for the projections and for the block."""
    rng = np.random.default_rng(8)
    H, T = 2048, 2
    lin = util.HostLinear.affine4(rng, 40, H).dev(orn, ctx)
    moe = util.HostMoe(rng, H=H, E=64, I=512, top_k=8, gate_kind=util.AFFINE4)
    w = moe.dev(orn, ctx)
    bufs = [ctx.alloc(T * H * 2 + 256) for _ in range(7)]
    for b in bufs: b.zero()

    class Off:
        def __init__(self, b): self.ptr = type(b.ptr)(b.ptr.value + 2)

    try:
        for fuse in (1, 0):
            orn.set_option("fuse_norm", fuse)
            for i in range(5):
                res, y, wn, h, nm = (Off(b) if j == i else b for j, b in enumerate(bufs[:5]))
                with pytest.raises(orn.OrnithError, match="aligned"):
                    orn.add_rms_linear_multi(ctx, [lin], res, y, wn, 1e-6, T, h, nm, [bufs[5]])
                with pytest.raises(orn.OrnithError, match="aligned"):
                    orn.add_rms_moe_block(ctx, w, res, y, wn, 1e-6, T, h, nm, bufs[6])
    finally:
        orn.set_option("fuse_norm", 1)
        for b in bufs: b.free()
        lin.free(); moe.free()


def _lin(rng, bits, O, K):
    return (util.HostLinear.affine4 if bits == 4 else util.HostLinear.affine8)(rng, O, K)


def _orc_lin(lin, xb):
    M = xb.shape[0]
    want = np.empty((M, lin.O), np.uint16)
    if lin.mode == "affine4":
        oracle().orc_affine4_gather_qmv(p(lin.w), p(lin.scales), p(lin.biases), 1, lin.O, lin.K, p(xb), None, None, M, p(want))
    else:
        oracle().orc_affine8_qmv(p(lin.w), p(lin.scales), p(lin.biases), lin.O, lin.K, p(xb), M, p(want))
    return want


@pytest.mark.parametrize("K,mats", [
    (1024, [(4, 257), (8, 33)]), (2048, [(4, 1000), (4, 36), (8, 256), (8, 1)]), (4096, [(4, 515), (8, 40)]),
    # more rows than the chip holds at once: a wavefront walks several groups, the last ones ragged
    (2048, [(4, 12289), (8, 9)]), (4096, [(4, 9001)]), (1024, [(4, 30011)]), (2048, [(8, 4099)])])
def test_affine_projections_sharing_a_launch_bit_exact(orn, ctx, K, mats):
    """Both bit widths in one launch, at each width of the kernel and every split of the activation rows over
    it (1 to 9 rows), ragged matrices among them."""
    rng = np.random.default_rng(K + len(mats))
    lins = [_lin(rng, b, O, K) for b, O in mats]
    dls = [l.dev(orn, ctx) for l in lins]
    for M in (1, 2, 3, 4, 5, 9):
        xb = util.bf16_normal(rng, (M, K))
        dx, ys = ctx.to_device(xb), [ctx.alloc(M * l.O * 2) for l in lins]
        ctx.linear_matmul_multi(dls, dx, M, ys)
        for l, y in zip(lins, ys):
            assert np.array_equal(y.download(np.uint16, (M, l.O)), _orc_lin(l, xb)), (M, l.mode, l.O)
        for b in (dx, *ys): b.free()
    for d in dls: d.free()


@pytest.mark.parametrize("mats", [[(4, 40)], [(8, 256), (8, 1)], [(4, 8192), (4, 4096)], [(4, 8192), (4, 513), (4, 512)],
                                  [(4, 12301)]])
def test_affine_projections_with_the_norm_in_their_head_bit_exact(orn, ctx, mats):
    """The residual add and the norm inside the projections' launch (width 2048, one to four rows; five take it in
    front): h, the normed rows and every projection against the oracle's add_rms_norm and mat-vecs."""
    rng = np.random.default_rng(len(mats))
    H = 2048
    lins = [_lin(rng, b, O, H) for b, O in mats]
    dls = [l.dev(orn, ctx) for l in lins]
    wn = util.bf16_normal(rng, (H,))
    dwn = ctx.to_device(wn)
    for M in (1, 2, 3, 4, 5):
        res, y = util.bf16_normal(rng, (M, H)), util.bf16_normal(rng, (M, H))
        wh, wnormed = util.orc_add_rms_norm(res, y, wn)
        bufs = [ctx.to_device(res), ctx.to_device(y), ctx.alloc(M * H * 2), ctx.alloc(M * H * 2)]
        ys = [ctx.alloc(M * l.O * 2) for l in lins]
        orn.add_rms_linear_multi(ctx, dls, bufs[0], bufs[1], dwn, 1e-6, M, bufs[2], bufs[3], ys)
        assert np.array_equal(bufs[2].download(np.uint16, (M, H)), wh) and np.array_equal(bufs[3].download(np.uint16, (M, H)), wnormed), M
        for l, yy in zip(lins, ys):
            assert np.array_equal(yy.download(np.uint16, (M, l.O)), _orc_lin(l, wnormed)), (M, l.mode, l.O)
        for b in bufs + ys: b.free()
    dwn.free()
    for d in dls: d.free()


# (2048, 512): the published artifact's block; 4096, 1024 and 256: the other widths of its kernels; 512 and 320: the
# kernels of any width
@pytest.mark.parametrize("H,I", [(2048, 512), (4096, 256), (1024, 256), (512, 320)])
def test_affine_block_at_every_launch_size_bit_exact(orn, ctx, H, I):
    """1 to 5, 9 and 16 tokens go through every row count a wavefront of the up launch takes (1, 2 and 4 times
    two) and every column count of the down launch (8, 16, 32, 64): ids, scores and output of the operator, and
    the layer's form with the norm in the router's head, by bits."""
    rng = np.random.default_rng(H + I)
    moe = util.HostMoe(rng, H=H, E=64, I=I, top_k=8, gate_kind=util.AFFINE4)
    w = moe.dev(orn, ctx)
    wn = util.bf16_normal(rng, (H,))
    dwn = ctx.to_device(wn)
    for T in (1, 2, 3, 4, 5, 9, 16):
        res, y = util.bf16_normal(rng, (T, H)), util.bf16_normal(rng, (T, H))
        wh, xb = util.orc_add_rms_norm(res, y, wn)
        want, winds, wscores, _ = util.orc_moe_block(moe, xb, T)
        bufs = [ctx.to_device(a) for a in (xb, res, y)] + [ctx.alloc(T * H * 2) for _ in range(3)] + [ctx.alloc(T * 32), ctx.alloc(T * 16)]
        dx, dres, dy, dh, dn, out, inds, scores = bufs
        ctx.moe_block(w, dx, T, out, inds, scores)
        assert np.array_equal(inds.download(np.uint32, (T, 8)), winds) and np.array_equal(scores.download(np.uint16, (T, 8)), wscores), T
        assert np.array_equal(out.download(np.uint16, (T, H)), want), T
        out.zero()
        orn.add_rms_moe_block(ctx, w, dres, dy, dwn, 1e-6, T, dh, dn, out)
        assert np.array_equal(dh.download(np.uint16, (T, H)), wh) and np.array_equal(dn.download(np.uint16, (T, H)), xb), T
        assert np.array_equal(out.download(np.uint16, (T, H)), want), T
        for b in bufs: b.free()
    dwn.free(); moe.free()


@pytest.mark.parametrize("bits,O,K", [(4, 513, 2048), (8, 256, 2048), (4, 2048, 4096)])
def test_affine_linear_is_exact_at_prompt_widths_without_gemms(orn, ctx, bits, O, K):
    """gemm_rows = 0 brings the exact sums back at every width (from 32 rows on the default is a GEMM)."""
    rng = np.random.default_rng(O)
    lin = _lin(rng, bits, O, K)
    dl = lin.dev(orn, ctx)
    M = 70
    xb = util.bf16_normal(rng, (M, K))
    dx, dy = ctx.to_device(xb), ctx.alloc(M * O * 2)
    try:
        orn.set_option("gemm_rows", 0)
        ctx.linear_matmul(dl, dx, M, dy)
        assert np.array_equal(dy.download(np.uint16, (M, O)), _orc_lin(lin, xb))
    finally:
        orn.set_option("gemm_rows", 32)
        for b in (dx, dy): b.free()
        dl.free()
