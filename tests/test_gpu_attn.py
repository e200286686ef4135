"""GPU parity: attention prep (q/k norm + RoPE + KV append) and split-K decode attention
with the output gate vs the oracle, bit for bit."""
import numpy as np
import pytest

import util

pytestmark = pytest.mark.gpu


def _mk(rng, T, Hq, Hkv, hd, cap, offset):
    qg = util.bf16_normal(rng, (T, Hq, 2 * hd)); kx = util.bf16_normal(rng, (T, Hkv, hd)); vx = util.bf16_normal(rng, (T, Hkv, hd))
    qw = util.bf16_normal(rng, (hd,)); kw = util.bf16_normal(rng, (hd,))
    kc = np.zeros((Hkv, cap, hd), np.uint16); vc = np.zeros((Hkv, cap, hd), np.uint16)
    kc[:, :offset] = util.bf16_normal(rng, (Hkv, offset, hd)); vc[:, :offset] = util.bf16_normal(rng, (Hkv, offset, hd))
    # rows past the end hold NaN patterns: nothing may read them
    kc[:, offset + T:] = 0x7FC0; vc[:, offset + T:] = 0x7FC0
    return qg, kx, vx, qw, kw, kc, vc


@pytest.mark.parametrize("T,Hq,Hkv,hd,cap,offset", [
    (1, 16, 2, 256, 4096, 4000), (2, 16, 2, 256, 4096, 255), (4, 16, 2, 256, 4096, 1021),
    # decode widths in short contexts (prep folded into the attention launch): first rows of a
    # cache, new rows across the end of a key block, the widest folded call, head_dim 128
    (1, 16, 2, 256, 4096, 0), (2, 16, 2, 256, 4096, 51), (4, 16, 2, 256, 4096, 254), (8, 16, 2, 256, 4096, 250),
    (8, 16, 2, 256, 4096, 100), (3, 8, 2, 128, 1024, 255), (5, 4, 4, 256, 512, 300),
    (3, 4, 1, 256, 512, 0), (2, 4, 2, 128, 768, 300), (1, 2, 2, 256, 256, 7),
    # many live key blocks: the launch switches to four heads of a KV group a workgroup (same sums)
    (4, 16, 2, 256, 4096, 4000), (4, 16, 2, 128, 4096, 3000),
    # ... with KV groups that are no multiple of four heads (three, one, two, six, five), and of eight (ragged last block)
    (8, 6, 2, 256, 8192, 8000), (4, 16, 16, 256, 2048, 1500), (4, 16, 8, 256, 2048, 1500), (2, 24, 4, 256, 4096, 3000),
    (7, 10, 2, 128, 4096, 3300), (3, 16, 2, 256, 8192, 7000),
    # the 1024-thread form numbered by die: from three blocks on, odd numbers of them, ragged KV groups, new rows across a block's
    # end, as many workgroups a die as it has compute units, and one row more (block fastest, or the other form)
    (1, 16, 2, 256, 4096, 513), (1, 16, 2, 256, 4096, 2300), (2, 16, 2, 256, 4096, 1790), (1, 6, 2, 128, 4096, 3300),
    (3, 5, 1, 256, 2048, 766), (4, 16, 2, 256, 4096, 800), (5, 16, 2, 256, 4096, 700), (1, 16, 16, 256, 2048, 600),
    # eight heads a workgroup: new rows across a block's end, a last block of new rows alone, ragged KV groups (six, five, twelve
    # heads), head width 128, more rows than the prep is done for
    (8, 16, 2, 256, 4096, 2556), (4, 16, 2, 256, 8192, 5120), (8, 12, 2, 256, 4096, 2300), (7, 5, 1, 256, 8192, 6000),
    (4, 24, 2, 128, 4096, 3500), (4, 16, 2, 128, 8192, 5000), (9, 16, 2, 256, 4096, 1900),
    # ... from one workgroup of the other form more than there are compute units: the last call before that, and the first
    (4, 16, 2, 256, 4096, 1020), (4, 16, 1, 128, 4096, 1021),
    # 16-row prompt chunks inside the first key block (one finishing launch, of two rounds from 17 rows on) and across
    # its end (enough rows for the four-head form, which leaves the finishing to the merge launch)
    (16, 16, 2, 256, 4096, 35), (16, 16, 2, 128, 4096, 0), (31, 16, 2, 256, 4096, 200), (31, 17, 1, 256, 4096, 0),
    (16, 16, 2, 256, 4096, 250),
    # the long-context configuration: a depth-3 verify window at the end of a 16384-row cache
    (4, 16, 2, 256, 16384, 16380), (1, 16, 2, 256, 16384, 6621)])
def test_attention_bit_exact(orn, ctx, T, Hq, Hkv, hd, cap, offset):
    rng = np.random.default_rng(T * 1000 + offset)
    qg, kx, vx, qw, kw, kc, vc = _mk(rng, T, Hq, Hkv, hd, cap, offset)
    rd = 64 if hd == 256 else 32
    c, s = util.orc_rope_table(cap, rd, 1e7)
    dc, ds = ctx.rope_table(cap, rd, 1e7)
    assert np.array_equal(dc.download(np.float32, c.shape), c) and np.array_equal(ds.download(np.float32, s.shape), s)
    d = [ctx.to_device(a) for a in (qg, kx, vx, qw, kw)]
    dkc, dvc = ctx.to_device(kc), ctx.to_device(vc)
    dq, dout = ctx.alloc(T * Hq * hd * 2), ctx.alloc(T * Hq * hd * 2)
    wkc, wvc = kc.copy(), vc.copy()
    wq, wgate = util.orc_attn_prep(qg, kx, vx, qw, kw, rd, c, s, offset, wkc, wvc)
    want = util.orc_sdpa(wq, wkc, wvc, wgate, offset, hd ** -0.5)
    for use_dev_offset in (False, True):
        doff = ctx.to_device(np.array([offset], np.int32)) if use_dev_offset else None
        dkc.upload(kc); dvc.upload(vc)
        ctx.attn_prep(*d, T, Hq, Hkv, hd, rd, 1e-6, dc, ds, cap, 0 if use_dev_offset else offset, cap, dq, dkc, dvc, d_offset=doff)
        assert np.array_equal(dq.download(np.uint16, wq.shape), wq)
        assert np.array_equal(dkc.download(np.uint16, kc.shape), wkc) and np.array_equal(dvc.download(np.uint16, vc.shape), wvc)
        ctx.sdpa_decode_gated(dq, dkc, dvc, d[0], T, Hq, Hkv, hd, 0 if use_dev_offset else offset, cap, hd ** -0.5, dout, d_offset=doff)
        assert np.array_equal(dout.download(np.uint16, want.shape), want), use_dev_offset
        if doff: doff.free()
    # prep + attention as one call (one launch at decode widths in short contexts, a prep launch
    # first otherwise; with the fold switched off it is always two): same output, same caches
    for fold in (1, 0):
        orn.set_option("fuse_attn_prep", fold)
        dkc.upload(kc); dvc.upload(vc); dout.zero(); dq.zero()
        ctx.attn_decode(*d, T, Hq, Hkv, hd, rd, 1e-6, dc, ds, cap, offset, cap, hd ** -0.5, dq, dkc, dvc, dout)
        assert np.array_equal(dout.download(np.uint16, want.shape), want), ("attn_decode", fold)
        assert np.array_equal(dkc.download(np.uint16, kc.shape), wkc) and np.array_equal(dvc.download(np.uint16, vc.shape), wvc), fold
        # the rotated queries: of every form but the folded one of a head a workgroup (as many as are one round of a 256-unit device)
        blocks = (offset + T - 1) // 256 + 1
        if not fold or T > 8 or blocks * Hq * T > (512 if blocks == 1 else 256):
            assert np.array_equal(dq.download(np.uint16, wq.shape), wq), ("rotated queries", fold)
    orn.set_option("fuse_attn_prep", 1)
    for b in d + [dkc, dvc, dq, dout, dc, ds]: b.free()


@pytest.mark.parametrize("cache_off,vx_off", [(8, 0), (0, 4), (8, 4)])
def test_attention_of_less_aligned_operands(orn, ctx, cache_off, vx_off):
    """Caches that are aligned to 8 bytes only, raw value rows to 4, at a size of the eight-head form: the same bits as aligned ones
    (without them the caches' rows could not go to LDS 16 bytes a lane)"""
    import ctypes as C
    T, Hq, Hkv, hd, cap, offset, rd = 4, 16, 2, 256, 4096, 2554, 64
    rng = np.random.default_rng(5)
    qg, kx, vx, qw, kw, kc, vc = _mk(rng, T, Hq, Hkv, hd, cap, offset)
    c, s = util.orc_rope_table(cap, rd, 1e7)
    dc, ds = ctx.rope_table(cap, rd, 1e7)
    wkc, wvc = kc.copy(), vc.copy()
    wq, wgate = util.orc_attn_prep(qg, kx, vx, qw, kw, rd, c, s, offset, wkc, wvc)
    want = util.orc_sdpa(wq, wkc, wvc, wgate, offset, hd ** -0.5)

    class At:                                         # a device address some bytes into a buffer
        def __init__(self, a, off):
            self.a, self.off = a, off
            self.buf = ctx.alloc(a.nbytes + 16)
            self.buf.upload(self.bytes(a))
            self.ptr = C.c_void_p(self.buf.ptr.value + off)

        def bytes(self, a):
            return np.concatenate([np.zeros(self.off, np.uint8), a.reshape(-1).view(np.uint8), np.zeros(16 - self.off, np.uint8)])

        def get(self):
            return self.buf.download(np.uint8, self.a.nbytes + 16)[self.off:self.off + self.a.nbytes].view(np.uint16).reshape(self.a.shape)

    d = [At(qg, 0), At(kx, 0), At(vx, vx_off), At(qw, 0), At(kw, 0)]
    dk, dv, dq, dout = At(kc, cache_off), At(vc, cache_off), ctx.alloc(T * Hq * hd * 2), ctx.alloc(T * Hq * hd * 2)
    ctx.attn_decode(*d, T, Hq, Hkv, hd, rd, 1e-6, dc, ds, cap, offset, cap, hd ** -0.5, dq, dk, dv, dout)
    assert np.array_equal(dout.download(np.uint16, want.shape), want)
    assert np.array_equal(dq.download(np.uint16, wq.shape), wq)
    assert np.array_equal(dk.get(), wkc) and np.array_equal(dv.get(), wvc)
    for b in [x.buf for x in d + [dk, dv]] + [dq, dout, dc, ds]: b.free()


# the matrix-core forms (four heads a workgroup, and eight; groups of eight and of three heads, head widths 256 and 128) and the
# 1024-thread one, inside the first key block and past it
@pytest.mark.parametrize("T,Hq,Hkv,hd,cap,offset", [(4, 16, 2, 256, 4096, 2500), (4, 16, 2, 128, 4096, 3000), (8, 6, 2, 256, 8192, 8000),
                                                    (2, 16, 2, 256, 4096, 51), (2, 16, 2, 256, 4096, 600), (8, 16, 2, 256, 4096, 2300)])
def test_attention_special_values(orn, ctx, T, Hq, Hkv, hd, cap, offset):
    """Subnormal keys and values, score products below the normal range, infinities and NaNs in keys and values:
    the oracle's values, NaN for NaN."""
    rng = np.random.default_rng(offset)
    q, gate = util.bf16_normal(rng, (T, Hq, hd)), util.bf16_normal(rng, (T, Hq, hd))
    k0, v0 = (rng.standard_normal((Hkv, cap, hd)).astype(np.float32) for _ in range(2))
    dq, dg, out = ctx.to_device(q), ctx.to_device(np.concatenate([np.zeros_like(gate), gate], -1)), ctx.alloc(T * Hq * hd * 2)
    dk, dv = ctx.alloc(k0.size * 2), ctx.alloc(v0.size * 2)

    def values(v): v[0, 3, 5], v[0, 4, 6], v[0, 9, 6], v[1, 7, 1] = np.inf, np.inf, -np.inf, np.nan
    cases = {"subnormal values": lambda k, v: v.__imul__(np.float32(1e-39)),
             "subnormal keys": lambda k, v: k.__imul__(np.float32(1e-39)),
             "products below the normal range": lambda k, v: k.__imul__(np.float32(1e-37)),
             "infinite and NaN values": lambda k, v: values(v),
             "an infinite key": lambda k, v: k[0, 3].fill(np.inf),
             "a key of minus infinity": lambda k, v: k[0, 7, :1].fill(-np.inf),
             "a NaN key": lambda k, v: k[0, 3, :1].fill(np.nan)}
    for name, change in cases.items():
        k, v = k0.copy(), v0.copy()
        change(k, v)
        kb, vb = util.f32_to_bf16(k), util.f32_to_bf16(v)
        dk.upload(kb); dv.upload(vb)
        ctx.sdpa_decode_gated(dq, dk, dv, dg, T, Hq, Hkv, hd, offset, cap, hd ** -0.5, out)
        want = util.orc_sdpa(q, kb, vb, gate, offset, hd ** -0.5)
        assert util.same_values(out.download(np.uint16, want.shape), want), name
        assert not np.isnan(util.bf16_to_f32(want)).all(), name
    for b in (dq, dg, out, dk, dv): b.free()
