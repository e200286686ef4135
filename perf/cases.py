"""The work a user of this library has it do, as cases that can be timed and compared.

Four families, all through the public entry points of the binding package:

  decode    a whole short request: reset the caches, take a prompt of a few tokens and generate.
            `generate_step` (depth 0) or `generate_step_mtp` (speculative, FR-Spec draft head) on
            the full 40-layer model, in either weight format, greedy or sampled.
  prefill   a prompt of `rows` tokens through the same model in one forward call
            (`ornith_model_forward` on device ids, post-norm hidden rows out).
  ops       the operators an engine of its own would call one by one: the k-quant mat-vec, the
            sparse MoE block, one gated-delta layer step, attention over a long cache.

Formats: "kq" is the k-quant artifact (Q4_K / Q6_K projections and experts, 8-bit embedding),
"affine4" the published one (4-bit affine group 32 everywhere, 8-bit router); the MTP head is
dense bf16 in both. Weights are random-init of the Qwen3.5-35B-A3B shape with zero mean and
outputs of unit variance, the projections that end a branch scaled down so that no single layer
outweighs the residual stream. A program loads its model once and
serves many requests with it: the models live as long as the process, and a case's seed makes the
prompt, the sampler's stream and the operators' inputs.
"""
import ctypes as C
import importlib
import math

import numpy as np
import torch

orn = importlib.import_module("ornith-rs_amd")

CFG = orn.TextConfig.qwen35_35b_a3b()
H, E, I, V, TOP_K, LAYERS = 2048, 256, 512, 248320, 8, 40
CONV, HK, HV, DK, HQ, HKV, HD = 8192, 16, 32, 128, 16, 2, 256
FRSPEC_IDS = 32768
MAX_ROWS = 8192            # a prompt of up to this many tokens goes through in one call
BRANCH = 0.03              # size of what one branch adds to a residual stream of unit size (scaled init of deep stacks)
DRAFT_HIT = 0.65           # share of drafts that the trunk agrees with, as on ordinary text


# ---- cases ---------------------------------------------------------------------------------
def listed():
    return [
        # the smallest calls: one projection (a gated-delta layer's last) for four verify rows
        dict(name="matvec-q4k-2048x4096", op="matvec", kind="q4k", O=2048, K=4096, M=4, dtype="bf16"),
        # one MoE block at the verify width of depth-1 speculation
        dict(name="moe-block-2", op="moe", rows=2, layer=7),
        # one gated-delta layer at the same width, with a state snapshot for every row
        dict(name="gdn-layer-2", op="gdn", rows=2),
        # a depth-3 verify window at the end of a long conversation
        dict(name="attention-4-at-6621", op="attention", rows=4, context=6621),
        # chat without speculation
        dict(name="decode-greedy", op="decode", format="kq", depth=0, prompt=13, tokens=64, sampler="greedy"),
        # the usual setting: depth-1 speculation with the reduced draft vocabulary
        dict(name="decode-mtp1-greedy", op="decode", format="kq", depth=1, prompt=13, tokens=64, sampler="greedy"),
        # sampled, depth 3, probability-ratio acceptance
        dict(name="decode-mtp3-sampled", op="decode", format="kq", depth=3, prompt=16, tokens=40, sampler="ratio"),
        # the published 4-bit artifact
        dict(name="decode-affine4-mtp1", op="decode", format="affine4", depth=1, prompt=9, tokens=48, sampler="greedy"),
        # a question, a page, a long document
        dict(name="prefill-51", op="prefill", format="kq", rows=51),
        dict(name="prefill-700", op="prefill", format="kq", rows=700),
        dict(name="prefill-6621", op="prefill", format="kq", rows=6621),
        # a page through the published artifact
        dict(name="prefill-affine4-600", op="prefill", format="affine4", rows=600),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    family = rng.choice(["matvec", "moe", "gdn", "attention", "decode", "decode", "prefill", "prefill", "prefill4"])
    if family == "matvec":
        # projections of one to sixteen rows, down to a single head and up to the pruned lm_head
        return dict(op="matvec", kind=rng.choice(["q4k", "q6k"]), O=_log(rng, 64, 32768), K=rng.choice([512, 1024, 2048, 4096]),
                    M=rng.randint(1, 16), dtype=rng.choice(["f32", "bf16"]))
    if family == "moe":
        return dict(op="moe", rows=rng.choice([1, 2, 3, 4, 5, 8, 9, 16]), layer=rng.randrange(LAYERS))
    if family == "gdn":
        return dict(op="gdn", rows=rng.randint(1, 16))
    if family == "attention":
        return dict(op="attention", rows=rng.randint(1, 9), context=_log(rng, 8, 16300))
    if family == "decode":
        depth = rng.randint(0, 4)
        return dict(op="decode", format=rng.choice(["kq", "kq", "affine4"]), depth=depth, prompt=rng.randint(1, 16),
                    tokens=_log(rng, 12, 64), sampler=rng.choice(["greedy", "greedy", "top_p", "ratio"]))
    if family == "prefill":
        return dict(op="prefill", format="kq", rows=_log(rng, 17, 6621))
    return dict(op="prefill", format="affine4", rows=_log(rng, 17, 600))


# ---- what a pass cannot do without ---------------------------------------------------------------
BITS = {"q4k": 144 / 256, "q6k": 210 / 256, "affine4": 0.625, "affine8": 1 + 4 / 64, "bf16": 2.0}
GDN_W = (CONV + HV * DK) * H + H * HV * DK       # qkv + z, out
ATT_W = (2 * HQ * HD + 2 * HKV * HD) * H + H * HQ * HD
STATE = HV * DK * DK * 4


def _distinct(rows):
    """Experts that `rows` tokens of independent routing touch, on average."""
    return E * (1.0 - (1.0 - TOP_K / E) ** rows)


def _trunk(fmt, rows):
    """(weight bytes, operations) of one forward call of `rows` tokens, without the output head."""
    kq = fmt == "kq"
    lo, hi = BITS["q4k" if kq else "affine4"], BITS["q6k" if kq else "affine4"]
    ex = I * H * (2 * lo + hi)
    moe = (_distinct(rows) + 1) * ex + E * H * BITS["q6k" if kq else "affine8"] + H * 1.06
    nbytes = 30 * (GDN_W * lo + 2 * HV * H * 2) + 10 * ATT_W * hi + 40 * moe
    ops = 2.0 * rows * (30 * (GDN_W + 2 * HV * H) + 10 * ATT_W + 40 * (E * H + (TOP_K + 1) * 3 * I * H))
    ops += 30 * rows * HV * DK * DK * 8.0 + 10 * rows * rows * HQ * HD * 2.0
    return nbytes, ops


def work(case):
    op = case["op"]
    if op == "matvec":
        es = 4 if case["dtype"] == "f32" else 2
        n = case["O"] * case["K"]
        return {"bytes": n * BITS[case["kind"]] + case["M"] * (case["O"] + case["K"]) * es, "flops": 2.0 * n * case["M"]}
    if op == "moe":
        T = case["rows"]
        ex = I * H * (2 * BITS["q4k"] + BITS["q6k"])
        return {"bytes": (_distinct(T) + 1) * ex + E * H * BITS["q6k"] + T * H * 4 + T * TOP_K * 6,
                "flops": 2.0 * T * (E * H + (TOP_K + 1) * 3 * I * H)}
    if op == "gdn":
        T = case["rows"]
        return {"bytes": GDN_W * BITS["q4k"] + 2 * HV * H * 2 + STATE * (1 + T) + T * (2 * H + CONV) * 2 + 4 * CONV * 2,
                "flops": 2.0 * T * (GDN_W + 2 * HV * H) + T * HV * DK * DK * 8.0}
    if op == "attention":
        T, n = case["rows"], case["context"] + case["rows"]
        return {"bytes": 2 * HKV * n * HD * 2 + T * (3 * HQ + 4 * HKV) * HD * 2, "flops": 4.0 * T * n * HQ * HD}
    if op == "prefill":
        nbytes, ops = _trunk(case["format"], case["rows"])
        return {"bytes": nbytes + 30 * STATE + 10 * 2 * HKV * case["rows"] * HD * 2 + case["rows"] * (4 + 2 * H), "flops": ops}
    # decode: the prompt, then a cycle of depth + 1 verified rows for every 1 + accepted tokens
    d, fmt = case["depth"], case["format"]
    per_cycle = 1.0 + (sum(DRAFT_HIT ** (i + 1) for i in range(d)) if case["sampler"] == "greedy" else 0.0)
    cycles = case["tokens"] / per_cycle
    b0, f0 = _trunk(fmt, case["prompt"])
    b1, f1 = _trunk(fmt, d + 1)
    head = V * H * BITS["q4k" if fmt == "kq" else "affine4"]
    draft = 2.0 * (2 * H * H + ATT_W + E * H + (TOP_K + 1) * 3 * I * H) + FRSPEC_IDS * H * BITS["q4k" if fmt == "kq" else "affine4"]
    state = 30 * STATE * (2 + d)
    return {"bytes": b0 + head + cycles * (b1 + head + state + d * draft),
            "flops": f0 + cycles * (f1 + 2.0 * (d + 1) * V * H + d * draft)}


def tolerance(case):
    if case["op"] == "prefill":
        # bf16 activations and weights rounded to bf16 on the way to the matrix cores, through 40
        # layers: two orders of summation differ by 0.006 to 0.008; a router tie that falls the
        # other way changes single rows (hence max)
        return {"rel": 0.015, "max": 0.5}
    return "exact"         # token ids, and bf16 / fp32 results whose order of summation is fixed


# ---- models ---------------------------------------------------------------------------------------
class _Buf:
    """A torch tensor where the binding expects one of its device buffers."""

    def __init__(self, t):
        self.t, self.ptr = t, C.c_void_p(t.data_ptr())


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _bytes(g, shape):
    return torch.randint(0, 256, shape, generator=g, device="cuda", dtype=torch.uint8)


def _normal(g, shape, std=1.0, mean=0.0):
    return (torch.randn(shape, generator=g, device="cuda") * std + mean).to(torch.bfloat16)


def _kquant(g, kind, lead, K, gain=1.0):
    """(codes, scales, dm) of [lead, K] weights: fields drawn directly, weights zero-mean."""
    nb = K // 256
    if kind == "q4k":
        sc = torch.randint(0, 64, lead + (nb, 8), generator=g, device="cuda", dtype=torch.uint8)
        lo, hi = sc[..., :4], sc[..., 4:]
        # scale and minimum of a sub-block are the same six bits; dmin = 7.5 d centres the codes
        top = (hi >> 4) << 6
        scales = torch.cat([lo | top, lo | top, (hi & 15) | ((hi & 15) << 4)], -1)
        d = torch.randn(lead + (nb,), generator=g, device="cuda").abs() * gain / (168.3 * math.sqrt(K))
        return _bytes(g, lead + (nb * 128,)), scales, torch.stack([d, 7.5 * d], -1).to(torch.float16)
    scales = torch.randint(-64, 64, lead + (nb, 16), generator=g, device="cuda", dtype=torch.int8).view(torch.uint8)
    d = torch.randn(lead + (nb, 1), generator=g, device="cuda").abs() * gain / (682.9 * math.sqrt(K))
    return _bytes(g, lead + (nb * 192,)), scales, d.to(torch.float16)


def _affine(g, bits, lead, K, gain=1.0):
    group = 64 if bits == 8 else 32
    spread, half = (73.9, 127.5) if bits == 8 else (4.61, 7.5)
    s = (torch.rand(lead + (K // group,), generator=g, device="cuda") + 0.5) * gain / (spread * math.sqrt(K))
    s = s.to(torch.bfloat16)
    return _bytes(g, lead + (K * bits // 8,)), s, (s.float() * -half).to(torch.bfloat16)


def _host(t):
    """A device tensor as numpy (bf16 and f16 as their bits)."""
    if t.dtype in (torch.bfloat16, torch.float16):
        t = t.view(torch.int16)
    a = t.cpu().numpy()
    return a.view(np.uint16) if a.dtype == np.int16 else a


class _Loader:
    def __init__(self, ctx, fmt, seed):
        self.ws, self.fmt, self.g = orn.WeightStore(ctx), fmt, _gen(seed)
        self.stage = torch.empty(E * I * H, dtype=torch.uint8, pin_memory=True)

    def put(self, name, t, code, view=None):
        raw = t.contiguous().reshape(-1).view(torch.uint8)
        if raw.numel() <= self.stage.numel():          # through pinned memory, one copy each way
            self.stage[:raw.numel()].copy_(raw)
            a = self.stage[:raw.numel()].numpy()
        else:
            a = raw.cpu().numpy()
        shape = tuple(t.shape)
        if view is not None:
            a, shape = a.view(view), shape[:-1] + (shape[-1] // np.dtype(view).itemsize,)
        else:
            a = a.view({orn.DT_BF16: np.uint16, orn.DT_F16: np.uint16, orn.DT_U8: np.uint8}[code])
        self.ws.put(name, a.reshape(shape), code)

    def linear(self, path, kind, O, K, lead=(), gain=1.0):
        if kind == "bf16":
            self.put(path + ".weight", _normal(self.g, lead + (O, K), gain / math.sqrt(K)), orn.DT_BF16)
        elif kind.startswith("affine"):
            w, s, b = _affine(self.g, int(kind[-1]), lead + (O,), K, gain)
            self.put(path + ".weight", w, orn.DT_U32, np.uint32)
            self.put(path + ".scales", s, orn.DT_BF16)
            self.put(path + ".biases", b, orn.DT_BF16)
        else:
            q, s, d = _kquant(self.g, kind, lead + (O,), K, gain)
            self.put(path + ".weight", q, orn.DT_U32, np.uint32)
            self.put(path + ".scales", s, orn.DT_U8)
            self.put(path + ".dm", d, orn.DT_F16)

    def norm(self, name, n):
        self.put(name, _normal(self.g, (n,), 0.1, 1.0), orn.DT_BF16)

    def attention(self, p, kind):
        self.linear(p + "q_proj", kind, 2 * HQ * HD, H)
        self.linear(p + "k_proj", kind, HKV * HD, H)
        self.linear(p + "v_proj", kind, HKV * HD, H)
        self.linear(p + "o_proj", kind, H, HQ * HD, gain=BRANCH)
        self.norm(p + "q_norm.weight", HD)
        self.norm(p + "k_norm.weight", HD)

    def moe(self, p, router, up, down, egate):
        self.linear(p + "gate", router, E, H)
        self.linear(p + "switch_mlp.gate_proj", up, I, H, (E,))
        self.linear(p + "switch_mlp.up_proj", up, I, H, (E,))
        self.linear(p + "switch_mlp.down_proj", down, H, I, (E,), BRANCH)
        self.linear(p + "shared_expert.gate_proj", up, I, H)
        self.linear(p + "shared_expert.up_proj", up, I, H)
        self.linear(p + "shared_expert.down_proj", down, H, I, gain=BRANCH)
        self.linear(p + "shared_expert_gate", egate, 1, H)

    def model(self):
        kq, P = self.fmt == "kq", "language_model.model."
        lo, hi, emb = ("q4k", "q6k", "affine8") if kq else ("affine4", "affine4", "affine4")
        self.linear(P + "embed_tokens", emb, V, H, gain=math.sqrt(H))
        self.linear("language_model.lm_head", lo, V, H)
        self.norm(P + "norm.weight", H)
        for i in range(LAYERS):
            p = P + "layers.%d." % i
            self.norm(p + "input_layernorm.weight", H)
            self.norm(p + "post_attention_layernorm.weight", H)
            if CFG.is_linear(i):
                g = p + "linear_attn."
                self.linear(g + "in_proj_qkv", lo, CONV, H)
                self.linear(g + "in_proj_z", lo, HV * DK, H)
                self.linear(g + "out_proj", lo, H, HV * DK, gain=BRANCH)
                self.linear(g + "in_proj_a", "bf16", HV, H)
                self.linear(g + "in_proj_b", "bf16", HV, H)
                self.put(g + "conv1d.weight", _normal(self.g, (CONV, 4, 1), 0.5), orn.DT_BF16)
                self.put(g + "dt_bias", _normal(self.g, (HV,), 0.5), orn.DT_BF16)
                self.put(g + "A_log", _normal(self.g, (HV,), 0.5), orn.DT_BF16)
                self.norm(g + "norm.weight", DK)
            else:
                self.attention(p + "self_attn.", hi)
            self.moe(p + "mlp.", "q6k" if kq else "affine8", lo, hi, emb)
        for n in ("pre_fc_norm_embedding", "pre_fc_norm_hidden", "norm"):
            self.norm("mtp.%s.weight" % n, H)
        m = "mtp.layers.0."
        self.norm(m + "input_layernorm.weight", H)
        self.norm(m + "post_attention_layernorm.weight", H)
        self.linear("mtp.fc", "bf16", H, 2 * H)
        self.attention(m + "self_attn.", "bf16")
        self.moe(m + "mlp.", "bf16", "bf16", "bf16", "bf16")
        torch.cuda.synchronize()
        return self.ws


_ctx = None
_models = {}


def _context():
    global _ctx
    if _ctx is None:
        _ctx = orn.Ctx(0)
    return _ctx


def _model(fmt):
    """(model, weights, FR-Spec head) of a format, loaded on first use."""
    if fmt not in _models:
        ws = _Loader(_context(), fmt, 1 if fmt == "kq" else 2).model()
        model = orn.TextModel(_context(), ws, CFG)
        model.set_max_rows(MAX_ROWS)
        ids = np.random.default_rng(1).permutation(V)[:FRSPEC_IDS].astype(np.uint32)
        _models[fmt] = (model, ws, orn.FrSpec(model, ids=ids))
        torch.cuda.empty_cache()
    return _models[fmt]


# ---- prepare and run --------------------------------------------------------------------------------
class _State:
    """What a request keeps; the library's objects in it are closed with it."""

    def __init__(self, case):
        self.case, self.close = case, []

    def __del__(self):
        for o in self.close:
            (o.close if hasattr(o, "close") else o.free)()


def _sampler(kind, seed):
    if kind == "greedy":
        return orn.Sampler.greedy()
    accept, rng = (orn.ACCEPT_RATIO, orn.RNG_PHILOX) if kind == "ratio" else (orn.ACCEPT_EQUALITY, orn.RNG_THREEFRY)
    return orn.Sampler(1, 0.8, 0.95, 0, seed, accept, rng)


def prepare(case, seed):
    s = _State(case)
    {"matvec": _prep_matvec, "moe": _prep_moe, "gdn": _prep_gdn, "attention": _prep_attention, "decode": _prep_decode,
     "prefill": _prep_prefill}[case["op"]](s, case, seed)
    return s


def run(s):
    return {"matvec": _run_matvec, "moe": _run_moe, "gdn": _run_gdn, "attention": _run_attention, "decode": _run_decode,
            "prefill": _run_prefill}[s.case["op"]](s)


def _empty(shape, dtype=torch.bfloat16):
    return _Buf(torch.empty(shape, device="cuda", dtype=dtype))


def _prep_matvec(s, c, seed):
    g, ctx = _gen(seed), _context()
    q, sc, d = _kquant(g, c["kind"], (c["O"],), c["K"])
    s.w = orn.KMatrix(ctx, orn.Q4K if c["kind"] == "q4k" else orn.Q6K, _host(q), _host(sc), _host(d), 1, c["O"], c["K"])
    s.close.append(s.w)
    dt, s.dt = (torch.float32, orn.F32) if c["dtype"] == "f32" else (torch.bfloat16, orn.BF16)
    s.x = _Buf(torch.randn((c["M"], c["K"]), generator=g, device="cuda").to(dt))
    s.y = _empty((c["M"], c["O"]), dt)


def _run_matvec(s):
    _ctx.kq_qmv(s.w, s.x, s.dt, s.case["M"], s.y, s.dt)
    return s.y.t


def _prep_moe(s, c, seed):
    T = c["rows"]
    s.w = _model("kq")[0].moe_weights(c["layer"])
    s.x = _Buf(_normal(_gen(seed), (T, H)))
    s.out, s.inds, s.scores = _empty((T, H)), _empty((T, TOP_K), torch.int32), _empty((T, TOP_K))


def _run_moe(s):
    _ctx.moe_block(s.w, s.x, s.case["rows"], s.out, s.inds, s.scores)
    return [s.out.t, s.inds.t, s.scores.t]


def _prep_gdn(s, c, seed):
    g, ctx, T = _gen(seed), _context(), c["rows"]

    def lin(O, K):
        l = orn.Linear.kquant(ctx, orn.Q4K, *[_host(t) for t in _kquant(g, "q4k", (O,), K)], O, K)
        s.close.append(l)
        return l

    s.qkv_w, s.z_w, s.out_w = lin(CONV, H), lin(HV * DK, H), lin(H, HV * DK)
    s.x, s.conv, s.cw = _Buf(_normal(g, (T, H))), _Buf(_normal(g, (3, CONV))), _Buf(_normal(g, (CONV, 4), 0.5))
    s.wa, s.wb = _Buf(_normal(g, (HV, H), H ** -0.5)), _Buf(_normal(g, (HV, H), H ** -0.5))
    s.a_log, s.dt, s.nw = _Buf(_normal(g, (HV,), 0.5)), _Buf(_normal(g, (HV,), 0.5)), _Buf(_normal(g, (DK,), 0.1, 1.0))
    s.S0 = _Buf(torch.randn((HV, DK, DK), generator=g, device="cuda") * 0.1)
    s.qkv, s.z, s.gated, s.r = _empty((T, CONV)), _empty((T, HV * DK)), _empty((T, HV * DK)), _empty((T, H))
    s.snaps, s.window = _empty((T, HV, DK, DK), torch.float32), _empty((3 + T, CONV))


def _run_gdn(s):
    T = s.case["rows"]
    _ctx.linear_matmul_multi([s.qkv_w, s.z_w], s.x, T, [s.qkv, s.z])
    orn.gdn_step(_ctx, s.conv, s.qkv, s.cw, s.wa, s.wb, s.x, H, s.a_log, s.dt, T, 4, HK, DK, HV, DK, s.S0, s.snaps, True,
                 s.nw, s.z, s.window, s.gated)
    _ctx.linear_matmul(s.out_w, s.gated, T, s.r)
    return [s.r.t, s.snaps.t, s.window.t]


def _prep_attention(s, c, seed):
    g, ctx, T, n = _gen(seed), _context(), c["rows"], c["context"]
    s.cap = (n + T + 255) // 256 * 256
    s.cos, s.sin = ctx.rope_table(s.cap, 64, 1e7)
    s.close += [s.cos, s.sin]
    s.qg, s.kx, s.vx = (_Buf(_normal(g, (T, w))) for w in (2 * HQ * HD, HKV * HD, HKV * HD))
    s.qw, s.kw = _Buf(_normal(g, (HD,), 0.1, 1.0)), _Buf(_normal(g, (HD,), 0.1, 1.0))
    s.k, s.v = _Buf(_normal(g, (HKV, s.cap, HD))), _Buf(_normal(g, (HKV, s.cap, HD)))
    s.q, s.out = _empty((T, HQ * HD)), _empty((T, HQ * HD))


def _run_attention(s):
    T, n = s.case["rows"], s.case["context"]
    _ctx.attn_decode(s.qg, s.kx, s.vx, s.qw, s.kw, T, HQ, HKV, HD, 64, 1e-6, s.cos, s.sin, s.cap, n, s.cap, HD ** -0.5,
                     s.q, s.k, s.v, s.out)
    return [s.out.t, s.k.t[:, n:n + T], s.v.t[:, n:n + T]]      # the output and the rows it appended


def _prep_decode(s, c, seed):
    s.model, ws, s.fr = _model(c["format"])
    d, n = c["depth"], c["prompt"] + c["tokens"] + c["depth"] + 2
    s.caches = s.model.make_cache(n, d + 1)
    s.close.append(s.caches)
    rng = np.random.default_rng(seed)
    s.prompt = rng.integers(0, V, c["prompt"]).astype(np.uint32)
    s.sampler = _sampler(c["sampler"], seed)
    s.head = None
    if d:
        s.head = orn.MtpHead(s.model, ws, c["tokens"] + d + 2)
        s.close.append(s.head)
        if c["sampler"] == "greedy":
            # random weights would never agree with their own head: hand the loop drafts of which
            # as many are right as a trained head's are
            script = np.array(orn.generate_step(s.model, s.caches, s.prompt, c["tokens"]), np.uint32)
            wrong = rng.random(len(script)) >= DRAFT_HIT
            script[wrong] = (script[wrong] + 1) % V
            s.head.force_drafts(script)


def _run_decode(s):
    c = s.case
    s.caches.reset()
    if not c["depth"]:
        return np.array(orn.generate_step(s.model, s.caches, s.prompt, c["tokens"], s.sampler), np.int64)
    toks, st = orn.generate_step_mtp(s.model, s.head, s.fr, s.caches, s.prompt, c["depth"], c["tokens"], s.sampler)
    return [np.array(toks, np.int64), np.array([st.cycles, st.drafted, st.accepted], np.int64)]


def _prep_prefill(s, c, seed):
    s.model = _model(c["format"])[0]
    s.caches = s.model.make_cache(c["rows"] + 64, 4)
    s.close.append(s.caches)
    s.ids = torch.randint(0, V, (c["rows"],), generator=_gen(seed), device="cuda", dtype=torch.int32)
    s.hidden = torch.empty((c["rows"], H), device="cuda", dtype=torch.bfloat16)


def _run_prefill(s):
    s.caches.reset()
    rc = orn.lib().ornith_model_forward(s.model.h, s.caches.h, C.c_void_p(s.ids.data_ptr()), s.case["rows"], 0,
                                        C.c_void_p(s.hidden.data_ptr()))
    if rc:
        raise orn.OrnithError(orn.lib().ornith_last_error().decode())
    return s.hidden
