"""Measured cases: the calls a program that serves a model with this library makes, at the sizes it makes them.

Each case is one pass through the public entry points (the C ABI of include/*.h through wzy_amd), with
weights and workspaces laid out once as a serving program keeps them.  The kinds:

  gdn          the attention half of one gated-delta-rule layer of a decode step or verify window:
               hyper-connection read, grouped input projections, delta-rule step, output projection
  qsa          the attention half of one sparse-attention layer: grouped projections, norms + RoPE + INT8
               KV and indexer append, block scores + top-2048, attention, output projection
  moe          the mixture-of-experts block of a decode step or verify window
  head         the LM head of a decode step or verify window and its argmax / top-16
  gemm         one dense projection of a prefill chunk
  moe_prefill  the mixture-of-experts block of a prefill chunk
  decode       a decode step (T = 1) or verify window (T > 1) of a whole stage, logits read back
  prefill      a prompt through the chunked prefill of a whole stage up to its first logits

Shapes: "base" is the synthetic benchmark model (n_embd 2048, 512 experts top-10 of 512, vocab 151,936),
"wide" the same blocks at n_embd 2560, n_ff 640, vocab 248,320.  Stages run 2 or 4 layers instead of 48
and a 32,768-row vocabulary, so that the head's share of a step stays small, as it is at 48 layers.  A
prompt's logits are those of its last token, a decode step after the chunk: they see the chunk through the
state it left, so a stage of two layers shows what the first layer's blocks computed for every row.
"""
import ctypes as C
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "wzy-flash-serve_amd"))
import wzy_amd  # noqa: E402

DEV = "cuda"
HC, LR, EPS = 4, 320, 1e-6
SHAPES = {"base": dict(D=2048, F=512), "wide": dict(D=2560, F=640)}
HK, E, K = 16, 512, 10                            # GDN key heads of 128; experts, experts per token
QH, KVH, HD, NROT, IH, IDIM, BLK, TOPK = 24, 2, 256, 64, 4, 128, 4, 2048
QD, KVD = QH * HD, KVH * HD
STAGE_VOCAB = 32768
# dense projections of a prefill chunk: N, K, weights
PROJ = {"gdn_qkv": (6144, 2048, "q8"), "gdn_out": (2048, 2048, "q8"), "qsa_q": (12288, 2048, "q8"),
        "qsa_out": (2048, 6144, "q8"), "hc_down": (320, 8192, "q8"), "kv": (512, 2048, "q8"),
        "indexer_q": (512, 2048, "bf16"), "wide_qkv": (10240, 2560, "q8")}


def listed():
    return [
        # one decoded token: the three kinds of layer work and the head, one row each
        dict(name="gdn_t1", kind="gdn", T=1, hv=16),
        dict(name="moe_t1", kind="moe", T=1, shape="base", K=10),
        dict(name="head_t1", kind="head", T=1, shape="base", V=151936),
        # a verify window of a speculative step, the context at its largest
        dict(name="moe_t4", kind="moe", T=4, shape="base", K=10),
        dict(name="qsa_t4_262k", kind="qsa", T=4, ctx=262140),
        # a short prompt: just above where prompts go through the chunked prefill
        dict(name="gemm_250", kind="gemm", M=250, proj="qsa_q", out="f32"),
        dict(name="moe_prefill_307", kind="moe_prefill", n=307, shape="base"),
        # a long prompt's chunk
        dict(name="gemm_8192", kind="gemm", M=8192, proj="gdn_qkv", out="f32"),
        dict(name="moe_prefill_8192", kind="moe_prefill", n=8192, shape="base"),
        # whole stages: a token at a long context (three delta-rule layers, then a sparse-attention one), a
        # long prompt's chunk after it (one layer of each), a follow-up prompt (two sparse-attention layers)
        dict(name="decode_32k", kind="decode", layers=4, period=4, T=1, ctx=32768),
        dict(name="prefill_8192", kind="prefill", layers=2, period=2, n=8192, ctx=32768),
        dict(name="prefill_qsa_1301", kind="prefill", layers=2, period=1, n=1301, ctx=9001),
    ]


def log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gdn", "qsa", "moe", "head", "gemm", "gemm", "moe_prefill", "moe_prefill", "decode", "prefill",
                       "prefill"])
    T = rng.randint(1, 8)
    shape = rng.choice(["base", "base", "wide"])
    if kind == "gdn":
        return dict(kind=kind, T=T, hv=rng.choice([16, 32, 48]))
    if kind == "qsa":
        return dict(kind=kind, T=T, ctx=log_int(rng, 16, 262136))
    if kind == "moe":
        return dict(kind=kind, T=T, shape=shape, K=rng.randint(4, 12))
    if kind == "head":
        return dict(kind=kind, T=T, shape=shape, V=log_int(rng, 30000, 248320))
    if kind == "gemm":
        return dict(kind=kind, M=log_int(rng, 193, 12000), proj=rng.choice(sorted(PROJ)), out=rng.choice(["f32", "bf16"]))
    if kind == "moe_prefill":
        return dict(kind=kind, n=log_int(rng, 193, 12000), shape=shape)
    if kind == "decode":
        return dict(kind=kind, layers=4, period=4, T=T, ctx=log_int(rng, 16, 131072))
    return dict(kind=kind, layers=2, period=rng.choice([1, 2]), n=log_int(rng, 193, 6000),
                ctx=rng.choice([0, log_int(rng, 16, 32768)]))


# ---- inputs ----------------------------------------------------------------------------------------
class Gen:
    """Seeded tensors on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(seed)

    def normal(self, *shape, mean=0.0, sd=1.0):
        return torch.empty(shape, device=DEV).normal_(mean, sd, generator=self.g)

    def uniform(self, *shape, lo, hi):
        return torch.empty(shape, device=DEV).uniform_(lo, hi, generator=self.g)

    def ints(self, *shape, lo, hi, dtype=torch.int8):
        return torch.randint(lo, hi, shape, device=DEV, generator=self.g, dtype=dtype)

    def bf16(self, *shape, sd=1.0):
        return self.normal(*shape, sd=sd).to(torch.bfloat16)

    def rows(self, *shape):
        """bf16-representable N(0, 1) activations in fp32"""
        return self.bf16(*shape).float()

    def q8(self, rows, cols):
        """Q8_0 codes and fp16 scales per 32 of N(0, 1 / cols) weights"""
        w = self.normal(rows, cols // 32, 32, sd=cols ** -0.5)
        s = (w.abs().amax(2, keepdim=True) / 127).half()
        return (w / s.float()).round_().clamp_(-127, 127).to(torch.int8).view(rows, cols), s.view(rows, cols // 32)

    def experts(self, D, F):
        """NVFP4 plane records: uniform e2m1 codes, e4m3 block scales in [2^-5, 2^-3], tensor scales 1"""
        sizes = [D * F, 2 * F * D // 16, D * F // 2, D * F // 16]
        rec = torch.empty(E, wzy_amd.lib().wzy_nvfp4_expert_bytes(D, F), dtype=torch.uint8, device=DEV)
        at = 0
        for i, n in enumerate(sizes):
            lo, hi = ((0, 256), (16, 33))[i & 1]
            rec[:, at:at + n] = self.ints(E, n, lo=lo, hi=hi, dtype=torch.uint8)
            at += n
        rec[:, at:].view(torch.float32)[:] = torch.tensor([1.0, 1.0, 1.0, 0.0], device=DEV)
        return rec


def p(t):
    return None if t is None else t.data_ptr()


def stream():
    return torch.cuda.current_stream().cuda_stream or None


def moe_weights(g, D, F, top_k):
    w = dict(router=g.bf16(E, D, sd=0.02), sgate=g.bf16(D, sd=0.02), experts=g.experts(D, F), gate=g.q8(F, D),
             up=g.q8(F, D), down=g.q8(D, F))
    m = wzy_amd.MoeWeights()
    m.n_embd, m.n_ff, m.n_exp, m.top_k = D, F, E, top_k
    m.router, m.sgate, m.experts = p(w["router"]), p(w["sgate"]), p(w["experts"])
    m.sh_gate_q, m.sh_gate_s = p(w["gate"][0]), p(w["gate"][1])
    m.sh_up_q, m.sh_up_s = p(w["up"][0]), p(w["up"][1])
    m.sh_down_q, m.sh_down_s = p(w["down"][0]), p(w["down"][1])
    return w, m


def segs(*rows):
    """wzy_gemv_seg array from (codes or bf16 rows, scales or None, output, output row stride)"""
    a = (wzy_amd.GemvSeg * len(rows))()
    for s, (w, sc, y, ld) in zip(a, rows):
        s.w, s.s, s.y, s.rows, s.y_stride = p(w), p(sc), p(y), w.shape[0], ld
        s.kind = wzy_amd.GEMV_BF16 if sc is None else wzy_amd.GEMV_Q8
    return a


def rope_tables(ctx, dtype=torch.float32):
    ang = torch.arange(ctx, dtype=torch.float64, device=DEV)[:, None] * (
        1e7 ** (-torch.arange(NROT // 2, dtype=torch.float64, device=DEV) / (NROT // 2)))[None, :]
    return ang.cos().to(dtype), ang.sin().to(dtype)


def gdn_width(hv):
    """q|k|v channels, output channels"""
    return (2 * HK + hv) * 128, hv * 128


def gdn_inputs(case, seed):
    g, T, hv, D = Gen(seed), case["T"], case["hv"], 2048
    QKV, GV = gdn_width(hv)
    return dict(
        R=g.normal(T, HC, D), bo=g.normal(T, D), inj_prev=g.normal(T, HC), norm=g.normal(HC, D, mean=1.0, sd=0.02),
        down=g.q8(LR, HC * D), inj_w=g.bf16(HC, HC * D, sd=(HC * D) ** -0.5), up=g.q8(HC * D, LR), qkv_w=g.q8(QKV, D),
        z_w=g.q8(GV, D), a_w=g.bf16(hv, D, sd=D ** -0.5), b_w=g.bf16(hv, D, sd=D ** -0.5), out_w=g.q8(D, GV),
        ssm_a=g.uniform(hv, lo=-2.0, hi=-1.0), dt=g.normal(hv, mean=-3.0, sd=0.5), conv_w=g.normal(QKV, 4, sd=0.5),
        gamma=g.normal(128, mean=1.0, sd=0.02), hist=g.normal(QKV, 3), ssm=g.normal(hv, 128, 128, sd=0.1))


def qsa_inputs(case, seed):
    g, T, ctx, D = Gen(seed), case["T"], case["ctx"], 2048
    cap = ctx + 8
    pooled = torch.zeros(cap // BLK + 2, IDIM, dtype=torch.float16, device=DEV)
    pooled[:ctx // BLK] = g.normal(ctx // BLK, IDIM).half()
    dead = g.normal(IDIM)
    pooled[ctx // BLK] = dead.half()
    return dict(
        x=g.rows(T, D), q_w=g.q8(2 * QD, D), k_w=g.q8(KVD, D), v_w=g.q8(KVD, D), ik_w=g.bf16(IDIM, D, sd=D ** -0.5),
        iq_w=g.bf16(IH * IDIM, D, sd=D ** -0.5), out_w=g.q8(D, QD), q_norm=g.normal(HD, mean=1.0, sd=0.02),
        k_norm=g.normal(HD, mean=1.0, sd=0.02), iq_norm=g.normal(IDIM, mean=1.0, sd=0.02),
        ik_norm=g.normal(IDIM, mean=1.0, sd=0.02), kq=g.ints(cap, KVD, lo=-127, hi=128),
        ks=g.uniform(cap, KVD // 64, lo=2.0 ** -7, hi=1.5 * 2.0 ** -6).half(), vq=g.ints(cap, KVD, lo=-127, hi=128),
        vs=g.uniform(cap, KVD // 64, lo=2.0 ** -7, hi=1.5 * 2.0 ** -6).half(),
        tail=g.normal(BLK - 1, IDIM).half().float(), dead=dead, pooled=pooled)


def gemm_inputs(case, seed):
    g, M = Gen(seed), case["M"]
    N, k, kind = PROJ[case["proj"]]
    w = g.q8(N, k) if kind == "q8" else (g.bf16(N, k, sd=k ** -0.5), None)
    return g.bf16(M, k), w


def moe_inputs(case, seed):
    g, s = Gen(seed), SHAPES[case["shape"]]
    return (g.rows(case.get("T") or case["n"], s["D"]),) + moe_weights(g, s["D"], s["F"], case.get("K", K))


def head_inputs(case, seed):
    g, s = Gen(seed), SHAPES[case["shape"]]
    return g.rows(case["T"], s["D"]), g.bf16(case["V"], s["D"], sd=s["D"] ** -0.5)


def stage_cfg(case, cap):
    cfg = wzy_amd.default_cfg(cap)
    cfg.n_layers, cfg.qsa_period, cfg.n_vocab = case["layers"], case["period"], STAGE_VOCAB
    return cfg


def settle(stage, layers):
    """Two things the plain random model lacks and a trained one has: router rows large enough that a token's
    experts stand clear of the others (four times as large here), and tensor scales that bring an expert's
    pre-activations and output to the size of its input.  Without them one row in five sits at a routing
    tie that any rounding decides, and a tie moves the logits by a third."""
    rec = stage.lib.wzy_nvfp4_expert_bytes(stage.cfg.n_embd, stage.cfg.n_ff)
    scales = np.array([0.1, 0.1, 0.2, 0.0], np.float32)
    for l in range(layers):
        r = (stage.read(l, "router", np.uint16).astype(np.uint32) << 16).view(np.float32) * np.float32(4)
        stage.write(l, "router", (r.view(np.uint32) >> 16).astype(np.uint16))
        for e in range(l * E, (l + 1) * E):
            stage.lib.wzy_stage_write_tensor_range(stage.h, -1, b"experts", (e + 1) * rec - 16, scales.ctypes.data, 16)


def prepare(case, seed):
    lib, kind, f32 = wzy_amd.lib(), case["kind"], dict(device=DEV, dtype=torch.float32)
    i32 = dict(device=DEV, dtype=torch.int32)
    st = stream()
    if kind == "gdn":
        a, T, HV, D = gdn_inputs(case, seed), case["T"], case["hv"], 2048
        QKV, GV = gdn_width(HV)
        o = dict(R=torch.empty(T, HC, D, **f32), inj=torch.empty(T, HC, **f32), block=torch.empty(T, D, **f32),
                 hist=a["hist"], ssm=a["ssm"])
        t = dict(nsc=torch.empty(T, HC, **f32), lo=torch.empty(T, LR, **f32), mixed=torch.empty(T, D, **f32),
                 qkv=torch.empty(T, QKV, **f32), z=torch.empty(T, GV, **f32), ab=torch.empty(T, 2 * HV, **f32),
                 y=torch.empty(T, GV, **f32))
        ws = torch.zeros(lib.wzy_hc_read_workspace_bytes(HC, LR, T), dtype=torch.uint8, device=DEV)
        s_in = segs((*a["qkv_w"], t["qkv"], QKV), (*a["z_w"], t["z"], GV), (a["a_w"], None, t["ab"], 2 * HV),
                    (a["b_w"], None, t["ab"][:, HV:], 2 * HV))
        s_out = segs((*a["out_w"], o["block"], D))
        calls = [
            (lib.wzy_hc_read, (p(a["R"]), None, None, 0, p(a["bo"]), p(a["inj_prev"]), p(o["R"]), p(a["norm"]),
                               p(a["down"][0]), p(a["down"][1]), p(a["inj_w"]), p(a["up"][0]), p(a["up"][1]), p(t["nsc"]),
                               p(t["lo"]), p(o["inj"]), p(t["mixed"]), D, HC, LR, EPS, T, p(ws), ws.numel(), st)),
            (lib.wzy_gemv_segs, (s_in, 4, p(t["mixed"]), D, T, st)),
            (lib.wzy_gdn_step, (p(t["qkv"]), p(t["z"]), p(t["ab"]), p(a["dt"]), p(a["ssm_a"]), p(a["conv_w"]), p(a["hist"]),
                                p(a["ssm"]), p(a["gamma"]), EPS, p(t["y"]), HK, HV, T, None, None, st)),
            (lib.wzy_gemv_segs, (s_out, 1, p(t["y"]), GV, T, st))]
        return dict(calls=calls, out=o, keep=(a, t, ws))
    if kind == "qsa":
        a, T, ctx, D = qsa_inputs(case, seed), case["T"], case["ctx"], 2048
        cap = a["kq"].shape[0]
        dm = wzy_amd.QsaDims(QH, KVH, HD, NROT, IH, IDIM, BLK, TOPK, cap, 0, 0, EPS, 32768)
        max_b = cap // BLK + 2
        t = dict(qg=torch.empty(T, 2 * QD, **f32), kk=torch.empty(T, KVD, **f32), vv=torch.empty(T, KVD, **f32),
                 ik=torch.empty(T, IDIM, **f32), iq=torch.empty(T, IH * IDIM, **f32), sel=torch.zeros(T, TOPK, **i32),
                 att=torch.empty(T, QD, **f32), pos=torch.tensor([ctx], **i32), cs=rope_tables(cap))
        o = dict(block=torch.empty(T, D, **f32), scores=torch.zeros(T, max_b, **f32), count=torch.zeros(T, **i32),
                 k=a["kq"], ks=a["ks"], v=a["vq"], vs=a["vs"], tail=a["tail"], pooled=a["pooled"])
        ws = torch.zeros(lib.wzy_qsa_attend_workspace_bytes(C.byref(dm), T), dtype=torch.uint8, device=DEV)
        s_in = segs((*a["q_w"], t["qg"], 2 * QD), (*a["k_w"], t["kk"], KVD), (*a["v_w"], t["vv"], KVD),
                    (a["ik_w"], None, t["ik"], IDIM), (a["iq_w"], None, t["iq"], IH * IDIM))
        s_out = segs((*a["out_w"], o["block"], D))
        kv = (p(a["kq"]), p(a["ks"]), p(a["vq"]), p(a["vs"]))
        calls = [
            (lib.wzy_gemv_segs, (s_in, 5, p(a["x"]), D, T, st)),
            (lib.wzy_qsa_prepare, (C.byref(dm), p(t["pos"]), p(t["qg"]), p(t["kk"]), p(t["vv"]), p(t["iq"]), p(t["ik"]),
                                   p(a["q_norm"]), p(a["k_norm"]), p(a["iq_norm"]), p(a["ik_norm"]), p(t["cs"][0]),
                                   p(t["cs"][1]), *kv, p(a["tail"]), p(a["dead"]), p(a["pooled"]), T, st)),
            (lib.wzy_qsa_select, (C.byref(dm), p(t["pos"]), p(a["pooled"]), p(a["dead"]), p(t["iq"]), p(o["scores"]), max_b,
                                  p(t["sel"]), p(o["count"]), T, st)),
            (lib.wzy_qsa_attend, (C.byref(dm), p(t["pos"]), p(t["qg"]), *kv, p(t["sel"]), p(t["att"]), p(ws), ws.numel(),
                                  T, st)),
            (lib.wzy_gemv_segs, (s_out, 1, p(t["att"]), QD, T, st))]
        return dict(calls=calls, out=o, keep=(a, t, ws, dm))
    if kind in ("moe", "moe_prefill"):
        x, w, m = moe_inputs(case, seed)
        n, D = x.shape
        dims = (m.n_embd, m.n_ff, m.n_exp, m.top_k, n)
        need = lib.wzy_moe_workspace_bytes(*dims) if kind == "moe" else lib.wzy_moe_prefill_workspace_bytes(*dims)
        ws = torch.zeros(need, dtype=torch.uint8, device=DEV)
        o = dict(comb=torch.empty(n, D, **f32), ids=torch.empty(n, m.top_k, **i32), wts=torch.empty(n, m.top_k, **f32))
        fn = lib.wzy_moe_block if kind == "moe" else lib.wzy_moe_prefill
        call = (fn, (C.byref(m), p(x), n, p(o["comb"]), p(o["ids"]), p(o["wts"]), p(ws), ws.numel(), st))
        return dict(calls=[call], out=o, keep=(x, w, m, ws))
    if kind == "head":
        x, w = head_inputs(case, seed)
        (T, D), V = x.shape, w.shape[0]
        o = dict(logits=torch.empty(T, V, **f32), greedy=torch.empty(T, **i32), top_v=torch.empty(T, 16, **f32),
                 top_i=torch.empty(T, 16, **i32))
        calls = [(lib.wzy_gemv_bf16, (p(w), p(x), p(o["logits"]), V, D, T, 0, st)),
                 (lib.wzy_row_top16, (p(o["logits"]), V, T, p(o["greedy"]), p(o["top_v"]), p(o["top_i"]), st))]
        return dict(calls=calls, out=o, keep=(x, w))
    if kind == "gemm":
        a, (w, s) = gemm_inputs(case, seed)
        (M, k), N = a.shape, w.shape[0]
        y = torch.empty(M, N, device=DEV, dtype=torch.float32 if case["out"] == "f32" else torch.bfloat16)
        yf, yb = (p(y), None) if case["out"] == "f32" else (None, p(y))
        q, sc, b = (p(w), p(s), None) if s is not None else (None, None, p(w))
        return dict(calls=[(lib.wzy_gemm_bf16, (p(a), k, M, k, q, sc, b, N, yf, yb, N, st))], out=dict(y=y), keep=(a, w, s))
    n = case["T"] if kind == "decode" else case["n"]
    stage = wzy_amd.Stage(stage_cfg(case, case["ctx"] + n + 8))
    stage.load_synthetic(seed, case["ctx"])
    settle(stage, case["layers"])
    toks = np.random.default_rng(seed).integers(0, STAGE_VOCAB, n).astype(np.int32)
    return dict(stage=stage, toks=toks, case=case)


def run(state):
    if "calls" in state:
        for fn, args in state["calls"]:
            fn(*args)
        return state["out"]
    stage, toks, case = state["stage"], state["toks"], state["case"]
    if case["kind"] == "decode":                  # a window keeps its snapshots for the commit of a prefix
        T = len(toks)
        stage.forward(case["ctx"], toks, save_snaps=T > 1)
    else:                                         # the last prompt token is the first decode step
        T = 1
        stage.prefill(case["ctx"], toks[:-1])
        stage.forward(case["ctx"] + len(toks) - 1, toks[-1:])
    stage.sync()
    return dict(logits=stage.logits(T))


# ---- what a pass cannot do without ------------------------------------------------------------------
def q8b(rows, cols):
    return rows * cols * 34 // 32


def hc_macs(D):
    return HC * D * (HC + 2 * LR)


def hc_bytes(D):
    return q8b(LR, HC * D) + q8b(HC * D, LR) + 2 * HC * HC * D + 4 * HC * D


def gdn_macs(D, hv=16):
    qkv, gv = gdn_width(hv)
    return D * (qkv + gv + 2 * hv) + gv * D + 3 * hv * 128 * 128


def gdn_bytes(D, hv=16):
    qkv, gv = gdn_width(hv)
    return q8b(qkv + gv, D) + 4 * hv * D + q8b(D, gv) + 2 * hv * 128 * 128 * 4 + qkv * (2 * 3 + 4) * 4


def qsa_macs(D):
    return D * (2 * QD + 2 * KVD + IDIM + IH * IDIM) + QD * D


def qsa_bytes(D):
    return q8b(2 * QD + 2 * KVD, D) + 2 * (IDIM + IH * IDIM) * D + q8b(D, QD)


def qsa_ctx_work(ctx, rows):
    """flops of scores and attention of `rows` rows after ctx cells; the keys, scores and cells they read once"""
    n_kv = ctx + rows
    sel = min(n_kv, TOPK)
    scored = n_kv // BLK if n_kv > TOPK else 0
    flops = rows * (2 * IH * IDIM * scored + 4 * QH * HD * sel)
    cells = min(n_kv, rows * sel)
    return flops, scored * IDIM * 2 + cells * KVD * 2 * 33 // 32


def moe_macs(D, F, top_k=K):
    return E * D + (1 + top_k) * 3 * D * F


def moe_bytes(D, F, rows, top_k=K):
    hit = E * (1 - (1 - top_k / E) ** rows)       # experts that some row routes to
    return 2 * E * D + 3 * q8b(D, F) + int(hit * 3 * D * F * 9 / 16)


def work(case):
    kind = case["kind"]
    if kind == "gdn":
        T, D = case["T"], 2048
        return {"bytes": hc_bytes(D) + gdn_bytes(D, case["hv"]) + T * 4 * (2 * HC + 2) * D,
                "flops": 2 * T * (hc_macs(D) + gdn_macs(D, case["hv"]))}
    if kind == "qsa":
        T, D = case["T"], 2048
        flops, nbytes = qsa_ctx_work(case["ctx"], T)
        return {"bytes": qsa_bytes(D) + nbytes + T * 8 * D, "flops": 2 * T * qsa_macs(D) + flops}
    if kind in ("moe", "moe_prefill"):
        s, n, top_k = SHAPES[case["shape"]], case.get("T") or case["n"], case.get("K", K)
        return {"bytes": moe_bytes(s["D"], s["F"], n, top_k) + n * 8 * s["D"],
                "flops": 2 * n * moe_macs(s["D"], s["F"], top_k)}
    if kind == "head":
        D, V, T = SHAPES[case["shape"]]["D"], case["V"], case["T"]
        return {"bytes": 2 * V * D + 4 * T * (D + V), "flops": 2 * T * V * D}
    if kind == "gemm":
        N, k, w = PROJ[case["proj"]]
        M = case["M"]
        return {"bytes": 2 * M * k + (q8b(N, k) if w == "q8" else 2 * N * k) + M * N * (4 if case["out"] == "f32" else 2),
                "flops": 2 * M * N * k}
    s, L, ctx = SHAPES["base"], case["layers"], case["ctx"]
    rows, D = case["T"] if kind == "decode" else case["n"], s["D"]
    n_qsa = L // case["period"]
    f_ctx, b_ctx = qsa_ctx_work(ctx, rows)
    heads = case["T"] if kind == "decode" else 1
    layer = 2 * hc_macs(D) + moe_macs(D, s["F"])
    flops = rows * (L * layer + n_qsa * qsa_macs(D) + (L - n_qsa) * gdn_macs(D))
    nbytes = L * (2 * hc_bytes(D) + moe_bytes(D, s["F"], rows)) + n_qsa * (qsa_bytes(D) + b_ctx)
    nbytes += (L - n_qsa) * gdn_bytes(D) + hc_bytes(D) + STAGE_VOCAB * D * 2 + rows * D * 2 + heads * STAGE_VOCAB * 4
    return {"bytes": nbytes, "flops": 2 * (flops + heads * (STAGE_VOCAB * D + hc_macs(D))) + n_qsa * f_ctx}


# ---- tolerances -------------------------------------------------------------------------------------
def tolerance(case):
    """About four times the error measured against exact(), or against the same stage with its
    normalisation weights moved by one part in 2^24."""
    kind = case["kind"]
    if kind == "gemm":                            # fp32 sums of bf16 products; a bf16 output is rounded once
        return {"rel": 2.4e-6, "max": 2e-5} if case["out"] == "f32" else {"rel": 2e-3, "max": 1e-2}
    if kind == "head":                            # fp32 sums; near-ties among the top 16 may swap
        return {"rel": 4e-7, "max": 1e-5, "differ": 0.005}
    if kind == "moe":                             # int8 activation codes beside a rounding tie may flip: 2.6e-3
        return {"rel": 1e-2, "max": 0.1}
    if kind == "moe_prefill":                     # bf16 activations: 1.7e-3
        return {"rel": 5e-3, "max": 5e-2, "differ": 1e-4}
    if kind == "gdn":                             # 2e-7 unless an int8 code flips
        return {"rel": 2e-3, "max": 3e-2}
    if kind == "qsa":                             # fp16 operands past 32,768 cells; cells at the selection's edge
        return {"rel": 1e-2, "max": 0.1, "differ": 1e-4}
    # 16-bit and int8 rounding flips spread over the layers: 1e-3 to 1e-2
    return {"rel": 3e-2, "max": 0.3}


# ---- the same values in 64 bits -----------------------------------------------------------------------
E2M1 = (0, 0.5, 1, 1.5, 2, 3, 4, 6, 0, -0.5, -1, -1.5, -2, -3, -4, -6)


def quant(x, n):
    """the activation quantisation of the Q8_0 / NVFP4 products: int8 codes per n values, scale amax / 127"""
    v = x.view(*x.shape[:-1], -1, n)
    a = v.abs().amax(-1, keepdim=True)
    return ((v * torch.where(a > 0, 127 / a, a)).round() * (a / 127)).view(x.shape)


def deq8(w, bf16=False):
    v = w[0].double() * w[1].double().repeat_interleave(32, 1)
    return v.to(torch.bfloat16).double() if bf16 else v


def nvfp4(codes, scales):
    """[rows, cols] values from code bytes [rows, cols / 2] and e4m3 scales [rows, cols / 16]"""
    lut = torch.tensor(E2M1, dtype=torch.float64, device=DEV)
    c = codes.view(codes.shape[0], -1, 8).long()
    v = torch.cat((lut[c & 15], lut[c >> 4]), 2)
    return (v * scales.contiguous().view(torch.float8_e4m3fn).double()[:, :, None]).view(codes.shape[0], -1)


def expert(rec, D, F):
    """gate|up [2F, D] and down [D, F] of one record"""
    at, m = 0, []
    for rows, cols in ((2 * F, D), (D, F)):
        c, s = rows * cols // 2, rows * cols // 16
        m.append(nvfp4(rec[at:at + c].view(rows, -1), rec[at + c:at + c + s].view(rows, -1)))
        at += c + s
    return m


def swiglu(g, u):
    return g * torch.sigmoid(g) * u


def route(logits, top_k):
    prob = torch.softmax(logits, 1)
    val, ids = torch.sort(prob, dim=1, descending=True, stable=True)
    val, ids = val[:, :top_k], ids[:, :top_k]
    return ids, val / val.sum(1, keepdim=True).clamp_min(2.0 ** -14)


def exact_moe(case, seed):
    s = SHAPES[case["shape"]]
    D, F = s["D"], s["F"]
    x32, w, _ = moe_inputs(case, seed)
    decode = case["kind"] == "moe"                # the prefill multiplies bf16 values, the decode int8 codes
    x = x32.double()
    ids, wts = route(x @ w["router"].double().T, case.get("K", K))
    qa = (lambda v, n: quant(v, n)) if decode else (lambda v, n: v)
    gate, up, down = (deq8(w[k], bf16=not decode) for k in ("gate", "up", "down"))
    xs = qa(x, 32)
    shared = qa(swiglu(xs @ gate.T, xs @ up.T), 32) @ down.T
    comb = shared * torch.sigmoid(x @ w["sgate"].double())[:, None]
    xr = qa(x, 16)
    for e in ids.unique().tolist():
        rows, slot = (ids == e).nonzero(as_tuple=True)
        gu, dn = expert(w["experts"][e], D, F)
        h = xr[rows] @ gu.T
        comb.index_add_(0, rows, (qa(swiglu(h[:, :F], h[:, F:]), 16) @ dn.T) * wts[rows, slot][:, None])
    return dict(comb=comb, ids=None, wts=wts)


def exact_gdn(case, seed):
    a = gdn_inputs(case, seed)
    d = {k: v.double() for k, v in a.items() if torch.is_tensor(v)}
    T, D = case["T"], 2048
    R = d["R"] + d["bo"][:, None, :] * (2 * torch.sigmoid(d["inj_prev"] / HC))[:, :, None]
    xn = R * (R.square().mean(2, keepdim=True) + EPS).rsqrt() * d["norm"]
    flat = xn.reshape(T, HC * D)
    lo = quant(flat, 32) @ deq8(a["down"]).T / HC
    lo = lo * torch.sigmoid(lo)
    inj = flat @ d["inj_w"].T
    gate = torch.sigmoid(quant(lo, 32) @ deq8(a["up"]).T).view(T, HC, D)
    mixed = (xn * gate).mean(1)
    mq = quant(mixed, 32)
    qkv, z = mq @ deq8(a["qkv_w"]).T, mq @ deq8(a["z_w"]).T
    decay = torch.exp(torch.nn.functional.softplus(mixed @ d["a_w"].T + d["dt"]) * d["ssm_a"])
    beta = torch.sigmoid(mixed @ d["b_w"].T)
    hist, S, ys = d["hist"], d["ssm"], []
    for t in range(T):
        win = torch.cat((hist, qkv[t][:, None]), 1)
        hist = win[:, 1:]
        c = (win * d["conv_w"]).sum(1)
        c = (c * torch.sigmoid(c)).view(-1, 128)
        qk = c[:2 * HK] * (c[:2 * HK].square().sum(1, keepdim=True) + EPS).rsqrt()
        q, k, v = qk[:HK].repeat(case["hv"] // HK, 1), qk[HK:].repeat(case["hv"] // HK, 1), c[2 * HK:]
        S = S * decay[t][:, None, None]
        delta = (v - (S * k[:, :, None]).sum(1)) * beta[t][:, None]
        S = S + k[:, :, None] * delta[:, None, :]
        o = (S * q[:, :, None]).sum(1) * 128 ** -0.5
        o = o * (o.square().mean(1, keepdim=True) + EPS).rsqrt() * d["gamma"]
        ys.append(o.reshape(-1) * torch.sigmoid(z[t]))
    block = quant(torch.stack(ys), 32) @ deq8(a["out_w"]).T
    return dict(R=R, inj=inj, block=block, hist=hist, ssm=S)


def exact_qsa(case, seed):
    a = qsa_inputs(case, seed)
    d = {k: v.double() for k, v in a.items() if torch.is_tensor(v) and k not in ("kq", "vq", "ks", "vs", "pooled")}
    T, ctx = case["T"], case["ctx"]
    cap = a["kq"].shape[0]
    cos, sin = rope_tables(cap, torch.float64)

    def norm_rope(v, gamma, pos):                 # v [.., n], pos an index of the tables
        v = v * (v.square().mean(-1, keepdim=True) + EPS).rsqrt() * gamma
        h = NROT // 2
        x, y = v[..., :h], v[..., h:NROT]
        return torch.cat((x * cos[pos] - y * sin[pos], x * sin[pos] + y * cos[pos], v[..., NROT:]), -1)

    xq = quant(d["x"], 32)
    qg = (xq @ deq8(a["q_w"]).T).view(T, QH, 2, HD)
    kk, vv = (xq @ deq8(a["k_w"]).T).view(T, KVH, HD), (xq @ deq8(a["v_w"]).T).view(T, KVH, HD)
    ik, iq = d["x"] @ d["ik_w"].T, (d["x"] @ d["iq_w"].T).view(T, IH, IDIM)

    def append(codes, scales, t, row):
        v = row.reshape(-1, 64)
        s = (v.abs().amax(1, keepdim=True) / 127).half()
        codes[ctx + t] = (v / s.double()).round().clamp(-127, 127).to(torch.int8).view(-1)
        scales[ctx + t] = s.view(-1)

    pooled, tail, dead = a["pooled"].clone(), d["tail"].clone(), d["dead"]
    kq, ks, vq, vs = (a[k].clone() for k in ("kq", "ks", "vq", "vs"))
    scores = torch.zeros(T, cap // BLK + 2, dtype=torch.float64, device=DEV)
    for t in range(T):
        append(kq, ks, t, norm_rope(kk[t], d["k_norm"], ctx + t))
        append(vq, vs, t, vv[t])
        raw, b = ik[t].half().double(), (ctx + t) // BLK
        if (ctx + t) % BLK < BLK - 1:
            tail[(ctx + t) % BLK] = raw
        else:
            m = (tail.sum(0) + raw) / BLK
            pooled[b] = norm_rope(m, d["ik_norm"], b * BLK).half()
            pooled[b + 1] = dead.half()
    att = torch.empty(T, QH, HD, dtype=torch.float64, device=DEV)
    for t in range(T):
        n_kv = ctx + t + 1
        if n_kv > TOPK:
            nb = n_kv // BLK
            q = norm_rope(iq[t], d["iq_norm"], ctx + t)
            sc = (pooled[:nb].double() @ q.half().double().T).clamp_min(0).sum(1)
            op = (q @ dead).clamp_min(0).sum() + (1e9 if n_kv % BLK else 0)
            scores[t, :nb], scores[t, nb] = sc, op
            left, room = n_kv - nb * BLK, TOPK
            cells = list(range(nb * BLK, n_kv))
            room -= left
            top = torch.sort(sc, descending=True, stable=True)[1][:-(-room // BLK)]
            cells = torch.cat((torch.tensor(cells, device=DEV, dtype=torch.int64),
                               (top[:, None] * BLK + torch.arange(BLK, device=DEV)).view(-1)[:room]))
        else:
            cells = torch.arange(n_kv, device=DEV)
        q = norm_rope(qg[t, :, 0], d["q_norm"], ctx + t)
        for j in range(KVH):
            sl, sg = slice(j * HD, (j + 1) * HD), slice(j * HD // 64, (j + 1) * HD // 64)
            Kc = kq[cells][:, sl].double() * ks[cells][:, sg].double().repeat_interleave(64, 1)
            Vc = vq[cells][:, sl].double() * vs[cells][:, sg].double().repeat_interleave(64, 1)
            h = slice(j * QH // KVH, (j + 1) * QH // KVH)
            att[t, h] = torch.softmax(q[h] @ Kc.T / 16, 1) @ Vc
    att = att * torch.sigmoid(qg[:, :, 1])
    block = quant(att.view(T, QD), 32) @ deq8(a["out_w"]).T
    return dict(block=block, scores=scores, count=None, k=None, ks=None, v=None, vs=None, tail=tail, pooled=None)


def exact(case, seed):
    kind = case["kind"]
    if kind == "gdn":
        return exact_gdn(case, seed)
    if kind == "qsa":
        return exact_qsa(case, seed)
    if kind in ("moe", "moe_prefill"):
        return exact_moe(case, seed)
    if kind == "head":
        x, w = head_inputs(case, seed)
        logits = torch.cat([x.double() @ b.double().T for b in w.split(16384)], 1)
        return dict(logits=logits, greedy=None, top_v=logits.topk(16, 1)[0], top_i=None)
    if kind == "gemm":
        a, w = gemm_inputs(case, seed)
        return dict(y=a.double() @ (deq8(w, bf16=True) if w[1] is not None else w[0].double()).T)
    return None        # a stage's weights are its own synthetic ones, which no plain code here can make
