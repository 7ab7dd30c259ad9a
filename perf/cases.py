"""The work a host of this library has it do, as measurable cases.

A translation server on these kernels spends its time in the decode step of
each token (batch-1 int8 products, attention over the KV cache, MoE rows), in
the prefill of prompts of some tens to some hundreds of tokens (batched f16
MFMA products, causal attention, grouped experts) and, where the host drives
single layers through the C ABI itself, in those same products one at a time.
Every case goes through the public entry points (the package's classes or the
device-pointer calls of include/hyq.h). Formats and shapes are those of the
1.8B, 7B and 30B-A3B-style models that bench.py and the tests build.

Weights are random packed blocks whose scales give the decoded rows a norm
near one, as trained linears have; activations are N(0, 1) rows.
"""
import importlib.util
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "hy-mt-rs_amd")


def _package():
    if "hy_mt_rs_amd" not in sys.modules:
        spec = importlib.util.spec_from_file_location(
            "hy_mt_rs_amd", os.path.join(PKG, "__init__.py"), submodule_search_locations=[PKG])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["hy_mt_rs_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["hy_mt_rs_amd"]


hyq = _package()
FMT = hyq.DTYPES
BLOCK = {"F32": (1, 4), "F16": (1, 2), "Q8_0": (32, 34), "Q4_K": (256, 144), "Q6_K": (256, 210),
         "Q2_0C": (512, 130), "STQ1_0": (256, 42)}
EPS = 1e-5
ROPE_BASE = 11158840.0
VOCAB = 120818
_ctx = None


def context():
    """The one context (device and stream) a host thread keeps."""
    global _ctx
    if _ctx is None:
        _ctx = hyq.Context(0)
    return _ctx


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # one decode token through a layer's FFN, driven call by call: the
        # smallest work a host asks for, where launches count (1.8B 2Bit)
        dict(name="ffn_decode_1p8b", kind="ffn", fmt="Q2_0C", down="Q2_0C", hidden=2048,
             ffn=6144),
        # the same for the 7B Q4_K_M mix: weights from HBM
        dict(name="ffn_decode_7b", kind="ffn", fmt="Q4_K", down="Q6_K", hidden=4096, ffn=14336),
        # one decode token through a layer's attention block, over the KV
        # cache of a page-long text
        dict(name="attn_decode_1p8b", kind="attn", fmt="Q2_0C", hidden=2048, heads=16,
             kv_heads=4, pos=1100),
        # one decode token through an MoE layer (64 experts, 8 used)
        dict(name="moe_decode", kind="moe", fmt="Q4_K", down="Q4_K", shared="Q8_0", tokens=1,
             experts=64, used=8, hidden=2048, mid=1536, smid=1536),
        # a sentence-long prompt through one linear
        dict(name="linear_q2c_sentence", kind="linear", fmt="Q2_0C", rows=6144, cols=2048,
             batch=21),
        # a paragraph, one token over a tile, through the 7B down projection
        dict(name="linear_q6k_ragged", kind="linear", fmt="Q6_K", rows=4096, cols=14336,
             batch=130),
        # a long prompt through the 7B gate projection
        dict(name="linear_q4k_512", kind="linear", fmt="Q4_K", rows=14336, cols=4096, batch=512),
        # the causal attention of a prompt's second part
        dict(name="attn_prefill", kind="attn_rows", heads=16, kv_heads=4, n=500, pos=1500),
        # a paragraph, and a long prompt, through an MoE layer
        dict(name="moe_64", kind="moe", fmt="Q4_K", down="Q4_K", shared="Q8_0", tokens=64,
             experts=64, used=8, hidden=2048, mid=1536, smid=1536),
        dict(name="moe_prefill", kind="moe", fmt="Q4_K", down="Q4_K", shared="Q8_0", tokens=500,
             experts=64, used=8, hidden=2048, mid=1536, smid=1536),
        # the whole 1.8B 2Bit model: 16 greedy tokens and one whose logits
        # the host samples from; and a prompt
        dict(name="generate_1p8b", kind="generate", fmt="Q2_0C", layers=32, hidden=2048, heads=16,
             kv_heads=4, ffn=6144, vocab=VOCAB, pos=1024, steps=16),
        dict(name="prefill_1p8b", kind="prefill", fmt="Q2_0C", layers=32, hidden=2048, heads=16,
             kv_heads=4, ffn=6144, vocab=VOCAB, n=777),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["linear", "ffn", "attn", "head", "attn_rows", "moe", "generate",
                        "prefill"], [8, 2, 2, 1, 3, 4, 1, 2])[0]
    quant = rng.choice(["Q2_0C", "STQ1_0", "Q4_K", "Q6_K", "Q8_0"])
    heads = rng.choice([(16, 4), (32, 8), (8, 2), (12, 4)])
    if kind == "linear":
        fmt = rng.choice([quant, quant, quant, quant, "F16"])
        return dict(kind=kind, fmt=fmt, rows=_log_int(rng, 512, 16384),
                    cols=512 * _log_int(rng, 2, 28), batch=_log_int(rng, 2, 1024))
    if kind == "ffn":
        return dict(kind=kind, fmt=quant, down=rng.choice([quant, "Q6_K"]),
                    hidden=512 * _log_int(rng, 2, 8), ffn=512 * _log_int(rng, 6, 28))
    if kind == "attn":
        return dict(kind=kind, fmt=quant, hidden=512 * _log_int(rng, 2, 8), heads=heads[0],
                    kv_heads=heads[1], pos=_log_int(rng, 16, 16000))
    if kind == "head":
        return dict(kind=kind, fmt=rng.choice(["Q6_K", "Q4_K", "Q8_0"]),
                    rows=_log_int(rng, 30000, 130000), cols=512 * _log_int(rng, 2, 8))
    if kind == "attn_rows":
        return dict(kind=kind, heads=heads[0], kv_heads=heads[1], n=_log_int(rng, 2, 1000),
                    pos=rng.choice([0, _log_int(rng, 16, 4000)]))
    if kind == "moe":
        tokens = rng.choice([1, _log_int(rng, 2, 16), _log_int(rng, 17, 128),
                             _log_int(rng, 129, 700)])
        fmt = rng.choice(["Q4_K", "Q4_K", "Q2_0C", "Q8_0"])
        return dict(kind=kind, fmt=fmt, down=rng.choice([fmt, fmt, "Q6_K"]), shared="Q8_0",
                    tokens=tokens, experts=rng.choice([32, 64]), used=rng.choice([4, 6, 8]),
                    hidden=512 * rng.randint(2, 4), mid=512 * rng.randint(1, 3),
                    smid=512 * rng.randint(1, 3))
    model = dict(kind=kind, fmt=rng.choice(["Q2_0C", "STQ1_0", "Q4_K"]), layers=rng.randint(2, 16),
                 hidden=512 * rng.randint(2, 4), heads=16, kv_heads=4,
                 ffn=512 * rng.randint(4, 12), vocab=_log_int(rng, 8000, VOCAB))
    if kind == "generate":
        return dict(model, pos=_log_int(rng, 16, 2000), steps=rng.randint(4, 16))
    n = _log_int(rng, 8, 777)
    return dict(model, n=n + 1 if n % 256 == 1 else n)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
class Source:
    """Seeded random tensors on the GPU, in the order they are asked for."""

    def __init__(self, seed):
        self.g = torch.Generator("cuda")
        self.g.manual_seed(int(seed) * 7919 + 13)

    def normal(self, *shape):
        return torch.randn(shape, generator=self.g, device="cuda", dtype=torch.float32)

    def ints(self, lo, hi, *shape):
        return torch.randint(lo, hi, shape, generator=self.g, device="cuda", dtype=torch.int32)

    def norm_vector(self, n):
        return 1.0 + 0.02 * self.normal(n)

    def blocks(self, fmt, rows, cols):
        """[blocks, block bytes] packed rows of about unit norm."""
        length, size = BLOCK[fmt]
        nb = rows * cols // length
        target = cols ** -0.5
        if fmt in ("F32", "F16"):
            v = self.normal(nb, 1) * target
            return (v if fmt == "F32" else v.half()).view(torch.uint8)
        b = torch.randint(0, 256, (nb, size), generator=self.g, device="cuda", dtype=torch.uint8)
        # block scales spread by a quarter around the one for the target deviation
        unit = {"Q8_0": 73.9, "Q4_K": 205.0, "Q6_K": 1365.0, "Q2_0C": 2.24, "STQ1_0": 0.87}[fmt]
        d = (torch.exp(0.25 * self.normal(nb)) * (target / unit)).half()
        at = {"Q8_0": 0, "Q4_K": 0, "Q6_K": 208, "Q2_0C": 0, "STQ1_0": 40}[fmt]
        b[:, at:at + 2] = d.view(torch.uint8).view(nb, 2)
        if fmt == "Q4_K":  # minimums that centre the weights
            b[:, 2:4] = (7.5 * d.float()).half().view(torch.uint8).view(nb, 2)
        return b


def _upload(fmt, blocks, dims):
    return context().upload(FMT[fmt], blocks.cpu().numpy().reshape(-1), dims)


def _tensors(case, seed):
    """The seeded inputs of a case: packed blocks and f32 vectors, by name."""
    s, c = Source(seed), case
    kind = c["kind"]
    t = {}
    if kind == "linear":
        t["w"] = s.blocks(c["fmt"], c["rows"], c["cols"])
        t["x"] = s.normal(c["batch"], c["cols"])
    elif kind == "ffn":
        H, F = c["hidden"], c["ffn"]
        t["gate"], t["up"] = s.blocks(c["fmt"], F, H), s.blocks(c["fmt"], F, H)
        t["down"] = s.blocks(c["down"], H, F)
        t["norm"], t["x"] = s.norm_vector(H), s.normal(H)
    elif kind == "attn":
        H, Q, KV = c["hidden"], c["heads"] * 128, c["kv_heads"] * 128
        for n, r, k in (("q", Q, H), ("k", KV, H), ("v", KV, H), ("o", H, Q)):
            t[n] = s.blocks(c["fmt"], r, k)
        t["norm"], t["x"] = s.norm_vector(H), s.normal(H)
        t["qn"], t["kn"] = s.norm_vector(128), s.norm_vector(128)
        t["kc"], t["vc"] = s.normal(c["pos"] + 1, KV), s.normal(c["pos"] + 1, KV)
    elif kind == "head":
        t["w"] = s.blocks(c["fmt"], c["rows"], c["cols"])
        t["norm"], t["x"] = s.norm_vector(c["cols"]), s.normal(c["cols"])
    elif kind == "attn_rows":
        KV, P = c["kv_heads"] * 128, c["pos"] + c["n"]
        t["q"] = s.normal(c["n"], c["heads"] * 128)
        t["kc"], t["vc"] = s.normal(P, KV), s.normal(P, KV)
    elif kind == "moe":
        H, M, S, E = c["hidden"], c["mid"], c["smid"], c["experts"]
        t["router"] = s.blocks("F32", E, H)
        t["bias"] = 0.1 * s.normal(E)
        t["gate"], t["up"] = s.blocks(c["fmt"], E * M, H), s.blocks(c["fmt"], E * M, H)
        t["down"] = s.blocks(c["down"], E * H, M)
        t["sgate"], t["sup"] = s.blocks(c["shared"], S, H), s.blocks(c["shared"], S, H)
        t["sdown"] = s.blocks(c["shared"], H, S)
        t["x"] = s.normal(c["tokens"], H)
    else:
        H, F, Q, KV = c["hidden"], c["ffn"], c["heads"] * 128, c["kv_heads"] * 128
        for l in range(c["layers"]):
            for n, r, k in (("q", Q, H), ("k", KV, H), ("v", KV, H), ("o", H, Q), ("gate", F, H),
                            ("up", F, H), ("down", H, F)):
                t[f"{n}{l}"] = s.blocks(c["fmt"], r, k)
            t[f"an{l}"], t[f"fn{l}"] = s.norm_vector(H), s.norm_vector(H)
            t[f"qn{l}"], t[f"kn{l}"] = s.norm_vector(128), s.norm_vector(128)
        t["embed"] = s.blocks("Q6_K", c["vocab"], H)
        t["on"] = s.norm_vector(H)
        if kind == "generate":
            t["token"] = s.ints(0, c["vocab"], 1)
            t["kc"] = s.normal(c["layers"], c["pos"], KV)
            t["vc"] = s.normal(c["layers"], c["pos"], KV)
        else:
            t["tokens"] = s.ints(0, c["vocab"], c["n"])
    return t


def _frequencies():
    j = torch.arange(64, device="cuda", dtype=torch.float64)
    return (ROPE_BASE ** (-2.0 * j / 128)).float()


def prepare(case, seed):
    c, t, ctx = case, _tensors(case, seed), context()
    kind = c["kind"]
    f32 = dict(device="cuda", dtype=torch.float32)
    s = dict(case=c)
    if kind == "linear":
        s.update(w=_upload(c["fmt"], t["w"], (c["cols"], c["rows"])), x=t["x"],
                 y=torch.empty(c["batch"], c["rows"], **f32))
    elif kind == "ffn":
        H, F = c["hidden"], c["ffn"]
        s.update(gate=_upload(c["fmt"], t["gate"], (H, F)), up=_upload(c["fmt"], t["up"], (H, F)),
                 down=_upload(c["down"], t["down"], (F, H)), norm=t["norm"], x=t["x"],
                 q8=ctx.q8(H), q8h=ctx.q8(F), h=torch.empty(F, **f32), y=torch.empty(H, **f32))
    elif kind == "attn":
        H, Q, KV = c["hidden"], c["heads"] * 128, c["kv_heads"] * 128
        n = hyq.lib().hyq_attention_scratch_floats(c["pos"] + 1, c["heads"])
        s.update(wq=_upload(c["fmt"], t["q"], (H, Q)), wk=_upload(c["fmt"], t["k"], (H, KV)),
                 wv=_upload(c["fmt"], t["v"], (H, KV)), wo=_upload(c["fmt"], t["o"], (Q, H)),
                 norm=t["norm"], x=t["x"], qn=t["qn"], kn=t["kn"], kc=t["kc"], vc=t["vc"],
                 q8=ctx.q8(H), q8a=ctx.q8(Q), q=torch.empty(Q, **f32), k=torch.empty(KV, **f32),
                 v=torch.empty(KV, **f32), att=torch.empty(Q, **f32), y=torch.empty(H, **f32),
                 freq=_frequencies(), pos=torch.tensor([c["pos"]], device="cuda",
                                                       dtype=torch.int32),
                 scratch=torch.empty(n, **f32))
    elif kind == "head":
        s.update(w=_upload(c["fmt"], t["w"], (c["cols"], c["rows"])), norm=t["norm"], x=t["x"],
                 q8=ctx.q8(c["cols"]), y=torch.empty(c["rows"], **f32),
                 scratch=torch.empty(128, **f32),
                 token=torch.zeros(1, device="cuda", dtype=torch.int32))
    elif kind == "attn_rows":
        P = c["pos"] + c["n"]
        n = hyq.lib().hyq_attention_rows_scratch_floats(P, c["heads"], c["n"])
        s.update(q=t["q"], kc=t["kc"], vc=t["vc"], scratch=torch.empty(n, **f32),
                 pos=torch.tensor([c["pos"]], device="cuda", dtype=torch.int32),
                 y=torch.empty(c["n"], c["heads"] * 128, **f32))
    elif kind == "moe":
        H, M, S, E = c["hidden"], c["mid"], c["smid"], c["experts"]
        cfg = hyq.MoeConfig(E, c["used"], M, S, 1, 2.5)
        n = hyq.lib().hyq_moe_forward_scratch_bytes(hyq.ctypes.byref(cfg), H, c["tokens"])
        s.update(cfg=cfg, router=_upload("F32", t["router"], (H, E)), bias=t["bias"],
                 gate=_upload(c["fmt"], t["gate"], (H, M, E)),
                 up=_upload(c["fmt"], t["up"], (H, M, E)),
                 down=_upload(c["down"], t["down"], (M, H, E)),
                 sgate=_upload(c["shared"], t["sgate"], (H, S)),
                 sup=_upload(c["shared"], t["sup"], (H, S)),
                 sdown=_upload(c["shared"], t["sdown"], (S, H)), x=t["x"], nbytes=n,
                 scratch=torch.empty(n, device="cuda", dtype=torch.uint8),
                 y=torch.empty(c["tokens"], H, **f32))
    else:
        s.update(_decoder(c, t))
    return s


def _decoder(c, t):
    H, F, Q, KV = c["hidden"], c["ffn"], c["heads"] * 128, c["kv_heads"] * 128
    ctx, fmt = context(), c["fmt"]
    cfg = hyq.DenseConfig(c["layers"], H, c["heads"], c["kv_heads"], 128, F, c["vocab"],
                          ROPE_BASE, EPS)
    length = c["pos"] + c["steps"] + 1 if c["kind"] == "generate" else c["n"]
    dec = hyq.DenseDecoder(ctx, cfg, length)
    for l in range(c["layers"]):
        W = {n: _upload(fmt, t[f"{n}{l}"], d)
             for n, d in (("q", (H, Q)), ("k", (H, KV)), ("v", (H, KV)), ("o", (Q, H)),
                          ("gate", (H, F)), ("up", (H, F)), ("down", (F, H)))}
        dec.set_layer(l, W["q"], W["k"], W["v"], W["o"], W["gate"], W["up"], W["down"],
                      *[t[f"{n}{l}"].cpu().numpy() for n in ("an", "fn", "qn", "kn")])
    E = _upload("Q6_K", t["embed"], (H, c["vocab"]))
    dec.set_output(E, E, t["on"].cpu().numpy())
    if c["kind"] == "generate":
        for l in range(c["layers"]):
            dec.load_kv(l, t["kc"][l].cpu().numpy(), t["vc"][l].cpu().numpy())
        return dict(dec=dec, token=int(t["token"][0]))
    return dict(dec=dec, tokens=t["tokens"].cpu().numpy())


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(s):
    c, L, h, ok = s["case"], hyq.lib(), context().handle, hyq.check
    kind = c["kind"]
    if kind == "linear":
        ok(L.hyq_matmul_d(h, s["w"].handle, s["x"].data_ptr(), c["batch"], s["y"].data_ptr()))
        return s["y"]
    if kind == "ffn":
        x, y = s["x"].data_ptr(), s["y"].data_ptr()
        ok(L.hyq_rms_norm_q8_d(h, x, s["norm"].data_ptr(), c["hidden"], EPS, None,
                               s["q8"].handle))
        ok(L.hyq_gate_up_silu_q8_d(h, s["gate"].handle, s["up"].handle, s["q8"].handle,
                                   s["h"].data_ptr()))
        ok(L.hyq_quantize_q8_d(h, s["h"].data_ptr(), c["ffn"], s["q8h"].handle))
        ok(L.hyq_gemv_q8_d(h, s["down"].handle, s["q8h"].handle, x, y))
        return {"h": s["h"], "y": s["y"]}
    if kind == "attn":
        q, k, v = s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr()
        ok(L.hyq_rms_norm_q8_d(h, s["x"].data_ptr(), s["norm"].data_ptr(), c["hidden"], EPS,
                               None, s["q8"].handle))
        ok(L.hyq_gemv_qkv_q8_d(h, s["wq"].handle, s["wk"].handle, s["wv"].handle,
                               s["q8"].handle, q, k, v))
        ok(L.hyq_attention_rope_d(h, q, k, v, s["qn"].data_ptr(), s["kn"].data_ptr(),
                                  s["freq"].data_ptr(), s["pos"].data_ptr(), c["pos"] + 1,
                                  c["heads"], c["kv_heads"], 128, EPS, 0, s["kc"].data_ptr(),
                                  s["vc"].data_ptr(), s["scratch"].data_ptr(),
                                  s["att"].data_ptr()))
        ok(L.hyq_quantize_q8_d(h, s["att"].data_ptr(), c["heads"] * 128, s["q8a"].handle))
        ok(L.hyq_gemv_q8_d(h, s["wo"].handle, s["q8a"].handle, s["x"].data_ptr(),
                           s["y"].data_ptr()))
        return {"att": s["att"], "kc": s["kc"], "vc": s["vc"], "y": s["y"]}
    if kind == "head":
        ok(L.hyq_rms_norm_q8_d(h, s["x"].data_ptr(), s["norm"].data_ptr(), c["cols"], EPS, None,
                               s["q8"].handle))
        ok(L.hyq_gemv_q8_d(h, s["w"].handle, s["q8"].handle, None, s["y"].data_ptr()))
        ok(L.hyq_argmax_d(h, s["y"].data_ptr(), c["rows"], s["scratch"].data_ptr(),
                          s["token"].data_ptr()))
        return {"logits": s["y"], "token": s["token"]}
    if kind == "attn_rows":
        ok(L.hyq_attention_rows_d(h, s["q"].data_ptr(), s["kc"].data_ptr(), s["vc"].data_ptr(),
                                  s["pos"].data_ptr(), c["n"], c["pos"] + c["n"], c["heads"],
                                  c["kv_heads"], 128, s["scratch"].data_ptr(),
                                  s["y"].data_ptr()))
        return s["y"]
    if kind == "moe":
        ok(L.hyq_moe_forward_d(h, hyq.ctypes.byref(s["cfg"]), s["router"].handle,
                               s["bias"].data_ptr(), s["gate"].handle, s["up"].handle,
                               s["down"].handle, s["sgate"].handle, s["sup"].handle,
                               s["sdown"].handle, s["x"].data_ptr(), c["tokens"],
                               s["scratch"].data_ptr(), s["nbytes"], s["y"].data_ptr()))
        return s["y"]
    dec = s["dec"]
    if kind == "generate":
        dec.position = c["pos"]
        tokens = dec.generate(s["token"], c["steps"])
        logits, _ = dec.forward(int(tokens[-1]))
        return {"tokens": tokens, "logits": logits}
    dec.position = 0
    logits, token = dec.prefill(s["tokens"])
    return {"logits": logits, "token": token}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _wbytes(fmt, rows, cols):
    length, size = BLOCK[fmt]
    return rows * cols // length * size


def work(case):
    c = case
    kind = c["kind"]
    if kind == "linear":
        R, K, B = c["rows"], c["cols"], c["batch"]
        return dict(bytes=_wbytes(c["fmt"], R, K) + 4 * B * (R + K), flops=2 * B * R * K)
    if kind == "head":
        R, K = c["rows"], c["cols"]
        return dict(bytes=_wbytes(c["fmt"], R, K) + 4 * (R + 2 * K), flops=2 * R * K)
    if kind == "ffn":
        H, F = c["hidden"], c["ffn"]
        return dict(bytes=2 * _wbytes(c["fmt"], F, H) + _wbytes(c["down"], H, F) +
                    4 * (3 * H + F), flops=6 * H * F)
    if kind == "attn":
        H, Q, KV, P = c["hidden"], c["heads"] * 128, c["kv_heads"] * 128, c["pos"] + 1
        w = _wbytes(c["fmt"], 2 * Q + 2 * KV, H)
        return dict(bytes=w + 8 * P * KV + 4 * (3 * H + Q), flops=2 * H * (2 * Q + 2 * KV) +
                    4 * P * Q)
    if kind == "attn_rows":
        Q, KV, n, p = c["heads"] * 128, c["kv_heads"] * 128, c["n"], c["pos"]
        return dict(bytes=8 * (p + n) * KV + 8 * n * Q,
                    flops=4 * Q * (n * p + n * (n + 1) // 2))
    if kind == "moe":
        H, M, S, E, T, U = (c[k] for k in ("hidden", "mid", "smid", "experts", "tokens", "used"))
        touched = E * (1 - (1 - U / E) ** T)  # experts that some token chose
        w = 2 * _wbytes(c["fmt"], M, H) + _wbytes(c["down"], H, M)
        ws = 3 * _wbytes(c["shared"], S, H)
        return dict(bytes=touched * w + ws + 4 * E * H + 8 * T * H,
                    flops=T * (2 * E * H + 6 * H * S + U * 6 * H * M))
    H, F, Q, KV = c["hidden"], c["ffn"], c["heads"] * 128, c["kv_heads"] * 128
    mats = ((2 * Q + 2 * KV), H), (3 * F, H)
    layer = sum(_wbytes(c["fmt"], r, k) for r, k in mats)
    macs = sum(r * k for r, k in mats)
    head = _wbytes("Q6_K", c["vocab"], H)
    if kind == "generate":
        n, p = c["steps"] + 1, c["pos"] + c["steps"] / 2
        return dict(bytes=n * (c["layers"] * (layer + 8 * p * KV) + head),
                    flops=n * (c["layers"] * (2 * macs + 4 * p * Q) + 2 * c["vocab"] * H))
    n = c["n"]
    return dict(bytes=c["layers"] * (layer + 8 * n * KV) + head + 4 * c["vocab"],
                flops=c["layers"] * (2 * n * macs + 2 * n * n * Q) + 2 * c["vocab"] * H)


def tolerance(case):
    c = case
    kind = c["kind"]
    if kind == "linear":
        # batched products of quantized weights round both operands to f16
        # (2^-11 each: 2.6e-4 of the result); F16 weights are f32 sums
        return {"rel": 1e-5} if c["fmt"] == "F16" else {"rel": 1e-3}
    if kind in ("ffn", "attn", "head"):
        # f32 sums, and int8 codes of rows that another summation order may
        # put on the other side of a rounding midpoint: one code in a row
        # of 2048 moves a product by about 6e-4 of its norm
        return {"rel": 1e-3}
    if kind == "attn_rows":
        return {"rel": 1e-5}
    if kind == "moe":
        # int8 codes for one token as above, else f16 operands in each of
        # two products in a row
        return {"rel": 1e-3} if c["tokens"] == 1 else {"rel": 3e-3}
    # a whole random-init model: one code or one f16 rounding grows through
    # the layers that follow
    return {"rel": 3e-2}


# ---------------------------------------------------------------------------
# the same in 64 bits, in plain torch
# ---------------------------------------------------------------------------
_CODEBOOK = [0xa9, 0x89, 0x29, 0x09, 0xa6, 0x86, 0x26, 0x06, 0x9a, 0x92, 0x1a, 0x12, 0x6a, 0x62,
             0x4a, 0x42, 0x01, 0x21, 0x81, 0xa1, 0x04, 0x24, 0x84, 0xa4, 0x10, 0x18, 0x90, 0x98,
             0x40, 0x48, 0x60, 0x68]


def _half(b):
    return b.contiguous().view(torch.float16).double()


def _bits(b, shifts, mask):
    """[n, len(shifts), m] fields of bytes [n, m]."""
    sh = torch.tensor(shifts, device=b.device, dtype=torch.int32)
    return (b.int()[:, None, :] >> sh[None, :, None]) & mask


def decoded(fmt, b, rows, cols):
    """The f64 values [rows, cols] of packed blocks [n, block bytes]."""
    n = b.shape[0]
    if fmt == "F32":
        v = b.contiguous().view(torch.float32).double()
    elif fmt == "F16":
        v = _half(b)
    elif fmt == "Q8_0":
        v = _half(b[:, :2]) * b[:, 2:].contiguous().view(torch.int8).double()
    elif fmt == "Q2_0C":
        code = _bits(b[:, 2:], [0, 2, 4, 6], 3).transpose(1, 2).reshape(n, 512)
        v = (2 * code - 3).double() * _half(b[:, :2])
    elif fmt == "STQ1_0":
        nib = _bits(b[:, :32], [0, 4], 15).transpose(1, 2).reshape(n, 64)
        sign = _bits(b[:, 32:40], list(range(8)), 1).transpose(1, 2).reshape(n, 64)
        book = torch.tensor(_CODEBOOK, device=b.device, dtype=torch.int32)
        e = book[(sign * 16 + nib).long()].view(n, 4, 1, 16)
        sh = torch.tensor([0, 2, 4, 6], device=b.device, dtype=torch.int32).view(1, 1, 4, 1)
        v = (((e >> sh) & 3) - 1).reshape(n, 256).double() * _half(b[:, 40:42])
    elif fmt == "Q4_K":
        d, dmin, sc = _half(b[:, :2]), _half(b[:, 2:4]), b[:, 4:16].int()
        lo, mid, hi = sc[:, :4], sc[:, 4:8], sc[:, 8:12]
        s = torch.cat([lo & 63, (hi & 15) | ((lo >> 6) << 4)], 1).double()
        m = torch.cat([mid & 63, (hi >> 4) | ((mid >> 6) << 4)], 1).double()
        q = _bits(b[:, 16:].reshape(n * 4, 32), [0, 4], 15).reshape(n, 8, 32).double()
        v = (d * s)[:, :, None] * q - (dmin * m)[:, :, None]
    else:  # Q6_K
        ql = b[:, :128].reshape(n * 2, 64)
        qh = b[:, 128:192].reshape(n * 2, 32)
        low = _bits(ql, [0, 4], 15).reshape(n * 2, 4, 32)
        high = _bits(qh, [0, 2, 4, 6], 3)
        q = (low | (high << 4)).reshape(n, 16, 16).double() - 32
        s = _half(b[:, 208:210]) * b[:, 192:208].contiguous().view(torch.int8).double()
        v = s[:, :, None] * q
    return v.reshape(rows, cols)


def _quantized(x):
    """The int8 activations' values (one f32 scale per 256, ties to even)."""
    x = x.float().view(-1, 256)
    top = x.abs().amax(1, keepdim=True)
    zero = top == 0
    one = torch.ones_like(top)
    inv = torch.where(zero, 0 * one, 127.0 * one / torch.where(zero, one, top))
    q = torch.clamp(torch.round(x * inv), -128, 127).double()
    return (q * (top / 127.0).double()).reshape(-1)


def _rms(x, w):
    x = x.double()
    return x * (w.double() / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS))


def _silu(g):
    return g / (1 + torch.exp(-g))


def _rope(x, p):
    """x [n, heads, 128] at positions p [n], halves rotated."""
    a = p.double()[:, None] * _frequencies().double()[None, :]
    cs, sn = torch.cos(a)[:, None, :], torch.sin(a)[:, None, :]
    u, v = x[..., :64], x[..., 64:]
    return torch.cat([u * cs - v * sn, v * cs + u * sn], -1)


def _attend(q, k, v, first):
    """Causal attention of q [n, heads, 128] over k, v [p, kv heads, 128]:
    row i sees positions up to first + i."""
    n, heads, _ = q.shape
    kvh = k.shape[1]
    out = torch.empty_like(q)
    seen = torch.arange(k.shape[0], device=q.device)[None, :] <= (
        first + torch.arange(n, device=q.device)[:, None])
    for h in range(heads):
        kk, vv = k[:, h * kvh // heads], v[:, h * kvh // heads]
        s = (q[:, h] @ kk.T.contiguous()) / math.sqrt(128.0)
        p = torch.softmax(torch.where(seen, s, torch.full_like(s, -math.inf)), 1)
        out[:, h] = p @ vv.contiguous()
    return out


def exact(case, seed):
    c = case
    kind = c["kind"]
    if kind == "generate":
        # the greedy tokens feed back and every row is rounded to int8
        # codes: in 64 bits it is another chain
        return None
    t = _tensors(case, seed)
    if kind == "linear":
        w = decoded(c["fmt"], t["w"], c["rows"], c["cols"])
        return t["x"].double() @ w.T.contiguous()
    if kind == "head":
        w = decoded(c["fmt"], t["w"], c["rows"], c["cols"])
        y = w @ _quantized(_rms(t["x"], t["norm"]))
        return {"logits": y, "token": None}
    if kind == "ffn":
        H, F = c["hidden"], c["ffn"]
        x = _quantized(_rms(t["x"], t["norm"]))
        h = _silu(decoded(c["fmt"], t["gate"], F, H) @ x) * (decoded(c["fmt"], t["up"], F, H) @ x)
        y = t["x"].double() + decoded(c["down"], t["down"], H, F) @ _quantized(h)
        return {"h": h, "y": y}
    if kind == "attn":
        H, Q, KV = c["hidden"], c["heads"] * 128, c["kv_heads"] * 128
        x = _quantized(_rms(t["x"], t["norm"]))
        q, k, v = (decoded(c["fmt"], t[n], r, H) @ x for n, r in (("q", Q), ("k", KV), ("v", KV)))
        at = torch.tensor([c["pos"]], device="cuda")
        q = _rms(_rope(q.view(1, -1, 128), at), t["qn"])
        k = _rms(_rope(k.view(1, -1, 128), at), t["kn"])
        kc, vc = t["kc"].double(), t["vc"].double()
        kc[c["pos"]], vc[c["pos"]] = k.reshape(-1), v
        att = _attend(q, kc.view(-1, c["kv_heads"], 128), vc.view(-1, c["kv_heads"], 128),
                      c["pos"]).reshape(-1)
        y = t["x"].double() + decoded(c["fmt"], t["o"], H, Q) @ _quantized(att)
        return {"att": att, "kc": kc, "vc": vc, "y": y}
    if kind == "attn_rows":
        q = t["q"].double().view(c["n"], -1, 128)
        kc, vc = (t[n].double().view(-1, c["kv_heads"], 128) for n in ("kc", "vc"))
        return _attend(q, kc, vc, c["pos"]).reshape(c["n"], -1)
    if kind == "moe":
        return _moe64(c, t)
    return _prefill64(c, t)


def _moe64(c, t):
    H, M, S, E, T = (c[k] for k in ("hidden", "mid", "smid", "experts", "tokens"))
    act = _quantized if T == 1 else (lambda v: v)  # one token: int8 rows

    def ffn(x, g, u, d):
        if T == 1:
            h = act((_silu(g @ act(x.reshape(-1))) * (u @ act(x.reshape(-1)))).reshape(-1))
            return (d @ h).view(1, -1)
        return (_silu(x @ g.T.contiguous()) * (x @ u.T.contiguous())) @ d.T.contiguous()

    x = t["x"].double()
    p = torch.sigmoid(x @ decoded("F32", t["router"], E, H).T.contiguous())
    chosen = torch.topk(p + t["bias"].double(), c["used"], 1).indices
    w = torch.gather(p, 1, chosen)
    w = w / w.sum(1, keepdim=True) * 2.5
    y = ffn(x, decoded(c["shared"], t["sgate"], S, H), decoded(c["shared"], t["sup"], S, H),
            decoded(c["shared"], t["sdown"], H, S))
    gate, up, down = (t[n].view(E, -1, t[n].shape[1]) for n in ("gate", "up", "down"))
    for e in range(E):
        rows, at = torch.nonzero(chosen == e, as_tuple=True)
        if rows.numel():
            y[rows] += w[rows, at][:, None] * ffn(
                x[rows], decoded(c["fmt"], gate[e], M, H), decoded(c["fmt"], up[e], M, H),
                decoded(c["down"], down[e], H, M))
    return y


def _prefill64(c, t):
    H, F, Q, KV, n = c["hidden"], c["ffn"], c["heads"] * 128, c["kv_heads"] * 128, c["n"]
    emb = t["embed"].view(c["vocab"], -1, BLOCK["Q6_K"][1])
    x = decoded("Q6_K", emb[t["tokens"].long()].reshape(-1, BLOCK["Q6_K"][1]), n, H)
    at = torch.arange(n, device="cuda")

    def mul(v, name, l, r, k):
        return v @ decoded(c["fmt"], t[f"{name}{l}"], r, k).T.contiguous()

    for l in range(c["layers"]):
        z = _rms(x, t[f"an{l}"])
        q, k, v = (mul(z, m, l, r, H).view(n, -1, 128) for m, r in (("q", Q), ("k", KV),
                                                                    ("v", KV)))
        q, k = _rms(_rope(q, at), t[f"qn{l}"]), _rms(_rope(k, at), t[f"kn{l}"])
        x = x + mul(_attend(q, k, v, 0).reshape(n, Q), "o", l, H, Q)
        z = _rms(x, t[f"fn{l}"])
        x = x + mul(_silu(mul(z, "gate", l, F, H)) * mul(z, "up", l, F, H), "down", l, H, F)
    z = _quantized(_rms(x[-1], t["on"]))
    logits = torch.empty(c["vocab"], device="cuda", dtype=torch.float64)
    for r in range(0, c["vocab"], 16384):
        r1 = min(c["vocab"], r + 16384)
        logits[r:r1] = decoded("Q6_K", emb[r:r1].reshape(-1, BLOCK["Q6_K"][1]), r1 - r, H) @ z
    return {"logits": logits, "token": None}
