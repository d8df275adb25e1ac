"""The work that users of this framework have it do, as cases that can be timed and checked.

Every case goes through the public entry points (the C ABI of include/*.h by way of
crispembed_amd.mq, and the encoder / decoder runners).  The kinds:

  mul_mat   one GGML_OP_MUL_MAT: fp32 rows in, fp32 rows out, any weight type
  ffn       an encoder's feed-forward block: up projection, bias, GELU, down projection, bias
  decode    the mat-muls of one decode step of a whole decoder (q|k|v, o, gate|up, down per layer)
  attn      an encoder's attention over a padded batch (ggml_flash_attn_ext with an F16 mask)
  causal    a decoder's attention over q|k|v rows, grouped-query, causal
  bert      the BERT-encoder runner, token ids to pooled embeddings
  decoder   the decoder-embedder runner, token ids to pooled embeddings

Weights are quantized here by plain rounding (no scale search), in GGUF's block layouts, from
N(0, 0.02); activations are N(0, 1), as a normalised layer input is.
"""
import ctypes
import math

import numpy as np
import torch

from crispembed_amd import mq
from crispembed_amd.bert import BertEncoder
from crispembed_amd.decoder import DecoderEmbedder

TYPES = {"q8_0": mq.TYPE_Q8_0, "q4_K": mq.TYPE_Q4_K, "q6_K": mq.TYPE_Q6_K, "f16": mq.TYPE_F16}
BLOCK = {"q8_0": (32, 34), "q4_K": (256, 144), "q6_K": (256, 210), "f16": (1, 2)}  # values, bytes


# ------------------------------------------------------------------------------- cases ----
def listed():
    return [
        # the FFN-up product of a MiniLM-L6 batch of 32 x 128 tokens
        dict(name="mul_mat_q8_0_minilm_up", kind="mul_mat", type="q8_0", m=4096, n=1536, k=384),
        # the FFN-up product of XLM-R-large / BGE-M3, 16 x 512 tokens
        dict(name="mul_mat_q4_K_bge_up", kind="mul_mat", type="q4_K", m=8192, n=4096, k=1024),
        # a ragged batch of a few sentences through a layer whose width is no tile multiple
        dict(name="mul_mat_q6_K_ragged", kind="mul_mat", type="q6_K", m=517, n=1096, k=3072),
        # an unquantized model's projection over a medium batch
        dict(name="mul_mat_f16_medium", kind="mul_mat", type="f16", m=2048, n=1024, k=1024),
        # the logits of one new token: Qwen3-VL-2B's lm_head
        dict(name="mul_mat_q6_K_lm_head", kind="mul_mat", type="q6_K", m=1, n=151936, k=2048),
        # the whole feed-forward block of BGE-M3 over 16 x 512 tokens
        dict(name="ffn_q4_K_bge", kind="ffn", type="q4_K", m=8192, h=1024, f=4096),
        # one decode step of Qwen3-VL-2B's text decoder, one sequence
        dict(name="decode_q4_K_one_token", kind="decode", type="q4_K", m=1, layers=28, h=2048, f=6144, q=2048, kv=1024),
        # attention of a base-size encoder over a padded batch of uneven sentences
        dict(name="attn_padded_hd64", kind="attn", B=16, T=203, heads=12, hd=64),
        # attention of Qwen3-Embedding-0.6B over 16 documents of 512 tokens
        dict(name="causal_qwen3_16x512", kind="causal", B=16, T=512, heads=16, kv_heads=8, hd=128),
        # one short query through MiniLM-L6: latency
        dict(name="bert_minilm_one_sentence", kind="bert", type="q8_0", B=1, T=16, layers=6, h=384, heads=12, f=1536),
        # a batch of documents through MiniLM-L6: throughput
        dict(name="bert_minilm_32x128", kind="bert", type="q8_0", B=32, T=128, layers=6, h=384, heads=12, f=1536),
        # a batch of documents through layers of Qwen3-Embedding-0.6B's shape
        dict(name="decoder_qwen3_16x512", kind="decoder", type="q4_K", B=16, T=512, layers=4, h=1024, heads=16,
             kv_heads=8, hd=128, f=3072),
    ]


def draw(rng):
    def logint(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["mul_mat", "mul_mat", "mul_mat", "mul_mat", "ffn", "decode", "attn", "causal", "bert",
                       "decoder"])
    if kind == "mul_mat":
        t = rng.choice(["q8_0", "q4_K", "q4_K", "q6_K", "f16"])
        k = 256 * logint(1, 24) if t in ("q4_K", "q6_K") else 32 * logint(4, 160)
        n = logint(64, 6144)
        m = logint(1, min(8192, max(64, 2 ** 35 // (n * k))))
        return dict(kind=kind, type=t, m=m, n=n, k=k)
    if kind == "ffn":
        h = rng.choice([384, 768, 1024])
        t = "q8_0" if h == 384 else rng.choice(["q8_0", "q4_K", "q4_K", "q6_K"])
        return dict(kind=kind, type=t, m=logint(33, 8192), h=h, f=4 * h)
    if kind == "decode":
        h, f, q, kv = rng.choice([(2048, 6144, 2048, 1024), (1024, 3072, 2048, 1024)])
        return dict(kind=kind, type=rng.choice(["q4_K", "q6_K"]), m=rng.randint(1, 8), layers=rng.choice([12, 28]), h=h,
                    f=f, q=q, kv=kv)
    if kind == "attn":
        T = logint(16, 512)
        return dict(kind=kind, B=logint(1, max(1, 4096 // T)), T=T, heads=rng.choice([6, 12, 16]),
                    hd=rng.choice([32, 64]))
    if kind == "causal":
        T = logint(16, 1024)
        heads, kv = rng.choice([(16, 8), (8, 8), (14, 2)])
        return dict(kind=kind, B=logint(1, max(1, 8192 // T)), T=T, heads=heads, kv_heads=kv, hd=rng.choice([64, 128]))
    if kind == "bert":
        T = logint(4, 512)
        t = rng.choice(["q8_0", "q8_0", "q4_K", "f16"])
        h, heads, f = (384, 12, 1536) if t == "q8_0" else (768, 12, 3072)
        return dict(kind=kind, type=t, B=logint(1, max(1, 4096 // T)), T=T, layers=6 if h == 384 else 3, h=h, heads=heads,
                    f=f)
    T = logint(8, 512)
    return dict(kind="decoder", type=rng.choice(["q4_K", "q4_K", "q6_K"]), B=logint(1, max(1, 8192 // T)), T=T, layers=4,
                h=1024, heads=16, kv_heads=8, hd=128, f=3072)


# ---------------------------------------------------------------------- GGUF weights ----
class Rand:
    """Seeded device tensors."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def normal(self, *shape, std=1.0, mean=0.0):
        return torch.randn(*shape, generator=self.g, device="cuda", dtype=torch.float32).mul_(std).add_(mean)

    def ints(self, lo, hi, *shape):
        return torch.randint(lo, hi, shape, generator=self.g, device="cuda", dtype=torch.int32)

    def weight(self, t, n, k, std=0.02):
        """GGUF rows of an n x k weight, uint8 [n, row bytes]."""
        rows = max(1, (1 << 26) // k)  # a few hundred MB at a time
        return torch.cat([quantize(t, self.normal(min(rows, n - r), k, std=std)) for r in range(0, n, rows)])


def f16_bytes(x):
    return x.to(torch.float16).unsqueeze(-1).view(torch.uint8)


def quantize(t, w):
    n, k = w.shape
    if t == "f16":
        return w.to(torch.float16).view(torch.uint8)
    if t == "q8_0":
        b = w.view(-1, 32)
        d = (b.abs().amax(1) / 127).to(torch.float16)
        q = torch.round(b / d.float().clamp_min(1e-12)[:, None]).clamp(-127, 127).to(torch.int8)
        return torch.cat([f16_bytes(d), q.view(torch.uint8)], 1).view(n, -1)
    if t == "q4_K":
        b = w.view(-1, 8, 32)
        lo = b.amin(2).clamp_max(0)
        step = (b.amax(2) - lo) / 15
        d = (step.amax(1) / 63).to(torch.float16)
        dm = ((-lo).amax(1) / 63).to(torch.float16)
        df, dmf = d.float().clamp_min(1e-12)[:, None], dm.float().clamp_min(1e-12)[:, None]
        sc, mn = torch.round(step / df).clamp(0, 63), torch.round(-lo / dmf).clamp(0, 63)
        q = torch.round((b + (dmf * mn)[..., None]) / (df * sc).clamp_min(1e-12)[..., None]).clamp(0, 15).to(torch.uint8)
        sc, mn = sc.to(torch.uint8), mn.to(torch.uint8)
        packed = torch.cat([sc[:, :4] | (sc[:, 4:] >> 4 << 6), mn[:, :4] | (mn[:, 4:] >> 4 << 6),
                            (sc[:, 4:] & 15) | (mn[:, 4:] & 15) << 4], 1)
        qs = (q[:, 0::2] | q[:, 1::2] << 4).reshape(-1, 128)
        return torch.cat([f16_bytes(d), f16_bytes(dm), packed, qs], 1).view(n, -1)
    b = w.view(-1, 16, 16)  # q6_K
    big = torch.gather(b, 2, b.abs().argmax(2, keepdim=True))[..., 0]
    step = -big / 32
    top = torch.gather(step, 1, step.abs().argmax(1, keepdim=True))[:, 0]
    d = (-top / 128).to(torch.float16)
    df = torch.where(d == 0, torch.full_like(top, 1e-12), d.float())[:, None]
    sc = torch.round(step / df).clamp(-128, 127)
    s = df * sc
    q = torch.round(b / torch.where(s == 0, torch.full_like(s, 1e-12), s)[..., None]).clamp(-32, 31).add(32)
    q = q.to(torch.uint8).view(-1, 2, 4, 32)
    low = q & 15
    ql = torch.cat([low[:, :, 0] | low[:, :, 2] << 4, low[:, :, 1] | low[:, :, 3] << 4], 2).reshape(-1, 128)
    h = q >> 4
    qh = (h[:, :, 0] | h[:, :, 1] << 2 | h[:, :, 2] << 4 | h[:, :, 3] << 6).reshape(-1, 64)
    return torch.cat([ql, qh, sc.to(torch.int8).view(torch.uint8), f16_bytes(d)], 1).view(n, -1)


def dequantize(t, rows, k):
    """The values that GGUF rows stand for, fp64 [n, k]."""
    n = rows.shape[0]
    if t == "f16":
        return rows.view(torch.float16).double()
    b = rows.reshape(-1, BLOCK[t][1])

    def half(i):
        return b[:, i:i + 2].contiguous().view(torch.float16).double()

    if t == "q8_0":
        return (half(0) * b[:, 2:].contiguous().view(torch.int8).double()).view(n, k)
    if t == "q4_K":
        s = b[:, 4:16]
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | (s[:, :4] >> 6 << 4)], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | (s[:, 4:8] >> 6 << 4)], 1).double()
        qs = b[:, 16:].reshape(-1, 4, 32)
        q = torch.stack([qs & 15, qs >> 4], 2).view(-1, 8, 32).double()
        return (q * (half(0) * sc)[..., None] - (half(2) * mn)[..., None]).view(n, k)
    ql, qh = b[:, :128].reshape(-1, 2, 64), b[:, 128:192].reshape(-1, 2, 32)
    sc = b[:, 192:208].contiguous().view(torch.int8).double()
    q = torch.stack([(ql[:, :, :32] & 15) | (qh & 3) << 4, (ql[:, :, 32:] & 15) | (qh >> 2 & 3) << 4,
                     (ql[:, :, :32] >> 4) | (qh >> 4 & 3) << 4, (ql[:, :, 32:] >> 4) | (qh >> 6) << 4], 2)
    return ((q.double() - 32).view(-1, 16, 16) * (half(208) * sc)[..., None]).view(n, k)


def act_values(t, x):
    """The values an fp32 activation stands for after ggml's activation quantization, fp64."""
    x = x.to(torch.float32)
    if t == "f16":
        return x.to(torch.float16).double()
    if t == "q8_0":
        b = x.reshape(-1, 32)
        amax = b.abs().amax(1, keepdim=True).double()
        inv = torch.where(amax > 0, 127 / amax, torch.zeros_like(amax)).float()
        return ((amax / 127).float().to(torch.float16).double() * torch.round(b * inv).double()).view(x.shape)
    b = x.reshape(-1, 256)
    big = torch.gather(b, 1, b.abs().argmax(1, keepdim=True)).double()
    inv = torch.where(big != 0, -127 / big, torch.zeros_like(big)).float()
    d = torch.where(inv != 0, 1 / inv.double(), torch.zeros_like(big)).float().double()
    return (d * torch.round(inv * b).clamp_max(127).double()).view(x.shape)


def product(t, x, rows, bias=None):
    """x (requantized as ggml does) times the weight's values, fp64."""
    k = x.shape[-1]
    y = act_values(t, x) @ dequantize(t, rows, k).t()
    return y if bias is None else y + bias.double()


# ------------------------------------------------------------------------ the library ----
def ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def ptrs(ts):
    return (ctypes.c_void_p * len(ts))(*[t.data_ptr() for t in ts])


def i64s(v):
    return (ctypes.c_int64 * len(v))(*v)


def image(t, rows, k):
    """A prepared weight image on the device."""
    L, n = mq.lib(), rows.shape[0]
    img = torch.empty(L.mq_weight_image_bytes(TYPES[t], n, k), dtype=torch.uint8, device="cuda")
    img[:rows.numel()] = rows.reshape(-1)
    mq.check(L.mq_weight_prepare(TYPES[t], ptr(img), n, k, 0, n, stream()))
    return img


def workspace(t, m, k):
    return torch.empty(mq.lib().mq_workspace_bytes(TYPES[t], m, k), dtype=torch.uint8, device="cuda")


def host(t):
    return t.cpu().numpy()


# ---------------------------------------------------------------------------- mul_mat ----
def mul_mat_inputs(c, seed):
    r = Rand(seed)
    return r.weight(c["type"], c["n"], c["k"]), r.normal(c["m"], c["k"])


def mul_mat_prepare(c, seed):
    rows, x = mul_mat_inputs(c, seed)
    return dict(x=x, img=image(c["type"], rows, c["k"]), ws=workspace(c["type"], c["m"], c["k"]),
                y=torch.empty(c["m"], c["n"], device="cuda"))


def mul_mat_run(c, s):
    mq.check(mq.lib().mq_mul_mat(TYPES[c["type"]], ptr(s["img"]), c["n"], c["k"], ptr(s["x"]), c["k"], c["m"], ptr(s["y"]),
                                 c["n"], ptr(s["ws"]), s["ws"].numel(), stream()))
    return s["y"]


def mul_mat_exact(c, seed):
    rows, x = mul_mat_inputs(c, seed)
    return torch.cat([product(c["type"], x, part) for part in rows.split(1 << 14)], 1)


# -------------------------------------------------------------------------------- ffn ----
def ffn_inputs(c, seed):
    r, t, h, f = Rand(seed), c["type"], c["h"], c["f"]
    return dict(up=r.weight(t, f, h), down=r.weight(t, h, f), x=r.normal(c["m"], h), b1=r.normal(f, std=0.02),
                b2=r.normal(h, std=0.02))


def ffn_prepare(c, seed):
    s, t, m = ffn_inputs(c, seed), c["type"], c["m"]
    up, down = image(t, s.pop("up"), c["h"]), image(t, s.pop("down"), c["f"])
    s.update(up=up, down=down, ws1=workspace(t, m, c["h"]), ws2=workspace(t, m, c["f"]),
             y=torch.empty(m, c["h"], device="cuda"))
    s["fused"] = mq.lib().mq_mul_mat_q_requant_supported(TYPES[t], TYPES[t], m, c["f"])
    s["mid"] = None if s["fused"] else torch.empty(m, c["f"], device="cuda")
    return s


def ffn_run(c, s):
    L, t, m, h, f, st, gemm = mq.lib(), TYPES[c["type"]], c["m"], c["h"], c["f"], stream(), mq.PATH_GEMM
    ws1, ws2 = s["ws1"], s["ws2"]
    mq.check(L.mq_quantize_act(t, ptr(s["x"]), h, m, h, ptr(ws1), ws1.numel(), gemm, st))
    if s["fused"]:
        mq.check(L.mq_mul_mat_q_requant(t, ptr(s["up"]), f, h, ptr(ws1), m, ptr(s["b1"]), mq.PRE_GELU_ERF, t, ptr(ws2),
                                        ws2.numel(), st))
    else:
        mq.check(L.mq_mul_mat_q(t, ptr(s["up"]), f, h, ptr(ws1), m, ptr(s["mid"]), f, gemm, st))
        mq.check(L.mq_quantize_act_ex(t, ptr(s["mid"]), f, m, f, ptr(s["b1"]), mq.PRE_GELU_ERF, ptr(ws2), ws2.numel(),
                                      gemm, st))
    mq.check(L.mq_mul_mat_q_ex(t, ptr(s["down"]), h, f, ptr(ws2), m, ptr(s["y"]), h, ptr(s["b2"]), gemm, st))
    return s["y"]


def gelu(x):
    return 0.5 * x * (1 + torch.erf(x / math.sqrt(2)))


def ffn_exact(c, seed):
    s, t = ffn_inputs(c, seed), c["type"]
    return product(t, gelu(product(t, s["x"], s["up"], s["b1"])), s["down"], s["b2"])


# ----------------------------------------------------------------------------- decode ----
def decode_shapes(c):
    """(group of out-features, in-features) of a layer's four products."""
    return [([c["q"], c["kv"], c["kv"]], c["h"]), ([c["h"]], c["q"]), ([c["f"], c["f"]], c["h"]), ([c["h"]], c["f"])]


def decode_inputs(c, seed):
    r = Rand(seed)
    return [[([r.weight(c["type"], n, k) for n in ns], r.normal(c["m"], k), r.normal(c["m"], k)) for ns, k in decode_shapes(c)]
            for _ in range(c["layers"])]


def decode_prepare(c, seed):
    """The step is captured once in a HIP graph and replayed for every token, as a serving loop does."""
    L, t, m = mq.lib(), TYPES[c["type"]], c["m"]
    calls, outs = [], [torch.empty(c["layers"], m, sum(ns), device="cuda") for ns, _ in decode_shapes(c)]
    for il, products in enumerate(decode_inputs(c, seed)):
        for i, (ws, x, x2) in enumerate(products):
            k, ns = x.shape[1], [w.shape[0] for w in ws]
            imgs = [image(c["type"], w, k) for w in ws]
            ys = outs[i][il].split(ns, 1)  # q|k|v and gate|up rows side by side
            args = (t, len(ws), ptrs(imgs), i64s(ns), k, ptr(x), k, ptr(x2) if i == 3 else None, k,
                    mq.PRE_SILU_MUL if i == 3 else mq.PRE_NONE, m, ptrs(ys), i64s([sum(ns)] * len(ns)), None)
            calls.append((args, imgs, x, x2))
    side = torch.cuda.Stream()

    def step():
        st = ctypes.c_void_p(side.cuda_stream)
        for args, *_ in calls:
            mq.check(L.mq_mul_mat_gemv(*args, st))

    torch.cuda.synchronize()
    step()
    side.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        step()
    torch.cuda.synchronize()
    return dict(graph=graph, calls=calls, outs=outs, side=side)


def decode_run(c, s):
    s["graph"].replay()
    return s["outs"]


def decode_exact(c, seed):
    outs = [[] for _ in decode_shapes(c)]
    for products in decode_inputs(c, seed):
        for i, (ws, x, x2) in enumerate(products):
            x = torch.nn.functional.silu(x.double()) * x2.double() if i == 3 else x
            outs[i].append(torch.cat([product(c["type"], x, w) for w in ws], 1))
    return [torch.stack(o) for o in outs]


# -------------------------------------------------------------------------- attention ----
def lengths(c, seed):
    """Token counts of a padded batch, the longest filling it."""
    n = torch.randint(max(1, c["T"] // 4), c["T"] + 1, (c["B"],), generator=torch.Generator().manual_seed(seed))
    n[0] = c["T"]
    return n


def attn_inputs(c, seed):
    r, h = Rand(seed), c["heads"] * c["hd"]
    qkv = r.normal(c["B"] * c["T"], 3 * h)
    live = torch.arange(c["T"])[None, :] < lengths(c, seed)[:, None]  # [B, key]
    mask = torch.where(live, 0.0, -math.inf)[:, None, None, :].expand(c["B"], 1, c["T"], c["T"])
    return qkv, mask.to(torch.float16).contiguous().cuda()


def attn_prepare(c, seed):
    B, T, nh, hd = c["B"], c["T"], c["heads"], c["hd"]
    h = nh * hd
    qkv, mask = attn_inputs(c, seed)
    out = torch.empty(B * T, h, device="cuda")

    def cols(i):  # [hd, T, heads, B] over the q|k|v rows
        return mq.view(qkv[:, i * h:], mq.TYPE_F32, (hd, T, nh, B), (4, 12 * h, 4 * hd, 12 * h * T))

    views = [cols(0), cols(1), cols(2), mq.view(mask), mq.view(out, mq.TYPE_F32, (hd, nh, T, B), (4, 4 * hd, 4 * h, 4 * h * T))]
    ws = torch.empty(mq.lib().mq_op_flash_attn_workspace_bytes(ctypes.byref(views[1])), dtype=torch.uint8, device="cuda")
    return dict(qkv=qkv, mask=mask, out=out, views=views, ws=ws)


def attn_run(c, s):
    mq.check(mq.lib().mq_op_flash_attn(*[ctypes.byref(v) for v in s["views"]], 1 / math.sqrt(c["hd"]), ptr(s["ws"]),
                                       s["ws"].numel(), stream()))
    return s["out"]


def attention(q, k, v, bias):
    """softmax(q k^T / sqrt(hd) + bias) v per head, fp64; q, k, v [B, T, heads, hd]."""
    q, k, v = (t.double().transpose(1, 2) for t in (q, k, v))
    g = q.shape[1] // k.shape[1]
    k, v = k.repeat_interleave(g, 1), v.repeat_interleave(g, 1)
    p = torch.softmax(torch.matmul(q, k.transpose(2, 3).contiguous()) / math.sqrt(q.shape[3]) + bias, 3)
    return torch.matmul(p, v).transpose(1, 2).flatten(2).flatten(0, 1)


def causal_bias(T):
    return torch.full((T, T), -math.inf, dtype=torch.float64, device="cuda").triu(1)


def attn_exact(c, seed):
    qkv, mask = attn_inputs(c, seed)
    return attention(*qkv.view(c["B"], c["T"], 3, c["heads"], c["hd"]).unbind(2), mask.double())


def causal_inputs(c, seed):
    return Rand(seed).normal(c["B"] * c["T"], (c["heads"] + 2 * c["kv_heads"]) * c["hd"])


def causal_prepare(c, seed):
    ws = mq.lib().mq_attention_workspace_bytes(c["B"], c["T"], c["kv_heads"], c["hd"])
    return dict(qkv=causal_inputs(c, seed), out=torch.empty(c["B"] * c["T"], c["heads"] * c["hd"], device="cuda"),
                ws=torch.empty(ws, dtype=torch.uint8, device="cuda"))


def causal_run(c, s):
    qkv, out = s["qkv"], s["out"]
    mq.check(mq.lib().mq_attention(ptr(qkv), qkv.shape[1], ptr(out), out.shape[1], c["B"], c["T"], c["heads"], c["kv_heads"],
                                   c["hd"], 1 / math.sqrt(c["hd"]), 1, ptr(s["ws"]), s["ws"].numel(), stream()))
    return out


def causal_exact(c, seed):
    qkv = causal_inputs(c, seed).view(c["B"], c["T"], -1, c["hd"])
    return attention(*qkv.split([c["heads"], c["kv_heads"], c["kv_heads"]], 2), causal_bias(c["T"]))


# ------------------------------------------------------------------------------- bert ----
VOCAB = 30522
EPS_LN, EPS_RMS, THETA = 1e-12, 1e-6, 1e6


def bert_inputs(c, seed):
    r, t, h, f = Rand(seed), c["type"], c["h"], c["f"]
    w = dict(tok=r.normal(VOCAB, h, std=0.02), pos=r.normal(512, h, std=0.02), type=r.normal(2, h, std=0.02),
             ln_w=r.normal(h, std=0.02, mean=1), ln_b=r.normal(h, std=0.02), layers=[])
    for _ in range(c["layers"]):
        lay = {}
        for nm, n, k in (("q", h, h), ("k", h, h), ("v", h, h), ("o", h, h), ("fc1", f, h), ("fc2", h, f)):
            lay["w" + nm], lay["b" + nm] = r.weight(t, n, k), r.normal(n, std=0.02)
        for nm in ("ln1", "ln2"):
            lay[nm + "_w"], lay[nm + "_b"] = r.normal(h, std=0.02, mean=1), r.normal(h, std=0.02)
        w["layers"].append(lay)
    return w, r.ints(1000, VOCAB, c["B"], c["T"])


def to_host(w):
    return {k: [to_host(lay) for lay in v] if k == "layers" else host(v) for k, v in w.items()}


def bert_prepare(c, seed):
    w, ids = bert_inputs(c, seed)
    hp = dict(n_layer=c["layers"], n_embd=c["h"], n_head=c["heads"], n_ff=c["f"], n_vocab=VOCAB, n_max_pos=512, n_type=2,
              layer_norm_eps=EPS_LN)
    return dict(model=BertEncoder(hp, TYPES[c["type"]], to_host(w)), ids=ids,
                out=torch.empty(c["B"], c["h"], device="cuda"),
                hidden=torch.empty(c["B"] * c["T"], c["h"], device="cuda"))


def model_run(c, s):
    s["model"].encode(s["ids"].data_ptr(), c["B"], c["T"], s["out"].data_ptr(), stream(), hidden_dev=s["hidden"].data_ptr())
    return dict(pooled=s["out"], hidden=s["hidden"])


def layer_norm(x, w, b):
    x = x.double()
    return torch.nn.functional.layer_norm(x, x.shape[-1:], w.double(), b.double(), EPS_LN)


def pool(rows):
    return rows / torch.sqrt((rows * rows).sum(1, keepdim=True).clamp_min(1e-12))


def bert_exact(c, seed):
    w, ids = bert_inputs(c, seed)
    t, B, T = c["type"], c["B"], c["T"]
    x = w["tok"].double()[ids.flatten().long()] + w["pos"].double()[:T].repeat(B, 1) + w["type"].double()[0]
    x = layer_norm(x, w["ln_w"], w["ln_b"])
    for lay in w["layers"]:
        qkv = [product(t, x, lay["w" + n], lay["b" + n]).view(B, T, c["heads"], -1) for n in "qkv"]
        x = layer_norm(x + product(t, attention(*qkv, 0.0), lay["wo"], lay["bo"]), lay["ln1_w"], lay["ln1_b"])
        mid = gelu(product(t, x, lay["wfc1"], lay["bfc1"]))
        x = layer_norm(x + product(t, mid, lay["wfc2"], lay["bfc2"]), lay["ln2_w"], lay["ln2_b"])
    return dict(pooled=pool(x.view(B, T, -1).mean(1)), hidden=x)


# ---------------------------------------------------------------------------- decoder ----
def decoder_inputs(c, seed):
    r, t, h, f, hd = Rand(seed), c["type"], c["h"], c["f"], c["hd"]
    qd, kvd = c["heads"] * hd, c["kv_heads"] * hd
    w = dict(tok=r.normal(VOCAB, h, std=0.02), out_norm=r.normal(h, std=0.02, mean=1), layers=[])
    for _ in range(c["layers"]):
        lay = {"w" + nm: r.weight(t, n, k) for nm, n, k in (("q", qd, h), ("k", kvd, h), ("v", kvd, h), ("o", h, qd),
                                                            ("gate", f, h), ("up", f, h), ("down", h, f))}
        for nm, n in (("attn_norm", h), ("ffn_norm", h), ("q_norm", hd), ("k_norm", hd)):
            lay[nm] = r.normal(n, std=0.02, mean=1)
        w["layers"].append(lay)
    return w, r.ints(0, VOCAB, c["B"], c["T"])


def decoder_prepare(c, seed):
    w, ids = decoder_inputs(c, seed)
    hp = dict(n_layer=c["layers"], n_embd=c["h"], n_head=c["heads"], n_kv_head=c["kv_heads"], head_dim=c["hd"],
              n_ff=c["f"], n_vocab=VOCAB, rms_norm_eps=EPS_RMS, rope_theta=THETA, causal=1, pooling=2)
    return dict(model=DecoderEmbedder(hp, TYPES[c["type"]], to_host(w)), ids=ids,
                out=torch.empty(c["B"], c["h"], device="cuda"),
                hidden=torch.empty(c["B"] * c["T"], c["h"], device="cuda"))


def rms_norm(x, w):
    x = x.double()
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS_RMS) * w.double()


def rope(x):
    """NEOX rotation of x [B, T, heads, hd] at positions 0 .. T-1."""
    T, half = x.shape[1], x.shape[3] // 2
    angle = torch.arange(T, device="cuda", dtype=torch.float64)[:, None] * \
        THETA ** (-torch.arange(half, device="cuda", dtype=torch.float64) / half)
    co, si = angle.cos()[None, :, None], angle.sin()[None, :, None]
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * co - b * si, a * si + b * co], 3)


def decoder_exact(c, seed):
    w, ids = decoder_inputs(c, seed)
    t, B, T, hd = c["type"], c["B"], c["T"], c["hd"]
    x, bias = w["tok"].double()[ids.flatten().long()], causal_bias(T)
    for lay in w["layers"]:
        y = rms_norm(x, lay["attn_norm"])
        q, k, v = (product(t, y, lay["w" + n]).view(B, T, -1, hd) for n in "qkv")
        a = attention(rope(rms_norm(q, lay["q_norm"])), rope(rms_norm(k, lay["k_norm"])), v, bias)
        x = x + product(t, a, lay["wo"])
        y = rms_norm(x, lay["ffn_norm"])
        y = torch.nn.functional.silu(product(t, y, lay["wgate"])) * product(t, y, lay["wup"])
        x = x + product(t, y, lay["wdown"])
    return dict(pooled=pool(rms_norm(x.view(B, T, -1)[:, -1], w["out_norm"])), hidden=x)


# ------------------------------------------------------------------------ entry points ----
KINDS = {
    "mul_mat": (mul_mat_prepare, mul_mat_run, mul_mat_exact),
    "ffn": (ffn_prepare, ffn_run, ffn_exact),
    "decode": (decode_prepare, decode_run, decode_exact),
    "attn": (attn_prepare, attn_run, attn_exact),
    "causal": (causal_prepare, causal_run, causal_exact),
    "bert": (bert_prepare, model_run, bert_exact),
    "decoder": (decoder_prepare, model_run, decoder_exact),
}


def prepare(case, seed):
    s = KINDS[case["kind"]][0](case, seed)
    s["case"] = case
    return s


def run(state):
    return KINDS[state["case"]["kind"]][1](state["case"], state)


def exact(case, seed):
    return KINDS[case["kind"]][2](case, seed)


def weight_bytes(t, n, k):
    return n * k // BLOCK[t][0] * BLOCK[t][1]


def work(case):
    c, kind = case, case["kind"]
    if kind == "mul_mat":
        m, n, k = c["m"], c["n"], c["k"]
        return dict(bytes=weight_bytes(c["type"], n, k) + 4 * m * (n + k), flops=2 * m * n * k)
    if kind == "ffn":
        m, h, f = c["m"], c["h"], c["f"]
        return dict(bytes=2 * weight_bytes(c["type"], f, h) + 8 * m * h + 4 * (f + h), flops=4 * m * h * f)
    if kind == "decode":
        nk = [(sum(ns), k, 2 if i == 3 else 1) for i, (ns, k) in enumerate(decode_shapes(c))]
        return dict(bytes=c["layers"] * sum(weight_bytes(c["type"], n, k) + 4 * c["m"] * (n + g * k) for n, k, g in nk),
                    flops=c["layers"] * sum(2 * c["m"] * n * k for n, k, _ in nk))
    B, T = c["B"], c["T"]
    if kind == "attn":
        h = c["heads"] * c["hd"]
        return dict(bytes=16 * B * T * h + 2 * B * T * T, flops=4 * B * T * T * h)
    if kind == "causal":
        h, kv = c["heads"] * c["hd"], c["kv_heads"] * c["hd"]
        return dict(bytes=8 * B * T * (h + kv), flops=2 * B * T * (T + 1) * h)
    h, f, m, n = c["h"], c["f"], B * T, c["layers"]
    if kind == "bert":
        per, attn = 4 * h * h + 2 * h * f, 4 * m * T * h
    else:
        qd, kvd = c["heads"] * c["hd"], c["kv_heads"] * c["hd"]
        per, attn = h * (2 * qd + 2 * kvd) + 3 * h * f, 2 * m * (T + 1) * qd
    return dict(bytes=n * weight_bytes(c["type"], 1, per) + 4 * m * (1 + 2 * h) + 4 * B * h, flops=n * (2 * m * per + attn))


def tolerance(case):
    """About four times what the path shows against exact() over the ranges of draw()."""
    kind = case["kind"]
    if kind == "mul_mat":
        return {"rel": 1e-6}  # 4e-8 .. 2e-7: fp32 sums of exact products
    if kind == "decode":
        return {"rel": 1e-3}  # fp32 sums; the gated product's rounding can move one of its 8-bit values
    if kind in ("attn", "causal"):
        return {"rel": 3e-6}  # 5e-7: operands of 22 bits, fp32 sums
    if kind == "ffn":
        return {"rel": 2e-4}  # 5e-5: GELU values that another rounding moves to the next 8-bit value
    # whole models: those moves add up over the layers, and the decoder's residual stream starts
    # as small as what its layers add to it
    return {"rel": 1.5e-2} if kind == "bert" else {"rel": 8e-2}
