"""End to end: the BERT-encoder runner (all mul_mats on the quantized GPU path, the
other ops as fp32 kernels) against the CPU reference encoder on the same weight bytes
and token ids.  Gate: cosine of the pooled embeddings >= 0.99999."""
import ctypes

import numpy as np
import pytest

import bert_oracle
import oracle_ffi as O
from gpu_util import host, stream

pytestmark = pytest.mark.gpu

COSINE_MIN = 0.99999
SMALL = dict(n_layer=2, n_embd=128, n_head=4, n_ff=512, n_vocab=1000, n_max_pos=64, n_type=2, layer_norm_eps=1e-12)


def _run(hp, wtype, B, T, name):
    import torch
    from crispembed_amd import bert, synth
    W = bert.synthetic_weights(hp, wtype, name=name)
    ids = synth.integers(f"{name}/ids_{B}x{T}", (B, T), min(1000, hp["n_vocab"] // 2), hp["n_vocab"] - 1)
    enc = bert.BertEncoder(hp, wtype, W)
    ids_d = torch.from_numpy(ids.ravel().copy()).cuda()
    out = torch.empty((B, hp["n_embd"]), dtype=torch.float32, device="cuda")
    hid = torch.empty((B * T, hp["n_embd"]), dtype=torch.float32, device="cuda")
    enc.encode(ids_d.data_ptr(), B, T, out.data_ptr(), stream(), hidden_dev=hid.data_ptr())
    return W, ids, host(out), host(hid)


def _check(hp, wtype, B, T, name, oracle, variant=O.Q8_0_X86):
    W, ids, pooled, hidden = _run(hp, wtype, B, T, name)
    ref_pooled, ref_hidden = bert_oracle.encode(oracle, hp, wtype, W, ids, variant=variant)
    cos = (pooled * ref_pooled).sum(-1) / (np.linalg.norm(pooled, axis=-1) * np.linalg.norm(ref_pooled, axis=-1))
    rel = np.abs(hidden - ref_hidden).max() / np.abs(ref_hidden).max()
    row = (np.linalg.norm(hidden - ref_hidden, axis=1) / np.linalg.norm(ref_hidden, axis=1)).max()
    print(f"{name}: min cosine {cos.min():.8f}, hidden max rel err {rel:.2e}, worst row {row:.2e}")
    assert np.isfinite(pooled).all()
    assert np.allclose(np.linalg.norm(pooled, axis=-1), 1.0, atol=1e-5)
    assert cos.min() >= COSINE_MIN
    return cos.min(), rel, row


@pytest.mark.parametrize("wtype", [O.Q8_0, O.Q4_K, O.Q6_K, O.F16])
def test_small_encoder(oracle, wtype):
    hp = dict(SMALL)
    if wtype in (O.Q4_K, O.Q6_K):
        hp.update(n_embd=256, n_head=4, n_ff=512)  # K-quants need k % 256 == 0
    _check(hp, wtype, 3, 16, f"small_{wtype}", oracle)


@pytest.mark.parametrize("B,T", [(2, 4), (1, 16), (2, 16)])
def test_small_encoder_gemv_rows(oracle, B, T, monkeypatch):
    """The runner's general path at a few rows (MQ_BERT_ROWS=0: no few-row layers): B*T <= 8, where every
    mul_mat takes the GEMV path, and 9-32 rows, where the FFN-down product is the GEMM's."""
    monkeypatch.setenv("MQ_BERT_ROWS", "0")
    _check(dict(SMALL), O.Q8_0, B, T, "small_gemv", oracle)


def test_minilm_l6_full_batch(oracle):
    """MiniLM-L6 shape, Q8_0, 32 sequences x 128 tokens (the embeddings/sec workload)."""
    from crispembed_amd import bert
    _check(dict(bert.MINILM_L6), O.Q8_0, 32, 128, "minilm", oracle)


@pytest.mark.parametrize("n_head", [8, 4, 2])
def test_q8_0_fused_path_head_dims(oracle, n_head):
    """The runner's Q8_0 path with every producer quantizing for its GEMM (norm, attention, FFN-up)
    and K / V written by the qkv GEMM as attention fragments, at head_dim 32, 64 and 128 (128:
    the attention's rows quantized after it)."""
    hp = dict(SMALL)
    hp.update(n_embd=256, n_head=n_head, n_ff=512, n_max_pos=128)
    _check(hp, O.Q8_0, 8, 64, f"fused_hd{256 // n_head}", oracle)


def test_kv_direct_equals_kv_pass(monkeypatch):
    """K / V fragments stored by the qkv GEMM are the bytes the attention's K / V pass writes:
    embeddings and hidden states bit-identical with MQ_BERT_KV_PASS=1 (the separate pass)."""
    hp = dict(SMALL)
    hp.update(n_embd=256, n_head=4, n_ff=512, n_max_pos=128)
    a = _run(hp, O.Q8_0, 8, 64, "kvd")
    monkeypatch.setenv("MQ_BERT_KV_PASS", "1")
    b = _run(hp, O.Q8_0, 8, 64, "kvd")
    assert np.array_equal(a[2], b[2]) and np.array_equal(a[3], b[3])


@pytest.mark.parametrize("H,nh,F,B,T", [
    (384, 12, 1536, 1, 1), (384, 12, 1536, 1, 31), (384, 12, 1536, 11, 3), (384, 12, 1536, 4, 32), (128, 4, 160, 3, 11),
    (512, 8, 512, 4, 32), (768, 12, 3072, 2, 32), (1024, 8, 4096, 5, 7), (96, 3, 544, 1, 16), (256, 2, 512, 1, 1),
    (256, 2, 512, 1, 16), (1024, 8, 4096, 2, 14), (128, 1, 160, 3, 31)])
@pytest.mark.parametrize("variant", [0, 1, 2])
def test_few_rows(oracle, H, nh, F, B, T, variant):
    """The Q8_0 runner at a few rows: the few-row layers up to 32 rows (head_dim 128: up to 128 where no
    other path takes it), the GEMM path past them, edges of the 32-row tiles and of the 32-key
    attention, rows of every register width, widths that are no multiple of 128, the three rounding
    variants of the quantizer, against the CPU encoder.  Every row's hidden state is within 2e-2: a
    rounding moves an 8-bit value by 1/127 of its block's largest, 1e-3 of a row over K >= 384 (4e-3
    over the smallest K here), and a handful of the eight products' values meet such a tie; a wrong row
    or column of a tile is off by its own size."""
    from crispembed_amd import mq
    hp = dict(SMALL)
    hp.update(n_embd=H, n_head=nh, n_ff=F, n_max_pos=128)
    L = mq.lib()
    saved = L.mq_q8_0_variant()
    mq.check(L.mq_set_q8_0_variant(variant))
    try:
        assert _check(hp, O.Q8_0, B, T, f"rows_{H}_{F}", oracle, variant)[2] <= 2e-2
    finally:
        mq.check(L.mq_set_q8_0_variant(saved))


@pytest.mark.parametrize("H,nh,F,B,T", [
    *[(96, 3, 544, 1, t) for t in range(1, 33)], *[(128, 2, 160, 1, t) for t in range(1, 33)],
    (384, 12, 1536, 1, 16), (384, 12, 1536, 2, 4), (384, 6, 1536, 3, 3), (384, 12, 1536, 2, 16), (384, 12, 1536, 11, 3),
    (512, 8, 2048, 4, 8), (768, 12, 3072, 2, 13), (1024, 16, 4096, 1, 31), (1024, 32, 4064, 5, 6), (992, 31, 32, 1, 9)])
def test_few_rows_equal_the_general_path(H, nh, F, B, T, monkeypatch):
    """The few-row layers change launches, not values: embeddings and hidden states are the bits of the
    general path (MQ_BERT_ROWS=0), at every sequence length (the attention's key ranges and blocks
    follow it), head_dim 32 and 64, row widths that are no multiple of 64 and of every step count,
    under and over the 8 rows at which the FFN-down product's sums change, and just past 32 rows."""
    hp = dict(SMALL)
    hp.update(n_embd=H, n_head=nh, n_ff=F)
    a = _run(hp, O.Q8_0, B, T, f"rows_eq_{H}_{nh}")
    monkeypatch.setenv("MQ_BERT_ROWS", "0")
    b = _run(hp, O.Q8_0, B, T, f"rows_eq_{H}_{nh}")
    assert np.array_equal(a[3], b[3]) and np.array_equal(a[2], b[2])


def _variant_blocks(n):
    """n values >= 6 (multiples of 32: Q8_0 blocks) that the three rounding variants quantize differently:
    in every other block the scale is 1 and the values are ties (REF rounds them away from 0, the
    others to even); in the rest 127 / max and 1 / (max / 127) are different floats and some values lie
    where one rounds up and the other down (X86 against NEON and REF)."""
    f = np.float32
    tie = np.array([127.0] + [6.5 + 2 * (i % 50) for i in range(31)], f)
    rng = np.random.default_rng(3)
    best = []
    while len(best) < 16:
        amax = f(rng.uniform(64, 127))
        a, b = f(127) / amax, f(1) / (amax / f(127))
        best = []
        for j in range(16, 127):
            x = f((j + 0.5) / np.float64(a))
            for c in (np.nextafter(x, f(0)), x, np.nextafter(x, f(999))):
                if np.rint(c * a) != np.rint(c * b):
                    best.append(c)
                    break
    edge = np.array(([amax] + best * 2)[:32], f)
    return np.concatenate([tie if i % 2 == 0 else edge for i in range(n // 32)])


@pytest.mark.parametrize("store", ["embedding", "attention", "norm1", "norm2", "gelu"])
@pytest.mark.parametrize("B,T", [(3, 1), (16, 1)])
def test_few_rows_quantizer_variants(store, B, T, monkeypatch):
    """Each place where the few-row layers quantize an activation follows the rounding variant: the
    values there are made constants that the three variants quantize differently (a LayerNorm weight of
    0 leaves its bias; one token attends to itself, so a V weight of 0 leaves V's bias; GELU is the
    identity on an FFN-up bias >= 6).  The outputs of the variants differ, and each is the general
    path's, whose quantizer is tested by itself, bit for bit."""
    import torch
    from crispembed_amd import bert, mq, synth
    hp = dict(SMALL)
    hp.update(n_embd=128, n_head=4, n_ff=160)
    W = bert.synthetic_weights(hp, O.Q8_0, name="variants")
    H, zero = _variant_blocks(128), np.zeros(128, np.float32)
    lay = W["layers"][0]
    if store == "embedding":
        W["ln_w"], W["ln_b"] = zero, H
    elif store == "attention":
        lay["wv"], lay["bv"] = np.zeros_like(lay["wv"]), H
    elif store == "norm1":
        lay["ln1_w"], lay["ln1_b"] = zero, H
    elif store == "norm2":
        lay["ln2_w"], lay["ln2_b"] = zero, H
    else:
        lay["wfc1"], lay["bfc1"] = np.zeros_like(lay["wfc1"]), _variant_blocks(160)
    enc = bert.BertEncoder(hp, O.Q8_0, W)
    ids = torch.from_numpy(synth.integers("variants/ids", (B * T,), 400, 999).copy()).cuda()
    L = mq.lib()
    saved, seen = L.mq_q8_0_variant(), []
    try:
        for variant in (0, 1, 2):
            mq.check(L.mq_set_q8_0_variant(variant))
            got = []
            for rows in ("32", "0"):
                monkeypatch.setenv("MQ_BERT_ROWS", rows)
                out = torch.empty((B, 128), dtype=torch.float32, device="cuda")
                hid = torch.empty((B * T, 128), dtype=torch.float32, device="cuda")
                enc.encode(ids.data_ptr(), B, T, out.data_ptr(), stream(), hidden_dev=hid.data_ptr())
                got.append(host(hid).copy())
            assert np.array_equal(got[0], got[1])
            seen.append(got[0])
    finally:
        mq.check(L.mq_set_q8_0_variant(saved))
    for i, j in ((0, 1), (1, 2), (0, 2)):
        assert not np.array_equal(seen[i], seen[j])


@pytest.mark.parametrize("n_head,B,T", [(12, 1, 16), (12, 2, 16), (3, 1, 30)])
def test_short_encode_captured_after_a_long_one(n_head, B, T):
    """A handle that has encoded its largest batch allocates nothing for a shorter one, whatever layers
    that takes: the short encode is captured (an allocation would break the capture) and every replay
    gives the eager bits, with other work between the replays."""
    import torch
    from crispembed_amd import bert, synth
    hp = dict(SMALL)
    hp.update(n_embd=384, n_head=n_head, n_ff=1536)
    enc = bert.BertEncoder(hp, O.Q8_0, bert.synthetic_weights(hp, O.Q8_0, name="cap"))
    ids = torch.from_numpy(synth.integers("cap/ids", (8, 64), 400, 999).ravel().copy()).cuda()
    big = torch.empty((8, 384), dtype=torch.float32, device="cuda")
    out = torch.empty((B, 384), dtype=torch.float32, device="cuda")
    hid = torch.empty((B * T, 384), dtype=torch.float32, device="cuda")
    side = torch.cuda.Stream()

    def encode(b, t, o, h=None):
        enc.encode(ids.data_ptr(), b, t, o.data_ptr(), ctypes.c_void_p(side.cuda_stream),
                   hidden_dev=h.data_ptr() if h is not None else None)

    torch.cuda.synchronize()
    encode(8, 64, big)
    side.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        encode(B, T, out, hid)
    torch.cuda.synchronize()
    encode(B, T, out, hid)
    side.synchronize()
    ref = host(out).copy(), host(hid).copy()
    for _ in range(3):
        encode(8, 64, big)
        side.synchronize()
        out.fill_(float("nan")), hid.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        assert np.array_equal(host(out), ref[0]) and np.array_equal(host(hid), ref[1])
