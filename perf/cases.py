"""Performance cases of the Q4_K / Q6_K path: what a program that serves a
Llama model calls, over the sizes it calls it with.

Every case goes through the public entry points (the package's functions, the
C ABI behind them, Runner and BatchRunner).  Weights are drawn as a
quantizer leaves them: Q4_K blocks whose mins centre the weights on zero, Q6_K
blocks whose scales use the whole int8 range.  Activations are normal with
a spread of channel gains.  exact() restates each path in float64 with plain
torch, without the package.

Kinds of case:
  qkv          one token's fused Q / K / V projection (FP32 arithmetic)
  head         one token's LM head with its greedy pick
  ffn          the feed-forward block of n tokens, FP32 arithmetic, one call a
               layer: n from a few sequences decoding together, through a
               decode batch, to a prefill chunk
  ffn_i8       the same in the INT8 arithmetic: x quantized, then the block
  multi        the fused projections of n tokens sharing x (QKV of a batch), in
               either arithmetic
  attn         attention of a ragged batch over the KV cache: sequences x
               chunk tokens at the end of each sequence's context
  norm         RMSNorm and per-32 quantization of n tokens in one call
  decode       a whole decode step of one sequence, with logits
  prefill      a whole batched step over one sequence's prompt chunk, with the
               last token's logits
"""
import ctypes
import importlib.util
import math
import pathlib
import sys

import numpy as np
import torch

PACKAGE = "inferencer_jetson_amd"
Q4, Q6, Q6S = 12, 14, 114
DEV = "cuda:0"

# Widths of the two models that the package's workloads use.
M1 = dict(dim=2048, hidden=8192, heads=32, kv_heads=8, vocab=128256)
M3 = dict(dim=3072, hidden=8192, heads=24, kv_heads=8, vocab=128256)


def _qk():
    if PACKAGE not in sys.modules:
        folder = pathlib.Path.cwd() / "inferencer-jetson_amd"
        spec = importlib.util.spec_from_file_location(PACKAGE, folder / "__init__.py",
                                                      submodule_search_locations=[str(folder)])
        mod = importlib.util.module_from_spec(spec)
        sys.modules[PACKAGE] = mod
        spec.loader.exec_module(mod)
    return sys.modules[PACKAGE]


# ------------------------------------------------------------------ cases --

def listed():
    return [
        # The smallest call of a decode step: one token's Q, K and V of the 1B.
        dict(name="qkv_1b_1", kind="qkv", dim=2048, kv_dim=512, v_type=Q6),
        # The largest matrix of a decode step: the tied LM head and the pick.
        dict(name="head_1b", kind="head", cols=2048, rows=128256, type=Q6S),
        # Four sequences decoding together (or four speculated tokens), 3B.
        dict(name="ffn_3b_4", kind="ffn", dim=3072, hidden=8192, tokens=4, layers=8, down_type=Q6),
        # A decode batch of 32 sequences, 3B, every layer's weights cold.
        dict(name="ffn_3b_32", kind="ffn", dim=3072, hidden=8192, tokens=32, layers=8, down_type=Q6S),
        # A prefill chunk of an odd length, 3B.
        dict(name="ffn_3b_517", kind="ffn", dim=3072, hidden=8192, tokens=517, layers=2, down_type=Q6S),
        # The decode batch and the prefill chunk in the INT8 arithmetic.
        dict(name="ffn_i8_3b_32", kind="ffn_i8", dim=3072, hidden=8192, tokens=32, layers=8, down_type=Q6S),
        dict(name="ffn_i8_3b_517", kind="ffn_i8", dim=3072, hidden=8192, tokens=517, layers=2, down_type=Q6S),
        # One layer's attention of 32 ragged sequences decoding, 1B heads.
        dict(name="attn_decode_32", kind="attn", heads=32, kv_heads=8, head_dim=64, seqs=32, chunk=1, ctx_lo=64,
             ctx_hi=2048),
        # One layer's attention of a 512-token prefill chunk that continues a
        # 600-token context, 3B heads.
        dict(name="attn_prefill_512", kind="attn", heads=24, kv_heads=8, head_dim=128, seqs=1, chunk=512, ctx_lo=1112,
             ctx_hi=1112),
        # The normalisation in front of a batched layer, 256 tokens.
        dict(name="norm_256", kind="norm", dim=3072, tokens=256),
        # A decode step of the 1B at position 700, FP32 arithmetic (what a new
        # runner computes in).
        dict(name="decode_1b", kind="decode", model="1b", layers=16, pos=700, context=1024, int8=False),
        # A prompt of 480 tokens through the 1B in one step, FP32 arithmetic.
        dict(name="prefill_1b_480", kind="prefill", model="1b", layers=16, tokens=480, pos=0, context=1024, int8=False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["qkv", "head", "ffn", "ffn", "ffn", "ffn_i8", "ffn_i8", "multi", "multi", "attn", "attn", "norm",
                       "decode", "prefill"])
    width = lambda lo, hi: 256 * _log(rng, lo, hi)
    if kind == "qkv":
        return dict(kind=kind, dim=width(4, 16), kv_dim=256 * rng.randint(1, 4), v_type=rng.choice([Q4, Q6, Q6S]))
    if kind == "head":
        return dict(kind=kind, cols=width(4, 12), rows=_log(rng, 16000, 130000), type=rng.choice([Q4, Q6, Q6S]))
    if kind in ("ffn", "ffn_i8"):
        return dict(kind=kind, dim=width(4, 12), hidden=width(16, 32), tokens=_log(rng, 2, 512), layers=2,
                    down_type=rng.choice([Q4, Q6, Q6S]))
    if kind == "multi":
        return dict(kind=kind, dim=width(4, 12), kv_dim=256 * rng.randint(1, 4), tokens=_log(rng, 2, 768),
                    v_type=rng.choice([Q4, Q6, Q6S]), int8=rng.random() < 0.4)
    if kind == "attn":
        heads, kv_heads, hd = rng.choice([(32, 8, 64), (24, 8, 128), (16, 8, 64), (8, 8, 128)])
        if rng.random() < 0.5:
            lo = _log(rng, 16, 1024)
            return dict(kind=kind, heads=heads, kv_heads=kv_heads, head_dim=hd, seqs=_log(rng, 1, 48), chunk=1,
                        ctx_lo=lo, ctx_hi=lo + rng.randint(0, 1024))
        chunk = _log(rng, 8, 512)
        lo = chunk + rng.randint(0, 700)
        return dict(kind=kind, heads=heads, kv_heads=kv_heads, head_dim=hd, seqs=max(1, min(4, 512 // chunk)),
                    chunk=chunk, ctx_lo=lo, ctx_hi=lo + rng.randint(0, 200))
    if kind == "norm":
        return dict(kind=kind, dim=width(4, 16), tokens=_log(rng, 1, 768))
    if kind == "decode":
        return dict(kind=kind, model=rng.choice(["1b", "3b"]), layers=rng.randint(2, 4), pos=_log(rng, 4, 1000),
                    context=1024, int8=rng.random() < 0.5)
    return dict(kind=kind, model=rng.choice(["1b", "3b"]), layers=rng.randint(2, 4), tokens=_log(rng, 9, 480),
                pos=rng.randint(0, 300), context=1024, int8=rng.random() < 0.3)


# ----------------------------------------------------------------- inputs --

def _gen(seed, stream):
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) * 1000003 + stream) % (1 << 62))
    return g


def _rand(shape, g, lo, hi):
    return torch.rand(shape, device=DEV, generator=g) * (hi - lo) + lo


def _halves(v):
    """fp16 bytes [.., 2] of float values."""
    return v.to(torch.float16).unsqueeze(-1).view(torch.uint8)


def _blocks(qtype, rows, nb, g):
    """rows x nb super-blocks in the GGUF layout, weights of about 0.02 rms."""
    if qtype == Q4:
        out = torch.randint(0, 256, (rows, nb, 144), dtype=torch.uint8, device=DEV, generator=g)
        sc = torch.randint(16, 64, (rows, nb, 8), dtype=torch.int32, device=DEV, generator=g)
        # The mins follow the scales: sub-blocks are centred on zero.
        mn = (sc + torch.randint(-2, 3, sc.shape, dtype=torch.int32, device=DEV, generator=g)).clamp(0, 63)
        a, b, m, n = sc[..., :4], sc[..., 4:], mn[..., :4], mn[..., 4:]
        packed = torch.cat([a | ((b >> 4) << 6), m | ((n >> 4) << 6), (b & 15) | ((n & 15) << 4)], -1)
        out[..., 4:16] = packed.to(torch.uint8)
        d = _rand((rows, nb), g, 0.7e-4, 1.5e-4).to(torch.float16).float()
        out[..., 0:2] = _halves(d)
        out[..., 2:4] = _halves(7.5 * d)
        return out
    out = torch.randint(0, 256, (rows, nb, 210), dtype=torch.uint8, device=DEV, generator=g)
    sc = torch.randint(40, 128, (rows, nb, 16), dtype=torch.int32, device=DEV, generator=g)
    sc = torch.where(torch.rand(sc.shape, device=DEV, generator=g) < 0.5, sc, -sc)
    sc[..., 0] = -128
    out[..., 192:208] = (sc & 255).to(torch.uint8)
    out[..., 208:210] = _halves(_rand((rows, nb), g, 0.8e-5, 1.6e-5))
    return out


def _weights(qtype, cols, rows, seed, stream):
    """Bytes of a quantized matrix as a GGUF file holds it (Q6 for either
    Q6_K layout)."""
    return _blocks(Q4 if qtype == Q4 else Q6, rows, cols // 256, _gen(seed, stream)).reshape(-1)


def _tensor(qk, qtype, cols, rows, seed, stream):
    t = qk.Tensor((cols, rows), Q4 if qtype == Q4 else Q6, _weights(qtype, cols, rows, seed, stream))
    return qk.split_q6k(t, torch.cuda.current_stream()) if qtype == Q6S else t


def _activations(n, cols, seed, stream):
    g = _gen(seed, stream)
    gains = torch.exp(0.5 * torch.randn(cols, device=DEV, generator=g))
    return torch.randn((n, cols), device=DEV, generator=g) * gains


def _empty(*shape, dtype=torch.float32):
    return torch.empty(shape, dtype=dtype, device=DEV)


def _buffer(nbytes):
    return torch.empty(max(int(nbytes), 256), dtype=torch.uint8, device=DEV)


def _contexts(case):
    """Context length of each sequence after its chunk, spread over the range."""
    lo, hi = case["ctx_lo"], case["ctx_hi"]
    return [max(case["chunk"], lo + int((hi - lo) * (((i + 1) * 0.6180339887) % 1.0))) for i in range(case["seqs"])]


def _attn_tokens(case):
    """(position, first cache row) of every token, and the cache's rows."""
    tokens, row = [], 0
    for ctx in _contexts(case):
        tokens += [(ctx - case["chunk"] + i, row) for i in range(case["chunk"])]
        row += ctx
    return tokens, row


def _config(case):
    m = M1 if case["model"] == "1b" else M3
    return dict(m, layers=case["layers"], context=case["context"], eps=1e-5, rope_theta=500000.0)


def _shapes(cfg):
    dim, hidden, kv = cfg["dim"], cfg["hidden"], cfg["dim"] // cfg["heads"] * cfg["kv_heads"]
    # The Q4_K_M mix: V and down in Q6_K, the rest in Q4_K.
    return [("q", Q4, dim, dim), ("k", Q4, dim, kv), ("v", Q6, dim, kv), ("o", Q4, dim, dim),
            ("gate", Q4, dim, hidden), ("up", Q4, dim, hidden), ("down", Q6, hidden, dim)]


def _model_parts(cfg, seed):
    """The model's matrices and norm gains, one at a time: (layer, name,
    type, cols, rows, bytes or gains).  Layer -1 holds the token table and
    the output norm."""
    def gains(stream):
        return _rand((cfg["dim"],), _gen(seed, stream), 0.6, 1.4)
    yield -1, "token_embd", Q6, cfg["dim"], cfg["vocab"], _weights(Q6, cfg["dim"], cfg["vocab"], seed, 7)
    yield -1, "output_norm", 0, cfg["dim"], 1, gains(8)
    for l in range(cfg["layers"]):
        for j, (name, qtype, cols, rows) in enumerate(_shapes(cfg)):
            yield l, name, qtype, cols, rows, _weights(qtype, cols, rows, seed, 100 + 16 * l + j)
        yield l, "attn_norm", 0, cfg["dim"], 1, gains(108 + 16 * l)
        yield l, "ffn_norm", 0, cfg["dim"], 1, gains(109 + 16 * l)


def _model_weights(cfg, seed):
    """The weights dictionary that Runner and BatchRunner take (host arrays)."""
    w = dict(embd_type=Q6, output=None, output_type=0, layers=[{} for _ in range(cfg["layers"])])
    for l, name, qtype, _, _, data in _model_parts(cfg, seed):
        where = w if l < 0 else w["layers"][l]
        where[name] = data.cpu().numpy()
        if l >= 0 and qtype:
            where[name + "_type"] = qtype
    return w


def _cache_rows(cfg, n, seed, stream):
    """Keys or values of positions 0..n-1, [layers][n][kv_dim]."""
    kv = cfg["dim"] // cfg["heads"] * cfg["kv_heads"]
    return torch.randn((cfg["layers"], n, kv), device=DEV, generator=_gen(seed, stream))


def _prompt(cfg, n, seed):
    return torch.randint(0, cfg["vocab"], (n,), device=DEV, generator=_gen(seed, 9)).tolist()


class _Buffer:
    """The CUDA array interface of a float32 device buffer."""

    def __init__(self, ptr, shape):
        self.__cuda_array_interface__ = dict(shape=shape, typestr="<f4", data=(ptr, False), version=2)


def _view(runner, ptr, shape):
    """The runner's own buffer as a tensor.  The buffer is freed with the
    runner, so the tensor holds on to it."""
    t = torch.as_tensor(_Buffer(ptr, shape), device=DEV)
    t.runner = runner
    return t


# --------------------------------------------------------------- the path --

def prepare(case, seed):
    qk = _qk()
    kind = case["kind"]
    s = dict(kind=kind, qk=qk, case=case, stream=torch.cuda.current_stream())
    if kind == "qkv":
        dim, kv = case["dim"], case["kv_dim"]
        s.update(x=_activations(1, dim, seed, 1)[0].contiguous(), q=_empty(dim), k=_empty(kv), v=_empty(kv),
                 wq=_tensor(qk, Q4, dim, dim, seed, 2), wk=_tensor(qk, Q4, dim, kv, seed, 3),
                 wv=_tensor(qk, case["v_type"], dim, kv, seed, 4))
    elif kind == "head":
        cols, rows = case["cols"], case["rows"]
        s.update(x=_activations(1, cols, seed, 1)[0].contiguous(), w=_tensor(qk, case["type"], cols, rows, seed, 2),
                 y=_empty(rows), token=_empty(1, dtype=torch.int32),
                 ws=_buffer(qk.lib().qk_gemv_argmax_workspace_bytes()))
    elif kind in ("ffn", "ffn_i8"):
        dim, hidden, n = case["dim"], case["hidden"], case["tokens"]
        s.update(x=_activations(n, dim, seed, 1), y=[_empty(n, dim) for _ in range(case["layers"])],
                 layers=[(_tensor(qk, Q4, dim, hidden, seed, 10 + 3 * l), _tensor(qk, Q4, dim, hidden, seed, 11 + 3 * l),
                          _tensor(qk, case["down_type"], hidden, dim, seed, 12 + 3 * l))
                         for l in range(case["layers"])])
        size = qk.lib().qk_ffn_batched_workspace_bytes if kind == "ffn" else \
            qk.lib().qk_ffn_batched_i8_workspace_bytes
        s.update(ws=_buffer(size(dim, hidden, n)))
        if kind == "ffn_i8":
            s.update(xq=_empty(n, dim, dtype=torch.int8), xs=_empty(n, dim // 32))
    elif kind == "multi":
        dim, kv, n = case["dim"], case["kv_dim"], case["tokens"]
        s.update(x=_activations(n, dim, seed, 1), q=_empty(n, dim), k=_empty(n, kv), v=_empty(n, kv),
                 wq=_tensor(qk, Q4, dim, dim, seed, 2), wk=_tensor(qk, Q4, dim, kv, seed, 3),
                 wv=_tensor(qk, case["v_type"], dim, kv, seed, 4))
        size = qk.lib().qk_gemv_batched_i8_workspace_bytes if case["int8"] else \
            qk.lib().qk_gemv_batched_workspace_bytes
        s.update(ws=_buffer(size(dim, dim + 2 * kv, n)))
        if case["int8"]:
            s.update(xq=_empty(n, dim, dtype=torch.int8), xs=_empty(n, dim // 32))
        s["mats"] = qk._matrices([(s["wq"], s["q"]), (s["wk"], s["k"]), (s["wv"], s["v"])])
    elif kind == "attn":
        heads, kvh, hd = case["heads"], case["kv_heads"], case["head_dim"]
        tokens, rows = _attn_tokens(case)
        g = _gen(seed, 1)
        desc = torch.tensor([[pos | (i << 32), row] for i, (pos, row) in enumerate(tokens)], dtype=torch.int64)
        top = max(pos for pos, _ in tokens)
        n = len(tokens)
        s.update(q=torch.randn((n, heads * hd), device=DEV, generator=g),
                 key=torch.randn((rows, kvh * hd), device=DEV, generator=g),
                 value=torch.randn((rows, kvh * hd), device=DEV, generator=g), desc=desc.to(DEV), top=top, rows=rows,
                 n=n, out=_empty(n, heads * hd))
        s.update(ws=_buffer(qk.lib().qk_attention_split_workspace_bytes(n, heads, kvh, hd, top, 0)))
    elif kind == "norm":
        n, dim = case["tokens"], case["dim"]
        s.update(x=_activations(n, dim, seed, 1), w=_rand((dim,), _gen(seed, 2), 0.6, 1.4), out=_empty(n, dim),
                 xq=_empty(n, dim, dtype=torch.int8), xs=_empty(n, dim // 32))
    elif kind == "decode":
        cfg = _config(case)
        run_ = qk.Runner(cfg, _model_weights(cfg, seed), s["stream"])
        if case["int8"]:
            run_.set_int8(True, True)
        keys = torch.zeros((cfg["layers"], cfg["context"], cfg["dim"] // cfg["heads"] * cfg["kv_heads"]))
        values = torch.zeros_like(keys)
        keys[:, :case["pos"]] = _cache_rows(cfg, case["pos"], seed, 5).cpu()
        values[:, :case["pos"]] = _cache_rows(cfg, case["pos"], seed, 6).cpu()
        run_.load_kv(keys.numpy(), values.numpy())
        s.update(runner=run_, token=_prompt(cfg, 1, seed)[0], cfg=cfg,
                 logits=_view(run_, run_.logits_ptr(), (cfg["vocab"],)))
    else:
        cfg = _config(case)
        n, pos = case["tokens"], case["pos"]
        run_ = qk.BatchRunner(cfg, _model_weights(cfg, seed), n, n + pos, s["stream"])
        if case["int8"]:
            run_.set_int8(True, True)
        if pos:
            run_.load_kv_rows(0, _cache_rows(cfg, pos, seed, 5).cpu().numpy(),
                              _cache_rows(cfg, pos, seed, 6).cpu().numpy())
        p = ctypes.c_void_p()
        qk.check(qk.lib().qk_llama_batch_logits(run_.handle, ctypes.byref(p)), "logits")
        s.update(runner=run_, tokens=_prompt(cfg, n, seed), positions=list(range(pos, pos + n)), zeros=[0] * n, cfg=cfg,
                 logits=_view(run_, p.value, (1, cfg["vocab"])))
    return s


def run(s):
    qk, kind, case, st = s["qk"], s["kind"], s["case"], s["stream"]
    lib, h = qk.lib(), s["stream"].cuda_stream
    if kind == "qkv":
        # As qkv() asks, V may be Q4_K or Q6_K in either layout.
        qk.qkv(s["wq"], s["wk"], s["wv"], s["x"], s["q"], s["k"], s["v"], case["dim"], case["kv_dim"], st)
        return [s["q"], s["k"], s["v"]]
    if kind == "head":
        qk.matvec_argmax(s["w"], s["x"], s["y"], s["token"], s["ws"], st)
        return [s["y"], s["token"]]
    if kind == "ffn":
        dim, hidden, n = case["dim"], case["hidden"], case["tokens"]
        for (g, u, d), y in zip(s["layers"], s["y"]):
            qk.check(lib.qk_ffn_batched_f32(g.type, g.gpu, u.type, u.gpu, d.type, d.gpu, s["x"].data_ptr(), dim,
                                            y.data_ptr(), dim, dim, hidden, n, 0, s["ws"].data_ptr(), s["ws"].numel(),
                                            h), "ffn")
        return list(s["y"])
    if kind == "ffn_i8":
        dim, hidden, n = case["dim"], case["hidden"], case["tokens"]
        qk.quantize(s["x"], s["xq"], s["xs"], dim, n, stream=st)
        for (g, u, d), y in zip(s["layers"], s["y"]):
            qk.check(lib.qk_ffn_batched_i8(g.type, g.gpu, u.type, u.gpu, d.type, d.gpu, s["xq"].data_ptr(), dim,
                                           s["xs"].data_ptr(), dim // 32, y.data_ptr(), dim, dim, hidden, n, 0,
                                           s["ws"].data_ptr(), s["ws"].numel(), h), "ffn_i8")
        return [s["xq"], s["xs"]] + list(s["y"])
    if kind == "multi" and case["int8"]:
        n, dim = case["tokens"], case["dim"]
        qk.quantize(s["x"], s["xq"], s["xs"], dim, n, stream=st)
        qk.check(lib.qk_gemv_multi_batched_i8(s["mats"], 3, s["xq"].data_ptr(), dim, s["xs"].data_ptr(), dim // 32,
                                              dim, n, s["ws"].data_ptr(), s["ws"].numel(), h), "multi_i8")
        return [s["q"], s["k"], s["v"]]
    if kind == "multi":
        qk.check(lib.qk_gemv_multi_batched_f32(s["mats"], 3, s["x"].data_ptr(), case["dim"], case["dim"],
                                               case["tokens"], s["ws"].data_ptr(), s["ws"].numel(), h), "multi")
        return [s["q"], s["k"], s["v"]]
    if kind == "attn":
        qk.check(lib.qk_attention_split_f32(s["q"].data_ptr(), s["key"].data_ptr(), s["value"].data_ptr(),
                                            s["out"].data_ptr(), 0, s["rows"], s["desc"].data_ptr(), s["n"], s["top"],
                                            case["heads"], case["kv_heads"], case["head_dim"], 0, s["ws"].data_ptr(),
                                            s["ws"].numel(), h), "attention")
        return [s["out"]]
    if kind == "norm":
        qk.rmsnorm_quantize(s["x"], s["w"], s["out"], s["xq"], s["xs"], case["dim"], case["tokens"], stream=st)
        return [s["out"], s["xq"], s["xs"]]
    if kind == "decode":
        s["runner"].forward(s["token"], case["pos"], True)
        return [s["logits"]]
    s["runner"].forward(s["tokens"], s["positions"], s["zeros"], seq=s["zeros"], logit_rows=[case["tokens"] - 1])
    return [s["logits"]]


# ------------------------------------------------------- work, tolerance --

def _bytes(qtype, cols, rows):
    return rows * (cols // 256) * (144 if qtype == Q4 else 210)


def work(case):
    kind = case["kind"]
    if kind in ("qkv", "multi"):
        n, dim, kv = case.get("tokens", 1), case["dim"], case["kv_dim"]
        return dict(bytes=_bytes(Q4, dim, dim + kv) + _bytes(case["v_type"], dim, kv) + 4 * n * (2 * dim + 2 * kv),
                    flops=2 * n * dim * (dim + 2 * kv))
    if kind == "head":
        return dict(bytes=_bytes(case["type"], case["cols"], case["rows"]) + 4 * (case["cols"] + case["rows"]),
                    flops=2 * case["cols"] * case["rows"])
    if kind in ("ffn", "ffn_i8"):
        dim, hidden, n, L = case["dim"], case["hidden"], case["tokens"], case["layers"]
        w = 2 * _bytes(Q4, dim, hidden) + _bytes(case["down_type"], hidden, dim)
        return dict(bytes=L * (w + 4 * n * dim) + 4 * n * dim + (n * (dim + dim // 8) if kind == "ffn_i8" else 0),
                    flops=L * 6 * n * dim * hidden)
    if kind == "attn":
        # Each cache row once, however many tokens of its sequence read it.
        hd, rows = case["head_dim"], sum(_contexts(case))
        pairs = sum(pos + 1 for pos, _ in _attn_tokens(case)[0])
        n = case["seqs"] * case["chunk"]
        return dict(bytes=8 * rows * case["kv_heads"] * hd + 8 * n * case["heads"] * hd,
                    flops=4 * pairs * case["heads"] * hd)
    if kind == "norm":
        n, dim = case["tokens"], case["dim"]
        return dict(bytes=n * (4 * dim + 4 * dim + dim + dim // 8) + 4 * dim, flops=6 * n * dim)
    cfg = _config(case)
    n, pos = case.get("tokens", 1), case["pos"]
    kv = cfg["dim"] // cfg["heads"] * cfg["kv_heads"]
    w = sum(_bytes(t, c, r) for _, t, c, r in _shapes(cfg))
    m = sum(c * r for _, t, c, r in _shapes(cfg))
    pairs = sum(pos + i + 1 for i in range(n))
    return dict(bytes=cfg["layers"] * (w + 8 * kv * (pos + n)) + _bytes(Q6, cfg["dim"], cfg["vocab"] + n) +
                4 * cfg["vocab"],
                flops=cfg["layers"] * (2 * n * m + 4 * pairs * cfg["dim"]) + 2 * cfg["dim"] * cfg["vocab"])


def tolerance(case):
    kind = case["kind"]
    if kind in ("qkv", "multi", "ffn"):
        # 22-bit activations, exact integer weights, float32 sums.
        return dict(rel=4e-6)
    if kind == "head":
        # The same; the picked row is a whole value of its own.
        return dict(rel=4e-6)
    if kind == "attn":
        return dict(rel=1e-6)
    if kind == "norm":
        # A value within rounding of a midpoint may take either code.
        return dict(rel=3e-7, differ=2e-4)
    if kind == "ffn_i8":
        # The hidden codes are rounded in between: one that lies within
        # rounding of a midpoint moves its outputs by half a step.
        return dict(rel=8e-4)
    if case["int8"]:
        # As above, through every layer: the flips of one layer move the
        # inputs of the next ones, and so flip more.
        return dict(rel=3e-2, max=3e-1)
    return dict(rel=2e-4)


# ------------------------------------------------------------------ exact --

def _decode(qtype, data, cols, rows):
    """The float64 matrix [rows][cols] of GGUF block bytes."""
    nb = cols // 256
    if qtype == Q4:
        b = data.view(rows, nb, 144)
        d = b[..., 0:2].contiguous().view(torch.float16).double()
        dmin = b[..., 2:4].contiguous().view(torch.float16).double()
        s = b[..., 4:16].to(torch.int32)
        sc = torch.cat([s[..., 0:4] & 63, (s[..., 8:12] & 15) | ((s[..., 0:4] >> 6) << 4)], -1).double()
        mn = torch.cat([s[..., 4:8] & 63, (s[..., 8:12] >> 4) | ((s[..., 4:8] >> 6) << 4)], -1).double()
        q = b[..., 16:].reshape(rows, nb, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 3).reshape(rows, nb, 8, 32).double()
        return (q * (d * sc).unsqueeze(-1) - (dmin * mn).unsqueeze(-1)).reshape(rows, cols)
    b = data.view(rows, nb, 210)
    ql = b[..., :128].reshape(rows, nb, 2, 1, 64)
    low = torch.cat([ql & 15, ql >> 4], 3).reshape(rows, nb, 2, 4, 32)
    shift = torch.tensor([0, 2, 4, 6], dtype=torch.uint8, device=data.device).view(4, 1)
    high = (b[..., 128:192].reshape(rows, nb, 2, 1, 32) >> shift) & 3
    code = (low | (high << 4)).double() - 32
    scale = b[..., 208:210].contiguous().view(torch.float16).double() * \
        b[..., 192:208].contiguous().view(torch.int8).double()
    return (code.reshape(rows, nb, 16, 16) * scale.unsqueeze(-1)).reshape(rows, cols)


def _matmul(qtype, data, cols, rows, x):
    """x [n][cols] (float64) times the matrix, transposed: [n][rows]."""
    qtype = Q4 if qtype == Q4 else Q6
    step = max(1, (1 << 26) // cols)
    per = cols // 256 * (144 if qtype == Q4 else 210)
    out = []
    for r in range(0, rows, step):
        m = min(step, rows - r)
        out.append(x @ _decode(qtype, data[r * per:(r + m) * per], cols, m).T)
    return torch.cat(out, 1)


def _silu_mul(g, u):
    return g / (1 + torch.exp(-g)) * u


def _codes(x):
    """Per-32 codes and scales of the rows of x (float64)."""
    n, cols = x.shape
    g = x.view(n, cols // 32, 32)
    amax = g.abs().amax(-1)
    scale = torch.where(amax > 0, amax / 127, torch.ones_like(amax))
    return torch.round(g / scale.unsqueeze(-1)).clamp(-127, 127).reshape(n, cols), scale


def _coded(x):
    q, scale = _codes(x)
    return (q.view(x.shape[0], -1, 32) * scale.unsqueeze(-1)).reshape(x.shape)


def _norm(x, w, eps=1e-5):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _attend(q, k, v, heads, kv_heads, first):
    """q [n][heads*hd] at positions first.. over k, v [rows][kv_heads*hd]."""
    n, rows = q.shape[0], k.shape[0]
    hd = q.shape[1] // heads
    mask = torch.arange(rows, device=q.device)[None, :] > first + torch.arange(n, device=q.device)[:, None]
    out = torch.empty_like(q)
    for h in range(heads):
        kv = h // (heads // kv_heads)
        s = q[:, h * hd:(h + 1) * hd] @ k[:, kv * hd:(kv + 1) * hd].T / math.sqrt(hd)
        p = torch.softmax(s.masked_fill(mask, -math.inf), -1)
        out[:, h * hd:(h + 1) * hd] = p @ v[:, kv * hd:(kv + 1) * hd]
    return out


def _rotate(x, hd, first, theta):
    """Adjacent pairs rotated; the angle is a float32 value, as in the tables."""
    n = x.shape[0]
    freq = np.power(np.float32(theta), -2 * np.arange(hd // 2, dtype=np.float32) / np.float32(hd)).astype(np.float32)
    angle = (np.arange(first, first + n, dtype=np.float32)[:, None] * freq).astype(np.float32)
    a = torch.from_numpy(angle).to(x.device).double()[:, None]
    y = x.view(n, -1, hd // 2, 2)
    c, s = torch.cos(a), torch.sin(a)
    return torch.stack([y[..., 0] * c - y[..., 1] * s, y[..., 0] * s + y[..., 1] * c], -1).reshape(x.shape)


def _exact_model(case, seed):
    cfg = _config(case)
    n, pos = case.get("tokens", 1), case["pos"]
    hd = cfg["dim"] // cfg["heads"]
    keys, values = _cache_rows(cfg, pos, seed, 5).double(), _cache_rows(cfg, pos, seed, 6).double()
    parts, w, layer = _model_parts(cfg, seed), {}, -1
    x = None
    for l, name, qtype, cols, rows, data in parts:
        if l < 0:
            if name == "token_embd":
                table = data
                per = cols // 256 * 210
                ids = torch.tensor(_prompt(cfg, n, seed), device=DEV)
                x = _decode(Q6, table.view(rows, per)[ids].reshape(-1), cols, n)
            else:
                out_norm = data.double()
            continue
        w[name] = (qtype, data, cols, rows) if qtype else data.double()
        if name != "ffn_norm":
            continue
        mm = lambda key, t: _matmul(w[key][0], w[key][1], w[key][2], w[key][3], t)
        h = _norm(x, w["attn_norm"])
        q, k, v = mm("q", h), mm("k", h), mm("v", h)
        q, k = _rotate(q, hd, pos, cfg["rope_theta"]), _rotate(k, hd, pos, cfg["rope_theta"])
        a = _attend(q, torch.cat([keys[l], k]), torch.cat([values[l], v]), cfg["heads"], cfg["kv_heads"], pos)
        x = x + mm("o", a)
        h = _norm(x, w["ffn_norm"])
        x = x + mm("down", _silu_mul(mm("gate", h), mm("up", h)))
        w = {}
    y = _matmul(Q6, table, cfg["dim"], cfg["vocab"], _norm(x[-1:], out_norm))
    return [y[0] if case["kind"] == "decode" else y]


def exact(case, seed):
    kind = case["kind"]
    if kind in ("qkv", "multi"):
        dim, kv = case["dim"], case["kv_dim"]
        x = _activations(case.get("tokens", 1), dim, seed, 1).double()
        if case.get("int8"):
            x = _coded(x)
        out = [_matmul(t, _weights(t, dim, r, seed, i), dim, r, x)
               for t, r, i in ((Q4, dim, 2), (Q4, kv, 3), (case["v_type"], kv, 4))]
        return [t[0] for t in out] if kind == "qkv" else out
    if kind == "head":
        x = _activations(1, case["cols"], seed, 1).double()
        y = _matmul(case["type"], _weights(case["type"], case["cols"], case["rows"], seed, 2), case["cols"],
                    case["rows"], x)[0]
        return [y, None]
    if kind == "ffn_i8":
        # The block's outputs depend on which hidden codes round up, so
        # their distance from 64 bits says how many lay near a midpoint, not
        # how exact the sums are: "multi" covers those.
        q, scale = _codes(_activations(case["tokens"], case["dim"], seed, 1).double())
        return [q.to(torch.int8), scale] + [None] * case["layers"]
    if kind == "ffn":
        dim, hidden, t = case["dim"], case["hidden"], case["down_type"]
        x = _activations(case["tokens"], dim, seed, 1).double()
        out = []
        for l in range(case["layers"]):
            g = _matmul(Q4, _weights(Q4, dim, hidden, seed, 10 + 3 * l), dim, hidden, x)
            u = _matmul(Q4, _weights(Q4, dim, hidden, seed, 11 + 3 * l), dim, hidden, x)
            out.append(_matmul(t, _weights(t, hidden, dim, seed, 12 + 3 * l), hidden, dim, _silu_mul(g, u)))
        return out
    if kind == "attn":
        heads, kvh, hd, chunk = case["heads"], case["kv_heads"], case["head_dim"], case["chunk"]
        tokens, rows = _attn_tokens(case)
        g = _gen(seed, 1)
        q = torch.randn((len(tokens), heads * hd), device=DEV, generator=g).double()
        key = torch.randn((rows, kvh * hd), device=DEV, generator=g).double()
        value = torch.randn((rows, kvh * hd), device=DEV, generator=g).double()
        out, row = [], 0
        for i, ctx in enumerate(_contexts(case)):
            out.append(_attend(q[i * chunk:(i + 1) * chunk], key[row:row + ctx], value[row:row + ctx], heads, kvh,
                               ctx - chunk))
            row += ctx
        return [torch.cat(out)]
    if kind == "norm":
        x = _activations(case["tokens"], case["dim"], seed, 1).double()
        y = _norm(x, _rand((case["dim"],), _gen(seed, 2), 0.6, 1.4).double())
        q, scale = _codes(y)
        return [y, q.to(torch.int8), scale]
    return [None] if case["int8"] else _exact_model(case, seed)   # codes in every layer: as for "ffn_i8"
