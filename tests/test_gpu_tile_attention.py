"""Attention of prefill chunks over shared rows (csrc/qk_tile_attention.hip)
against float64: head layouts of every wave count, chunk lengths around the
16-token tile and context lengths around the 32-row tile, chunks that begin or
end inside a tile, tokens left to the per-token kernel, and values that are
not finite in rows an earlier token must not see."""
import ctypes

import numpy as np
import pytest

from conftest import rel_l2, to_dev

pytestmark = pytest.mark.gpu
# fp32 products and sums over at most 700 rows and 128 dimensions: a score is
# within about sqrt(128) * 2^-24 of its terms, a probability within that, the
# output's sum within sqrt(700) * 2^-24: below 2e-6.
TOL = 2e-6


def reference(q, key, value, tokens, heads, kvh, hd):
    """Float64 softmax attention of every (pos, first row) token."""
    out = np.empty((len(tokens), heads * hd))
    group = heads // kvh
    k64, v64 = key.astype(np.float64), value.astype(np.float64)
    for t, (pos, row) in enumerate(tokens):
        for h in range(heads):
            c = slice(h // group * hd, h // group * hd + hd)
            s = k64[row:row + pos + 1, c] @ q[t, h * hd:(h + 1) * hd].astype(np.float64) / np.sqrt(hd)
            p = np.exp(s - s.max())
            out[t, h * hd:(h + 1) * hd] = p @ v64[row:row + pos + 1, c] / p.sum()
    return out


def tiles(qk, tokens, cache_rows, heads, kvh, hd):
    """Whether the call tries tiles (its descriptors are on the device)."""
    rule = qk.lib().qk_rule_tile_attention
    rule.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_int64] + [ctypes.c_int] * 3
    return bool(rule(len(tokens), max(p for p, _ in tokens), cache_rows, heads, kvh, hd))


def run(qk, t, q, key, value, tokens, heads, kvh, hd, split_rows=0):
    n, rows = len(tokens), key.shape[0]
    top = max(p for p, _ in tokens)
    desc = to_dev(t, np.array([[p | (i << 32), r] for i, (p, r) in enumerate(tokens)], dtype=np.int64))
    nb = qk.lib().qk_attention_split_workspace_bytes(n, heads, kvh, hd, top, split_rows)
    ws = t.empty(max(nb, 256), dtype=t.uint8, device="cuda")
    out = t.full((n, heads * hd), float("nan"), device="cuda")
    qd, kd, vd = to_dev(t, q), to_dev(t, key), to_dev(t, value)
    qk.check(qk.lib().qk_attention_split_f32(qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), out.data_ptr(), 0, rows,
                                             desc.data_ptr(), n, top, heads, kvh, hd, split_rows, ws.data_ptr(),
                                             ws.numel(), None), "attention")
    t.cuda.synchronize()
    return out.cpu().numpy()


def batch(rng, seqs, heads, kvh, hd):
    """seqs: (rows after the chunk, chunk tokens) of each sequence."""
    tokens, row = [], 0
    for ctx, chunk in seqs:
        tokens += [(ctx - chunk + i, row) for i in range(chunk)]
        row += ctx
    draw = lambda n, w: rng.standard_normal((n, w)).astype(np.float32)
    return draw(len(tokens), heads * hd), draw(row, kvh * hd), draw(row, kvh * hd), tokens


LAYOUTS = [(8, 8, 64), (16, 8, 64), (24, 8, 128), (32, 8, 64), (48, 8, 128), (64, 8, 64)]


def check_chunks(qk, t, rng, q, key, value, tokens, heads, kvh, hd):
    assert tiles(qk, tokens, len(key), heads, kvh, hd)
    got = run(qk, t, q, key, value, tokens, heads, kvh, hd)
    pick = sorted(set(rng.integers(0, len(tokens), 24).tolist() + [0, 1, 15, 16, len(tokens) - 1]))
    want = reference(q[pick], key, value, [tokens[i] for i in pick], heads, kvh, hd)
    assert rel_l2(got[pick], want) < TOL
    # Every token, against the per-token form (a split size given asks for it).
    assert rel_l2(got, run(qk, t, q, key, value, tokens, heads, kvh, hd, split_rows=256)) < TOL


@pytest.mark.parametrize("heads,kvh,hd", LAYOUTS)
@pytest.mark.parametrize("seqs", [[(512, 512)], [(540, 507)]])
def test_one_chunk(qk, torch_gpu, heads, kvh, hd, seqs):
    rng = np.random.default_rng(heads * 1000)
    check_chunks(qk, torch_gpu, rng, *batch(rng, seqs, heads, kvh, hd), heads, kvh, hd)


@pytest.mark.parametrize("heads,kvh,hd", LAYOUTS[:4])
@pytest.mark.parametrize("seqs", [[(640, 300), (333, 205)], [(640, 480), (33, 17)], [(200, 150), (300, 181), (260, 170)]])
def test_chunks_of_several_sequences(qk, torch_gpu, heads, kvh, hd, seqs):
    """Tiles of two sequences, of a sequence's end and a short one, and of one
    token of one and fifteen of another."""
    rng = np.random.default_rng(heads * 1000 + len(seqs))
    check_chunks(qk, torch_gpu, rng, *batch(rng, seqs, heads, kvh, hd), heads, kvh, hd)


@pytest.mark.parametrize("heads,kvh,hd", LAYOUTS)
def test_tile_of_two_runs(qk, torch_gpu, heads, kvh, hd):
    """Two runs over the rows of one sequence that meet inside a tile, in every
    head layout: tokens 0..299 and, in the same call, 251..462."""
    rng = np.random.default_rng(heads * 1000 + 5)
    q, key, value, _ = batch(rng, [(463, 512 - 49)], heads, kvh, hd)
    q = rng.standard_normal((512, heads * hd)).astype(np.float32)
    tokens = [(i, 0) for i in range(300)] + [(i, 0) for i in range(251, 463)]
    check_chunks(qk, torch_gpu, rng, q, key, value, tokens, heads, kvh, hd)


def test_decodes_beside_a_chunk(qk, torch_gpu):
    """16-token tiles with more than two sequences go one token at a time."""
    heads, kvh, hd = 32, 8, 64
    rng = np.random.default_rng(7)
    q, key, value, tokens = batch(rng, [(500, 460)] + [(40 + i, 1) for i in range(20)], heads, kvh, hd)
    assert tiles(qk, tokens, len(key), heads, kvh, hd)
    got = run(qk, torch_gpu, q, key, value, tokens, heads, kvh, hd)
    pick = [0, 200, 459] + list(range(460, 480))
    want = reference(q[pick], key, value, [tokens[i] for i in pick], heads, kvh, hd)
    assert rel_l2(got[pick], want) < TOL


def step_mode(qk, tokens, cfg):
    """The decode driver's choice: 0 none, 1 tiles and the other tokens one by
    one, 2 every token in a tile."""
    desc = (qk.qk_batch_token * len(tokens))(*(qk.qk_batch_token(p, 0, r) for p, r in tokens))
    return qk.lib().qk_rule_tile_attention_step(desc, len(tokens), cfg["heads"], cfg["kv_heads"],
                                                cfg["dim"] // cfg["heads"])


@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("heads,kv_heads,hd,chunk,decodes", [
    (16, 8, 64, (0, 301), 0), (16, 8, 64, (37, 331), 20), (8, 4, 128, (200, 509), 0), (8, 4, 128, (200, 505), 19),
    (8, 8, 64, (0, 347), 19)])
def test_driver_chunk(qk, torch_gpu, workloads, synth, int8, heads, kv_heads, hd, chunk, decodes):
    """A chunk, alone and beside decodes (of long and short contexts, so that
    their rows are split and merged), in the batched driver's own cache layout
    with the o projection's records (FP32) or codes (INT8) from the attention:
    every token's logits against the same step with its tokens in reverse order.
    Those tokens form no runs, so they take the per-token form; the products do
    not depend on the order."""
    pre, n = chunk
    cfg = dict(dim=heads * hd, layers=2, heads=heads, kv_heads=kv_heads, hidden=512, vocab=300, context=1024, eps=1e-5,
               rope_theta=10000.0)
    W, ctx, kv = workloads.llama_weights(cfg, 31), cfg["context"], kv_heads * hd
    S = 1 + decodes
    entries = [(0, pre + i) for i in range(n)] + [(1 + i, 40 + 47 * i) for i in range(decodes)]   # (sequence, position)
    tokens = [(p, s * ctx) for s, p in entries]
    assert step_mode(qk, tokens, cfg) == (1 if decodes else 2)
    assert step_mode(qk, tokens[::-1], cfg) == 0
    caches = [synth.normal_f32(cfg["layers"] * S * ctx * kv, 32, i).reshape(cfg["layers"], S * ctx, kv) for i in (0, 1)]
    ids = [int(v) for v in synth.uniform_i32(len(entries), 32, 5, 0, cfg["vocab"] - 1)]

    def step(order):
        br = qk.BatchRunner(cfg, W, max_tokens=len(entries), cache_rows=S * ctx)
        br.set_int8(int8, int8)
        br.load_kv(*caches)
        pick = [entries[i] for i in order]
        br.forward([ids[i] for i in order], [p for _, p in pick], [s * ctx for s, _ in pick], seq=[s for s, _ in pick],
                   logit_rows=list(range(len(order))))
        lg = br.logits(len(order))
        br.close()
        out = np.empty_like(lg)
        out[order] = lg
        return out

    got, want = step(list(range(len(entries)))), step(list(range(len(entries)))[::-1])
    errs = np.array([rel_l2(a, b) for a, b in zip(got, want)])
    # FP32: the forms' roundings (2e-7 of an output each) through two layers,
    # magnified where a random score is large.  INT8: a code within them of a
    # midpoint moves by one of 127, in few tokens.
    assert np.isfinite(got).all() and np.median(errs) < 1e-6 and errs.max() < (5e-2 if int8 else 2e-3)


def test_later_rows_not_finite(qk, torch_gpu):
    """Infinite or NaN values in a later token's row reach that token only."""
    heads, kvh, hd = 24, 8, 128
    rng = np.random.default_rng(8)
    q, key, value, tokens = batch(rng, [(500, 500)], heads, kvh, hd)
    clean = run(qk, torch_gpu, q, key, value, tokens, heads, kvh, hd)
    value[300, 5], value[421, hd + 7] = np.inf, np.nan
    key[421, 3 * hd] = np.nan
    got = run(qk, torch_gpu, q, key, value, tokens, heads, kvh, hd)
    assert rel_l2(got[:300], clean[:300]) < TOL
    assert np.isfinite(got[:300]).all() and not np.isfinite(got[300:, 5]).any()
    per_token = run(qk, torch_gpu, q, key, value, tokens, heads, kvh, hd, split_rows=512)
    assert np.array_equal(np.isfinite(got), np.isfinite(per_token))
    assert rel_l2(got[np.isfinite(got)], per_token[np.isfinite(got)]) < TOL


def test_poisoned_sequence_time(qk, torch_gpu):
    """A non-finite early row makes every result of its sequence non-finite, at
    the cost of a clean one: every tile is taken once, whatever it holds."""
    t = torch_gpu
    heads, kvh, hd = 24, 8, 128
    rng = np.random.default_rng(9)
    q, key, value, tokens = batch(rng, [(1000, 500)], heads, kvh, hd)
    n, top = len(tokens), tokens[-1][0]
    desc = to_dev(t, np.array([[p | (i << 32), r] for i, (p, r) in enumerate(tokens)], dtype=np.int64))
    ws = t.empty(qk.lib().qk_attention_split_workspace_bytes(n, heads, kvh, hd, top, 0), dtype=t.uint8, device="cuda")
    out, qd, kd = t.empty((n, heads * hd), device="cuda"), to_dev(t, q), to_dev(t, key)

    def best(vd):
        times = []
        for _ in range(5):
            a, b = t.cuda.Event(enable_timing=True), t.cuda.Event(enable_timing=True)
            a.record()
            qk.check(qk.lib().qk_attention_split_f32(
                qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), out.data_ptr(), 0, len(key), desc.data_ptr(), n, top, heads,
                kvh, hd, 0, ws.data_ptr(), ws.numel(), t.cuda.current_stream().cuda_stream), "attention")
            b.record()
            t.cuda.synchronize()
            times.append(a.elapsed_time(b))
        return min(times)

    clean = best(to_dev(t, value))
    value[3] = np.nan
    assert best(to_dev(t, value)) < 3 * clean
    assert t.isnan(out).all()


def test_rows_at_a_run_end_not_finite(qk, torch_gpu):
    """Infinities in the rows of the chunk's own tokens, among them the first
    and last of a 16-token tile and of a 32-row tile: a token that sees one has
    it in its result (two of opposite sign: NaN), one that does not is untouched."""
    heads, kvh, hd = 32, 8, 64
    rng = np.random.default_rng(10)
    q, key, value, tokens = batch(rng, [(700, 500)], heads, kvh, hd)
    clean = run(qk, torch_gpu, q, key, value, tokens, heads, kvh, hd, split_rows=704)
    want = clean.copy()
    group = heads // kvh
    for tok, h, d, v in [(0, 0, 3, np.inf), (15, 1, 60, -np.inf), (16, 2, 0, np.nan), (56, 3, 63, np.inf),
                         (87, 4, 33, -np.inf), (88, 4, 33, np.inf), (499, 7, 17, np.inf)]:
        value[200 + tok, h * hd + d] = v
        for g in range(group):
            with np.errstate(invalid="ignore"):
                want[tok:, (h * group + g) * hd + d] += v
    got = run(qk, torch_gpu, q, key, value, tokens, heads, kvh, hd)
    finite = np.isfinite(want)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isfinite(got), finite)
    assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
    assert rel_l2(got[finite], want[finite]) < TOL


@pytest.mark.parametrize("heads,kvh,hd", [(24, 8, 128), (32, 8, 64)])
@pytest.mark.parametrize("ctx,chunk", [(512, 512), (1112, 512)])
def test_error_against_float64(qk, torch_gpu, heads, kvh, hd, ctx, chunk):
    """The tile form is as exact as the per-token form (a split size given asks
    for that): both errors are RMS over some 10^6 outputs of the same inputs,
    so 2 % covers the draw."""
    t = torch_gpu
    rng = np.random.default_rng(11)
    q, key, value, tokens = batch(rng, [(ctx, chunk)], heads, kvh, hd)
    want = np.empty_like(q, dtype=np.float64)
    mask = t.arange(ctx)[None, :] > t.tensor([p for p, _ in tokens])[:, None]
    for h in range(heads):
        c, kv = slice(h * hd, (h + 1) * hd), slice(h * kvh // heads * hd, (h * kvh // heads + 1) * hd)
        s = t.from_numpy(q[:, c]).double() @ t.from_numpy(key[:, kv]).double().T / hd ** 0.5
        want[:, c] = (t.softmax(s.masked_fill(mask, -float("inf")), 1) @ t.from_numpy(value[:, kv]).double()).numpy()
    tile = rel_l2(run(qk, t, q, key, value, tokens, heads, kvh, hd), want)
    per_token = rel_l2(run(qk, t, q, key, value, tokens, heads, kvh, hd, split_rows=ctx), want)
    assert tile < 1.02 * per_token


def test_cache_with_room(qk, torch_gpu):
    """A chunk takes the tile form whatever room its cache has beside it."""
    heads, kvh, hd = 24, 8, 128
    rng = np.random.default_rng(12)
    q, key, value, tokens = batch(rng, [(1112, 512)], heads, kvh, hd)
    want = run(qk, torch_gpu, q, key, value, tokens, heads, kvh, hd)
    assert tiles(qk, tokens, 1112, heads, kvh, hd)
    for room in (1113, 4096, 65536):
        assert tiles(qk, tokens, room, heads, kvh, hd)
        pad = np.zeros((room, kvh * hd), np.float32)
        pad[:1112] = key
        vpad = np.full((room, kvh * hd), np.nan, np.float32)
        vpad[:1112] = value
        assert np.array_equal(run(qk, torch_gpu, q, pad, vpad, tokens, heads, kvh, hd), want)


@pytest.mark.parametrize("heads,kvh,hd", [(32, 8, 64), (24, 8, 128), (16, 8, 64), (8, 8, 128)])
def test_decode_batches_stay_per_token(qk, torch_gpu, heads, kvh, hd):
    for lengths in ([700] * 32, list(range(64, 2048, 31)), [300] * 300, [4096] * 8):
        tokens = [(n - 1, sum(lengths[:i])) for i, n in enumerate(lengths)]
        for cache in (sum(lengths), 4 * sum(lengths)):
            assert not tiles(qk, tokens, cache, heads, kvh, hd)
