"""Products of 2 to 7 tokens (csrc/qk_few.hip): row counts around the 16-row
tile and the two-tile step, one to thirty-two blocks a row (one or two a wave,
with and without a second block in the last wave), every storage type alone and
mixed, scales over the whole int8 range, the feed-forward block's pair, its down
product and residual, SiLU(x) * up and the RMSNorm staged by the decode driver,
values that are not finite.  few_pays decides which calls come here (enough
weight bytes for the token count); every test asks it."""
import ctypes

import numpy as np
import pytest

from conftest import rel_l2, to_dev
from test_gpu_tile_gemm import Q4_K, Q6_K, Q6_K_SPLIT, TOL, check, matrix

pytestmark = pytest.mark.gpu


def few(qk, mats, cols, ntok, pair=False):
    """Whether a call over mats ((type, rows) each) comes here."""
    arr = (qk.qk_matrix * len(mats))(*(qk.qk_matrix(ty, rows, None, None) for ty, rows in mats))
    return bool(qk.lib().qk_rule_few_tokens(arr, len(mats), cols, ntok, int(pair)))


@pytest.mark.parametrize("qtype", [Q4_K, Q6_K, Q6_K_SPLIT])
@pytest.mark.parametrize("ntok,cols,rows", [(7, 256, 140001), (7, 768, 32015), (4, 2048, 65541), (6, 3072, 16400),
                                            (5, 4096, 12001), (7, 7424, 4093), (7, 7936, 3900), (7, 8192, 3899),
                                            (7, 8192, 3700), (4, 2048, 128256)])
def test_edges(qk, torch_gpu, oracle, workloads, synth, qtype, ntok, cols, rows):
    x = synth.normal_f32(ntok * cols, 61, ntok).reshape(ntok, cols)
    assert few(qk, [(qtype, rows)], cols, ntok)
    check(qk, torch_gpu, oracle, [matrix(qk, torch_gpu, workloads, synth, qtype, cols, rows, 60 + ntok)], x, cols)


@pytest.mark.parametrize("ntok,cols", [(7, 2048), (5, 2560), (4, 3072)])
def test_mixed_types(qk, torch_gpu, oracle, workloads, synth, ntok, cols):
    x = synth.normal_f32(ntok * cols, 62, ntok).reshape(ntok, cols)
    mats = [(Q4_K, 16500), (Q6_K, 96), (Q6_K_SPLIT, 257), (Q4_K, 20)]
    assert few(qk, mats, cols, ntok)
    tensors = [matrix(qk, torch_gpu, workloads, synth, ty, cols, rows, 70 + i) for i, (ty, rows) in enumerate(mats)]
    check(qk, torch_gpu, oracle, tensors, x, cols)


@pytest.mark.parametrize("types", [(Q4_K, Q4_K, Q6_K), (Q4_K, Q6_K, Q4_K), (Q6_K_SPLIT, Q6_K_SPLIT, Q6_K_SPLIT)])
@pytest.mark.parametrize("ntok,dim,hidden", [(7, 2048, 8192), (5, 3072, 8192), (7, 1536, 8192), (7, 4096, 4096),
                                             (6, 3840, 4608)])
def test_ffn(qk, torch_gpu, oracle, workloads, synth, types, ntok, dim, hidden):
    """Gate and up of one type in one launch with SiLU * up; down here or by the
    GEMV kernels (small products)."""
    t = torch_gpu
    if types[0] == types[1]:
        assert few(qk, [(types[0], hidden), (types[1], hidden)], dim, ntok, True)
    if types[2] == Q6_K_SPLIT and (dim, hidden) in ((3072, 8192), (4096, 4096)):
        assert few(qk, [(types[2], dim)], hidden, ntok)
    x = synth.normal_f32(ntok * dim, 63, ntok).reshape(ntok, dim) * 0.05
    shapes = [(dim, hidden), (dim, hidden), (hidden, dim)]
    (g, wg, tg), (u, wu, tu), (d, wd, td) = [matrix(qk, t, workloads, synth, ty, c, r, 80 + i)
                                             for i, (ty, (c, r)) in enumerate(zip(types, shapes))]
    a = oracle.gemv_f64(tg, wg, x, dim, hidden)
    h = a / (1.0 + np.exp(-np.clip(a, -700, 700))) * oracle.gemv_f64(tu, wu, x, dim, hidden)
    # The oracle takes fp32 rows: a scale that keeps their rounding at 2^-24.
    want = x + oracle.gemv_f64(td, wd, h.astype(np.float32), hidden, dim)
    nb = qk.lib().qk_ffn_batched_workspace_bytes(dim, hidden, ntok)
    ws = t.empty(max(nb, 256), dtype=t.uint8, device="cuda")
    y = to_dev(t, x)
    qk.check(qk.lib().qk_ffn_batched_f32(g.type, g.gpu, u.type, u.gpu, d.type, d.gpu, y.data_ptr(), dim, y.data_ptr(), dim,
                                         dim, hidden, ntok, 1, ws.data_ptr(), nb, None), "ffn")
    t.cuda.synchronize()
    # Two products and SiLU: the errors of gate and up double in h.
    assert rel_l2(y.cpu().numpy(), want) < 4 * TOL


@pytest.mark.parametrize("qtype", [Q4_K, Q6_K, Q6_K_SPLIT])
@pytest.mark.parametrize("ntok,cols,rows", [(4, 2048, 65541), (7, 7936, 3900)])
@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
def test_not_finite(qk, torch_gpu, workloads, synth, qtype, ntok, cols, rows, value):
    """A non-finite activation poisons its own token's outputs only."""
    t = torch_gpu
    x = synth.normal_f32(ntok * cols, 64, 1).reshape(ntok, cols)
    x[2, 700] = value
    assert few(qk, [(qtype, rows)], cols, ntok)
    ten, _, _ = matrix(qk, t, workloads, synth, qtype, cols, rows, 90)
    y = t.empty((ntok, rows), device="cuda")
    qk.batch_matvec(ten, to_dev(t, x), y, cols, rows, ntok)
    t.cuda.synchronize()
    got = y.cpu().numpy()
    assert np.isnan(got[2]).all() and np.isfinite(np.delete(got, 2, 0)).all()


def test_pair_not_finite(qk, torch_gpu, workloads, synth):
    t = torch_gpu
    ntok, dim, hidden = 7, 4096, 4096
    x = synth.normal_f32(ntok * dim, 66, 1).reshape(ntok, dim) * 0.05
    x[3, 17], x[5, 4095] = np.nan, np.inf
    (g, _, _), (u, _, _), (d, _, _) = [matrix(qk, t, workloads, synth, ty, c, r, 92 + i) for i, (ty, c, r) in
                                       enumerate([(Q4_K, dim, hidden), (Q4_K, dim, hidden), (Q6_K_SPLIT, hidden, dim)])]
    assert few(qk, [(Q4_K, hidden)] * 2, dim, ntok, True) and few(qk, [(Q6_K_SPLIT, dim)], hidden, ntok)
    nb = qk.lib().qk_ffn_batched_workspace_bytes(dim, hidden, ntok)
    ws, y = t.empty(nb, dtype=t.uint8, device="cuda"), t.empty((ntok, dim), device="cuda")
    xd = to_dev(t, x)
    qk.check(qk.lib().qk_ffn_batched_f32(Q4_K, g.gpu, Q4_K, u.gpu, Q6_K_SPLIT, d.gpu, xd.data_ptr(), dim, y.data_ptr(), dim,
                                         dim, hidden, ntok, 0, ws.data_ptr(), nb, None), "ffn")
    t.cuda.synchronize()
    got = y.cpu().numpy()
    assert np.isnan(got[[3, 5]]).all() and np.isfinite(got[[0, 1, 2, 4, 6]]).all()


@pytest.mark.parametrize("up_type", [Q4_K, Q6_K])
@pytest.mark.parametrize("ntok,dim,hidden,heads,kv_heads", [(7, 4096, 4096, 32, 8), (5, 3072, 8192, 24, 8)])
def test_driver_step(qk, torch_gpu, oracle, workloads, synth, up_type, ntok, dim, hidden, heads, kv_heads):
    """Sequences decoding in the batched driver (which holds Q6_K in the split
    layout): gate / up with the RMSNorm staged here, of one type (the pair) or of
    two (down then stages SiLU * up), down accumulated into x, one block a wave and
    two; each sequence against its own oracle model."""
    cfg = dict(dim=dim, layers=2, heads=heads, kv_heads=kv_heads, hidden=hidden, vocab=300, context=32, eps=1e-5,
               rope_theta=10000.0)
    W = workloads.llama_weights(cfg, 27, mix=dict(workloads.MIX_1B, up=up_type))
    for i, L in enumerate(W["layers"]):
        L["attn_norm"] = 1.0 + 0.2 * synth.normal_f32(dim, 27, 500 + i)
        L["ffn_norm"] = 1.0 + 0.2 * synth.normal_f32(dim, 27, 510 + i)
    pair = [(Q4_K, hidden), (Q4_K if up_type == Q4_K else Q6_K_SPLIT, hidden)]
    assert few(qk, pair, dim, ntok, True) == (up_type == Q4_K) and few(qk, pair, dim, ntok)
    assert few(qk, [(Q6_K_SPLIT, dim)], hidden, ntok)
    br = qk.BatchRunner(cfg, W, max_tokens=ntok, cache_rows=ntok * cfg["context"])
    orcs = [oracle.Llama(cfg, W) for _ in range(ntok)]
    tokens = [int(v) for v in synth.uniform_i32(ntok, 27, 71, 0, cfg["vocab"] - 1)]
    for pos in range(2):
        br.forward(tokens, [pos] * ntok, [s * cfg["context"] for s in range(ntok)], True)
        lg = br.logits(ntok)
        want = [orcs[s].forward(tokens[s], pos, True) for s in range(ntok)]
        for s in range(ntok):
            assert rel_l2(lg[s], want[s][1]) < 1e-4
        tokens = [o for o, _ in want]
    br.close()


def test_infinite_scale_in_the_last_block(qk, torch_gpu, oracle, workloads, synth):
    """31 blocks a row, two a wave: the wave without a second block adds nothing.
    Where the row's last block has an infinite scale, its high and low products
    are infinite, of one sign in about half of the outputs; the last block again
    over zeros would make every one NaN."""
    t = torch_gpu
    ntok, cols, rows = 7, 31 * 256, 4096
    assert few(qk, [(Q4_K, rows)], cols, ntok)
    x = synth.normal_f32(ntok * cols, 65, ntok).reshape(ntok, cols)
    w, _ = workloads.gemv_case(Q4_K, cols, rows, seed=91)
    w = w.reshape(rows, 31, 144).copy()
    w[::5, 30, 0:2] = np.array([np.inf], np.float16).view(np.uint8)
    ten, y = qk.Tensor((cols, rows), Q4_K, to_dev(t, w.reshape(-1))), t.empty((ntok, rows), device="cuda")
    qk.batch_matvec(ten, to_dev(t, x), y, cols, rows, ntok)
    t.cuda.synchronize()
    y = y.cpu().numpy()
    assert not np.isfinite(y[:, ::5]).any() and 0.3 < np.isinf(y[:, ::5]).mean() < 0.7
    keep = np.arange(rows) % 5 != 0
    w[::5, 30, 0:2] = 0
    assert rel_l2(y[:, keep], oracle.gemv_f64(Q4_K, w.reshape(-1), x, cols, rows)[:, keep]) < TOL
