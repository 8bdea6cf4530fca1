"""The matrix-core GEMM of two token tiles and more (csrc/qk_tile_gemm.h) at
the edges of its tiles: token counts around multiples of 32 and 64, row counts
around multiples of 32 and 128, one block and odd block counts, every storage
type alone and mixed in one launch, with and without split sums."""
import re

import numpy as np
import pytest

from conftest import rel_l2, to_dev

pytestmark = pytest.mark.gpu
Q4_K, Q6_K, Q6_K_SPLIT = 12, 14, 114
# Activations carry 22 bits (2^-22 of a value), the fp32 sums of a block's 256
# products up to about sqrt(256) roundings of 2^-24: 1.2e-6 together.
TOL = 2e-6


def matrix(qk, t, workloads, synth, qtype, cols, rows, seed):
    """(tensor, host bytes as the oracle reads them, oracle type)."""
    if qtype == Q4_K:
        w, _ = workloads.gemv_case(Q4_K, cols, rows, seed=seed)
        return qk.Tensor((cols, rows), Q4_K, to_dev(t, w)), w, Q4_K
    w = synth.quant_matrix(Q6_K, cols, rows, seed, 1).reshape(-1, 210).copy()
    # Every third block's scales over the whole int8 range: the wave takes
    # the third chain where one of its rows has such a block.
    wide = synth.uniform_i32(w.shape[0] * 16, seed, 2, -128, 127).astype(np.int8).reshape(-1, 16)
    w[::3, 192:208] = wide[::3].view(np.uint8)
    w = w.reshape(-1)
    g = qk.Tensor((cols, rows), Q6_K, to_dev(t, w))
    if qtype == Q6_K:
        return g, w, Q6_K
    s = qk.split_q6k(g)
    t.cuda.synchronize()
    return s, w, Q6_K


def check(qk, t, oracle, tensors, x, cols, extra=0):
    ntok = x.shape[0]
    rows = [ten.rows() for ten, _, _ in tensors]
    nws = qk.batch_workspace_bytes(cols, sum(rows), ntok) + extra
    ws = t.empty(max(nws, 256), dtype=t.uint8, device="cuda")
    ys = [t.full((ntok, r), float("nan"), device="cuda") for r in rows]
    xd = to_dev(t, x)
    arr = qk._matrices([(ten, y) for (ten, _, _), y in zip(tensors, ys)])
    qk.check(qk.lib().qk_gemv_multi_batched_f32(arr, len(tensors), xd.data_ptr(), cols, cols, ntok, ws.data_ptr(), nws,
                                                None), "multi batched")
    t.cuda.synchronize()
    for (ten, w, qtype), y in zip(tensors, ys):
        want = oracle.gemv_f64(qtype, w, x, cols, ten.rows())
        # Over all tokens: one output of one row may cancel to far below its
        # terms (its error is bounded by their size, not its own); the norm
        # over the tokens does not.
        assert rel_l2(y.cpu().numpy(), want) < TOL, qtype


@pytest.mark.parametrize("qtype", [Q4_K, Q6_K, Q6_K_SPLIT])
@pytest.mark.parametrize("ntok,cols,rows", [(33, 256, 31), (64, 512, 129), (65, 768, 128), (97, 2048, 640),
                                            (128, 1280, 33), (129, 3072, 257)])
def test_edges(qk, torch_gpu, oracle, workloads, synth, qtype, ntok, cols, rows):
    x = synth.normal_f32(ntok * cols, 31, ntok).reshape(ntok, cols)
    check(qk, torch_gpu, oracle, [matrix(qk, torch_gpu, workloads, synth, qtype, cols, rows, 30 + ntok)], x, cols)


@pytest.mark.parametrize("ntok", [34, 96, 161])
def test_mixed_types(qk, torch_gpu, oracle, workloads, synth, ntok):
    cols = 1024
    x = synth.normal_f32(ntok * cols, 32, ntok).reshape(ntok, cols)
    tensors = [matrix(qk, torch_gpu, workloads, synth, ty, cols, rows, 40 + i)
               for i, (ty, rows) in enumerate([(Q4_K, 130), (Q6_K, 96), (Q6_K_SPLIT, 257), (Q4_K, 1)])]
    check(qk, torch_gpu, oracle, tensors, x, cols)


def test_large_workspace_splits(qk, torch_gpu, oracle, workloads, synth):
    """Room for more splits than the queried size holds."""
    ntok, cols, rows = 40, 4096, 200
    x = synth.normal_f32(ntok * cols, 33, ntok).reshape(ntok, cols)
    t = torch_gpu
    check(qk, t, oracle, [matrix(qk, t, workloads, synth, Q4_K, cols, rows, 50)], x, cols, extra=8 << 20)


@pytest.mark.parametrize("qtype", [Q4_K, Q6_K_SPLIT])
def test_error_of_long_rows(qk, torch_gpu, workloads, synth, qtype):
    """32-block rows of 517 tokens are as exact as the same tokens 32 at a time
    (the kernel of one token tile, whose sums are at most four blocks long):
    both errors are RMS over a million outputs, so 2 % covers the draw."""
    t = torch_gpu
    ntok, cols, rows = 517, 8192, 3072
    g = t.Generator(device="cuda").manual_seed(5)
    x = t.randn((ntok, cols), device="cuda", generator=g) * t.exp(0.5 * t.randn(cols, device="cuda", generator=g))
    if qtype == Q4_K:   # mins that centre the weights, as a quantizer leaves them
        w, _ = workloads.gemv_case(Q4_K, cols, rows, seed=55)
        w = w.reshape(-1, 144).copy()
        sc = synth.uniform_i32(w.shape[0] * 8, 56, 2, 16, 63).astype(np.uint8).reshape(-1, 8)
        a, b = sc[:, :4], sc[:, 4:]
        w[:, 4:16] = np.concatenate([a | (b >> 4) << 6, a | (b >> 4) << 6, b & 15 | (b & 15) << 4], 1)
        w[:, 0:2], w[:, 2:4] = np.array([1e-4], np.float16).view(np.uint8), np.array([7.5e-4], np.float16).view(np.uint8)
        ten = qk.Tensor((cols, rows), Q4_K, to_dev(t, w.reshape(-1)))
    else:
        ten, _, _ = matrix(qk, t, workloads, synth, qtype, cols, rows, 57)
    dense = t.empty((rows, cols), device="cuda")
    qk.dequant_rows(ten, dense, 0, rows)
    want = x.double() @ dense.double().T
    ws = t.empty(qk.batch_workspace_bytes(cols, rows, ntok), dtype=t.uint8, device="cuda")

    def error(step):
        y = t.empty((ntok, rows), device="cuda")
        for i in range(0, ntok, step):
            n = min(step, ntok - i)
            qk.check(qk.lib().qk_gemv_batched_f32(ten.type, ten.gpu, x[i:].data_ptr(), cols, y[i:].data_ptr(), rows, cols,
                                                  rows, n, ws.data_ptr(), ws.numel(), None), "batched")
        t.cuda.synchronize()
        return float((y.double() - want).norm() / want.norm())

    assert error(ntok) < 1.02 * error(32)


def sizes_of(qk, call, query):
    """The queried size, more, and the least size the call takes."""
    with pytest.raises(qk.QKError) as e:
        call(256)
    least = int(re.search(r"smaller than (\d+) bytes", str(e.value))[1])
    assert least <= query
    return query, query + (64 << 20), least


@pytest.mark.parametrize("ntok,cols,rows", [(40, 4096, 200), (97, 8192, 640), (256, 2048, 512)])
def test_bits_do_not_depend_on_a_larger_workspace(qk, torch_gpu, workloads, synth, ntok, cols, rows):
    t = torch_gpu
    ten, _, _ = matrix(qk, t, workloads, synth, Q4_K, cols, rows, 51)
    x = to_dev(t, synth.normal_f32(ntok * cols, 34, ntok))
    query = qk.batch_workspace_bytes(cols, rows, ntok)
    ws = t.empty(query + (64 << 20), dtype=t.uint8, device="cuda")

    def call(n):
        y = t.empty((ntok, rows), device="cuda")
        qk.check(qk.lib().qk_gemv_batched_f32(Q4_K, ten.gpu, x.data_ptr(), cols, y.data_ptr(), rows, cols, rows, ntok,
                                              ws.data_ptr(), n, None), "batched")
        t.cuda.synchronize()
        return y.cpu().numpy()

    queried, more, least = (call(n) for n in sizes_of(qk, call, query))
    assert np.array_equal(queried, more)
    assert rel_l2(least, queried) < TOL


@pytest.mark.parametrize("ntok,dim,hidden", [(64, 1024, 2816), (130, 3072, 8192)])
def test_ffn_bits_do_not_depend_on_a_larger_workspace(qk, torch_gpu, workloads, synth, ntok, dim, hidden):
    t = torch_gpu
    g, u, d = (matrix(qk, t, workloads, synth, Q4_K, c, r, 52 + i)[0]
               for i, (c, r) in enumerate([(dim, hidden), (dim, hidden), (hidden, dim)]))
    x = to_dev(t, synth.normal_f32(ntok * dim, 35, ntok) * np.float32(0.05))
    query = qk.lib().qk_ffn_batched_workspace_bytes(dim, hidden, ntok)
    ws = t.empty(query + (64 << 20), dtype=t.uint8, device="cuda")

    def call(n):
        y = t.empty((ntok, dim), device="cuda")
        qk.check(qk.lib().qk_ffn_batched_f32(Q4_K, g.gpu, Q4_K, u.gpu, Q4_K, d.gpu, x.data_ptr(), dim, y.data_ptr(), dim,
                                             dim, hidden, ntok, 0, ws.data_ptr(), n, None), "ffn")
        t.cuda.synchronize()
        return y.cpu().numpy()

    queried, more, least = (call(n) for n in sizes_of(qk, call, query))
    assert np.array_equal(queried, more)
    assert rel_l2(least, queried) < 4 * TOL
