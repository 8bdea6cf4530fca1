"""INT8 products of more (row tile, token tile) units than the chip holds at
once (csrc/qk_tile_i8.hip): ragged token and row tiles, split rows, the gate /
up pair, accumulation, strided inputs and outputs, and a workspace too small
for the planned splits.

Integer blocks (d = dmin = 1) with unit scales make every partial sum an exact
integer below 2^24, so the outputs equal an int64 product bit for bit; random
blocks are compared with the fp64 combine.  Its bar: an output adds K / 32
products of fp32 operands, each rounded a few times, so the relative error of
the whole is below about sqrt(K / 32) * 2^-24 * a small factor: 1e-5 as for the
integer matrix cores."""
import numpy as np
import pytest

from conftest import rel_l2, to_dev
from test_gpu_int8_matrix_core import Q4_K, Q6_K, _integer_blocks
from test_gpu_tile_gemm import sizes_of

pytestmark = pytest.mark.gpu


def _dense(t, qk, qtype, w, cols, rows):
    out = t.empty((rows, cols), device="cuda")
    wd = to_dev(t, w)
    qk.check(qk.lib().qk_dequant_rows(qtype, wd.data_ptr(), out.data_ptr(), cols, 0, rows, None), "dequant")
    t.cuda.synchronize()
    return out.cpu().double()


@pytest.mark.parametrize("qtype", [Q4_K, Q6_K])
@pytest.mark.parametrize("cols,rows,ntok", [(5632, 2050, 300), (8192, 1055, 545), (4096, 4096, 161),
                                            (20480, 2050, 130)])
def test_exact_ragged(qk, torch_gpu, synth, qtype, cols, rows, ntok):
    t = torch_gpu
    w = _integer_blocks(qtype, synth.quant_matrix(qtype, cols, rows, 5, 1), cols, rows)
    dense = _dense(t, qk, qtype, w, cols, rows)
    g = t.Generator().manual_seed(3)
    ldxq, ldsc, ldy = cols + 32, cols // 32 + 3, rows + 5
    # Small codes keep whole sums below 2^24 (scale * code <= 4096).
    xq = t.randint(-1, 2, (ntok, ldxq), generator=g, dtype=t.int8)
    xq *= (t.rand(ntok, ldxq, generator=g) < 0.1).to(t.int8)
    want = xq[:, :cols].double() @ dense.T
    assert want.abs().max() < 2 ** 24
    L = qk.lib()
    n = L.qk_gemv_batched_i8_workspace_bytes(cols, rows, ntok)
    ws = t.empty(n, dtype=t.uint8, device="cuda")
    wd, xd, xs = to_dev(t, w), xq.cuda(), t.ones(ntok, ldsc, device="cuda")
    y = t.full((ntok, ldy), 7.0, device="cuda")
    qk.check(L.qk_gemv_batched_i8(qtype, wd.data_ptr(), xd.data_ptr(), ldxq, xs.data_ptr(), ldsc, y.data_ptr(), ldy,
                                  cols, rows, ntok, ws.data_ptr(), n, None), "batched INT8")
    t.cuda.synchronize()
    got = y.cpu().double()
    assert (got[:, :rows] == want).all()
    assert (got[:, rows:] == 7.0).all()


def _centred_blocks(synth, cols, rows, seed):
    """Q4_K blocks as a quantizer leaves them: min = scale, dmin = 7.5 d, so
    that a sub-block's mins centre its codes on zero."""
    w = synth.quant_matrix(Q4_K, cols, rows, seed, 1).reshape(-1, 144).copy()
    sc = synth.uniform_i32(w.shape[0] * 8, seed, 2, 16, 63).astype(np.uint8).reshape(-1, 8)
    a, b = sc[:, :4], sc[:, 4:]
    w[:, 4:16] = np.concatenate([a | (b >> 4) << 6, a | (b >> 4) << 6, b & 15 | (b & 15) << 4], 1)
    d = w[:, :2].copy().view(np.float16).astype(np.float32)
    d = np.float16(1e-4) * (1 + np.abs(d) / (1 + np.abs(d)))
    w[:, :2] = d.astype(np.float16).view(np.uint8)
    w[:, 2:4] = (7.5 * d.astype(np.float16)).astype(np.float16).view(np.uint8)
    return w.reshape(-1)


@pytest.mark.parametrize("qtype", [Q4_K, Q6_K])
@pytest.mark.parametrize("cols,rows,ntok", [(8192, 3072, 256), (8192, 2050, 517), (14336, 4096, 256), (8192, 8192, 1000)])
def test_rounding(qk, torch_gpu, synth, qtype, cols, rows, ntok):
    """The fp32 sums' own error.  A rounding is 0.42 * 2^-24 of its result
    (RMS).  The eight dots of a block are summed one after the other: 4.5
    roundings of the block's size (RMS of the running sums).  A Q4_K block of
    centred weights has dots of 1.9 times its own size and mins of 1.6 times,
    the latter rounded once more before they are summed: 1.9^2 * 4.5 + 1.6^2 *
    5.5 = 30, and two where they meet.  The nb blocks' running sum: nb / 2."""
    t = torch_gpu
    nb = cols // 256
    w = _centred_blocks(synth, cols, rows, 13) if qtype == Q4_K else synth.quant_matrix(Q6_K, cols, rows, 13, 1)
    dense = _dense(t, qk, qtype, w, cols, rows)
    g = t.Generator().manual_seed(17)
    xq = t.randn(ntok, cols, generator=g).mul(40).round().clamp(-127, 127).to(t.int8)
    xs = t.rand(ntok, cols // 32, generator=g) * 1e-2 + 1e-2
    want = (xq.double() * xs.double().repeat_interleave(32, 1)) @ dense.T
    L = qk.lib()
    n = L.qk_gemv_batched_i8_workspace_bytes(cols, rows, ntok)
    ws = t.empty(n, dtype=t.uint8, device="cuda")
    wd, xd, sd = to_dev(t, w), xq.cuda(), xs.cuda()
    y = t.empty(ntok, rows, device="cuda")
    qk.check(L.qk_gemv_batched_i8(qtype, wd.data_ptr(), xd.data_ptr(), cols, sd.data_ptr(), cols // 32, y.data_ptr(),
                                  rows, cols, rows, ntok, ws.data_ptr(), n, None), "batched INT8")
    t.cuda.synchronize()
    roundings = (32 if qtype == Q4_K else 4.5) + nb / 2
    assert rel_l2(y.cpu().numpy(), want.numpy()) < 0.42 * 2 ** -24 * roundings ** 0.5


@pytest.mark.parametrize("down", [Q4_K, Q6_K])
@pytest.mark.parametrize("dim,hidden,ntok", [(2048, 5632, 97), (3072, 8192, 200), (1024, 2816, 517), (5120, 5632, 200)])
def test_ffn(qk, torch_gpu, synth, down, dim, hidden, ntok):
    t = torch_gpu
    ws = [synth.quant_matrix(Q4_K, dim, hidden, 9, i) for i in (1, 2)]
    ws.append(synth.quant_matrix(down, hidden, dim, 9, 3))
    g, u = (_dense(t, qk, Q4_K, ws[i], dim, hidden) for i in (0, 1))
    d = _dense(t, qk, down, ws[2], hidden, dim)
    gen = t.Generator().manual_seed(11)
    xq = t.randint(-128, 128, (ntok, dim), generator=gen, dtype=t.int8)
    xs = t.rand(ntok, dim // 32, generator=gen) * 2e-4 + 1e-5
    x = xq.double() * xs.double().repeat_interleave(32, 1)
    a = x @ g.T
    h = (a / (1 + t.exp(-a)) * (x @ u.T)).view(ntok, hidden // 32, 32)
    scale = (h.abs().amax(2, keepdim=True) / 127).float().double()
    scale = t.where(scale > 0, scale, t.ones_like(scale))
    hq = (t.round(h / scale).clamp(-127, 127) * scale).view(ntok, hidden)
    y0 = t.randn(ntok, dim, generator=gen)
    want = hq @ d.T
    L = qk.lib()
    n = L.qk_ffn_batched_i8_workspace_bytes(dim, hidden, ntok)
    dev = [to_dev(t, w) for w in ws]
    xd, sd, work = xq.cuda(), xs.cuda(), t.empty(n, dtype=t.uint8, device="cuda")
    for accumulate in (0, 1):
        y = y0.cuda()
        qk.check(L.qk_ffn_batched_i8(Q4_K, dev[0].data_ptr(), Q4_K, dev[1].data_ptr(), down, dev[2].data_ptr(),
                                     xd.data_ptr(), dim, sd.data_ptr(), dim // 32, y.data_ptr(), dim, dim, hidden, ntok,
                                     accumulate, work.data_ptr(), n, None), "INT8 FFN")
        t.cuda.synchronize()
        ref = want + y0.double() if accumulate else want
        # h in fp32 is off by some 2^-20 of itself, so a share of about
        # 127 * 2^-20 of the codes rounds the other way, by 1 / 127 of the
        # group's peak (some three times its RMS): sqrt(127 * 2^-20) * 3 / 127
        # = 2.6e-4 of the whole.
        assert rel_l2(y.cpu().numpy(), ref.numpy()) < 5e-4


@pytest.mark.parametrize("qtype,cols,rows,ntok", [(Q4_K, 8192, 3072, 256), (Q6_K, 8192, 2048, 300), (Q6_K, 5632, 2048, 400)])
def test_bits_do_not_depend_on_a_larger_workspace(qk, torch_gpu, synth, qtype, cols, rows, ntok):
    """The queried size and a larger one give the same bits; the least size that
    is accepted holds fewer splits."""
    t = torch_gpu
    g = t.Generator().manual_seed(19)
    w = to_dev(t, synth.quant_matrix(qtype, cols, rows, 15, 1))
    xq = t.randint(-127, 128, (ntok, cols), generator=g, dtype=t.int8).cuda()
    xs = (t.rand(ntok, cols // 32, generator=g) * 1e-2).cuda()
    L = qk.lib()
    query = L.qk_gemv_batched_i8_workspace_bytes(cols, rows, ntok)
    ws = t.empty(query + (64 << 20), dtype=t.uint8, device="cuda")

    def call(n):
        y = t.empty(ntok, rows, device="cuda")
        qk.check(L.qk_gemv_batched_i8(qtype, w.data_ptr(), xq.data_ptr(), cols, xs.data_ptr(), cols // 32, y.data_ptr(),
                                      rows, cols, rows, ntok, ws.data_ptr(), n, None), "batched INT8")
        t.cuda.synchronize()
        return y.cpu().numpy()

    queried, more, least = (call(n) for n in sizes_of(qk, call, query))
    assert np.array_equal(queried, more)
    assert rel_l2(least, queried) < 1e-6


def test_ffn_bits_do_not_depend_on_a_larger_workspace(qk, torch_gpu, synth):
    t = torch_gpu
    dim, hidden, ntok = 2048, 8192, 256
    g = t.Generator().manual_seed(23)
    w = [to_dev(t, synth.quant_matrix(ty, c, r, 16, i)) for i, (ty, c, r) in
         enumerate([(Q4_K, dim, hidden), (Q4_K, dim, hidden), (Q6_K, hidden, dim)])]
    xq = t.randint(-127, 128, (ntok, dim), generator=g, dtype=t.int8).cuda()
    xs = (t.rand(ntok, dim // 32, generator=g) * 2e-4).cuda()
    L = qk.lib()
    query = L.qk_ffn_batched_i8_workspace_bytes(dim, hidden, ntok)
    ws = t.empty(query + (64 << 20), dtype=t.uint8, device="cuda")

    def call(n):
        y = t.empty(ntok, dim, device="cuda")
        qk.check(L.qk_ffn_batched_i8(Q4_K, w[0].data_ptr(), Q4_K, w[1].data_ptr(), Q6_K, w[2].data_ptr(), xq.data_ptr(),
                                     dim, xs.data_ptr(), dim // 32, y.data_ptr(), dim, dim, hidden, ntok, 0,
                                     ws.data_ptr(), n, None), "INT8 FFN")
        t.cuda.synchronize()
        return y.cpu().numpy()

    queried, more, least = (call(n) for n in sizes_of(qk, call, query))
    assert np.array_equal(queried, more)
    assert rel_l2(least, queried) < 1e-6
