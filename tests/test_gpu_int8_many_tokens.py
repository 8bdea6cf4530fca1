"""INT8 products of more (row tile, token tile) units than the chip holds at
once (csrc/qk_tile_i8.hip): ragged token and row tiles, rows in one piece and
split, short and long sums, the gate / up pair, several matrices of one type,
accumulation, strided inputs and outputs, every storage type, workspaces at and
beyond the queried size and below it.  Every test of the kernel asks the dispatch
rule whether its call comes here.

Integer blocks (d = dmin = 1) with unit scales make every partial sum an exact
integer below 2^24, so the outputs equal an int64 product bit for bit; the
rounding of random blocks is held to a derived bar (test_rounding)."""
import numpy as np
import pytest

from conftest import rel_l2, to_dev
from test_gpu_int8_matrix_core import Q4_K, Q6_K, _integer_blocks
from test_gpu_tile_gemm import Q6_K_SPLIT, sizes_of

pytestmark = pytest.mark.gpu


def splits(qk, mats, cols, ntok, pair=False):
    """The row splits of a call over mats ((type, rows) each) that comes here, or
    0."""
    arr = (qk.qk_matrix * len(mats))(*(qk.qk_matrix(ty, rows, None, None) for ty, rows in mats))
    return qk.lib().qk_rule_tile_i8(arr, len(mats), cols, ntok, int(pair))


def _dense(t, qk, qtype, w, cols, rows):
    out = t.empty((rows, cols), device="cuda")
    wd = to_dev(t, w)
    qk.check(qk.lib().qk_dequant_rows(qtype, wd.data_ptr(), out.data_ptr(), cols, 0, rows, None), "dequant")
    t.cuda.synchronize()
    return out.cpu().double()


def _tensor(t, qk, qtype, w, cols, rows):
    """The device matrix of GGUF block bytes, in the split layout for Q6_K_SPLIT."""
    ten = qk.Tensor((cols, rows), Q4_K if qtype == Q4_K else Q6_K, to_dev(t, w))
    if qtype == Q6_K_SPLIT:
        ten = qk.split_q6k(ten)
        t.cuda.synchronize()
    return ten


def _sparse_codes(t, g, ntok, ldxq):
    """Small codes: whole sums stay below 2^24 (scale * code <= 4096)."""
    xq = t.randint(-1, 2, (ntok, ldxq), generator=g, dtype=t.int8)
    return xq * (t.rand(ntok, ldxq, generator=g) < 0.1).to(t.int8)


@pytest.mark.parametrize("qtype", [Q4_K, Q6_K, Q6_K_SPLIT])
@pytest.mark.parametrize("cols,rows,ntok,here", [
    (5632, 2050, 300, True), (8192, 1055, 545, True), (4096, 4096, 193, True), (8192, 8191, 1000, True),
    (20480, 2050, 130, None)])   # the last: Q4_K by the looping int32 kernel, in ten splits
def test_exact_ragged(qk, torch_gpu, synth, qtype, cols, rows, ntok, here):
    t = torch_gpu
    base = Q4_K if qtype == Q4_K else Q6_K
    assert bool(splits(qk, [(qtype, rows)], cols, ntok)) == (qtype != Q4_K if here is None else here)
    w = _integer_blocks(base, synth.quant_matrix(base, cols, rows, 5, 1), cols, rows)
    dense = _dense(t, qk, base, w, cols, rows)
    g = t.Generator().manual_seed(3)
    ldxq, ldsc, ldy = cols + 32, cols // 32 + 3, rows + 5
    xq = _sparse_codes(t, g, ntok, ldxq)
    want = xq[:, :cols].double() @ dense.T
    assert want.abs().max() < 2 ** 24
    L = qk.lib()
    n = L.qk_gemv_batched_i8_workspace_bytes(cols, rows, ntok)
    ws = t.empty(n, dtype=t.uint8, device="cuda")
    ten, xd, xs = _tensor(t, qk, qtype, w, cols, rows), xq.cuda(), t.ones(ntok, ldsc, device="cuda")
    y = t.full((ntok, ldy), 7.0, device="cuda")
    qk.check(L.qk_gemv_batched_i8(ten.type, ten.gpu, xd.data_ptr(), ldxq, xs.data_ptr(), ldsc, y.data_ptr(), ldy,
                                  cols, rows, ntok, ws.data_ptr(), n, None), "batched INT8")
    t.cuda.synchronize()
    got = y.cpu().double()
    assert (got[:, :rows] == want).all()
    assert (got[:, rows:] == 7.0).all()


@pytest.mark.parametrize("qtype", [Q4_K, Q6_K, Q6_K_SPLIT])
@pytest.mark.parametrize("cols,ntok", [(4096, 300), (8192, 517)])
def test_several_matrices(qk, torch_gpu, synth, qtype, cols, ntok):
    """One launch over matrices of one type with ragged rows: each one's row
    groups, split sums and outputs are its own."""
    t = torch_gpu
    base = Q4_K if qtype == Q4_K else Q6_K
    rows = [1027, 33, 700]
    assert splits(qk, [(qtype, r) for r in rows], cols, ntok) > 1
    ws_ = [_integer_blocks(base, synth.quant_matrix(base, cols, r, 6, i), cols, r) for i, r in enumerate(rows)]
    xq = _sparse_codes(t, t.Generator().manual_seed(4), ntok, cols)
    tens = [_tensor(t, qk, qtype, w, cols, r) for w, r in zip(ws_, rows)]
    ys = [t.empty((ntok, r), device="cuda") for r in rows]
    xd, xs = xq.cuda(), t.ones(ntok, cols // 32, device="cuda")
    L = qk.lib()
    n = L.qk_gemv_batched_i8_workspace_bytes(cols, sum(rows), ntok)
    ws = t.empty(n, dtype=t.uint8, device="cuda")
    qk.check(L.qk_gemv_multi_batched_i8(qk._matrices(list(zip(tens, ys))), 3, xd.data_ptr(), cols, xs.data_ptr(),
                                        cols // 32, cols, ntok, ws.data_ptr(), n, None), "multi INT8")
    t.cuda.synchronize()
    for w, r, y in zip(ws_, rows, ys):
        assert (y.cpu().double() == xq.double() @ _dense(t, qk, base, w, cols, r).T).all()


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
    assert splits(qk, [(qtype, rows)], cols, ntok)
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


@pytest.mark.parametrize("down", [Q4_K, Q6_K, Q6_K_SPLIT])
@pytest.mark.parametrize("gate", [Q4_K, Q6_K_SPLIT])
@pytest.mark.parametrize("dim,hidden,ntok", [(2048, 5632, 200), (3072, 8192, 200), (1024, 2816, 517), (5120, 5632, 200)])
def test_ffn(qk, torch_gpu, synth, gate, down, dim, hidden, ntok):
    """The pair, its quantized outputs, and down with and without the residual
    (1024 x 2816: down by the int32 kernels)."""
    t = torch_gpu
    assert splits(qk, [(gate, hidden)] * 2, dim, ntok, True)
    assert bool(splits(qk, [(down, dim)], hidden, ntok)) == (dim > 1024)
    gb, db = (Q4_K if ty == Q4_K else Q6_K for ty in (gate, down))
    ws = [synth.quant_matrix(gb, dim, hidden, 9, i) for i in (1, 2)]
    ws.append(synth.quant_matrix(db, hidden, dim, 9, 3))
    g, u = (_dense(t, qk, gb, ws[i], dim, hidden) for i in (0, 1))
    d = _dense(t, qk, db, ws[2], hidden, dim)
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
    gd, ud, dd = (_tensor(t, qk, ty, w, c, r) for ty, w, c, r in
                  [(gate, ws[0], dim, hidden), (gate, ws[1], dim, hidden), (down, ws[2], hidden, dim)])
    xd, sd, work = xq.cuda(), xs.cuda(), t.empty(n, dtype=t.uint8, device="cuda")
    for accumulate in (0, 1):
        y = y0.cuda()
        qk.check(L.qk_ffn_batched_i8(gate, gd.gpu, gate, ud.gpu, down, dd.gpu, xd.data_ptr(), dim, sd.data_ptr(), dim // 32, y.data_ptr(), dim, dim, hidden, ntok,
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
