"""Products of 2 to 7 tokens (csrc/qk_few.hip): row counts around the 16-row
tile and the two-tile step, one to thirty-two blocks a row (one or two a wave),
every storage type alone and mixed, scales over the whole int8 range, the
feed-forward block's pair and residual, values that are not finite.  The sizes
are those that few_pays takes (enough weight bytes for the token count); the
small ones beside them go to the GEMV kernels."""
import numpy as np
import pytest

from conftest import rel_l2, to_dev
from test_gpu_tile_gemm import Q4_K, Q6_K, Q6_K_SPLIT, TOL, check, matrix

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("qtype", [Q4_K, Q6_K, Q6_K_SPLIT])
@pytest.mark.parametrize("ntok,cols,rows", [(7, 256, 66001), (7, 768, 32015), (4, 2048, 65541), (6, 3072, 16400),
                                            (5, 4096, 12001), (7, 4352, 3903), (7, 8192, 3899), (7, 8192, 3700),
                                            (3, 1024, 20)])
def test_edges(qk, torch_gpu, oracle, workloads, synth, qtype, ntok, cols, rows):
    x = synth.normal_f32(ntok * cols, 61, ntok).reshape(ntok, cols)
    check(qk, torch_gpu, oracle, [matrix(qk, torch_gpu, workloads, synth, qtype, cols, rows, 60 + ntok)], x, cols)


@pytest.mark.parametrize("ntok,cols", [(7, 2048), (5, 2560), (3, 512)])
def test_mixed_types(qk, torch_gpu, oracle, workloads, synth, ntok, cols):
    x = synth.normal_f32(ntok * cols, 62, ntok).reshape(ntok, cols)
    tensors = [matrix(qk, torch_gpu, workloads, synth, ty, cols, rows, 70 + i)
               for i, (ty, rows) in enumerate([(Q4_K, 16500), (Q6_K, 96), (Q6_K_SPLIT, 257), (Q4_K, 20)])]
    check(qk, torch_gpu, oracle, tensors, x, cols)


@pytest.mark.parametrize("types", [(Q4_K, Q4_K, Q6_K), (Q4_K, Q6_K, Q4_K), (Q6_K_SPLIT, Q6_K_SPLIT, Q6_K_SPLIT)])
@pytest.mark.parametrize("ntok,dim,hidden", [(7, 2048, 4096), (5, 3072, 4096), (7, 1024, 8192), (2, 512, 768)])
def test_ffn(qk, torch_gpu, oracle, workloads, synth, types, ntok, dim, hidden):
    t = torch_gpu
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


def test_not_finite(qk, torch_gpu, workloads, synth):
    """A non-finite activation poisons its own token's outputs only."""
    t = torch_gpu
    ntok, cols, rows = 4, 1024, 100
    x = synth.normal_f32(ntok * cols, 64, 1).reshape(ntok, cols)
    x[2, 700] = np.inf
    ten, _, _ = matrix(qk, t, workloads, synth, Q4_K, cols, rows, 90)
    y = t.empty((ntok, rows), device="cuda")
    qk.batch_matvec(ten, to_dev(t, x), y, cols, rows, ntok)
    t.cuda.synchronize()
    got = y.cpu().numpy()
    assert np.isnan(got[2]).all() and np.isfinite(got[[0, 1, 3]]).all()


def test_infinite_scale_in_the_last_block(qk, torch_gpu, oracle, workloads, synth):
    """31 blocks a row, two a wave: the wave without a second block adds nothing.
    Where the row's last block has an infinite scale, its high and low products
    are infinite, of one sign in about half of the outputs; the last block again
    over zeros would make every one NaN."""
    t = torch_gpu
    ntok, cols, rows = 7, 31 * 256, 4096
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
