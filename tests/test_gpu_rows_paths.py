"""The rows GEMV whose waves hold their activations (gemvw_kernel) at its
edges, against the oracle's float64 linear over dequant() with the
reference's conditioning tolerance (tests/test_ops_gpu.cu:199-206): one tile
and a few, ragged last tiles, tile counts around a chunk of 4, waves with
one, two and four groups, several K ranges, several matrices, every packing
of the rows."""
import numpy as np
import pytest
import torch

from infer_amd import ops
from oracle import oracle as O
from tests.gpu_util import QFix, bias_of, check_linear, out_buffer, say

pytestmark = pytest.mark.gpu


# (row counts of the matrices, K): the kernel serves MANY at every row count
# of the test, LONG up to 16 rows, and of SOME only part (test_routes.py
# asserts which; the other kernels the rest)
MANY = [((16389, 1, 40), 1024), ((1025, 17), 16384), ((1030,), 16640)]
LONG = [((1,), 16640), ((17,), 16384), ((250, 33), 16640)]
SOME = [((1,), 6144), ((17,), 8960), ((250, 33), 8960), ((1025,), 6400), ((1024, 500), 256),
        ((4609,), 3584), ((16400,), 512), ((1100, 16, 5), 12800)]


@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("Ns,K", SOME + MANY + LONG)
def test_rows_edges(kind, Ns, K):
    rng = np.random.default_rng(sum(Ns) + K + kind)
    Ws = [QFix(rng, N, K, kind, sd=0.02) for N in Ns]
    bs = [bias_of(rng, N) for N in Ns]
    for M in (5, 8, 9, 16, 17, 32):
        x = rng.standard_normal((M, K), dtype=np.float32)
        x[:, rng.integers(0, K, 2)] *= 50.0
        ys = [out_buffer(M, N) for N in Ns]
        say("rows edges", kind, Ns, K, M)
        ops.gemv_multi(torch.from_numpy(x).cuda(), [W.view for W in Ws], [b[1] for b in bs], M, K, ys)
        torch.cuda.synchronize()
        for W, b, y, N in zip(Ws, bs, ys, Ns):
            check_linear(y, x, W, b[0], M, f"rows kind={kind} {Ns}x{K} M={M}")


@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("M", [5, 16, 32])
@pytest.mark.parametrize("K", [8960, 16384])
def test_rows_non_finite(kind, M, K):
    """inf and NaN in a row make that row non-finite and leave the others
    bit for bit as they are (K = 8960 at 5 rows on the 1-row kernel, the
    rest on this one)."""
    N = 1600
    rng = np.random.default_rng(3 + kind)
    W = QFix(rng, N, K, kind, sd=0.02)
    x = rng.standard_normal((M, K), dtype=np.float32)
    bad = x.copy()
    bad[1, 200], bad[M - 1, K - 1] = np.inf, np.nan
    ys = []
    for v in (x, bad):
        y = torch.empty(M, N, device="cuda")
        ops.launch_gemv_batched_q(torch.from_numpy(v).cuda(), W.view, None, M, K, N, y)
        ys.append(y)
    torch.cuda.synchronize()
    keep = [m for m in range(M) if m not in (1, M - 1)]
    assert torch.equal(ys[0][keep], ys[1][keep])
    assert not torch.isfinite(ys[1][[1, M - 1]]).any()


# (N of 3 ranges' sums inside and beyond the no-allocation scratch)
SCRATCH = dict(inside=38000, beyond=48000, K=6144, M=32)


@pytest.mark.parametrize("N", [SCRATCH["inside"], SCRATCH["beyond"]])
def test_rows_small_scratch(N):
    """More range sums than the no-allocation scratch holds: another route,
    the same result."""
    K, M, kind = SCRATCH["K"], SCRATCH["M"], 1
    rng = np.random.default_rng(11)
    W = QFix(rng, N, K, kind, sd=0.02)
    x = rng.standard_normal((M, K), dtype=np.float32)
    y = out_buffer(M, N)
    ops.gemv_noalloc(torch.from_numpy(x).cuda(), W.view, None, M, K, N, y)
    torch.cuda.synchronize()
    check_linear(y, x, W, None, M, "rows, small scratch")
