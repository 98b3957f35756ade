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


# (row counts of the matrices, K): K = 6144 / 8960 / 12800 take the kernel at
# any row count (G >= 48), the others from 17 rows on or on enough tiles
@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("Ns,K", [((1,), 6144), ((17,), 8960), ((250, 33), 8960), ((1025,), 6400), ((1024, 500), 256),
                                  ((4609,), 3584), ((16400,), 512), ((1100, 16, 5), 12800)])
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
def test_rows_non_finite(kind, M):
    """inf and NaN in a row make that row non-finite and leave the others
    bit for bit as they are."""
    N, K = 1600, 8960
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


def test_rows_small_scratch():
    """More range sums than the no-allocation scratch holds: another route,
    the same result."""
    N, K, M, kind = 38000, 6144, 32, 1
    rng = np.random.default_rng(11)
    W = QFix(rng, N, K, kind, sd=0.02)
    x = rng.standard_normal((M, K), dtype=np.float32)
    y = out_buffer(M, N)
    ops.gemv_noalloc(torch.from_numpy(x).cuda(), W.view, None, M, K, N, y)
    torch.cuda.synchronize()
    check_linear(y, x, W, None, M, "rows, small scratch")
