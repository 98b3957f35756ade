"""Ragged rows at 1..16 activation rows (the kernels' unaligned 16-byte loads
and the shift in a row's last group): rows of under and just over 16 bytes,
ending on every byte of a chunk, against the oracle's float64 linear over
dequant() with the reference's conditioning tolerance
(tests/test_ops_gpu.cu:199-206)."""
import numpy as np
import pytest
import torch

from infer_amd import ops
from tests.gpu_util import QFix, bias_of, check_linear, out_buffer, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("K", [14, 16, 30, 32, 34, 126, 130, 142, 250, 300, 1030, 2050, 4098, 9000])
def test_ragged_rows(kind, K):
    rng = np.random.default_rng(K * 3 + kind)
    for N, k in ((1, K), (35, K), (200, K + (1 if kind == 0 else 2))):
        W = QFix(rng, N, k, kind)
        bb, bd = bias_of(rng, N)
        for M in (1, 2, 4, 5, 9, 16):
            x = rng.standard_normal((M, k), dtype=np.float32)
            y = out_buffer(M, N)
            say("ragged rows", kind, N, k, M)
            ops.launch_gemv_batched_q(torch.from_numpy(x).cuda(), W.view, bd, M, k, N, y)
            torch.cuda.synchronize()
            check_linear(y, x, W, bb, M, f"ragged kind={kind} {N}x{k} M={M}")
