"""The prefill GEMM's load paths at their edges, against the oracle's
float64 linear over dequant() with the reference's conditioning tolerance
(tests/test_ops_gpu.cu:199-206)."""
import numpy as np
import pytest
import torch

from infer_amd import ops
from oracle import oracle as O
from tests.gpu_util import QFix, bias_of, check_linear, out_buffer, say
from tests.test_gpu_routes import Packed, check_sampled

pytestmark = pytest.mark.gpu


def shifted(a, by):
    """The array on the device, starting `by` elements into its allocation
    and ending with it."""
    t = torch.from_numpy(np.ascontiguousarray(a)).cuda()
    buf = torch.zeros(t.numel() + by, dtype=t.dtype, device="cuda")
    buf[by:] = t.view(-1)
    return buf[by:]


# (N, K): rows of one 16-byte chunk and less, rows that end inside a chunk
# and inside a dword, one row past a tile, K of one step and a bit, several
# K ranges; whole groups, for unaligned inputs
@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("N,K", [(1, 14), (3, 16), (5, 30), (2, 32), (129, 34), (64, 66), (65, 130), (257, 1022),
                                 (31, 2050), (128, 256)])
def test_unaligned_rows(kind, N, K):
    rng = np.random.default_rng(1000 * N + K + kind)
    Ks = [K] if kind == 1 or K % 128 == 0 else [K, K + 1]  # int8 rows of odd length too
    for k in Ks:
        W = QFix(rng, N, k, kind)
        bb, bd = bias_of(rng, N)
        for T in (33, 70, 129):
            x = rng.standard_normal((T, k), dtype=np.float32)
            for by in (0, 1):
                y = out_buffer(T, N)
                say("unaligned fp32", kind, N, k, T, by)
                ops.launch_gemm_tiled_q(shifted(x, by), W.view, bd, T, k, N, y)
                torch.cuda.synchronize()
                check_linear(y, x, W, bb, T, f"fp32 kind={kind} {N}x{k} T={T} +{by}")
                xb = O.f32_to_bf16(x)
                y = out_buffer(T, N)
                say("unaligned bf16", kind, N, k, T, by)
                ops.launch_gemm_bf16x(shifted(xb.view(np.int16), by), W.view, bd, T, k, N, y)
                torch.cuda.synchronize()
                check_linear(y, O.bf16_to_f32(xb), W, bb, T, f"bf16 kind={kind} {N}x{k} T={T} +{by}")


@pytest.mark.parametrize("kind", [0, 1])
def test_unaligned_rows_ignore_what_follows(kind):
    """The columns past a row's end are the next row's: non-finite values
    there (the next activation row) must not reach this row's outputs."""
    N, K, T = 40, 202, 66
    rng = np.random.default_rng(9 + kind)
    W = QFix(rng, N, K, kind)
    x = rng.standard_normal((T, K), dtype=np.float32)
    x[1::2] = np.inf
    want, _ = O.linear_dq_f64(x[0::2], W.dq, None)
    for bf16 in (False, True):
        xs = O.f32_to_bf16(x) if bf16 else x
        y = out_buffer(T, N)
        if bf16:
            ops.launch_gemm_bf16x(torch.from_numpy(xs.view(np.int16)).cuda(), W.view, None, T, K, N, y)
            want, _ = O.linear_dq_f64(O.bf16_to_f32(xs)[0::2], W.dq, None)
        else:
            ops.launch_gemm_tiled_q(torch.from_numpy(xs).cuda(), W.view, None, T, K, N, y)
        torch.cuda.synchronize()
        got = y.cpu().numpy()[:T * N].reshape(T, N)
        assert np.all(np.isfinite(got[0::2])) and not np.any(np.isfinite(got[1::2]))
        assert np.abs(got[0::2] - want).max() <= 5e-6 * np.abs(want).max() * 8


# The wide tiles (iq_gemmw.hip): 128- and 256-row tiles of bf16 and 128-row
# tiles of fp32 activations, all K ranges of split tiles, rows and columns
# past the last tile, N that is no multiple of 4 (the reduction's scalar
# stores); whole rounds of tiles beside split ones are in test_gpu_routes
# (the 7B gate at T = 1024).  Which of these calls the wide tiles serve is
# in test_routes.py.
WIDE = [(18947, 3584, (100, 201)), (3587, 18944, (257, 450)), (8192, 4096, (513,))]


@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("N,K,Ts", WIDE)
def test_wide_tiles(kind, N, K, Ts):
    rng = np.random.default_rng(N + kind)
    W = QFix(rng, N, K, kind, sd=0.02)
    bb, bd = bias_of(rng, N)
    for T in Ts:
        x = rng.standard_normal((T, K), dtype=np.float32)
        x[:, rng.integers(0, K, 3)] *= 40.0
        y = out_buffer(T, N)
        say("wide tiles fp32", kind, N, K, T)
        ops.launch_gemm_tiled_q(torch.from_numpy(x).cuda(), W.view, bd, T, K, N, y)
        torch.cuda.synchronize()
        check_linear(y, x, W, bb, T, f"wide fp32 kind={kind} {N}x{K} T={T}")
        xb = O.f32_to_bf16(x)
        y = out_buffer(T, N)
        say("wide tiles bf16", kind, N, K, T)
        ops.launch_gemm_bf16x(torch.from_numpy(xb.view(np.int16)).cuda(), W.view, bd, T, K, N, y)
        torch.cuda.synchronize()
        check_linear(y, O.bf16_to_f32(xb), W, bb, T, f"wide bf16 kind={kind} {N}x{K} T={T}")


# Row counts around the one from which the 7B gate takes wide tiles: 129, 160
# and 177 stay on the narrow ones, 240 takes wide tiles but for int4 with
# fp32 activations (3 row blocks in the last tile's second wave).
@pytest.mark.parametrize("kind", [0, 1])
def test_wide_tiles_row_blocks(kind):
    N, K = 18944, 3584
    rng = np.random.default_rng(31 + kind)
    W = QFix(rng, N, K, kind, sd=0.02)
    for T in (129, 160, 177, 240):
        x = rng.standard_normal((T, K), dtype=np.float32)
        y = out_buffer(T, N)
        say("wide tiles, row blocks", kind, N, K, T)
        ops.launch_gemm_tiled_q(torch.from_numpy(x).cuda(), W.view, None, T, K, N, y)
        torch.cuda.synchronize()
        check_linear(y, x, W, None, T, f"row blocks fp32 kind={kind} T={T}")
        xb = O.f32_to_bf16(x)
        y = out_buffer(T, N)
        ops.launch_gemm_bf16x(torch.from_numpy(xb.view(np.int16)).cuda(), W.view, None, T, K, N, y)
        torch.cuda.synchronize()
        check_linear(y, O.bf16_to_f32(xb), W, None, T, f"row blocks bf16 kind={kind} T={T}")


# Row counts with 1, 2 or 3 of the 4 row blocks of the last 128-row tile's
# first wave in use and none of its second, and all and 1, 2 or 3, for both
# kinds and activation types (test_routes.py asserts it); bf16 at T = 600 and
# 700 the same on 256-row tiles.
LAST_BLOCKS = (18947, 3584, (400, 410, 430, 450, 470, 490, 600, 700))


@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("T", LAST_BLOCKS[2])
def test_wide_tiles_last_row_blocks(kind, T):
    N, K, _ = LAST_BLOCKS
    rng = np.random.default_rng(47 + 2 * T + kind)
    W = Packed(rng, N, K, kind)
    bb, bd = bias_of(rng, N)
    x = rng.standard_normal((T, K), dtype=np.float32)
    y = out_buffer(T, N)
    say("wide tiles, last row blocks", kind, T)
    ops.launch_gemm_tiled_q(torch.from_numpy(x).cuda(), W.view, bd, T, K, N, y)
    torch.cuda.synchronize()
    check_sampled(y, x, W, T, rng, f"last row blocks fp32 kind={kind} T={T}", bb)
    xb = O.f32_to_bf16(x)
    y = out_buffer(T, N)
    ops.launch_gemm_bf16x(torch.from_numpy(xb.view(np.int16)).cuda(), W.view, bd, T, K, N, y)
    torch.cuda.synchronize()
    check_sampled(y, O.bf16_to_f32(xb), W, T, rng, f"last row blocks bf16 kind={kind} T={T}", bb)


# (bf16 at 8192 x 4096 runs the narrow tiles, at 18944 x 3584 128-row wide
# ones, at 3587 x 18944 256-row ones, whose last tile has 4 of 8 row blocks)
NON_FINITE = [(8192, 4096, 513), (18944, 3584, 450), (3587, 18944, 700)]


@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("N,K,T", NON_FINITE)
def test_wide_tiles_non_finite_rows(kind, N, K, T):
    """A row with inf or NaN gives a non-finite output row and leaves the
    other rows as they are."""
    rng = np.random.default_rng(77 + kind)
    W = QFix(rng, N, K, kind, sd=0.02)
    x = rng.standard_normal((T, K), dtype=np.float32)
    bad = x.copy()
    bad[5, 100], bad[300, K - 1], bad[T - 1, 0] = np.inf, np.nan, -np.inf
    rows = [5, 300, T - 1]
    for bf16 in (False, True):
        ys = []
        for v in (x, bad):
            y = torch.empty(T, N, device="cuda")
            if bf16:
                xb = torch.from_numpy(O.f32_to_bf16(v).view(np.int16)).cuda()
                ops.launch_gemm_bf16x(xb, W.view, None, T, K, N, y)
            else:
                ops.launch_gemm_tiled_q(torch.from_numpy(v).cuda(), W.view, None, T, K, N, y)
            ys.append(y)
        torch.cuda.synchronize()
        keep = torch.ones(T, dtype=torch.bool, device="cuda")
        keep[rows] = False
        assert torch.equal(ys[0][keep], ys[1][keep])
        assert not torch.isfinite(ys[1][rows]).all(1).any()
