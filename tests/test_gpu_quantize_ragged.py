"""On-device quantize of rows that are not whole 128-column groups, bit for
bit against the oracle: rows ending inside a 16-column chunk, inside a 4-byte
word and on either, the matrix's last value included; rows short enough to
share a wave; what follows a row
(the next row, here with NaN and infinities in it) must not reach its codes;
inputs off 16-byte alignment; nothing is written past the codes."""
import numpy as np
import pytest
import torch

from infer_amd import ops
from oracle import oracle as O
from tests.gpu_util import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("rows,cols", [(1, 1), (3, 2), (2, 15), (5, 16), (3, 17), (9, 127), (4, 129), (7, 143), (6, 1023),
                                       (5, 1024 + 16), (4, 1025), (3, 2049), (700, 300), (3000, 131),
                                       # rows that share a wave: 8, 4 or 2, and a last wave with fewer
                                       (8, 100), (17, 99), (9, 255), (4, 250), (5, 257), (2, 383), (3, 385), (2051, 511), (4, 513)])
def test_quantize_ragged_rows(kind, rows, cols):
    if kind == 1:
        cols += cols % 2
    rng = np.random.default_rng(rows * 10007 + cols + kind)
    w = O.seeded_bf16(rng, (rows, cols), 0.05)
    w[1::3, 0] = np.array([0x7FC0, 0x7F80, 0xFF80], np.uint16)[rng.integers(0, 3, len(w[1::3]))]  # NaN, +-inf
    q, s, z = O.quantize(w, kind)
    for by in (0, 1):
        buf = torch.zeros(rows * cols + by, dtype=torch.int16, device="cuda")
        buf[by:] = torch.from_numpy(w.view(np.int16).reshape(-1)).cuda()
        out = ops.alloc_quant(kind, rows, cols)
        n = out.q.numel()
        big = torch.full((n + 32,), 0xA5, dtype=torch.uint8, device="cuda")
        out = ops.QuantView(kind, rows, cols, big[:n], out.scales, out.zeros)
        say("quantize ragged", kind, rows, cols, by)
        ops.quantize(buf[by:].view(rows, cols), kind, out=out)
        torch.cuda.synchronize()
        assert np.array_equal(big[:n].cpu().numpy(), q.reshape(-1))
        assert bool((big[n:] == 0xA5).all())
        assert np.array_equal(out.scales.cpu().numpy().view(np.uint16), s.reshape(-1))
        if kind == 1:
            assert np.array_equal(out.zeros.cpu().numpy(), z.reshape(-1))
