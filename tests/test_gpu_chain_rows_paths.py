"""Chain stages at 5..32 rows on the kernel whose waves hold their
activations (gemvw_kernel's chain instances): one wave a workgroup (more rows
than its row factors' first set), two groups a wave, four, K split (down of
36 and 128 groups at any row count, from 17 rows also 28 groups), both kinds,
SwiGLU pairs, residuals, the sums of squares handed to the next stage; stage
by stage against the oracle on the chain's own inputs."""
import numpy as np
import pytest
import torch

from infer_amd import chain as C
from tests.gpu_util import say
from tests.test_gpu_chain import RowView, check_step, make_model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B", [5, 8, 9, 17, 24, 32])
@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("H,I,nh,nkv", [(256, 512, 2, 1), (1024, 2304, 8, 2), (1536, 3072, 12, 2), (3584, 4608, 28, 4),
                                         (256, 16384, 2, 1)])
def test_chain_rows_holding_waves(H, I, nh, nkv, kind, B):
    rng = np.random.default_rng(H + 7 * B + kind)
    host, dev = make_model(rng, H=H, I=I, nh=nh, nkv=nkv, hd=128, V=1000, L=2, kind=kind, head_kind=0)
    tokens = [int(t) for t in rng.integers(0, 1000, B)]
    say("chain rows, holding waves", H, I, kind, B)
    step = C.DecodeStep(dev, rows=B)
    step.step(tokens)
    torch.cuda.synchronize()
    pick = np.random.default_rng(5)
    for b in sorted({0, 4, B // 2, B - 1}):
        check_step(RowView(step, b), host, idx_of=lambda n: np.unique(np.r_[0, n - 1, pick.choice(n, min(n, 200))]))
    first = step.logits.clone()
    step.step(tokens)
    torch.cuda.synchronize()
    assert torch.equal(first, step.logits)
