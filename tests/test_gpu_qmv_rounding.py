"""GPU test of lmoe_qmv_rows' fused multiply-add (rounded to odd in float32, then to bf16) where its rounding decides: the
bits of the oracle on rows full of exact ties, of exact cancellations (signed zeros) and of sums far apart in exponent, and
on group sizes that do not divide the 512-element step."""
import numpy as np
import pytest
import torch

from oracle import qmv

pytestmark = pytest.mark.gpu


def dev_bf16(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).cuda().bfloat16()


@pytest.mark.parametrize("K,N,G", [(16, 1, 16), (96, 9, 48), (1056, 37, 48), (2048, 65, 1024), (1536, 24, 512)])
@pytest.mark.parametrize("kind", ["ties", "cancel", "apart"])
def test_qmv_rounding_bits(K, N, G, kind):
    from larder_amd import trunk
    rng = np.random.default_rng(K + N)
    wq = rng.integers(0, 2 ** 32, (N, K // 8), dtype=np.uint64).astype(np.uint32)
    s = qmv.bf16(np.exp2(rng.integers(-3, 2, (N, K // G))))
    b = qmv.bf16(-np.exp2(rng.integers(-3, 3, (N, K // G))))
    x = qmv.bf16((1 + rng.integers(0, 128, (8, K)) / 128) * np.exp2(rng.integers(-2, 3, (8, K))) *
                 rng.choice([-1.0, 1.0], (8, K)))
    if kind == "cancel":  # the second half of a row repeats the first half's weights against -x: slots return to zero
        h = K // 2 // 512 * 512
        if h:
            x[:, h:2 * h] = -x[:, :h]
            wq[:, h // 8:h // 4] = wq[:, :h // 8]
            s[:], b[:] = s[:, :1], b[:, :1]
        else:
            x[:, ::2] = 0.0
    if kind == "apart":
        x = qmv.bf16(x * np.exp2(rng.integers(-30, 31, (8, K))))
    W = (torch.from_numpy(wq.view(np.int32)).cuda(), dev_bf16(s), dev_bf16(b))
    for t in (1, 3, 8):
        got = trunk.qmv_rows(dev_bf16(x[:t]), *W, G).float().cpu().numpy()
        assert (got.view(np.uint32) == qmv.qmv_rows(x[:t], wq, s, b, G).view(np.uint32)).all(), (K, N, G, kind, t)
