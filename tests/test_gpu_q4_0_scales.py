"""GPU test of the grouped Q4_0 GEMM at the largest block scales: (q - 8) d fits f16 for small |q - 8| though 8 d does
not. With a power of two for d, down's rows are exactly d times those at d = 1 (f32 accumulation and output)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


# one-unit K steps (K % 128 != 0) and two-unit ones; 64 is one step, which does not split
@pytest.mark.parametrize("bm,ks,I", [(32, 1, 64), (64, 1, 64), (128, 1, 64), (32, 1, 256), (32, 2, 256), (64, 1, 256),
                                     (128, 1, 256)])
@pytest.mark.parametrize("d", [8192.0, -8192.0, 16384.0])
def test_scales_past_an_eighth_of_f16(bm, ks, d, I):
    from larder_amd import grouped
    E, H, R = 3, 256, 2 * bm + 5
    rng = np.random.default_rng(7)
    q = rng.integers(5, 12, (E, H, I // 32, 32), dtype=np.uint8)  # |q - 8| <= 3: 3 x 16384 fits f16

    def blocks(scale):
        b = np.empty((E, H, I // 32, 18), np.uint8)
        b[..., :2] = np.array([scale], np.float16).view(np.uint8)
        b[..., 2:] = q[..., :16] | (q[..., 16:] << 4)
        return torch.from_numpy(b.reshape(E, H, -1)).cuda()

    ids = torch.from_numpy(rng.integers(0, E, R).astype(np.int32)).cuda()
    h = torch.from_numpy(rng.standard_normal((R, I)).astype(np.float16)).cuda()
    G = grouped.Grouping(R, E, bm=bm).run(ids)
    y = [torch.zeros((R, H), dtype=torch.float32, device="cuda") for _ in range(2)]
    for out, scale in zip(y, (np.sign(d), d)):  # the matrix core's sums need not mirror under a change of sign
        grouped.down(h, G, blocks(scale), "Q4_0", out, ksplit=ks)
    assert torch.isfinite(y[1]).all() and (y[0] != 0).any()
    assert torch.equal(y[1], y[0] * abs(d))
