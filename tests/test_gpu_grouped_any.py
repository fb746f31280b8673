"""GPU tests of the grouped GEMMs that decode Q4_1 / Q8_0 / Q5_K / Q6_K blocks themselves (lmoe_grouped_*_any): the bits
of the f16-weight GEMMs on the dequantized experts, and the oracle's outputs."""
import numpy as np
import pytest
import torch

from oracle import gguf, moe

pytestmark = pytest.mark.gpu
BAR = 2e-3
# group sizes around the 16-row fragments, the 64-row tile and two tiles, and an empty group
SIZES = [0, 1, 15, 16, 17, 31, 33, 48, 49, 63, 64, 65, 200]


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("t,H,I", [("Q8_0", 256, 128), ("Q8_0", 512, 384), ("Q4_1", 256, 128), ("Q4_1", 768, 640),
                                   ("Q5_K", 256, 256), ("Q5_K", 768, 512), ("Q6_K", 256, 256), ("Q6_K", 512, 768)])
@pytest.mark.parametrize("bm", [64, 128])
def test_any_gemms_equal_f16_weights(t, H, I, bm):
    """Contractions of one step (128 weights), an odd count of steps and one super-block up; a slot past the experts."""
    from larder_amd import grouped
    rng = np.random.default_rng(H + I + bm)
    E = len(SIZES)
    types = (t,) * 3
    w = tuple(gguf.random_experts(rng, E, r, c, t) for r, c in ((I, H), (I, H), (H, I)))
    wd = tuple(dev(b) for b in w)
    w16 = tuple(grouped.gemm_weights(b, t) for b in wd)
    slots = np.concatenate([np.full(n, e) for e, n in enumerate(SIZES)]).astype(np.int32)
    rng.shuffle(slots)
    slots[3] = E + 1
    R = slots.size
    x = dev(rng.standard_normal((R, H)).astype(np.float16))
    G = grouped.Grouping(R, E, bm=bm).run(dev(slots))
    assert grouped._decodes_in_gemm(t, H, bm) and grouped._decodes_in_gemm(t, I, bm)
    n = int(G.offsets[-1])
    h = [torch.empty((R, I), dtype=torch.float16, device="cuda") for _ in range(2)]
    for i in range(2):
        grouped.gate_up(x, G, 1, wd[0], wd[1], types, h[i], w16=w16[:2] if i else None)
    assert torch.equal(h[0][:n].view(torch.int16), h[1][:n].view(torch.int16))
    for dt, bits in ((torch.float32, torch.int32), (torch.float16, torch.int16)):
        y = [torch.empty((R, H), dtype=dt, device="cuda") for _ in range(2)]
        for i in range(2):
            grouped.down(h[0], G, wd[2], t, y[i], w16=w16[2] if i else None)
        assert torch.equal(y[0][:n].view(bits), y[1][:n].view(bits))
    order = G.order.cpu().numpy()
    valid = slots[order] < E
    _, want = moe.gemv(x.float().cpu().numpy(), w, slots, 1, types)
    assert moe.rel_l2(y[0].float().cpu().numpy()[valid], want[order][valid]) < BAR
