"""Where the grouped GEMMs of the block types beyond Q4 take an f16 copy made first and where they decode the blocks
(grouped._dequant_pays): the measured points on both sides of the line, and the same bits on either route."""
from types import SimpleNamespace

import pytest
import torch

from larder_amd import _lib, grouped


def grouping(rows_an_expert, E, bm=64):
    R = rows_an_expert * E
    return SimpleNamespace(R=R, E=E, bm=bm, max_tiles=-(-R // bm) + E)


# (type, matrices, their rows, contraction, experts): the most rows an expert measured faster on blocks, the least on a copy
LINES = [
    ("Q6_K", 2, 768, 2048, 128, 512, 1024), ("Q5_K", 2, 768, 2048, 128, 512, 1024), ("Q8_0", 2, 768, 2048, 128, 1024, 1536),
    ("Q4_1", 2, 768, 2048, 128, 2048, None), ("Q6_K", 1, 2048, 768, 128, 512, 768), ("Q8_0", 1, 2048, 768, 128, 768, 1536),
    ("Q4_1", 1, 2048, 768, 128, 2048, None), ("Q8_0", 2, 1408, 2048, 60, 1024, 2048), ("Q8_0", 1, 2048, 1408, 60, 1024, 1536),
    ("Q6_K", 1, 2048, 512, 256, 256, 768), ("Q6_K", 1, 2048, 512, 1, 4096, None), ("Q6_K", 2, 512, 2048, 1, 1024, None),
    ("Q6_K", 1, 2048, 5632, 1, None, 16), ("Q5_K", 1, 2048, 5632, 1, None, 16), ("Q8_0", 2, 5632, 2048, 1, 4096, None),
]


@pytest.mark.parametrize("t,mats,rows,K,E,blocks,copy", LINES)
def test_rule_on_both_sides(t, mats, rows, K, E, blocks, copy):
    if blocks is not None:
        assert not grouped._dequant_pays(t, mats, rows, K, grouping(blocks, E))
        assert not grouped._dequant_pays(t, mats, rows, K, grouping(1, E))
    if copy is not None:
        assert grouped._dequant_pays(t, mats, rows, K, grouping(copy, E))


def test_rule_keeps_what_only_blocks_take():
    """down's f16-weight GEMM takes at most 4 GiB of h, padded to its tiles; the blocks' takes them unpadded."""
    g = grouping(2 ** 21 // 8, 8)
    assert not grouped._dequant_pays("Q6_K", 1, 2048, 1024, g)
    assert grouped._dequant_pays("Q6_K", 1, 2048, 1024, grouping(2 ** 20 // 8, 8))


@pytest.mark.gpu
@pytest.mark.parametrize("t", ("Q6_K", "Q5_K", "Q8_0"))
def test_both_routes_same_bits(t, monkeypatch):
    """A gate/up and a down where the copy pays (one expert, long rows), with a row past the experts."""
    K = 8192
    gen = torch.Generator(device="cuda").manual_seed(3)
    from larder_amd import gguf_experts
    wg, wu, wd = (gguf_experts._random_q4(1, 256, K, t, gen) for _ in range(3))
    R = 37
    ids = torch.zeros(R, dtype=torch.int32, device="cuda")
    ids[5] = 1
    G = grouped.Grouping(R, 1, bm=64).run(ids)
    x = torch.randn((R, K), generator=gen, device="cuda").half()
    names = []
    monkeypatch.setattr(grouped, "call", lambda name, *a: (names.append(name), _lib.call(name, *a)))

    def both():
        h = torch.zeros((R, 256), dtype=torch.float16, device="cuda")
        y = torch.zeros((R, 256), dtype=torch.float32, device="cuda")
        grouped.gate_up(x, G, 1, wg, wu, (t, t), h, prepped=True)
        grouped.down(x, G, wd, t, y)
        return h, y

    copied = both()
    assert names == ["lmoe_dequant_gemm_f16"] * 2 + ["lmoe_grouped_gate_up_f16w", "lmoe_dequant_gemm_f16",
                                                    "lmoe_grouped_down_f16w"]
    names.clear()
    monkeypatch.setattr(grouped, "_dequant_pays", lambda *a: False)
    decoded = both()
    assert names == ["lmoe_grouped_gate_up_any", "lmoe_grouped_down_any"]
    assert all(torch.equal(a, b) for a, b in zip(copied, decoded)) and bool(copied[1].any())
