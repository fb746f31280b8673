"""GPU test of lmoe_grouped_down_rows (down's rows straight to the caller's order and dtype) and lmoe_rows_to_gemm_f16
against the GEMM in grouped order, unsorted and rounded by torch: the same values; rows past the experts zero."""
import numpy as np
import pytest
import torch

from oracle import gguf

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t,bm,ks", [("Q4_0", 32, 1), ("Q4_0", 32, 2), ("Q4_0", 64, 1), ("Q4_0", 128, 1), ("Q4_K", 32, 1),
                                     ("Q4_K", 64, 1), ("Q4_K", 128, 1), ("Q8_0", 64, 1), ("Q6_K", 128, 1)])
@pytest.mark.parametrize("odt", [torch.float32, torch.float16, torch.bfloat16])
def test_down_rows(t, bm, ks, odt):
    from larder_amd import grouped
    from larder_amd._lib import call, dcode, ptr, qcode, stream
    H, I, sizes = 512, 256, [0, 1, 15, 31, 33, 64, 129]
    rng = np.random.default_rng(bm + ks)
    E = len(sizes)
    wd = torch.from_numpy(gguf.random_experts(rng, E, H, I, t)).cuda()
    slots = np.concatenate([np.full(n, e) for e, n in enumerate(sizes)] + [[E, -1, E + 7]]).astype(np.int32)
    rng.shuffle(slots)
    ids = torch.from_numpy(slots).cuda()
    R = slots.size
    x = torch.from_numpy(rng.standard_normal((R, I)).astype(np.float32)).cuda()
    G = grouped.Grouping(R, E, bm=bm).run(ids)
    xh = torch.empty((R, I), dtype=torch.float16, device="cuda")
    out = torch.full((R, H), 7.0, dtype=odt, device="cuda")
    # the conversion clears the rows of out (of x's width) that no expert writes; out is cleared at its own width here
    clear = torch.full((R, I), 7.0, dtype=odt, device="cuda")
    call("lmoe_rows_to_gemm_f16", ptr(x), dcode(x.dtype), R, I, ptr(ids), E, ptr(xh), ptr(clear), dcode(odt), stream())
    assert torch.equal(xh, grouped.as_gemm_f16(x))
    bad = (ids < 0) | (ids >= E)
    assert (clear[bad] == 0).all() and (clear[~bad] == 7).all()
    h = xh[G.order.long()]
    y = torch.zeros((R, H), dtype=torch.float32, device="cuda")
    grouped.down(h, G, wd, t, y, ksplit=ks)
    ws = torch.empty(ks * R * H, dtype=torch.float32, device="cuda")
    call("lmoe_grouped_down_rows", ptr(h), R, ptr(G.order), ptr(G.offsets), ptr(G.tiles), ptr(G.n_tiles), G.max_tiles, bm,
         ks, ptr(ws), ptr(wd), qcode(t), E, I, H, ptr(out), dcode(odt), stream())
    want = y[G.inv.long()].to(odt)
    assert torch.equal(out[~bad], want[~bad]) and (out[bad] == 7).all()


@pytest.mark.parametrize("t,bm,ks", [("Q4_0", 32, 1), ("Q4_0", 32, 2), ("Q4_0", 128, 1), ("Q4_K", 64, 1), ("Q8_0", 64, 1)])
def test_down_rows_zero_signs_f16(t, bm, ks):
    """Negative sums of 2^-28, below half of f16's least value: +0, the bits of the grouped f16 rows unsorted by the combine."""
    from larder_amd import grouped
    from larder_amd._lib import F16, call, ptr, qcode, stream
    E, R, H, I = 2, 37, 256, 256
    be, bb = {"Q4_0": (32, 18), "Q8_0": (32, 34), "Q4_K": (256, 144)}[t]
    b = torch.zeros((E, H, I // be, bb), dtype=torch.uint8)
    neg = torch.tensor([2.0 ** -14]).half().view(torch.uint8)
    b[..., :2] = neg  # d
    if t == "Q4_0":  # weights (q - 8) d = -d, and +d in every other row
        b[:, :, :, 2:] = 0x77
        b[:, ::2, :, 2:] = 0x99
    elif t == "Q8_0":
        b[:, :, :, 2:] = 0xFF
        b[:, ::2, :, 2:] = 1
    else:  # q d sc - dmin m with q = 0, m = 1 in every sub-block: -dmin; q = 2, sc = 1 in every other row: +d
        b[..., 2:4] = neg
        b[..., 4:12] = 1
        b[..., 12:16] = 0x11
        b[:, ::2, :, 16:] = 0x22
    wd = b.reshape(E, H, -1).cuda()
    h = torch.zeros((R, I), dtype=torch.float16, device="cuda")
    h[:, 0] = 2.0 ** -14
    G = grouped.Grouping(R, E, bm=bm).run((torch.arange(R, dtype=torch.int32) % E).cuda())
    y = torch.zeros((R, H), dtype=torch.float16, device="cuda")
    grouped.down(h, G, wd, t, y, ksplit=ks)
    assert (y[:, 1::2].view(torch.int16) == -2 ** 15).all()  # -0 in the grouped rows: the case is met
    want, out = torch.empty_like(y), torch.empty_like(y)
    call("lmoe_combine_sorted", ptr(y), F16, ptr(G.inv), None, R, 1, H, None, None, 0, None, 0, ptr(want), F16, stream())
    ws = torch.empty(ks * R * H, dtype=torch.float32, device="cuda")
    call("lmoe_grouped_down_rows", ptr(h), R, ptr(G.order), ptr(G.offsets), ptr(G.tiles), ptr(G.n_tiles), G.max_tiles, bm,
         ks, ptr(ws), ptr(wd), qcode(t), E, I, H, ptr(out), F16, stream())
    assert torch.equal(out.view(torch.int16), want.view(torch.int16))
