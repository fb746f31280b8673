"""GPU tests of the drop-in block's one-launch steps against the launches they stand for: the shared expert's gate, up and
SwiGLU (lmoe_qmv_swiglu_rows), probs' best-last order (lmoe_router_probs) and tail (lmoe_combine_rows)."""
import numpy as np
import pytest
import torch

from oracle import qmv

pytestmark = pytest.mark.gpu


def _weight(rng, N, K, G):
    wq, s, b = qmv.quantize_affine4((rng.standard_normal((N, K)) * 0.05).astype(np.float32), G)
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).cuda().bfloat16()  # noqa: E731
    return torch.from_numpy(wq.view(np.int32)).cuda(), d(s), d(b), G


@pytest.mark.parametrize("T,N,K,G", [(1, 512, 2048, 64), (3, 33, 528, 16), (8, 5, 64, 32), (9, 64, 1056, 48)])
def test_qmv_swiglu_same_bits(T, N, K, G):
    from larder_amd import trunk
    from larder_amd._lib import call, ptr, stream
    rng = np.random.default_rng(T + N)
    gate, up = _weight(rng, N, K, G), _weight(rng, N, K, G)
    x = torch.from_numpy(rng.standard_normal((T, K)).astype(np.float32)).cuda().bfloat16()
    g, u = trunk.qmv_rows(x, *gate), trunk.qmv_rows(x, *up)
    want = torch.empty_like(g)
    call("lmoe_swiglu_bf16", ptr(g), ptr(u), g.numel(), ptr(want), stream())
    got = torch.empty_like(g)
    call("lmoe_qmv_swiglu_rows", ptr(x), T, *(ptr(t) for t in gate[:3] + up[:3]), N, K, G, ptr(got), stream())
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))


def _column_slices(w):
    """An affine weight's tensors as column slices of wider buffers."""
    wide = [torch.cat([t, t.flip(0)[:, :8]], 1)[:, :t.shape[1]] for t in w[:3]]
    assert not any(t.is_contiguous() for t in wide)
    return (*wide, w[3])


def test_shared_expert_rows_of_strided_weights():
    """Weights, scales and biases of gate and up that are column slices: the contiguous call's bits."""
    from larder_amd import trunk
    rng = np.random.default_rng(11)
    gate, up, down = _weight(rng, 256, 512, 64), _weight(rng, 256, 512, 64), _weight(rng, 512, 256, 64)
    x = torch.from_numpy(rng.standard_normal((5, 512)).astype(np.float32)).cuda().bfloat16()
    want = trunk.shared_expert_rows(x, gate, up, down)
    got = trunk.shared_expert_rows(x, _column_slices(gate), _column_slices(up), down)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))


def test_qmv_rows_of_strided_weights():
    from larder_amd import trunk
    rng = np.random.default_rng(12)
    w = _weight(rng, 96, 512, 64)
    x = torch.from_numpy(rng.standard_normal((5, 512)).astype(np.float32)).cuda().bfloat16()
    want, got = trunk.qmv_rows(x, *w), trunk.qmv_rows(x, *_column_slices(w))
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("T,E,k", [(1, 256, 8), (5, 512, 10), (4, 60, 4), (67, 9, 9), (3, 1024, 32)])
def test_probs_is_topk_reversed(T, E, k):
    from larder_amd import route
    lg = torch.randn((T, E), generator=torch.Generator(device="cuda").manual_seed(E), device="cuda").bfloat16()
    ids, sc = route.topk(lg, k, True)
    inds, scores = route.probs(lg, k, True)
    assert torch.equal(inds, ids.flip(-1)) and torch.equal(scores, sc.flip(-1))


@pytest.mark.parametrize("k", [1, 2, 3, 7, 8, 11, 15, 16])
@pytest.mark.parametrize("dt", [torch.float32, torch.float16, torch.bfloat16])
def test_tail_every_row_count_and_dtype(k, dt):
    """Any count of rows a token, aligned and odd widths, shared rows and gates in y's dtype."""
    from larder_amd import route
    g = torch.Generator(device="cuda").manual_seed(k)
    r = lambda *s: torch.randn(s, generator=g, device="cuda")  # noqa: E731
    for D in (64, 2056, 33):
        y, sc, sh, gate = r(3, k, D).to(dt), r(3, k), r(3, D).to(dt), r(3, 1).to(dt)
        want = (y.double() * sc.double()[..., None]).sum(-2)
        tol = {torch.float32: 1e-5, torch.float16: 1e-3, torch.bfloat16: 8e-3}[dt]  # one rounding of the output
        for shared in (None, sh):
            w = want if shared is None else want + torch.sigmoid(gate.double()) * sh.double()
            got = route.tail(y, sc, shared, None if shared is None else gate).double()
            assert float((got - w).norm() / w.norm()) < tol


@pytest.mark.parametrize("D", [64, 33])
@pytest.mark.parametrize("y_dt,sh_dt,gate_dt", [(torch.bfloat16, torch.float32, torch.float16),
                                                (torch.float16, torch.bfloat16, torch.float32),
                                                (torch.float32, torch.float16, torch.bfloat16),
                                                (torch.bfloat16, torch.float64, torch.float16),
                                                (torch.float32, torch.bfloat16, torch.float64)])
def test_tail_mixed_dtypes(y_dt, sh_dt, gate_dt, D):
    """y, shared rows and gates of three dtypes (float64 is read as float32): what float32 copies of the two give, bit for
    bit, and the sum in float64."""
    from larder_amd import route
    g = torch.Generator(device="cuda").manual_seed(D)
    r = lambda *s: torch.randn(s, generator=g, device="cuda")  # noqa: E731
    y, sc, sh, gate = r(3, 8, D).to(y_dt), r(3, 8), r(3, D).double().to(sh_dt), r(3, 1).double().to(gate_dt)
    got = route.tail(y, sc, sh, gate)
    assert got.dtype == y_dt and torch.equal(got, route.tail(y, sc, sh.float(), gate.float()))
    want = (y.double() * sc.double()[..., None]).sum(-2) + torch.sigmoid(gate.double()) * sh.double()
    tol = {torch.float32: 1e-5, torch.float16: 1e-3, torch.bfloat16: 8e-3}[y_dt]  # one rounding of the output
    assert float((got.double() - want).norm() / want.norm()) < tol
