"""A call that takes strided tensors hands the library contiguous copies: each must live until the launch has gone out, or the
allocator gives its block to the next copy. On the CPU, with the library call replaced by one that looks at the copies."""
import weakref

import pytest
import torch

from larder_amd import grouped, trunk


def _wide(t):
    """t's values as a column slice of a wider buffer (not contiguous)."""
    buf = torch.empty(t.shape[:-1] + (t.shape[-1] + 8,), dtype=t.dtype, device=t.device)
    buf[..., :t.shape[-1]] = t
    return buf[..., :t.shape[-1]]


def _affine(n, k, g, wide=True):
    parts = (torch.zeros((n, k // 8), dtype=torch.int32), torch.ones((n, k // g), dtype=torch.bfloat16),
             torch.ones((n, k // g), dtype=torch.bfloat16))
    return tuple(_wide(p) if wide else p for p in parts) + (g,)


@pytest.fixture
def launches(monkeypatch):
    """Names of the library calls made; every tensor that a call has a pointer of is alive when it goes out."""
    held, names = [], []

    def ptr(t):
        if t is None:
            return None
        assert t.is_contiguous()
        held.append(weakref.ref(t))
        return t.data_ptr()

    def call(name, *args):
        gone = sum(r() is None for r in held)
        assert not gone, f"{name}: {gone} of its {len(held)} tensors were freed before the launch"
        held.clear()
        names.append(name)

    for module in (grouped, trunk):
        monkeypatch.setattr(module, "ptr", ptr)
        monkeypatch.setattr(module, "call", call)
        monkeypatch.setattr(module, "stream", lambda: None)
    return names


def test_shared_expert_rows_holds_its_copies(launches):
    x = _wide(torch.zeros((3, 64), dtype=torch.bfloat16))
    trunk.shared_expert_rows(x, _affine(32, 64, 32), _affine(32, 64, 32), _affine(64, 32, 32, wide=False))
    assert launches == ["lmoe_qmv_swiglu_rows", "lmoe_qmv_rows"]


def test_qmv_rows_holds_its_copies(launches):
    x = _wide(torch.zeros((3, 64), dtype=torch.bfloat16))
    trunk.qmv_rows(x, *_affine(32, 64, 32))
    assert launches == ["lmoe_qmv_rows"]


def test_stream_copy_holds_its_copy(built_lib, launches):
    grouped.stream_copy(_wide(torch.zeros((2, 128, 2048 // 32 * 18), dtype=torch.uint8)), "Q4_0")
    assert launches == ["lmoe_stream_repack"]
