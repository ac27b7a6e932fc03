"""The inference step's whole-layer call on inputs of every layout that the
separate ops take: rows at any offset and stride."""

import pytest
import torch

from redpanda_amd import layer_step
from tests.test_gpu_layer_step import _model, _ply, _state

pytestmark = pytest.mark.gpu
dev = "cuda"


def _offset(x, by):
    store = torch.zeros(x.numel() + by, device=dev)
    return store[by:].view_as(x).copy_(x)


def _columns(x, by, row):
    big = torch.zeros(x.shape[0], row, device=dev)
    return big[:, by:by + x.shape[1]].copy_(x)


LAYOUTS = {
    "contiguous, off 16 bytes": lambda x: _offset(x, 1),
    "columns off 16 bytes": lambda x: _columns(x, 2, 68),
    "odd row stride": lambda x: _columns(x, 0, 65),
    "even row stride": lambda x: _columns(x, 4, 76),
    "transposed": lambda x: x.t().contiguous().t(),
}


@pytest.mark.parametrize("R", [1, 3])
@pytest.mark.parametrize("layout", list(LAYOUTS))
def test_rows_of_any_layout(gpu_lib, monkeypatch, layout, R):
    m = _model()
    x = torch.randn(R, 64, generator=torch.Generator().manual_seed(R)).to(dev)
    cache = _state(m, R, "full")
    want = _ply(m, x, cache, monkeypatch, True)
    xl = LAYOUTS[layout](x)
    assert torch.equal(xl, x) and layer_step.usable(m, xl)
    got = _ply(m, xl, cache, monkeypatch, True)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    assert _ply(m, xl, cache, monkeypatch, False)[0].shape == (R, 64)  # the separate ops take it too
