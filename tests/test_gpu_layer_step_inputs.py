"""The inference step's whole-layer call on inputs of every layout that the
separate ops take: rows at any offset and stride, gate parameters of any
stride."""

import pytest
import torch
import torch.nn as nn

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


@pytest.mark.parametrize("names", [("A_log_mag", "A_phase"), ("track_theta",), ("A_log",)])
def test_gate_parameters_of_any_stride(gpu_lib, monkeypatch, names):
    """Gates computed from transposed views keep their strides."""
    m = _model(use_complex="A_log" not in names)
    x = torch.randn(5, 64, generator=torch.Generator().manual_seed(7)).to(dev)
    cache = _state(m, 5, "full")
    want = _ply(m, x, cache, monkeypatch, True)
    for layer in m.layers:
        for n in names:
            p = getattr(layer["mixer"], n).detach()
            setattr(layer["mixer"], n, nn.Parameter(p.t().contiguous().t()))
        assert not all(t is None or t.is_contiguous() for t in layer["mixer"]._gates(False))
    assert layer_step.usable(m, x)
    assert all(torch.equal(a, b) for a, b in zip(_ply(m, x, cache, monkeypatch, True), want))


def test_gates_of_other_sizes_are_refused_before_the_launch(gpu_lib, monkeypatch):
    """As the separate ops refuse them; another split of the same d_state runs."""
    x = torch.randn(5, 64, device=dev)
    m = _model()
    m.layers[0]["mixer"].track_theta = nn.Parameter(torch.zeros(128, 8, device=dev))
    with pytest.raises(ValueError, match="d_state"):
        _ply(m, x, None, monkeypatch, True)
    m = _model()
    m.layers[0]["mixer"].track_theta = nn.Parameter(torch.zeros(64, 4, device=dev))
    with pytest.raises(ValueError, match="gates"):
        _ply(m, x, None, monkeypatch, True)
    m = _model()
    mx = m.layers[0]["mixer"]
    mx.A_log_mag, mx.A_phase = (nn.Parameter(p.detach()[:, :12].clone())
                                for p in (mx.A_log_mag, mx.A_phase))
    mx.track_theta = nn.Parameter(torch.zeros(128, 8, device=dev))
    new, old = (_ply(m, x, None, monkeypatch, fused) for fused in (True, False))
    assert all(float((a - b).norm() / b.norm()) <= 5e-6 for a, b in zip(new, old))
