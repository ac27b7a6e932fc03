"""The inference step's whole-layer call (redpanda_amd/layer_step.py,
rp_layer_step) against the separate ops it replaces and the float64 oracle
block, at the edges of its tiles, in every state form, and the calls that must
not take it."""

import ctypes

import pytest
import torch
import torch.nn as nn

from redpanda_amd import _lib, layer_step
from redpanda_amd.mamba import Mamba, MambaConfig
from redpanda_amd.step import compact_beta

pytestmark = pytest.mark.gpu
dev = "cuda"


def _model(seed=3, n_layer=2, **kw):
    torch.manual_seed(seed)
    cfg = MambaConfig(**{**dict(d_model=64, n_layer=n_layer, vocab_size=64, d_state=20,
                                n_track_state=4, mimo_p=2), **kw})
    m = Mamba(cfg).eval()
    with torch.no_grad():
        for name, p in m.named_parameters():
            if name.endswith("A_phase"):
                p.uniform_(-1.2, 1.2)
            elif "norm" in name:
                p.uniform_(0.5, 1.5)
            elif p.dim() == 2 and "embedding" not in name and "A_" not in name and "track" not in name:
                p.normal_(0, p.shape[1] ** -0.5)
    return m.to(dev)


def _state(m, R, form, seed=5):
    g = torch.Generator(device=dev).manual_seed(seed)
    D, N = m.config.d_inner, m.config.d_state
    rn = lambda *s: torch.randn(*s, generator=g, device=dev)
    if form == "none":
        return None
    if form == "shared":
        return [(rn(1, D, N).expand(R, D, N), rn(1, D, N).expand(R, D, N)) for _ in m.layers]
    if form == "rank1":
        return [(rn(R, D, N), compact_beta(rn(R, D) * 0.1, rn(R, N))) for _ in m.layers]
    return [(rn(R, D, N), rn(R, D, N) * 0.1) for _ in m.layers]


def _ply(m, x, cache, monkeypatch, fused, **kw):
    if not fused:
        monkeypatch.setattr(layer_step, "MAX_ROWS", 0)
    with torch.no_grad():
        y, c = m.step(input_embed=x, cache=cache, **kw)
    monkeypatch.undo()
    return [y, *(t for st in c for t in st)]


def rel(a, b):
    a, b = a.detach().double(), b.detach().double()
    return float((a - b).norm() / b.norm())


@pytest.mark.parametrize("R,form,kw", [
    (1, "none", {}),
    (15, "full", dict(d_model=20, dt_rank=4)),             # K of 20 and 40: a partial slice of 16
    (16, "rank1", dict(d_model=72, mimo_p=1, d_state=7, n_track_state=2, dt_rank=4)),  # N P odd
    (17, "shared", dict(d_model=64, bias=True)),
    (33, "full", dict(use_bcnorm=False, d_state=16, n_track_state=0, use_complex=False)),
    (64, "full", dict(d_model=384, d_state=32, n_track_state=0)),
    (130, "rank1", dict(d_model=512)),
    (256, "full", dict(d_model=512, mimo_p=4)),
])
def test_layer_step_matches_the_separate_ops(gpu_lib, monkeypatch, R, form, kw):
    """Same result as the separate launches: fp32 sums in another order.  A
    dot of K <= 1024 terms differs by about sqrt(K) 2^-24 (2e-6) of its
    terms' norm, twice through a layer's depth."""
    m = _model(**kw)
    x = torch.randn(R, m.config.d_model, generator=torch.Generator().manual_seed(R)).to(dev)
    assert layer_step.usable(m, x)
    cache = _state(m, R, form)
    compact = form == "rank1"
    new = _ply(m, x, cache, monkeypatch, True, compact=compact)
    old = _ply(m, x, cache, monkeypatch, False, compact=compact)
    for a, b in zip(new, old):
        assert a.shape == b.shape and a.dtype == b.dtype
        assert rel(a, b) <= 5e-6
    # into caller buffers, and without the final norm
    bufs = [(torch.empty_like(new[1 + 2 * i]), torch.empty_like(new[2 + 2 * i]))
            for i in range(len(m.layers))]
    again = _ply(m, x, cache, monkeypatch, True, compact=compact, out_cache=bufs)
    assert all(torch.equal(a, b) for a, b in zip(again, new))
    assert again[1] is bufs[0][0]
    raw = _ply(m, x, cache, monkeypatch, True, compact=compact, apply_final_norm=False)
    assert rel(m.norm_f(raw[0]), new[0]) <= 1e-6


def test_layer_step_distance_from_float64(gpu_lib, monkeypatch):
    """No further from float64 than the separate ops (within 1.2x: the sums'
    order only) over a 4-layer ply from a fresh state."""
    from oracle import model_ref
    m = _model(n_layer=4, d_model=256)
    cfg = m.config
    ref = model_ref.Mamba(model_ref.MambaConfig(vocab_size=64, n_layer=4, d_model=256, d_state=20,
                                                n_track_state=4, mimo_p=2)).eval()
    ref.load_state_dict({k: v.cpu() for k, v in m.state_dict().items()})
    x = torch.randn(24, cfg.d_model, generator=torch.Generator().manual_seed(9))
    ref = ref.double()
    for mod in ref.modules():  # the reference keeps its gates in fp32
        if hasattr(mod, "_compute_A"):
            mag = -torch.exp(mod.A_log_mag)
            Ar, Ai, Tk = (mag * torch.cos(mod.A_phase), mag * torch.sin(mod.A_phase),
                          torch.tanh(mod.track_theta))
            mod._compute_A = lambda Ar=Ar, Ai=Ai: (Ar, Ai)
            mod._track_gate = lambda Tk=Tk: Tk
    with torch.no_grad():
        want, _ = ref.step(input_embed=x.double())
    new = _ply(m, x.to(dev), None, monkeypatch, True)
    old = _ply(m, x.to(dev), None, monkeypatch, False)
    e_new, e_old = rel(new[0].cpu(), want), rel(old[0].cpu(), want)
    print(f"layer step vs float64: {e_new:.2e}, separate ops {e_old:.2e}", flush=True)
    assert e_new <= max(1.2 * e_old, 1e-7)


def test_layer_step_rows_are_independent(gpu_lib, monkeypatch):
    """A row's result does not depend on the batch it is in (the same tiles
    of 16 rows, K split the same way)."""
    m = _model(d_model=128)
    x = torch.randn(70, 128, generator=torch.Generator().manual_seed(4)).to(dev)
    cache = _state(m, 70, "full")
    full = _ply(m, x, cache, monkeypatch, True)
    for lo, hi in ((0, 1), (16, 37), (69, 70)):
        part = _ply(m, x[lo:hi], [(h[lo:hi].clone(), b[lo:hi].clone()) for h, b in cache],
                    monkeypatch, True)
        assert all(torch.equal(a, b[lo:hi]) for a, b in zip(part, full))


class _Scaled(nn.Linear):
    def forward(self, x):
        return super().forward(x) * 2


def test_layer_step_is_not_taken_where_it_would_change_the_call(gpu_lib):
    x = torch.randn(4, 64, device=dev)
    assert layer_step.usable(_model(), x)
    m = _model()
    m.layers[1]["mixer"].x_proj.register_forward_hook(lambda mod, i, o: o)
    assert not layer_step.usable(m, x)
    m = _model()
    lin = m.layers[0]["mixer"].in_proj
    new = _Scaled(lin.in_features, lin.out_features, bias=False).to(dev)
    m.layers[0]["mixer"].in_proj = new
    assert not layer_step.usable(m, x)
    assert not layer_step.usable(_model().half(), x)
    m = _model()
    w = m.layers[0]["mixer"].out_proj.weight
    store = torch.empty(w.numel() + 1, device=dev)
    m.layers[0]["mixer"].out_proj.weight = nn.Parameter(store[1:].view_as(w))  # off 16 bytes
    assert not layer_step.usable(m, x)
    m = _model()
    m.layers[0]["mixer"].dt_proj.weight = nn.Parameter(
        torch.empty(4, 128, device=dev).t())  # a transposed view
    assert not layer_step.usable(m, x)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert not layer_step.usable(_model(), x)
    assert not layer_step.usable(_model(), torch.randn(layer_step.MAX_ROWS + 1, 64, device=dev))
    with pytest.raises(ValueError):
        with torch.no_grad():
            m = _model()
            m.step(input_embed=x, cache=[(torch.zeros(4, 8, 8, device=dev),) * 2] * 2)


def test_layer_step_check_refuses(gpu_lib):
    lib = _lib.load()
    m = _model()
    a = _lib.LayerStepArgs()
    a.R, a.d_model, a.D, a.N, a.NR, a.NT, a.P, a.dt_rank = 4, 64, 128, 20, 16, 4, 2, 4
    assert lib.rp_layer_step_work_bytes(ctypes.byref(a)) > 0
    assert lib.rp_layer_step_check(ctypes.byref(a)) < 0  # NULL operands
    assert lib.rp_layer_step(ctypes.byref(a), None) < 0
    a.d_model = 66
    assert lib.rp_layer_step_work_bytes(ctypes.byref(a)) < 0
    a.d_model, a.P = 64, 9  # BCNorm's own limit, refused before any launch
    t = torch.zeros(1 << 16, device=dev)
    for k, _ in _lib.LayerStepArgs._fields_[8:]:
        if k in ("x", "norm_w", "in_w", "xp_w", "dtp_w", "out_w", "A_real", "A_imag", "track",
                 "Dskip", "work"):
            setattr(a, k, t.data_ptr())
    a.x_sr = 64
    o = torch.zeros(3, 1 << 16, device=dev)
    a.h_out, a.beta_out, a.x_out = (o[i].data_ptr() for i in range(3))
    a.work_bytes = lib.rp_layer_step_work_bytes(ctypes.byref(a))
    w = torch.empty(a.work_bytes, dtype=torch.uint8, device=dev)
    a.work = w.data_ptr()
    assert lib.rp_layer_step(ctypes.byref(a), None) < 0
    assert b"P <= 8" in lib.rp_last_error()
    a.P, a.work_bytes = 2, 256
    assert lib.rp_layer_step(ctypes.byref(a), None) < 0
    assert m is not None
