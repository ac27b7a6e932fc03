"""The scan backward's general instantiations (64-bit addresses, arrays of any
size) against its FAST ones, bit for bit, over what both accept: every lane
shape, whole and partial channel tiles, both directions, every storage type,
softplus on load, 16-bit gradients and the 16-lane tile walk.

A launch takes the general form when an array spans 4 GiB or more, so u is
given as a view of the same values whose batch rows lie that far apart."""

import pytest
import torch

from tests import hip_capi
from tests.test_gpu_scan import make_case

pytestmark = pytest.mark.gpu
dev = "cuda"
F32, BF16, F16 = torch.float32, torch.bfloat16, torch.float16
# (delta, u, B and C): the types that the FAST form has instantiations for, and a mix
MIXES = {"fp32": (F32, F32, F32), "bf16": (BF16, BF16, BF16), "fp16": (F16, F16, F16),
         "model bf16": (F32, BF16, F32), "mixed": (F16, F32, BF16)}
SPAN = 1 << 32


@pytest.fixture(scope="module")
def store():
    buf = torch.empty(SPAN + (1 << 22), dtype=torch.uint8, device=dev)
    yield buf
    del buf
    torch.cuda.empty_cache()


def _far(t, store):
    """The values of t (B >= 2, L, X) with batch rows SPAN / (B - 1) bytes apart."""
    B, L, X = t.shape
    es = t.element_size()
    sb = -(-SPAN // (B - 1)) // 256 * 256 + 256
    assert sb >= L * X * es and (B - 1) * sb + L * X * es <= store.numel()
    v = store.view(t.dtype).as_strided((B, L, X), (sb // es, X, 1))
    v.copy_(t.to(dev))
    assert ((B - 1) * v.stride(0) + L * X) * es >= SPAN
    return v


def _same(a, b):
    return a.dtype == b.dtype and torch.equal(a.view(torch.uint8), b.view(torch.uint8))


@pytest.mark.parametrize("bidir", [False, True])
@pytest.mark.parametrize("mix,softplus", [(k, False) for k in MIXES] + [("bf16", True)])
@pytest.mark.parametrize("B,L,D,NR,NT", [
    (2, 37, 130, 12, 4),    # 4 lanes, a tile of 64 channels, one whole and a partial one beyond
    (3, 34, 33, 32, 8),     # 8 lanes, one channel past a tile
    (2, 35, 32, 20, 8),     # 8 lanes with pad states
    (2, 33, 23, 64, 8),     # 16 lanes, a partial tile
    (1100, 6, 72, 64, 8),   # 16 lanes, tiles walked 4 to a workgroup, the last one partial
])
def test_general_equals_fast(gpu_lib, monkeypatch, store, B, L, D, NR, NT, mix, softplus, bidir):
    monkeypatch.setattr(hip_capi, "_dev", lambda t: None if t is None else (
        t if t.is_cuda else t.to(dev).contiguous()))
    c = make_case(1500 + D + L, B=B, L=L, D=D, NR=NR, NT=NT)
    if softplus:
        c["delta"] = torch.log(torch.expm1(c["delta"]))
    td, tu, ts = MIXES[mix]
    for k, t in (("delta", td), ("u", tu), ("Bc", ts), ("Cc", ts)):
        c[k] = c[k].to(t)
    far = dict(c, u=_far(c["u"], store))
    for in_storage in (False, True):
        y0, g0 = hip_capi.scan_fwd_bwd(c, bidir, softplus=softplus, grad_in_storage=in_storage)
        y1, g1 = hip_capi.scan_fwd_bwd(far, bidir, softplus=softplus, grad_in_storage=in_storage)
        assert _same(y0, y1)
        for k in g0:
            assert g0[k] is None and g1[k] is None or _same(g0[k], g1[k]), (k, in_storage)
