"""The scan forward's instantiations by storage type and launch size: every
type combination gives the bits of fp32 storage of the same values, for whole
and partial channel tiles, full and short blocks, few and many workgroups, with
and without softplus on load, checkpoints and the final state."""

import pytest
import torch

from redpanda_amd.scan import hip_scan_with_state, hip_trapezoidal_scan
from tests.test_gpu_scan import make_case

pytestmark = pytest.mark.gpu
dev = "cuda"
F32, BF16, F16 = torch.float32, torch.bfloat16, torch.float16
MIXES = {"bf16": (BF16, BF16, BF16), "fp16": (F16, F16, F16), "model bf16": (BF16, BF16, F32),
         "model fp16": (F16, F16, F32), "reference autocast": (F32, BF16, F32),
         "any": (F32, F16, BF16)}
# (B, L, D, NR, NT): 4, 8 and 16 lanes; one channel, whole tiles, one past a
# tile; lengths around the blocks of 32 (16 above 40 states); few workgroups
# and more than the launcher's limit
SHAPES = [(2, 33, 65, 12, 4), (1, 32, 1, 32, 0), (2, 31, 64, 32, 8), (1, 64, 33, 32, 8),
          (2, 35, 17, 64, 8), (1100, 17, 33, 32, 0), (1100, 33, 48, 64, 8)]


def _run(ins, prm, nr, n, bidir, sp):
    with torch.no_grad():
        y = hip_trapezoidal_scan(*ins, *prm, nr, n, bidirectional=bidir, delta_softplus=sp)
    leaves = [t.clone().requires_grad_(True) for t in ins]
    yt = hip_trapezoidal_scan(*leaves, *prm, nr, n, bidirectional=bidir, delta_softplus=sp)
    assert torch.equal(y, yt.detach())  # with and without checkpoints
    return y


@pytest.mark.parametrize("sp", [False, True])
@pytest.mark.parametrize("mix", list(MIXES))
@pytest.mark.parametrize("shape", SHAPES)
def test_storage_types_give_the_fp32_bits(gpu_lib, shape, mix, sp):
    B, L, D, NR, NT = shape
    c = make_case(1300 + D + L, B=B, L=L, D=D, NR=NR, NT=NT)
    td, tu, ts = MIXES[mix]
    if sp:
        c["delta"] = torch.log(torch.expm1(c["delta"]))
    ins = [c[k].to(t).to(dev) for k, t in zip(("delta", "u", "Bc", "Cc"), (td, tu, ts, ts))]
    prm = [None if c[k] is None else c[k].to(dev) for k in ("Ar", "Ai", "Tk")]
    f32 = [t.float() for t in ins]
    for bidir in (False, True):
        want = _run(f32, prm, NR, NR + NT, bidir, sp)
        assert torch.equal(_run(ins, prm, NR, NR + NT, bidir, sp), want), bidir
    with torch.no_grad():
        y0, (h0, b0) = hip_scan_with_state(*f32, *prm, delta_softplus=sp)
        y1, (h1, b1) = hip_scan_with_state(*ins, *prm, delta_softplus=sp)
    assert torch.equal(y0, y1) and torch.equal(h0, h1) and torch.equal(b0, b1)


@pytest.mark.parametrize("D,NR,NT", [(33, 32, 0), (70, 12, 4), (40, 64, 8)])
def test_few_and_many_workgroups_agree(gpu_lib, D, NR, NT):
    """A row alone (the few-workgroups instantiation) and among 1100 rows."""
    c = make_case(1400 + D, B=1100, L=37, D=D, NR=NR, NT=NT)
    ins = [c[k].to(dev) for k in ("delta", "u", "Bc", "Cc")]
    prm = [None if c[k] is None else c[k].to(dev) for k in ("Ar", "Ai", "Tk")]
    with torch.no_grad():
        y, (h, b) = hip_scan_with_state(*ins, *prm)
        for r in (0, 611, 1099):
            yr, (hr, br) = hip_scan_with_state(*(t[r:r + 1] for t in ins), *prm)
            assert torch.equal(yr[0], y[r]) and torch.equal(hr[0], h[r]) and torch.equal(br[0], b[r])
