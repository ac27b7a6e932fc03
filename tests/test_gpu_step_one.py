"""The step tile kernel's one-rollout instantiation and its vector loads of the
gate parameters, bit for bit against a length-1 scan from the same state (the
lane-layout arithmetic): every lane shape, gate kind and beta form, at one and
several rollouts per workgroup, whole and partial channel tiles, and gate rows
that are no multiple of 16 bytes or not 16-byte aligned (the scalar loads)."""

import pytest
import torch

from redpanda_amd.scan import hip_scan_with_state
from redpanda_amd.step import compact_beta, full_beta, hip_step
from tests.test_gpu_step import make_step_case

pytestmark = pytest.mark.gpu
dev = "cuda"


def _shift(t, by):
    """The same values `by` floats past a 16-byte boundary."""
    if t is None:
        return None
    store = torch.empty(t.numel() + 4, device=dev)
    v = store[by:by + t.numel()].view_as(t)
    v.copy_(t)
    return v


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("form", ["full", "rank1", "none"])
@pytest.mark.parametrize("R,D,NR,NT", [
    (1, 256, 16, 4), (7, 100, 12, 8), (3, 192, 32, 0), (5, 70, 32, 8), (2, 128, 20, 8),
    (4, 96, 64, 0), (3, 64, 64, 8), (2, 32, 112, 16), (3, 80, 88, 4), (4, 128, 14, 6),
    (900, 256, 16, 4), (700, 256, 64, 0), (600, 128, 30, 6),
])
def test_step_matches_scan_bitwise(gpu_lib, R, D, NR, NT, form, shift):
    c = {k: (v.to(dev) if torch.is_tensor(v) else v)
         for k, v in make_step_case(31 * R + NR, R=R, D=D, NR=NR, NT=NT).items()}
    x = torch.log(torch.expm1(c["delta"]))
    prm = [_shift(c[k], shift) for k in ("Ar", "Ai", "Tk")]
    N = NR + NT
    if form == "rank1":
        bp = compact_beta(c["u"] * 0.1, c["Cc"])
        step_state, scan_state = (c["h"], bp), (c["h"], full_beta(bp, D))
    elif form == "full":
        step_state = scan_state = (c["h"], c["beta"])
    else:
        step_state = scan_state = None
    with torch.no_grad():
        y, (h, b) = hip_step(x, c["u"], c["Bc"], c["Cc"], *prm, torch.zeros(D, device=dev),
                             step_state, delta_softplus=True)
        ys, (hs, bs) = hip_scan_with_state(x[:, None], c["u"][:, None], c["Bc"][:, None],
                                           c["Cc"][:, None], c["Ar"], c["Ai"], c["Tk"],
                                           state=scan_state, delta_softplus=True)
    if form == "rank1":
        assert b.shape == (R, D + N)
        b = full_beta(b, D)
    assert torch.equal(y, ys[:, 0]) and torch.equal(h, hs) and torch.equal(b, bs)
