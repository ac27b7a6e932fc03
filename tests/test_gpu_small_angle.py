"""The sine in the scan backward: the A_imag gradient of a scan whose terms all
have one sign, so that an error the sine repeats at every step is not averaged
away, against float64, by bands of the rotation angle dt A_imag."""

import pytest
import torch

from oracle import scan_ref
from redpanda_amd.scan import hip_trapezoidal_scan

pytestmark = pytest.mark.gpu
dev = "cuda"


@pytest.mark.parametrize("NR,NT", [(16, 4), (32, 8), (64, 8)])
@pytest.mark.parametrize("lo,hi", [(1e-4, 5e-4), (5e-4, 1e-3), (1e-3, 1.5e-3), (1.5e-3, 3e-3),
                                   (3e-3, 1e-2), (1e-2, 0.1), (0.1, 0.3)])
def test_sine_is_unbiased_at_every_angle(gpu_lib, lo, hi, NR, NT):
    """Over 256 channels x NR states the mean relative error of d A_imag is
    below 1e-7.  What repeats from state to state is the rounding of the
    constants: the step 2 pi / 256 (2.8e-8 relative) and its reciprocal (at
    most 6e-8); the other roundings are independent between states and leave
    about 2^-23 / sqrt(256 NR) = 2e-9 of their own.  A sine that drops its cubic
    term within steps of 2 pi / 2048 is off by 2.4e-7 around 1.2e-3."""
    gen = torch.Generator().manual_seed(int(lo * 1e6) + NR)
    rnd = lambda *s: torch.rand(*s, generator=gen)
    B, L, D, N = 1, 8, 256, NR + NT
    dt = (0.01 + 0.01 * rnd(1, 1, D)).expand(B, L, D).contiguous()
    ang = torch.exp(torch.log(torch.tensor(lo)) + rnd(D, NR) * torch.log(torch.tensor(hi / lo)))
    Ai = ang / dt[0, 0, :, None]
    Ar = -(0.5 + rnd(D, NR))
    Tk = 0.9 * rnd(D, NT)
    # all positive (angles up to 8 x 0.3 / 2 keep the signs): every term of
    # d A_imag is negative
    u, Bc, Cc, dy = (0.5 + rnd(B, L, k) for k in (D, N, N, D))
    leaves = [t.to(dev) for t in (dt, u, Bc, Cc, Ar)] + [Ai.to(dev).requires_grad_(True), Tk.to(dev)]
    y = hip_trapezoidal_scan(*leaves, NR, N)
    got, = torch.autograd.grad(y, leaves[5], dy.to(dev))
    Ai64 = Ai.double().requires_grad_(True)
    y64 = scan_ref.scan_sequential(*(t.double() for t in (dt, u, Bc, Cc, Ar)), Ai64, Tk.double())[0]
    want, = torch.autograd.grad(y64, Ai64, dy.double())
    assert (want < 0).all()
    err = (got.double().cpu() - want) / want
    mean, rms = float(err.mean()), float(err.square().mean().sqrt())
    print(f"d A_imag at {lo:g}-{hi:g} rad, {NR}+{NT}: mean {mean:+.2e}, rms {rms:.2e}", flush=True)
    assert abs(mean) <= 1e-7
