"""The scan backward across storage types: the same values stored in 16 bits,
at odd element offsets and row strides, give the bits that fp32 storage gives
(every load converts exactly), in each of the backward's type instantiations
(all fp32, all bf16, the model's mix, any other mix) and lane shapes, with
whole and partial channel tiles and last chunks of every length."""

import pytest
import torch

from redpanda_amd.scan import hip_trapezoidal_scan
from tests.test_gpu_scan import make_case

pytestmark = pytest.mark.gpu
dev = "cuda"
F32, BF16, F16 = torch.float32, torch.bfloat16, torch.float16
MIXES = {"bf16": (BF16, BF16, BF16, BF16), "fp16": (F16, F16, F16, F16),
         "model bf16": (F32, BF16, F32, F32), "model fp16": (F32, F16, F32, F32),
         "f32 u": (BF16, F32, F16, BF16), "mixed": (F16, BF16, BF16, F32)}
# (B, L, D, NR, NT): 4 lanes partial tile; 8 lanes one channel, whole tiles and
# one past; 16 lanes; 16 lanes with a tile walk (whole and partial tiles)
SHAPES = [(2, 4, 65, 12, 4), (1, 1, 1, 32, 8), (2, 5, 32, 32, 8), (2, 11, 33, 32, 0),
          (1, 7, 17, 64, 8), (1100, 6, 72, 64, 8)]


def _odd(t):
    """The values of t as a view at an odd offset with an odd row stride."""
    X = t.shape[-1]
    row = X + 2 + X % 2 + 1  # odd for every X
    big = torch.zeros(*t.shape[:-1], row, dtype=t.dtype, device=dev)
    big[..., 1:1 + X] = t.to(dev)
    return big[..., 1:1 + X]


def _run(ins, prm, nr, n, dy, bidir):
    leaves = [t.detach().requires_grad_(True) for t in ins] + [
        None if t is None else t.to(dev).requires_grad_(True) for t in prm]
    y = hip_trapezoidal_scan(*leaves, nr, n, bidirectional=bidir)
    need = [t for t in leaves if t is not None]
    return y.detach(), torch.autograd.grad(y, need, dy.to(dev))


@pytest.mark.parametrize("bidir", [False, True])
@pytest.mark.parametrize("mix", list(MIXES))
@pytest.mark.parametrize("shape", SHAPES)
def test_storage_types_give_the_fp32_bits(gpu_lib, shape, mix, bidir):
    B, L, D, NR, NT = shape
    c = make_case(1200 + D + L, B=B, L=L, D=D, NR=NR, NT=NT)
    types = MIXES[mix]
    ins = [c[k].to(t) for k, t in zip(("delta", "u", "Bc", "Cc"), types)]
    prm = [c[k] for k in ("Ar", "Ai", "Tk")]
    y0, g0 = _run([t.float().to(dev) for t in ins], prm, NR, NR + NT, c["dy"], bidir)
    y1, g1 = _run([_odd(t) for t in ins], prm, NR, NR + NT, c["dy"], bidir)
    assert torch.equal(y0, y1)
    for k, (a, b) in enumerate(zip(g0, g1)):
        want = a.to(types[k]) if k < 4 else a
        assert b.dtype == want.dtype and torch.equal(b, want), k
