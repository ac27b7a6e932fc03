"""hip_step refuses parameters that hold other than the values it reads,
before any launch."""

import pytest
import torch

from redpanda_amd.step import hip_step

pytestmark = pytest.mark.gpu
dev = "cuda"


def _z(*s):
    return torch.zeros(*s, device=dev)


@pytest.mark.parametrize("which,shape", [("Ar", (31, 12)), ("Ai", (32, 8)), ("Tk", (1, 4)),
                                         ("D", (1,)), ("wB", (1,)), ("wC", (16,))])
def test_parameters_of_other_sizes_are_refused(gpu_lib, which, shape):
    R, D, N, P = 3, 32, 16, 2
    t = dict(Ar=_z(D, 12), Ai=_z(D, 12), Tk=_z(D, 4), D=_z(D), wB=_z(N * P), wC=_z(N * P))
    t[which] = _z(*shape)
    with torch.no_grad(), pytest.raises(ValueError, match="must"):
        hip_step(_z(R, D), _z(R, D), None, None, t["Ar"], t["Ai"], t["Tk"], t["D"],
                 bcnorm=(_z(R, N * P), _z(R, N * P), t["wB"], t["wC"], P, 1e-5, True))
    if which in ("Ar", "Ai", "Tk", "D"):
        with torch.no_grad(), pytest.raises(ValueError, match="must"):
            hip_step(_z(R, D), _z(R, D), _z(R, N), _z(R, N), t["Ar"], t["Ai"], t["Tk"], t["D"])
