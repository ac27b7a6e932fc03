"""One Mamba-3 layer of the inference step as a single library call.

`hip_layer_step` is the body of Mamba.step's pre-norm loop for one layer
(engine/mamba.py:592-597 around Mamba3Block.step, :440-498): x + out_proj of
the gated step of norm(x), with the norm, SiLU and residual add folded into
small-batch fp32 projections (rp_layer_step: five launches, six where BCNorm does
not fit the step's prologue, where the separate ops take seven and eight, and one
call from Python where they take eight).  Inference only.
"""

import ctypes

import torch
import torch.nn as nn
from torch.nn.modules import module as _nn_module

from redpanda_amd import _lib, mamba
from redpanda_amd.step import _f32c, _state_pair

# The most rows that take this path, by width (d_model, at expand 2).  A
# projection's workgroup here reads all of its x rows for 16 columns of W, which
# costs more than its launch saves once rows and width grow; the library's GEMMs
# share both in larger tiles.  Microseconds per layer of a replayed ply, this path / the separate ops
# (eager: the larger of this and the host's 48 / 150):
#   d_model  256   64 rows 25 / 74,  256 35 / 200,  512 56 / 63
#   d_model  512   64 34 / 51,  256 64 / 67,  384 87 / 78
#   d_model  640   128 65 / 66,  144 65 / 63,  256 93 / 81
#   d_model  768   64 47 / 53,  128 72 / 72,  144 79 / 68,  256 105 / 88
#   d_model 1024   64 53 / 63,  128 82 / 85,  144 104 / 88,  256 130 / 105
#   d_model 1280   48 73 / 75,  64 93 / 89
#   d_model 1536   32 76 / 87,  48 99 / 96,  128 151 / 125
#   d_model 2048   32 100 / 108,  48 119 / 118,  128 209 / 159,  256 374 / 239
# (Replayed and eager plies take the same path, so that they give the same bits.)
MAX_ROWS = 256


def max_rows(width):
    if width <= 512:
        return MAX_ROWS
    return MAX_ROWS // 2 if width <= 1024 else min(MAX_ROWS // 2, (1 << 16) // width)


_LINEAR_FORWARD = nn.Linear.forward
_PLAIN = (nn.Parameter, torch.Tensor)  # a tensor subclass computes its own product


def _plain_linear(m, out_features, in_features):
    """The (tensor, shape) pairs of a Linear of this shape that computes just
    that, or None: no subclass, parametrization, hook or forward of its own
    (offloading and quantising wrappers set one on the instance) that a direct
    use of its weight would pass by."""
    if (type(m) is not nn.Linear or m._forward_hooks or m._forward_pre_hooks or
            "forward" in m.__dict__):
        return None
    # (the dictionaries, not the attributes: this runs for every layer of a ply)
    ps = m._parameters
    pairs = [(ps.get("weight"), (out_features, in_features))]
    if ps.get("bias") is not None:
        pairs.append((ps["bias"], (out_features,)))
    return pairs


# what hip_layer_step does in Mamba3Block's place
_BLOCK_METHODS = frozenset(("step", "_ssm_proj_raw"))


def _layer_tensors(layer, d):
    """The (tensor, shape) pairs that hip_layer_step reads of a layer on rows of
    d floats, or None where the separate ops must run."""
    mx, norm = layer["mixer"], layer["norm"]
    # a block whose step is not Mamba3Block's own has to run it
    if type(mx) is not mamba.Mamba3Block or not _BLOCK_METHODS.isdisjoint(mx.__dict__):
        return None
    cfg = mx.config
    D, r, np2 = cfg.d_inner, cfg.dt_rank, 2 * cfg.d_state * cfg.mimo_p
    if cfg.d_model != d or d % 4 or D % 4 or r % 4 or cfg.mimo_p > 8:
        return None
    mods = mx._modules
    pairs = [(norm._parameters.get("weight"), (d,)), (mx._parameters.get("D"), (D,))]
    for name, n_out, n_in in (("in_proj", 2 * D, d), ("x_proj", r + np2, D), ("dt_proj", D, r),
                              ("out_proj", d, D)):
        lin = _plain_linear(mods.get(name), n_out, n_in)
        if lin is None:
            return None
        pairs += lin
    if cfg.use_bcnorm:
        for name in ("b_norm", "c_norm"):
            pairs.append((mods[name]._parameters.get("weight"), (np2 // 2,)))
    return pairs


def usable(model, x):
    """Whether Mamba.step's inference loop may take hip_layer_step for the
    rows x (R, d_model) fp32: a small batch for the width, plain fp32 projections, and every
    tensor of the configured shape, on x's device, contiguous and 16-byte
    aligned (the kernels read them by these shapes; where one differs, the
    separate ops refuse or convert it)."""
    R, d = x.shape
    if (not 0 < R <= max_rows(max(d, model.config.d_inner // 2)) or
            torch.is_autocast_enabled("cuda")):
        return False
    if _nn_module._global_forward_hooks or _nn_module._global_forward_pre_hooks:
        return False
    if nn.Linear.forward is not _LINEAR_FORWARD or mamba.Mamba3Block.step is not mamba._BLOCK_STEP:
        return False  # replaced for every instance
    dev = x.device
    bits = 0
    for layer in model.layers:
        pairs = _layer_tensors(layer, d)
        if pairs is None:
            return False
        for w, shape in pairs:
            if (type(w) not in _PLAIN or w.shape != shape or w.dtype is not torch.float32 or
                    w.device != dev or not w.is_contiguous()):
                return False
            bits |= w.data_ptr()
    return not bits & 15


def _vector_rows(x):
    """(tensor, row stride): the rows of x (R, d) where the kernels can read
    them as 16-byte vectors, x itself or a copy.  (contiguous() would return a
    misaligned x, or one row of another stride, as it is.)  A stride shorter
    than a row is left to the library, which refuses it."""
    R, d = x.shape
    if x.stride(-1) != 1:
        x = x.contiguous()
    sr = x.stride(0)
    if sr >= d:
        if R == 1:
            sr = d
        if sr % 4 or x.data_ptr() & 15:
            x, sr = torch.empty((R, d), dtype=x.dtype, device=x.device).copy_(x), d
    return x, sr


def _gate_rows(gates, D, N):
    """(A_real, A_imag, track) as fp32 rows of the D channels: the parameters
    they come from may be views of any stride, which the gates keep."""
    Ar, Ai, Tk = (None if t is None else _f32c(t) for t in gates)
    NR = 0 if Ar is None else Ar.shape[-1]
    NT = 0 if Tk is None else Tk.shape[-1]
    if NR + NT != N:
        raise ValueError(f"step: n_rot ({NR}) + n_track ({NT}) != d_state ({N})")
    for t, n in ((Ar, NR), (Ai, NR), (Tk, NT)):
        if t is not None and t.shape != (D, n):
            raise ValueError(f"step: gates {tuple(t.shape)} must be {(D, n)}")
    return Ar, Ai, Tk


def hip_layer_step(x, layer, state, compact=False, out=None):
    """(x + layer(x), (h, beta)) for rows x (R, d_model) fp32 that `usable`
    accepted; state, compact and out as in Mamba3Block.step."""
    lib = _lib.load()
    mx = layer["mixer"]
    cfg = mx.config
    R, D, N = x.shape[0], cfg.d_inner, cfg.d_state
    dev = x.device
    x, x_sr = _vector_rows(x)
    Ar, Ai, Tk = _gate_rows(mx._gates(False), D, N)
    a = _lib.LayerStepArgs()
    a.R, a.d_model, a.D, a.N, a.P, a.dt_rank = R, cfg.d_model, D, N, cfg.mimo_p, cfg.dt_rank
    a.NR = 0 if Ar is None else Ar.shape[1]
    a.NT = 0 if Tk is None else Tk.shape[1]
    h_in = beta_in = None
    rank1 = bool(compact)
    if state is not None:
        h_in, beta_in, broadcast, rank1 = _state_pair(state[0], state[1], R, D, N)
        a.h_in, a.beta_in, a.broadcast_state = h_in.data_ptr(), beta_in.data_ptr(), broadcast
    bshape = (R, D + N) if rank1 else (R, D, N)
    f32 = dict(dtype=torch.float32, device=dev)
    if out is None:
        h_out, beta_out = torch.empty((R, D, N), **f32), torch.empty(bshape, **f32)
    else:
        h_out, beta_out = out
        for name, t, shp in (("h", h_out, (R, D, N)), ("beta", beta_out, bshape)):
            if (t.shape != shp or t.dtype != torch.float32 or t.device != dev or
                    not t.is_contiguous()):
                raise ValueError(f"step: out {name} must be a contiguous fp32 {shp} tensor on {dev}")
    x_out = torch.empty((R, cfg.d_model), **f32)
    norm = layer["norm"]
    a.x, a.x_sr, a.norm_w, a.norm_eps = x.data_ptr(), x_sr, norm.weight.data_ptr(), norm.eps
    for pre, lin in (("in", mx.in_proj), ("xp", mx.x_proj), ("dtp", mx.dt_proj), ("out", mx.out_proj)):
        setattr(a, pre + "_w", lin.weight.data_ptr())
        if lin.bias is not None:
            setattr(a, pre + "_b", lin.bias.data_ptr())
    if cfg.use_bcnorm:
        a.bn_wB, a.bn_wC, a.bn_eps = (mx.b_norm.weight.data_ptr(), mx.c_norm.weight.data_ptr(),
                                      mx.b_norm.eps)
    a.A_real, a.A_imag, a.track = _lib.ptr(Ar), _lib.ptr(Ai), _lib.ptr(Tk)
    a.Dskip = mx.D.data_ptr()
    a.h_out, a.beta_out, a.x_out = h_out.data_ptr(), beta_out.data_ptr(), x_out.data_ptr()
    a.beta_rank1 = 1 if rank1 else 0
    nbytes = lib.rp_layer_step_work_bytes(ctypes.byref(a))
    _lib.check(0 if nbytes >= 0 else -1, lib)
    work = torch.empty(nbytes, dtype=torch.uint8, device=dev)
    a.work, a.work_bytes = work.data_ptr(), nbytes
    _lib.check(lib.rp_layer_step(ctypes.byref(a), _lib.stream_of(dev)), lib)
    return x_out, (h_out, beta_out)
