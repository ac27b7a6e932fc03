"""The workloads whose speed this framework answers for.

Each case is one call, or one training step, that a program makes through the
public entry points: the selective scan and its gradients, the scan that primes
a search cache, the batched O(1) step, a whole search ply, a rollout replayed
from HIP graphs, and a Mamba layer trained forward and backward.  Sizes are the
repository's own configurations (the model defaults, tests/test_gpu_configs.py,
bench.py) and odd ones between them.  `draw` gives more cases of the same kinds
over the whole ranges.

`exact` restates each path in float64 plain torch, without this package.
"""

import math

import torch
import torch.nn.functional as F

DEV = "cuda:0"
DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}

# Flops of one (token, direction, channel, state) update: the gate (an exp, a
# cos or sin), hb, h and y forward; the gate with its sine, the adjoint and the
# gradient terms backward.
SCAN_FWD_FLOPS = 12
SCAN_BWD_FLOPS = 30


# ---------------------------------------------------------------- the cases

def listed():
    return [
        # The reference's own CPU configuration: one causal real-decay layer in
        # fp32, forward and backward.  Latency and launches are all of it.
        dict(name="scan_small_train", kind="scan", B=8, L=64, D=256, NR=16, NT=0, imag=False,
             bi=False, dtype="fp32", train=True),
        # A training step of the evaluation model's scan: 256 boards of 64
        # tokens, both directions, inputs stored in bf16 (bench.py's headline).
        dict(name="scan_eval_train", kind="scan", B=256, L=64, D=1536, NR=32, NT=8, imag=True,
             bi=True, dtype="bf16", train=True),
        # Scoring a ragged batch of positions with the evaluation model's scan:
        # forward only, odd batch and length, fp16.
        dict(name="scan_eval_infer", kind="scan", B=75, L=69, D=1536, NR=32, NT=8, imag=True,
             bi=True, dtype="fp16", train=False),
        # Long games: one causal layer over 2048 tokens with 72 states, fp32,
        # forward and backward.  The largest case.
        dict(name="scan_long_train", kind="scan", B=64, L=2048, D=1024, NR=64, NT=8, imag=True,
             bi=False, dtype="fp32", train=True),
        # Training the search model on middling sequences: one causal scan at
        # its default state size with a channel count that is no multiple of a
        # tile, fp32.
        dict(name="scan_mid_train", kind="scan", B=12, L=250, D=1000, NR=32, NT=0, imag=True,
             bi=False, dtype="fp32", train=True),
        # Priming a search cache: one board through one causal layer, forward
        # only, the final state kept (the search model's default width).
        dict(name="scan_prime_board", kind="prime", B=1, L=67, D=768, NR=32, NT=0),
        # The batched step that advances 4096 rollouts by one token, gated, full
        # beta (bench.py's step).
        dict(name="step_4096", kind="step", R=4096, D=1024, NR=16, NT=4, form="full"),
        # The same for an odd number of rollouts at the search model's default
        # width with the compact (rank-1) cache.
        dict(name="step_rank1_777", kind="step", R=777, D=768, NR=32, NT=0, form="rank1"),
        # One eager ply of a whole search model for the rows of one simulation
        # budget, with the continuation head's logits.
        dict(name="ply_search_64", kind="ply", R=64, d_model=384, n_layer=12, d_state=32,
             n_track=0, p=2),
        # A rollout of 8 plies replayed from HIP graphs at a small batch
        # (bench.py's search backbone: 8 layers, 16 + 4 states).
        dict(name="rollout_graph_12", kind="graph", R=12, d_model=512, n_layer=8, d_state=20,
             n_track=4, p=2, plies=8),
        # Training the evaluation model's layer under bf16 autocast: output,
        # input gradient and every parameter gradient.
        dict(name="layer_eval_train", kind="layer", B=256, L=64, d_model=768, d_state=40, n_track=8,
             p=4, bi=True, amp="bf16"),
        # Training one causal search-model layer on a small odd batch in fp32.
        dict(name="layer_small_train", kind="layer", B=9, L=71, d_model=384, d_state=32, n_track=0,
             p=2, bi=False, amp="fp32"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _states(rng):
    n = rng.choice([16, 20, 24, 32, 36, 40, 64, 72])
    nt = rng.choice([0, 4, 8])
    return n - nt, nt


def draw(rng):
    kind = rng.choice(["scan", "scan", "scan", "prime", "step", "step", "ply", "graph", "layer",
                       "layer"])
    if kind == "scan":
        nr, nt = _states(rng)
        L = _log(rng, 20, 1200)
        D = rng.choice([256, 384, 512, 768, 1000, 1024, 1500, 1536])
        B = max(1, min(256, int(_log(rng, 2e5, 4e7) / (L * D))))
        imag = rng.random() < 0.85
        return dict(kind=kind, B=B, L=L, D=D, NR=nr, NT=nt, imag=imag, bi=rng.random() < 0.5,
                    dtype=rng.choice(["fp32", "bf16", "fp16"]), train=rng.random() < 0.7)
    if kind == "prime":
        nr, nt = _states(rng)
        return dict(kind=kind, B=rng.choice([1, 1, 2, 5, 16]), L=_log(rng, 20, 300),
                    D=rng.choice([512, 768, 1000, 1024]), NR=nr, NT=nt)
    if kind == "step":
        nr, nt = _states(rng)
        return dict(kind=kind, R=_log(rng, 1, 4096), D=rng.choice([512, 768, 1000, 1024]), NR=nr,
                    NT=nt, form=rng.choice(["full", "rank1", "shared"]))
    if kind == "ply":
        return dict(kind=kind, R=_log(rng, 1, 1024), d_model=rng.choice([256, 384, 512]),
                    n_layer=rng.choice([2, 4, 8]), d_state=rng.choice([16, 20, 32]), n_track=4,
                    p=rng.choice([1, 2, 4]))
    if kind == "graph":
        return dict(kind=kind, R=_log(rng, 1, 512), d_model=rng.choice([256, 384, 512]),
                    n_layer=rng.choice([2, 4, 8]), d_state=rng.choice([16, 20, 32]), n_track=4,
                    p=rng.choice([1, 2]), plies=rng.randint(2, 8))
    d_state, n_track = rng.choice([(16, 4), (20, 4), (32, 0), (40, 8), (64, 8)])
    return dict(kind="layer", B=_log(rng, 2, 128), L=_log(rng, 20, 100),
                d_model=rng.choice([256, 384, 512, 768]), d_state=d_state, n_track=n_track,
                p=rng.choice([2, 4]), bi=rng.random() < 0.5,
                amp=rng.choice(["fp32", "bf16", "fp16"]))


# ---------------------------------------------------------------- inputs

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) & 0x7FFFFFFF)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV)


def _gates(g, D, NR, NT, imag=True):
    Ar = Ai = Tk = None
    if NR:
        Ar = -torch.exp(torch.rand(D, NR, generator=g, device=DEV) * 3.0)
        if imag:
            Ai = (torch.rand(D, NR, generator=g, device=DEV) * 2 - 1) * math.pi
    if NT:
        Tk = torch.tanh(_randn(g, D, NT) * 1.5)
    return Ar, Ai, Tk


def _scan_inputs(case, seed):
    g = _gen(seed)
    B, L, D, NR, NT = (case[k] for k in ("B", "L", "D", "NR", "NT"))
    dt = DTYPES[case["dtype"]]
    s = dict(delta=F.softplus(_randn(g, B, L, D) * 0.5 - 2.0).to(dt), u=_randn(g, B, L, D).to(dt),
             Bc=_randn(g, B, L, NR + NT).to(dt), Cc=_randn(g, B, L, NR + NT).to(dt))
    s["Ar"], s["Ai"], s["Tk"] = _gates(g, D, NR, NT, case["imag"])
    if case["train"]:
        s["dy"] = _randn(g, B, L, D)
    return s


def _prime_inputs(case, seed):
    g = _gen(seed)
    B, L, D, NR, NT = (case[k] for k in ("B", "L", "D", "NR", "NT"))
    s = dict(x=_randn(g, B, L, D) * 0.5 - 2.0, u=_randn(g, B, L, D), Bc=_randn(g, B, L, NR + NT),
             Cc=_randn(g, B, L, NR + NT))
    s["Ar"], s["Ai"], s["Tk"] = _gates(g, D, NR, NT)
    return s


def _step_inputs(case, seed):
    g = _gen(seed)
    R, D, NR, NT = (case[k] for k in ("R", "D", "NR", "NT"))
    N = NR + NT
    s = dict(x=_randn(g, R, D) * 0.5 - 2.0, u=_randn(g, R, D), Bc=_randn(g, R, N),
             Cc=_randn(g, R, N), z=_randn(g, R, D), Dk=1.0 + 0.2 * _randn(g, D))
    s["Ar"], s["Ai"], s["Tk"] = _gates(g, D, NR, NT)
    rows = 1 if case["form"] == "shared" else R
    s["h"] = _randn(g, rows, D, N)
    if case["form"] == "rank1":
        s["beta"] = torch.cat([0.13 * _randn(g, R, D), _randn(g, R, N)], dim=-1)
    else:
        s["beta"] = 0.13 * _randn(g, rows, D, N)
    if case["form"] == "shared":
        s["h"], s["beta"] = s["h"].expand(R, D, N), s["beta"].expand(R, D, N)
    return s


def _settle(module, g):
    """Weights as a trained model has them: rotational phases and norm weights
    off their initial constants, the projections at their fan-in scale."""
    for name, p in module.named_parameters():
        leaf = name.rsplit(".", 1)[-1]
        with torch.no_grad():
            if leaf == "A_phase":
                p.copy_((_randn(g, *p.shape) * 0.5).clamp(-1.4, 1.4))
            elif leaf == "weight" and p.dim() == 2 and "embedding" not in name:
                p.copy_(_randn(g, *p.shape) / math.sqrt(p.shape[1]))
            elif leaf == "weight" and p.dim() == 2:
                p.copy_(_randn(g, *p.shape))
            elif leaf == "weight":
                p.copy_(1.0 + 0.1 * _randn(g, *p.shape))
            elif leaf == "track_theta":
                p.add_(0.1 * _randn(g, *p.shape))


def _config(case, bi=False):
    from redpanda_amd.mamba import MambaConfig
    return MambaConfig(d_model=case["d_model"], n_layer=case.get("n_layer", 1), vocab_size=8192,
                       d_state=case["d_state"], n_track_state=case["n_track"], mimo_p=case["p"],
                       bidirectional=bi)


def _model(case, seed):
    from redpanda_amd.mamba import Mamba
    torch.manual_seed(seed)
    with torch.device(DEV):
        m = Mamba(_config(case)).eval()
    g = _gen(seed)
    _settle(m, g)
    head = _randn(g, 8192, case["d_model"]) / math.sqrt(case["d_model"])
    return m, head, g


def _cache(case, g):
    D, N, R = 2 * case["d_model"], case["d_state"], case["R"]
    return [(_randn(g, R, D, N) * 0.3, _randn(g, R, D, N) * 0.03) for _ in range(case["n_layer"])]


def prepare(case, seed):
    kind = case["kind"]
    if kind == "scan":
        s = _scan_inputs(case, seed)
        if case["train"]:
            s["leaves"] = [s[k].requires_grad_(True) for k in ("delta", "u", "Bc", "Cc", "Ar", "Ai", "Tk")
                           if s[k] is not None]
    elif kind == "prime":
        s = _prime_inputs(case, seed)
    elif kind == "step":
        s = _step_inputs(case, seed)
    elif kind == "ply":
        m, head, g = _model(case, seed)
        s = dict(model=m, head=head, cache=_cache(case, g),
                 tok=torch.randint(0, 8192, (case["R"],), generator=g, device=DEV))
    elif kind == "graph":
        from redpanda_amd.step_graph import StepGraph
        m, head, g = _model(case, seed)
        cache = _cache(case, g)
        toks = torch.randint(0, 8192, (case["plies"], case["R"]), generator=g, device=DEV)
        s = dict(model=m, head=head, cache=cache, tok=toks, graph=StepGraph(m, case["R"]))
    else:
        from redpanda_amd.mamba import Mamba3Block
        torch.manual_seed(seed)
        g = _gen(seed)
        with torch.device(DEV):
            blk = Mamba3Block(_config(case, case["bi"]))
        _settle(blk, g)
        x = _randn(g, case["B"], case["L"], case["d_model"]).requires_grad_(True)
        s = dict(block=blk, x=x, dout=_randn(g, *x.shape), leaves=[x, *blk.parameters()])
    s["case"] = case
    return s


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "scan":
        from redpanda_amd.scan import triton_trapezoidal_scan
        n, nr = case["NR"] + case["NT"], case["NR"]
        args = [state[k] for k in ("delta", "u", "Bc", "Cc", "Ar", "Ai", "Tk")]
        if not case["train"]:
            with torch.no_grad():
                return triton_trapezoidal_scan(*args, nr, n, bidirectional=case["bi"])
        y = triton_trapezoidal_scan(*args, nr, n, bidirectional=case["bi"])
        return [y.detach(), *torch.autograd.grad(y, state["leaves"], state["dy"])]
    if kind == "prime":
        from redpanda_amd.scan import hip_scan_with_state
        with torch.no_grad():
            y, (h, beta) = hip_scan_with_state(
                *(state[k] for k in ("x", "u", "Bc", "Cc", "Ar", "Ai", "Tk")), delta_softplus=True)
        return [y, h, beta]
    if kind == "step":
        from redpanda_amd.step import hip_step
        y, (h, beta) = hip_step(*(state[k] for k in ("x", "u", "Bc", "Cc", "Ar", "Ai", "Tk", "Dk")),
                                (state["h"], state["beta"]), delta_softplus=True, z=state["z"])
        return [y, h, beta]
    if kind == "ply":
        with torch.no_grad():
            hid, cache = state["model"].step(token_id=state["tok"], cache=state["cache"])
            return [hid, F.linear(hid, state["head"]), *(t for st in cache for t in st)]
    if kind == "graph":
        with torch.no_grad():
            sg, hids = state["graph"], []
            sg.load(state["cache"])
            for t in range(case["plies"]):
                hid, cache = sg(token_id=state["tok"][t])
                hids.append(hid.clone())
            return [torch.stack(hids), F.linear(hid, state["head"]), *(t for st in cache for t in st)]
    amp = DTYPES[case["amp"]]
    with torch.autocast("cuda", dtype=amp, enabled=amp != torch.float32):
        out = state["block"](state["x"])
    return [out.detach(), *torch.autograd.grad(out, state["leaves"], state["dout"].to(out.dtype))]


# ---------------------------------------------------------------- the work

def _ply_work(case, R):
    d, D, N, p = case["d_model"], 2 * case["d_model"], case["d_state"], case["p"]
    r = math.ceil(d / 16)
    w = d * 2 * D + D * (r + 2 * N * p) + r * D + D * d
    # the weights and the cache in once and the cache out once, however many plies
    plies = case.get("plies", 1)
    return ((4 * w + 16 * R * D * N) * case["n_layer"],
            (2 * R * w + 12 * R * D * N) * case["n_layer"] * plies)


def work(case):
    kind = case["kind"]
    if kind == "scan":
        B, L, D, N = case["B"], case["L"], case["D"], case["NR"] + case["NT"]
        s = DTYPES[case["dtype"]].itemsize
        ins = B * L * (2 * D + 2 * N) * s
        params = 4 * D * (case["NR"] * (2 if case["imag"] else 1) + case["NT"])
        upd = B * L * D * N * (2 if case["bi"] else 1)
        nbytes, flops = ins + 4 * B * L * D + params, SCAN_FWD_FLOPS * upd
        if case["train"]:
            # the gradients out, dy in; the inputs stay in hand
            nbytes += ins + 4 * B * L * D + params
            flops += SCAN_BWD_FLOPS * upd
        return dict(bytes=nbytes, flops=flops)
    if kind == "prime":
        B, L, D, N = case["B"], case["L"], case["D"], case["NR"] + case["NT"]
        return dict(bytes=4 * (B * L * (3 * D + 2 * N) + 2 * D * N + 2 * B * D * N),
                    flops=SCAN_FWD_FLOPS * B * L * D * N)
    if kind == "step":
        R, D, N = case["R"], case["D"], case["NR"] + case["NT"]
        state = {"full": 16 * R * D * N, "rank1": 8 * R * D * N + 8 * R * (D + N),
                 "shared": 8 * R * D * N + 8 * D * N}[case["form"]]
        return dict(bytes=state + 4 * R * (4 * D + 2 * N) + 8 * D * N, flops=12 * R * D * N)
    if kind in ("ply", "graph"):
        R, head = case["R"], 8192 * case["d_model"]
        nbytes, flops = _ply_work(case, R)
        return dict(bytes=nbytes + 4 * (head + R * 8192), flops=flops + 2 * R * head)
    d, D, N, p = case["d_model"], 2 * case["d_model"], case["d_state"], case["p"]
    T = case["B"] * case["L"]
    r = math.ceil(d / 16)
    w = d * 2 * D + D * (r + 2 * N * p) + r * D + D * d
    upd = T * D * N * (2 if case["bi"] else 1)
    return dict(bytes=4 * (4 * T * d + 2 * w + 4 * D * N),
                flops=6 * T * w + (SCAN_FWD_FLOPS + SCAN_BWD_FLOPS) * upd)


def tolerance(case):
    # about four times the distance from `exact` that the path measures
    kind = case["kind"]
    if kind == "scan":
        if case["dtype"] == "fp32" or not case["train"]:
            # fp32 sums over the sequence; longer ones carry more roundings
            return {"rel": 1e-6 if case["L"] <= 512 else 3e-6}
        # gradients leave in the inputs' 16-bit types: half an ulp of those
        return {"rel": 8e-3 if case["dtype"] == "bf16" else 1e-3}
    if kind == "layer":
        return {"rel": {"fp32": 5e-6, "fp16": 5e-3, "bf16": 3e-2}[case["amp"]]}
    if kind in ("ply", "graph"):
        return {"rel": 1.2e-5}
    return {"rel": 5e-7}


# ---------------------------------------------------------------- in 64 bits

def _d(t):
    return None if t is None else t.detach().double()


def _run64(delta, u, Bc, Cc, Ar, Ai, Tk, h, hb):
    """The trapezoidal recurrence over (B, T, ...) from (h, beta / 2)."""
    parts = []
    if Ar is not None:
        g = torch.exp(delta[..., None] * Ar)
        parts.append(g if Ai is None else g * torch.cos(delta[..., None] * Ai))
    if Tk is not None:
        parts.append(Tk.expand(*delta.shape, Tk.shape[-1]))
    g = torch.cat(parts, -1) if len(parts) > 1 else parts[0]
    hbs = 0.5 * (delta * u)[..., None] * Bc[:, :, None, :]
    ys = []
    for t in range(delta.shape[1]):
        h = g[:, t] * (h + hb) + hbs[:, t]
        hb = hbs[:, t]
        ys.append((h * Cc[:, t, None, :]).sum(-1))
    return torch.stack(ys, 1), h, hb


def _span(B, D, N):
    return max(1, min(32, int(4e8 / (B * D * N))))


class _Scan64(torch.autograd.Function):
    """One causal scan in float64, its backward recomputed span by span."""

    @staticmethod
    def forward(ctx, delta, u, Bc, Cc, Ar, Ai, Tk):
        B, L, D = u.shape
        N = Bc.shape[-1]
        step = _span(B, D, N)
        h = torch.zeros(B, D, N, dtype=torch.float64, device=u.device)
        hb, ys, entry = h, [], []
        for t in range(0, L, step):
            entry.append((h, hb))
            s = slice(t, t + step)
            y, h, hb = _run64(delta[:, s], u[:, s], Bc[:, s], Cc[:, s], Ar, Ai, Tk, h, hb)
            ys.append(y)
        ctx.ins, ctx.entry, ctx.step = (delta, u, Bc, Cc, Ar, Ai, Tk), entry, step
        ctx.mark_non_differentiable(h, hb)
        return torch.cat(ys, 1), h, hb

    @staticmethod
    def backward(ctx, dy, _dh, _dhb):
        ins, step = ctx.ins, ctx.step
        L = ins[0].shape[1]
        grads = [None if t is None else torch.zeros_like(t) for t in ins]
        dh = dhb = torch.zeros_like(ctx.entry[0][0])
        for i in range(len(ctx.entry) - 1, -1, -1):
            s = slice(i * step, min(L, (i + 1) * step))
            with torch.enable_grad():
                loc = [None if t is None else (t[:, s] if k < 4 else t).detach().requires_grad_(True)
                       for k, t in enumerate(ins)]
                st = [t.detach().requires_grad_(True) for t in ctx.entry[i]]
                y, h, hb = _run64(*loc, *st)
                need = [t for t in loc if t is not None] + st
                got = torch.autograd.grad([y, h, hb], need, [dy[:, s], dh, dhb], allow_unused=True)
            got = list(got)
            dhb, dh = got.pop(), got.pop()
            for k in range(7):
                if ins[k] is not None:
                    gk = got.pop(0)
                    if gk is None:
                        continue
                    if k < 4:
                        grads[k][:, s] = gk
                    else:
                        grads[k] += gk
        return tuple(grads)


def _scan64(delta, u, Bc, Cc, Ar, Ai, Tk, bi):
    y, h, hb = _Scan64.apply(delta, u, Bc, Cc, Ar, Ai, Tk)
    if bi:
        yr, _, _ = _Scan64.apply(delta.flip(1), u.flip(1), Bc.flip(1), Cc.flip(1), Ar, Ai, Tk)
        y = y + yr.flip(1)
    return y, h, hb


def _norm64(x, w, eps=1e-5):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * w


def _proj64(P, x, case):
    """(x_branch, z, delta, Bc, Cc) of a layer's parameters P for inputs x."""
    n, p = case["d_state"], case["p"]
    xb, z = (x @ P["in_proj.weight"].T).chunk(2, -1)
    xb = F.silu(xb)
    r = P["dt_proj.weight"].shape[1]
    dt, B, C = (xb @ P["x_proj.weight"].T + P["x_proj.bias"]).split([r, n * p, n * p], -1)
    B = _norm64(B, P["b_norm.weight"]).unflatten(-1, (n, p)).sum(-1)
    C = _norm64(C, P["c_norm.weight"]).unflatten(-1, (n, p)).sum(-1)
    return xb, z, F.softplus(dt @ P["dt_proj.weight"].T + P["dt_proj.bias"]), B, C


def _gates64(P):
    mag = -torch.exp(P["A_log_mag"])
    Tk = torch.tanh(P["track_theta"]) if "track_theta" in P else None
    return mag * torch.cos(P["A_phase"]), mag * torch.sin(P["A_phase"]), Tk


def _step64(delta, u, Bc, Cc, Ar, Ai, Tk, Dk, h, beta):
    y, h, hb = _run64(delta[:, None], u[:, None], Bc[:, None], Cc[:, None], Ar, Ai, Tk, h, 0.5 * beta)
    return y[:, 0] + u * Dk, h, 2.0 * hb


def _ply64(P, layers, tok, cache, case):
    x, new = P["embedding.weight"][tok], []
    for L, (h, beta) in zip(layers, cache):
        xb, z, delta, B, C = _proj64(L, _norm64(x, L["norm.weight"]), case)
        y, h, beta = _step64(delta, xb, B, C, *_gates64(L), L["D"], h, beta)
        x = x + (y * F.silu(z)) @ L["out_proj.weight"].T
        new.append((h, beta))
    return _norm64(x, P["norm_f.weight"]), new


def exact(case, seed):
    kind = case["kind"]
    if kind == "scan":
        s = _scan_inputs(case, seed)
        ins = [_d(s[k]) for k in ("delta", "u", "Bc", "Cc", "Ar", "Ai", "Tk")]
        if not case["train"]:
            with torch.no_grad():
                return _scan64(*ins, case["bi"])[0]
        leaves = [t.requires_grad_(True) for t in ins if t is not None]
        y, _, _ = _scan64(*ins, case["bi"])
        return [y.detach(), *torch.autograd.grad(y, leaves, _d(s["dy"]))]
    if kind == "prime":
        s = _prime_inputs(case, seed)
        with torch.no_grad():
            y, h, hb = _scan64(F.softplus(_d(s["x"])), *(_d(s[k]) for k in
                               ("u", "Bc", "Cc", "Ar", "Ai", "Tk")), False)
        return [y, h, 2.0 * hb]
    if kind == "step":
        s = _step_inputs(case, seed)
        D = case["D"]
        u, B = _d(s["u"]), _d(s["Bc"])
        beta = _d(s["beta"])
        if case["form"] == "rank1":
            beta = beta[:, :D, None] * beta[:, None, D:]
        delta = F.softplus(_d(s["x"]))
        y, h, b = _step64(delta, u, B, *(_d(s[k]) for k in ("Cc", "Ar", "Ai", "Tk", "Dk")),
                          _d(s["h"]), beta)
        if case["form"] == "rank1":
            b = torch.cat([delta * u, B], -1)
        return [y * F.silu(_d(s["z"])), h, b]
    if kind in ("ply", "graph"):
        m, head, g = _model(case, seed)
        cache = [(_d(h), _d(b)) for h, b in _cache(case, g)]
        plies = (case["plies"],) if kind == "graph" else ()
        toks = torch.randint(0, 8192, (*plies, case["R"]), generator=g, device=DEV)
        P = {k: _d(v) for k, v in m.named_parameters()}
        layers = []
        for i in range(case["n_layer"]):
            pre = f"layers.{i}."
            L = {k[len(pre) + 6:]: v for k, v in P.items() if k.startswith(pre + "mixer.")}
            L["norm.weight"] = P[pre + "norm.weight"]
            layers.append(L)
        with torch.no_grad():
            if kind == "ply":
                hid, cache = _ply64(P, layers, toks, cache, case)
                return [hid, hid @ _d(head).T, *(t for st in cache for t in st)]
            hids = []
            for t in range(case["plies"]):
                hid, cache = _ply64(P, layers, toks[t], cache, case)
                hids.append(hid)
            return [torch.stack(hids), hid @ _d(head).T, *(t for st in cache for t in st)]
    s = prepare(case, seed)
    x = _d(s["x"]).requires_grad_(True)
    P = {k: _d(v).requires_grad_(True) for k, v in s["block"].named_parameters()}
    xb, z, delta, B, C = _proj64(P, x, case)
    y, _, _ = _scan64(delta, xb, B, C, *_gates64(P), case["bi"])
    y = (y + (2 if case["bi"] else 1) * xb * P["D"]) * F.silu(z)
    out = y @ P["out_proj.weight"].T
    return [out.detach(), *torch.autograd.grad(out, [x, *P.values()], _d(s["dout"]))]
