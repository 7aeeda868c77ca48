"""What is timed: the work a program has this package do, through its public layers, over the range of shapes, options
and directions in use. Every case runs one whole call (a forward, or a forward and backward that returns every
gradient) on inputs made from the seed, and ``exact`` restates it in float64 with plain torch operations.

Kinds of case:

    scan   an ``EWS`` / ``LogEWS`` layer on a batch of paths
    token  the token cache and the cached scan of a formal-language block
    mixer  a block's mixer epilogue on prefix rows
"""

from __future__ import annotations

import math
import os
import sys
from fractions import Fraction

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PACKAGE = os.path.join(ROOT, "exponentially-weighted-signature_amd")
if PACKAGE not in sys.path:
    sys.path.insert(0, PACKAGE)

F64 = torch.float64

# Options every scan case states; a case overrides what it needs.
SCAN = dict(kind="scan", layer="ews", gen="planes", B=1, L=2, d=2, N=2, leaf="plane_closed", q=0, M=0, vl="exact",
            chen="exact", mode="displacement", readout="prefix", dtype="float32", path="brownian", clock="uniform",
            block=0, train=True, clock_grad=False)


def _scan(**kw):
    return dict(SCAN, **kw)


# ------------------------------------------------------------------------------------------------------- the cases
def listed():
    return [
        # The smallest call: inference over a few short three-channel recordings with a diagonal generator. Launches
        # and their latency are all of it.
        _scan(name="diag8_forward", gen="diag", B=8, L=1024, d=8, leaf="series", q=8, train=False),
        # The headline training step: long regularly sampled recordings (EigenWorms' length), 8 rotation planes.
        _scan(name="planes16_train", B=32, L=17984, d=16),
        # A learned clock: irregular steps, the clock's gradient wanted too, a medium and odd length.
        _scan(name="planes16_learned_clock_train", B=32, L=1751, d=16, clock="learned", clock_grad=True),
        # The longest sequences: a 32 Hz physiological recording, 12 planes, the path in bfloat16.
        _scan(name="planes24_bf16_train", B=8, L=49920, d=24, dtype="bfloat16", path="sinusoids"),
        # Many token sequences of moderate length through the log-signature layer, 32 real decay rates, unit steps.
        _scan(name="logews_diag32_train", layer="log", gen="diag", B=256, L=512, d=32, leaf="series", q=12,
              path="tokens", clock="steps"),
        # A dense generator at depth 3 with an input-dependent clock: the reference's default leaf, training.
        _scan(name="dense16_depth3_train", gen="dense", B=16, L=4096, d=16, N=3, leaf="van_loan", M=20, vl="cayley",
              path="walk", clock="gated"),
        # The same model served with the series leaf: forward only.
        _scan(name="dense16_depth3_series_forward", gen="dense", B=16, L=4096, d=16, N=3, leaf="series", q=24,
              path="walk", clock="gated", train=False),
        # The layer's defaults on a generator wider than 16, irregular clock, one terminal state per sample.
        _scan(name="dense24_terminal_train", gen="dense", B=32, L=896, d=24, leaf="van_loan", M=20, vl="cayley",
              clock="irregular", readout="terminal", clock_grad=True),
        # A sequence classifier's block: skew-symmetric d = 17, one shared step per sample, mean readout.
        _scan(name="skew17_mean_train", gen="skew", B=32, L=896, d=17, leaf="van_loan", M=4, vl="euler",
              chen="cayley", mode="displacement_uniform", readout="mean", clock="linspace"),
        # The banked depth-1 block of the physiological model: 16 complex Jordan chains of 4, gated clock.
        _scan(name="chains64_train", gen="jordan_complex", B=8, L=49920, d=64, N=1, block=4, leaf="jordan_closed",
              clock="clamped", clock_grad=True),
        # A formal-language block: 8 tokens, 32 rotation planes, ragged masked sequences.
        dict(kind="token", name="token64_train", B=256, L=512, d=64, V=8),
        # The mixer epilogue of a long-sequence block: 399k rows of 601 numbers down to 24 channels.
        dict(kind="mixer", name="mixer24_train", B=8, R=49919, d=24, N=2, hidden=24, variant="live_rms"),
    ]


def _log(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    pick = rng.randrange(11)
    if pick == 0:
        return _scan(gen="diag", B=_log(rng, 1, 16), L=_log(rng, 64, 2048), d=rng.randint(3, 16), leaf="series", q=8,
                     train=False)
    if pick == 1:
        return _scan(B=_log(rng, 2, 32), L=_log(rng, 1000, 17984), d=16)
    if pick == 2:
        return _scan(B=_log(rng, 2, 32), L=_log(rng, 200, 3000), d=16, clock="learned", clock_grad=True)
    if pick == 3:
        return _scan(B=_log(rng, 1, 8), L=_log(rng, 3000, 49920), d=2 * rng.randint(4, 12),
                     dtype=rng.choice(["bfloat16", "float32"]), path="sinusoids")
    if pick == 4:
        return _scan(layer="log", gen="diag", B=rng.randint(128, 256), L=_log(rng, 100, 512), d=rng.randint(12, 32),
                     leaf="series", q=12, path="tokens", clock="steps")
    if pick == 5:
        return _scan(gen="dense", B=_log(rng, 2, 16), L=_log(rng, 400, 4096), d=rng.randint(8, 16),
                     N=rng.choice([2, 3, 3]), leaf="van_loan", M=20, vl="cayley", path="walk", clock="gated")
    if pick == 6:
        return _scan(gen="dense", B=_log(rng, 2, 16), L=_log(rng, 400, 4096), d=rng.randint(8, 16), N=3,
                     leaf="series", q=24, path="walk", clock="gated", train=False)
    if pick == 7:
        return _scan(gen="dense", B=_log(rng, 4, 32), L=_log(rng, 100, 896), d=rng.randint(17, 28), leaf="van_loan",
                     M=20, vl="cayley", clock="irregular", readout=rng.choice(["terminal", "mean"]), clock_grad=True)
    if pick == 8:
        return _scan(gen="skew", B=_log(rng, 4, 32), L=_log(rng, 100, 896), d=rng.randint(17, 28), leaf="van_loan",
                     M=4, vl="euler", chen="cayley", mode="displacement_uniform", readout="mean", clock="linspace")
    if pick == 9:
        kind, size = rng.choice([("real", 2), ("real", 4), ("complex", 4), ("complex", 6)])
        return _scan(gen="jordan_" + kind, B=_log(rng, 1, 8), L=_log(rng, 3000, 49920),
                     d=size * rng.randint(4, 64 // size), N=1, block=size, leaf="jordan_closed", clock="clamped",
                     clock_grad=True)
    if rng.random() < 0.5:
        return dict(kind="token", B=_log(rng, 32, 256), L=_log(rng, 100, 512), d=2 * rng.randint(10, 32),
                    V=rng.randint(3, 8))
    return dict(kind="mixer", B=_log(rng, 1, 8), R=_log(rng, 3000, 49919), d=rng.randint(8, 24), N=2,
                hidden=rng.randint(12, 64), variant=rng.choice(["live_rms", "static_gain"]))


# ------------------------------------------------------------------------------------------------------ the inputs
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _generator(case, seed):
    g = torch.Generator(device=_device())
    g.manual_seed(1000003 * int(seed) + 17 * case["B"] + case["d"])
    return g


def _path(case, g):
    """(B, L, d) float32: what a block hands to its layer, a low-dimensional signal lifted to d channels."""
    B, L, d = case["B"], case["L"], case["d"]
    dev = _device()
    c = min(6, d)
    lift = torch.randn(d, c, generator=g, device=dev) / math.sqrt(c)
    if case["path"] == "brownian":  # increments of variance 1 / L
        raw = torch.randn(B, L, c, generator=g, device=dev, dtype=F64).cumsum(1) / math.sqrt(L)
    elif case["path"] == "walk":  # unit increments (a standardised feature stream)
        raw = torch.randn(B, L, c, generator=g, device=dev, dtype=F64).cumsum(1)
    elif case["path"] == "sinusoids":  # four tones a channel at 32 Hz and noise
        t = torch.arange(L, device=dev, dtype=F64) / 32.0
        raw = 0.22 * torch.randn(B, L, c, generator=g, device=dev, dtype=F64)
        for _ in range(4):
            f = 0.5 + 2.5 * torch.rand(B, 1, c, generator=g, device=dev, dtype=F64)
            ph = 2 * math.pi * torch.rand(B, 1, c, generator=g, device=dev, dtype=F64)
            raw += torch.sin(2 * math.pi * f * t[None, :, None] + ph)
    else:  # "tokens": an embedding of 8 letters, read as the path's values
        emb = torch.randn(8, d, generator=g, device=dev) / math.sqrt(d)
        return emb[torch.randint(0, 8, (B, L), generator=g, device=dev)].contiguous()
    return (raw @ lift.to(F64).t()).to(torch.float32).contiguous()


def _clock(case, g):
    """(B, L) float32 clock values."""
    B, L = case["B"], case["L"]
    dev = _device()
    kind = case["clock"]
    if kind == "uniform":  # k / L
        return (torch.arange(L, device=dev, dtype=F64) / L).expand(B, L).to(torch.float32).contiguous()
    if kind == "steps":  # the block's default clock, one unit a token
        return torch.arange(L, device=dev, dtype=torch.float32).expand(B, L).contiguous()
    if kind == "linspace":
        return torch.linspace(-1.0, 1.0, L, device=dev, dtype=F64).expand(B, L).to(torch.float32).contiguous()
    if kind == "irregular":  # uniformly spread steps about 1 / L
        inc = (0.5 + torch.rand(B, L, generator=g, device=dev, dtype=F64)) / L
    elif kind == "learned":  # a token-gated clock scaled to a fixed horizon
        inc = torch.nn.functional.softplus(torch.randn(B, L, generator=g, device=dev, dtype=F64)) * (4.0 / L)
    elif kind == "clamped":  # a clamped gate: some steps stand still
        inc = (0.5 + 0.6 * torch.randn(B, L, generator=g, device=dev, dtype=F64)).clamp(0.0, 1.0) * (2.0 / L)
    else:  # "gated": softplus of the input's increment, steps of order one
        inc = torch.nn.functional.softplus(0.9 * torch.randn(B, L, generator=g, device=dev, dtype=F64))
    inc[:, 0] = 0.0
    return inc.cumsum(1).to(torch.float32)


def _inverse_softplus(x):
    return torch.log(torch.expm1(x))


def _generator_values(case, g):
    """The generator's trainable numbers by name, float32."""
    d, dev = case["d"], _device()
    gen = case["gen"]

    def uniform(n, lo, hi):
        return lo + (hi - lo) * torch.rand(n, generator=g, device=dev)

    if gen == "planes":  # damping in (0.01, 1), frequency in (0, pi)
        return {"v": _inverse_softplus(uniform(d // 2, 0.01, 1.0)), "u": torch.logit(uniform(d // 2, 0.02, 0.98))}
    if gen == "diag":
        return {"theta": _inverse_softplus(uniform(d, 0.1, 2.0))}
    if gen == "dense":
        X = torch.randn(d, d, generator=g, device=dev) * math.sqrt(0.1)
        return {"matrix": torch.diag(torch.nn.functional.softplus(uniform(d, 0.0, 1.0))) - (X - X.t()) / math.sqrt(2)}
    if gen == "skew":
        X = torch.randn(d, d, generator=g, device=dev) * 0.1
        return {"matrix": X - X.t()}
    K = d // case["block"]
    rate = _inverse_softplus(uniform(K, 0.005, 0.5))
    if gen == "jordan_real":
        return {"chains": rate[:, None].contiguous()}
    return {"chains": torch.stack([rate, uniform(K, -15.0, 15.0)], 1)}


def _param(case, values):
    import ews_mi355x as E

    gen, d = case["gen"], case["d"]
    if gen == "planes":
        return E.AParamDampedRotation(values["v"].clone(), values["u"].clone(), d, omega_scale=math.pi)
    if gen == "diag":
        return E.AParamEFM(values["theta"].clone())
    if gen in ("dense", "skew"):
        return E.AParamGeneral(values["matrix"].clone())
    K = d // case["block"]
    return E.AParamJordanRepeated([case["block"]] * K, [gen.split("_")[1]] * K, [row.clone() for row in values["chains"]])


def _layer(case, values):
    import ews_mi355x as E

    kw = dict(N=case["N"], leaf=case["leaf"], van_loan_expm=case["vl"], chen_expm=case["chen"],
              reweighting_mode=case["mode"])
    if case["M"]:
        kw["M"] = case["M"]
    if case["q"]:
        kw["series_q"] = case["q"]
    if case["gen"].startswith("jordan"):
        kw.update(combine="block_kernel", jordan_flows=True)
    return (E.LogEWS if case["layer"] == "log" else E.EWS)(_param(case, values), **kw).to(_device())


def _width(case):
    d, N = case["d"], case["N"]
    if case["layer"] == "log":
        return d + d * (d - 1) // 2
    return 1 + sum(d**k for k in range(1, N + 1))


def _cotangent(case, g):
    shape = (case["B"], _width(case)) if case["readout"] != "prefix" else (case["B"], case["L"] - 1, _width(case))
    return torch.randn(shape, generator=g, device=_device())


def _scan_inputs(case, seed):
    g = _generator(case, seed)
    path, clock, values = _path(case, g), _clock(case, g), _generator_values(case, g)
    return path.to(getattr(torch, case["dtype"])), clock, values, _cotangent(case, g) if case["train"] else None


def _token_inputs(case, seed):
    g, dev = _generator(case, seed), _device()
    B, L, d, V = case["B"], case["L"], case["d"], case["V"]
    dx = 0.3 * torch.randn(V, d, generator=g, device=dev)
    dth = 0.05 + 0.35 * torch.rand(V, generator=g, device=dev)
    v, u = torch.randn(d // 2, generator=g, device=dev), torch.randn(d // 2, generator=g, device=dev)
    tok = torch.randint(0, V, (B, L), generator=g, device=dev)
    lens = torch.randint(L // 4, L + 1, (B,), generator=g, device=dev)
    mask = torch.arange(L, device=dev)[None, :] < lens[:, None]
    return dx, dth, v, u, tok, mask, torch.randn(B, L, d, generator=g, device=dev) / math.sqrt(d)


def _mixer_inputs(case, seed):
    g, dev = _generator(case, seed), _device()
    B, R, d, N, H = case["B"], case["R"], case["d"], case["N"], case["hidden"]
    D = sum(d**k for k in range(1, N + 1))
    rows = torch.randn(B, R, 1 + D, generator=g, device=dev)
    rows[..., 0] = 1.0
    rows[..., 1 + d:] *= 0.3  # the levels differ in scale
    lim = 1.0 / math.sqrt(D)
    weight = lim * (2 * torch.rand(H, D, generator=g, device=dev) - 1)
    bias = lim * (2 * torch.rand(H, generator=g, device=dev) - 1)
    gains = 0.5 + torch.rand(N, generator=g, device=dev)
    return rows, weight, bias, gains, torch.randn(B, R + 1, H, generator=g, device=dev)


# -------------------------------------------------------------------------------------------- the calls that count
def prepare(case, seed):
    if case["kind"] == "scan":
        path, clock, values, g = _scan_inputs(case, seed)
        layer = _layer(case, values)
        if not case["train"]:
            layer.eval()
        path.requires_grad_(case["train"])
        clock.requires_grad_(case["clock_grad"])
        return {"case": case, "layer": layer, "path": path, "clock": clock, "g": g}
    if case["kind"] == "token":
        import ews_mi355x as E

        dx, dth, v, u, tok, mask, g = _token_inputs(case, seed)
        param = E.AParamDampedRotation(v, u, case["d"], omega_scale=2.0).to(_device())
        return {"case": case, "param": param, "dx": dx.requires_grad_(True), "dth": dth.requires_grad_(True),
                "tok": tok, "mask": mask, "g": g}
    import ews_mi355x as E

    rows, weight, bias, gains, g = _mixer_inputs(case, seed)
    mixer = E.MixerEpilogue(case["d"], case["N"], case["hidden"], graded_variant=case["variant"]).to(_device())
    with torch.no_grad():
        mixer.c_down.weight.copy_(weight)
        mixer.c_down.bias.copy_(bias)
        mixer.graded.gains.copy_(gains)
    return {"case": case, "mixer": mixer, "rows": rows.requires_grad_(True), "g": g}


def run(state):
    kind = state["case"]["kind"]
    if kind == "scan":
        layer, path, clock, readout = state["layer"], state["path"], state["clock"], state["case"]["readout"]
        if not state["case"]["train"]:
            with torch.no_grad():
                return {"out": layer(path, clock, readout=readout)}
        inputs = [path] + ([clock] if clock.requires_grad else []) + list(layer.parameters())
        out = layer(path, clock, readout=readout)
        return {"out": out.detach(), "grads": list(torch.autograd.grad(out, inputs, state["g"]))}
    if kind == "token":
        import ews_mi355x as E

        param, d = state["param"], state["case"]["d"]
        P, D = E.build_token_cache(state["dx"], state["dth"], param(), 4, 1, "exact", "exact", "van_loan")
        out = E.token_cached_prefix_scan(state["tok"], state["mask"], P, D, d, 1)
        inputs = [state["dx"], state["dth"]] + list(param.parameters())
        return {"out": out.detach(), "grads": list(torch.autograd.grad(out, inputs, state["g"]))}
    mixer = state["mixer"]
    out = mixer(state["rows"])
    inputs = [state["rows"], mixer.c_down.weight, mixer.c_down.bias, mixer.graded.gains]
    return {"out": out.detach(), "grads": list(torch.autograd.grad(out, inputs, state["g"]))}


def work(case):
    """Compulsory bytes (each input read once, each output written once) and the multiply-adds of the recursion or
    contraction itself, times three for a forward and backward."""
    if case["kind"] == "token":
        n = case["B"] * case["L"]
        return {"bytes": n * (4 * case["d"] * 2 + 8 + 1), "flops": 3 * n * 4 * case["d"]}
    if case["kind"] == "mixer":
        n, D, H = case["B"] * case["R"], case["d"] + case["d"] ** 2, case["hidden"]
        return {"bytes": 4 * n * (2 * (D + 1) + 2 * H), "flops": 3 * n * 2 * D * H}
    B, L, d, N, W = case["B"], case["L"], case["d"], case["N"], _width(case)
    s = 2 if case["dtype"] == "bfloat16" else 4
    rows = B * W * (L - 1 if case["readout"] == "prefix" else 1)
    nbytes = B * L * (s * d + 4) + 4 * rows
    if case["train"]:
        nbytes += 4 * rows + B * L * s * d + (4 * B * L if case["clock_grad"] else 0)
    bs = {"planes": 2, "diag": 1, "dense": d, "skew": d}.get(case["gen"], case["block"])
    step = sum(2 * k * d**k * bs + 2 * (k - 1) * d**k for k in range(1, N + 1))
    return {"bytes": nbytes, "flops": (3 if case["train"] else 1) * B * (L - 1) * step}


def tolerance(case):
    """Relative 2-norm bounds, about four times the largest distance from float64 that this path shows on any output:
    7e-6 for float32 recursions of up to 50k steps, 1.2e-5 for the wide dense generators (whose float32 step matrices
    are reused at every step); a bfloat16 path rounds its gradient to 8 bits (1.7e-3)."""
    if case.get("dtype") == "bfloat16":
        return {"rel": 8e-3, "max": 0.1}
    if case.get("gen") in ("dense", "skew") and case["d"] > 16:
        return {"rel": 5e-5, "max": 5e-3}
    return {"rel": 3e-5, "max": 3e-3}


# -------------------------------------------------------------------------------------------------- the same in 64 bits
def exact(case, seed):
    if case["kind"] == "scan":
        return _exact_scan(case, seed)
    if case["kind"] == "token":
        return _exact_token(case, seed)
    return _exact_mixer(case, seed)


def _blocks(case, values):
    """The generator's diagonal blocks (nb, bs, bs) from its trainable numbers, differentiable."""
    gen, d = case["gen"], case["d"]
    if gen == "planes":
        a, b = torch.nn.functional.softplus(values["v"]), math.pi * torch.sigmoid(values["u"])
        return torch.stack([torch.stack([a, -b], -1), torch.stack([b, a], -1)], -2)
    if gen == "diag":
        return torch.nn.functional.softplus(values["theta"])[:, None, None]
    if gen in ("dense", "skew"):
        return values["matrix"][None]
    bs, P = case["block"], values["chains"]
    a = torch.nn.functional.softplus(P[:, 0])[:, None, None]
    eye = torch.eye(bs, dtype=F64, device=P.device)
    if gen == "jordan_real":
        return a * eye + torch.diag(torch.ones(bs - 1, dtype=F64, device=P.device), 1)
    rot = torch.tensor([[0.0, -1.0], [1.0, 0.0]], dtype=F64, device=P.device)
    rot = torch.block_diag(*[rot] * (bs // 2))
    return a * eye + P[:, 1][:, None, None] * rot + torch.diag(torch.ones(bs - 2, dtype=F64, device=P.device), 2)


def _expm(X, norm):
    """exp of a batch of matrices whose 1-norms are at most ``norm``: degree-20 Taylor and repeated squaring."""
    s = max(0, math.ceil(math.log2(max(norm, 1e-30))) + 1)
    Y = X / 2.0**s
    eye = torch.eye(X.shape[-1], dtype=X.dtype, device=X.device)
    E = eye + Y / 20
    for k in range(19, 0, -1):
        E = eye + Y @ E / k
    for _ in range(s):
        E = E @ E
    return E


def _scheme(X, how, norm):
    eye = torch.eye(X.shape[-1], dtype=X.dtype, device=X.device)
    if how == "cayley":
        return torch.linalg.solve(eye - X / 2, eye + X / 2)
    return _expm(X, norm)


def _apply(F, T, axis):
    """Block-diagonal F (n, nb, bs, bs) on one tensor axis of T (n, d, ..)."""
    n, nb, bs = F.shape[:3]
    X = torch.movedim(T, axis, 1)
    rest = X.shape[2:]
    Y = torch.matmul(F, X.reshape(n, nb, bs, -1)).reshape((n, nb * bs) + rest)
    return torch.movedim(Y, 1, axis)


def _outer(a, b):
    return a.reshape(a.shape + (1,) * (b.dim() - 1)) * b.reshape(b.shape[:1] + (1,) * (a.dim() - 1) + b.shape[1:])


def _chen(S, F, s):
    """S flowed by F along every axis, then the truncated tensor product with s."""
    flowed = []
    for k, x in enumerate(S, 1):
        for ax in range(1, k + 1):
            x = _apply(F, x, ax)
        flowed.append(x)
    out = []
    for k in range(len(S)):
        x = flowed[k] + s[k]
        for j in range(k):
            x = x + _outer(flowed[j], s[k - j - 1])
        out.append(x)
    return out


def _prefix(levels, F, B):
    """Prefix states of B samples (levels and flows given for B * n intervals, sample-major): chunks of about sqrt(n)
    intervals step together, their ends are scanned, each chunk's rows take its carry."""
    n = levels[0].shape[0] // B
    T = max(1, int(math.sqrt(n)))
    C = -(-n // T)
    pad = C * T - n
    eye = torch.eye(F.shape[-1], dtype=F64, device=F.device).expand((B, pad) + F.shape[1:])
    Fc = torch.cat([F.reshape((B, n) + F.shape[1:]), eye], 1).reshape((B * C, T) + F.shape[1:])
    Lc = []
    for x in levels:
        x = x.reshape((B, n) + x.shape[1:])
        x = torch.cat([x, torch.zeros((B, pad) + x.shape[2:], dtype=F64, device=x.device)], 1)
        Lc.append(x.reshape((B * C, T) + x.shape[2:]))
    S, P = [x[:, 0] for x in Lc], Fc[:, 0]
    rows, flows = [S], [P]
    for t in range(1, T):
        S, P = _chen(S, Fc[:, t], [x[:, t] for x in Lc]), Fc[:, t] @ P
        rows.append(S)
        flows.append(P)
    ends = [x.reshape((B, C) + x.shape[1:]) for x in S]
    Pe = P.reshape((B, C) + P.shape[1:])
    carry = [[torch.zeros_like(x[:, 0]) for x in ends]]
    for c in range(C - 1):
        carry.append(_chen(carry[-1], Pe[:, c], [x[:, c] for x in ends]))
    carry = [torch.stack([c[k] for c in carry], 1).flatten(0, 1) for k in range(len(levels))]
    out = [_chen(carry, flows[t], rows[t]) for t in range(T)]
    out = [torch.stack([o[k] for o in out], 1) for k in range(len(levels))]
    return [x.reshape((B, C * T) + x.shape[2:])[:, :n] for x in out]


def _series(v, h, A, N, q):
    """The order-q series of an interval's iterated integrals: letters b_p = (-h A)^p v / p!, and the coefficient of
    b_m1 (x) .. (x) b_mk (total order at most q) is prod_j 1 / (m_j + .. + m_k + k - j + 1)."""
    b = [v]
    for p in range(1, q + 1):
        b.append((-h / p)[:, None] * _apply(A[None].expand((v.shape[0],) + A.shape), b[-1], 1))
    b = torch.stack(b, 1)  # (n, q + 1, d)
    r = range(q + 1)
    dev = v.device
    c1 = torch.tensor([1.0 / (p + 1) for p in r], dtype=F64, device=dev)
    out = [torch.einsum("p,npi->ni", c1, b)]
    if N >= 2:
        c2 = torch.tensor([[float(Fraction(1, (a + e + 2) * (e + 1))) if a + e <= q else 0.0 for e in r] for a in r],
                          dtype=F64, device=dev)
        out.append(torch.matmul(torch.einsum("ae,nai->nie", c2, b), b))
    if N >= 3:
        c3 = torch.tensor([[[float(Fraction(1, (a + e + f + 3) * (e + f + 2) * (f + 1))) if a + e + f <= q else 0.0
                             for f in r] for e in r] for a in r], dtype=F64, device=dev)
        n, _, d = b.shape
        G = torch.einsum("aef,nai->nfie", c3, b)  # (n, f, i, e)
        G = torch.matmul(G.reshape(n, -1, q + 1), b).reshape(n, q + 1, d * d)
        out.append(torch.matmul(G.transpose(1, 2), b).reshape(n, d, d, d))
    return out


def _integrals(v, h, A, N, norm):
    """The interval's iterated integrals themselves: an order-16 series on a 2^s-th of it, then s Chen doublings."""
    s = max(0, math.ceil(math.log2(max(norm, 1e-30))) + 2)
    w, step = v / 2.0**s, h / 2.0**s
    S = _series(w, step, A, N, 16)
    for k in range(s):
        F = _expm(-(step * 2.0**k)[:, None, None, None] * A, max(norm, 1e-30) * 2.0 ** (k - s))
        S = _chen(S, F, S)
    return S


def _van_loan(v, h, A, N, M, how, norm):
    """The signature of the M + 1 reweighted knots of each interval: increments Delta_M = V w, Delta_{m-1} = P Delta_m
    with w = v / M, P the inverse of the scheme's exp(a), a = h A / M, and V its integral."""
    n, d = v.shape
    a = (h / M)[:, None, None] * A[0]
    eye = torch.eye(d, dtype=F64, device=v.device)
    if how == "cayley":
        V = torch.linalg.inv(eye + a / 2)
        P = 2 * V - eye
    else:  # euler
        P = V = torch.linalg.inv(eye + a)
    if a.shape[0] == 1:
        P, V = P.expand(n, d, d), V.expand(n, d, d)
    step = [torch.matmul(V, (v / M)[..., None])[..., 0]]
    for _ in range(M - 1):
        step.append(torch.matmul(P, step[-1][..., None])[..., 0])
    S = None
    for x in reversed(step):
        seg = [x]
        for k in range(2, N + 1):
            seg.append(_outer(seg[-1], x) / k)
        if S is None:
            S = seg
        else:
            S = [S[k] + seg[k] + sum(_outer(S[j], seg[k - j - 1]) for j in range(k)) for k in range(N)]
    return S


def _exact_scan(case, seed):
    path, clock, values, g = _scan_inputs(case, seed)
    B, L, d, N = case["B"], case["L"], case["d"], case["N"]
    values = {k: x.to(F64).requires_grad_(case["train"]) for k, x in values.items()}
    path = path.to(F64)
    clock = clock.to(F64)
    n = L - 1
    group = max(1, min(B, int(4e7 / (n * d**N))))
    outs, gpath, gclock = [], [], []
    gvals = {k: torch.zeros_like(x) for k, x in values.items()}
    for b0 in range(0, B, group):
        p = path[b0:b0 + group].clone().requires_grad_(case["train"])
        c = clock[b0:b0 + group].clone().requires_grad_(case["train"])
        with torch.set_grad_enabled(case["train"]):
            out = _exact_rows(case, p, c, _blocks(case, values))
        outs.append(out.detach())
        if case["train"]:
            names = list(values)
            got = torch.autograd.grad(out, [p, c] + [values[k] for k in names], g[b0:b0 + group].to(F64))
            gpath.append(got[0])
            gclock.append(got[1])
            for k, x in zip(names, got[2:]):
                gvals[k] += x
        del out
    answer = {"out": torch.cat(outs)}
    if case["train"]:
        grads = [torch.cat(gpath)] + ([torch.cat(gclock)] if case["clock_grad"] else [])
        order = {"planes": ["v", "u"], "diag": ["theta"], "dense": ["matrix"], "skew": ["matrix"]}
        for k in order.get(case["gen"], ["chains"]):
            grads += list(gvals[k]) if k == "chains" else [gvals[k]]
        answer["grads"] = grads
    return answer


def _exact_rows(case, path, clock, A):
    B, L, d = path.shape
    N, n = case["N"], L - 1
    v = (path[:, 1:] - path[:, :-1]).reshape(B * n, d)
    h = (clock[:, 1:] - clock[:, :-1]).reshape(B * n)
    shared = case["mode"] == "displacement_uniform"
    norm = float(A.detach().abs().sum(-2).max() * h.detach().abs().max())
    if shared:  # one step a sample: its first
        h = h.reshape(B, n)[:, :1].expand(B, n).reshape(B * n)
    if case["leaf"] == "series":
        S = _series(v, h, A, N, case["q"])
    elif case["leaf"] == "van_loan":
        if shared:
            parts = [_van_loan(v[b * n:(b + 1) * n], h[b * n:b * n + 1], A, N, case["M"], case["vl"], norm)
                     for b in range(B)]
            S = [torch.cat([x[k] for x in parts]) for k in range(N)]
        else:
            S = _van_loan(v, h, A, N, case["M"], case["vl"], norm)
    else:
        S = _integrals(v, h, A, N, norm)
    if shared:
        F = _scheme(-h.reshape(B, n)[:, 0][:, None, None, None] * A, case["chen"], norm)
        F = F[:, None].expand((B, n) + F.shape[1:]).reshape((B * n,) + F.shape[1:])
    else:
        F = _scheme(-h[:, None, None, None] * A, case["chen"], norm)
    rows = _prefix(S, F, B)
    if case["layer"] == "log":
        i, j = torch.triu_indices(d, d, 1, device=path.device)
        area = rows[1] - 0.5 * rows[0][..., :, None] * rows[0][..., None, :]
        return torch.cat([rows[0], area[:, :, i, j]], -1)
    flat = torch.cat([torch.ones((B, n, 1), dtype=F64, device=path.device)] + [x.reshape(B, n, -1) for x in rows], -1)
    if case["readout"] == "terminal":
        return flat[:, -1]
    if case["readout"] == "mean":
        return flat.mean(1)
    return flat


def _exact_token(case, seed):
    dx, dth, v, u, tok, mask, g = _token_inputs(case, seed)
    B, L, d = case["B"], case["L"], case["d"]
    dx, dth, v, u = (x.to(F64).requires_grad_(True) for x in (dx, dth, v, u))
    a, b = torch.nn.functional.softplus(v), 2.0 * torch.sigmoid(u)
    A = torch.stack([torch.stack([a, -b], -1), torch.stack([b, a], -1)], -2)
    norm = float(A.detach().abs().sum(-2).max() * dth.detach().abs().max())
    P = _integrals(dx, dth, A, 1, norm)[0]  # at depth 1 exact exponentials make the Van Loan leaf the integral itself
    D = _expm(-dth[:, None, None, None] * A, norm)
    on = mask.reshape(-1)
    F = torch.where(on[:, None, None, None], D[tok.reshape(-1)], torch.eye(2, dtype=F64, device=D.device))
    s = torch.where(on[:, None], P[tok.reshape(-1)], torch.zeros((), dtype=F64, device=D.device))
    out = _prefix([s], F, B)[0]
    return {"out": out.detach(), "grads": list(torch.autograd.grad(out, [dx, dth, v, u], g.to(F64)))}


def _exact_mixer(case, seed):
    rows, weight, bias, gains, g = _mixer_inputs(case, seed)
    d, N = case["d"], case["N"]
    rows, weight, bias, gains = (x.to(F64).requires_grad_(True) for x in (rows, weight, bias, gains))
    x = torch.cat([torch.zeros_like(rows[:, :1, 1:]), rows[:, :, 1:]], 1)  # a zero row before the first interval
    parts, st = [], 0
    for k in range(N):
        blk = x[..., st:st + d ** (k + 1)]
        st += d ** (k + 1)
        if case["variant"] == "live_rms":
            ms = (blk * blk).mean(-1, keepdim=True)
            rms = torch.where(ms > 0, torch.sqrt(torch.where(ms > 0, ms, torch.ones_like(ms))), torch.zeros_like(ms))
            blk = blk / (rms + 1e-3)
        parts.append(gains[k] * blk)
    out = torch.cat(parts, -1) @ weight.t() + bias
    return {"out": out.detach(), "grads": list(torch.autograd.grad(out, [rows, weight, bias, gains], g.to(F64)))}
