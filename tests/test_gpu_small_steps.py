"""Irregular clocks under the small-step coefficient model, forward and every gradient, against the float64 oracle:
chunks whose steps can be inverted and chunks too contractive for it, planes and real diagonals on every lane map, the
d = 16 pair-group forward with chunks of every class in one call, the chunk lengths the library suits to few intervals,
steps on both sides of the model's radius, clocks that turn inside a chunk, in other units, and recordings padded with
NaN. Bars as the repository's: forward 1e-5, gradients 1e-4."""

import ctypes

import numpy as np
import pytest
import torch

from ews_mi355x import _native as nat
from ews_mi355x import ops
from oracle import ews_oracle as O

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _rel(a, b):
    a, b = a.detach().cpu().double(), b.detach().double()
    return float((a - b).abs().max() / b.abs().max().clamp_min(1e-300))


def _check(structure, d, N, B, L, steps, damp, readout="prefix", chunk=0, bf16=False, flow="per_interval", freq=3.0,
           rows=None, clock_grad=True):
    """steps (L,): the clock's steps (the first unused). rows: the prefix rows that the loss sees (all)."""
    rng = np.random.default_rng(L + d)
    path = torch.tensor(np.cumsum(rng.normal(size=(B, L, d)) * 0.2, 1), dtype=torch.float32)
    path = path.to(torch.bfloat16) if bf16 else path
    clock = torch.tensor(np.cumsum(np.stack([steps * rng.uniform(0.9, 1.1) for _ in range(B)]), 1), dtype=torch.float32)
    if structure == "planes":
        w = np.stack([rng.uniform(*damp, d // 2), rng.uniform(0.0, freq, d // 2)], -1)
        w = torch.tensor(w, dtype=torch.float32)
    else:
        w = torch.tensor(rng.uniform(*damp, d), dtype=torch.float32)
    p, c, q = path.to(DEV).requires_grad_(), clock.to(DEV).requires_grad_(clock_grad), w.to(DEV).requires_grad_()
    out = ops.diag_scan(p, c, q, N, structure, flow, readout, True, chunk=chunk)
    g = torch.tensor(rng.normal(size=tuple(out.shape)), dtype=torch.float32)
    if rows is not None:
        g[:, rows:] = 0.0
    got = torch.autograd.grad(out, [p, q] + ([c] if clock_grad else []), g.to(DEV))
    rp, rc, rq = (x.double().requires_grad_() for x in (path, clock, w))
    if structure == "planes":
        A = torch.block_diag(*[torch.stack([torch.stack([r[0], r[1]]), torch.stack([-r[1], r[0]])]) for r in rq])
    else:
        A = torch.diag(rq)
    mode = {"per_interval": "displacement", "cached": "displacement_uniform"}[flow]
    ref = O.ews(rp, rc, A, N, readout, leaf="plane_closed" if structure == "planes" else "diag_closed",
                reweighting_mode=mode, terminal_reduce="assoc")
    want = torch.autograd.grad(ref, [rp, rq] + ([rc] if clock_grad else []), g.double())
    errs = [_rel(out, ref)] + [_rel(a, b) for a, b in zip(got, want)]
    print(f"{structure} d={d} N={N} B={B} L={L} {readout} chunk={chunk} errs={['%.1e' % e for e in errs]}", flush=True)
    assert errs[0] < 1e-5, errs
    assert errs[1] < (1e-2 if bf16 else 1e-4) and max(errs[2:]) < 1e-4, errs


def _steps(L, lo, hi, seed=0):
    return np.random.default_rng(seed).uniform(lo, hi, L)


@pytest.mark.parametrize("structure,d,N", [("planes", 6, 2), ("planes", 16, 2), ("planes", 20, 2), ("planes", 24, 2),
                                           ("planes", 10, 1), ("real_diag", 5, 2), ("real_diag", 12, 2),
                                           ("real_diag", 32, 2)])
@pytest.mark.parametrize("damp", [(0.01, 1.0), (3.0, 6.0)])
def test_small_steps(structure, d, N, damp):
    # 2 max|u| h: 0.4 at |u| = 6.7 and h = 0.03; damping above 3 contracts a 16-step chunk by more than ln 2 / 2
    L = 83
    _check(structure, d, N, 2, L, _steps(L, 0.002, 0.028), damp)


@pytest.mark.parametrize("structure,d", [("planes", 16), ("planes", 12), ("real_diag", 9)])
def test_every_class_in_one_call(structure, d):
    L = 4 * 64 + 64 + 9
    s = np.full(L, 2.0**-8)  # uniform chunks
    s[1 + 64:1 + 128] = _steps(64, 0.001, 0.01)  # small steps
    s[1 + 192:1 + 256] = _steps(64, 0.05, 0.6)  # steps outside the radius
    s[1 + 230] = 0.0
    for chunk in (64, 16):
        _check(structure, d, 2, 2, L, s, (0.01, 1.0), chunk=chunk)


@pytest.mark.parametrize("readout", ["terminal", "mean", "max"])
def test_small_steps_readouts(readout):
    _check("planes", 8, 2, 2, 70, _steps(70, 0.002, 0.02), (0.01, 1.0), readout=readout)


@pytest.mark.parametrize("d", [16, 18])
def test_small_steps_bf16_path(d):
    _check("planes", d, 2, 2, 70, _steps(70, 0.002, 0.02), (0.01, 1.0), bf16=True)


def test_small_steps_cached_flow():
    _check("planes", 6, 2, 2, 70, _steps(70, 0.002, 0.02), (0.01, 1.0), flow="cached")


@pytest.mark.parametrize("structure,d,N", [("planes", 16, 2), ("planes", 12, 2), ("planes", 24, 2), ("planes", 10, 1),
                                           ("real_diag", 9, 2), ("real_diag", 5, 1)])
@pytest.mark.parametrize("sign", [1.0, -1.0])
def test_clock_that_turns(structure, d, N, sign):
    """A clock that turns inside a chunk: its net step is near zero, but the states contract by e^11 on the way (sign
    -1: a growing generator on a clock that starts backwards), so that the steps cannot be inverted from the chunk's
    end. The loss sees the first rows only, or all of them."""
    s = sign * np.r_[0.0, np.full(32, 0.17), np.full(32, -0.17), _steps(60, 0.1, 0.17)]
    for rows in (8, None):
        _check(structure, d, N, 2, len(s), s, sorted((0.9 * sign, sign)), chunk=64, freq=0.2, rows=rows)


@pytest.mark.parametrize("structure,d", [("planes", 16), ("planes", 12), ("planes", 24), ("real_diag", 9)])
@pytest.mark.parametrize("unit", [2.0**-20, 2.0**26, 2.0**13])
@pytest.mark.parametrize("regular", [False, True])
def test_units_of_the_clock(structure, d, unit, regular):
    """The same problem with the clock in other units: steps near 1e-8 or 1e6, generators near 1e6 or 1e-8, whose powers
    leave the float32 range where h u does not."""
    L = 83
    s = np.full(L, 2.0**-6) if regular else _steps(L, 0.002, 0.028)
    _check(structure, d, 2, 2, L, s * unit, (0.01 / unit, 1.0 / unit), freq=3.0 / unit, clock_grad=not regular)


def test_suited_chunk_lengths():
    """The library's choice: 64 intervals where there are many, 16 where few, 0 on the sequential kernels, and an
    error code (never a choice) for a descriptor it refuses."""
    lib = nat.load()

    def suited(B, L, d, structure=nat.STRUCT_PLANES, chunk=0, readout="prefix"):
        return lib.ews_diag_suited_chunk(ctypes.byref(ops.make_desc(
            B, L, d, 2, structure, nat.FLOW_PER_INTERVAL, readout, True, nat.DTYPE_F32, chunk)))

    assert suited(32, 17984, 16) == 64 and suited(2, 1500, 16) == 16 and suited(8, 49920, 24) == 64
    assert suited(1, 3000, 24) == 16 and suited(8, 1024, 8, nat.STRUCT_REAL_DIAG) == 64
    assert suited(256, 512, 32, nat.STRUCT_REAL_DIAG, readout="log_prefix") == 0
    assert suited(2, 100, 16, chunk=40) == 40
    assert suited(2, 100, 34) < 0


@pytest.mark.parametrize("structure,d", [("planes", 10), ("real_diag", 5)])
@pytest.mark.parametrize("chunk", [16, 64])
def test_depth1_rows_before_missing_values(structure, d, chunk):
    """Recordings padded with NaN at depth 1, the loss on rows before the padding: the path's and the clock's gradients
    there are those of the recordings cut before it."""
    rng = np.random.default_rng(8)
    B, L, cut, seen = 2, 64, 45, 40
    path = torch.tensor(np.cumsum(rng.normal(size=(B, L, d)) * 0.3, 1), dtype=torch.float32)
    path[:, cut:] = float("nan")
    clock = torch.tensor(np.cumsum(rng.uniform(0.001, 0.02, size=(B, L)), 1), dtype=torch.float32).to(DEV)
    w = torch.tensor(rng.uniform(0.01, 0.4, size=(d // 2, 2) if structure == "planes" else d), dtype=torch.float32)
    g = torch.tensor(rng.normal(size=(B, seen, 1 + d)), dtype=torch.float32).to(DEV)
    res = []
    for n in (L, cut):
        p, c = path[:, :n].to(DEV).requires_grad_(), clock[:, :n].clone().requires_grad_()
        out = ops.diag_scan(p, c, w.to(DEV), 1, structure, "per_interval", "prefix", True, chunk=chunk)
        res.append(torch.autograd.grad((out[:, :seen] * g).sum(), [p, c]))
    (gp, gc), (wp, wc) = res
    errs = [_rel(gp[:, :cut], wp.cpu()), _rel(gc[:, :cut - 1], wc[:, :cut - 1].cpu())]
    print(structure, chunk, errs)
    assert errs[0] < 1e-5 and errs[1] < 1e-5, errs
