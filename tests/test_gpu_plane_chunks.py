"""Uniform clocks on rotation planes of every lane map of the wave-per-chunk kernels (two chunks or one per wavefront,
rows whose pair count is no multiple of four), against the float64 oracle: short and ragged last chunks, chunks that
cannot be stepped backwards, chunks that are uniform only to the looser bound next to strict ones, steps that differ by
as much as they are long within the strict bound, with and without the clock's gradient, rows, log rows and reductions.
Bars as the repository's: forward 1e-5, gradients 1e-4."""

import numpy as np
import pytest
import torch

from ews_mi355x import ops
from oracle import ews_oracle as O

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _rel(a, b):
    a, b = a.detach().cpu().double(), b.detach().double()
    return float((a - b).abs().max() / b.abs().max().clamp_min(1e-300))


def _check(d, B, steps, damp, readout="prefix", chunk=0, bf16=False, clock_grad=True, freq=3.0):
    """steps (L,): the clock's steps (the first is its start). Planes: damping in damp, frequencies in [0, freq]."""
    L = len(steps)
    rng = np.random.default_rng(L + d)
    path = torch.tensor(np.cumsum(rng.normal(size=(B, L, d)) * 0.2, 1), dtype=torch.float32)
    path = path.to(torch.bfloat16) if bf16 else path
    clock = torch.tensor(np.cumsum(steps)[None].repeat(B, 0), dtype=torch.float32)
    w = torch.tensor(np.stack([rng.uniform(*damp, d // 2), rng.uniform(0.0, freq, d // 2)], -1), dtype=torch.float32)
    p, c, q = path.to(DEV).requires_grad_(), clock.to(DEV).requires_grad_(clock_grad), w.to(DEV).requires_grad_()
    out = ops.diag_scan(p, c, q, 2, "planes", "per_interval", readout, readout != "log_prefix", chunk=chunk)
    g = torch.tensor(rng.normal(size=tuple(out.shape)), dtype=torch.float32)
    got = torch.autograd.grad(out, [p, q] + ([c] if clock_grad else []), g.to(DEV))
    rp, rc, rq = (x.double().requires_grad_() for x in (path, clock, w))
    A = torch.block_diag(*[torch.stack([torch.stack([r[0], r[1]]), torch.stack([-r[1], r[0]])]) for r in rq])
    ref = O.ews(rp, rc, A, 2, "prefix" if readout == "log_prefix" else readout, leaf="plane_closed",
                terminal_reduce="assoc")
    if readout == "log_prefix":  # level 1 and level 2 - x (x) x / 2 at the words i < j
        x, S = ref[..., 1:1 + d], ref[..., 1 + d:].unflatten(-1, (d, d))
        i, j = torch.triu_indices(d, d, 1)
        ref = torch.cat([x, S[..., i, j] - 0.5 * x[..., i] * x[..., j]], -1)
    want = torch.autograd.grad(ref, [rp, rq] + ([rc] if clock_grad else []), g.double())
    errs = [_rel(out, ref)] + [_rel(a, b) for a, b in zip(got, want)]
    print(f"d={d} B={B} L={L} {readout} chunk={chunk} errs={['%.1e' % e for e in errs]}", flush=True)
    assert errs[0] < 1e-5, errs
    assert errs[1] < (1e-2 if bf16 else 1e-4) and max(errs[2:]) < 1e-4, errs


def _uniform(L, h):
    return np.r_[0.0, np.full(L - 1, h)]


@pytest.mark.parametrize("d", [6, 8, 10, 14, 18, 20, 24, 26, 32])
@pytest.mark.parametrize("clock_grad", [False, True])
def test_widths(d, clock_grad):
    # h a power of two: every step and running sum is exact, so that each chunk is strict
    _check(d, 3, _uniform(150, 2.0**-9), (0.1, 1.0), clock_grad=clock_grad)


@pytest.mark.parametrize("d,L", [(12, 2), (24, 2), (12, 65), (24, 66), (24, 16 * 4 * 3 + 2)])
@pytest.mark.parametrize("chunk", [0, 4, 64])
def test_lengths(d, L, chunk):
    _check(d, 2, _uniform(L, 2.0**-8), (0.1, 1.0), chunk=chunk, clock_grad=False)


@pytest.mark.parametrize("d", [12, 24])
@pytest.mark.parametrize("h,damp", [(0.25, (0.05, 0.2)), (0.125, (2.0, 4.0)), (2.0**-8, (0.1, 1.0))])
def test_large_and_contractive_steps(d, h, damp):
    # beyond the small-step model's radius, and contracting past what the inverse recursion is used for
    _check(d, 2, _uniform(140, h), damp, clock_grad=False)


@pytest.mark.parametrize("d", [12, 24])
def test_strict_and_loose_chunks(d):
    steps = _uniform(400, 2.0**-9)
    steps[100:200] *= 1.0 + 2e-4 * np.random.default_rng(0).uniform(-1, 1, 100)
    steps[300:330] *= np.random.default_rng(1).uniform(0.2, 3.0, 30)
    _check(d, 2, steps, (0.1, 1.0), clock_grad=False)


def _irregular(L, h, start=0.0):
    return np.r_[start, np.random.default_rng(2).uniform(0.2, 1.8, L - 1) * h]


@pytest.mark.parametrize("d", [8, 12, 16, 24, 32])
@pytest.mark.parametrize("rate,h", [(0.0, 2.0**-4), (1e-5, 2.0**-8), (2e-2, 2e-5)])
def test_steps_that_differ_within_constant_coefficients(d, rate, h):
    # max|u| times the steps' deviation is far below the bound of constant coefficients, the deviation itself 80% of a
    # step: the parameter gradients weigh each step's cotangents with its own length
    _check(d, 2, _irregular(140, h), (0.0, rate), clock_grad=False, freq=rate)


@pytest.mark.parametrize("d", [12, 16, 24])
def test_float32_uniform_clock(d):
    # a uniform clock whose float32 values near 1 leave steps of 2e-5 off by 3e-3 of themselves
    _check(d, 2, _uniform(300, 2.0e-5) + np.r_[0.9, np.zeros(299)], (0.1, 1.0), clock_grad=False)


@pytest.mark.parametrize("d", [8, 24, 32])
@pytest.mark.parametrize("clock_grad", [False, True])
def test_rounding_that_grows_past_the_strict_bound(d, clock_grad):
    # steps of 5e-3 on a clock from 1.5 to 8.5: with max|u| near 3 the chunks miss the strict bound from 2 on
    _check(d, 2, np.r_[1.5, np.full(1400, 5e-3)], (0.1, 1.0), clock_grad=clock_grad)


@pytest.mark.parametrize("d", [12, 24])
@pytest.mark.parametrize("readout", ["log_prefix", "terminal", "mean"])
def test_readouts(d, readout):
    _check(d, 2, _uniform(150, 2.0**-9), (0.1, 1.0), readout=readout, clock_grad=False)


def test_many_groups_and_bf16():
    # 4-interval chunks: 19 groups of the carry scan, more than one block of staged flows
    _check(12, 1, _uniform(1200, 2.0**-10), (0.1, 1.0), chunk=4, clock_grad=False)
    _check(24, 2, _uniform(300, 2.0**-10), (0.1, 1.0), bf16=True, clock_grad=False)
