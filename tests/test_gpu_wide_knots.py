"""Van Loan leaf on wide dense generators at the edges of the knot tiles (one knot, a part of a tile, whole tiles, three and
four of them), on the series path and off it (large steps) and with the shared pair, against the float64 oracle: forward
1e-5, gradients 1e-4."""

import numpy as np
import pytest
import torch

from ews_mi355x import ops
from oracle import ews_oracle as O

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _check(d, N, M, h, mode="displacement", scheme="cayley"):
    rng = np.random.default_rng(d + M)
    B, L = 2, 21
    path = torch.tensor(np.cumsum(rng.normal(size=(B, L, d)) * 0.2, 1), dtype=torch.float32)
    steps = np.full((B, L), h) if mode != "displacement" else rng.uniform(0.5, 1.5, size=(B, L)) * h
    clock = torch.tensor(np.cumsum(steps, 1), dtype=torch.float32)
    A = torch.tensor(0.5 * rng.normal(size=(d, d)) / np.sqrt(d) + np.eye(d), dtype=torch.float32)
    leaf = ops.DenseLeaf("van_loan", M=M, van_loan_expm=scheme, reweighting_mode=mode)
    flow = {"displacement": "per_interval", "displacement_uniform": "cached"}[mode]
    x = [v.to(DEV).requires_grad_() for v in (path, clock, A)]
    out = ops.dense_scan(*x, N, leaf.q, flow, "prefix", True, leaf=leaf)
    g = torch.tensor(rng.normal(size=tuple(out.shape)), dtype=torch.float32)
    got = [out.detach()] + list(torch.autograd.grad(out, x, g.to(DEV)))
    r = [v.double().requires_grad_() for v in (path, clock, A)]
    ref = O.ews(*r, N, "prefix", leaf="van_loan", M=M, van_loan_expm=scheme, terminal_reduce="assoc", reweighting_mode=mode)
    want = [ref.detach()] + list(torch.autograd.grad(ref, r, g.double()))
    errs = [float((a.cpu().double() - b).abs().max() / b.abs().max()) for a, b in zip(got, want)]
    print(f"d={d} N={N} M={M} h={h} {mode} {scheme} errs={['%.1e' % e for e in errs]}", flush=True)
    assert errs[0] < 1e-5 and max(errs[1:]) < 1e-4, errs


@pytest.mark.parametrize("M", [1, 2, 4, 7, 16, 17, 20, 32, 33, 48, 64])
@pytest.mark.parametrize("N", [1, 2])
def test_series_knots(M, N):
    _check(24, N, M, 0.02)


@pytest.mark.parametrize("d,M", [(17, 5), (32, 21), (20, 64)])
@pytest.mark.parametrize("scheme", ["exact", "pade"])
def test_widths_and_schemes(d, M, scheme):
    _check(d, 2, M, 0.02, scheme=scheme)


@pytest.mark.parametrize("M", [3, 18])
def test_off_the_series_path_and_shared_pair(M):
    _check(19, 2, M, 0.3 * M)
    _check(24, 2, M, 0.02, mode="displacement_uniform")


@pytest.mark.parametrize("mode", ["displacement_uniform", "displacement_uniform_basepoint"])
@pytest.mark.parametrize("M", [3, 20])
def test_zero_shared_step(mode, M):
    """A zero shared step fixes the Van Loan pair to the identity: it adds nothing to the clock's gradient, whatever the
    workspace held before (the rest of that gradient is the flows')."""
    rng = np.random.default_rng(M)
    B, L, d = 3, 7, 21
    path = torch.tensor(np.cumsum(rng.normal(size=(B, L, d)) * 0.2, 1), dtype=torch.float32)
    steps = rng.uniform(0.01, 0.02, size=(B, L))
    steps[1, 1:3] = 0.0
    clock = torch.tensor(np.cumsum(steps, 1), dtype=torch.float32)
    A = torch.tensor(0.5 * rng.normal(size=(d, d)) / np.sqrt(d), dtype=torch.float32)
    leaf = ops.DenseLeaf("van_loan", M=M, van_loan_expm="exact", reweighting_mode=mode)
    flow = {"displacement_uniform": "cached", "displacement_uniform_basepoint": "cached_basepoint"}[mode]
    g = torch.tensor(rng.normal(size=(B, L - 1, d + d * d)), dtype=torch.float32)
    r = [v.double().requires_grad_() for v in (path, clock, A)]
    ref = O.ews(*r, 2, "prefix", leaf="van_loan", M=M, van_loan_expm="exact", terminal_reduce="assoc",
                reweighting_mode=mode)[..., 1:]
    want = torch.autograd.grad(ref, r, g.double())
    for keep in (False, True):
        junk = [torch.full((1 << n,), 1e6, device=DEV) for n in (16, 18, 20, 22, 24) for _ in range(24)]
        del junk
        x = [v.to(DEV).requires_grad_() for v in (path, clock, A)]
        out = ops.dense_scan(*x, 2, leaf.q, flow, "prefix", False, leaf=leaf, keep=keep)
        got = torch.autograd.grad(out, x, g.to(DEV))
        errs = [float((a.cpu().double() - b).abs().max() / b.abs().max()) for a, b in zip(got, want)]
        print(f"{mode} M={M} keep={keep} errs={['%.1e' % e for e in errs]}", flush=True)
        assert max(errs) < 1e-4, errs
