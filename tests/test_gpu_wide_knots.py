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
