"""Van Loan leaf gradients at the edges of the knot adjoint's blocks (full tiles of 16 knots, a padded tile, quads, one
knot, the most knots), depths 1 to 3, against the float64 oracle. Bar as the repository's: gradients 1e-4."""

import numpy as np
import pytest
import torch

from ews_mi355x import ops
from oracle import ews_oracle as O

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _check(B, L, d, N, M, scheme, seed, damp=0.5, spread=1.0):
    rng = np.random.default_rng(seed)
    path = torch.tensor(np.cumsum(rng.normal(size=(B, L, d)) * 0.2, 1), dtype=torch.float32)
    clock = torch.tensor(np.cumsum(rng.uniform(0.02, 0.06, size=(B, L)), 1), dtype=torch.float32)
    A = torch.tensor(spread * rng.normal(size=(d, d)) / np.sqrt(d) + damp * np.eye(d), dtype=torch.float32)
    leaf = ops.DenseLeaf("van_loan", M=M, van_loan_expm=scheme)
    x = [v.to(DEV).requires_grad_() for v in (path, clock, A)]
    out = ops.dense_scan(*x, N, leaf.q, "per_interval", "prefix", True, leaf=leaf)
    g = torch.tensor(rng.normal(size=tuple(out.shape)), dtype=torch.float32)
    got = torch.autograd.grad(out, x, g.to(DEV))
    r = [v.double().requires_grad_() for v in (path, clock, A)]
    ref = O.ews(*r, N, "prefix", leaf="van_loan", M=M, van_loan_expm=scheme, terminal_reduce="assoc")
    want = torch.autograd.grad(ref, r, g.double())
    errs = [float((a.cpu().double() - b).abs().max() / b.abs().max()) for a, b in zip(got, want)]
    print(f"N={N} d={d} M={M} {scheme} errs={['%.1e' % e for e in errs]}", flush=True)
    assert max(errs) < 1e-4, errs


@pytest.mark.parametrize("M", [1, 2, 4, 5, 8, 9, 15, 16, 17, 20, 24, 25, 33, 64])
def test_knot_counts(M):
    _check(2, 7, 16, 3, M, "cayley", M)


@pytest.mark.parametrize("N", [1, 2, 3])
@pytest.mark.parametrize("M", [3, 20, 27])
@pytest.mark.parametrize("scheme", ["cayley", "exact"])
def test_depths_and_padding(N, M, scheme):
    _check(3, 9, 11, N, M, scheme, 40 + M)


def test_more_intervals_than_wavefronts():
    # 2150 intervals on 512 workgroups of four. Every eigenvalue decays (real parts above 1): with the default spread one
    # grows over the 17 units of the clock, rows reach 4e11 and the clock's gradient is a difference of such terms
    _check(5, 431, 4, 3, 6, "cayley", 7, damp=1.5, spread=0.5)
