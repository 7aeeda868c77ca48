"""The chain adjoint's two sources of a step's states (inverted steps, or states recomputed from the chunk's carry when
it contracts too strongly), every reach of the phi series, chunk edges and the reference-step clock shares, against the
float64 oracle's exact integrals at depth 1. Bars as the repository's: forward 1e-5, gradients 1e-4."""

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


def _generator(kind, size, K, rates, seed):
    rng = np.random.default_rng(seed)
    A = torch.zeros(K * size, K * size, dtype=torch.float64)
    for j in range(K):
        f = j * size
        a, b = rates[j % len(rates)], rng.uniform(-3, 3)
        if kind == "real":
            A[f:f + size, f:f + size] = a * torch.eye(size) + torch.diag(torch.ones(size - 1), 1)
        else:
            k = size // 2
            A[f:f + size, f:f + size] = torch.block_diag(*[torch.tensor([[a, -b], [b, a]])] * k) + torch.diag(
                torch.ones(size - 2), 2)
    return A.float()


@pytest.mark.parametrize("kind,size,K", [("real", 1, 5), ("real", 2, 3), ("real", 4, 4), ("complex", 2, 4),
                                         ("complex", 4, 4), ("complex", 6, 2), ("complex", 8, 2)])
@pytest.mark.parametrize("rates,step", [((0.3, 0.01), 1e-4),   # 7 terms, inverted
                                        ((0.4,), 0.03),        # 13 terms, inverted
                                        ((0.2, 1.5), 0.5),     # 28 terms; chunks of 32 not inverted
                                        ((0.05, 9.0), 0.4)])   # the recurrence beyond |x| = 2, strong contraction
def test_states_and_series_reach(kind, size, K, rates, step):
    rng = np.random.default_rng(K + size)
    d, B = K * size, 2
    for L, chunk in ((72, 32), (20, 0), (2, 0), (35, 1)):
        path = torch.tensor(np.cumsum(rng.normal(size=(B, L, d)) * 0.3, 1), dtype=torch.float32)
        clock = torch.tensor(np.cumsum(rng.uniform(0.0, 2 * step, size=(B, L)), 1), dtype=torch.float32)
        A = _generator(kind, size, K, rates, 3)
        p, c, a = (x.to(DEV).requires_grad_() for x in (path, clock, A))
        out = ops.chain_scan(p, c, a, kind, size, chunk=chunk)
        g = torch.tensor(rng.normal(size=tuple(out.shape)), dtype=torch.float32)
        gp, gc, _ = torch.autograd.grad(out, [p, c, a], g.to(DEV))
        rp, rc = path.double().requires_grad_(), clock.double().requires_grad_()
        ref = O.ews(rp, rc, A.double(), 1, "prefix", leaf="exact")
        wp, wc = torch.autograd.grad(ref, [rp, rc], g.double())
        errs = [_rel(out, ref), _rel(gp, wp), _rel(gc, wc)]
        print(f"{kind} {size} K={K} rates={rates} step={step} L={L} chunk={chunk}: {['%.1e' % e for e in errs]}")
        assert errs[0] < 1e-5 and errs[1] < 1e-4 and errs[2] < 1e-4, errs


@pytest.mark.parametrize("chunk", [1, 2, 8])
def test_reference_step_shares(chunk):
    """Cached flows and leaf: every interval at theta1 - theta0, whose clock gradient lands on knots 0 and 1."""
    rng = np.random.default_rng(4)
    B, L, d = 2, 19, 8
    path = torch.tensor(np.cumsum(rng.normal(size=(B, L, d)) * 0.3, 1), dtype=torch.float32)
    clock = torch.tensor(np.cumsum(rng.uniform(0.02, 0.05, size=(B, L)), 1), dtype=torch.float32)
    A = _generator("complex", 2, 4, (0.3, 0.8), 5)
    for flow, mode in (("cached", "displacement_uniform"), ("cached_basepoint", "displacement_uniform_basepoint")):
        p, c, a = path.to(DEV).requires_grad_(), clock.to(DEV).requires_grad_(), A.to(DEV)
        out = ops.chain_scan(p, c, a, "complex", 2, flow, flow, chunk=chunk)
        g = torch.tensor(rng.normal(size=tuple(out.shape)), dtype=torch.float32)
        gp, gc = torch.autograd.grad(out, [p, c], g.to(DEV))
        rp, rc = path.double().requires_grad_(), clock.double().requires_grad_()
        ref = O.ews(rp, rc, A.double(), 1, "prefix", leaf="van_loan", M=4, van_loan_expm="exact",
                    reweighting_mode=mode, terminal_reduce="assoc")
        wp, wc = torch.autograd.grad(ref, [rp, rc], g.double())
        errs = [_rel(out, ref), _rel(gp, wp), _rel(gc, wc)]
        print(flow, chunk, errs)
        assert errs[0] < 1e-5 and errs[1] < 1e-4 and errs[2] < 1e-4, errs


@pytest.mark.parametrize("kind,size,K", [("real", 1, 5), ("real", 2, 3), ("complex", 2, 4), ("complex", 4, 4)])
@pytest.mark.parametrize("chunk", [0, 32, 64])
def test_rows_before_missing_values(kind, size, K, chunk):
    """Recordings padded with NaN, the loss on rows before the padding: the path's and the clock's gradients there are
    those of the recordings cut before it (the states before a step never come from a chunk's end that is not finite)."""
    rng = np.random.default_rng(8)
    B, L, cut, seen = 2, 64, 45, 40
    path = torch.tensor(np.cumsum(rng.normal(size=(B, L, K * size)) * 0.3, 1), dtype=torch.float32)
    path[:, cut:] = float("nan")
    clock = torch.tensor(np.cumsum(rng.uniform(0.0, 0.02, size=(B, L)), 1), dtype=torch.float32).to(DEV)
    A = _generator(kind, size, K, (0.3, 0.01), 3).to(DEV)
    g = torch.tensor(rng.normal(size=(B, seen, 1 + K * size)), dtype=torch.float32).to(DEV)
    res = []
    for n in (L, cut):
        p, c = path[:, :n].to(DEV).requires_grad_(), clock[:, :n].clone().requires_grad_()
        out = ops.chain_scan(p, c, A, kind, size, chunk=chunk)
        res.append(torch.autograd.grad((out[:, :seen] * g).sum(), [p, c]))
    (gp, gc), (wp, wc) = res
    errs = [_rel(gp[:, :cut], wp.cpu()), _rel(gc[:, :cut - 1], wc[:, :cut - 1].cpu())]
    print(kind, size, chunk, errs)
    assert errs[0] < 1e-5 and errs[1] < 1e-5, errs
