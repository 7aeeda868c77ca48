"""The depth-1 cached scan with a sample's steps split over wavefronts, and the chain-structured token cache, against the
float64 oracle: every block size, step counts around the span edges, masks with padding at the end and inside, caches too
large to stage, and the gradients to the tokens' increments and steps and to the chain parameters. Bars as the
repository's: forward 1e-5, gradients 1e-4."""

import numpy as np
import pytest
import torch

import ews_mi355x as E
from oracle import token_oracle as TO

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _rel(a, b):
    a, b = a.detach().cpu().double(), b.detach().double()
    return float((a - b).abs().max() / b.abs().max().clamp_min(1e-300))


def _blocks(rng, V, d, bs):
    D = np.zeros((V, d, d), np.float32)
    for f in range(0, d, bs):
        D[:, f:f + bs, f:f + bs] = 0.8 * np.eye(bs) + 0.1 * rng.normal(size=(V, bs, bs)) / np.sqrt(bs)
    return torch.tensor(D)


@pytest.mark.parametrize("bs,d", [(1, 20), (2, 18), (2, 64), (3, 21), (4, 64), (6, 24), (8, 64)])
@pytest.mark.parametrize("n", [64, 261])
def test_spans_against_the_oracle(bs, d, n):
    rng = np.random.default_rng(bs * 100 + n)
    V, B = 5, 3
    P = torch.tensor(rng.normal(size=(V, d)), dtype=torch.float32)
    D = _blocks(rng, V, d, bs)
    tok = torch.tensor(rng.integers(0, V, size=(B, n)))
    mask = torch.tensor(rng.random((B, n)) > 0.1)
    mask[1, n // 2:] = False
    g = torch.tensor(rng.normal(size=(B, n, d)), dtype=torch.float32)
    p, q = P.to(DEV).requires_grad_(), D.to(DEV).requires_grad_()
    out = E.token_cached_prefix_scan(tok.to(DEV), mask.to(DEV), p, q, d, 1, block=bs)
    gp, gq = torch.autograd.grad(out, [p, q], g.to(DEV))
    rp, rq = P.double().requires_grad_(), D.double().requires_grad_()
    ref = TO.token_cached_prefix_scan_depth1(tok, mask, rp, rq)
    wp, wq = torch.autograd.grad(ref, [rp, rq], g.double())
    on = torch.block_diag(*[torch.ones(bs, bs)] * (d // bs)).double()
    errs = [_rel(out, ref), _rel(gp, wp), _rel(gq, wq * on)]
    print(f"bs={bs} d={d} n={n}: {['%.1e' % e for e in errs]}")
    assert errs[0] < 1e-5 and errs[1] < 1e-4 and errs[2] < 1e-4, errs
    assert float((gq.cpu().double() * (1 - on)).abs().max()) == 0.0


@pytest.mark.parametrize("B", [1, 700])
def test_span_counts_by_batch(B):
    """One to eight wavefronts a sample (by the batch), the same rows and gradients."""
    rng = np.random.default_rng(B)
    d, V, n = 18, 3, 300
    P, D = torch.tensor(rng.normal(size=(V, d)), dtype=torch.float32).to(DEV), _blocks(rng, V, d, 2).to(DEV)
    tok = torch.tensor(rng.integers(0, V, size=(1, n))).to(DEV)
    one = E.token_cached_prefix_scan(tok.expand(5000, n).contiguous(), None, P, D, d, 1, block=2)[:1]  # NW = 1
    many = E.token_cached_prefix_scan(tok.expand(B, n).contiguous(), None, P, D, d, 1, block=2)
    assert _rel(many[:1], one.cpu()) < 2e-6 and torch.equal(many[:1], many[-1:])


@pytest.mark.parametrize("kind,size", [("real", 1), ("real", 3), ("complex", 2), ("complex", 4), ("complex", 8)])
@pytest.mark.parametrize("q", [0, 5])
def test_chain_cache(kind, size, q):
    rng = np.random.default_rng(size + q)
    K = 24 // size
    d, V = K * size, 4
    rate, freq = rng.uniform(0.1, 1.5, K), rng.uniform(-2, 2, K)

    def A_of(r, f):
        blocks = []
        for j in range(K):
            if kind == "real":
                blocks.append(r[j] * torch.eye(size, dtype=r.dtype) + torch.diag(torch.ones(size - 1, dtype=r.dtype), 1))
            else:
                k = size // 2
                R = torch.stack([torch.stack([r[j], -f[j]]), torch.stack([f[j], r[j]])])
                blocks.append(torch.kron(torch.eye(k, dtype=r.dtype), R) +
                              torch.diag(torch.ones(size - 2, dtype=r.dtype), 2))
        return torch.block_diag(*blocks)

    def leaves(dtype):
        return [torch.tensor(x, dtype=torch.float32).to(dtype).requires_grad_()
                for x in (rng2.normal(size=(V, d)), rng2.uniform(0.0, 1.2, V), rate, freq)]

    rng2 = np.random.default_rng(7)
    ref_in = leaves(torch.float64)
    rng2 = np.random.default_rng(7)
    got_in = leaves(torch.float32)
    leaf = dict(leaf="series", series_q=q) if q else dict(leaf="van_loan")
    A = A_of(got_in[2], got_in[3])
    P, D = E.build_token_cache(got_in[0].to(DEV), got_in[1].to(DEV), A.to(DEV), 4, 1, "exact", "exact", chain=(kind, size),
                               **leaf)
    rP, rD = TO.build_token_cache(ref_in[0], ref_in[1], A_of(ref_in[2], ref_in[3]), 4, 1, "exact", "exact", **leaf)
    gP = torch.tensor(rng.normal(size=(V, d)), dtype=torch.float32)
    gD = torch.tensor(rng.normal(size=(V, d, d)), dtype=torch.float32)
    use = got_in if kind == "complex" else got_in[:3]
    got = torch.autograd.grad([P, D], use, [gP.to(DEV), gD.to(DEV)])
    # the chain's gradient lands on the entries it is read from: the parameters', summed over the chain's coordinates
    want = torch.autograd.grad([rP, rD], ref_in if kind == "complex" else ref_in[:3], [gP.double(), gD.double()])
    errs = [_rel(P, rP), _rel(D, rD)] + [_rel(a, b) for a, b in zip(got[:2], want[:2])]
    # A's slots repeat a parameter; the kernels put its whole gradient on the chain's first slot
    errs += [_rel(a, b) for a, b in zip(got[2:], want[2:])]
    print(f"{kind} {size} q={q}: {['%.1e' % e for e in errs]}")
    assert errs[0] < 1e-5 and errs[1] < 1e-5 and max(errs[2:]) < 1e-4, errs


def test_chain_cache_refuses_what_it_cannot_build():
    dx, dth, A = torch.zeros(2, 18), torch.ones(2), torch.eye(18)
    with pytest.raises(RuntimeError, match="HIP device only"):
        E.build_token_cache(dx, dth, A, 4, 1, chain=("real", 1))
    with pytest.raises(ValueError, match="unsupported chain"):
        E.build_token_cache(dx.to(DEV), dth.to(DEV), A.to(DEV), 4, 1, chain=("real", 4))
