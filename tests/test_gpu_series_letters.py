"""Depth-3 series local terms: stages of the letters (orders about multiples of twelve), a generator so large that the
powers A^m / m! leave the float32 range while h A stays moderate, and steps so large that those of h do (a clock in raw
seconds), against the float64 oracle (bar 1e-5). Steps have h ||A||_1 above 0.48: within it the cayley flow itself is a
series in those powers, which a large A overflows."""

import numpy as np
import pytest
import torch

from ews_mi355x import ops
from oracle import ews_oracle as O

pytestmark = pytest.mark.gpu

DEV = "cuda"


@pytest.mark.parametrize("q", [1, 4, 11, 12, 13, 16, 24, 25, 36, 40])
@pytest.mark.parametrize("scale", [1.0, 2e4, 4e-2, 4e-4, 1e-4, 1e-6])
def test_letters(q, scale):
    rng = np.random.default_rng(q)
    d, L = 7, 9
    path = torch.tensor(np.cumsum(rng.normal(size=(2, L, d)) * 0.3, 1), dtype=torch.float32)
    clock = torch.tensor(np.cumsum(rng.uniform(0.6, 0.9, size=(2, L)) / scale, 1), dtype=torch.float32)
    A = torch.tensor((rng.normal(size=(d, d)) / np.sqrt(d) + np.eye(d)) * scale, dtype=torch.float32)
    assert float((clock[:, 1:] - clock[:, :-1]).min() * A.abs().sum(0).max()) > 0.48
    leaf = ops.DenseLeaf("series", q=q, chen_expm="cayley")  # rational flows: no power of A in them
    out = ops.dense_scan(path.to(DEV), clock.to(DEV), A.to(DEV), 3, q, "per_interval", "prefix", True, leaf=leaf)
    ref = O.ews(path.double(), clock.double(), A.double(), 3, "prefix", leaf="series", series_q=q, chen_expm="cayley",
                terminal_reduce="assoc")
    assert bool(torch.isfinite(out).all())
    err = float((out.cpu().double() - ref).abs().max() / ref.abs().max())
    print(f"q={q} scale={scale} {err:.1e}", flush=True)
    assert err < 1e-5


@pytest.mark.parametrize("q", [1, 12, 24, 40])
@pytest.mark.parametrize("scale", [1.0, 2e4, 4e-4, 1e-4])
def test_gradients_in_units_of_the_clock(q, scale):
    rng = np.random.default_rng(q)
    d, L = 5, 7
    path = torch.tensor(np.cumsum(rng.normal(size=(2, L, d)) * 0.3, 1), dtype=torch.float32)
    clock = torch.tensor(np.cumsum(rng.uniform(0.6, 0.9, size=(2, L)) / scale, 1), dtype=torch.float32)
    A = torch.tensor((rng.normal(size=(d, d)) / np.sqrt(d) + np.eye(d)) * scale, dtype=torch.float32)
    leaf = ops.DenseLeaf("series", q=q, chen_expm="cayley")
    p, c, a = (x.to(DEV).requires_grad_() for x in (path, clock, A))
    out = ops.dense_scan(p, c, a, 3, q, "per_interval", "prefix", True, leaf=leaf)
    g = torch.tensor(rng.normal(size=tuple(out.shape)), dtype=torch.float32)
    got = torch.autograd.grad(out, [p, c, a], g.to(DEV))
    r = [x.double().requires_grad_() for x in (path, clock, A)]
    ref = O.ews(*r, 3, "prefix", leaf="series", series_q=q, chen_expm="cayley", terminal_reduce="assoc")
    want = torch.autograd.grad(ref, r, g.double())
    errs = [float((x.cpu().double() - y).abs().max() / y.abs().max()) for x, y in zip(got, want)]
    print(f"q={q} scale={scale} {['%.1e' % e for e in errs]}", flush=True)
    assert max(errs) < 1e-4, errs
