"""Mixer epilogue forward at the row counts where c_down goes into LDS (every CU a full workgroup of row tiles) and just
below, ragged last tiles, depths 1 to 3, one to four hidden tiles, against the float64 oracle (forward bar 1e-5)."""

import pytest
import torch

import ews_mi355x as E
from oracle import mixer_oracle as MO

pytestmark = pytest.mark.gpu

DEV = "cuda"


@pytest.mark.parametrize("d,N,hidden,B,R", [(5, 1, 3, 1, 65536), (5, 2, 24, 2, 32767), (5, 2, 24, 3, 21851),
                                            (3, 3, 40, 2, 40003), (17, 2, 33, 1, 65545), (4, 2, 64, 7, 9999)])
@pytest.mark.parametrize("basepoint", [False, True])
def test_forward(d, N, hidden, B, R, basepoint):
    torch.manual_seed(d + R)
    m = E.MixerEpilogue(d, N, hidden, graded_prescale="binomial" if d == 5 else None, basepoint=basepoint).to(DEV)
    x = torch.randn(B, R, 1 + m.D)
    x[..., 0] = 1.0
    got = m(x.to(DEV)).detach().cpu().double()
    W, b, g = (v.detach().cpu().double() for v in (m.c_down.weight, m.c_down.bias, m.graded.gains))
    ref = MO.mixer_epilogue(x.double(), W, b, d, N, "live_rms", m.graded.eps, gains=g, lam=None, basepoint=basepoint,
                            prescale=d == 5)
    assert got.shape == ref.shape
    err = float((got - ref).abs().max() / ref.abs().max())
    print(f"d={d} N={N} hidden={hidden} B={B} R={R} {err:.1e}", flush=True)
    assert err < 1e-5
