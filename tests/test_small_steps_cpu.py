"""The small-step polynomials of the coefficients (csrc/ews_numerics.h) on the host against divided differences of exp
by their Taylor sums in float64, up to the radius that the kernels admit. Bars: a few float32 roundings for the values
and their d/dh, plus the remainders of degrees 6 and 7 at the radius (2e-8 of the value, 1e-7 of a node derivative)."""

import ctypes
import math
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "exponentially-weighted-signature_amd", "csrc")


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    out = tmp_path_factory.mktemp("shim") / "libsmallstep.so"
    subprocess.check_call(["g++", "-O2", "-shared", "-fPIC", "-I", CSRC, "-o", str(out),
                           os.path.join(HERE, "native", "smallstep_shim.cpp")])
    lib = ctypes.CDLL(str(out))
    lib.shim_radius.restype = lib.shim_max.restype = ctypes.c_float
    lib.shim_small.argtypes = [ctypes.c_float, ctypes.c_float]
    return lib


def _ptr(a):
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_float))


def _f(z):
    return np.ascontiguousarray(np.stack([z.real, z.imag], -1).astype(np.float32))


def _hom(m, nodes):
    """Complete homogeneous polynomial of degree m."""
    if len(nodes) == 1:
        return nodes[0] ** m
    return sum(nodes[-1] ** i * _hom(m - i, nodes[:-1]) for i in range(m + 1))


def _dd(nodes):
    """exp[0, nodes..] = sum_m h_m(nodes) / (m + len(nodes))!."""
    return sum(_hom(m, nodes) / math.factorial(m + len(nodes)) for m in range(22))


@pytest.mark.parametrize("share", [1e-3, 0.3, 1.0])
def test_values_and_step_derivatives(shim, share):
    rng = np.random.default_rng(int(share * 1000))
    n, R = 60, shim.shim_radius() * share
    u = rng.uniform(0.2, 1.0, n) * np.exp(1j * rng.uniform(0, 2 * np.pi, n))
    v = u + rng.uniform(0.2, 1.0, n) * np.exp(1j * rng.uniform(0, 2 * np.pi, n))
    h = np.full(n, R / 2)  # 2 max|u| |h| at the radius
    u, v, h = u.astype(np.complex64), v.astype(np.complex64), h.astype(np.float32)
    out = np.zeros((n, 8), np.float32)
    shim.shim_poly(n, _ptr(h), _ptr(_f(u)), _ptr(_f(v)), _ptr(out))
    got = out[:, 0::2] + 1j * out[:, 1::2]
    for i in range(n):
        x, y, ui, vi = complex(h[i] * u[i]), complex(h[i] * v[i]), complex(u[i]), complex(v[i])
        ref = [_dd([x]), _dd([x, x]) * ui, _dd([x, y]), _dd([x, x, y]) * ui + _dd([x, y, y]) * vi]
        for k, bar in enumerate((3e-7, 5e-7, 3e-7, 1e-6)):
            assert abs(got[i, k] - ref[k]) <= bar * max(1.0, abs(ref[k])), (i, k, got[i, k], ref[k])


def test_node_cotangents_through_moments(shim):
    rng = np.random.default_rng(5)
    n = 64
    u, v = np.complex64(-0.6 + 0.8j), np.complex64(-1.0 + 1.7j)
    h = (rng.uniform(0.0, 1.0, n) * shim.shim_radius() / 2).astype(np.float32)
    g = (rng.normal(size=n) + 1j * rng.normal(size=n)).astype(np.complex64)
    out = np.zeros(6, np.float32)
    shim.shim_moments(n, _ptr(h), _ptr(_f(g)), _ptr(_f(np.array([u]))), _ptr(_f(np.array([v]))), _ptr(out))
    got = out[0::2] + 1j * out[1::2]
    ref = [0, 0, 0]
    for hi, gi in zip(h.astype(np.float64), g.astype(np.complex128)):
        x, y = hi * complex(u), hi * complex(v)
        for k, d in enumerate((_dd([x, x]), _dd([x, x, y]), _dd([x, y, y]))):
            ref[k] += hi * gi * np.conj(d)
    size = float(np.sum(h * np.abs(g)))
    for k in range(3):  # float32 sums of 64 terms: 64 roundings of the summed magnitudes at most
        assert abs(got[k] - ref[k]) <= 64 * 6e-8 * size, (k, got[k], ref[k])


@pytest.mark.parametrize("side", [0, 1])
def test_at_the_bounds_of_u_and_h(shim, side):
    """At the largest generator with its steps, and at the largest step with its generators: the values and the node
    cotangents are those of the same h u in moderate units; past either bound the model is refused."""
    R = shim.shim_radius()
    U, H = (shim.shim_max(0), R / 2 / shim.shim_max(0)) if side == 0 else (R / 2 / shim.shim_max(1), shim.shim_max(1))
    assert shim.shim_small(U * (1 - 1e-6), H * (1 - 1e-6))
    assert not shim.shim_small(U * (1.01 if side == 0 else 1.0), H / 2 if side == 0 else H * 1.01)
    assert not shim.shim_small(float("nan"), H) and not shim.shim_small(U, float("nan"))
    rng = np.random.default_rng(9)
    n, k = 40, 2.0 ** (round(math.log2(U)))  # a power of two: the same problem in moderate units
    u = (U * np.exp(1j * rng.uniform(0, 2 * np.pi, n))).astype(np.complex64)
    v = (2 * U * np.exp(1j * rng.uniform(0, 2 * np.pi, n))).astype(np.complex64)
    h = (rng.uniform(0.1, 1.0, n) * H).astype(np.float32)
    g = (rng.normal(size=n) + 1j * rng.normal(size=n)).astype(np.complex64)
    outs = []
    for f in (1.0, k):
        uf, vf, hf = (u / f).astype(np.complex64), (v / f).astype(np.complex64), (h * f).astype(np.float32)
        a, b = np.zeros((n, 8), np.float32), np.zeros(6, np.float32)
        shim.shim_poly(n, _ptr(hf), _ptr(_f(uf)), _ptr(_f(vf)), _ptr(a))
        shim.shim_moments(n, _ptr(hf), _ptr(_f(g)), _ptr(_f(uf[:1])), _ptr(_f(vf[:1])), _ptr(b))
        a = a.reshape(n, 4, 2) * np.array([1.0, f, 1.0, f])[None, :, None]  # d/dh scales with u
        outs.append((a, b / f))
    for x, y in zip(*outs):
        assert np.isfinite(x).all() and np.max(np.abs(x - y)) <= 1e-6 * np.max(np.abs(y))
