"""The order in which the FP32 wavefront recurrence adds up a point.

Fitted standing-wave coefficients are large and cancel, so that another order of
the same sums is further from the surface than the rounding of its values, and a
transform of the surface (NIT) whose target law is flat or not monotone makes
visible steps of the difference.  The order is therefore held to the bit, against
its definition carried out here operation by operation on the CPU:

  part[k] = sum of phi(k, i, j) zeta(t - k, x - i, y - j), (i, j) != (0, 0), a chain
            of FMAs from zero in row-major order of (i, j);
  the parts of slices t - P0 + 1 .. t - 1, each closed by the FMA with
  phi(k, 0, 0) zeta(t - k, x, y), and then part[0], added one by one with
  compensation (TwoSum; the errors in a second sum);
  zeta = eps + ((sum + errors) + phi(0, 0, 0) eps).
"""
import numpy as np
import pytest
import torch

import arma_amd
import pyoracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def fma(a, b, c):
    """a b + c of float32 values, rounded once: exact in 64 bits but for the sum,
    whose rounding to odd lets the second rounding decide as the first would."""
    p = a.astype(np.float64) * b.astype(np.float64)
    c = c.astype(np.float64)
    s = p + c
    bb = s - p
    err = (p - (s - bb)) + (c - bb)
    even = (s.view(np.int64) & 1) == 0
    odd = np.where((err != 0) & even, np.nextafter(s, np.copysign(np.inf, err)), s)
    return odd.astype(np.float32)


def defined(eps, phi):
    p0, p1, p2 = phi.shape
    phi = phi.astype(np.float32)
    nt, nx, ny = eps.shape
    z = np.zeros((nt + p0, nx + p1, ny + p2), np.float32)
    T, X, Y = np.indices(eps.shape)
    plane = (T + X + Y).ravel()
    order = np.argsort(plane, kind="stable")
    ends = np.searchsorted(plane[order], np.arange(plane.max() + 2))
    for s in range(plane.max() + 1):
        at = order[ends[s]:ends[s + 1]]
        t, x, y = T.ravel()[at], X.ravel()[at], Y.ravel()[at]
        total = np.zeros(len(at), np.float32)
        errors = np.zeros(len(at), np.float32)
        for k in range(p0 - 1, -1, -1):
            v = np.zeros(len(at), np.float32)
            for m in range(1, p1 * p2):
                i, j = divmod(m, p2)
                v = fma(phi[k, i, j], z[t - k + p0, x - i + p1, y - j + p2], v)
            if k:
                v = fma(phi[k, 0, 0], z[t - k + p0, x + p1, y + p2], v)
            r = total + v
            bb = r - total
            errors = errors + ((total - (r - bb)) + (v - bb))
            total = r
        e = eps[t, x, y]
        z[t + p0, x + p1, y + p2] = e + ((total + errors) + phi[0, 0, 0] * e)
    return z[p0:, p1:, p2:]


def fitted(kind, order, alpha, beta):
    acf = O.acf(kind, (10, 10, 10), velocity=beta, alpha=(alpha,) * 3,
                beta=(beta, beta) if kind == O.STANDING else (-beta, 0.0))
    return O.yw_choi(acf, order)[0]


def drawn(shape):
    phi = np.random.default_rng(2).standard_normal(shape) * (0.3 / np.prod(shape) ** 0.5)
    phi[0, 0, 0] = 0.02
    return phi


@pytest.mark.parametrize("name,phi,shape", [
    ("standing, order 3", lambda: fitted(O.STANDING, 3, 0.06, 0.8), (40, 35, 37)),
    ("standing, order 5", lambda: fitted(O.STANDING, 5, 0.06, 0.8), (24, 35, 37)),
    ("standing, order 7", lambda: fitted(O.STANDING, 7, 0.06, 0.8), (20, 20, 37)),
    ("standing, order 9", lambda: fitted(O.STANDING, 9, 0.07, 0.6), (20, 18, 20)),
    ("propagating, order 7", lambda: fitted(O.PROPAGATING, 7, 0.04, 1.2), (60, 35, 37)),
    ("streamed taps", lambda: drawn((4, 3, 6)), (40, 35, 37)),
    ("one slice", lambda: drawn((1, 4, 4)), (40, 35, 37)),
    ("one column", lambda: drawn((6, 1, 1)), (40, 35, 37)),
], ids=lambda v: v.replace(", ", "-").replace(" ", "-") if isinstance(v, str) else "")
def test_sums_in_their_order(hip_ctx, name, phi, shape):
    phi = phi()
    eps = (np.random.default_rng(9).standard_normal(shape) * 0.1).astype(np.float32)
    z = torch.from_numpy(eps.copy()).to(DEV)
    d = hip_ctx.ar_desc(shape, phi, 1.0, [arma_amd.mt19937_params()],
                        algorithm=arma_amd.AR_WAVEFRONT, precision=arma_amd.FP32)
    hip_ctx.ar_recurrence(d, z)
    np.testing.assert_array_equal(z.cpu().numpy(), defined(eps, phi))
