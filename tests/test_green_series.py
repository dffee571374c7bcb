"""The series of the Green function away from the origin (izh_field.hip,
igf_far): the mean of 1/r over a cell as the Taylor series of 1/r averaged over
the cell, up to derivatives of the source's order, from the source's distance on.

A term of order 2n adds at most (|s|/r)^2n P_2n over the cell's points s, so at
rho half diagonals the truncated terms come to at most the sum of
rho^-2n / (2n + 1): the mean of |s|^2n over a box is largest, 1 / (2n + 1) of
its half diagonal's power, where the box is a needle.  Checked in extended
precision against a 20-point Gauss rule per axis (its own error: below 5e-16)."""
import itertools
import math
import os
import re

import numpy as np
import pytest

from conftest import ROOT

SRC = open(os.path.join(ROOT, "impact-z_amd", "csrc", "izh_field.hip")).read()
ORDER = int(re.search(r"constexpr int kIgfOrder = (\d+);", SRC).group(1))
FAR = float(re.search(r"constexpr double kIgfFar = ([\d.]+);", SRC).group(1))
LD = np.longdouble


def derivative(orders):
    """d^(orders) 1/r = P(x, y, z) / r^m: (P as {exponents: coefficient}, m)."""
    p, m = {(0, 0, 0): 1}, 1
    for axis, times in enumerate(orders):
        for _ in range(times):
            q = {}
            for e, c in p.items():
                up = list(e)
                up[axis] += 1
                q[tuple(up)] = q.get(tuple(up), 0) - m * c
                if e[axis]:
                    for other in range(3):
                        f = list(e)
                        f[axis] -= 1
                        f[other] += 2
                        q[tuple(f)] = q.get(tuple(f), 0) + e[axis] * c
            p, m = q, m + 2
    return p, m


TERMS = [(n, *derivative([2 * k for k in n]))
         for n in itertools.product(range(ORDER + 1), repeat=3) if sum(n) <= ORDER]


def series(x, y, z, h):
    r = np.sqrt(x * x + y * y + z * z)
    out = np.zeros_like(r)
    for n, p, m in TERMS:
        w = LD(1)
        for a in range(3):
            w *= LD(h[a]) ** (2 * n[a]) / (LD(4) ** n[a] * math.factorial(2 * n[a] + 1))
        poly = sum(c * x ** e[0] * y ** e[1] * z ** e[2] for e, c in p.items() if c)
        out += w * poly / r ** m
    return out


def cell_mean(x, y, z, h):
    t, w = np.polynomial.legendre.leggauss(20)
    t, w = t.astype(LD) / 2, w.astype(LD) / 2
    out = np.zeros_like(x)
    for i, j in itertools.product(range(20), repeat=2):
        rho2 = (x + t[i] * h[0]) ** 2 + (y + t[j] * h[1]) ** 2
        zz = z[:, None] + t[None, :] * h[2]
        out += w[i] * w[j] * np.sum(w / np.sqrt(rho2[:, None] + zz * zz), axis=1)
    return out


@pytest.mark.parametrize("h", [(1, 1, 0.2), (1, 1, 1), (1, 1, 4), (1, 4, 16), (0.7, 1, 2.5),
                               (1, 1, 30), (1, 30, 30)])
def test_series_is_the_cell_mean(h):
    h = np.array(h, dtype=LD)
    half = np.sqrt(np.sum(h * h)) / 2
    d = np.abs(np.random.default_rng(3).normal(size=(60, 3)))
    d = np.vstack([d, np.eye(3), np.ones((1, 3)), [[1, 1, 0], [0, 1, 1], [1, 0, 1]]]).astype(LD)
    d /= np.linalg.norm(d.astype(float), axis=1)[:, None]
    for far in (FAR, 2 * FAR, 64.0):
        bound = 5e-16 + sum(far ** (-2 * n) / (2 * n + 1) for n in range(ORDER + 1, ORDER + 8))
        p = d * far * half
        want = cell_mean(p[:, 0], p[:, 1], p[:, 2], h)
        got = series(p[:, 0], p[:, 1], p[:, 2], h)
        assert np.max(np.abs(got / want - 1)) < bound, far
