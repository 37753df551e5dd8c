"""The nodes at which the series path sums near lines (radiobear_amd/csrc/far.hpp): a line whose poles
lie on or outside the ellipse of an interval of columns is its Chebyshev interpolant there.  The
error, relative to the line's own value at each column, is evaluated in long double at the kernels'
numbers of nodes and ellipses for the line forms that leave most of it: a narrow Gross line (a = 0, a
near-double pole) and a narrow Ben-Reuven / Van Vleck-Weisskopf line (c = a |p|), with the pole
anywhere on the ellipse and intervals from a few percent wide to four decades.

It stays under one FP32 rounding (2^-24) in FP32 mode and under the ten roundings of an FP64 term
(10 x 2^-53) in FP64 mode."""
import os
import re

import numpy as np
import pytest

LD = np.longdouble
HERE = os.path.dirname(os.path.abspath(__file__))


def kernel_constant(name):
    """{'fp32': a, 'fp64': b} of a `F32 ? a : b` constant."""
    with open(os.path.join(HERE, '..', 'radiobear_amd', 'csrc', 'far.hpp')) as fp:
        m = re.search(re.escape(name) + r'[^;{]*[{=][^;]*?F32 \? ([0-9.]+) : ([0-9.]+);', fp.read())
    assert m, name
    return {'fp32': float(m.group(1)), 'fp64': float(m.group(2))}


def interpolation_error(term, lo, hi, n):
    c, r = (lo + hi) / 2, (hi - lo) / 2
    angle = (2 * np.arange(n, dtype=LD) + 1) * (np.arctan(LD(1)) * 4) / (2 * n)
    value = term(c + r * np.cos(angle))
    coef = [(LD(2) if m else LD(1)) / n * np.sum(value * np.cos(m * angle)) for m in range(n)]
    u = np.linspace(-1, 1, 201).astype(LD)
    b1 = b2 = np.zeros_like(u)
    for m in range(n - 1, 0, -1):
        b1, b2 = 2 * u * b1 - b2 + coef[m], b1
    exact = term(c + r * u)
    return float(np.max(np.abs(u * b1 - b2 + coef[0] - exact) / np.abs(exact)))


def worst(n, rho):
    out = 0.0
    for ratio in (1.032, 1.1, 1.5, 2.0, 4.0, 10.0, 100.0, 1e4):
        hi = LD(100)
        lo = hi / LD(ratio)
        c, r = (lo + hi) / 2, (hi - lo) / 2
        for th in np.linspace(0.0, np.pi, 25):
            z = c + r * (rho * np.exp(1j * th) + np.exp(-1j * th) / rho) / 2
            if z.real < 0:
                continue
            p = np.clongdouble(z) ** 2
            Ds, h = p.real, p.imag ** 2
            if th in (0.0, np.pi):
                h = Ds * Ds * LD(1e-12)   # narrow, not of no width
            for a, k in ((0, 1), (1, np.sqrt(Ds * Ds + h))):
                out = max(out, interpolation_error(lambda f: (a * f * f + k) / ((f * f - Ds) ** 2 + h), lo, hi, n))
    return out


@pytest.mark.parametrize('mode,bound', [('fp32', 2.0 ** -24), ('fp64', 10 * 2.0 ** -53)])
def test_nodes_within_a_terms_roundings(mode, bound):
    n = int(kernel_constant('constexpr int nodes')[mode])
    assert worst(n, kernel_constant('node_rho()')[mode]) < bound
