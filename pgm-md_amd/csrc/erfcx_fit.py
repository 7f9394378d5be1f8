"""The coefficients of the pair kernels' polynomials in device.hpp, highest degree first (Horner order).

erfcxFast  exp(x^2) erfc(x) = t Q(t), t = 1/(1 + x/2), x in [0, 4.5], with Q of degree 8 fitted for the least maximum
           relative error by iteratively reweighted least squares (Lawson's method) on Chebyshev nodes in t, in FP32.
ErfcxD     (x + K) exp(x^2) erfc(x) over x >= 0 as a polynomial of degree 24 in u = (x - K)/(x + K), K = 2.5: its
           Chebyshev series (60 nodes, 60 digits) cut there and written in powers of u, in FP64 (the mapping of
           Shepherd and Laframboise, Math. Comp. 36, 249, 1981).
ExpD       exp(r) for |r| <= ln 2 / 2: 1 + r + r^2/2 + r^3 q(r), q the Chebyshev series of degree 8 of
           (exp(r) - 1 - r - r^2/2)/r^3 (40 nodes), in FP64.
Prints the coefficients and the polynomials' maximum relative errors.

    python pgm-md_amd/csrc/erfcx_fit.py
"""

import mpmath as mp
import numpy as np
from scipy.special import erfcx

DEG, XMAX, NODES, ITERS = 8, 4.5, 4000, 60


def fit():
    t0 = 1.0 / (1.0 + XMAX / 2.0)
    k = np.arange(NODES)
    t = 0.5 * (1.0 + t0) + 0.5 * (1.0 - t0) * np.cos(np.pi * (k + 0.5) / NODES)
    f = erfcx(2.0 * (1.0 / t - 1.0)) / t
    w = np.ones_like(f)
    best = None
    V = np.vander(t, DEG + 1)
    for _ in range(ITERS):
        c, *_ = np.linalg.lstsq(V * (w / f)[:, None], w, rcond=None)
        rel = (V @ c - f) / f
        m = np.abs(rel).max()
        if best is None or m < best[0]:
            best = (m, c.copy())
        w = w * (1.0 + 5.0 * np.abs(rel) / m)
    return best


def chebyshev(f, nodes, degree):
    """The Chebyshev series of f on [-1, 1] from that many nodes, cut at degree, in powers: lowest first."""
    theta = [mp.pi * (k + mp.mpf(1) / 2) / nodes for k in range(nodes)]
    values = [f(mp.cos(a)) for a in theta]
    out = [mp.mpf(0)] * (degree + 1)
    lower, power = [mp.mpf(0)], [mp.mpf(1)]  # T_{j-1}, T_j
    for j in range(degree + 1):
        c = (2 if j else 1) * sum(v * mp.cos(j * a) for v, a in zip(values, theta)) / nodes
        for k, v in enumerate(power):
            out[k] += c * v
        following = [mp.mpf(0)] + [(2 if j else 1) * v for v in power]
        if j:
            for k, v in enumerate(lower):
                following[k] -= v
        lower, power = power, following
    return out


def fit_erfcx64(K=2.5, degree=24):
    with mp.workdps(60):
        K = mp.mpf(K)

        def scaled(x):
            return mp.exp(x * x) * mp.erfc(x)

        c = chebyshev(lambda u: scaled(K * (1 + u) / (1 - u)) * (K * (1 + u) / (1 - u) + K), 60, degree)
        grid = [mp.mpf(k) / 16 for k in range(16 * 27)]
        err = max(abs(mp.polyval(c[::-1], (x - K) / (x + K)) / (x + K) / scaled(x) - 1) for x in grid)
        return float(err), [float(v) for v in c[::-1]]


def fit_exp64(degree=8):
    with mp.workdps(60):
        h = mp.log(2) / 2

        def tail(v):
            r = v * h
            return (mp.exp(r) - 1 - r - r * r / 2) / r**3 if abs(r) > mp.mpf(10) ** -15 else mp.mpf(1) / 6

        c = [v / h**j for j, v in enumerate(chebyshev(tail, 40, degree))]
        c = [mp.mpf(1), mp.mpf(1), mp.mpf(1) / 2] + c
        grid = [h * (mp.mpf(k) / 200 - 1) for k in range(401)]
        err = max(abs(mp.polyval(c[::-1], r) / mp.exp(r) - 1) for r in grid)
        return float(err), [float(v) for v in c[::-1]]


if __name__ == "__main__":
    for name, (err, c), digits in (("erfcxFast", fit(), 9), ("ErfcxD", fit_erfcx64(), 17), ("ExpD", fit_exp64(), 17)):
        if name == "erfcxFast":
            c = c.astype(np.float32)
        print(name + ": " + ", ".join(f"{v:.{digits}e}" for v in c))
        print(f"max relative error of the polynomial: {err:.2e}")
