"""Quadrature rules at the edges of their kernels' loops and lanes, against multi-precision values.

Gauss-Legendre: every node and weight is one rounding of a value with twice FP64's digits: 2 ulp allowed.
Matsubara: the nodes are those of the FP64 matrix, whose entries carry up to four roundings each, and the
Sturm pivots' backward error is of the same form; a relative perturbation eps of every entry moves
an eigenvalue by at most kappa eps with kappa = |z|^T |A| |z| / (lambda z^T z), so 8 kappa eps bounds the
eigenvalue, half of it the node, and twice that (the vector's own perturbation beside) the weight.
"""
import mpmath as mp
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _gl_node(n, x):
    """The Gauss-Legendre node next to x and its weight on [0,1] in 50 digits."""
    z = 2 * mp.mpf(float(x)) - 1
    for _ in range(3):
        p0, p1 = mp.mpf(1), z
        for j in range(2, n + 1):
            p0, p1 = p1, ((2 * j - 1) * z * p1 - (j - 1) * p0) / j
        dp = n * (z * p1 - p0) / (z * z - 1)
        z -= p1 / dp
    return (1 + z) / 2, 1 / ((1 - z * z) * dp * dp)


# below, at and past the 64 roots of a block, the unrolled loops' remainders, and the largest order
@pytest.mark.parametrize("n", [2, 3, 4, 9, 63, 64, 65, 127, 128, 129, 131, 500, 4096])
def test_gl_nodes_to_the_last_digits(gpu, n):
    print(f"[case] gl order {n}", flush=True)
    x, w = gpu.gl_generate(n)
    assert np.all(np.diff(x) > 0) and np.array_equal(w, w[::-1])
    with mp.workdps(50):
        for i in sorted({0, 1, n // 3, (n - 1) // 2, n // 2, n - 1}):
            mx, mw = _gl_node(n, x[i])
            assert abs(x[i] - mx) <= 4.5e-16 * mx, (n, i)
            assert abs(w[i] - mw) <= 4.5e-16 * mw, (n, i)


def test_gl_order_one(gpu):
    print("[case] gl order 1", flush=True)
    x, w = gpu.gl_generate(1)
    assert x[0] == 0.5 and w[0] == 1.0


# a vacuum rule's half length at, past and far past the degrees whose reciprocals are tabulated in LDS (the
# last would need more LDS than a CU has); E = 1/2 maps the lower half onto [0,1] itself
@pytest.mark.parametrize("h", [4096, 4097, 5001, 11000])
def test_long_vacuum_rules(gpu, h):
    print(f"[case] vacuum rule of {2 * h} nodes", flush=True)
    x, w, T = gpu.matsubara_generate(0.0, 0.5, 2, 32, 128, 2 * h, 0)
    assert T == 0.0 and len(x) == 2 * h and np.all(np.diff(x) > 0)
    with mp.workdps(50):
        for i in (0, h // 3, h // 2, h - 1):
            mx, mw = _gl_node(h, x[i])
            assert abs(x[i] - mx) <= 4.5e-16 * mx, (h, i)
            assert abs(w[i] * 2 * mp.pi - mw) <= 9e-16 * mw, (h, i)  # two more roundings
            lx = mp.exp(mp.log(5e5) * mx)
            assert abs(x[h + i] - lx) <= 1e-14 * lx, (h, i)  # 13 roundings of the exponent log(5e5) x, and its own
            lw = mw * mp.log(5e5) * lx
            assert abs(w[h + i] * 2 * mp.pi - lw) <= 1.2e-14 * lw, (h, i)
    qp = gpu.QuadratureProvider(vacuum_quad_size=2 * h)
    assert np.array_equal(qp.get_matsubara_points(0.0, 0.5), x)


# the count's groups of eight steps and their remainders, one and several entries per lane
@pytest.mark.parametrize("n", [1, 2, 3, 8, 9, 10, 17, 32, 64, 65, 128, 200])
def test_matsubara_nodes_against_multiprecision(gpu, n):
    print(f"[case] matsubara n={n}", flush=True)
    T = 0.1
    x, w, _ = gpu.matsubara_generate(T, 1.0, 1, n, n, 48, 1)
    assert len(x) == n and np.all(np.diff(x) < 0)
    # the vector's forward recurrence multiplies a rounding by up to 1e7 per component
    with mp.workdps(60 + 8 * n):
        a = [2 * mp.pi ** 2 / (4 * j + 1) / (4 * j + 5) for j in range(n)]
        a[0] = mp.pi ** 2 / 15
        b = [mp.pi ** 4 / ((4 * j + 3) * (4 * j + 7)) / (4 * j + 5) ** 2 for j in range(n)]
        for k in sorted({0, min(1, n - 1), n // 2, n - 1}):
            lam = (2 * mp.pi * T / mp.mpf(float(x[k]))) ** 2
            for _ in range(3 + (60 + 8 * n).bit_length()):  # Newton on the characteristic polynomial
                p0, p1, d0, d1 = mp.mpf(1), a[0] - lam, mp.mpf(0), mp.mpf(-1)
                for j in range(1, n):
                    p0, p1, d0, d1 = p1, (a[j] - lam) * p1 - b[j - 1] * p0, d1, (a[j] - lam) * d1 - p1 - b[j - 1] * d0
                lam -= p1 / d1
            z = [mp.mpf(1)]  # eigenvector: e_j z_{j+1} = (lam - a_j) z_j - e_{j-1} z_{j-1}
            for j in range(n - 1):
                z.append(((lam - a[j]) * z[j] - (mp.sqrt(b[j - 1]) * z[j - 1] if j else 0)) / mp.sqrt(b[j]))
            s = sum(v * v for v in z)
            kappa = (sum(a[j] * z[j] ** 2 for j in range(n)) +
                     2 * sum(mp.sqrt(b[j]) * abs(z[j] * z[j + 1]) for j in range(n - 1))) / (lam * s)
            tol = 8 * kappa * mp.mpf(2) ** -52
            node, weight = 2 * mp.pi * T / mp.sqrt(lam), T * mp.pi ** 2 / 6 / s / lam
            assert abs(x[k] / node - 1) <= tol / 2, (n, k, float(x[k] / node - 1), float(tol))
            assert abs(w[k] / weight - 1) <= 2 * tol, (n, k, float(w[k] / weight - 1), float(tol))
