"""The threshold and finite-T batches at the sizes where their work split changes, against the oracle.

Tolerance 1e-13: each term differs from the oracle's by a few roundings (the reciprocal within 1 ulp,
at most five products), and both add positive terms or, near a pole, terms of one sign per node.
"""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

TOL = 1e-13


# register tiles of 64, 128 and 256 nodes and the loop beyond them; groups of eight integrals, one
# wave, one block of 16 waves, and more groups than resident waves
@pytest.mark.parametrize("nx", [1, 2, 63, 64, 65, 128, 129, 256, 257, 600])
@pytest.mark.parametrize("n,k,d", [(1, 1.0, 4), (7, 1e-3, 2), (8, 30.0, 7), (9, 1.0, 3), (1025, 0.2, 5),
                                   (33003, 1.0, 4)])
def test_threshold_sizes(gpu, qp, nx, n, k, d):
    if n > 5000 and nx > 257:
        n = 5001
    m2 = np.random.default_rng(n + nx).uniform(-0.9, 4.0, n) * k * k
    x, w = qp.get_points(nx), qp.get_weights(nx)
    ref = O.c0_threshold(m2, x, w, 20.0, k, 1.0, d)
    d_m2, d_x, d_w = (gpu.DeviceArray.from_host(a) for a in (m2, x, w))
    out = gpu.DeviceArray.from_host(np.full(n + 9, -1.0))
    for mode in (gpu.FP64, gpu.MIXED):
        print(f"[case] threshold n={n} nx={nx} k={k} d={d} mode={mode}", flush=True)
        gpu.threshold_batch(d_m2, d_x, d_w, out, 20.0, k, mode, d)
        got = out.to_host()
        assert np.all(got[n:] == -1.0)  # nothing past the last integral
        assert np.abs(got[:n] / ref - 1).max() <= TOL


# both sides of the batch size at which the kernel changes; the first integrals of a larger batch are the same
# bits as alone, in either kernel
@pytest.mark.parametrize("nx,limit", [(7, 4096), (64, 4096), (100, 4096), (256, 4096), (257, 7680), (600, 7680),
                                      (1024, 7680)])
def test_threshold_bits_across_the_kernels(gpu, qp, nx, limit):
    m2 = np.random.default_rng(nx).uniform(-0.9, 4.0, limit + 13)
    x, w = qp.get_points(nx), qp.get_weights(nx)
    ref = O.c0_threshold(m2, x, w, 20.0, 1.0, 1.0, 4)
    d_x, d_w = (gpu.DeviceArray.from_host(a) for a in (x, w))
    for mode in (gpu.FP64, gpu.MIXED):
        res = []
        for n in (5, limit, limit + 1, limit + 13):
            print(f"[case] threshold n={n} nx={nx} mode={mode}", flush=True)
            out = gpu.DeviceArray(n)
            gpu.threshold_batch(gpu.DeviceArray.from_host(m2[:n]), d_x, d_w, out, 20.0, 1.0, mode, 4)
            res.append(out.to_host())
            assert np.abs(res[-1] / ref[:n] - 1).max() <= TOL
        for r in res[:-1]:
            assert np.array_equal(r, res[-1][:len(r)])


def test_threshold_special_masses(gpu, qp):
    # infinite masses give 0, NaN gives NaN; a neighbour in the same group of eight is not touched
    x, w = qp.get_points(33), qp.get_weights(33)
    m2 = np.array([0.5, np.inf, np.nan, 1e300, -np.inf, 0.5, 0.25, 0.5, 0.5])
    d_m2, d_x, d_w = (gpu.DeviceArray.from_host(a) for a in (m2, x, w))
    out = gpu.DeviceArray(len(m2))
    print("[case] threshold special masses", flush=True)
    gpu.threshold_batch(d_m2, d_x, d_w, out, 20.0, 1.0, gpu.FP64, 4)
    got = out.to_host()
    ref = O.c0_threshold(np.array([0.5, 0.25]), x, w, 20.0, 1.0, 1.0, 4)
    assert np.all(got[[1, 3, 4]] == 0.0) and np.isnan(got[2])
    assert np.abs(got[[0, 5, 7, 8]] / ref[0] - 1).max() <= TOL and abs(got[6] / ref[1] - 1) <= TOL


# Matsubara rules around the 64-lane chunk and the powers of two of a last chunk's lane split; nx
# around the waves' radial strides; scales k far from 1
@pytest.mark.parametrize("nm", [1, 2, 3, 5, 16, 17, 31, 32, 33, 64, 65, 66, 96, 97, 130])
@pytest.mark.parametrize("nx,k,radial_mode", [(1, 1.0, 1), (37, 1e-3, 0), (64, 1e18, 1), (65, 1e-20, 0),
                                              (1024, 1.0, 1)])
def test_finite_T_sizes(gpu, qp, nm, nx, k, radial_mode):
    rng = np.random.default_rng(nm + nx)
    n, d = 9, 4
    T = k * rng.choice([0.05, 0.1, 0.3], n)
    T[3] = 0.0  # no zero mode
    p0 = 2 * np.pi * T * rng.integers(0, 5, n)
    pabs = 2.0 * k * rng.random(n)
    m1, m2 = k * k * rng.uniform(-0.5, 3, n), k * k * rng.uniform(-0.5, 3, n)
    lens = np.array([nm, max(1, nm - 1), nm + 1])
    off = np.concatenate([[0], np.cumsum(lens)[:-1]])
    rules = [(2 * np.pi * 0.1 * k * np.arange(1, m + 1), np.full(m, 0.1 * k)) for m in lens]
    sel = rng.integers(0, 3, n)
    x, w = qp.get_points(nx), qp.get_weights(nx)
    extent = 6.0 * k if radial_mode else 20.0
    ref = O.c2_finiteT(T, p0, pabs, m1, m2, [rules[s] for s in sel], x, w, extent, k, 1.0, d, radial_mode)
    A = gpu.DeviceArray.from_host
    dev = {"T": A(T), "p0": A(p0), "pabs": A(pabs), "m1": A(m1), "m2": A(m2),
           "mx": A(np.concatenate([r[0] for r in rules])), "mw": A(np.concatenate([r[1] for r in rules])),
           "m_off": A(off[sel].astype(np.int32)), "m_n": A(lens[sel].astype(np.int32)), "x": A(x), "w": A(w)}
    out = gpu.DeviceArray(n)
    try:
        for block in (0, 64, 256):
            gpu.ft_set_block(block)
            for mode in (gpu.FP64, gpu.MIXED):
                print(f"[case] finite-T nm={nm} nx={nx} k={k} block={block} mode={mode}", flush=True)
                gpu.ft_batch(dev, out, extent, k, mode, d, radial_mode)
                assert np.abs(out.to_host() / ref - 1).max() <= TOL
    finally:
        gpu.ft_set_block(0)


def _ft(gpu, T, p0, pabs, m1, m2, rules, x, w, extent, k, d, radial_mode, block, tol=TOL):
    """ft_batch in both modes against the oracle: finite values to `tol`, zeros, infinities and NaNs alike."""
    T, p0, pabs, m1, m2 = np.broadcast_arrays(*(np.asarray(a, float) for a in (T, p0, pabs, m1, m2)))
    # the oracle adds the zero mode beside its first node: a node of weight 0 where there is none
    with np.errstate(all="ignore"):
        ref = O.c2_finiteT(T, p0, pabs, m1, m2, [r if len(r[0]) else (np.ones(1), np.zeros(1)) for r in rules],
                           x, w, extent, k, 1.0, d, radial_mode)
    lens = np.array([len(r[0]) for r in rules], np.int32)
    off = np.concatenate([[0], np.cumsum(lens)[:-1]]).astype(np.int32)
    pad = np.ones(1)  # the concatenation may be empty
    A = gpu.DeviceArray.from_host
    dev = {"T": A(T), "p0": A(p0), "pabs": A(pabs), "m1": A(m1), "m2": A(m2),
           "mx": A(np.concatenate([r[0] for r in rules] + [pad])),
           "mw": A(np.concatenate([r[1] for r in rules] + [pad])),
           "m_off": A(off), "m_n": A(lens), "x": A(x), "w": A(w)}
    out = gpu.DeviceArray(len(T))
    try:
        gpu.ft_set_block(block)
        for mode in (gpu.FP64, gpu.MIXED):
            print(f"[case] finite-T k={k} nx={len(x)} radial_mode={radial_mode} block={block} mode={mode}", flush=True)
            gpu.ft_batch(dev, out, extent, k, mode, d, radial_mode)
            got = out.to_host()
            fin = np.isfinite(ref) & (ref != 0)
            assert np.array_equal(got[~fin], ref[~fin], equal_nan=True), (got, ref)
            assert np.all(np.abs(got[fin] / ref[fin] - 1) <= tol), np.abs(got / ref - 1)
    finally:
        gpu.ft_set_block(0)


# the direction every flow runs: k falls while temperature, momenta and masses stay (products of three
# denominators over k^2 leave the FP32 range near k = 1e-6); and masses that stay where k grows
@pytest.mark.parametrize("k", [1e-3, 1e-5, 3e-6, 1e-6, 1e-8, 1e-15, 1e6])
@pytest.mark.parametrize("radial_mode", [0, 1])
@pytest.mark.parametrize("block", [0, 64])
def test_finite_T_scale_against_fixed_masses(gpu, qp, k, radial_mode, block):
    rng = np.random.default_rng(5)
    n = 8
    T = np.array([0.05, 0.1, 0.3, 0.0, 0.1, 2.0, 0.1, 0.3])
    rules = [(2 * np.pi * max(t, 0.1) * np.arange(1, m + 1), np.full(m, max(t, 0.1)))
             for t, m in zip(T, (64, 96, 17, 48, 3, 66, 130, 33))]
    m1, m2 = rng.uniform(0.01, 3, n), rng.uniform(0.01, 3, n)
    m1[4], m2[4] = 1e4, 1e-4
    extent = 6.0 * k if radial_mode else 20.0
    _ft(gpu, T, 2 * np.pi * T * rng.integers(0, 5, n), rng.uniform(0, 1, n), m1, m2, rules, qp.get_points(48),
        qp.get_weights(48), extent, k, 4, radial_mode, block)


@pytest.mark.parametrize("block", [0, 64, 512])
@pytest.mark.parametrize("k", [1.0, 1e-40, 1e40])
def test_finite_T_huge_masses(gpu, qp, k, block):
    # masses past the range of a product of denominators, infinite and NaN ones: 0, the small value or NaN, and
    # ordinary neighbours beside them; scales k where such products leave the FP64 range altogether
    k2 = k * k
    m1 = np.array([0.5, 1.0, 1.0, 1.0, 1.0, 1e60, np.inf, np.nan, 1.0, 1e60, -0.5]) * k2
    m2 = np.array([0.5, 1e120 / k2, 1e160 / k2, np.inf, np.nan, 1.0, 1.0, 1.0, -np.inf, 1e110, 0.25]) * k2
    n = len(m1)
    T = np.where(np.arange(n) % 2, 0.1, 0.0) * k
    rules = [(2 * np.pi * 0.1 * k * np.arange(1, m + 1), np.full(m, 0.1 * k))
             for m in (64, 65, 5, 130, 1, 33, 64, 2, 17, 64, 66)]
    _ft(gpu, T, 0.3 * k, 0.7 * k, m1, m2, rules, qp.get_points(37), qp.get_weights(37), 20.0, k, 4, 0, block)


@pytest.mark.parametrize("block", [0, 256])
def test_finite_T_huge_external_and_frequencies(gpu, qp, block):
    p0 = np.array([0.3, 1e80, 1e120, np.inf, 0.3, 0.3, 0.3])
    pabs = np.array([0.7, 0.7, 0.7, 0.7, 1e90, np.inf, 0.7])
    rules = [(np.geomspace(1e-3, top, m), np.full(m, 0.1)) for top, m in
             ((10.0, 64), (10.0, 65), (10.0, 64), (10.0, 33), (10.0, 5), (10.0, 64), (1e95, 130))]
    _ft(gpu, 0.1, p0, pabs, 0.5, 0.25, rules, qp.get_points(37), qp.get_weights(37), 20.0, 1.0, 4, 0, block)


@pytest.mark.parametrize("block", [0, 64])
def test_finite_T_vanishing_denominators(gpu, qp, block):
    # one radial node at q^2 = 49, whose regulator e^-49 is below a rounding, so the masses cancel q^2 exactly:
    # a zero d1 in the zero mode, a zero d2 there and in a frequency pair: infinite, as by three divisions
    x, w = np.array([0.98]), np.array([1.0])
    q2 = float(np.sqrt(0.98 * 50.0) ** 2)
    assert q2 + np.exp(-q2) == q2
    rules = [(np.array([0.5, 2.0]), np.array([0.1, 0.1]))] * 5
    T = np.array([0.1, 0.1, 0.0, 0.0, 0.1])
    p0 = np.array([0.3, 0.0, 2.0, 0.3, 0.3])
    m1 = np.array([-q2, 0.5, 0.5, -q2, 0.5])
    m2 = np.array([0.25, -q2, -q2, 0.25, 0.25])
    _ft(gpu, T, p0, 0.0, m1, m2, rules, x, w, 50.0, 1.0, 4, 0, block)


@pytest.mark.parametrize("block", [0, 64])
@pytest.mark.parametrize("nx", [1, 48])
def test_finite_T_zero_mode_alone(gpu, qp, nx, block):
    # integrals without Matsubara nodes: the zero mode, or nothing at T = 0.  (The lanes' share of such a rule
    # is a static_assert beside the kernel.)
    T = np.array([0.1, 0.0, 0.3])
    rules = [(np.zeros(0), np.zeros(0))] * 2 + [(np.array([1.0]), np.array([0.3]))]
    _ft(gpu, T, 0.3, 0.7, 0.5, 0.25, rules, qp.get_points(nx), qp.get_weights(nx), 20.0, 1.0, 4, 0, block)
