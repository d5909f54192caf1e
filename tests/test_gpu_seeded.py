"""The seeded FP64 form of the self-energy batch (table-driven log and exp, hardware reciprocal and
reciprocal-square-root estimates) against the oracle's library-call arithmetic, at the edges of what
its rule admits, and next to integrals that the rule leaves to the general form.

Tolerance 1e-13: every evaluation differs from the oracle's by a few roundings (each log, exp, root
and reciprocal within 1 ulp, the table index by 255 roundings of slope <= |dZ|), and both sums add
up to 64*64*1024 positive terms in FP64 pairwise per lane, wave and tile (a few tens of eps).
"""
import os
import tempfile

import numpy as np
import pytest

from diffrg_amd import isa_count as I
from oracle import oracle as O

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
TOL = 1e-13


@pytest.mark.gpu
@pytest.mark.parametrize("start,stop,bias", [(1e-3, 40.0, 6.0), (1e-3, 40.0, 0.01), (1e-3, 40.0, 11.0), (1e-3, 40.0, 1.99),
                                             (1e-30, 3.0, 6.0), (0.5, 8.0, 2.0), (0.09, 40.0, 6.0)])
@pytest.mark.parametrize("k", [1.0, 0.03])  # bias 0.01 and 1.99: the general form, on the rule's other side
def test_seeded_fp64_matches_oracle(gpu, qp, start, stop, bias, k):
    rng = np.random.default_rng(3)
    n_tab = [2, 3, 31, 32, 255, 256, 64, 128]
    nq = [1, 3, 64, 129, 17, 64, 300, 16]
    na = [2, 64, 8, 16, 32, 4, 8, 64]
    # p = 0, on the table's ends, far outside, and where |p - q| passes near 0
    p = [0.0, start, stop, 3 * stop, k, 2.5 * k, 0.7 * k, 4.4 * k]
    tables = [1.0 + 0.5 * np.tanh(rng.uniform(-2, 2, n)) for n in n_tab]
    xq = [(qp.get_points(v), qp.get_weights(v)) for v in nq]
    xa = [(qp.get_points(v), qp.get_weights(v)) for v in na]
    coords = [O.logcoord(n, start, stop, bias) for n in n_tab]
    ref = O.c1_selfenergy(p, tables, coords, xq, xa, 20.0, k)
    out = gpu.DeviceArray(len(p))
    b = gpu.SEBatch(qp, p, nq, na, tables, start, stop, bias, x_extent=20.0, k=k)
    for block, tile, grid in ((256, 8192, 0), (64, 1024, 0), (1024, 65536, 0), (512, 4096, 16)):
        b.set_shape(block, tile, grid)
        print(f"[case] seeded start={start} bias={bias} k={k} block={block} grid={grid}", flush=True)
        b.run(out, gpu.FP64)
        err = np.abs(out.to_host() / ref - 1)
        print(f"  max rel err {err.max():.2e}", flush=True)
        assert err.max() <= TOL


@pytest.mark.gpu
def test_general_fp64_beside_seeded(gpu, qp):
    # a falling coordinate map, a log argument that turns negative at y = 0, an infinite table value
    # and start 0 keep the general form; one such integral sends the whole batch to the kernel that
    # holds both forms, where the seeded integrals give the same bits as alone
    rng = np.random.default_rng(4)
    z = 1.0 + 0.5 * np.tanh(rng.uniform(-2, 2, 48))
    zinf = z.copy()
    zinf[-1] = np.inf
    start = np.array([1e-3, 1e-3, 1.0, 1e-3, 0.0, 1e-3])
    stop = np.array([40.0, 40.0, 2.0, 40.0, 40.0, 40.0])
    bias = np.array([6.0, -2.0, 6.0, 6.0, 6.0, 6.0])
    tables = [z, z.copy(), z.copy(), zinf, z.copy(), z.copy()]
    p = np.array([1.0, 0.5, 3.0, 2.0, 1e-3, 7.0])
    xq = [(qp.get_points(32), qp.get_weights(32))] * 6
    xa = [(qp.get_points(16), qp.get_weights(16))] * 6
    coords = [O.logcoord(48, a, b, c) for a, b, c in zip(start, stop, bias)]
    ref = O.c1_selfenergy(p, tables, coords, xq, xa, 20.0, 1.0)
    out, one = gpu.DeviceArray(6), gpu.DeviceArray(1)
    print("[case] general and seeded FP64 forms in one batch", flush=True)
    gpu.SEBatch(qp, p, 32, 16, tables, start, stop, bias).run(out, gpu.FP64)
    got = out.to_host()
    assert np.abs(got / ref - 1).max() <= TOL
    for i in range(6):
        gpu.SEBatch(qp, p[i:i + 1], 32, 16, tables[i:i + 1], start[i], stop[i], bias[i]).run(one, gpu.FP64)
        assert one.to_host()[0] == got[i]


@pytest.mark.gpu
def test_seeded_and_unroll_queries(gpu, qp):
    z = np.linspace(1.0, 1.5, 48)
    start = np.array([1e-3, 1e-3, 0.0, 1e-3])
    bias = np.array([6.0, 1.0, 6.0, 2.0])
    tables = [z.copy() for _ in bias]
    b = gpu.SEBatch(qp, np.ones(4), 32, 16, tables, start, 40.0, bias)
    assert list(b.seeded) == [True, False, False, True]
    # the kernel that holds both FP64 forms takes one radial node per step
    assert b.unroll(gpu.FP64) == 1 and b.unroll(gpu.MIXED) == 2
    thin = gpu.SEBatch(qp, np.ones(4), 32, 16, tables, 1e-3, 40.0, 6.0)
    assert thin.seeded.all() and thin.unroll(gpu.FP64) == thin.unroll(gpu.MIXED) == 2
    thick = gpu.SEBatch(qp, np.ones(300), 64, 64, [z] * 300, 1e-3, 40.0, 6.0)
    assert thick.unroll(gpu.FP64) == thick.unroll(gpu.MIXED) == 1


@pytest.mark.skipif(not os.path.exists(I.B.HIPCC), reason="hipcc not found")
def test_seeded_loop_counts_match_bench():
    import bench
    with tempfile.TemporaryDirectory() as d:
        loops = I.inner_loops(I.compile_asm(os.path.join(ROOT, "diffrg_amd", "csrc", "integrals.hip"), d))
    # kSeededOnly kernels: two transcendental instructions per evaluation; with unroll 2 a paired loop of
    # four evaluations comes first
    for block, unroll, want in ((256, 1, ["pairs", "single"]), (512, 2, ["pairs2", "pairs", "single"])):
        body = [c for n, c in loops if f"se_kernelILi2ELi{block}ELi{unroll}E" in n and c["trans"] in (4, 8)]
        body.sort(key=lambda c: (-c["trans"], c["lds"]))
        assert len(body) == len(want)
        for kind, c in zip(want, body):
            evals = c["trans"] // 2
            assert bench.SE_OPS["seeded"][kind] == (c["flop"] / evals, c["valu"] / evals), (kind, c)
