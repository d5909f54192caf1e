"""The flow step kernel over the run lengths and lane splits its host rule can choose: a flow alone
(short runs, 32 lanes per integral), in a crowd (long runs, 8 lanes, several passes) and against the
oracle.  The node sums are one tree whatever the split, so results are the same bits; against the
oracle 300 steps of a contracting flow carry a few roundings per step (1e-12 absolute of values < 5).
"""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _serve(gpu, qp, flows, nx, n_steps):
    fs = gpu.FlowServer(qp, hbm_budget=1 << 24, max_resident=96, nx=nx, n_steps=n_steps, k_end=0.3,
                        steps_per_launch=25)
    # grid spacing 0.1: the explicit steps' stability limit goes with its square
    ids = [fs.submit(n, T, rho_max=0.1 * (n - 1)) for n, T in flows]
    while fs.progress()[0]:
        pass
    out = [fs.result(i)[0] for i in ids]
    fs.close()
    return out


# the smallest grids, lengths that do not divide into the runs, and the largest grid; nodes below, at and
# past a chunk of 64
@pytest.mark.parametrize("nx", [3, 64, 65, 130])
def test_flow_bits_do_not_depend_on_the_cut(gpu, qp, nx):
    flows = [(4, 0.2), (5, 0.05), (7, 0.3), (64, 0.1), (65, 0.02), (129, 0.15), (1024, 0.25)]
    crowd = flows + [(300 + 13 * i, 0.02 + 0.005 * i) for i in range(50)]
    print(f"[case] flows alone and among {len(crowd)}, nx={nx}", flush=True)
    mix = _serve(gpu, qp, crowd, nx, 50)
    few = _serve(gpu, qp, flows + [(700, 0.1), (900, 0.2)], nx, 50)
    for i, f in enumerate(flows):
        alone = _serve(gpu, qp, [f], nx, 50)[0]
        assert np.array_equal(alone, mix[i]) and np.array_equal(alone, few[i]), f


@pytest.mark.parametrize("n,T,nx", [(4, 0.2, 64), (5, 0.01, 64), (97, 0.3, 64), (97, 0.05, 7), (200, 0.1, 100),
                                    (4096, 0.1, 64)])
def test_flow_edges_vs_oracle(gpu, qp, n, T, nx):
    steps = 300 if n < 1000 else 40
    print(f"[case] flow n={n} T={T} nx={nx}, {steps} steps", flush=True)
    rho_max = 4.0 if n < 100 else 0.1 * (n - 1)
    fs = gpu.FlowServer(qp, hbm_budget=1 << 24, max_resident=2, nx=nx, n_steps=steps, k_end=0.3, steps_per_launch=25)
    i = fs.submit(n, T, rho_max=rho_max)
    while fs.progress()[0]:
        pass
    u = fs.result(i)[0]
    fs.close()
    ref = O.flow_lpa(O.flow_params(n, rho_max, T, 0.0, 4.0, 0.2, 1.0), qp.get_points(nx), qp.get_weights(nx), 20.0, 1.0,
                     0.3, steps)
    assert np.max(np.abs(u - ref)) <= 1e-12
