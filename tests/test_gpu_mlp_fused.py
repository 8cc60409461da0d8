"""Fused network kernels (gm_mlp.hip) at the edges of their tiles, and the
direct row output against forward + gm_surrogate_post.

Tolerances as in test_gpu_mlp.py (two-term BF16 activations against FP64).  The
direct rows apply the same formulas to the same outputs: a few ulp of FP32.
"""
import numpy as np
import pytest

from oracle import mlp as O

pytestmark = pytest.mark.gpu


def _setup(dims, n):
    from geosmie_amd.surrogate import init_params
    rng = np.random.default_rng(n + sum(dims))
    p = init_params(dims, n)
    for _, b, _, n_out in O.layout(dims)[0]:
        p[b:b + n_out] = rng.uniform(-0.3, 0.3, n_out)
    x = rng.standard_normal((n, dims[0])).astype(np.float32)
    t = rng.standard_normal((n, dims[-1])).astype(np.float32)
    return p, x, t, rng.uniform(0.5, 2.0, dims[-1]).astype(np.float32)


# rows around one and two 64-row blocks; widths at and past the 16-, 32-, 64- and
# 128-feature splits of the wavefronts; 257 (layer by layer), and one layer and two
# with 33 or 64 features between them (forward layer by layer, gradients fused)
@pytest.mark.parametrize("dims,n", [((6, 256, 35), 63), ((6, 256, 35), 64), ((32, 33, 16), 65),
                                    ((33, 128, 129, 3), 128), ((256, 65, 256), 129),
                                    ((5, 7), 200), ((256, 256), 70), ((6, 64, 35), 65),
                                    ((32, 33, 20, 16), 65), ((5, 7, 7, 7), 200),
                                    ((6, 257, 4), 65)])
def test_tile_edges_vs_oracle(gpu, dims, n):
    from geosmie_amd import _lib
    from geosmie_amd.surrogate import MLP
    p, x, t, cw = _setup(dims, n)
    f = lambda a: _lib.to_dev(a, np.float32)
    mlp = MLP(dims, params=p, weight_terms=2)
    y = mlp.forward(f(x)).cpu().numpy()
    ref = O.forward(p, dims, x, terms=2)
    assert np.max(np.abs(y - ref)) <= 2e-4 * np.abs(ref).max()
    loss = float(mlp.grad(f(x), f(t), f(cw)).item())
    g = mlp.g.cpu().numpy().astype(np.float64)
    lref, gref = O.loss_grad(p, dims, x, t, cw, terms=2)
    assert abs(loss - lref) <= 1e-4 * abs(lref)
    for w, b, _, n_out in O.layout(dims)[0]:
        for lo, hi in ((w, b), (b, b + n_out)):
            assert np.linalg.norm(g[lo:hi] - gref[lo:hi]) <= 2e-3 * np.linalg.norm(gref[lo:hi])


@pytest.mark.parametrize("hidden,n,baseline", [((256,), 65, True), ((40,), 130, False),
                                               ((40, 40), 130, False), ((300,), 65, True)])
def test_rows_match_forward_and_post(gpu, hidden, n, baseline):
    import torch
    from geosmie_amd import _lib
    from geosmie_amd._lib import ptr
    from geosmie_amd.surrogate import MLP, make_queries
    dims = (6, *hidden, 35)
    p, x, _, _ = _setup(dims, n)
    rng = np.random.default_rng(n)
    q = make_queries(rng.uniform(0.01, 5, n), rng.uniform(1.4, 2.6, n), rng.uniform(1.3, 1.8, n),
                     rng.uniform(1e-6, 1, n), rng.uniform(0.2, 40, n), rng.uniform(1, 2, n))
    f = lambda a: _lib.to_dev(a, np.float32)
    d_x, d_q = f(x), f(q)
    mean, std = f(rng.uniform(-1, 1, 35)), f(rng.uniform(0.1, 1, 35))
    mlp = MLP(dims, params=p)
    y = mlp.forward(d_x)
    want, got = torch.empty_like(y), torch.empty_like(y)
    L, h, s = _lib.lib(), _lib.ctx(), _lib.stream()
    dq = ptr(d_q) if baseline else None
    _lib.check(L.gm_surrogate_post(h, n, 35, dq, 1.33, ptr(y), ptr(mean), ptr(std), ptr(want), s))
    _lib.check(L.gm_surrogate_rows(h, mlp.n_layers, mlp._cd, n, ptr(mlp.p), ptr(d_x), dq, 1.33,
                                   ptr(mean), ptr(std), ptr(got), s))
    # exp(t + ln B) with |t + ln B| < 30: 2 ulp of its argument
    np.testing.assert_allclose(got.cpu().numpy(), want.cpu().numpy(), rtol=4e-6, atol=1e-7)
