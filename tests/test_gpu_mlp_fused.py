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
# with 33, 48 or 64 features between them (forward layer by layer but for the large
# batch with few inputs and outputs, gradients fused)
@pytest.mark.parametrize("dims,n", [((6, 256, 35), 63), ((6, 256, 35), 64), ((32, 33, 16), 65),
                                    ((33, 128, 129, 3), 128), ((256, 65, 256), 129),
                                    ((5, 7), 200), ((256, 256), 70), ((6, 64, 35), 65),
                                    ((6, 48, 8), 65535), ((6, 48, 8), 65536),
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


def _bf16(v):
    u = np.ascontiguousarray(v, np.float32).view(np.uint32)
    return (((u + 0x7fff + ((u >> 16) & 1)) >> 16) << 16).astype(np.uint32).view(np.float32)


def _pair(a):
    """hi + lo, the two BF16 terms that an activation is kept in."""
    a = np.float32(a)
    h = _bf16(a)
    return h.astype(np.float64) + _bf16(a - h)


def test_silu_error(gpu):
    """SiLU of the fused kernel, read back through a last layer that is the identity:
    weights 0 and bias z in the first.  The pair of BF16 terms hides an error unless
    it moves a value over a rounding boundary, so z are taken whose exact SiLU lies
    between 1.27e-7 (the stated error for z > 0 is 1.25e-7) and 1.8e-7 from one,
    relative: all of them come out as the exact value's pair.  Large arguments keep
    their limits."""
    from geosmie_amd import _lib
    from geosmie_amd.surrogate import MLP
    dims, w = (1, 256, 256), 256
    p = np.zeros(O.layout(dims)[1], np.float32)
    (_, b0, _, _), (w1, _, _, _) = O.layout(dims)[0]
    p[w1:w1 + w * w] = np.eye(w, dtype=np.float32).ravel()
    x = _lib.to_dev(np.ones((1, 1)), np.float32)

    def run(z):
        p[b0:b0 + w] = z
        return MLP(dims, params=p).forward(x).cpu().numpy()[0].astype(np.float64)

    def silu(z):
        return z / (1.0 + np.exp(-z.astype(np.float64)))
    z = np.linspace(0.05, 10.0, 1 << 21).astype(np.float32)
    exact = silu(z)
    near = lambda r: np.stack([_pair(exact * (1.0 + f * r)) == _pair(exact) for f in (-1, 1)])
    z = z[near(1.27e-7).all(0) & ~near(1.8e-7).all(0)]
    assert z.size >= 64 * w
    z = z[np.linspace(0, z.size - 1, 64 * w).astype(int)]
    got = np.concatenate([run(c) for c in z.reshape(-1, w)])
    assert np.array_equal(got, _pair(silu(z)))
    z = np.linspace(-80.0, 80.0, w).astype(np.float32)
    assert np.all(np.abs(run(z) - silu(z)) <= (2.0 ** -17 + 3e-6) * np.abs(silu(z)))
    z = np.resize(np.float32([-3e38, -1e4, -104.0, -88.0, 0.0, 104.0, 1e4, 3e38]), w)
    got = run(z)
    assert np.all(np.abs(got - np.maximum(z, 0)) <= 2.0 ** -17 * np.maximum(z, 0) + 1e-35)
    z[3] = np.nan
    assert np.isnan(run(z)).all()
