"""Network passes at the edges of their 64-row tiles: one row, a tile less,
whole and more, and batches whose workgroups take several tiles each (256 of
them for the gradients, 768 forward), against the oracle."""
import numpy as np
import pytest

from oracle import mlp_oracle as M

pytestmark = pytest.mark.gpu
F32 = np.float32
# Where GPU and oracle round an operand to bf16 differently it moves by 2^-8;
# the longest chain, to the first layer's weights, goes through six products.
TOL = 6 * 2.0 ** -8


def rel(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30))


def _network(vg, n):
    rng = np.random.default_rng(n)
    p = (M.init_params(12) + 0.05 * rng.standard_normal(M.N_PARAMS)).astype(F32)
    m = vg.Mlp()
    m.set_params(p)
    return rng, p, m, rng.standard_normal((n, M.N_IN)).astype(F32)


@pytest.mark.parametrize("n", [1, 15, 63, 64, 65, 4097, 16384, 16385, 33000])
def test_gradients_of_batch_sizes(vg, n):
    print(f"[case] mlp gradients n={n}", flush=True)
    rng, p, m, X = _network(vg, n)
    T = rng.standard_normal((n, 3)).astype(F32)
    B = rng.standard_normal((n, 3, 3)).astype(F32) if n % 2 else None
    loss, g = m.gradients(vg.DeviceArray.from_numpy(X), vg.DeviceArray.from_numpy(T), n,
                          basis=None if B is None else vg.DeviceArray.from_numpy(B))
    lw, gw = M.backward(p, X, T, emulate_bf16=True, B=B)
    assert abs(loss - lw) < TOL * lw
    o = 0
    for name, shp in M.SHAPES:
        k = int(np.prod(shp))
        assert rel(g[o:o + k], gw[o:o + k]) < TOL, name
        o += k


@pytest.mark.parametrize("n", [1, 63, 64, 65, 49152, 49153, 70001])
@pytest.mark.parametrize("in_place", [False, True])
def test_forward_of_batch_sizes(vg, n, in_place):
    print(f"[case] mlp forward n={n} in place {in_place}", flush=True)
    _, p, m, X = _network(vg, n)
    want, _ = M.forward(p, X, emulate_bf16=True)
    dx = vg.DeviceArray.from_numpy(X)
    dy = dx if in_place else vg.DeviceArray.zeros((n, 3))
    m.forward(dx, n, dy)
    vg.synchronize()
    got = dy.numpy().ravel()[:3 * n].reshape(n, 3)
    assert rel(got, want) < TOL
