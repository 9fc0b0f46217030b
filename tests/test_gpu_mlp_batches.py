"""Network passes at the edges of their 64-row tiles: one row, a tile less,
whole and more, and batches whose workgroups take several tiles each (256 of
them for the gradients, 768 forward), against the oracle."""
import numpy as np
import pytest

from oracle import mlp_oracle as M

pytestmark = pytest.mark.gpu
F32 = np.float32
# An operand that FP32 and FP64 leave on either side of a tie is rounded to
# bf16 differently and moves by 2^-8.  Differences of a few 2^-24 do so to
# about one operand in 2^13, so a product's error is some 2^-8 2^-6.5 = 4e-5,
# and six products' on the way to the first layer's weights 1e-4 (1.2e-4 was
# the largest seen); ten times that.
TOL = 1e-3


def rel(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30))


def _network(vg, n):
    rng = np.random.default_rng(n)
    p = (M.init_params(12) + 0.05 * rng.standard_normal(M.N_PARAMS)).astype(F32)
    m = vg.Mlp()
    m.set_params(p)
    return rng, p, m, rng.standard_normal((n, M.N_IN)).astype(F32)


# Rows of a tile, and of all workgroups' first, second, ... tiles.
TILE, ROUND_GRAD, ROUND_FORWARD = 64, 256 * 64, 768 * 64


def groups(n, size):
    """The rows of each round of tiles, and of the last tile by itself."""
    edges = list(range(0, n, size)) + [n]
    last = (n - 1) // TILE * TILE
    if last not in edges:
        edges.insert(-1, last)
    return [slice(a, b) for a, b in zip(edges, edges[1:])]


@pytest.mark.parametrize("n", [1, 15, 63, 64, 65, 4097, 16384, 16385, 33000])
def test_gradients_of_batch_sizes(vg, n):
    """Targets far from the outputs, so that the rows' gradients add up like
    random vectors and no common part hides a few of them, and farther in
    smaller groups of rows, so that each has the same share."""
    print(f"[case] mlp gradients n={n}", flush=True)
    rng, p, m, X = _network(vg, n)
    T = 30 * rng.standard_normal((n, 3)).astype(F32)
    parts = groups(n, ROUND_GRAD)
    for g in parts:
        T[g] *= F32(np.sqrt(n / (g.stop - g.start)))
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
    # a group of rows left out, or a tile of one, would show
    tiles = [slice(r.start, min(r.start + TILE, r.stop)) for r in parts if n > ROUND_GRAD]
    for left_out in parts + tiles:
        r = np.r_[left_out]
        if len(r) == n:
            continue
        _, gp = M.backward(p, X[r], T[r], emulate_bf16=True, B=None if B is None else B[r])
        assert np.linalg.norm(gp) * len(r) / n > 20 * TOL * np.linalg.norm(gw)


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
    for r in groups(n, ROUND_FORWARD):
        assert rel(got[r], want[r]) < TOL
    # every row: a few operands of it rounded differently (0.007 was the largest
    # seen); a row left out would be off by itself, which few are short enough
    # to hide
    bound = 8 * 2.0 ** -8 * np.sqrt(np.mean(want ** 2) * 3)
    assert np.linalg.norm(got - want, axis=1).max() < bound
    assert np.mean(np.linalg.norm(want, axis=1) > 2 * bound) > 0.99
