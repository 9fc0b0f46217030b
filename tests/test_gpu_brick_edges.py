"""The near-field walk at the grid's upper faces, where a 4x4x4 brick holds
fewer points: rows run along the first axis with four points and take 4, 16
or 64 lanes.  Every combination of 1..4 points on the brick's axes, one
vorton size and a different size per vorton (the per-cluster size form)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
F32 = np.float32


def rel_l2(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


@pytest.mark.parametrize("own_sizes", [False, True])
@pytest.mark.parametrize("order", [0, 1])
@pytest.mark.parametrize("cells", [(1, 1, 4), (4, 1, 1), (1, 6, 6), (2, 2, 2), (3, 3, 3),
                                   (4, 4, 4), (6, 2, 4), (4, 8, 2), (2, 6, 3), (12, 3, 6),
                                   (8, 4, 16), (24, 6, 1)])
def test_brick_edges(vg, oracle, cells, order, own_sizes):
    print(f"[case] brick edges, cells {cells}, order {order}, own sizes {own_sizes}", flush=True)
    rng = np.random.default_rng(sum(c * 31 ** i for i, c in enumerate(cells)))
    n = 1500
    ext = np.array(cells, np.float64) * 0.25
    pos = (rng.uniform(0.02, 0.98, (n, 3)) * ext).astype(F32)
    om = rng.normal(size=(n, 3)).astype(F32)
    og = oracle.define_shape(int(np.prod(cells)), np.zeros(3), ext, pow2=False)
    assert og.shape == tuple(c + 1 for c in cells) and not oracle.nested_has_orphans(og)
    size = (0.1 * rng.uniform(0.5, 2.0, n)).astype(F32) if own_sizes else np.full(n, 0.1, F32)
    dp, dw = vg.DeviceArray.from_numpy(pos), vg.DeviceArray.from_numpy(om)
    ds = vg.DeviceArray.from_numpy(np.repeat(size[:, None], 3, axis=1))
    v = vg.Vortons()
    v.pos, v.angvel, v.size = dp.ptr.value, dw.ptr.value, ds.ptr.value
    v.stride, v.n, v.uniform_size = 3, n, 0.0
    g = vg.GridDesc.from_fields(og)
    t = vg.Tree()
    t.build(g, v)
    out = vg.DeviceArray.zeros((g.capacity, 3))
    t.velocity_grid_mac(g, out, 1, order, 1.0, 1.0, 1)
    vg.synchronize()
    got = out.numpy().reshape(g.np[2], g.np[1], g.np[0], 3)
    ot = oracle.InfluenceTree(og, pos, om, size)
    want = oracle.mac_velocity_grid(ot, og, pos, om, size, 1, order, 1.0, 1.0, 1, threads=8)
    want = want.reshape(got.shape)
    # FP32 sums of up to 1500 terms of random sign in another order: a few
    # ulp of the partial sums, 1e-5 leaves a factor of ten; the faces, which
    # the short bricks hold, by themselves too
    assert rel_l2(got, want) < 1e-5
    for face in (np.s_[-1], np.s_[:, -1], np.s_[:, :, -1]):
        assert rel_l2(got[face], want[face]) < 1e-5
