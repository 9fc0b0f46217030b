"""Trees whose upper layers are formed by one workgroup: where those begin at
the first layer, with the largest layer a workgroup takes (and the smallest it
does not), one layer only, and decimations other than two, bit for bit against
the oracle's."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
F32 = np.float32


@pytest.mark.parametrize("n,shape", [
    (2, (1, 1, 1)), (8, (1, 1, 1)), (64, (1, 1, 1)), (300, (1, 2, 3)), (4096, (1, 1, 1)),
    (4096, (1, 0.1, 4)), (4096, (1, 0.02, 0.9)), (5000, (3, 1, 2)), (60000, (1, 1, 1.7)),
])
def test_tree_top_layers(vg, oracle, n, shape):
    print(f"[case] tree n={n} shape={shape}", flush=True)
    rng = np.random.default_rng(n)
    pos = (rng.random((n, 3)) * np.array(shape)).astype(F32)
    om = rng.standard_normal((n, 3)).astype(F32)
    og = oracle.grid_for(pos, 0.01)
    ot = oracle.InfluenceTree(og, pos, om, 0.02)
    dp, dw = vg.DeviceArray.from_numpy(pos), vg.DeviceArray.from_numpy(om)
    t = vg.Tree()
    t.build(vg.GridDesc.from_fields(og), vg.vortons_view(dp, dw, n, uniform_size=0.02))
    vg.synchronize()
    assert t.depth == ot.depth
    for l in range(ot.depth):
        g1, p1, w1, s1 = t.layer(l)
        g2, p2, w2, s2 = ot.layer(l)
        print(l, list(g2.np))
        assert list(g1.np) == list(g2.np)
        assert np.array_equal(s1, s2) and np.array_equal(w1, w2) and np.array_equal(p1, p2), l
