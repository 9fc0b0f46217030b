"""The viscous exchange's chain form (fractions precomputed, one component
per workgroup) at the sizes where it changes: cells of one vorton up to more
than two chunks of 64 lanes, a neighbourhood just within and just past the
partners that fit a wave's LDS buffer, and slices that fit the LDS and that
do not.  Bit for bit against the CPU oracle, with dead vortons."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
F32 = np.float32


def run(vg, oracle, og, pos, om, size, rng, dead=0.15):
    n = len(pos)
    birth = np.where(rng.random(n) < dead, -1, 5).astype(np.int32)
    dp, dw = vg.DeviceArray.from_numpy(pos), vg.DeviceArray.from_numpy(om)
    db = vg.DeviceArray.from_numpy(birth)
    t = vg.Tree()
    t.build(vg.GridDesc.from_fields(og), vg.vortons_view(dp, dw, n, uniform_size=size))
    t.pse_diffuse(dw, 0.5, 0.2, birth=db, birth_stride=1)
    vg.synchronize()
    want = oracle.pse_diffuse(og, pos, om, size, 0.5, 0.2, alive=birth >= 0)
    assert np.array_equal(dw.numpy(), want)


@pytest.mark.parametrize("blob", [1, 2, 3, 63, 64, 65, 127, 128, 129, 700, 2399, 2401])
def test_chunks_of_here_vortons(vg, oracle, blob):
    """One cell of `blob` vortons (its neighbours hold none) among cells of a
    few."""
    print(f"[case] PSE chain, a cell of {blob} vortons", flush=True)
    rng = np.random.default_rng(blob)
    cells, h = (8, 6, 5), 0.25
    ext = np.array(cells) * h
    pos = (rng.uniform(0.02, 0.98, (300, 3)) * ext)
    around = np.all(np.abs(pos - np.array([4.5, 3.5, 2.5]) * h) < 1.6 * h, axis=1)
    lump = (np.array([4, 3, 2]) + rng.uniform(0.1, 0.9, (blob, 3))) * h
    pos = np.concatenate([pos[~around], lump]).astype(F32)
    om = rng.normal(size=pos.shape).astype(F32)
    og = oracle.define_shape(int(np.prod(cells)), np.zeros(3), ext, pow2=False)
    assert og.shape == tuple(c + 1 for c in cells)
    run(vg, oracle, og, pos, om, 0.2, rng)


def test_slices_past_the_lds(vg, oracle):
    """A thin slab: 50,000 vortons in two slices (200 KB a component)."""
    print("[case] PSE chain, 100,000 vortons in a slab of four slices", flush=True)
    rng = np.random.default_rng(9)
    cells = (96, 96, 4)
    ext = np.array(cells) * 0.02
    pos = (rng.uniform(0.001, 0.999, (100000, 3)) * ext).astype(F32)
    om = rng.normal(size=pos.shape).astype(F32)
    og = oracle.define_shape(int(np.prod(cells)), np.zeros(3), ext, pow2=False)
    assert og.shape == tuple(c + 1 for c in cells)
    run(vg, oracle, og, pos, om, 0.02, rng)


def kernels(vg, f):
    vg.profile_reset()
    vg.profile_enable(True)
    try:
        f()
        return {k for k in vg.profile_dump() if k.startswith("vg_pse_")}
    finally:
        vg.profile_enable(False)


@pytest.mark.parametrize("cells", [(513, 257, 1), (514, 258, 2), (512, 256, 1)])
@pytest.mark.parametrize("fractions", [None, "0"])
def test_flat_grids(vg, oracle, monkeypatch, cells, fractions):
    """Wavefront steps of more cells than the schedule deals, and of as many:
    cells of no vortons up to two chunks, with the fractions precomputed and in
    the serial exchange."""
    print(f"[case] PSE flat grid {cells}, fractions {fractions}", flush=True)
    if fractions is not None:
        monkeypatch.setenv("VG_PSE_FRACTIONS", fractions)
    rng = np.random.default_rng(sum(cells))
    h = 0.05
    ext = np.array(cells) * h
    pos = [rng.uniform(0.0005, 0.9995, (40000, 3)) * ext]
    for k in (3, 4, 5, 63, 64, 65, 130):
        at = np.array([rng.integers(c) for c in cells])
        pos.append((at + rng.uniform(0.1, 0.9, (k, 3))) * h)
    pos = np.concatenate(pos).astype(F32)
    om = rng.normal(size=pos.shape).astype(F32)
    og = oracle.define_shape(int(np.prod(cells)), np.zeros(3), ext, pow2=False)
    assert og.shape == tuple(c + 1 for c in cells)
    ran = kernels(vg, lambda: run(vg, oracle, og, pos, om, 0.04, rng))
    assert ("vg_pse_fractions" in ran) == (fractions is None)
    assert ("vg_pse_schedule" in ran) == (cells == (512, 256, 1))


@pytest.mark.parametrize("blob", [2401, 5000])
def test_cells_past_the_chain_keep_precomputed_fractions(vg, oracle, blob):
    """Cells of one wave's share of the fractions beside one of many."""
    print(f"[case] PSE fractions by rows, a cell of {blob} vortons", flush=True)
    rng = np.random.default_rng(blob)
    cells, h = (9, 8, 7), 0.25
    ext = np.array(cells) * h
    lump = (np.array([4, 3, 2]) + rng.uniform(0.1, 0.9, (blob, 3))) * h
    pos = np.concatenate([rng.uniform(0.002, 0.998, (9000, 3)) * ext, lump]).astype(F32)
    om = rng.normal(size=pos.shape).astype(F32)
    og = oracle.define_shape(int(np.prod(cells)), np.zeros(3), ext, pow2=False)
    assert og.shape == tuple(c + 1 for c in cells)
    assert "vg_pse_fractions" in kernels(vg, lambda: run(vg, oracle, og, pos, om, 0.2, rng))


@pytest.mark.parametrize("dead", [0.4, 0.95])
def test_zeros_keep_their_sign(vg, oracle, dead):
    """Components of -0 and +0 beside others, in cells of one vorton up to two
    chunks: alone, adopted, exchanged, and past dead vortons; the bits of the
    oracle's, not their values."""
    print(f"[case] PSE signed zeros, {dead} dead", flush=True)
    rng = np.random.default_rng(5)
    cells, h = (10, 8, 6), 0.25
    ext = np.array(cells) * h
    lumps = [(np.array([rng.integers(c) for c in cells]) + rng.uniform(0.1, 0.9, (k, 3))) * h
             for k in (1, 2, 3, 64, 70)]
    pos = np.concatenate([rng.uniform(0.002, 0.998, (400, 3)) * ext] + lumps).astype(F32)
    om = rng.normal(size=pos.shape).astype(F32)
    om[rng.random(om.shape) < 0.4] = F32(-0.0)
    om[rng.random(om.shape) < 0.1] = F32(0.0)
    og = oracle.define_shape(int(np.prod(cells)), np.zeros(3), ext, pow2=False)
    assert og.shape == tuple(c + 1 for c in cells)
    birth = np.where(rng.random(len(pos)) < dead, -1, 5).astype(np.int32)
    want = oracle.pse_diffuse(og, pos, om, 0.02, 0.5, 0.2, alive=birth >= 0)
    # (what a live vorton touches loses it: dead ones have it)
    assert np.count_nonzero((want == 0) & np.signbit(want)) > 10
    dp, dw = vg.DeviceArray.from_numpy(pos), vg.DeviceArray.from_numpy(om)
    db = vg.DeviceArray.from_numpy(birth)
    t = vg.Tree()
    t.build(vg.GridDesc.from_fields(og), vg.vortons_view(dp, dw, len(pos), uniform_size=0.02))
    t.pse_diffuse(dw, 0.5, 0.2, birth=db, birth_stride=1)
    vg.synchronize()
    assert np.array_equal(dw.numpy().view(np.uint32), want.view(np.uint32))
