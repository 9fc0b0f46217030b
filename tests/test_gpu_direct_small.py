"""The direct sums' fine blocks (128 queries by whole tiles of 256 sources):
the edges of the query block, of a tile and of a wave's quarter of it, one
source and one query, and the split over several tiles, against the CPU
oracle; strided vortons with their own sizes included."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
F32 = np.float32


@pytest.mark.parametrize("policy", [0, 1])
@pytest.mark.parametrize("n,nq", [(1, 1), (63, 127), (64, 128), (65, 129), (255, 64), (256, 1),
                                  (257, 300), (1023, 513), (4097, 4095), (12345, 77)])
def test_fine_blocks(vg, oracle, n, nq, policy):
    print(f"[case] direct sum, {n} vortons, {nq} queries, policy {policy}", flush=True)
    rng = np.random.default_rng(n + nq)
    rec = rng.normal(size=(n, 18)).astype(F32)
    rec[:, 13] = rng.uniform(0.05, 0.3, n)
    q = rng.normal(size=(nq, 4)).astype(F32)
    d, dq = vg.DeviceArray.from_numpy(rec), vg.DeviceArray.from_numpy(q)
    v = vg.Vortons()
    v.pos, v.angvel, v.size = d.ptr.value, d.offset(9).value, d.offset(13).value
    v.stride, v.n, v.uniform_size = 18, n, 0.0
    pos, om, size = (np.ascontiguousarray(a) for a in (rec[:, 0:3], rec[:, 9:12], rec[:, 13]))
    pts = np.ascontiguousarray(q[:, :3])
    for gpu, cpu in ((vg.direct_velocity, oracle.direct_velocity),
                     (vg.direct_vecpot, oracle.direct_vecpot)):
        out = vg.DeviceArray.zeros((nq, 3))
        gpu(v, dq, nq, out, 1.3, 0.7, policy, q_stride=4)
        vg.synchronize()
        want = cpu(pos, om, size, pts, 1.3, 0.7, policy=policy, threads=8)
        # FP32 terms of random sign summed in another order
        assert np.linalg.norm(out.numpy() - want) <= 1e-5 * np.linalg.norm(want)


@pytest.mark.parametrize("partials", [1, 15, 16, 17, 32, 33, 2000])
def test_partials_of_many_tiles(vg, oracle, partials):
    """A tile per workgroup and their sum, which takes 16 of them at a time:
    the edges of those, and the time of many (few queries by many vortons)."""
    n, nq = 256 * partials, 64
    print(f"[case] direct sum, {partials} partials", flush=True)
    rng = np.random.default_rng(partials)
    pos, om, q = (rng.normal(size=(k, 3)).astype(F32) for k in (n, n, nq))
    dp, dw, dq = (vg.DeviceArray.from_numpy(a) for a in (pos, om, q))
    v = vg.vortons_view(dp, dw, n, uniform_size=0.2)
    out = vg.DeviceArray.zeros((nq, 3))
    vg.direct_velocity(v, dq, nq, out, policy=1)
    vg.profile_reset()
    vg.profile_enable(True)
    try:
        vg.direct_velocity(v, dq, nq, out, policy=1)
        vg.synchronize()
        ms, _ = vg.profile_get("vg_direct_reduce")
    finally:
        vg.profile_enable(False)
    want = oracle.direct_velocity_f64(pos, om, np.full(n, 0.2, F32), q, threads=8)
    # FP32 terms of random sign; 64-bit sums, which a serial FP32 one of
    # 512,000 terms misses by 1.3e-5
    assert np.linalg.norm(out.numpy() - want) <= 1e-5 * np.linalg.norm(want)
    # 2000 partials: 75 us with 16 loads under way, 480 with one
    assert ms < 0.2


def _sum(vg, v, q, nq, out, stride):
    """The kernels of a sum."""
    vg.profile_reset()
    vg.profile_enable(True)
    try:
        vg.direct_velocity(v, q, nq, out, 1.3, 0.7, 1, q_stride=stride)
        vg.synchronize()
        return set(vg.profile_dump())
    finally:
        vg.profile_enable(False)


@pytest.mark.parametrize("n,nq", [(1, 1), (200, 20000), (256, 130), (300, 140000), (257, 300)])
def test_one_share_of_the_sources_goes_out_directly(vg, oracle, n, nq):
    """One launch where the sources are not split, several where they are; an
    output that holds the vortons, or the queries at another stride, is written
    once all have been read, to the same bits."""
    print(f"[case] direct sum, {n} vortons at {nq} points, outputs among the inputs", flush=True)
    rng = np.random.default_rng(n + nq)
    pos, om, q = (rng.normal(size=(k, 3)).astype(F32) for k in (n, n, nq))
    dp, dw, dq = (vg.DeviceArray.from_numpy(a) for a in (pos, om, q))
    v = vg.vortons_view(dp, dw, n, uniform_size=0.2)
    out = vg.DeviceArray.zeros((nq, 3))
    split = n > 256 and nq < 131000
    assert ("vg_direct_reduce" in _sum(vg, v, dq, nq, out, 3)) == split
    got = out.numpy()
    want = oracle.direct_velocity(pos, om, np.full(n, 0.2, F32), q, 1.3, 0.7, policy=1, threads=8)
    assert np.linalg.norm(got - want) <= 1e-5 * np.linalg.norm(want)
    # the vortons within the output, first as positions, then as vorticities
    for field in (0, 1):
        whole = rng.normal(size=(max(n, nq), 3)).astype(F32)
        whole[:n] = (pos, om)[field]
        both = vg.DeviceArray.from_numpy(whole)
        u = vg.vortons_view(both, dw, n, uniform_size=0.2) if field == 0 else \
            vg.vortons_view(dp, both, n, uniform_size=0.2)
        assert "vg_direct_reduce" in _sum(vg, u, dq, nq, both, 3)
        assert np.array_equal(both.numpy()[:nq], got)
    # the queries' own places, and other ones
    same = vg.DeviceArray.from_numpy(q)
    assert ("vg_direct_reduce" in _sum(vg, v, same, nq, same, 3)) == split
    assert np.array_equal(same.numpy(), got)
    wide = np.zeros((nq, 5), F32)
    wide[:, :3] = q
    apart = vg.DeviceArray.from_numpy(wide)
    assert "vg_direct_reduce" in _sum(vg, v, apart, nq, apart, 5)
    assert np.array_equal(apart.numpy().ravel()[:3 * nq].reshape(nq, 3), got)
