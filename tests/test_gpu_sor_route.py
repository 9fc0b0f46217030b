"""Which form a zebra SOR solve takes: the row kernels where a block of rows
in LDS has more around it than in it, or too few passes to make up for the
launches around them, blocks or one launch elsewhere; and no launch of more
than about a millisecond.  The forms give the same bits (the oracle's)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
F32 = np.float32


def solve(vg, shape, steps, u0=None, f=None, again=False):
    """Kernels of a solve ({name: (launches, ms)}), its grid and its result;
    again: of the second of two."""
    g = vg.GridDesc()
    for a in range(3):
        e = F32(0.01 * (a + 3) * (shape[a] - 1))
        g.extent[a], g.np[a] = e, shape[a]
        g.cell[a], g.cpe[a] = e / F32(shape[a] - 1), F32(shape[a] - 1) / e
    zero = u0 is None
    u = vg.DeviceArray.zeros((g.capacity, 3)) if zero else vg.DeviceArray.from_numpy(u0)
    lap = vg.DeviceArray.zeros((g.capacity, 3)) if zero else vg.DeviceArray.from_numpy(f)
    if again:
        vg.sor_solve(g, vg.DeviceArray.zeros((g.capacity, 3)), lap, steps)
    vg.profile_reset()
    vg.profile_enable(True)
    try:
        vg.sor_solve(g, u, lap, steps)
        vg.synchronize()
        kernels = {k: v for k, v in vg.profile_dump().items() if k.startswith("vg_sor_")}
    finally:
        vg.profile_enable(False)
    return kernels, g, u


def exact(oracle, g, u0, f, steps):
    og = oracle.define_shape(len(u0), np.zeros(3), np.ones(3), pow2=False)
    for a in range(3):
        og.np[a], og.cell[a], og.cpe[a] = g.np[a], g.cell[a], g.cpe[a]
        og.extent[a] = g.extent[a]
    return oracle.solve_vector_poisson(og, u0, f, steps)


@pytest.mark.parametrize("again", [False, True])
@pytest.mark.parametrize("shape,steps", [((33, 33, 33), 1), ((3, 321, 428), 8), ((5, 38, 281), 2),
                                         ((257, 257, 257), 1), ((321, 321, 321), 2),
                                         ((317, 434, 67), 2)])
def test_rows(vg, shape, steps, again):
    print(f"[case] SOR by rows {shape}, {steps} steps", flush=True)
    kernels, _, _ = solve(vg, shape, steps, again=again)
    assert {k: c for k, (c, _) in kernels.items()} == {"vg_sor_rows": 2 * steps}


@pytest.mark.parametrize("shape,steps", [((33, 41, 50), 1), ((65, 65, 65), 1), ((65, 65, 65), 2),
                                         ((129, 129, 129), 1)])
def test_rows_without_an_allocation_at_hand(vg, shape, steps):
    """Solves shorter than the time a first allocation of their scratch takes."""
    print(f"[case] SOR by rows, first solve {shape}, {steps} steps", flush=True)
    solve(vg, (3, 3, 3), 1)
    kernels, _, _ = solve(vg, shape, steps)
    assert set(kernels) == {"vg_sor_rows"}


@pytest.mark.parametrize("shape,steps,again", [
    ((129, 129, 129), 16, False), ((65, 65, 129), 16, False), ((65, 65, 65), 2, True),
    ((33, 33, 65), 16, True), ((65, 65, 67), 3, True), ((65, 36, 129), 16, True),
    ((67, 50, 41), 2, True), ((129, 20, 70), 2, True), ((257, 12, 19), 5, True),
    ((9, 129, 131), 7, True), ((41, 39, 25), 5, False)])
def test_blocks(vg, oracle, shape, steps, again):
    """Blocks with a remainder on either axis, short last launches among them."""
    print(f"[case] SOR in blocks {shape}, {steps} steps", flush=True)
    rng = np.random.default_rng(sum(shape))
    u0, f = (rng.normal(size=(int(np.prod(shape)), 3)).astype(F32) for _ in range(2))
    solve(vg, (3, 3, 3), 1)
    kernels, g, u = solve(vg, shape, steps, u0, f, again)
    assert set(kernels) == {"vg_sor_planes", "vg_sor_block"}
    assert kernels["vg_sor_block"][0] <= steps
    assert np.array_equal(u.numpy(), exact(oracle, g, u0, f, steps))


# passes of 0.7, 10 and 20 us
@pytest.mark.parametrize("shape,steps", [((3, 3, 3), 2000), ((1025, 5, 5), 120), ((2049, 3, 3), 150)])
def test_launches_stay_short(vg, oracle, shape, steps):
    print(f"[case] SOR whole grid {shape}, {steps} steps", flush=True)
    rng = np.random.default_rng(sum(shape))
    n = int(np.prod(shape))
    u0, f = (rng.normal(size=(n, 3)).astype(F32) for _ in range(2))
    kernels, g, u = solve(vg, shape, steps, u0, f)
    assert set(kernels) == {"vg_sor_block"}
    launches, ms = kernels["vg_sor_block"]
    print(f"{launches} launches, {ms:.2f} ms", flush=True)
    # the plan's estimate was measured within a factor of two
    assert launches >= 2 and ms / launches < 2.0
    assert np.array_equal(u.numpy(), exact(oracle, g, u0, f, steps))
