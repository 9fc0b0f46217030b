"""The zebra SOR's LDS form at the sizes where it changes: grids that fit one
workgroup (all passes in one launch) down to one interior point, grids dealt
in blocks with a remainder on either axis, step counts that leave a short
last launch, rows of one chunk, of a chunk more or less, and the grids that
keep the row kernels (an even number of points along x).  Bit for bit against
the CPU oracle's sequential sweep."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
F32 = np.float32


@pytest.mark.parametrize("shape,steps", [
    ((3, 3, 3), 1), ((3, 5, 9), 16), ((5, 3, 4), 3), ((9, 9, 17), 16), ((11, 10, 3), 5),
    ((17, 17, 33), 16), ((19, 24, 25), 4), ((33, 33, 9), 16), ((33, 33, 65), 16),
    ((65, 65, 67), 3), ((65, 36, 129), 16), ((67, 50, 41), 1), ((129, 20, 70), 2),
    ((257, 12, 19), 5), ((9, 129, 131), 7), ((10, 129, 131), 3), ((8, 17, 17), 16),
    ((3, 3, 3), 700)])
def test_sor_block(vg, oracle, shape, steps):
    print(f"[case] SOR grid {shape}, {steps} steps", flush=True)
    rng = np.random.default_rng(sum(shape) + steps)
    ext = np.array([c - 1 for c in shape], np.float64) * np.array([0.05, 0.06, 0.04])
    og = oracle.define_shape(int(np.prod([c - 1 for c in shape])), np.zeros(3), ext, pow2=False)
    g = vg.GridDesc.from_fields(og)
    for a in range(3):
        og.np[a] = g.np[a] = shape[a]
        og.cell[a] = g.cell[a] = F32(ext[a]) / F32(shape[a] - 1)
        og.cpe[a] = g.cpe[a] = F32(shape[a] - 1) / F32(ext[a])
    n = int(np.prod(shape))
    f = rng.normal(size=(n, 3)).astype(F32)
    u0 = rng.normal(size=(n, 3)).astype(F32)
    sol, lap = vg.DeviceArray.from_numpy(u0), vg.DeviceArray.from_numpy(f)
    vg.sor_solve(g, sol, lap, steps)
    vg.synchronize()
    assert np.array_equal(sol.numpy(), oracle.solve_vector_poisson(og, u0, f, steps))
    assert np.array_equal(lap.numpy(), f)
