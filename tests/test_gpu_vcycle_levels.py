"""V-cycles whose coarse levels run in one launch: grids all of whose levels
fit LDS, only the coarsest, or none (a coarsest level past it), coarsest levels
within a wave and beyond, long and flat ones, against the system in 64
bits."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu
F32 = np.float32


# cells per axis, and the cycles that take the relative residual to 1e-6 with
# a launch per step
@pytest.mark.parametrize("cells,cycles", [
    ((2, 2, 2), 1),      # one interior point, the coarsest itself
    ((4, 4, 4), 4),     # two levels, the coarsest within a wave
    ((4, 6, 8), 5),     # coarsest 3x4x5, 60 points
    ((6, 10, 6), 5),    # coarsest beyond a wave
    ((20, 12, 28), 5),  # odd row counts on every level
    ((16, 16, 32), 5),  # the largest first level of a doubling grid
    ((18, 18, 18), 5),  # first level and coarsest (9 cells) in one workgroup
    ((13, 9, 11), 1),    # one level, in double
    ((23, 23, 23), 1),   # one level, past LDS
    ((2, 2, 500), 1),   # one level of long rows along z
    ((500, 2, 3), 1),   # and along x
    ((48, 64, 32), 5),  # launches per level down to the ones that fit
])
def test_vcycle_levels(vg, cells, cycles):
    print(f"[case] v-cycle cells {cells}", flush=True)
    rng = np.random.default_rng(sum(cells))
    np_ = [c + 1 for c in cells]
    ext = [c / max(cells) for c in cells]
    h = [float(F32(e) / F32(c)) for e, c in zip(ext, cells)]
    g = vg.GridDesc()
    for k in range(3):
        g.extent[k], g.cell[k], g.cpe[k], g.np[k] = ext[k], h[k], 1 / h[k], np_[k]
    inner = [c - 1 for c in cells]
    f = np.zeros((np_[2], np_[1], np_[0], 3), F32)
    f[1:-1, 1:-1, 1:-1] = rng.standard_normal((inner[2], inner[1], inner[0], 3))
    a = vg.DeviceArray.zeros((f.size // 3, 3))
    rel, took = vg.Multigrid().vcycle_solve(g, a, vg.DeviceArray.from_numpy(f.reshape(-1, 3)),
                                            tol=1e-6, max_cycles=80)
    vg.synchronize()
    got = a.numpy().reshape(f.shape).astype(np.float64)
    print(f"rel {rel:.2e} in {took} cycles")
    assert rel <= 1e-6 and took <= cycles
    d2 = [sp.diags_array([np.ones(n - 1), -2 * np.ones(n), np.ones(n - 1)], offsets=[-1, 0, 1]) / s ** 2
          for n, s in zip(inner, h)]
    one = [sp.eye_array(n) for n in inner]
    lap = (sp.kron(sp.kron(one[2], one[1]), d2[0]) + sp.kron(sp.kron(one[2], d2[1]), one[0]) +
           sp.kron(sp.kron(d2[2], one[1]), one[0]))
    b = f[1:-1, 1:-1, 1:-1].reshape(-1, 3).astype(np.float64)
    e = got[1:-1, 1:-1, 1:-1].reshape(-1, 3)
    # `a` is the solution rounded to 32 bits, whose residual that moves
    norm = sum(4 / s ** 2 for s in h)
    bound = 1.01e-6 * np.linalg.norm(b) + norm * 2.0 ** -24 * np.linalg.norm(e)
    assert np.linalg.norm(lap @ e - b) <= bound
