"""The zebra SOR's scratch: a solve or a cascade recorded into a graph takes
none that it does not have (rows and whole grids need none), and a cascade
keeps none that no layer of it reads.  Replays against the eager result, bit
for bit, with eager work between them."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
F32 = np.float32


def grid(vg, shape):
    g = vg.GridDesc()
    for a in range(3):
        e = F32(0.05 * (a + 2) * (shape[a] - 1))
        g.extent[a], g.np[a] = e, shape[a]
        g.cell[a], g.cpe[a] = e / F32(shape[a] - 1), F32(shape[a] - 1) / e
    return g


class Graph:
    """What f(stream) launches, recorded in the mode that refuses allocations."""

    def __init__(self, vg, stream, f):
        self.lib, self.stream = vg.lib(), stream
        graph, self.exec = C.c_void_p(), C.c_void_p()
        assert self.lib.hipStreamBeginCapture(stream.handle, 0) == 0
        try:
            f(stream)
        finally:
            ended = self.lib.hipStreamEndCapture(stream.handle, C.byref(graph))
        assert ended == 0
        assert self.lib.hipGraphInstantiate(C.byref(self.exec), graph, None, None,
                                            C.c_size_t(0)) == 0
        self.lib.hipGraphDestroy(graph)

    def launch(self):
        assert self.lib.hipGraphLaunch(self.exec, self.stream.handle) == 0
        self.stream.sync()

    def __del__(self):
        if self.exec:
            self.lib.hipGraphExecDestroy(self.exec)


def replays(vg, stream, run, result):
    """Recorded passes equal the eager one, whatever runs between them."""
    run(stream)
    stream.sync()
    want = result()
    g = Graph(vg, stream, run)
    for _ in range(3):
        g.launch()
        assert np.array_equal(result(), want)
        run(stream)
        stream.sync()
        assert np.array_equal(result(), want)


@pytest.mark.parametrize("shape", [(9, 9, 17), (33, 33, 65), (65, 65, 67), (8, 17, 17)])
def test_recorded_solve(vg, shape):
    """Whole grids, grids dealt in blocks when there is scratch, row kernels."""
    print(f"[case] recorded SOR solve {shape}", flush=True)
    rng = np.random.default_rng(sum(shape))
    g = grid(vg, shape)
    u0, f = (rng.normal(size=(g.capacity, 3)).astype(F32) for _ in range(2))
    first, lap = vg.DeviceArray.from_numpy(u0), vg.DeviceArray.from_numpy(f)
    u = vg.DeviceArray.zeros(u0.shape)
    s = vg.Stream()

    def run(stream):
        assert vg.lib().hipMemcpyAsync(u.ptr, first.ptr, C.c_size_t(u0.nbytes), 3,
                                       stream.handle) == 0
        vg.sor_solve(g, u, lap, 5, stream=stream)

    replays(vg, s, run, u.numpy)


@pytest.mark.parametrize("first,shape", [
    ((33, 33, 33), (33, 34, 34)),  # more scratch on the finest layer alone
    ((5, 5, 5), (6, 5, 5)),        # a finest layer of row kernels
    ((65, 65, 65), (65, 65, 65)),  # the scratch is there
])
def test_recorded_cascade(vg, first, shape):
    """A cascade whose coarse layers an earlier grid's buffers hold."""
    print(f"[case] recorded cascade {shape} after {first}", flush=True)
    rng = np.random.default_rng(sum(shape))
    s, m = vg.Stream(), vg.Multigrid()
    g0, g = grid(vg, first), grid(vg, shape)
    zero = vg.DeviceArray.zeros((g0.capacity, 3))
    m.cascade(g0, zero, zero, 3, stream=s)
    s.sync()
    f = rng.normal(size=(g.capacity, 3)).astype(F32)
    a, w = vg.DeviceArray.from_numpy(f), vg.DeviceArray.from_numpy(rng.permutation(f))

    def run(stream):
        m.cascade(g, a, w, 3, stream=stream)  # the interior starts from zero

    recorded = Graph(vg, s, run)  # before any eager pass on this grid
    recorded.launch()
    want = a.numpy()
    other = vg.Multigrid()
    for _ in range(2):
        other.cascade(g, a, w, 3, stream=s)
        s.sync()
        assert np.array_equal(a.numpy(), want)
        recorded.launch()
        assert np.array_equal(a.numpy(), want)


def test_cascade_keeps_no_unread_scratch(vg):
    """Row kernels (an even number of points along x) on every layer: the
    coarse layers' fields and no more."""
    shape = (128, 128, 128)
    print(f"[case] cascade memory {shape}", flush=True)

    def free():
        f, t = C.c_size_t(), C.c_size_t()
        assert vg.lib().hipMemGetInfo(C.byref(f), C.byref(t)) == 0
        return f.value

    g = grid(vg, shape)
    a = vg.DeviceArray.zeros((g.capacity, 3))
    warm = vg.Multigrid()
    warm.cascade(g, a, a, 2)
    vg.synchronize()
    before, m = free(), vg.Multigrid()
    m.cascade(g, a, a, 2)
    vg.synchronize()
    took = before - free()
    layers, _ = vg.nested_layers(g)
    # an allocation takes whole pages, of 2 MiB at most: far below the 75 MB
    # that the finest layer's scratch would be
    assert took <= sum(2 * 12 * l.capacity + 2 * (2 << 20) for l in layers[1:])
