"""Boxes at the edges of the launch shapes against the oracle, bit for bit."""
import pytest

from conftest import assert_states_equal
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def box_state(shape, dims=3, seed=11):
    """A seeded state on a box of any shape: periodic plane waves."""
    import numpy as np

    from pluto_amd import problems as P
    rng = np.random.default_rng([seed, dims, *shape])
    nz, ny, nx = shape
    d = (1.0 / nx, 1.0 / ny, 1.0 / nz if dims == 3 else 1.0)

    def field():
        f = np.zeros(shape)
        for _ in range(6):
            k = rng.integers(-3, 4, 3)
            a = [2 * np.pi * k[c] * (np.arange(n) + 0.5) / n for c, n in enumerate((nx, ny, nz))]
            f += rng.standard_normal() * np.cos(a[0][None, None, :] + a[1][None, :, None]
                                                + a[2][:, None, None] * (dims == 3)
                                                + rng.uniform(0, 6.28))
        return f / 6.0

    a = [0.05 * field() for _ in range(3)]
    if dims == 2:
        a[0][:], a[1][:] = 0.0, 0.0
    b = P.curl_edges(*a, d, dims)
    v = np.stack([0.4 * field() for _ in range(3)])
    if dims == 2:
        v[2] = 0.0
    return P.assemble(1.0 + 0.3 * field(), v, 1.0 + 0.3 * field(), *b, dims, (1.0, 1.0, 1.0))


def check(shape, steps=2, dims=3, emf="uct_hll", **kw):
    from pluto_amd import native
    st = box_state(shape, dims)
    dt = 0.05 / max(shape)
    dom = native.Domain.from_state(st, emf_average=emf, **kw)
    dom.set_dt(dt)
    dom.run(steps)
    dom.sync()
    out = dom.get_state(st)
    dom.close()
    ref = st.copy()
    O.run(ref, steps, dt, emf=emf)
    assert_states_equal(out, ref, "%s" % (shape,))


# the z march and the CT march: 256 columns of the plane per workgroup (255,
# 256, 257 columns), segments of 1 plane and longer ones with a remainder (by
# size: 2, 4, 8 and 32 planes)
@pytest.mark.parametrize("shape", [(3, 17, 15), (5, 16, 16), (4, 257, 3), (7, 4, 64), (49, 48, 47),
                                   (65, 64, 63), (77, 93, 131), (161, 160, 160)])
def test_marches(shape):
    check(shape)


# the x/y row kernel: several rows a workgroup (nx 5, 16, 24, 100, with the
# last group cut by nz), one row, windows (nx 131, 257, 300, 515; one window
# and several), y segments with a remainder, both dimensions
@pytest.mark.parametrize("shape", [(9, 6, 5), (33, 40, 16), (17, 30, 24), (5, 50, 100), (6, 70, 131),
                                   (3, 9, 256), (3, 7, 257), (8, 33, 300), (3, 3, 515), (1, 40, 64),
                                   (1, 65, 130), (1, 33, 700)])
@pytest.mark.parametrize("seg", [0, 7])
def test_rows(shape, seg):
    from pluto_amd import native
    native.set_flux_kernel(1, seg)
    try:
        check(shape, dims=2 if shape[0] == 1 else 3)
    finally:
        native.set_flux_kernel()


# the LDS EMF: tiles cut at the row and plane ends, even rows (16-byte copies)
# and odd ones (4-byte), boxes narrower than a tile, z segments with a
# remainder, 2D
@pytest.mark.parametrize("kind,shape", [(k, s) for k in (1, 2, 3) for s in (
    (3, 3, 3), (5, 9, 31), (17, 8, 32), (18, 7, 33), (6, 10, 34), (33, 17, 66))]
    + [(3, s) for s in ((1, 3, 3), (1, 9, 32), (1, 25, 67))])   # (2D has one kernel)
def test_emf_tiles(shape, kind):
    from pluto_amd import native
    native.set_emf_kernel(kind)
    try:
        check(shape, dims=2 if shape[0] == 1 else 3)
    finally:
        native.set_emf_kernel()


# the face EMF averages marching up z: planes of less than one workgroup, one
# and several with a cut last one, segments of 1 plane, 2 with a remainder and
# 16 with a remainder; 2D (per cell)
@pytest.mark.parametrize("shape", [(3, 3, 3), (5, 16, 16), (7, 86, 3), (9, 17, 31), (33, 130, 130),
                                   (37, 181, 200), (19, 600, 450), (1, 9, 32)])
@pytest.mark.parametrize("emf", ["uct0", "uct_contact", "arithmetic"])
def test_emf_faces(shape, emf):
    check(shape, dims=2 if shape[0] == 1 else 3, emf=emf)


# the modular pipeline's EMF: register kernels on small boxes, the LDS one on
# larger and on narrow ones (either side of 300000 cells, 16-cell rows, 16-cell
# planes), 2D too
@pytest.mark.parametrize("shape", [(3, 3, 3), (20, 5, 3), (20, 6, 3), (9, 20, 15), (9, 20, 16), (64, 64, 73),
                                   (65, 65, 72), (1, 4, 3), (1, 20, 16), (1, 547, 548), (1, 549, 550)])
@pytest.mark.parametrize("kind", [0, 3])
def test_modular_emf(shape, kind):
    from pluto_amd import native
    native.set_emf_kernel(kind)
    try:
        check(shape, dims=2 if shape[0] == 1 else 3, pipeline=native.PIPELINE_MODULAR)
    finally:
        native.set_emf_kernel()


# read-back: less than one staging buffer (2^19 values), just over one and
# several with a cut last one, interior of a bounded box, single arrays
@pytest.mark.parametrize("shape", [(3, 4, 5), (36, 37, 36), (47, 50, 49), (90, 81, 77)])
@pytest.mark.parametrize("bounded", [False, True])
def test_readback(shape, bounded):
    import ctypes

    import numpy as np

    from pluto_amd import native
    st = box_state(shape)
    dom = native.Domain(st.shape, 3, st.spacing(), bounds=["periodic"] * 6 if bounded else None)
    dom.set_state(st)
    for _ in range(20):
        out = dom.get_state(st)
        assert_states_equal(out, st, "%s bounded %s" % (shape, bounded))
    one = np.full(shape, -1.0)
    native.check(native.lib().pgpu_get_state(dom.h, None, None, one.ctypes.data_as(
        ctypes.POINTER(ctypes.c_double)), None))
    assert np.array_equal(one, st.by)
    dom.close()


# a read waits for the steps queued before it, also one that asks for no array
def test_empty_read_waits():
    import time

    from pluto_amd import native
    L = native.lib()
    st = box_state((256, 256, 256))
    dom = native.Domain.from_state(st)
    bat = native.Batch([256])
    bat.set_patch(0, st)
    bat.set_dt(1e-4)
    dom.set_dt(1e-4, fixed=True)
    for obj, read in ((dom, lambda: L.pgpu_get_state(dom.h, None, None, None, None)),
                      (bat, lambda: L.pgpu_batch_get_patch(bat.h, 0, None, None, None, None))):
        obj.run(2)
        obj.sync()
        t0 = time.perf_counter()
        obj.run(60)   # 6 ms each
        native.check(read())
        t1 = time.perf_counter()
        obj.sync()
        t2 = time.perf_counter()
        print("run and empty read %.3f s, then the wait %.4f s" % (t1 - t0, t2 - t1), flush=True)
        assert t2 - t1 < 0.1 * (t1 - t0)
        obj.close()


# while a read waits for the steps queued before it, the host's other processors
# are left alone (the threads that copy out start when there is something to copy)
def test_read_waits_idle():
    import ctypes
    import resource
    import time

    from pluto_amd import native
    st = box_state((256, 256, 256))
    dom = native.Domain.from_state(st)
    dom.set_dt(1e-4, fixed=True)
    out = st.copy()
    ptrs = [a.ctypes.data_as(ctypes.POINTER(ctypes.c_double)) for a in (out.bx, out.by, out.bz)]
    native.check(native.lib().pgpu_get_state(dom.h, None, *ptrs))   # (first allocations)
    dom.run(60)   # 6 ms each
    t0, c0 = time.perf_counter(), resource.getrusage(resource.RUSAGE_SELF)
    native.check(native.lib().pgpu_get_state(dom.h, None, *ptrs))
    t1, c1 = time.perf_counter(), resource.getrusage(resource.RUSAGE_SELF)
    dom.close()
    wall, cpu = t1 - t0, c1.ru_utime + c1.ru_stime - c0.ru_utime - c0.ru_stime
    print("read %.3f s, %.3f s of processor time" % (wall, cpu), flush=True)
    assert wall > 0.1
    assert cpu < 2.0 * wall   # one waiting thread, and the copies' 10 ms of eight


# pinned memory for what is read, not for the largest read there is
def test_small_read_pins_little():
    from pluto_amd import native
    st = box_state((3, 4, 5))
    native.Domain.from_state(st).get_state(st)   # (code and runtime in place)

    def mapped():
        with open("/proc/self/statm") as f:
            return int(f.read().split()[0]) * 4096

    doms = [native.Domain.from_state(st) for _ in range(8)]
    before = mapped()
    for d in doms:
        assert_states_equal(d.get_state(st), st, "small read")
    grown = mapped() - before
    print("8 small reads mapped %.2f MiB" % (grown / 2**20), flush=True)
    for d in doms:
        d.close()
    assert grown < 8 * 2**20   # (eight 660-value reads; 4 x 4 MiB each: 128 MiB)


# one object's reads in any order of sizes (the staging grows with them)
def test_reads_of_growing_size():
    from pluto_amd import native
    edges = [4, 6, 12, 20, 37, 64, 80]
    states = [box_state((n, n, n), seed=n) for n in edges]
    b = native.Batch(edges)
    for p, st in enumerate(states):
        b.set_patch(p, st)
    for p in (0, 2, 1, 4, 3, 6, 0, 5, 6, 2):
        assert_states_equal(b.get_patch(p), states[p], "patch %d" % p)
    b.close()
