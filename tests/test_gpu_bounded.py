"""Resident boxes with non-periodic sides (pgpu_domain_create_bounded):
the ghosted box stays on the device across steps, Boundary()'s fill
(boundary.c:120-292, ct_fill_mag_field.c) runs before every stage, and dt
comes from the device-side CFL reduction over PLUTO's ranges.  Against
PLUTO's own main loop with the same [Boundary] block (oracle/_ref/pluto3d,
the state loader setting the face below the first cell as the image of the
last face, as the bounded box does), bit for bit: states, dt and Mach per
dumped step.  div.B stays at round-off in the interior cells.  Periodic axes,
alone and beside outflow ones, also against the oracle, with lower faces that
differ from the last ones.
"""
import numpy as np
import pytest

from conftest import assert_states_equal

pytestmark = pytest.mark.gpu


def _say(msg):
    print(msg, flush=True)


@pytest.fixture(scope="module")
def native():
    from pluto_amd import native as N
    if N.device_count() < 1:
        pytest.fail("no HIP device visible")
    return N


def _box(shape, seed):
    from pluto_amd import problems as P
    nz, ny, nx = shape
    big = P.random_mhd_3d(max(shape), seed=seed)
    st = big.copy()
    st.prim = np.ascontiguousarray(big.prim[:, :nz, :ny, :nx])
    st.bx, st.by, st.bz = (np.ascontiguousarray(b[:nz, :ny, :nx]) for b in (big.bx, big.by, big.bz))
    n = max(shape)
    st.length = (nx / n, ny / n, nz / n)
    st.prim[4], st.prim[5], st.prim[6] = P.face_average(st.bx, st.by, st.bz)
    return st


CASES = {
    "outflow": (("outflow",) * 6, "hlld", "uct_hll"),
    "reflective": (("reflective",) * 6, "hlld", "uct_hll"),
    "mixed": (("reflective", "outflow", "periodic", "periodic", "eqtsymmetric", "axisymmetric"),
              "hlld", "uct_hll"),
    "outflow_hllc_arith": (("outflow", "outflow", "reflective", "outflow", "periodic", "periodic"),
                           "hllc", "arithmetic"),
    "all_periodic": (("periodic",) * 6, "hlld", "uct_hll"),
}


@pytest.mark.parametrize("case", sorted(CASES))
def test_bounded_domain_vs_pluto_main_loop(native, case):
    from oracle import refrun
    bounds, solver, emf = CASES[case]
    if not refrun.available(3, emf):
        pytest.skip("reference executables not built (make -C oracle/ref)")
    shape = (9, 10, 12)
    _say("case: bounded domain %s (%s, %s), box %s, 8 CFL steps" % (case, solver, emf, shape))
    st = _box(shape, seed=53)
    cpu = refrun.run(st, 8, dump=[1, 4], first_dt=1e-4, bounds=bounds, solver=solver, emf=emf)
    codes = {"hlld": native.SOLVER_HLLD, "hllc": native.SOLVER_HLLC}
    dom = native.Domain.from_state(st, bounds=bounds, solver=codes[solver],
                                   emf_average=native.EMF_AVERAGES[emf])
    dom.set_dt(1e-4, 0.4, 1.1)
    done = 0
    for s in sorted(cpu):
        dom.run(s - done)
        done = s
        h, ref = cpu[s]
        assert_states_equal(dom.get_state(st), ref, "%s step %d" % (case, s))
        sc = dom.scalars()
        assert sc["dt"] == h["dt"] and sc["maxmach"] == h["maxmach"], (case, s)
    dom.close()


def test_bounded_outflow_40cube_divb(native):
    from oracle import refrun
    from pluto_amd import problems as P
    if not refrun.available(3):
        pytest.skip("reference executables not built (make -C oracle/ref)")
    _say("case: bounded domain, outflow, 40^3, 5 CFL steps, div.B")
    st = P.random_mhd_3d(40, seed=59)
    bounds = ("outflow",) * 6
    cpu = refrun.run(st, 5, first_dt=1e-4, bounds=bounds)
    dom = native.Domain.from_state(st, bounds=bounds)
    dom.set_dt(1e-4, 0.4, 1.1)
    dom.run(5)
    out = dom.get_state(st)
    assert_states_equal(out, cpu[5][1], "outflow 40^3")
    # cells whose lower faces get_state returns (the upper faces of their neighbours)
    bmax = max(np.abs(out.bx).max(), np.abs(out.by).max(), np.abs(out.bz).max())
    assert np.abs(P.divb(out)[1:, 1:, 1:]).max() * out.spacing()[0] / bmax <= 1e-13
    assert not np.array_equal(out.prim, refrun.run(st, 5, first_dt=1e-4)[5][1].prim)
    dom.close()


def test_bounded_refusals(native):
    from pluto_amd import problems as P
    _say("case: bounded domains refuse what they do not run")
    st = P.random_mhd_3d(8, seed=1)
    b = ("outflow",) * 6
    with pytest.raises(native.PGPUError):
        native.Domain.from_state(st, bounds=b, precision=native.PGPU_PREC_FP32_FLUX)
    with pytest.raises(native.PGPUError):
        native.Domain.from_state(st, bounds=b, pipeline=native.PIPELINE_MODULAR)
    with pytest.raises(native.PGPUError):       # SHEARING
        native.Domain.from_state(st, bounds=("outflow",) * 5 + (6,))
    with pytest.raises(native.PGPUError):
        native.Domain(st.shape, 3, st.spacing(), bounds=b, nghost=9)
    # PLM + CT reads two cells beyond the interfaces PLUTO solves
    with pytest.raises(native.PGPUError):
        native.Domain(st.shape, 3, st.spacing(), bounds=b, nghost=1)
    # an axis is periodic on both sides or on neither
    with pytest.raises(native.PGPUError):
        native.Domain(st.shape, 3, st.spacing(),
                      bounds=("periodic", "outflow", "outflow", "outflow", "outflow", "outflow"))
    per0 = native.Domain.from_state(st)
    low = (np.zeros((8, 8)),) * 3
    with pytest.raises(native.PGPUError):
        per0.set_state(st, low=low)
    with pytest.raises(native.PGPUError):
        per0.low_faces()
    per0.close()
    dom = native.Domain.from_state(st, bounds=b)
    import ctypes
    from pluto_amd.native import check, lib
    ptrs = (ctypes.c_void_p * 8)()
    with pytest.raises(native.PGPUError):
        check(lib().pgpu_state_device_ptrs(dom.h, ptrs, None))
    per = native.Domain.from_state(st)
    out = np.zeros(32)
    with pytest.raises(native.PGPUError):
        check(lib().pgpu_state_error(per.h, dom.h, out.ctypes.data_as(ctypes.POINTER(ctypes.c_double))))
    per.close()
    dom.close()


def test_bounded_dbl_matches_pluto_and_restarts(native, tmp_path):
    """.dbl output of a bounded box (the interior with its own faces below the
    first cells) against PLUTO's own files from the same run with the same
    [Boundary], byte for byte; a restart from output #2 continues to #3
    exactly."""
    from oracle import refrun
    from test_dbl_io import _records
    if not refrun.available(3):
        pytest.skip("reference executables not built (make -C oracle/ref)")
    _say("case: bounded box .dbl output and restart vs PLUTO's files, 12x10x9")
    st = _box((9, 10, 12), seed=67)
    bounds = ("outflow", "reflective", "outflow", "outflow", "reflective", "outflow")
    ref_dir = tmp_path / "ref"
    ref_dir.mkdir()
    refrun.run(st, 4, first_dt=1e-4, bounds=bounds, dbl_every=1, keep_dir=str(ref_dir))
    recs = _records((ref_dir / "restart.out").read_bytes())
    assert len(recs) >= 4
    dom = native.Domain.from_state(st, bounds=bounds)
    dom.set_dt(1e-4, 0.4, 1.1)
    out = tmp_path / "lib"
    out.mkdir()
    done = 0
    for nfile, (nstep, _, _, _) in enumerate(recs[:4]):
        dom.run(nstep - done)
        done = nstep
        dom.write_dbl(str(out), nfile)
        name = "data.%04d.dbl" % nfile
        assert (out / name).read_bytes() == (ref_dir / name).read_bytes(), name
    assert (out / "dbl.out").read_text() == "".join(
        (ref_dir / "dbl.out").read_text().splitlines(True)[:4])
    dom.close()
    # restart from PLUTO's output #2
    dom = native.Domain.from_state(st, bounds=bounds)
    dom.set_dt(1.0, 0.4, 1.1)
    dom.read_dbl(str(ref_dir), 2)
    sc = dom.scalars()
    assert (sc["time"], sc["dt"], sc["step"]) == (recs[2][2], recs[2][3], recs[2][0])
    dom.run(recs[3][0] - recs[2][0])
    again = tmp_path / "again"
    again.mkdir()
    dom.write_dbl(str(again), 3)
    assert (again / "data.0003.dbl").read_bytes() == (ref_dir / "data.0003.dbl").read_bytes()
    dom.close()


def _open_box_field(n, seed):
    """A state on a non-periodic n^3 box of the unit cube whose field is the
    discrete curl (vec_pot_diff.c:139-169) of a vector potential that is not
    periodic, so the faces below the first cells are not images of the last
    ones.  Returns the state (upper faces) and the lower faces."""
    from pluto_amd import problems as P
    rng = np.random.default_rng(seed)
    d = 1.0 / n
    i = np.arange(-1, n)                       # edge/face index, -1 = below the box
    xc, xf = (i + 0.5) * d, (i + 1.0) * d      # cell centres, upper faces
    c = rng.uniform(0.5, 1.5, size=9)

    def ax(z, y, x):
        return 0.2 * np.sin(c[0] * 2.0 * y + 0.3) * np.cos(c[1] * 3.0 * z) + 0.1 * y * z * c[2]

    def ay(z, y, x):
        return 0.2 * np.cos(c[3] * 2.5 * x - 0.2) * np.sin(c[4] * 2.0 * z) + 0.1 * x * x * c[5]

    def az(z, y, x):
        return 0.3 * np.sin(c[6] * 3.0 * x) * np.sin(c[7] * 2.0 * y + 0.1) + 0.2 * x * y * c[8]

    g = lambda a, b, e: np.meshgrid(a, b, e, indexing="ij")
    AX = ax(*g(xf, xf, xc))        # (z_{k+1/2}, y_{j+1/2}, x_i)
    AY = ay(*g(xf, xc, xf))        # (z_{k+1/2}, y_j, x_{i+1/2})
    AZ = az(*g(xc, xf, xf))        # (z_k, y_{j+1/2}, x_{i+1/2})
    # faces with their index -1 included along their own axis (first entry)
    bx = (AZ[1:, 1:, :] - AZ[1:, :-1, :]) / d - (AY[1:, 1:, :] - AY[:-1, 1:, :]) / d
    by = -(AZ[1:, :, 1:] - AZ[1:, :, :-1]) / d + (AX[1:, :, 1:] - AX[:-1, :, 1:]) / d
    bz = (AY[:, 1:, 1:] - AY[:, 1:, :-1]) / d - (AX[:, 1:, 1:] - AX[:, :-1, 1:]) / d
    z, y, x = g(xc[1:], xc[1:], xc[1:])
    rho = 1.0 + 0.2 * np.sin(2.0 * np.pi * x) * np.cos(2.0 * np.pi * z)
    v = np.stack([0.3 * np.sin(2.0 * np.pi * y), 0.2 * np.cos(2.0 * np.pi * z),
                  0.25 * np.sin(2.0 * np.pi * x + 1.0)])
    p = 1.0 + 0.1 * np.cos(2.0 * np.pi * (x + y))
    st = P.assemble(rho, v, p, np.ascontiguousarray(bx[:, :, 1:]),
                    np.ascontiguousarray(by[:, 1:, :]), np.ascontiguousarray(bz[1:]), 3,
                    (1.0, 1.0, 1.0))
    low = (np.ascontiguousarray(bx[:, :, 0]), np.ascontiguousarray(by[:, 0, :]),
           np.ascontiguousarray(bz[0]))
    # the cell-centred field is the average with the true lower faces
    st.prim[4] = 0.5 * (bx[:, :, 1:] + bx[:, :, :-1])
    st.prim[5] = 0.5 * (by[:, 1:, :] + by[:, :-1, :])
    st.prim[6] = 0.5 * (bz[1:] + bz[:-1])
    return st, low


def _divb_all(st, low):
    """div.B of every cell, the first layer included, from the upper faces
    and the lower faces of the first cells."""
    dx, dy, dz = st.spacing()
    bx = np.concatenate([low[0][:, :, None], st.bx], axis=2)
    by = np.concatenate([low[1][:, None, :], st.by], axis=1)
    bz = np.concatenate([low[2][None], st.bz], axis=0)
    return np.diff(bx, axis=2) / dx + np.diff(by, axis=1) / dy + np.diff(bz, axis=0) / dz


def test_bounded_true_lower_faces_vs_pluto(native):
    """pgpu_set_state_bounded: a solenoidal field of a non-periodic potential,
    with the box's own faces below the first cells (as PLUTO's Startup sets
    Vs at IBEG-1), runs bit for bit like PLUTO's main loop given the same
    faces, and div.B stays at round-off in every cell, the first layer
    included (the image convention would break it there)."""
    from oracle import refrun
    if not refrun.available(3):
        pytest.skip("reference executables not built (make -C oracle/ref)")
    n = 12
    st, low = _open_box_field(n, seed=71)
    bmax = max(np.abs(b).max() for b in (st.bx, st.by, st.bz))
    assert np.abs(_divb_all(st, low)).max() / n / bmax <= 1e-13
    bounds = ("outflow", "outflow", "reflective", "outflow", "outflow", "eqtsymmetric")
    _say("case: bounded box with its own lower faces, %d^3, %s, 6 CFL steps" % (n, bounds))
    cpu = refrun.run(st, 6, dump=[2], first_dt=1e-4, bounds=bounds, low=low)
    dom = native.Domain(st.shape, 3, st.spacing(), bounds=bounds)
    dom.set_state(st, low=low)
    got_low = dom.low_faces()
    for a, b in zip(got_low, low):
        assert np.array_equal(a, b)
    dom.set_dt(1e-4, 0.4, 1.1)
    done = 0
    for s in sorted(cpu):
        dom.run(s - done)
        done = s
        h, ref = cpu[s]
        out = dom.get_state(st)
        assert_states_equal(out, ref, "lower faces step %d" % s)
        sc = dom.scalars()
        assert sc["dt"] == h["dt"] and sc["maxmach"] == h["maxmach"], s
        lo = dom.low_faces()
        bm = max(np.abs(b).max() for b in (out.bx, out.by, out.bz))
        assert np.abs(_divb_all(out, lo)).max() / n / bm <= 1e-13, s
    # the image convention differs from PLUTO's run with the true faces
    img = native.Domain.from_state(st, bounds=bounds)
    img.set_dt(1e-4, 0.4, 1.1)
    img.run(2)
    assert not np.array_equal(img.get_state(st).prim, cpu[2][1].prim)
    img.close()
    dom.close()


def _pluto_centres(n, ng, length):
    """PLUTO's cell centres along one uniform axis, ghosts included
    (set_grid.c:52-95: interior xl = xL + (i - iL)*dx, xr = xl + dx; the
    ghosts continue from the first and last interior cell; x = (xl + xr)/2)."""
    dx = length / float(n)
    xl = np.empty(n + 2 * ng)
    xr = np.empty(n + 2 * ng)
    for i in range(n):
        xl[ng + i] = 0.0 + float(i) * dx
        xr[ng + i] = xl[ng + i] + dx
    iL, iR = ng, ng + n - 1
    for i in range(ng):
        xl[i] = xl[iL] - (ng - i) * dx
        xr[i] = xl[i] + dx
        xl[iR + i + 1] = xl[iR] + (i + 1.0) * dx
        xr[iR + i + 1] = xl[iR] + (i + 2.0) * dx
    return 0.5 * (xl + xr)


def _userdef_hook(dom, x2):
    """The USERDEF sides of oracle/ref/init_io.c's UserDefBoundary on a slab:
    an inflow at X1_BEG (reading the first interior cell, the stage and the
    time), a zero-gradient copy with the normal velocity halved elsewhere;
    then the transverse cell-centred average of the side's ghost cells
    (ct_field_average.c:275-457)."""

    def hook(side, stage, slab):
        vc, vs = slab.arrays()
        lo, t = list(slab.lo), list(slab.tot)
        beg, end = list(slab.beg), list(slab.end)
        a = side // 2

        def rng(x, l, h):          # PLUTO index range -> slab slice
            return slice(l - lo[x], h - lo[x] + 1)

        # the centre box and face boxes (boundary.c:144-165)
        c_lo, c_hi = [0, 0, 0], [t[0] - 1, t[1] - 1, t[2] - 1]
        if side & 1:
            c_lo[a] = end[a] + 1
        else:
            c_hi[a] = beg[a] - 1

        def box(face):
            l, h = list(c_lo), list(c_hi)
            if face is not None:
                l[face] -= 1
            return (rng(2, l[2], h[2]), rng(1, l[1], h[1]), rng(0, l[0], h[0]))

        C = box(None)
        if side == 0:
            time = dom.scalars()["time"]
            xc = x2[c_lo[1]:c_hi[1] + 1][None, :, None]
            vc[0][C] = 1.2 + 0.5 * time
            vc[1][C] = 0.3
            vc[2][C] = 0.05 * stage
            vc[3][C] = 0.02 * xc
            vc[4][C] = 0.1
            vc[5][C] = 0.2
            vc[6][C] = -0.1
            vc[7][C] = vc[7][rng(2, c_lo[2], c_hi[2]), rng(1, c_lo[1], c_hi[1]),
                             rng(0, beg[0], beg[0])]
            vs[0][box(0)] = 0.1
            vs[1][box(1)] = 0.2
            l3, h3 = list(c_lo), list(c_hi)
            l3[2] -= 1
            vs[2][box(2)] = -0.1 + 0.01 * x2[l3[1]:h3[1] + 1][None, :, None]
        else:
            src = end[a] if side & 1 else beg[a]
            sl = [rng(2, c_lo[2], c_hi[2]), rng(1, c_lo[1], c_hi[1]), rng(0, c_lo[0], c_hi[0])]
            sl[2 - a] = rng(a, src, src)
            for q in range(8):
                vc[q][C] = vc[q][tuple(sl)]
            vc[1 + a][C] = 0.5 * vc[1 + a][tuple(sl)]
            for f in range(3):
                if f == a:
                    continue
                B = box(f)
                fl, fh = list(c_lo), list(c_hi)
                fl[f] -= 1
                ss = [rng(2, fl[2], fh[2]), rng(1, fl[1], fh[1]), rng(0, fl[0], fh[0])]
                ss[2 - a] = rng(a, src, src)
                vs[f][B] = vs[f][tuple(ss)]
        # CT_AverageTransverseMagField over the side's ghost cells
        Z, Y, X = C
        if a != 0:
            vc[4][C] = 0.5 * (vs[0][C] + vs[0][Z, Y, slice(X.start - 1, X.stop - 1)])
        if a != 1:
            vc[5][C] = 0.5 * (vs[1][C] + vs[1][Z, slice(Y.start - 1, Y.stop - 1), X])
        if a != 2:
            vc[6][C] = 0.5 * (vs[2][C] + vs[2][slice(Z.start - 1, Z.stop - 1), Y, X])

    return hook


@pytest.mark.parametrize("bounds", [
    ("userdef", "outflow", "periodic", "periodic", "reflective", "userdef"),
    ("userdef",) * 6])
def test_bounded_userdef_hook_vs_pluto(native, bounds):
    """USERDEF sides of a resident bounded box through a host hook
    (pgpu_set_userdef_boundary) written like oracle/ref/init_io.c's
    UserDefBoundary: states, dt and Mach bit for bit against PLUTO's main
    loop running that UserDefBoundary."""
    from oracle import refrun
    if not refrun.available(3):
        pytest.skip("reference executables not built (make -C oracle/ref)")
    shape = (9, 10, 12)
    _say("case: bounded box with USERDEF sides %s, %s, 5 CFL steps" % (bounds, shape))
    st = _box(shape, seed=83)
    cpu = refrun.run(st, 5, dump=[1, 3], first_dt=1e-4, bounds=bounds)
    dom = native.Domain.from_state(st, bounds=bounds)
    x2 = _pluto_centres(shape[1], 2, st.length[1])
    dom.set_userdef_boundary(_userdef_hook(dom, x2))
    dom.set_dt(1e-4, 0.4, 1.1)
    done = 0
    for s in sorted(cpu):
        dom.run(s - done)
        done = s
        h, ref = cpu[s]
        assert_states_equal(dom.get_state(st), ref, "USERDEF step %d" % s)
        sc = dom.scalars()
        assert sc["dt"] == h["dt"] and sc["maxmach"] == h["maxmach"], s
    # without a hook a USERDEF side is an error, not a silent skip
    dom.set_userdef_boundary(None)
    with pytest.raises(native.PGPUError, match="USERDEF"):
        dom.run(1)
    dom.close()


def _lower(faces):
    """The last face planes: what lies below the first cells of a periodic box."""
    bx, by, bz = faces
    return [bx[:, :, -1].copy(), by[:, -1, :].copy(), bz[-1].copy()]


def _centres_with(st, low):
    """The first cells' centred field as set_state(low=...) forms it."""
    st.prim[4][:, :, 0] = 0.5 * (st.bx[:, :, 0] + low[0])
    st.prim[5][:, 0, :] = 0.5 * (st.by[:, 0, :] + low[1])
    st.prim[6][0] = 0.5 * (st.bz[0] + low[2])


def _bounded_vs_oracle(native, st, low, bounds, nghost, what):
    from oracle import oracle as O
    dom = native.Domain(st.shape, 3, st.spacing(), bounds=bounds, nghost=nghost)
    dom.set_state(st, low=low)
    dom.set_dt(1e-3, 0.3, 1.1)
    dom.run(3)
    out = dom.get_state(st)
    lows = dom.low_faces()
    dom.close()
    ref = st.copy()
    _centres_with(ref, low)
    O.run(ref, 3, 1e-3, cfl=0.3)
    assert_states_equal(out, ref, what)
    return lows, _lower((ref.bx, ref.by, ref.bz))


# the ghost fill of periodic axes, the faces below the first cells differing
# from the last faces (which the fill replaces them by): extents equal to the
# ghost zones, odd and larger ones
@pytest.mark.parametrize("shape,nghost", [((3, 3, 3), 3), ((5, 7, 9), 2), ((12, 5, 17), 4), ((33, 20, 70), 2)])
def test_periodic_sides_with_other_lower_faces(native, shape, nghost):
    _say("case: bounded all-periodic %s, %d ghost zones, lower faces of their own" % (shape, nghost))
    st = _box(shape, seed=61)
    rng = np.random.default_rng(67)
    low = [a + 0.05 * rng.standard_normal(a.shape) for a in _lower((st.bx, st.by, st.bz))]
    lows, ref = _bounded_vs_oracle(native, st, low, ("periodic",) * 6, nghost, "all periodic %s" % (shape,))
    for a, b in zip(lows, ref):
        assert np.array_equal(a, b)


# periodic axes before outflow ones (X1 is filled first, X3 last: an outflow
# fill reads the faces below the first cells of the periodic axes after it as
# they were): a state that varies along one periodic axis only, so that an
# outflow ghost zone holds what a periodic one does (exactly: face areas are
# powers of two and the other axes' differences vanish)
@pytest.mark.parametrize("axis,periodic", [(0, 1), (0, 2), (1, 2)])
@pytest.mark.parametrize("extents,nghost", [((9, 4, 3), 2), ((3, 3, 3), 3), ((70, 5, 8), 2)])
def test_periodic_axes_before_outflow(native, axis, periodic, extents, nghost):
    from pluto_amd import problems as P
    n = [extents[(a - axis) % 3] for a in range(3)]   # x, y, z
    shape = (n[2], n[1], n[0])
    _say("case: bounded %s varying along axis %d, the first %d axes periodic" % (shape, axis, periodic))
    rng = np.random.default_rng(71)
    line = [1] * 3
    line[2 - axis] = n[axis]

    def wave(lo, amp):
        return np.broadcast_to((lo + amp * rng.standard_normal(n[axis])).reshape(line), shape).copy()

    b = [wave(0.3, 0.2) for _ in range(3)]
    b[axis][:] = 0.75
    v = np.stack([wave(0.0, 0.3) for _ in range(3)])
    st = P.assemble(wave(1.0, 0.1), v, wave(1.0, 0.1), *b, 3, tuple(0.25 * x for x in n))
    low = _lower(b)
    low[axis] += 0.0625
    bounds = ["periodic" if a < periodic else "outflow" for a in (0, 0, 1, 1, 2, 2)]
    _bounded_vs_oracle(native, st, low, bounds, nghost, "axis %d of %s" % (axis, shape))
