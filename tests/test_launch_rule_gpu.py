"""Launch shapes on extents that divide nothing: block orders over any block
count, balanced t-chunks, partly filled tile blocks, and the built-in rule's
own shapes.  Every kernel variant applies the same operations in the same
order, so each result is bitwise the gather kernel's in plain block order;
that one is held to the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = {0: 1e-13, 1: 2e-6, 2: 4e-3}  # as the hopping tests: storage precision F64, F32, F16


@pytest.fixture(scope="module")
def hp():
    from plqcd_amd import hopping
    return hopping


def set_shape(prec, shape):
    from plqcd_amd import capi
    if shape is None:
        assert capi.lib().plqcd_hip_hop_tuning_reset(prec) == 0
    else:
        assert capi.lib().plqcd_hip_hop_tuning(prec, *shape) == 0


def fields(hp, L, prec, links, R):
    V = int(np.prod(L))
    lat = hp.Lattice(L)
    u = hp.random_gauge_su3(V, 5)
    g = hp.Gauge(lat, prec, links).upload(u)
    fi, fo = hp.Field(lat, prec, R), hp.Field(lat, prec, R)
    qs = [hp.random_spinor(V, 50 + r) for r in range(R)]
    for r, q in enumerate(qs):
        fi.upload(q, r)
    return lat, g, fi, fo, qs, u


# order, group, block, tmarch, rb, tile_y, tile_z
SHAPES = [(1, 1, 64, 0, 1, 0, 0), (2, 8, 64, 0, 1, 0, 0), (2, 3, 128, 0, 1, 0, 0), (1, 1, 64, 1, 1, 0, 0),
          (2, 8, 64, 3, 1, 0, 0), (1, 1, 128, 4, 1, 0, 0), (2, 5, 64, 7, 1, 0, 0), (1, 1, 256, 64, 1, 0, 0), None]
TILES = [(1, 1, 256, 3, 1, 3, 1), (2, 8, 256, 4, 1, 3, 2), (1, 1, 256, 5, 1, 1, 7), (0, 1, 256, 64, 1, 6, 1)]


@pytest.mark.parametrize("L", [(4, 6, 14, 10), (10, 6, 14, 6)])
@pytest.mark.parametrize("prec,links,R", [(0, 18, 1), (1, 12, 1), (2, 18, 1), (0, 12, 3), (1, 18, 5), (2, 12, 12)])
def test_shapes_on_ragged_extents(hp, L, prec, links, R):
    import oracle
    lat, g, fi, fo, qs, u = fields(hp, L, prec, links, R)
    try:
        for mode in (hp.HOP_WILSON, hp.HOP_COMPAT):
            set_shape(prec, (0, 1, 256, 0, 1, 0, 0))
            hp.hop(g, fi, fo, hp.PARITY_ALL, mode)
            want = [fo.download(r) for r in range(R)]
            ref = oracle.hopping_full(qs[-1], u, L, mode)
            assert np.abs(want[-1] - ref).max() <= TOL[prec] * np.abs(ref).max()
            for shape in SHAPES + (TILES if R == 1 else []):
                set_shape(prec, shape)
                for r in range(R):
                    fo.upload(np.zeros_like(qs[0]), r)
                hp.hop(g, fi, fo, hp.PARITY_ALL, mode)
                for r in range(R):
                    assert np.array_equal(fo.download(r), want[r]), (mode, shape, r)
    finally:
        set_shape(prec, None)


def test_solver_shapes_on_ragged_extents(hp):
    """The norms' reduction chunks over balanced t-chunks and partly filled
    tiles: a solve takes the same iterates to the same bits."""
    from plqcd_amd import solver
    L = (8, 6, 10, 14)
    lat, g, b, x, qs, u = fields(hp, L, hp.PREC_F64, 18, 1)
    want = None
    try:
        for shape in ((0, 1, 256, 0, 1, 0, 0), (1, 1, 128, 5, 1, 0, 0), (1, 1, 256, 3, 1, 2, 5), None):
            set_shape(hp.PREC_F64, shape)
            st = solver.cg_solve(g, b, x, 0.12, 1e-10)
            got = (st[0]["iterations"], st[0]["true_residual"], x.download())
            assert st[0]["converged"]
            if want is None:
                want = got
            assert got[:2] == want[:2] and np.array_equal(got[2], want[2]), shape
    finally:
        set_shape(hp.PREC_F64, None)


def test_batch_of_small_ragged_lattices(hp):
    """Every item of a batch is bitwise its own launch."""
    shapes = [(4, 6, 14, 10), (4, 4, 4, 4), (6, 10, 4, 22)]
    sets = [fields(hp, L, hp.PREC_F32, 12, R) for L, R in zip(shapes, (4, 1, 12))]
    stream = hp.lib().plqcd_hip_lattice_stream(sets[0][0].h)
    for s in sets:
        s[0].set_stream(stream)
    for mode in (hp.HOP_WILSON, hp.HOP_COMPAT):
        want = []
        for lat, g, fi, fo, qs, u in sets:
            hp.hop(g, fi, fo, hp.PARITY_ALL, mode)
            want.append([fo.download(r) for r in range(fo.nrhs)])
            for r in range(fo.nrhs):
                fo.upload(np.zeros_like(qs[0]), r)
        hp.hop_batch([s[1] for s in sets], [s[2] for s in sets], [s[3] for s in sets], mode)
        for s, w in zip(sets, want):
            for r in range(s[3].nrhs):
                assert np.array_equal(s[3].download(r), w[r]), (s[0].L, mode, r)


# smallest lattices on which a half-lattice launch streams its links (a gauge
# field of 75 MiB) and sweeps slabs (200 MiB of the input), and one below both
@pytest.mark.parametrize("L,prec,links,R", [((16, 16, 18, 32), 0, 18, 1), ((16, 16, 18, 32), 0, 18, 4),
                                            ((12, 18, 10, 22), 0, 12, 12), ((20, 16, 18, 32), 1, 18, 12),
                                            ((4, 6, 6, 4), 2, 12, 5)])
def test_half_lattice_orders(hp, L, prec, links, R):
    """The built-in rule's orders and link loads give bitwise the plain order's
    output, on each parity, and leave the other alone."""
    lat, g, fi, fo, qs, u = fields(hp, L, prec, links, R)
    mark = np.full_like(qs[0], 3.0)
    half = len(mark) // 2
    try:
        for mode, parity in ((hp.HOP_WILSON, 0), (hp.HOP_COMPAT, 1)):
            mine = slice(parity * half, (parity + 1) * half)
            other = slice((1 - parity) * half, (2 - parity) * half)
            got = []
            for shape in ((0, 1, 256, 0, 1, 0, 0), None):
                set_shape(prec, shape)
                for r in range(R):
                    fo.upload(mark, r)
                hp.hop(g, fi, fo, parity, mode)
                got.append([fo.download(r) for r in range(R)])
            for want, out in zip(*got):
                assert np.array_equal(out[mine], want[mine])
                assert np.array_equal(out[other], mark[other])
                assert not np.array_equal(out[mine], mark[mine])
    finally:
        set_shape(prec, None)


@pytest.mark.parametrize("prec,links", [(0, 18), (2, 12)])
def test_iterations_enqueued_ahead(hp, prec, links):
    """Solves stopped after 1 .. 9 iterations (whole and broken groups of four,
    updates inside and at the end of one) take the iterates that direct
    launches without graphs take; the iteration count is exact."""
    from plqcd_amd import solver
    L = (4, 6, 4, 10)
    lat, g, b, x, qs, u = fields(hp, L, hp.PREC_F64, 18, 3)
    gs = None if prec == hp.PREC_F64 else hp.Gauge(lat, prec, links).upload(u)
    x2 = hp.Field(lat, hp.PREC_F64, 3)
    tol = [1e-10, 1e-3, 1e-6]  # slots that stop at different iterations
    for most in (1, 2, 3, 4, 5, 7, 8, 9, 200):
        st = solver.cg_solve(g, b, x, 0.12, tol, max_iter=most, sloppy=gs)
        st2 = solver.cg_solve(g, b, x2, 0.12, tol, max_iter=most, sloppy=gs, use_graph=False)
        for r in range(3):
            assert st[r]["iterations"] <= most
            assert st[r]["converged"] or st[r]["iterations"] == most
            assert st[r]["iterations"] == st2[r]["iterations"]
            assert np.array_equal(x.download(r), x2.download(r))
            # alone, the slot takes the same iterates
            b1, x1 = hp.Field(lat).upload(qs[r]), hp.Field(lat)
            s1 = solver.cg_solve(g, b1, x1, 0.12, tol[r], max_iter=most, sloppy=gs)[0]
            assert s1["iterations"] == st[r]["iterations"]
            assert np.array_equal(x1.download(), x.download(r))


@pytest.mark.parametrize("R", [1, 16, 17, 40])
def test_kappa_with_the_launch_and_from_memory(hp, R):
    """M, M^+ and the Schur operator with as many kappas as travel with a launch
    and one more: every RHS is bitwise its own one-RHS call."""
    from plqcd_amd import solver
    L = (4, 6, 4, 6)
    lat, g, fi, fo, qs, u = fields(hp, L, hp.PREC_F64, 18, R)
    ft = hp.Field(lat, hp.PREC_F64, R)
    f1, o1, t1 = hp.Field(lat), hp.Field(lat), hp.Field(lat)
    kap = [0.1 + 0.001 * r for r in range(R)]
    half = len(qs[0]) // 2
    for dagger in (False, True):
        solver.apply_m(g, fi, fo, kap, dagger)
        for r in (0, R // 2, R - 1):
            solver.apply_m(g, f1.upload(qs[r]), o1, kap[r], dagger)
            assert np.array_equal(fo.download(r), o1.download()), (dagger, r)
    solver.apply_schur(g, fi, ft, fo, kap, 1)
    for r in (0, R // 2, R - 1):
        solver.apply_schur(g, f1.upload(qs[r]), t1, o1, kap[r], 1)
        assert np.array_equal(fo.download(r)[half:], o1.download()[half:]), r
