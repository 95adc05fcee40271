"""The hybrid Schwarz multigrid preconditioner on the GPU (csrc/hsmg.hip)
against its oracle (oracle/hsmg.py, pinned in test_oracle_hsmg.py), and
GMRES + HSMG, the pressure solver of the shipped cases.

Bars (FP64): one application z = M^-1 r within 1e-10 of the oracle's,
relative to max|z|, at p = 7, 5 and 3 (the device's eigen-solver and sums
differ from numpy's in rounding only; the FDM result does not depend on the
eigenvector basis); GMRES + HSMG reaches 1e-9 in the same number of
iterations as the oracle's GMRES + HSMG (within 1) and far fewer than
Jacobi; the solution agrees with PCG's."""
import numpy as np
import pytest

import oracle
from oracle import hsmg as ohsmg
from oracle import krylov

pytestmark = pytest.mark.gpu

SHAPES = [(4, 3, 2, 8), (3, 3, 2, 6), (3, 2, 2, 4)]


@pytest.fixture(scope="module", params=SHAPES, ids=lambda s: f"{s[0]}x{s[1]}x{s[2]}_lx{s[3]}")
def pair(request):
    from nekoamd import device, sem
    device.init(0)
    nx, ny, nz, lx = request.param
    g = sem.BoxCase(nx, ny, nz, lx, jitter=0.05, seed=1234)
    M = sem.HSMG(g)
    Mo = ohsmg.HSMG(nx, ny, nz, lx)
    return g, M, Mo


def test_hsmg_apply_matches_oracle(pair):
    g, M, Mo = pair
    c = Mo.c3
    rng = np.random.default_rng(11)
    r = c.gs(c.B * rng.standard_normal(c.n))
    r[oracle.face_mask(c.nx, c.ny, c.nz, c.lx, oracle.PRS_DIRICHLET)] = 0.0
    z = g.field()
    M.apply(z, g.field(r))
    zr = Mo.apply(r)
    err = np.abs(z.get() - zr).max() / np.abs(zr).max()
    print(f"lx={c.lx}: HSMG apply error {err:.1e}")
    assert err < 1e-10


@pytest.mark.parametrize("graphs", [False, True], ids=["kernels", "graph"])
def test_repeated_applies_match_oracle(pair, graphs, monkeypatch):
    """Four applications in a row on different inputs, with eager work (a gs
    and host reads) between them, each within the bar.  With
    NEKOAMD_HIP_GRAPHS=1 when the multigrid is created, its coarse solve is a
    HIP graph recorded from kernel nodes on the first application and replayed
    on a side stream after: every replay equals the one-kernel result bit for
    bit (the same sums in the same order)."""
    from nekoamd import sem
    g, M, Mo = pair
    Mg = None
    if graphs:
        monkeypatch.setenv("NEKOAMD_HIP_GRAPHS", "1")
        Mg = sem.HSMG(g)
    c = Mo.c3
    mask = oracle.face_mask(c.nx, c.ny, c.nz, c.lx, oracle.PRS_DIRICHLET)
    rng = np.random.default_rng(21)
    z = g.field()
    zg = g.field()
    for k in range(4):
        r = c.gs(c.B * rng.standard_normal(c.n))
        r[mask] = 0.0
        rd = g.field(r)
        M.apply(z, rd)
        zr = Mo.apply(r)
        err = np.abs(z.get() - zr).max() / np.abs(zr).max()
        print(f"lx={c.lx} application {k}: error {err:.1e}")
        assert err < 1e-10, k
        if Mg is not None:
            Mg.apply(zg, rd)
            assert np.array_equal(zg.get(), z.get()), k
        g.gs.op(rd)                    # eager work between replays
        assert np.isfinite(rd.get()).all()


def test_gmres_hsmg_matches_oracle(pair):
    from nekoamd import sem
    g, M, Mo = pair
    c = Mo.c3
    maskh = oracle.face_mask(c.nx, c.ny, c.nz, c.lx, oracle.PRS_DIRICHLET)
    rng = np.random.default_rng(12)
    f = c.gs(c.B * rng.standard_normal(c.n))
    f[maskh] = 0.0

    def A(u):
        w = c.gs(c.ax(u))
        w[maskh] = 0.0
        return w

    xr, itr, _, rr, _ = krylov.gmres(A, Mo.apply, f, c.mult, c.volume, m=30, abstol=1e-9,
                                     max_iter=500)
    mask = g.mask(oracle.PRS_DIRICHLET)
    one = g.field(np.ones(c.n))
    gm = sem.GMRES(g, m=30)
    x = g.field()
    mon = gm.solve(x, g.field(f), M, mask, one, abstol=1e-9, max_iter=500)
    dd = g.field()
    g.jacobi(dd, one)
    xj = g.field()
    monj = gm.solve(xj, g.field(f), dd, mask, one, abstol=1e-9, max_iter=5000)
    err = np.abs(x.get() - xr).max() / np.abs(xr).max()
    print(f"lx={c.lx}: GMRES+HSMG iterations gpu {mon.iter} oracle {itr}; "
          f"GMRES+Jacobi {monj.iter}; x err {err:.1e}")
    assert mon.done == 1 and mon.res_final < 1e-9
    assert abs(mon.iter - itr) <= 1
    assert err < 1e-7
    assert mon.iter * 4 <= monj.iter
    assert np.abs(x.get() - xj.get()).max() < 1e-5 * np.abs(xj.get()).max()


def test_fp32_hsmg_inside_fp64_gmres(pair):
    """The FP32 data path (NEKOAMD_CG_MIXED): one application agrees with
    the FP64 one to FP32 rounding (5e-5 relative), and the FP64 flexible
    GMRES with it reaches 1e-9 on its FP64 residual with at most two more
    iterations than with the FP64 preconditioner."""
    from nekoamd import sem
    g, M, Mo = pair
    c = Mo.c3
    M32 = sem.HSMG(g, mixed=True)
    maskh = oracle.face_mask(c.nx, c.ny, c.nz, c.lx, oracle.PRS_DIRICHLET)
    rng = np.random.default_rng(13)
    f = c.gs(c.B * rng.standard_normal(c.n))
    f[maskh] = 0.0
    z64, z32 = g.field(), g.field()
    M.apply(z64, g.field(f))
    M32.apply(z32, g.field(f))
    d = np.abs(z32.get() - z64.get()).max() / np.abs(z64.get()).max()
    mask = g.mask(oracle.PRS_DIRICHLET)
    one = g.field(np.ones(c.n))
    gm = sem.GMRES(g, m=30)
    x64, x32 = g.field(), g.field()
    m64 = gm.solve(x64, g.field(f), M, mask, one, abstol=1e-9, max_iter=500)
    m32 = gm.solve(x32, g.field(f), M32, mask, one, abstol=1e-9, max_iter=500)
    err = np.abs(x32.get() - x64.get()).max() / np.abs(x64.get()).max()
    print(f"lx={c.lx}: FP32 vs FP64 HSMG apply {d:.1e}; GMRES iterations FP64 pc {m64.iter}, "
          f"FP32 pc {m32.iter}; solutions differ by {err:.1e}")
    assert d < 5e-5
    assert m32.done == 1 and m32.res_final < 1e-9
    assert m32.iter <= m64.iter + 2
    assert err < 1e-6


@pytest.mark.parametrize("box", [(1, 1, 1), (9, 7, 5), (12, 9, 7), (58, 58, 1), (61, 61, 1)])
def test_coarse_kernel_equals_launches(box, monkeypatch):
    """The coarse solve as one kernel against its launches (the ones a HIP
    graph records), bit for bit: one element, two blocks of vertices in one
    workgroup, a last workgroup with one block, the largest plane whose range
    fits the kernel and one past it (launches on both sides)."""
    from nekoamd import device, sem
    device.init(0)
    g = sem.BoxCase(*box, 4, jitter=0.05, seed=1234)
    M = sem.HSMG(g)
    monkeypatch.setenv("NEKOAMD_HIP_GRAPHS", "1")
    Mg = sem.HSMG(g)
    rng = np.random.default_rng(5)
    z, zg = g.field(), g.field()
    for _ in range(3):
        r = g.field(rng.standard_normal(g.n))
        g.gs.op(r)
        M.apply(z, r)
        Mg.apply(zg, r)
        assert np.array_equal(z.get(), zg.get()) and np.isfinite(z.get()).all()
        assert z.get().any()
        assert Mg.path == Mg.BY_LAUNCHES
        assert M.path == (M.BY_LAUNCHES if box[0] > 58 else M.ONE_KERNEL)


@pytest.mark.parametrize("box", [(1, 1, 1), (12, 9, 7), (16, 16, 16)])
def test_coarse_kernel_with_waits_given_up(box, monkeypatch):
    """All waits of the coarse kernel given up at once: the application is
    finished by one workgroup (its sums in another order: the rounding of ten
    iterations of a preconditioner, 1e-12), the next ones take the launches
    (bit for bit) and a new wait the kernel again.  Three applications queued
    without a host wait between them are right whichever of the two ways
    each takes."""
    from nekoamd import device, sem
    device.init(0)
    g = sem.BoxCase(*box, 4, jitter=0.05, seed=1234)
    M = sem.HSMG(g)
    monkeypatch.setenv("NEKOAMD_HIP_GRAPHS", "1")
    Mg = sem.HSMG(g)
    rng = np.random.default_rng(6)
    rs = [g.field(rng.standard_normal(g.n)) for _ in range(3)]
    zs = [g.field() for _ in rs]
    want = []
    for r, z in zip(rs, zs):
        g.gs.op(r)
        Mg.apply(z, r)
        want.append(z.get())

    def close(z, w):
        return np.abs(z.get() - w).max() <= 1e-12 * np.abs(w).max()

    z = zs[0]
    M.set_wait(0)
    M.apply(z, rs[0])
    assert M.path == M.ONE_WORKGROUP and close(z, want[0])
    for k in (1, 2):
        M.apply(z, rs[k])
        assert M.path == M.BY_LAUNCHES and np.array_equal(z.get(), want[k])
    M.set_wait(10**6)
    M.apply(z, rs[0])
    assert M.path == M.ONE_KERNEL and np.array_equal(z.get(), want[0])
    M.set_wait(0)
    for r, z in zip(rs, zs):
        M.apply(z, r)
    device.sync()
    assert all(close(z, w) for z, w in zip(zs, want))


@pytest.mark.parametrize("crs_iter", [1, 2, 10])
def test_captured_application_replays(crs_iter):
    """An application captured from the library stream by the caller: every
    replay, with eager applications between them, equals the eager result bit
    for bit.  One coarse iteration takes the launches."""
    import ctypes as C
    from nekoamd import device, sem
    from nekoamd._lib import lib
    device.init(0)
    hip = C.CDLL("libamdhip64.so")

    def ok(rc):
        assert rc == 0, rc
    stream = C.c_void_p(lib().nekoamd_stream())
    g = sem.BoxCase(16, 8, 8, 4, jitter=0.05, seed=1234)
    M = sem.HSMG(g, crs_iter=crs_iter)
    rng = np.random.default_rng(8)
    r, z, zg = g.field(), g.field(), g.field()
    other = g.field(rng.standard_normal(g.n))
    M.apply(z, r)  # the side stream is made on the first application
    assert M.path == (M.ONE_KERNEL if crs_iter > 1 else M.BY_LAUNCHES)
    graph, run = C.c_void_p(), C.c_void_p()
    ok(hip.hipStreamBeginCapture(stream, 2))  # relaxed
    M.apply(zg, r)
    ok(hip.hipStreamEndCapture(stream, C.byref(graph)))
    ok(hip.hipGraphInstantiate(C.byref(run), graph, None, None, 0))
    for k in range(5):
        v = g.field(rng.standard_normal(g.n))
        g.gs.op(v)
        r.copy_from(v)
        ok(hip.hipGraphLaunch(run, stream))
        device.sync()
        got = zg.get()
        if k % 2:
            M.apply(z, other)
        M.apply(z, r)
        assert np.array_equal(got, z.get()) and got.any()
    ok(hip.hipGraphExecDestroy(run))
    ok(hip.hipGraphDestroy(graph))
