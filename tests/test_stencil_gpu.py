"""GPU parity of the stencil engine (through libpattern's C ABI) vs the oracle.

Bar: bit-exact against the FP32 oracle (same rule, same operation order, no
contraction on either side).  The FP64 error is reported for the heat3D
workload (128^3, seed 42, 100 steps).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def run_dev(pa, g, nsteps, **kw):
    nz, ny, nx = (s - 2 for s in g.shape)
    a = pa.DeviceArray.from_numpy(g)
    b = a.clone()
    out = pa.heat3d_run_dev(a, b, nx, ny, nz, nsteps, **kw)
    pa.sync()
    return out.numpy()


@pytest.mark.parametrize("shape", [(1, 1, 1), (63, 7, 5), (65, 9, 17), (130, 3, 2), (64, 16, 33), (200, 33, 12)])
def test_lds25d_bitexact_ragged(pa, orc, gpu, shape):
    nx, ny, nz = shape
    g = pa.gen_heat3d(nx, ny, nz, seed=11)
    ref = orc.heat3d(g, 3)
    got = run_dev(pa, g, 3, variant=pa.PAT_STENCIL_LDS25D)
    assert np.array_equal(got, ref)


@pytest.mark.parametrize("bx,by,zc", [(64, 4, 1), (64, 8, 3), (64, 16, 8), (64, 8, 64), (32, 16, 5), (128, 4, 2),
                                      (128, 4, 7)])
def test_lds25d_tiles(pa, orc, gpu, bx, by, zc):
    nx, ny, nz = 97, 41, 23
    g = pa.gen_heat3d(nx, ny, nz, seed=12)
    ref = orc.heat3d(g, 4)
    got = run_dev(pa, g, 4, variant=pa.PAT_STENCIL_LDS25D, bx=bx, by=by, zc=zc)
    assert np.array_equal(got, ref)


@pytest.mark.parametrize("shape", [(1, 1, 1), (2, 3, 4), (60, 12, 5), (61, 13, 17), (130, 29, 2), (64, 57, 33),
                                   (200, 33, 12)])
@pytest.mark.parametrize("steps", [1, 2, 5])
def test_temporal2_bitexact_ragged(pa, orc, gpu, shape, steps):
    """Two fused sweeps per pass: every window and chunk edge, odd step counts."""
    nx, ny, nz = shape
    g = pa.gen_heat3d(nx, ny, nz, seed=21)
    ref = orc.heat3d(g, steps)
    for by, zc in ((16, 1), (32, 3), (16, 64), (8, 2), (8, 5)):
        got = run_dev(pa, g, steps, variant=pa.PAT_STENCIL_TEMPORAL2, bx=64, by=by, zc=zc)
        assert np.array_equal(got, ref), (by, zc)


def test_temporal2_handle_replay(pa, orc, gpu):
    nx, ny, nz = 70, 50, 40
    g = pa.gen_heat3d(nx, ny, nz, seed=15)
    s = pa.Stencil(nx, ny, nz)
    s.set_variant(pa.PAT_STENCIL_TEMPORAL2, 64, 32, 8)
    s.upload(g)
    s.run(7)
    s.run(7)  # replays the captured graph from the other buffer
    s.run(6)
    tot, kms = s.run_timed(3)
    got = s.download()
    s.close()
    assert len(kms) == 3 and np.all(kms > 0)
    assert np.array_equal(got, orc.heat3d(g, 23))


@pytest.mark.parametrize("shape", [(1, 1, 1), (2, 3, 4), (15, 17, 16), (16, 16, 16), (33, 9, 31), (61, 13, 17),
                                   (130, 29, 2)])
@pytest.mark.parametrize("steps", [1, 3, 4, 9])
def test_cubes_bitexact_ragged(pa, orc, gpu, shape, steps):
    """Several sweeps per launch on LDS blocks: every block edge, grids
    smaller than one block, step counts that leave sweeps over for the
    plain kernel."""
    nx, ny, nz = shape
    g = pa.gen_heat3d(nx, ny, nz, seed=23)
    ref = orc.heat3d(g, steps)
    for cube in range(5):
        got = run_dev(pa, g, steps, variant=pa.PAT_STENCIL_CUBES, bx=cube)
        assert np.array_equal(got, ref), cube


def test_cubes_handle_replay_and_errors(pa, orc, gpu):
    nx, ny, nz = 70, 50, 40
    g = pa.gen_heat3d(nx, ny, nz, seed=16)
    s = pa.Stencil(nx, ny, nz)
    with pytest.raises(RuntimeError):
        s.set_variant(pa.PAT_STENCIL_CUBES, 5, 0, 0)  # no such shape
    s.set_variant(pa.PAT_STENCIL_CUBES, 2, 0, 0)  # 16^3 blocks, 4 sweeps per launch
    s.upload(g)
    s.run(8)
    s.run(8)  # replays the captured graph from the other buffer
    s.run(5)
    tot, kms = s.run_timed(6)
    got = s.download()
    s.close()
    assert len(kms) == 6 and np.all(kms > 0)
    assert np.array_equal(got, orc.heat3d(g, 27))


def test_naive_bitexact(pa, orc, gpu):
    g = pa.gen_heat3d(45, 30, 20, seed=13)
    ref = orc.heat3d(g, 4)
    got = run_dev(pa, g, 4, variant=pa.PAT_STENCIL_GENERIC)
    assert np.array_equal(got, ref)


def test_heat3d_workload_128(pa, orc, gpu):
    """heat3D workload: 128^3, seed 42, 100 steps; bit-exact vs FP32 oracle."""
    n = 128
    g = pa.gen_heat3d(n, n, n, seed=42)
    ref = orc.heat3d(g, 100, threads=8)
    s = pa.Stencil(n, n, n, alpha=0.1)
    s.upload(g)
    s.run(100)
    got = s.download()
    s.close()
    assert np.array_equal(got, ref)
    ref64 = orc.heat3d(g.astype(np.float64), 100, dtype=np.float64)
    err = np.max(np.abs(got - ref64)) / np.max(np.abs(ref64))
    print(f"heat3d 128^3 x100: Linf={np.max(np.abs(got)):.6e} rel err vs FP64 {err:.3e}")
    assert err < 1e-5


def test_handle_graph_replay(pa, orc, gpu):
    nx, ny, nz = 70, 50, 40
    g = pa.gen_heat3d(nx, ny, nz, seed=14)
    s = pa.Stencil(nx, ny, nz)
    s.upload(g)
    s.run(7)
    s.run(7)  # replays the captured graph from the other buffer
    s.run(6)
    got = s.download()
    s.close()
    assert np.array_equal(got, orc.heat3d(g, 20))


def test_graph_timed_run_matches_run(pa, orc, gpu):
    """The timed replay advances the grid like run() (7 + 7 + 6 sweeps, so
    graphs start from both buffers) and reports a positive device time."""
    nx, ny, nz = 70, 50, 40
    g = pa.gen_heat3d(nx, ny, nz, seed=15)
    s = pa.Stencil(nx, ny, nz)
    s.upload(g)
    ms = [s.run_graph_timed(7), s.run_graph_timed(7), s.run_graph_timed(6)]
    got = s.download()
    s.close()
    assert all(t > 0 for t in ms)
    assert np.array_equal(got, orc.heat3d(g, 20))


def test_eigenmode_full_size_384(pa, gpu):
    """384^3 (over the 256 MB last-level cache): closed-form decay of a sine mode."""
    n, steps, alpha = 384, 10, 0.1
    k = np.sin(np.pi * np.arange(n + 2) / (n + 1))
    k[0] = k[-1] = 0.0
    g0 = (k[:, None, None] * k[None, :, None]) * k[None, None, :]
    g = pa.DeviceArray.from_numpy(g0.astype(np.float32))
    b = g.clone()
    out = pa.heat3d_run_dev(g, b, n, n, n, steps, alpha)
    pa.sync()
    lam = 1 + alpha * 3 * (2 * np.cos(np.pi / (n + 1)) - 2)
    err = np.max(np.abs(out.numpy() - g0 * lam ** steps))
    assert err < 1e-5


STRIPS = [(64, 16), (64, 32), (128, 16), (64, 48), (64, 64)]  # the strip forms' windows


def strip_run(pa, g, shape, sweeps, zc):
    import ctypes
    f = pa.lib().pat_internal_heat_strip
    f.restype = ctypes.c_int
    f.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int64, ctypes.c_int64, ctypes.c_int64, ctypes.c_float,
                  ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_void_p]
    nz, ny, nx = (n - 2 for n in g.shape)
    a = pa.DeviceArray.from_numpy(g)
    b = pa.DeviceArray.from_numpy(np.zeros_like(g))
    assert f(a.ptr, b.ptr, nx, ny, nz, 0.1, shape, sweeps, zc, None) == 0, pa.lib().pat_last_error()
    pa.sync()
    return b.numpy()


@pytest.mark.parametrize("sweeps", [1, 2, 3, 4, 6])
@pytest.mark.parametrize("shape", range(5))
def test_strip_windows_vs_oracle(pa, orc, gpu, shape, sweeps):
    """Every strip form at the edges of its window: narrower than it, as wide,
    one cell wider (two windows that overlap almost whole), two full windows
    and one cell more; one plane, fewer planes than sweeps, chunks with a
    remainder.  The first case's values include infinities and NaN next to the
    grid's faces, which must stay where the single sweep has them."""
    wx, wy = STRIPS[shape]
    two = [2 * w - 2 * sweeps for w in (wx, wy)]
    cases = [(wx - 1, wy - 3, 5, 2), (wx, wy, 7, 3), (wx + 1, wy + 1, 4, 4), (two[0], two[1], 9, 4),
             (two[0] + 1, two[1] + 1, 2, 1), (3, 2, 1, 1), (wx, 1, 12, 12), (1, wy + 5, 3, 2)]
    for i, (nx, ny, nz, zc) in enumerate(cases):
        g = pa.gen_heat3d(nx, ny, nz, seed=nx + ny)
        if i == 0:
            g[1, 1, 1], g[-2, -2, -2], g[2, -2, 3] = np.inf, np.nan, -np.inf
        got = strip_run(pa, g, shape, sweeps, zc)
        assert np.array_equal(got, orc.heat3d(g, sweeps), equal_nan=True), (nx, ny, nz, zc)


@pytest.mark.parametrize("sweeps", [1, 4, 6])
@pytest.mark.parametrize("shape", range(5))
def test_strip_windows_where_values_are_not_finite(pa, orc, gpu, shape, sweeps):
    """Grids of two windows and a cell (whose cells need no test against the
    grid's end): infinities and NaN at the faces and where the windows meet
    stay where the single sweep has them."""
    wx, wy = STRIPS[shape]
    nx, ny, nz = 2 * wx - 2 * sweeps + 1, 2 * wy - 2 * sweeps + 1, 9
    g = pa.gen_heat3d(nx, ny, nz, seed=4)
    for z, y, x, v in ((1, 1, 1, np.inf), (nz, ny, nx, np.nan), (1, ny, 3, -np.inf), (5, wy - sweeps, wx - sweeps, np.inf),
                       (7, wy - sweeps + 1, wx - sweeps + 1, np.nan), (4, 1, nx, -np.inf)):
        g[z, y, x] = v
    got = strip_run(pa, g, shape, sweeps, 4)
    assert np.array_equal(got, orc.heat3d(g, sweeps), equal_nan=True)


@pytest.mark.parametrize("shape", [(20, 18, 22), (64, 64, 64), (70, 40, 33)])
@pytest.mark.parametrize("variant", ["PAT_STENCIL_AUTO", "PAT_STENCIL_TEMPORAL2"])
def test_halo_values_are_kept(pa, orc, gpu, shape, variant):
    """A field whose halo is not zero (fixed boundary values): every step count
    equals the single sweeps, also after a field with a zero halo on the same
    handle, and a halo written through the device pointer holds for one step."""
    nx, ny, nz = shape
    rng = np.random.default_rng(3)
    zero = pa.gen_heat3d(nx, ny, nz, seed=5)
    fixed = rng.random((nz + 2, ny + 2, nx + 2), dtype=np.float32)
    s = pa.Stencil(nx, ny, nz)
    s.set_variant(getattr(pa, variant))
    for g in (zero, fixed, zero):
        s.upload(g)
        done = 0
        for steps in (1, 2, 7):
            s.run(steps)
            done += steps
            assert np.array_equal(s.download(), orc.heat3d(g, done)), steps
    s.upload(fixed)
    tot, kms = s.run_timed(3)
    assert np.array_equal(s.download(), orc.heat3d(fixed, 3))
    s.upload(zero)
    p = pa.c_vp()
    pa.call("pat_stencil_device_ptr", s.h, pa.ctypes.byref(p))
    pa.call("pat_memcpy_h2d", p, fixed.ctypes.data, fixed.nbytes, None)
    pa.sync()
    s.run(1)
    inside = (slice(1, -1),) * 3
    assert np.array_equal(s.download()[inside], orc.heat3d(fixed, 1)[inside])
    s.close()


def test_tuned_tile_of_the_next_grid(pa, gpu):
    """Grids that share a size class with one tuned before take a tile that
    fits them: none is slower than the two-sweep window of 64 x 16 cells (the
    tile they had before the strips), by the best of several runs in turn."""
    steps = 60

    def handle(n, variant=None):
        s = pa.Stencil(*n)
        if variant:
            s.set_variant(*variant)
        s.upload(pa.gen_heat3d(*n, seed=2))
        s.run(steps)
        return s

    handle((128, 128, 128)).close()  # tunes the class
    for n in ((129, 129, 129), (160, 160, 160), (176, 176, 176), (130, 170, 150), (148, 180, 133)):
        a, b = handle(n), handle(n, (pa.PAT_STENCIL_TEMPORAL2, 64, 16, 4))
        ta, tb = (min(s.run_graph_timed(steps) for _ in range(8)) for s in (a, b))
        tile = a.tile()
        a.close()
        b.close()
        assert ta <= tb, (n, tile, ta, tb)
