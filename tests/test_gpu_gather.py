"""The gather's branches at the sizes where they can go wrong, against the
oracle: the same bars as the parity tests (1e-5 relative L-inf over pixels
above 1e-6 of the maximum, 1e-6 on the image sum)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

LINF_TOL = 1e-5
SUM_TOL = 1e-6


@pytest.fixture(scope="module")
def B():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from illcrawl_amd import backend
    return backend


def rel_errors(a, ref):
    a, ref = np.asarray(a, np.float64), np.asarray(ref, np.float64)
    m = ref > 1e-6 * ref.max()
    return (float(np.max(np.abs(a[m] - ref[m]) / ref[m])),
            float(abs(a.sum() - ref.sum()) / abs(ref.sum())))


def lattice(nx, ny, x0, y0, step):
    pts = np.zeros((nx * ny, 4), np.float32)
    pts[:, 0] = np.tile(x0 + step * np.arange(nx), ny)
    pts[:, 1] = np.repeat(y0 + step * np.arange(ny), nx)
    return pts


def render(B, p4, h, pts, nx, **kw):
    b = B.ProjectiveSmoothingGrid(**kw)
    b.init_backend(p4.shape[0])
    b.setup_projected_particles(p4, h)
    b.setup_evaluation_points(pts, layout_nx=nx)
    b.run()
    return b.retrieve_results_f64().cpu().numpy()


@pytest.mark.parametrize("spread,target,step", [
    (0.0, 50, 1.0),     # every h the cell's largest and the grid's: nothing below the radius
    (0.05, 50, 1.0),    # h on both sides of the smallest radius of a tile
    (2.0, 2, 0.5),      # cells far smaller than h, sparse: row streaming
    (2.0, 400, 4.0),    # tiles of several cells with different radii
])
def test_search_box_is_skipped_only_where_it_drops_nothing(B, orc, spread, target, step):
    rng = np.random.default_rng(int(100 * spread) + target)
    n = 6000
    p4 = np.zeros((n, 4), np.float32)
    p4[: n // 2, :2] = rng.uniform(-100, 100, (n // 2, 2))
    p4[n // 2:, :2] = rng.normal(0, 8.0, (n - n // 2, 2))
    p4[:, 3] = rng.uniform(0.5, 1.5, n)
    h = (6.0 * np.exp(spread * rng.uniform(-1, 1, n))).astype(np.float32)
    pts = lattice(45, 37, -20 * step, -17 * step, step)
    print(f"search box: spread={spread} target={target} step={step}", flush=True)
    ref = orc.Grid(p4, h, target=target).gather_ref(pts, acc_mode=1)
    for tile in (None, (16, 16)):
        got = render(B, p4, h, pts, 45, target_particles_per_cell=target, tile=tile)
        linf, s = rel_errors(got, ref)
        print(f"  tile={tile} linf={linf:.2e} sum={s:.2e}", flush=True)
        assert linf < LINF_TOL and s < SUM_TOL


def batch_image(B, p4, h, view, tile, mode):
    r = B.BatchRenderer(mode=mode, kernel="quartic_ref", tile=tile)
    r.set_particles(p4[:, :3].copy(), p4[:, 3].copy(), h)
    r.set_views([view])
    r.render()
    return r.image_f64(0).cpu().numpy().reshape(-1)


@pytest.mark.parametrize("mode", ["reference", "exact"])
@pytest.mark.parametrize("nx,ny", [(1, 1), (1, 40), (33, 1), (8, 8), (17, 15), (50, 31)])
def test_tiles_with_far_and_near_particles(B, orc, mode, nx, ny):
    """Partial, one-row and one-column tiles of both sides, with supports from
    a fraction of a pixel to many tiles wide: particles whose support covers a
    tile (summed at the nodes), crosses it, or lies inside it."""
    rng = np.random.default_rng(nx * 100 + ny)
    n = 5000
    p4 = np.zeros((n, 4), np.float32)
    p4[:, :2] = rng.uniform(-150, 150, (n, 2))
    p4[:, 2] = rng.uniform(-10, 10, n)
    p4[:, 3] = rng.uniform(0.5, 1.5, n)
    h = np.exp(rng.uniform(np.log(0.3), np.log(120.0), n)).astype(np.float32)
    view = dict(position=np.array([0.0, 0.0, -20.0]), look_at=np.array([0.0, 0.0, 1.0]),
                roll=0.3, width=float(nx), nx=nx, ny=ny, depth=40.0)
    cam = orc.Camera(view["position"], view["look_at"], view["roll"], view["width"], nx, ny)
    pp = cam.project_particles(p4, view["depth"])
    pts = cam.pixel_points()
    ref = orc.Grid(pp, h).gather_ref(pts, acc_mode=1) if mode == "reference" else \
        orc.gather_exact(pp, h, pts, kind=0)
    for tile in ((16, 16, 64), (8, 8, 64), None):
        got = batch_image(B, p4, h, view, tile, mode)
        linf, s = rel_errors(got, ref)
        print(f"tiles {nx}x{ny} {mode} tile={tile}: linf={linf:.2e} sum={s:.2e}", flush=True)
        assert linf < LINF_TOL and s < SUM_TOL


def test_tile_side_follows_the_number_of_points(B, orc):
    """Both sides of the rule (16x16 tiles from 3 << 18 points): the images of
    a lattice one row shorter and one row longer agree with the oracle on
    sampled points."""
    rng = np.random.default_rng(3)
    n = 20000
    p4 = np.zeros((n, 4), np.float32)
    p4[:, :2] = rng.uniform(-300, 300, (n, 2))
    p4[:, 3] = rng.uniform(0.5, 1.5, n)
    h = rng.uniform(2.0, 90.0, n).astype(np.float32)
    nx = 1024
    for ny in (767, 768):
        pts = lattice(nx, ny, -200.0, -150.0, 0.39)
        got = render(B, p4, h, pts, nx)
        idx = rng.choice(nx * ny, 1200, replace=False)
        ref = orc.Grid(p4, h).gather_ref(pts[idx], acc_mode=1)
        linf, s = rel_errors(got[idx], ref)
        print(f"rule {nx}x{ny}: linf={linf:.2e} sum={s:.2e}", flush=True)
        assert linf < LINF_TOL and s < SUM_TOL


@pytest.mark.parametrize("kernel", ["quartic", "cubic"])
def test_coincident_points(B, orc, kernel):
    """A tile of no extent: every point the same."""
    rng = np.random.default_rng(5)
    n = 4000
    p4 = np.zeros((n, 4), np.float32)
    p4[:, :2] = rng.uniform(-40, 40, (n, 2))
    p4[:, 3] = 1.0
    h = rng.uniform(1.0, 60.0, n).astype(np.float32)
    pts = np.zeros((300, 4), np.float32)
    pts[:, 0], pts[:, 1] = 1.25, -2.5
    got = render(B, p4, h, pts, 20, mode="exact", kernel=kernel)
    ref = orc.gather_exact(p4, h, pts[:1], kind={"quartic": 1, "cubic": 2}[kernel])
    assert np.all(got == got[0])
    # the cubic kernel is tabulated: the parity tests' 2e-5
    assert abs(got[0] - ref[0]) / ref[0] < (2e-5 if kernel == "cubic" else LINF_TOL)


@pytest.mark.parametrize("nx,ny", [(1024, 771), (97, 43), (8, 1)])
def test_adjoint_tiles(B, orc, nx, ny):
    """Both tile sides of the adjoint (16x16 from 3 << 18 points), partial
    tiles, blocks without a gradient, and supports from a fraction of a pixel
    to most of the image (the nodes of 16x16 tiles).  1e-4 of each component's
    largest magnitude, as the adjoint tests."""
    rng = np.random.default_rng(nx)
    n = 300
    p4 = np.zeros((n, 4), np.float32)
    p4[:, 0], p4[:, 1] = rng.uniform(-0.6 * nx, 0.6 * nx, n), rng.uniform(-0.6 * ny, 0.6 * ny, n)
    p4[:, 3] = rng.uniform(0.5, 1.5, n)
    h = np.exp(rng.uniform(np.log(0.4), np.log(0.4 * max(nx, ny) + 2.0), n)).astype(np.float32)
    pts = lattice(nx, ny, -0.5 * nx, -0.5 * ny, 1.0)
    G = rng.normal(size=nx * ny).astype(np.float32)
    G.reshape(ny, nx)[: ny // 3, : nx // 3] = 0.0
    b = B.ProjectiveSmoothingGrid(mode="exact", kernel="quartic", target_particles_per_cell=40)
    b.init_backend(n)
    b.setup_projected_particles(p4, h)
    b.setup_evaluation_points(pts, layout_nx=nx)
    got = [t.cpu().numpy() for t in b.backward(torch.from_numpy(G).cuda(), 1.0)]
    ref = orc.backward_exact(p4, h, pts, G, kind=1)
    for name, a, r in zip(("w", "h", "x", "y"), got, ref):
        e = float(np.max(np.abs(a - r)) / np.max(np.abs(r)))
        print(f"adjoint {nx}x{ny} dL/d{name}: {e:.2e}", flush=True)
        assert e < 1e-4


SORT_SIZES = [1, 2, 1024, 1025, 131072, 131073, 1 << 20, (1 << 20) + 1]


def sort_input(n):
    rng = np.random.default_rng(n)
    p4 = np.zeros((n, 4), np.float32)
    p4[:, :2] = rng.normal(0, 30.0, (n, 2))
    p4[:, 3] = 1.0
    h = np.exp(rng.uniform(-8, 8, n)).astype(np.float32)
    h[rng.random(n) < 0.5] = 1.5
    return p4, h


@pytest.mark.parametrize("target", [40, 3])
def test_cells_hold_their_particles_by_descending_h(orc, tmp_path, target):
    """The order that the gather searches: by cell, in a cell by descending h (the
    top 16 bits of its pattern), ties in input order, at the sort's limits."""
    import os
    import subprocess
    from illcrawl_amd import build
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    if not os.path.exists(build.SORT):
        pytest.fail("sort_order is not built (run __graft_entry__.build())")
    for n in SORT_SIZES:
        p4, h = sort_input(n)
        p4.tofile(tmp_path / f"p4_{n}.f32")
        h.tofile(tmp_path / f"h_{n}.f32")
    r = subprocess.run([build.SORT, str(tmp_path), str(target)] + [str(n) for n in SORT_SIZES],
                       capture_output=True, text=True, timeout=100)
    print(r.stdout + r.stderr, flush=True)
    assert r.returncode == 0
    for n in SORT_SIZES:
        p4, h = sort_input(n)
        cell = orc.Grid(p4, h, target=target).keys(p4)
        order = np.lexsort((np.arange(n), -(h.view(np.uint32) >> 16).astype(np.int64), cell))
        assert np.array_equal(np.fromfile(tmp_path / f"perm_{n}.u32", np.uint32), order)
        assert np.array_equal(np.fromfile(tmp_path / f"key_{n}.u32", np.uint32), cell[order])


@pytest.mark.parametrize("n", SORT_SIZES)
def test_grid_sort_at_the_tile_and_path_limits(B, orc, n):
    """The sort's tiles of 1024 and 4096 rows and its three paths (digit counts
    by the passes, by a count launch, scanned): cells, ranges, max h and the
    reference's order (sorted again from the input's) equal the oracle's bit for
    bit."""
    p4, h = sort_input(n)
    b = B.ProjectiveSmoothingGrid(target_particles_per_cell=40)
    b.init_backend(n)
    b.setup_projected_particles(p4, h)
    g = orc.Grid(p4, h, target=40)
    cells, maxh, perm = b.export_grid()
    assert np.array_equal(cells.cpu().numpy(), g.cells)
    assert np.array_equal(maxh.cpu().numpy(), g.maxh_cell)
    assert np.array_equal(perm.cpu().numpy().astype(np.uint32), g.perm)
    print(f"sort n={n}: {g.ncells} cells", flush=True)


def odd_lattice(value, axes):
    """1024 x 771 points (16x16 tiles), three of them with `value` as `axes`."""
    nx, ny = 1024, 771
    pts = lattice(nx, ny, -0.05 * nx, -0.05 * ny, 0.1)
    odd = np.array([0, 385 * nx + 512, nx * ny - 1])
    pts[np.ix_(odd, axes)] = value
    near = [b * nx + a for c in odd for b in range(max(c // nx - 16, 0), min(c // nx + 17, ny), 3)
            for a in range(max(c % nx - 16, 0), min(c % nx + 17, nx), 3)]
    return pts, nx, odd, np.setdiff1d(np.unique(near), odd)


def wide_particles(n, seed):
    rng = np.random.default_rng(seed)
    p4 = np.zeros((n, 4), np.float32)
    p4[:, 0], p4[:, 1] = rng.uniform(-70, 70, n), rng.uniform(-60, 60, n)
    p4[:, 3] = rng.uniform(0.5, 1.5, n)
    return p4, np.exp(rng.uniform(np.log(0.5), np.log(60.0), n)).astype(np.float32)


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("axes", [[0], [0, 1]])
@pytest.mark.parametrize("mode,kernel", [("reference", "quartic_ref"), ("exact", "quartic"),
                                         ("exact", "cubic")])
def test_points_out_of_reach(B, orc, mode, kernel, axes, value):
    """A point with an infinite or NaN coordinate is worth 0, as the oracle has
    it, and its tile's other points lose nothing."""
    p4, h = wide_particles(2000, 7)
    pts, nx, odd, some = odd_lattice(value, axes)
    print(f"points out of reach: {mode} {kernel} {axes} {value}", flush=True)
    got = render(B, p4, h, pts, nx, mode=mode, kernel=kernel)
    ref = orc.Grid(p4, h).gather_ref(pts[some], acc_mode=1) if mode == "reference" else \
        orc.gather_exact(p4, h, pts[some], kind={"quartic": 1, "cubic": 2}[kernel])
    linf, s = rel_errors(got[some], ref)
    # the cubic kernel is tabulated: the parity tests' 2e-5
    assert linf < (2e-5 if kernel == "cubic" else LINF_TOL) and s < SUM_TOL
    assert np.all(got[odd] == 0.0)


def adjoint(B, p4, h, pts, nx, G):
    b = B.ProjectiveSmoothingGrid(mode="exact", kernel="quartic", target_particles_per_cell=40)
    b.init_backend(p4.shape[0])
    b.setup_projected_particles(p4, h)
    b.setup_evaluation_points(pts, layout_nx=nx)
    return [t.cpu().numpy() for t in b.backward(torch.from_numpy(G).cuda(), 1.0)]


@pytest.mark.parametrize("value", [np.inf, np.nan])
@pytest.mark.parametrize("axes", [[0], [0, 1]])
def test_adjoint_of_points_out_of_reach(B, orc, axes, value):
    """They add nothing to any particle's gradient."""
    p4, h = wide_particles(300, 8)
    pts, nx, odd, _ = odd_lattice(value, axes)
    G = np.random.default_rng(8).normal(size=pts.shape[0]).astype(np.float32)
    got = adjoint(B, p4, h, pts, nx, G)
    ref = orc.backward_exact(p4, h, pts, G, kind=1)
    for name, a, r in zip(("w", "h", "x", "y"), got, ref):
        e = float(np.max(np.abs(a - r)) / np.max(np.abs(r)))
        print(f"adjoint with points at {value} {axes} dL/d{name}: {e:.2e}", flush=True)
        assert e < 1e-4


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
def test_adjoint_of_a_point_without_a_finite_gradient(B, orc, value):
    """dL/dw of the particles that cover the point is that value (at the nodes
    of a tile it would meet weights of either sign); those a tile's diagonal
    beyond their support have the other points' gradient."""
    p4, h = wide_particles(300, 9)
    pts, nx, odd, _ = odd_lattice(0.0, [2])
    G = np.random.default_rng(9).normal(size=pts.shape[0]).astype(np.float32)
    c = odd[1]
    G[c] = 0.0
    ref = orc.backward_exact(p4, h, pts, G, kind=1)
    G[c] = value
    got = adjoint(B, p4, h, pts, nx, G)
    r = np.hypot(p4[:, 0] - pts[c, 0], p4[:, 1] - pts[c, 1])
    covers, clear = r < 0.999 * h, r > h + 0.1 * 16 * 1.5
    assert covers.sum() > 20 and clear.sum() > 20
    assert np.array_equal(got[0][covers], np.full(covers.sum(), value, np.float32), equal_nan=True)
    for name, a, x in zip(("w", "h", "x", "y"), got, ref):
        e = float(np.max(np.abs(a[clear] - x[clear])) / np.max(np.abs(x)))
        print(f"adjoint with a gradient of {value} dL/d{name}: {e:.2e}", flush=True)
        assert e < 1e-4


def pair_bound(pp, h, pts, kernel):
    """Rounding of the FP32 pairs (c s)^2.5, s = 1 - r^2/h^2, per point, with
    u = 2^-24.  The argument c s is a sum of terms of at most 1.5 c, each off by
    some 6 u: 24 u c in all, the value by 2.5 coef s^1.5 24 u; the power, the
    coefficient and a partial sum of 32 pairs by 50 u of it."""
    u = 2.0 ** -24
    norm = 3.5 / np.pi if kernel == "quartic" else 2.0 * 1.04445 * 1.066667
    h2 = h.astype(np.float64) ** 2
    coef = norm * np.abs(pp[:, 3].astype(np.float64)) / h2
    r2 = sum((pts[:, None, a].astype(np.float64) - pp[None, :, a].astype(np.float64)) ** 2
             for a in range(2))
    s = np.maximum(1.0 - r2 / h2, 0.0)
    return ((60 * u * s ** 1.5 + 50 * u * s ** 2.5 + (24 * u) ** 2.5) * coef).sum(1)


@pytest.mark.parametrize("mode,kernel", [("reference", "quartic_ref"), ("exact", "quartic"),
                                         ("exact", "cubic")])
@pytest.mark.parametrize("n", [1, 3, 5, 63, 66, 255, 256, 257])
def test_few_candidates_for_a_tile(B, orc, n, mode, kernel):
    """A 16x16 tile with fewer candidates than its four waves take at a time."""
    rng = np.random.default_rng(n)
    p4 = np.zeros((n, 4), np.float32)
    p4[:, :2] = rng.uniform(-7, 7, (n, 2))
    p4[:, 3] = rng.uniform(0.5, 1.5, n)
    h = np.exp(rng.uniform(np.log(0.8), np.log(30.0), n)).astype(np.float32)
    view = dict(position=np.array([0.0, 0.0, -20.0]), look_at=np.array([0.0, 0.0, 1.0]),
                roll=0.0, width=16.0, nx=16, ny=16, depth=40.0)
    cam = orc.Camera(view["position"], view["look_at"], view["roll"], view["width"], 16, 16)
    pp, pts = cam.project_particles(p4, view["depth"]), cam.pixel_points()
    ref = orc.Grid(pp, h).gather_ref(pts, acc_mode=1) if mode == "reference" else \
        orc.gather_exact(pp, h, pts, kind={"quartic": 1, "cubic": 2}[kernel])
    r = B.BatchRenderer(mode=mode, kernel=kernel, tile=(16, 16, 64))
    r.set_particles(p4[:, :3].copy(), p4[:, 3].copy(), h)
    r.set_views([view])
    r.render()
    got = r.image_f64(0).cpu().numpy().reshape(-1)
    print(f"few candidates n={n} {mode} {kernel}", flush=True)
    if kernel == "cubic":  # tabulated: the parity tests' 2e-5, of the largest value
        assert np.max(np.abs(got - ref)) < 2e-5 * ref.max()
    else:
        assert np.all(np.abs(got - ref) <= pair_bound(pp, h, pts, kernel))


@pytest.mark.parametrize("mode,kernel", [("reference", "quartic_ref"), ("exact", "quartic")])
@pytest.mark.parametrize("nx,ny,n,hmax", [
    (999, 603, 3500, 40.0),   # the last column and row of tiles with empty quarters
    (1041, 520, 2500, 3.0),   # supports within a tile, the last row half empty
])
def test_slab_stack_by_quarter_tiles(B, orc, nx, ny, n, hmax, mode, kernel):
    """Slab stacks of many tiles for their rows, summed by the quarters of
    16x16 tiles, against the oracle on sampled points (the last tiles' among
    them); a dense clump fills the lists many times over."""
    rng = np.random.default_rng(nx)
    p4 = np.zeros((n, 4), np.float32)
    p4[:, 0], p4[:, 1] = rng.uniform(-0.55 * nx, 0.55 * nx, n), rng.uniform(-0.55 * ny, 0.55 * ny, n)
    p4[: n // 3, :2] = rng.normal(0, 6.0, (n // 3, 2)) + (0.5 * nx - 8.0, 0.5 * ny - 9.0)
    p4[:, 2] = rng.uniform(0, 40, n)
    p4[:, 3] = rng.uniform(0.5, 1.5, n)
    h = np.exp(rng.uniform(np.log(0.4), np.log(hmax), n)).astype(np.float32)
    views = [dict(position=np.array([0.0, 0.0, 10.0 * k]), look_at=np.array([0.0, 0.0, 1.0]),
                  roll=0.0, width=float(nx), nx=nx, ny=ny, depth=10.0) for k in range(4)]
    r = B.BatchRenderer(mode=mode, kernel=kernel, tile=(16, 16, 64))
    r.set_particles(p4[:, :3].copy(), p4[:, 3].copy(), h)
    r.set_views(views)
    r.render()
    rows = sum(r.view_info(k)["num_particles"] for k in range(4))
    tiles = 4 * -(-nx // 16) * -(-ny // 16)
    assert tiles ** 2 >= 25000 * rows  # the rule's line
    x, y = rng.integers(0, nx, 1500), rng.integers(0, ny, 1500)
    x[:500], y[:500] = rng.integers(nx - 40, nx, 500), rng.integers(ny - 40, ny, 500)
    idx = y * nx + x
    for k, v in enumerate(views):
        cam = orc.Camera(v["position"], v["look_at"], v["roll"], v["width"], nx, ny)
        pp, pts = cam.project_particles(p4, v["depth"]), cam.pixel_points()[idx]
        ref = orc.Grid(pp, h).gather_ref(pts, acc_mode=1) if mode == "reference" else \
            orc.gather_exact(pp, h, pts, kind=1)
        got = r.image_f64(k).cpu().numpy().reshape(-1)[idx]
        off = np.abs(got - ref) / np.maximum(pair_bound(pp, h, pts, kernel), 1e-300)
        print(f"quarters {nx}x{ny} {mode} slab {k}: {off.max():.2f} of the bound", flush=True)
        assert ref.max() > 0 and off.max() <= 1.0
    eager = [r.image_f64(k) for k in range(4)]
    for _ in range(3):  # the graph's replays, with eager work between them
        r.render(graph=True)
        assert all(torch.equal(r.image_f64(k), eager[k]) for k in range(4))


# The nodes' interpolation errs by at most 3.3e-7 of a far particle's own value
# at a point of the tile, whatever the tile's shape (in FP64, over all directions
# and distances that the rule takes).  A sum over many particles averages their
# FP32 rounding (6e-8 left: three deviations of 5e-6 over 65536), but not the kernel
# constant's (2^-24 twice).
@pytest.mark.parametrize("nx,ny", [(16, 1), (1, 16), (16, 4), (3, 16), (16, 16)])
@pytest.mark.parametrize("of", ["diagonal", "side"])
def test_far_particles_of_strip_tiles(B, orc, nx, ny, of):
    """Particles 0.9 h from the tile's centre, along its longer side, whose
    supports are just wide enough by its half-diagonal, or by sqrt 2 times its
    larger half-side."""
    rng = np.random.default_rng(nx * 20 + ny)
    n, hx, hy = 65536, 0.5 * (nx - 1), 0.5 * (ny - 1)
    a = np.hypot(hx, hy) if of == "diagonal" else np.sqrt(2.0) * max(hx, hy)
    p4 = np.zeros((n, 4), np.float32)
    h = (a / (0.975 * (0.4 + 0.9 * 0.22) * 0.1) * (1.0 + 0.004 * rng.random(n))).astype(np.float32)
    p4[:, :2] = rng.uniform(-5e-4, 5e-4, (n, 2)) * h[:, None]
    p4[:, 0 if nx >= ny else 1] += 0.9 * h
    p4[:, 3] = rng.uniform(0.5, 1.5, n)
    view = dict(position=np.array([0.0, 0.0, -20.0]), look_at=np.array([0.0, 0.0, 1.0]),
                roll=0.0, width=float(nx), nx=nx, ny=ny, depth=40.0)
    cam = orc.Camera(view["position"], view["look_at"], view["roll"], view["width"], nx, ny)
    pts = cam.pixel_points()
    p4[:, :2] += 0.5 * (pts[:, :2].min(0) + pts[:, :2].max(0))  # the points are the pixels' corners
    r = B.BatchRenderer(mode="exact", kernel="quartic", tile=(16, 16, 64))
    r.set_particles(p4[:, :3].copy(), p4[:, 3].copy(), h)
    r.set_views([view])
    r.render()
    ref = orc.gather_exact(cam.project_particles(p4, view["depth"]), h, pts, kind=1)
    off = np.max(np.abs(r.image_f64(0).cpu().numpy().reshape(-1) / ref - 1.0))
    print(f"far strip {nx}x{ny} by the {of}: {off:.2e}", flush=True)
    assert off < 3.3e-7 + 2 * 2.0 ** -24 + 6e-8
