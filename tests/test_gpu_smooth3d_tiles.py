"""The volumetric gather at the edges of its tiles, against the FP64 sums.

The bound is the rounding of the FP32 pair w/h^3 s^2, s = 1 - r^2/h^2, with
u = 2^-24: r^2 is off by 5 u (a subtraction counts twice, three roundings), 1/h^2
by 2 u and s, one rounding more, by 7 u in all; the coefficient by 6 u, the
square and the product by 2 u, a partial sum of 32 pairs by 32 u.  So a point
may be off by u sum(coef (14 s + 40 s^2)), and by (7 u)^2 coef for a pair at
the edge of its support."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

U = 2.0 ** -24
SUM_TOL = 1e-6


def bound(p4, h, pts):
    coef = 1.05 * p4[:, 3].astype(np.float64) / h.astype(np.float64) ** 3
    xyz, h2 = p4[:, :3].astype(np.float64), h.astype(np.float64) ** 2
    out = np.empty(pts.shape[0])
    for i in range(0, pts.shape[0], 2048):
        q = pts[i:i + 2048, :3].astype(np.float64)
        r2 = sum((q[:, a, None] - xyz[None, :, a]) ** 2 for a in range(3))
        s = np.maximum(1.0 - r2 / h2, 0.0)
        out[i:i + 2048] = ((14 * U * s + 40 * U * s * s + (7 * U) ** 2) * coef).sum(1)
    return out


@pytest.fixture(scope="module")
def B():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from illcrawl_amd import backend
    return backend


@pytest.fixture(scope="module")
def orc():
    import oracle
    return oracle


@pytest.mark.parametrize("nx,ny,step,bend,hmax", [
    (1, 1, 1.0, 0.0, 30.0),        # one point
    (1, 300, 0.2, 0.0, 20.0),      # one column: no plane through the tile's corners
    (300, 1, 0.2, 0.0, 20.0),      # one row
    (17, 9, 1.0, 0.0, 60.0),       # a column and a row beyond a tile; cover particles
    (16, 16, 0.0, 0.0, 20.0),      # every point the same
    (40, 33, 1.0, 6.0, 12.0),      # points off their tile's plane
    (23, 48, 1.0, 1e9, 12.0),      # rows of far-apart slices in one tile
    (1024, 513, 0.1, 0.0, 12.0),   # 16 x 16 tiles, the last row of points alone
    (1000, 525, 0.1, 0.7, 12.0),   # the same, off their plane and a partial column
])
@pytest.mark.parametrize("mode,kernel", [("reference", "quartic_ref"), ("exact", "quartic")])
def test_tiles_match_the_sums(B, orc, nx, ny, step, bend, hmax, mode, kernel):
    rng = np.random.default_rng(nx * 1000 + ny)
    n = 3000
    p4 = np.concatenate([rng.uniform(0, 100, (n, 3)), rng.lognormal(0, 0.3, (n, 1))],
                        1).astype(np.float32)
    h = np.exp(rng.uniform(np.log(1.0), np.log(hmax), n)).astype(np.float32)
    u, v = np.meshgrid((np.arange(nx) - 0.5 * nx) * step, (np.arange(ny) - 0.5 * ny) * step)
    z = 30.0 * (np.arange(ny)[:, None] % 3 - 1.0) + 0 * u if bend > 1e8 else bend * np.sin(u + v)
    pts = np.zeros((nx * ny, 4), np.float32)
    pts[:, 0] = (50.0 + u).ravel()
    pts[:, 1] = (50.0 + 0.8 * v - 0.6 * z).ravel()
    pts[:, 2] = (50.0 + 0.6 * v + 0.8 * z).ravel()
    # past 20000 points, some of them (stride coprime to the tile side, both ends)
    some = np.unique(np.r_[0:pts.shape[0]:max(1, pts.shape[0] // 20000) | 1, pts.shape[0] - 1])
    print(f"tiles {nx} x {ny} step {step} bend {bend} {mode}", flush=True)
    g = B.GridSmoothing(mode=mode, kernel=kernel, target_particles_per_cell=64)
    g.init_backend(n)
    g.setup_particles(p4, [h])
    g.setup_evaluation_points(pts, layout_nx=nx)
    g.run()
    got = g.retrieve_results_f64().cpu().numpy()[some]
    if mode == "reference":
        ref = orc.Grid(p4, h, target=64).smooth3d_ref(pts[some], form=1)
    else:
        ref = orc.smooth3d_exact(p4, h, pts[some])
    assert ref.max() > 0
    off = np.abs(got - ref) / bound(p4, h, pts[some])
    print(f"  largest error {off.max():.3f} of its bound", flush=True)
    assert off.max() < 1.0
    assert abs(got.sum() - ref.sum()) < SUM_TOL * ref.sum()


@pytest.mark.parametrize("n,span,cluster", [
    (1, 0.0, False),               # one particle
    (700, 0.0, False),             # one h: one level, no level bits
    (257, 40.0, False),            # levels that the clamp at level 0 shares; a two-word key
    (20000, 6.0, True),            # most particles in one cell
    ((1 << 20) + 77, 3.0, True),   # cell maxima in ranges, the last workgroup partial
])
def test_level_index_matches_the_sums(B, orc, n, span, cluster):
    rng = np.random.default_rng(n)
    xyz = rng.uniform(0, 100, (n, 3))
    if cluster:
        xyz[: 3 * n // 4] = 50.0 + rng.normal(0, 0.4, (3 * n // 4, 3))
    w = rng.lognormal(0, 0.3, (n, 1))
    p4 = np.concatenate([xyz, w], 1).astype(np.float32)
    h = (20.0 * (n ** -0.3) * 2.0 ** (-span * rng.uniform(0, 1, n))).astype(np.float32)
    pts = np.zeros((96, 4), np.float32)
    pts[:, :3] = rng.uniform(0, 100, (96, 3))
    pts[48:, :3] = p4[rng.integers(0, n, 48), :3] + rng.normal(0, 0.05, (48, 3))
    print(f"level index n={n} span={span}", flush=True)
    g = B.GridSmoothing(mode="reference", kernel="quartic_ref", target_particles_per_cell=64)
    g.init_backend(n)
    g.setup_particles(p4, [h])
    g.setup_evaluation_points(pts)
    g.run()
    got = g.retrieve_results_f64().cpu().numpy()
    ref = orc.Grid(p4, h, target=64).smooth3d_ref(pts, form=1)
    assert ref.max() > 0
    assert np.all(np.abs(got - ref) <= bound(p4, h, pts))


def with_odd_points(nx, ny, value, axes):
    """A tilted lattice whose points `odd` have `value` as their coordinates `axes`."""
    u, v = np.meshgrid((np.arange(nx) - 0.5 * nx) * 0.2, (np.arange(ny) - 0.5 * ny) * 0.2)
    pts = np.zeros((nx * ny, 4), np.float32)
    pts[:, 0], pts[:, 1], pts[:, 2] = (50.0 + u).ravel(), (50.0 + v).ravel(), (50.0 + 0.3 * u).ravel()
    odd = np.array([0, nx * (ny // 2) + nx // 2, nx * ny - 1])
    pts[np.ix_(odd, axes)] = value
    return pts, odd


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, 1e25])
@pytest.mark.parametrize("axes", [[0], [2], [0, 1, 2]])
@pytest.mark.parametrize("nx,ny", [(40, 33), (1024, 513)])
@pytest.mark.parametrize("mode,kernel", [("reference", "quartic_ref"), ("exact", "quartic")])
def test_a_point_out_of_reach_takes_nothing_from_its_tile(B, orc, mode, kernel, nx, ny, axes,
                                                          value):
    rng = np.random.default_rng(nx)
    n = 2000
    p4 = np.concatenate([rng.uniform(30, 70, (n, 3)), rng.lognormal(0, 0.3, (n, 1))],
                        1).astype(np.float32)
    h = np.exp(rng.uniform(np.log(1.0), np.log(15.0), n)).astype(np.float32)
    pts, odd = with_odd_points(nx, ny, value, axes)
    print(f"odd points {value} {axes} {nx} x {ny} {mode}", flush=True)
    g = B.GridSmoothing(mode=mode, kernel=kernel, target_particles_per_cell=64)
    g.init_backend(n)
    g.setup_particles(p4, [h])
    g.setup_evaluation_points(pts, layout_nx=nx)
    g.run()
    got = g.retrieve_results_f64().cpu().numpy()
    # the odd points' neighbours (a tile's side away at most) and some others
    x, y = odd % nx, odd // nx
    near = [(b, a) for px, py in zip(x, y) for b in range(max(py - 16, 0), min(py + 17, ny), 3)
            for a in range(max(px - 16, 0), min(px + 17, nx), 3)]
    some = np.setdiff1d(np.unique([b * nx + a for b, a in near]), odd)
    ref = orc.Grid(p4, h, target=64).smooth3d_ref(pts[some], form=1) if mode == "reference" else \
        orc.smooth3d_exact(p4, h, pts[some])
    assert ref.max() > 0
    assert np.all(np.abs(got[some] - ref) <= bound(p4, h, pts[some]))
    assert np.all(got[odd] == 0.0)
