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
