"""Handles that differentiated passes take over from one another: the same
images, bit for bit, and gradients (1e-5 of their largest: the adjoint's sums are
in no fixed order) as passes on fresh handles."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def A():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from illcrawl_amd import autograd
    yield autograd
    autograd.release_handles()


def inputs(n, nx, seed):
    rng = np.random.default_rng(seed)
    pos = torch.tensor(rng.normal(0, 10, (n, 3)), dtype=torch.float32, device="cuda")
    w = torch.tensor(rng.uniform(0.5, 1.5, n), dtype=torch.float32, device="cuda")
    h = torch.tensor(rng.uniform(0.5, 4.0, n), dtype=torch.float32, device="cuda")
    cam = dict(position=(0.0, 0.0, -40.0), look_at=(0.0, 0.0, 1.0), up=(0.0, 1.0, 0.0), width=30.0,
               nx=nx, ny=nx, depth=80.0)
    g = torch.tensor(rng.normal(0, 1, (nx, nx)), dtype=torch.float32, device="cuda")
    return [t.requires_grad_() for t in (pos, w, h)], cam, g


def run(A, case, kernel="quartic"):
    x, cam, g = case
    img = A.projected_image(*x, cam, kernel=kernel)
    return img, torch.autograd.grad(img, x, g)


def same(a, b):
    assert torch.equal(a[0], b[0])
    for x, y in zip(a[1], b[1]):
        assert (x - y).abs().max() <= 1e-5 * y.abs().max()


@pytest.mark.parametrize("how", ["sizes", "alive", "streams", "threads", "retained", "failed"])
def test_taken_over_handles_give_fresh_results(A, how):
    cases = [inputs(n, nx, n) for n, nx in ((3000, 40), (700, 65), (9000, 24))]
    fresh = []
    for c in cases:
        A.release_handles()
        fresh.append(run(A, c))
    torch.cuda.synchronize()
    assert all(f[0].sum() > 0 and f[1][0].abs().max() > 0 for f in fresh)
    print(f"handles: {how}", flush=True)
    if how == "sizes":
        for k in (0, 1, 2, 1, 0, 2):
            same(run(A, cases[k]), fresh[k])
        a = run(A, cases[0], "cubic")
        same(run(A, cases[0]), fresh[0])
        same(run(A, cases[0], "cubic"), a)
    elif how == "alive":
        imgs = [A.projected_image(*x, cam) for x, cam, _ in cases]
        for k in (2, 0, 1):
            x, _, g = cases[k]
            same((imgs[k], torch.autograd.grad(imgs[k], x, g)), fresh[k])
    elif how == "streams":
        streams = [torch.cuda.Stream() for _ in range(3)]
        out = []
        for i in range(9):
            with torch.cuda.stream(streams[i % 3]):
                out.append(run(A, cases[i % 2]))
        torch.cuda.synchronize()
        for i, o in enumerate(out):
            same(o, fresh[i % 2])
    elif how == "threads":
        out = {}

        def work(i):
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(4):
                    out[i] = run(A, cases[i])
                torch.cuda.current_stream().synchronize()

        ts = [threading.Thread(target=work, args=(i,)) for i in range(3)]
        [t.start() for t in ts]
        [t.join() for t in ts]
        for i in range(3):
            same(out[i], fresh[i])
    elif how == "retained":
        x, cam, g = cases[0]
        img = A.projected_image(*x, cam)
        first = torch.autograd.grad(img, x, g, retain_graph=True)
        run(A, cases[1])
        same((img, torch.autograd.grad(img, x, g)), fresh[0])
        same((img, first), fresh[0])
    else:
        x, cam, g = cases[0]
        with pytest.raises(Exception):
            A.projected_image(x[0], x[1], x[2] * float("nan"), cam)
        same(run(A, cases[0]), fresh[0])
    assert all(len(q) <= A._POOL_SIZE for q in A._pool.values())


def test_large_passes_keep_nothing(A):
    A.release_handles()
    run(A, inputs(A._POOL_ROWS + 1, 16, 5))
    assert not any(A._pool.values())


def test_kept_handles_are_bounded_over_all_configurations(A):
    """Passes of many configurations leave no more handles than passes of one,
    the newest, and none of their points."""
    A.release_handles()
    case = inputs(500, 20, 1)
    x, cam, g = case
    fresh = run(A, case)
    for target in (8, 20, 50, 120, 300, 700, 900, 2000):
        for kernel in ("quartic", "cubic"):
            img = A.projected_image(*x, cam, kernel=kernel, target_particles_per_cell=target)
            torch.autograd.grad(img, x, g)
            del img
    kept = [e for q in A._pool.values() for e in q]
    print(f"handles kept: {len(kept)}", flush=True)
    assert 0 < len(kept) <= A._POOL_SIZE
    assert not any(p._keep for e in kept for p in e if hasattr(p, "_keep"))
    same(run(A, case), fresh)
