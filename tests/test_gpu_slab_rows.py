"""The rows that a slab stack's pass lists per 2048-particle tile, at the list's
edges: the images equal the per-view pass's bit for bit (the same rows in the same
order), which a view that is no slab brings about."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("n,slabs,thickness", [
    (6000, 6, 3300.0),   # every particle in two slabs: up to 4096 rows a tile, two rounds
    (4096, 6, 1700.0),   # about one slab each: the list's end
    (5001, 40, 260.0),   # many slabs, the last tile partial
    (2049, 6, 3.0),      # nearly all rows empty, slabs without any
])
def test_slab_rows_equal_the_per_view_pass(n, slabs, thickness):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from illcrawl_amd import backend as B, synth
    print(f"slab rows n={n} slabs={slabs} thickness={thickness}", flush=True)
    snap = synth.make_snapshot(n, 7, 10000.0, n_halos=2, rs_range=(300.0, 600.0), gas=True)
    tab = synth.gaunt_table_1d()
    views = synth.slab_views(snap.box, n_slabs=slabs, thickness=thickness, nx=48, width=8000.0,
                             quantity=1)
    for v in views:
        v["scale"] = 1.0
    other = synth.centred_view(snap.box, look_at=(0.3, 0.2, 0.9), width=6000.0, nx=48)
    other.update(quantity=1, scale=1.0)
    images = []
    for vs in (views, views + [other]):
        r = B.BatchRenderer(mode="reference", kernel="quartic_ref")
        r.set_particles(snap.pos, snap.mass, snap.hsml, snap.rho, snap.temp, snap.xe)
        r.set_gaunt_table(*tab)
        r.set_views(vs)
        r.render()
        images.append([r.image_f64(k).cpu().numpy() for k in range(slabs)])
    assert thickness < 10 or sum(i.sum() for i in images[0]) > 0
    for a, b in zip(*images):
        assert np.array_equal(a, b)
