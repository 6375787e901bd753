"""What batches hand out, at the sizes where it stops fitting the pinned memory it goes through (needs an MI355X): a
2 MiB block takes the results and up to 3 n + 1,024 records, or the chunk positions and as many infos, or two lists of
as many draws; beyond, the device copies them. Every job is the same lone block: six quads, one record."""
import numpy as np
import pytest

import cases
from hypercraft_amd import hcm, workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 12154, 12180, 15118, 15119, 17100, 17200])
def test_records_infos_and_draws_around_the_pinned_block(ctx, n):
    blocks, light, nbr = cases.lone_block()
    store = hcm.Store(ctx, 27)
    store.upload(blocks, light)
    batch = hcm.Batch(ctx, store, np.tile(nbr, (n, 1)))
    print(f"export: {n} jobs", flush=True)
    batch.run()
    assert batch.totals() == (6 * n, n)
    res = batch.results()
    assert (res["status"] == 0).all() and (res["mesh_count"] == 1).all() and (res["quad_count"] == 6).all()
    res2, recs, verts, idx = batch.download()
    assert np.array_equal(res, res2)
    assert np.array_equal(np.sort(recs["job"]), np.arange(n)) and np.array_equal(recs["job"][res["first_mesh"]], np.arange(n))
    assert np.array_equal(np.sort(recs["first_quad"]), 6 * np.arange(n)) and (recs["aabb"] == [80, 112, 96, 96, 128, 112]).all()
    first = verts[:24]
    assert np.array_equal(verts.reshape(n, 24, 2), np.broadcast_to(first, (n, 24, 2))) and idx.size == 36 * n
    infos = batch.mesh_infos(np.zeros((n, 3), np.int32))
    assert infos.shape[0] == n and (infos["index_count"] == 36).all()
    assert np.array_equal(np.sort(infos["first_index"]), 36 * np.arange(n)) and (infos["aabb"] == [5, 7, 6, 6, 8, 7]).all()
    eye = np.array([5.5, 7.5, -20.0], np.float32)
    for target, kept in (((5.5, 7.5, 6.5), n), ((5.5, 7.5, -60.0), 0)):
        for _ in range(2):  # the counts start from zero again
            opaque, clear = batch.cull(eye, workloads.look_at_projection(eye, target))
            assert len(opaque) == kept and len(clear) == 0
            assert np.array_equal(np.sort(opaque["first_instance"]), np.arange(kept))
    batch.close()
    store.close()


@pytest.mark.parametrize("width,height", [(1, 2), (3, 1), (127, 129), (256, 128), (257, 129), (255, 257), (640, 361), (1, 16384), (513, 1025)])
def test_depth_levels_around_the_one_workgroup_tail(ctx, width, height):
    """Levels of up to 16,384 texels are made by one workgroup, larger ones by a launch each."""
    import draw_oracle

    depth = np.random.default_rng(width).random((height, width), dtype=np.float32)
    ctx.set_depth(depth)
    want = draw_oracle.depth_pyramid(depth)
    for k, level in enumerate(want):
        assert np.array_equal(ctx.depth_level(k), level), f"level {k} of {width} x {height}"
