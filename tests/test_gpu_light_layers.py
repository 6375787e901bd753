"""The light rebuild across the layers its wavefronts hold (needs an MI355X): one light source per job at and beside
every edge of six layers along y, at the ends of the 46-cell window along each axis and at the edges of a chunk, in open
air, among random blocks and in a corridor that winds through all layers; sunlight from random heights. The rebuilt
light is the oracle's, byte for byte."""
import numpy as np
import pytest

import cases
from hypercraft_amd import hcm, workloads

pytestmark = pytest.mark.gpu
EDGES = (-15, -14, -10, -9, -4, -3, -1, 0, 2, 3, 8, 9, 14, 15, 16, 20, 21, 26, 27, 29, 30)


def world(kind, axis, rng):
    """One job's window as (48, 48, 48) blocks [y, z, x] from -16 for each edge: a glowstone there along `axis`."""
    out = []
    for at in EDGES:
        w = np.zeros((48, 48, 48), np.uint16)
        if kind == "blocks":
            w[rng.random(w.shape) < 0.3] = 1
        elif kind == "corridor":  # floors with one hole each, at alternating ends
            w[2::3] = 1
            w[2::6, 20:24, 20:24] = 0
            w[5::6, 24:28, 24:28] = 0
        pos = [24, 24, 24]
        pos[axis] = at + 16
        w[tuple(pos)] = workloads.GLOWSTONE
        out.append(w)
    return out


@pytest.mark.parametrize("kind", ["air", "blocks", "corridor"])
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_one_source_at_every_layer_edge(ctx, oracle, kind, axis):
    import os

    from conftest import GOLDEN

    levels = np.load(os.path.join(GOLDEN, "light.npz"))["light_levels"]
    rng = np.random.default_rng(axis)
    blocks, heights = [], []
    for w in world(kind, axis, rng):
        for d in workloads.SLOT_OFFSETS:
            x, y, z = 16 * (d + 1)
            blocks.append(w[y:y + 16, z:z + 16, x:x + 16].reshape(-1))
    blocks = np.stack(blocks)
    heights = np.full((blocks.shape[0], 256), 16, np.int8) if kind == "air" else cases.random_heights(axis, blocks.shape[0])
    n = len(EDGES)
    nbr = np.arange(27 * n, dtype=np.uint32).reshape(n, 27)
    want, _ = oracle.relight_many(levels, blocks, heights, nbr, 8, mesh=False, halo=True)
    store = hcm.Store(ctx, blocks.shape[0])
    store.upload(blocks, np.zeros(blocks.shape, np.uint8))
    store.upload_sunlight(heights)
    batch = hcm.Batch(ctx, store, nbr)
    batch.set_light(hcm.LIGHT_REBUILD)
    print(f"light layers: {kind}, axis {axis}", flush=True)
    batch.run()
    batch.sync()
    for j, at in enumerate(EDGES):
        assert np.array_equal(batch.fetch_light(j).reshape(-1), want[j].reshape(-1)), f"source at {at}"
    batch.close()
    store.close()
