"""The memory for dense chunks' face words grows with the launches that need it, also while an earlier launch that uses
the smaller one may still run (needs an MI355X). Checkerboards of up to 12,288 faces, against the oracle."""
import numpy as np
import pytest

import meshdigest
from hypercraft_amd import hcm, workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("threads", [256, 512])
def test_larger_launches_after_a_smaller_one(threads, oracle):
    rng = np.random.default_rng(threads)
    y, z, x = np.indices((16, 16, 16))
    odd = ((x + y + z) & 1).reshape(-1) == 1
    blocks = np.where(odd & (rng.random((54, 4096)) < 0.95), rng.integers(1, 4, (54, 4096)), 0).astype(np.uint16)
    light = rng.integers(0, 256, blocks.shape).astype(np.uint8)
    nbr = np.tile(np.arange(54, dtype=np.uint32).reshape(2, 27), (450, 1))
    want = [meshdigest.digest(oracle.mesh(*workloads.slice_jobs(blocks, light, nbr, j))) for j in range(2)]
    ctx = hcm.Context(pool_quads=900 * 12400)
    store = hcm.Store(ctx, 54)
    store.upload(blocks, light)
    ctx.set_tuning(wg_per_cu=1, threads=threads)
    few, many = hcm.Batch(ctx, store, nbr[:3]), hcm.Batch(ctx, store, nbr)
    for wg_per_cu in (1, 3, 2, 4):
        print(f"900 dense jobs, {wg_per_cu} x {threads} threads after 3 jobs", flush=True)
        ctx.set_tuning(wg_per_cu=1, threads=threads)
        few.run()
        many.run()
        ctx.set_tuning(wg_per_cu=wg_per_cu, threads=threads)
        many.run()  # the runs before it may still be on the device
        out = many.download()
        for j in range(0, 900, 23):
            assert meshdigest.digest(hcm.job_meshes(j, *out)) == want[j & 1], j
    few.close(), many.close(), store.close(), ctx.close()
