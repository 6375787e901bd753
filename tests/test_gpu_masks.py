"""Visibility masks, face words and merging on registries whose blocks show another texture on every face
(needs an MI355X): the classes of a block's six faces, its light passes and its collision are drawn at random, so that
every pair of face classes meets along every axis and direction, at the chunk's rim too, and bits of one face's plane
in another's would change the meshes. Whole numbers: the oracle's meshes, exactly."""
import numpy as np
import pytest

import cases
import meshdigest
from conftest import REGISTRY
from hypercraft_amd import hcm, workloads

pytestmark = pytest.mark.gpu


def shuffled_registry(tmp_path, seed):
    reg = cases.RegistryFile(REGISTRY)
    rng = np.random.default_rng(seed)
    full = np.unique(reg.rows["tex"])
    pool = np.concatenate([full[full != 0][rng.permutation((full != 0).sum())[:24]], [0, 0, 0]])
    plain = reg.rows["mesh"] == 0xFFFF
    plain[reg.row_of[0]] = False  # air stays air
    n = int(plain.sum())
    reg.rows["tex"][plain] = pool[rng.integers(0, pool.size, (n, 6))]
    reg.rows["transparency"][plain] = rng.integers(0, 3, n)
    reg.rows["collision"][plain] = rng.integers(0, 3, n)
    path = str(tmp_path / f"registry_{seed}.bin")
    reg.write(path)
    return reg, path


@pytest.mark.parametrize("seed,density,threads", [(1, 1.0, 256), (2, 0.5, 256), (3, 0.5, 128), (4, 0.7, 512), (5, 0.06, 256)])
def test_meshes_of_blocks_with_six_textures(tmp_path, seed, density, threads):
    import cpu_oracle

    reg, path = shuffled_registry(tmp_path, seed)
    orc = cpu_oracle.Oracle(path)
    values = cases.ALL_VALUES if seed % 2 else cases.ALL_VALUES[(cases.ALL_VALUES & 0xFF) != 15]
    rng = np.random.default_rng(100 + seed)
    n = 6
    blocks = np.where(rng.random((27 * n, 4096)) < density, values[rng.integers(0, values.size, (27 * n, 4096))], 0).astype(np.uint16)
    light = rng.integers(0, 256, blocks.shape).astype(np.uint8)
    nbr = np.arange(27 * n, dtype=np.uint32).reshape(n, 27)
    ctx = hcm.Context(pool_quads=1 << 20, registry=reg.c_registry(hcm))
    ctx.set_tuning(wg_per_cu=0, threads=threads)
    store = hcm.Store(ctx, blocks.shape[0])
    store.upload(blocks, light)
    batch = hcm.Batch(ctx, store, nbr)
    print(f"six textures: seed {seed}, density {density}, threads {threads}", flush=True)
    batch.run()
    batch.sync()
    out = batch.download()
    assert (out[0]["status"] == 0).all() and (out[0]["quad_count"] > 0).all()
    for j in range(n):
        b27, l27 = workloads.slice_jobs(blocks, light, nbr, j)
        want = meshdigest.digest(orc.mesh(b27, l27))
        assert meshdigest.digest(hcm.job_meshes(j, *out)) == want, f"job {j}"
        assert meshdigest.digest(ctx.mesh_chunk(b27, l27)) == want, f"job {j}, plain"
    batch.close()
    store.close()
    ctx.close()
