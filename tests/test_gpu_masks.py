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


def chunk_with_faces(n):
    """27 chunks whose middle one has exactly n visible faces: stone blocks apart from each other (six faces each), with
    stone beyond x, y and z = 15, which hides a face of the blocks along those sides."""
    fours = [(x, 15, 15) for x in range(1, 14, 2)]
    put = {0: [], 1: [(15, 15, 15)] + fours[:1], 2: fours[:2], 3: [(15, 15, 15)], 4: fours[:1], 5: [(15, 15, 15)] + fours[:2]}[n % 6]
    left = n - sum(3 if at[0] == 15 else 4 for at in put)
    inner = [(x, y, z) for y in range(14) for z in range(14) for x in range(14) if (x + y + z) % 2 == 0]
    put += inner[:left // 6]
    left -= 6 * min(left // 6, len(inner))
    b = np.zeros((16, 16, 16), np.uint16)  # [y, z, x]
    for x, y, z in put:
        b[y, z, x] = 1
    out = []
    for d in workloads.SLOT_OFFSETS:
        c = np.zeros((16, 16, 16), np.uint16)
        if not d.any():
            c = b
        elif (d == 1).any():
            c[0 if d[1] == 1 else slice(None), 0 if d[2] == 1 else slice(None), 0 if d[0] == 1 else slice(None)] = 1
        out.append(c.reshape(-1))
    return np.stack(out), left


@pytest.mark.parametrize("merge", [False, True])
@pytest.mark.parametrize("faces", [1, 2, 63, 64, 65, 128, 1343, 1344, 1345, 1471, 1472, 1473, 1536, 2496, 2497, 2688, 2689, 2944, 2945, 4416, 4417, 8232])
def test_face_counts_at_block_and_group_edges(ctx, oracle, faces, merge):
    """Visible faces are numbered by units of 64 mask bits, handled in blocks of 64 lanes and held in groups of up to
    1,344: counts at and beside those edges, with light that lets faces merge and light that does not."""
    if faces < 3:  # nothing apart has so few: a slab's top, and two
        b27 = [np.zeros(4096, np.uint16) if d[1] == 1 else np.ones(4096, np.uint16) for d in workloads.SLOT_OFFSETS]
        l27 = [np.zeros(4096, np.uint8)] * 27
    else:
        blocks, left = chunk_with_faces(faces)
        assert left == 0, (faces, left)
        b27 = list(blocks)
        rng = np.random.default_rng(faces)
        l27 = [np.full(4096, 0x3A, np.uint8) if merge else rng.integers(0, 256, 4096).astype(np.uint8) for _ in range(27)]
    print(f"{faces} faces, merge {merge}", flush=True)
    want = oracle.mesh(b27, l27)
    assert meshdigest.digest(ctx.mesh_chunk(b27, l27)) == meshdigest.digest(want)
    store = hcm.Store(ctx, 27)
    store.upload(np.stack(b27), np.stack(l27))
    for threads in (128, 256, 512):
        ctx.set_tuning(wg_per_cu=0, threads=threads)
        batch = hcm.Batch(ctx, store, np.arange(27, dtype=np.uint32).reshape(1, 27))
        batch.run()
        out = batch.download()
        batch.close()
        assert meshdigest.digest(hcm.job_meshes(0, *out)) == meshdigest.digest(want), threads
    ctx.set_tuning(wg_per_cu=0, threads=256)
    store.close()


@pytest.mark.parametrize("seed,reach,threads", [(1, 16, 256), (2, 17, 256), (3, 40, 512), (4, 255, 128), (5, 16, 512)])
def test_custom_meshes_with_any_vertices(tmp_path, seed, reach, threads):
    """Custom meshes whose faces have random corners, axes, light faces and textures (opaque and transparent pass), within
    their block (the light's interpolation in 16 bits) and past it (in 32, wrapping)."""
    import cpu_oracle

    reg = cases.RegistryFile(REGISTRY)
    rng = np.random.default_rng(seed)
    tex = np.unique(reg.rows["tex"])
    tex = tex[tex != 0]
    for m in reg.meshes:
        head = m[:16].view(np.uint32)
        if head[1] != 0:
            continue  # liquid flow
        head[0] = rng.integers(1, 17)
        faces = m[16:].reshape(16, 24)
        faces[:, 0] = rng.integers(0, 3, 16)
        faces[:, 1:3] = rng.integers(0, 6, (16, 2))
        faces[:, 4:6] = rng.choice(tex, 16).astype(np.uint16).reshape(16, 1).view(np.uint8)
        corners = faces[:, 8:].reshape(16, 4, 4)
        corners[..., :3] = rng.integers(0, reach + 1, (16, 4, 3))
        corners[..., 3] = rng.integers(0, 5, (16, 4))
    path = str(tmp_path / f"registry_custom_{seed}.bin")
    reg.write(path)
    orc = cpu_oracle.Oracle(path)
    values = cases.CUSTOM
    n = 4
    blocks = np.where(rng.random((27 * n, 4096)) < (0.02, 0.4)[seed % 2], values[rng.integers(0, values.size, (27 * n, 4096))], 0).astype(np.uint16)
    light = rng.integers(0, 256, blocks.shape).astype(np.uint8)
    nbr = np.arange(27 * n, dtype=np.uint32).reshape(n, 27)
    ctx = hcm.Context(pool_quads=1 << 20, registry=reg.c_registry(hcm))
    ctx.set_tuning(wg_per_cu=0, threads=threads)
    store = hcm.Store(ctx, blocks.shape[0])
    store.upload(blocks, light)
    batch = hcm.Batch(ctx, store, nbr)
    print(f"custom meshes: seed {seed}, reach {reach}, threads {threads}", flush=True)
    batch.run()
    out = batch.download()
    for j in range(n):
        b27, l27 = workloads.slice_jobs(blocks, light, nbr, j)
        want = meshdigest.digest(orc.mesh(b27, l27))
        assert meshdigest.digest(hcm.job_meshes(j, *out)) == want, f"job {j}"
        assert meshdigest.digest(ctx.mesh_chunk(b27, l27)) == want, f"job {j}, plain"
    batch.close()
    store.close()
    ctx.close()


@pytest.mark.parametrize("n", [255, 256, 257])
def test_batches_around_a_job_per_cu(n, oracle):
    """Up to a job per CU a batch runs in workgroups of 512 threads, unless a size was asked for; beyond, in 256."""
    rng = np.random.default_rng(n)
    values = np.concatenate([cases.CUSTOM, np.arange(1, 9, dtype=np.uint16)])
    blocks = np.where(rng.random((54, 4096)) < 0.1, values[rng.integers(0, values.size, (54, 4096))], 0).astype(np.uint16)
    light = rng.integers(0, 256, blocks.shape).astype(np.uint8)
    nbr = np.tile(np.arange(54, dtype=np.uint32).reshape(2, 27), (n, 1))[:n]
    want = [meshdigest.digest(oracle.mesh(*workloads.slice_jobs(blocks, light, nbr, j))) for j in range(2)]
    ctx = hcm.Context(pool_quads=1 << 21)
    store = hcm.Store(ctx, 54)
    store.upload(blocks, light)
    for asked in (None, 256, 512):
        if asked:
            ctx.set_tuning(wg_per_cu=0, threads=asked)
        batch = hcm.Batch(ctx, store, nbr)
        print(f"{n} jobs, threads {asked}", flush=True)
        for _ in range(2):
            batch.run()
        out = batch.download()
        for j in range(n):
            assert meshdigest.digest(hcm.job_meshes(j, *out)) == want[j & 1], (asked, j)
        batch.close()
    store.close()
    ctx.close()


@pytest.mark.parametrize("kind,seed,threads", [("mesh", 1, 256), ("face", 2, 256), ("both", 3, 512), ("cubes", 4, 256), ("both", 5, 128)])
def test_blocks_in_front_that_pass_no_light(tmp_path, kind, seed, threads):
    """Voxel words hold no light where a block passes none, unless the registry has such a block that a visible face may
    look at: one with a face that is not opaque, or with a mesh. Blocks that pass none and are opaque cubes need no more."""
    import cpu_oracle

    reg = cases.RegistryFile(REGISTRY)
    rng = np.random.default_rng(seed)
    flags = reg.tex_flags[np.minimum(reg.rows["tex"] & 0x1FFF, len(reg.tex_flags) - 1)]
    cube = (((reg.rows["tex"] & 0x1FFF) != 0) & ((flags & 5) == 0)).all(axis=1)
    mesh = reg.rows["mesh"] != 0xFFFF
    pick = {"mesh": mesh, "face": ~cube & ~mesh, "both": np.ones(len(mesh), bool), "cubes": cube & ~mesh}[kind]
    assert pick.any()
    reg.rows["transparency"][pick & (rng.random(len(mesh)) < 0.7)] = 0
    path = str(tmp_path / f"registry_{kind}.bin")
    reg.write(path)
    orc = cpu_oracle.Oracle(path)
    ids = np.arange(1, 256)
    values = np.unique(np.concatenate([cases.CUSTOM, ids[reg.row_of[ids] != reg.row_of[255]], ids[:40], ids[:40] | 0x100]))
    n = 3
    blocks = np.where(rng.random((27 * n, 4096)) < 0.4, values[rng.integers(0, values.size, (27 * n, 4096))], 0).astype(np.uint16)
    light = rng.integers(0, 256, blocks.shape).astype(np.uint8)
    nbr = np.arange(27 * n, dtype=np.uint32).reshape(n, 27)
    ctx = hcm.Context(pool_quads=1 << 20, registry=reg.c_registry(hcm))
    ctx.set_tuning(wg_per_cu=0, threads=threads)
    store = hcm.Store(ctx, blocks.shape[0])
    store.upload(blocks, light)
    batch = hcm.Batch(ctx, store, nbr)
    print(f"no light through {kind}: {threads} threads", flush=True)
    batch.run()
    out = batch.download()
    for j in range(n):
        b27, l27 = workloads.slice_jobs(blocks, light, nbr, j)
        want = meshdigest.digest(orc.mesh(b27, l27))
        assert meshdigest.digest(hcm.job_meshes(j, *out)) == want, f"job {j}"
        assert meshdigest.digest(ctx.mesh_chunk(b27, l27)) == want, f"job {j}, plain"
    batch.close()
    store.close()
    ctx.close()


@pytest.mark.parametrize("n,wg_per_cu,threads", [(3, 0, 0), (300, 0, 0), (2, 0, 128), (3, 0, 512), (1030, 4, 128)])
def test_dense_chunks_past_the_kept_faces(n, wg_per_cu, threads, oracle):
    """A batch's workgroups keep the words of a dense chunk's first 8,192 faces until its quads are written, as many of them
    as the memory was made for; past either they are computed again. Checkerboards of 12,288 faces and fewer."""
    rng = np.random.default_rng(n)
    y, z, x = np.indices((16, 16, 16))
    odd = ((x + y + z) & 1).reshape(-1) == 1
    solid = np.array([1, 2, 3, 9, 10, 4], np.uint16)
    blocks = np.where(odd & (rng.random((54, 4096)) < 0.9), solid[rng.integers(0, solid.size, (54, 4096))], 0).astype(np.uint16)
    blocks[26] = np.where(odd, 1, 0)  # the first job's own chunk (the neighbour slot of all coordinates 0)
    light = rng.integers(0, 256, blocks.shape).astype(np.uint8)
    nbr = np.tile(np.arange(54, dtype=np.uint32).reshape(2, 27), (n, 1))[:n]
    want = [meshdigest.digest(oracle.mesh(*workloads.slice_jobs(blocks, light, nbr, j))) for j in range(2)]
    ctx = hcm.Context(pool_quads=n * 13000)
    if threads:
        ctx.set_tuning(wg_per_cu=wg_per_cu, threads=threads)
    store = hcm.Store(ctx, 54)
    store.upload(blocks, light)
    batch = hcm.Batch(ctx, store, nbr)
    print(f"{n} dense jobs, {wg_per_cu} x {threads} threads", flush=True)
    for _ in range(2):
        batch.run()
    out = batch.download()
    assert out[0]["quad_count"][0] > 11000
    for j in range(0, n, 1 if n < 10 else 23):
        assert meshdigest.digest(hcm.job_meshes(j, *out)) == want[j & 1], j
    batch.close()
    store.close()
    ctx.close()
