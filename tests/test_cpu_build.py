"""Memory faults and allocations of the library, on the CPU build of its sources (tests/cpp/hipcpu; no GPU). With
HIPCPU_GUARD every device and pinned allocation ends at an inaccessible page, so that an access past one ends the
process: each check runs in one of its own."""
import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "hypercraft_amd", "_build", "cpu", "libhcm_cpu.so")


def dense(n):
    """n jobs whose own chunks are checkerboards of 12,288 faces, one quad each: two blocks in turn."""
    y, z, x = np.indices((16, 16, 16))
    odd = ((x + y + z) & 1).reshape(-1) == 1
    blocks = np.zeros((27, 4096), np.uint16)
    blocks[26] = np.where(odd, np.where(np.arange(4096) & 32, 1, 2), 0)
    light = np.random.default_rng(7).integers(0, 256, blocks.shape).astype(np.uint8)
    return blocks, light, np.tile(np.arange(27, dtype=np.uint32), (n, 1))


def batch_of(hcm, ctx, n):
    blocks, light, nbr = dense(n)
    store = hcm.Store(ctx, 27)
    store.upload(blocks, light)
    return hcm.Batch(ctx, store, nbr)


def check_download_of_a_full_pool(pool_quads):
    """A run that wants more quads than the pool has: what fits is handed out, and nothing past the pool is read."""
    from hypercraft_amd import hcm

    ctx = hcm.Context(pool_quads=pool_quads)
    batch = batch_of(hcm, ctx, 3)
    batch.run()
    wanted = batch.totals()[0]
    res, _, verts, idx = batch.download()
    full = res["status"] == hcm.HCM_ERR_POOL_FULL
    assert full.any() and wanted == res["quad_count"].sum() > pool_quads and wanted < 45000
    kept = int(res["quad_count"][~full].sum())  # the first chunks that fit: 12,288 quads each
    assert verts[: 4 * kept].any(axis=1).all() and not verts[4 * pool_quads :].any()
    assert idx.reshape(-1, 6)[:kept].any(axis=1).all() and not idx[6 * pool_quads :].any()


KEPT = 8192 * 10  # bytes of a workgroup's memory for dense chunks; the CPU build has two CUs


def count(hcm, name):
    f = getattr(hcm.lib(), "hipcpu_" + name)
    f.restype = ctypes.c_size_t
    return f()


def allocated(hcm):
    return count(hcm, "allocated")


def check_dense_memory_of_one_job():
    """The memory for dense chunks is that of the workgroups a batch can launch, whatever the tuning allows."""
    from hypercraft_amd import hcm

    ctx = hcm.Context(pool_quads=1 << 14)
    ctx.set_tuning(wg_per_cu=64, threads=256)
    before = allocated(hcm)
    batch = batch_of(hcm, ctx, 1)
    assert allocated(hcm) - before < 1 << 20  # (its store is 0.34 MB)
    batch.run()
    assert allocated(hcm) - before < 1 << 20 and batch.totals() == (12288, 1)


def check_dense_memory_grows():
    """A batch whose launches grow beyond the workgroups the memory was made for gets more of it, once."""
    from hypercraft_amd import hcm
    import meshdigest

    ctx = hcm.Context(pool_quads=12 * 12288)
    ctx.set_tuning(wg_per_cu=1, threads=256)
    batch = batch_of(hcm, ctx, 12)
    digests = []
    sizes = [allocated(hcm)]
    for wg_per_cu in (1, 3, 1, 3):
        ctx.set_tuning(wg_per_cu=wg_per_cu, threads=256)
        batch.run()
        sizes.append(allocated(hcm))
        out = batch.download()
        digests.append({meshdigest.digest(hcm.job_meshes(j, *out)) for j in range(12)})
    assert np.diff(sizes).tolist() == [0, 4 * KEPT, 0, 0], np.diff(sizes)
    assert len(digests[0]) == 1 and digests == digests[:1] * 4


def check_pinned_memory_touched():
    """A context touches its pinned input and little of its 2 MiB of pinned output before it has batches, and then as much
    as they are large."""
    from hypercraft_amd import hcm

    ctx = hcm.Context(pool_quads=1 << 16)
    touched = [count(hcm, "pinned_touched")]
    for n in (1, 37, 400, 37, 1000):
        batch_of(hcm, ctx, n)
        touched.append(count(hcm, "pinned_touched"))
    made, one, few, many, after, most = touched
    inputs = 27 * 4096 * 2 + 14400 + 5832
    assert inputs <= made <= inputs + (96 << 10)
    assert made <= one <= made + (96 << 10)  # (room for 1,027 records)
    assert 37 * 128 * 44 < few - made < 37 * 128 * 44 + (112 << 10)
    assert inputs + (2 << 20) - (64 << 10) <= many <= inputs + (2 << 20) + (64 << 10)
    assert many <= after <= most <= inputs + (2 << 20) + (64 << 10)


def check_tuning_round_trip():
    """What hcm_get_tuning returns, given back, changes nothing: with no workgroup size set, batches of few jobs still
    take another than the one it names."""
    from hypercraft_amd import hcm

    ctx = hcm.Context(pool_quads=1 << 14)
    fresh = ctx.get_tuning()
    assert fresh == {"wg_per_cu": 0, "threads": 256, "default_threads": True}
    ctx.set_tuning(**fresh)
    assert ctx.get_tuning() == fresh
    ctx.set_tuning(**dict(fresh, wg_per_cu=2))
    assert ctx.get_tuning() == dict(fresh, wg_per_cu=2)
    for threads in (128, 256, 512):
        ctx.set_tuning(wg_per_cu=2, threads=threads)
        asked = ctx.get_tuning()
        assert asked == {"wg_per_cu": 2, "threads": threads, "default_threads": False}
        ctx.set_tuning(**asked)
        assert ctx.get_tuning() == asked
    ctx.set_tuning(threads=0)
    assert ctx.get_tuning() == fresh


def check_retry_after_failed_allocation(n):
    """A call whose n-th allocation failed can be made again."""
    from hypercraft_amd import hcm, workloads

    ctx = hcm.Context(pool_quads=1 << 14)
    batch = batch_of(hcm, ctx, 1)

    def twice(call):
        hcm.lib().hipcpu_fail_allocation(n)
        try:
            call()
        except hcm.HcmError:
            pass
        hcm.lib().hipcpu_fail_allocation(0)
        return call()

    twice(lambda: batch.set_light(hcm.LIGHT_REBUILD))
    batch.run()
    assert batch.results()["status"][0] == 0
    infos = twice(lambda: batch.mesh_infos(np.zeros((1, 3), np.int32)))
    opaque, clear = batch.cull(np.array([8, 8, -20], np.float32), workloads.look_at_projection(np.array([8, 8, -20], np.float32), (8, 8, 8)))
    assert len(infos) == len(opaque) + len(clear) == 1


@pytest.fixture(scope="module", autouse=True)
def library():
    subprocess.run(["make", "-s", "-j4", "-C", os.path.join(ROOT, "tests", "cpp", "hipcpu")], check=True, timeout=900,
                   stderr=subprocess.DEVNULL)


def run(check, *args):
    env = dict(os.environ, HCM_LIB=LIB, HIPCPU_GUARD="1")
    p = subprocess.run([sys.executable, __file__, check.__name__, *map(str, args)], capture_output=True, text=True,
                       timeout=600, env=env)
    assert p.returncode == 0, f"exit status {p.returncode}\n" + (p.stdout + p.stderr)[-4000:]


# smaller than a chunk's 12,288 quads, one chunk's, two and a half chunks'
@pytest.mark.parametrize("pool_quads", [1000, 12288, 30000])
def test_download_of_a_full_pool(pool_quads):
    run(check_download_of_a_full_pool, pool_quads)


def test_dense_memory_of_one_job():
    run(check_dense_memory_of_one_job)


def test_dense_memory_grows():
    run(check_dense_memory_grows)


def test_pinned_memory_touched():
    run(check_pinned_memory_touched)


def test_tuning_round_trip():
    run(check_tuning_round_trip)


@pytest.mark.parametrize("n", [1, 2, 3, 4])
def test_retry_after_failed_allocation(n):
    run(check_retry_after_failed_allocation, n)


if __name__ == "__main__":
    sys.path[:0] = [ROOT, os.path.join(ROOT, "tests")]
    globals()[sys.argv[1]](*map(int, sys.argv[2:]))
