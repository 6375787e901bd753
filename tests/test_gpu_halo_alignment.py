"""Packed halos at every alignment (needs an MI355X): the staging takes 16-byte loads of blocks and 8-byte loads of
light where both arrays allow them, single elements elsewhere. One halo and several, at addresses that are a multiple
of neither, of one of them and of both, give the meshes of hcm_mesh_chunk (whole numbers: exactly)."""
import numpy as np
import pytest

import meshdigest
from hypercraft_amd import hcm, workloads
from test_zz_no_alloc import Hip

pytestmark = pytest.mark.gpu
QUADS, RECS = 1 << 16, 64


@pytest.mark.parametrize("n", [1, 3, 8])
@pytest.mark.parametrize("skew_blocks,skew_light", [(0, 0), (2, 0), (8, 4), (0, 1), (14, 7), (16, 8)])
def test_halos_at_any_alignment(ctx, n, skew_blocks, skew_light):
    import ctypes

    blocks, light, nbr = workloads.terrain_region(n=(2, 3, 2), seed=3, flags=hcm.HCM_GEN_PLANTS, y0=0)
    jobs = [workloads.slice_jobs(blocks, light, nbr, j) for j in range(n)]
    halos = [hcm.halo_of_chunks(*j) for j in jobs]
    hip = Hip()
    try:
        d_hb, d_hl = hip.alloc(n * hcm.HALO_BLOCKS * 2 + 32), hip.alloc(n * hcm.HALO_LIGHT + 32)
        hb, hl = ctypes.c_void_p(d_hb.value + skew_blocks), ctypes.c_void_p(d_hl.value + skew_light)
        hip.put(hb, np.stack([b.reshape(-1) for b, _ in halos]))
        hip.put(hl, np.stack([a.reshape(-1) for _, a in halos]))
        d_v, d_i, d_r = hip.alloc(QUADS * 32), hip.alloc(QUADS * 12), hip.alloc(RECS * 40)
        d_res = hip.alloc(n * hcm.JOB_RESULT_DTYPE.itemsize)
        print(f"{n} halos, blocks at +{skew_blocks}, light at +{skew_light}", flush=True)
        hcm.check("hcm_mesh_halos_noalloc", hcm.lib().hcm_mesh_halos_noalloc(ctx.ptr, hb, hl, n, d_v, d_i, QUADS, d_r, RECS, d_res, None))
        res = hip.get(d_res, np.zeros(n, hcm.JOB_RESULT_DTYPE))
        recs = hip.get(d_r, np.zeros(RECS, hcm.MESH_REC_DTYPE))
        verts = hip.get(d_v, np.zeros((QUADS * 4, 2), np.uint32))
        idx = hip.get(d_i, np.zeros(QUADS * 6, np.uint16))
        for j in range(n):
            assert meshdigest.digest(hcm.job_meshes(j, res, recs, verts, idx)) == meshdigest.digest(ctx.mesh_chunk(*jobs[j])), j
    finally:
        hip.free_all()
