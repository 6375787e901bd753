// hcm_light.hip -- gfx950 kernels of the light rebuild before meshing (client/src/ChunkMeshTask.cpp:48-111).
//
// The reference's mesh task rebuilds light over its chunk's [-15, 31)^3 neighbourhood: torchlight from
// the blocks' light levels, sunlight 15 at and above each column's sunlight height, then a first-in
// first-out propagation (client/include/client/BlockLightAlgo.hpp:44-73) that lowers the level by one
// per step into blocks that pass light indirectly, pruned where a level cannot reach the bound
// [-1, 17)^3 (BlockLightAlgo.hpp:32-42 with ChunkMeshTask.inl:53-56). The mesher reads only the 18^3
// cells of that bound. Along a path that ends in the bound with level >= 1, the level exceeds the
// distance to the bound at every cell, so the pruning never changes those cells: there the result is
// the max-plus fixpoint
//     L(v) = max(L0(v), max over the six neighbours u of L(u) - 1, when v passes light),
// whatever order the propagation runs in. This file computes it level by level on bit masks. With G_k
// the cells of level >= k,
//     G_15 = sources of level 15,   G_k = G_{k+1} | sources of level k | (dilate(G_{k+1}) & passable),
// one 46-bit x-row of the 46-wide window per lane; at step k only rows within distance k - 1 of the
// bound can still reach it. A cell's level is the largest k with the cell in G_k.
//
// Two kernels:
//   light_prep_kernel  one workgroup per store slot the batch reads: packs its blocks' light pass, its
//                      sunlit cells (from the sunlight heights), its level-15 torchlight sources and its
//                      torchlight levels into 16-bit x-rows (4 KB per slot);
//   light_kernel       one workgroup per job (persistent, per-XCD work queues): assembles the 46^3 window
//                      from the 27 slots' packed rows in registers, runs the sunlight and torchlight levels,
//                      and writes the 18^3 rebuilt light bytes (sun | torch << 4) the mesher reads.
#include <hip/hip_runtime.h>

#include "hcm_device.h"

namespace hcm {

namespace {

constexpr int kW = 46;                 // window [-15, 31) per axis
constexpr int kH = 18;                 // the mesher's halo [-1, 17) per axis
constexpr int kHRows = kH * kH;        // halo x-rows, index hz + 18 hy
constexpr int kHOff = 14;              // window index of halo index 0
constexpr int kLightThreads = 512;
constexpr int kLightWaves = kLightThreads / 64;
// A wavefront holds kPlanes layers of the window along y, a lane one row z of each (46 of the 64 lanes): a
// row's neighbours along z are the neighbouring lanes', those along y are in the lane's own registers but for
// the wavefront's first and last layer, which go through LDS. A level step of a layer is 16 VALU instructions
// and no LDS; eight wavefronts of six layers at 64 registers fill a CU's wavefronts four workgroups deep. The
// step is bound by VALU issue (91.1 M instructions for 4,096 jobs of the lit cave region, 148 us at full issue,
// 183 us measured; on another region of the kind, that of the figures below, 88.6 M, 144 and 174). The earlier kernel
// kept the whole window in LDS, one row per thread and step, with six LDS reads and a write per row: 223 us. Six
// wavefronts of eight layers took 207 us, a wavefront skipping steps that can change none of its rows 181 us (the
// skipped work is less than the bookkeeping).
constexpr int kPlanes = 6;
static_assert(kLightWaves * kPlanes >= kW && kW <= 64, "the wavefronts' layers cover the window");
constexpr int kEdgeLanes = 48; // rows of an exchanged layer: 46 and two that are always empty

// The wavefronts whose layers meet the halo record all of theirs: layers kHFirst .. kHFirst + kHLayers - 1.
constexpr int kHWave = kHOff / kPlanes, kHFirst = kHWave * kPlanes;
constexpr int kHWaves = (kHOff + kH + kPlanes - 1) / kPlanes - kHWave, kHLayers = kHWaves * kPlanes;
constexpr int kHRec = kHLayers * kH, kHBefore = (kHOff - kHFirst) * kH; // rows recorded per level, and those before the halo's

struct LightSmem {
	uint2 edge[2][kLightWaves][2][kEdgeLanes]; // by the step's parity: each wavefront's first and last layer
	uint32_t halo[15][kHRec];                  // G_1 .. G_15 over the halo's x-rows (bits past the 18th are others'), see kHRec
	uint32_t slots[27];
	uint32_t changed[3]; // per level step (rotating): some row of the step changed
	uint32_t levels;     // torchlight levels present in the 27 chunks
	uint32_t job;
};

// Neighbour-slot terms along an axis (CmpXYZ2NeighbourIndex, common/include/common/Position.hpp:138-145):
// L(-1) = 1, L(0) = 2, L(1) = 0.
__device__ __forceinline__ int slot_term(int v) { return v < 0 ? 1 : (v >= 16 ? 0 : 2); }

// The packed records of a window row: x in [-15, 0) from the -x chunk, [0, 16) from the centre column,
// [16, 31) from the +x chunk.
struct RowSrc {
	uint2 l, c, r;
};
// record 0: x = light pass | sunlit << 16, y = level-15 torchlight sources; record 1: the four bits of the
// torchlight level.
__device__ __forceinline__ RowSrc row_src(const LightParams &p, const LightSmem &s, int wy, int wz, int record) {
	const int y = wy - 15, z = wz - 15, yz = 3 * slot_term(y) + slot_term(z);
	const uint2 *rows = reinterpret_cast<const uint2 *>(p.packed) + 256 * record + (z & 15) + 16 * (y & 15);
	constexpr size_t stride = kLightSlotBytes / sizeof(uint2);
	return {rows[s.slots[9 + yz] * stride], rows[s.slots[18 + yz] * stride], rows[s.slots[yz] * stride]};
}
// The window row (lo, hi) of three 16-bit rows.
__device__ __forceinline__ uint2 window_row(uint32_t l, uint32_t c, uint32_t r) {
	return make_uint2((l >> 1) | (c << 15) | (r << 31), (r >> 1) & 0x3fffu);
}

// Lane z's value from lane z - 1 and z + 1 (0 beyond the wavefront): wave_shr:1, wave_shl:1.
__device__ __forceinline__ uint32_t from_prev(uint32_t v) { return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x138, 0xf, 0xf, true); }
__device__ __forceinline__ uint32_t from_next(uint32_t v) { return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x130, 0xf, 0xf, true); }

// The halo's x and z part of this wavefront's layers of G_k into s.halo.
__device__ __forceinline__ void record_halo(LightSmem &s, uint32_t k, int wave, int lane, const uint2 g[kPlanes]) {
	if ((unsigned)(wave - kHWave) >= (unsigned)kHWaves) // the same for the whole wavefront
		return;
	const int hz = lane - kHOff;
	if ((unsigned)hz < (unsigned)kH) {
		uint32_t *rec = s.halo[k - 1] + (wave - kHWave) * kPlanes * kH + hz;
#pragma unroll
		for (int q = 0; q < kPlanes; ++q)
			rec[q * kH] = (g[q].x >> kHOff) | (g[q].y << (32 - kHOff));
	}
}

// One channel from its G_15, with s.changed clear: G_k over the halo into s.halo[k - 1] for k down to the
// returned level; the lower ones equal that one. A step that adds no cell to its rows leaves G unchanged for
// every later step (each later step reads only rows of the earlier step), so the channel ends there unless
// sources enter at a lower level; one without a cell of level 15 ends at once.
__device__ __forceinline__ uint32_t propagate(const LightParams &p, LightSmem &s, int wave, int lane, uint2 g[kPlanes],
                                              const uint2 pass[kPlanes], bool inject) {
	record_halo(s, 15, wave, lane, g);
	uint32_t any = 0;
#pragma unroll
	for (int q = 0; q < kPlanes; ++q)
		any |= g[q].x | g[q].y;
	if (__ballot(any != 0) && lane == 0)
		s.changed[15 % 3] = 1;
	uint32_t end = 15;
#pragma unroll 1
	for (uint32_t k = 14; k >= 1; --k) {
		uint2(*edge)[2][kEdgeLanes] = s.edge[k & 1];
		if (lane < kEdgeLanes) {
			edge[wave][0][lane] = g[0];
			edge[wave][1][lane] = g[kPlanes - 1];
		}
		__syncthreads();
		if (!s.changed[(k + 1) % 3] && !(inject && (s.levels & ((2u << k) - 1u))))
			break;
		end = k;
		if (threadIdx.x == 0)
			s.changed[(k + 2) % 3] = 0; // the flag of step k - 1, last read before this step's barrier
		// rows past distance k - 1 of the bound cannot reach it any more
		if (kPlanes * wave + kPlanes <= 15 - int(k) || kPlanes * wave >= 31 + int(k))
			continue;
		const int el = min(lane, kEdgeLanes - 1);
		uint2 before = wave > 0 ? edge[wave - 1][1][el] : make_uint2(0, 0);
		const uint2 after = wave < kLightWaves - 1 ? edge[wave + 1][0][el] : make_uint2(0, 0);
		const bool inj = inject && ((s.levels >> k) & 1u);
		uint32_t changed = 0;
#pragma unroll
		for (int q = 0; q < kPlanes; ++q) {
			const uint2 o = g[q], up = q < kPlanes - 1 ? g[q + 1] : after;
			const uint32_t dx = (o.x << 1) | ((o.x >> 1) | (o.y << 31)) | before.x | up.x | from_prev(o.x) | from_next(o.x);
			const uint32_t dy = ((o.y << 1) | (o.x >> 31)) | (o.y >> 1) | before.y | up.y | from_prev(o.y) | from_next(o.y);
			uint2 n = make_uint2(o.x | (dx & pass[q].x), o.y | (dy & pass[q].y));
			changed |= (n.x ^ o.x) | (n.y ^ o.y);
			before = o;
			g[q] = n;
		}
		if (inj) { // sources of level k
			// (the layer index by way of readfirstlane, so that the addresses are not computed ahead of the steps and
			// held in registers through all of them)
			const int w0 = kPlanes * __builtin_amdgcn_readfirstlane(wave);
#pragma unroll
			for (int q = 0; q < kPlanes; ++q) {
				const RowSrc t = row_src(p, s, min(w0 + q, kW - 1), min(lane, kW - 1), 1);
				uint32_t ml = w0 + q < kW && lane < kW ? 0xffffu : 0u, mc = ml, mr = ml;
#pragma unroll
				for (int b = 0; b < 4; ++b) {
					const uint32_t flip = (k >> b) & 1u ? 0u : 0xffffu;
					ml &= ((b < 2 ? t.l.x : t.l.y) >> (16 * (b & 1))) ^ flip;
					mc &= ((b < 2 ? t.c.x : t.c.y) >> (16 * (b & 1))) ^ flip;
					mr &= ((b < 2 ? t.r.x : t.r.y) >> (16 * (b & 1))) ^ flip;
				}
				const uint2 src = window_row(ml, mc, mr);
				changed |= (src.x & ~g[q].x) | (src.y & ~g[q].y);
				g[q].x |= src.x, g[q].y |= src.y;
			}
		}
		record_halo(s, k, wave, lane, g);
		if (__ballot(changed != 0) && lane == 0)
			s.changed[k % 3] = 1;
	}
	__syncthreads();
	return end;
}

// The levels of halo row hr as four bit planes, from G_1 .. G_15 (each within the next lower one).
__device__ __forceinline__ void level_planes(const LightSmem &s, int hr, uint32_t end, uint32_t pl[4]) {
	uint32_t G[16];
#pragma unroll
	for (uint32_t k = 1; k < 16; ++k)
		G[k] = s.halo[max(k, end) - 1][kHBefore + hr];
	pl[3] = G[8];
	pl[2] = (G[4] & ~G[8]) | G[12];
	pl[1] = (G[2] & ~G[4]) | (G[6] & ~G[8]) | (G[10] & ~G[12]) | G[14];
	pl[0] = (G[1] & ~G[2]) | (G[3] & ~G[4]) | (G[5] & ~G[6]) | (G[7] & ~G[8]) | (G[9] & ~G[10]) | (G[11] & ~G[12]) |
	        (G[13] & ~G[14]) | G[15];
}

// Wavefront 0: the slot list of `job` and the torchlight levels present in its 27 chunks, into LDS.
__device__ __forceinline__ void light_slots(const LightParams &p, LightSmem &s, uint32_t job) {
	const int lane = threadIdx.x & 63;
	uint32_t slot = 0, lv = 0;
	if (lane < 27) {
		slot = p.nbr[27 * (size_t)job + lane];
		s.slots[lane] = slot;
		lv = p.levels[slot];
	}
#pragma unroll
	for (int d = 1; d < 64; d <<= 1)
		lv |= __shfl_xor(lv, d);
	if (lane == 0)
		s.levels = lv & ~1u;
}

// One job; s.slots and s.levels are in place and s.changed is clear (a barrier after them).
__device__ __forceinline__ void light_job(const LightParams &p, LightSmem &s, uint32_t job) {
	static_assert(kLightThreads >= kHRows, "one halo x-row per thread");
	const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	const bool torch = s.levels != 0;
	uint2 g[kPlanes], pass[kPlanes];
	uint32_t pl[8] = {}; // bit planes of the light bytes sun | torch << 4 (block/include/block/Light.hpp)
#pragma unroll 1
	for (int channel = 0;; ++channel) { // sunlight: 15 at and above the sunlight height (Chunk.hpp:73-79); then torchlight
		// (the layer index by way of readfirstlane, so that the addresses are not kept in registers through a channel)
		const int w0 = kPlanes * __builtin_amdgcn_readfirstlane(wave);
#pragma unroll
		for (int q = 0; q < kPlanes; ++q) { // lanes and layers past the window read some row of it and drop it
			const RowSrc t = row_src(p, s, min(w0 + q, kW - 1), min(lane, kW - 1), 0);
			const uint32_t in = w0 + q < kW && lane < kW ? ~0u : 0u, l = t.l.x & in, c = t.c.x & in, r = t.r.x & in;
			if (channel == 0) {
				pass[q] = window_row(l & 0xffffu, c & 0xffffu, r & 0xffffu);
				g[q] = window_row(l >> 16, c >> 16, r >> 16);
			} else
				g[q] = window_row(t.l.y & in, t.c.y & in, t.r.y & in);
		}
		const uint32_t end = propagate(p, s, wave, lane, g, pass, channel != 0);
		if (tid < kHRows)
			level_planes(s, tid, end, pl + 4);
		if (channel != 0)
			break;
#pragma unroll
		for (int b = 0; b < 4; ++b)
			pl[b] = pl[4 + b], pl[4 + b] = 0;
		if (!torch)
			break;
		if (tid < 3)
			s.changed[tid] = 0;
		__syncthreads(); // every halo row's sunlight level is read
	}
	if (tid < kHRows) { // one 20-byte record per halo x-row: the planes' bits 8 j + b transposed are byte j of word b
		exchange_bits<4>(pl);
		exchange_bits<2>(pl);
		exchange_bits<1>(pl);
		uint32_t w[5];
#pragma unroll
		for (int j = 0; j < 4; ++j) { // bytes x = 4 j .. 4 j + 3
			const int b = 4 * (j & 1), sh = 8 * (j >> 1);
			w[j] = ((pl[b] >> sh) & 0xffu) | ((pl[b + 1] >> sh) & 0xffu) << 8 | ((pl[b + 2] >> sh) & 0xffu) << 16 |
			       ((pl[b + 3] >> sh) & 0xffu) << 24;
		}
		w[4] = ((pl[0] >> 16) & 0xffu) | ((pl[1] >> 16) & 0xffu) << 8;
		const size_t at = (size_t)job * (kLightJobBytes / 4) + tid * (kLightRowBytes / 4);
#pragma unroll
		for (int q = 0; q < 5; ++q)
			reinterpret_cast<uint32_t *>(p.halo_light)[at + q] = w[q];
		if (p.halo_light_copy)
#pragma unroll
			for (int q = 0; q < 5; ++q)
				reinterpret_cast<uint32_t *>(p.halo_light_copy)[at + q] = w[q];
	}
}

} // namespace

__global__ __launch_bounds__(256) void light_prep_kernel(LightParams p) {
	__shared__ uint32_t s_levels;
	const uint32_t slot = p.slots[blockIdx.x];
	const int row = threadIdx.x, y = row >> 4, z = row & 15;
	if (row == 0)
		s_levels = 0;
	const uint16_t *src = p.blocks + (size_t)slot * HCM_CHUNK_VOXELS + row * 16;
	const uint4 b0 = *reinterpret_cast<const uint4 *>(src), b1 = *reinterpret_cast<const uint4 *>(src + 8);
	const uint4 hv = *reinterpret_cast<const uint4 *>(p.heights + (size_t)slot * 256 + 16 * z);
	if (p.blocks_copy) {
		uint4 *copy = reinterpret_cast<uint4 *>(p.blocks_copy + (size_t)slot * HCM_CHUNK_VOXELS + row * 16);
		copy[0] = b0, copy[1] = b1;
	}
	const uint32_t bw[8] = {b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, b1.z, b1.w};
	const uint32_t hw[4] = {hv.x, hv.y, hv.z, hv.w};
	uint32_t info[16];
#pragma unroll
	for (int x = 0; x < 16; ++x)
		info[x] = p.light_info[(bw[x >> 1] >> (16 * (x & 1))) & 0xffffu];
	uint32_t pass = 0, sun = 0, t0 = 0, t1 = 0, t2 = 0, t3 = 0, t15 = 0, lv = 0;
#pragma unroll
	for (int x = 0; x < 16; ++x) {
		const int h = int(int8_t(hw[x >> 2] >> (8 * (x & 3))));
		sun |= uint32_t(y >= h) << x; // Chunk::GetSunlight (Chunk.hpp:73-76)
		pass |= ((info[x] & kLightInfoPass) ? 1u : 0u) << x;
		const uint32_t l = info[x] & 15u;
		t0 |= (l & 1u) << x, t1 |= ((l >> 1) & 1u) << x, t2 |= ((l >> 2) & 1u) << x, t3 |= ((l >> 3) & 1u) << x;
		t15 |= (l == 15u ? 1u : 0u) << x;
		lv |= 1u << l;
	}
	uint2 *dst = reinterpret_cast<uint2 *>(p.packed + (size_t)slot * (kLightSlotBytes / 2)) + row;
	dst[0] = make_uint2(pass | sun << 16, t15);
	dst[256] = make_uint2(t0 | t1 << 16, t2 | t3 << 16);
	__syncthreads();
	if (lv & ~1u)
		atomicOr(&s_levels, lv & ~1u);
	__syncthreads();
	if (row == 0)
		p.levels[slot] = s_levels;
}

__global__ __launch_bounds__(kLightThreads, 8) void light_kernel(LightParams p) {
	__shared__ LightSmem s;
	__shared__ JobClaims claims;
	if (threadIdx.x == 0) // (only this lane uses it)
		claims.init(p.n_jobs);
	for (;;) {
		if (threadIdx.x < 64) { // wavefront 0 claims the next job and loads its slot list and levels
			uint32_t job = ~0u;
			if (threadIdx.x == 0) {
				job = claims.next(p.ctr);
				s.job = job;
				s.changed[0] = s.changed[1] = s.changed[2] = 0;
			}
			job = (uint32_t)__shfl((int)job, 0);
			if (job < p.n_jobs)
				light_slots(p, s, job);
		}
		__syncthreads();
		const uint32_t job = s.job;
		if (job >= p.n_jobs)
			break;
		light_job(p, s, job);
		__syncthreads();
	}
	// as in the mesh kernel: the last workgroup to finish clears the queues for the next run
	if (p.self_reset && threadIdx.x == 0) {
		claims_returned();
		if (atomicAdd(&p.ctr->done, 1u) == gridDim.x - 1) {
			for (uint32_t q = 0; q < kQueues; ++q)
				p.ctr->queue[q].v = 0;
			p.ctr->dry.v = 0;
			p.ctr->done = 0;
		}
	}
}

hipError_t launch_light_prep(const LightParams &p, hipStream_t stream) {
	if (p.n_slots == 0)
		return hipSuccess;
	hipLaunchKernelGGL(light_prep_kernel, dim3(p.n_slots), dim3(256), 0, stream, p);
	return hipGetLastError();
}

hipError_t launch_light(const LightParams &p, int grid, hipStream_t stream) {
	hipLaunchKernelGGL(light_kernel, dim3(grid), dim3(kLightThreads), 0, stream, p);
	return hipGetLastError();
}

int light_lds_bytes() {
	return (int)sizeof(LightSmem);
}

} // namespace hcm
