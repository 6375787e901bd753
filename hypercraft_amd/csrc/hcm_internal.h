// hcm_internal.h -- types shared by the gfx950 kernels (hcm_kernels.hip) and the host API (hcm_api.cpp).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/hcm.h"

namespace hcm {

constexpr int kMaxPid = 128;   // registry rows + dynamic liquid-texture rows kept in LDS
constexpr int kMaxCodes = 128; // distinct face textures kept in LDS
constexpr int kFlowPatterns = 17;

// Voxel word staged in LDS per halo voxel, laid out so that light4_init adds words as they are (the fields above the
// sums do not reach down into them): bit 0 zero and bits 1-4 the direct light pass, each four times; sunlight in bits
// 8-11, 1 for a block that passes indirect light in bit 14 and torchlight in bits 16-19, so that a sum of four
// has sunlight in bits 8-13, a count in bits 14-15 and torchlight in bits 16-21; the texture row in bits 23-29; flow.
constexpr int kVoxSunBit = 8, kVoxIndirectBit = 14, kVoxTorchBit = 16;
constexpr uint32_t kVoxDirect = 0x1eu;                   // VerticalLightPass || collision != solid (BlockMeshAlgo.hpp:119)
constexpr uint32_t kVoxIndirect = 1u << kVoxIndirectBit; // transparency != opaque (block/include/block/Block.hpp:70)
constexpr uint32_t kVoxSunTorch = 0xfu << kVoxSunBit | 0xfu << kVoxTorchBit;
constexpr uint32_t kVoxLight = kVoxSunTorch | kVoxIndirect;
constexpr int kVoxPidShift = 23; // texture row, 7 bits
constexpr uint32_t kVoxPidMask = 0x7fu;
constexpr uint32_t kVoxFlow = 1u << 30; // liquid flow (dynamic mesh and face textures)
// A block's template: in y its voxel word but for light; in x its face classes, flags, and kVoxSunTorch if its light counts.
constexpr uint32_t kTmplMesh = 1u; // has a custom mesh
constexpr uint32_t kTmplFlow = 2u;
constexpr uint32_t kTmplMeta = 4u; // (by block id) the texture row depends on the meta byte: the full table decides
constexpr int kVoxClassShift = 20; // 2-bit face class per BlockFace f at bit 20 + 2 f
// Face classes for BlockTexture::Show (texture/include/texture/BlockTexture.hpp:68-76)
constexpr uint32_t kClassEmpty = 0, kClassOpaque = 1, kClassTransparent = 2, kClassLiquid = 3;

// Code words: texture bits as the second word of a vertex has them, and in the upper bits, as a face word has them,
// the upper three of the code's own seven bits and whether its faces go to the transparent pass.
constexpr uint32_t kCodeVertex = 0x1fffu;
constexpr uint32_t kCodeLow = 0x0fffffffu;
constexpr uint32_t kCodeTransPass = 1u << 31;

// Texture-row flag (in rows[pid].y): a halo made of this row's block alone has visible faces.
constexpr uint32_t kRowSelfShow = 1u << 16;

// What a mesh workgroup holds in LDS for all its jobs, laid out in device memory as it is there: copied by one load per
// thread or two, where filling it from separate tables took dependent loads (37 plant chunks 22.9 us per pass, 22.15 so).
struct MeshTables {
	uint2 rows[kMaxPid];       // x = tc0..tc3 (8 bits each), y = tc4 | tc5 << 8 | kRowSelfShow | mesh << 24
	uint2 pid_vox[kMaxPid];    // templates by texture row
	uint2 tmpl_id[256];        // template by block id when the meta byte does not change it, else kTmplMeta
	uint32_t codes[kMaxCodes];
	// (sum << 2) / count of light4_init for every sum of lights of 0 to 15, by the fields of a sum of voxel words:
	// sunlight by sum | (count - 1) << 6 and moved up by the two bits a face word has it at, torchlight by
	// (count - 1) | sum << 2
	uint8_t sun_of[256], torch_of[256];
};
static_assert(sizeof(MeshTables) % 16 == 0, "copied in 16-byte words");

struct DevReg {
	const uint8_t *pid_of;         // [65536] Block::m_data -> texture row (pid)
	const hcm_custom_mesh *meshes; // [n_meshes]
	const uint32_t *mesh_sums;     // [n_meshes]: faces | (bit j: face j goes to the transparent pass) << 16
	uint32_t flow_pid_base;
	uint32_t flow_tex, flow_trans, src_id, flow_id;
};

// The persistent kernels' job list is cut into kQueues contiguous parts, one per XCD (gfx950 has 8,
// and workgroups are dispatched to them round-robin by workgroup id). A workgroup takes jobs from its
// own XCD's part first, so neighbouring chunks, which share halo data, are read through one L2; then it
// takes jobs from the other parts. The first jobs of a part belong to its workgroups, one each, so that only
// jobs beyond those are claimed by atomics, and a launch with no more jobs than workgroups makes none. Each
// counter sits on its own 256-byte line: all are hit by device-scope atomics, and atomics on one line are
// serialised where that line lives.
constexpr uint32_t kQueues = 8;

struct Counters {
	struct alignas(256) Line {
		uint32_t v;
	};
	Line queue[kQueues];               // jobs claimed from each part of the job list, past its workgroups' first ones
	Line dry;                          // bit q: part q had no job left for a claim
	alignas(256) uint32_t pool_cursor; // quads allocated in the pool
	alignas(256) uint32_t mesh_cursor; // mesh records allocated
	// self-resetting persistent runs: workgroups done; the last one copies the run's totals below and
	// clears every counter for the next run
	alignas(256) uint32_t done;
	uint32_t total_quads, total_meshes;
};

// Memory of a workgroup for the words (8 bytes) and descriptors (2) of a dense chunk's faces, from when it computes them
// until it emits their quads: the first 8,192, past which it computes them twice, as it does all without the memory.
// 1,000 chunks of random blocks (7,757 quads each) took 202.4 us computing all groups but the last twice, 181.6 so.
constexpr uint32_t kKeptFaces = 8192;
constexpr size_t kKeptBytes = kKeptFaces * 10;

// Device memory that no kernel writes: read by scalar loads where it is used.
#ifdef __HIP_DEVICE_COMPILE__
#define HCM_CONSTANT __attribute__((address_space(4)))
#else
#define HCM_CONSTANT
#endif

struct MeshParams {
	// By pointer: its members among the kernel's arguments were held in scalar registers from the start, which spilled
	// (4,096 cave chunks 78.5 us, 77.1 so).
	const HCM_CONSTANT DevReg *reg;
	const MeshTables *tables;
	uint32_t raw_front; // a block that passes no indirect light may stand in front of a visible face (or have a mesh)
	const uint16_t *blocks; // store: slot * 4096 + local
	const uint8_t *light;
	const uint32_t *nbr;    // 27 slots per job
	uint32_t n_jobs;
	uint32_t job_base; // per-chunk launches: job = job_base + blockIdx.x
	uint32_t persistent;
	uint32_t pool_cap; // quads
	Counters *ctr;
	uint2 *pool_verts;   // 4 vertices per quad
	uint16_t *pool_idx;  // 6 indices per quad
	hcm_mesh_rec *recs;
	uint32_t rec_cap;
	uint32_t self_reset; // persistent: the last workgroup to finish clears the counters (no reset kernel)
	hcm_job_result *results;
	// [n_jobs][kLightJobBytes]: each job's rebuilt light over its halo, or null: light from the store
	const uint8_t *halo_light;
	// Packed halos (include/hcm.h), job j's at j HCM_HALO_BLOCKS and j HCM_HALO_LIGHT, instead of a store (null:
	// the store). Launches of 512 threads. Any alignment, device or pinned host memory.
	const uint16_t *halo_in;
	const uint8_t *halo_in_light;
	uint8_t *kept;  // per workgroup kKeptBytes, or null
	uint32_t alone; // the launch's one job: its output starts at quad and record 0, the counters are not touched
};

// ---- light rebuild before meshing (client/src/ChunkMeshTask.cpp:48-111) ----
// Per store slot, the inputs of the light rebuild packed as 16-bit x-rows (bit x), two 8-byte records per row
// z + 16 y: first, for every row, the indirect light pass, the sunlit cells and the cells of torchlight level 15
// (16 bits unused); then, for every row, the four bits of the torchlight level.
constexpr size_t kLightSlotBytes = 2 * 256 * 8;
constexpr uint32_t kLightRowBytes = 20;                        // one halo x-row of rebuilt light (18 used)
constexpr uint32_t kLightJobBytes = 18 * 18 * kLightRowBytes; // rows hz + 18 hy
constexpr int kLightPerCu = 4; // workgroups of the persistent light kernel per CU: its 32 wavefronts
constexpr uint8_t kLightInfoPass = 0x10;     // light_info: level | kLightInfoPass when the block passes light
constexpr uint8_t kLightInfoVertical = 0x20; // ... | kLightInfoVertical when it passes sunlight straight down

struct LightParams {
	const uint16_t *blocks;    // store: slot * 4096 + local
	const int8_t *heights;     // store: slot * 256 + x + 16 z
	const uint8_t *light_info; // [65536] by Block::m_data
	const uint32_t *slots;     // the store slots the batch reads
	uint32_t n_slots;
	uint32_t n_jobs;
	uint16_t *packed;          // [store slots][kLightSlotBytes / 2]
	uint32_t *levels;          // [store slots]: bit l set when a voxel emits torchlight level l
	const uint32_t *nbr;       // 27 slots per job
	Counters *ctr;             // work queues of the persistent light kernel
	uint8_t *halo_light;       // [n_jobs][kLightJobBytes]
	uint8_t *halo_light_copy;  // a second copy of the same, or null
	uint16_t *blocks_copy;     // the packed slots' blocks as the packing pass read them, or null: slot * 4096 + local
	uint32_t self_reset;       // the last workgroup to finish clears the work queues (no reset kernel)
};

// One voxel edit of a device chunk store: slot, chunk-local index, block, light. local >= 4096 sets the
// slot's sunlight height local - 4096 (index x + 16 z) to the low byte of block instead.
struct VoxelEdit {
	uint32_t slot, local, block, light;
};

// Launchers (hcm_kernels.hip)
hipError_t launch_reset(Counters *ctr, hipStream_t stream);
hipError_t launch_mesh(const MeshParams &p, int threads, int grid, hipStream_t stream);
// staged chunk k (sblocks + 4096 k, and slight + 4096 k or sheights + 256 k; the unused one null) to store
// slot moves[i].y for k = moves[i].x, i < n; all arrays 16-byte aligned
hipError_t launch_upload_scatter(const uint16_t *sblocks, const uint8_t *slight, const int8_t *sheights,
                                 const uint2 *moves, uint32_t n, uint16_t *blocks, uint8_t *light, int8_t *heights,
                                 hipStream_t stream);
hipError_t launch_edits(uint16_t *blocks, uint8_t *light, int8_t *heights, const VoxelEdit *edits, uint32_t n,
                        hipStream_t stream);
int mesh_lds_bytes(int threads);

// What a run left on the device, copied to pinned host memory by one kernel: a launch and a synchronisation
// instead of copies that wait for one another (the totals say how much there is to copy).
struct ExportParams {
	const Counters *ctr = nullptr; // null: given_quads quads, no records
	uint32_t persistent = 1;       // totals: a persistent run's, else the cursors
	uint32_t given_quads = 0;
	const hcm_job_result *results = nullptr;
	uint32_t n_jobs = 0;
	const hcm_mesh_rec *recs = nullptr;
	uint32_t rec_cap = 0; // records there can be, and that fit out_recs
	const uint2 *verts = nullptr;
	const uint16_t *idx = nullptr;
	uint32_t quad_cap = 0; // quads that fit out_verts and out_idx: all of the run's or none
	uint32_t *out_totals = nullptr; // quads, mesh records
	hcm_job_result *out_results = nullptr;
	hcm_mesh_rec *out_recs = nullptr;
	uint2 *out_verts = nullptr;
	uint16_t *out_idx = nullptr;
};
hipError_t launch_export(const ExportParams &p, hipStream_t stream);
// Launchers (hcm_draw.hip)
// Depth hierarchy of the renderer's depth image (client/include/client/rg/DepthHierarchyPass.hpp:166-196):
// level 0 is the image, level i >= 1 is max(level i - 1 size >> 1, 1) per axis; the culling shader's
// texture holds levels 1 .. n_levels - 1 as its mips 0 .. n_levels - 2.
constexpr int kMaxDepthLevels = 16; // images up to 16384 x 16384 have at most 15 levels
struct DepthPyramid {
	const float *data = nullptr; // every level, level i at data + offset[i], row y at + y * width[i]
	uint32_t n_levels = 0;
	uint32_t width[kMaxDepthLevels] = {}, height[kMaxDepthLevels] = {}, offset[kMaxDepthLevels] = {};
};
struct CullParams {
	float view_pos[3];
	float view_proj[16]; // column-major
	DepthPyramid hiz;    // data == nullptr: frustum test only
};
// levels 1 .. h.n_levels - 1 from level 0, in `levels` (h.data's memory)
hipError_t launch_depth_levels(const DepthPyramid &h, float *levels, hipStream_t stream);
// The infos of the run's records (at most rec_cap); n receives their number, out2 (may be null) a second copy.
hipError_t launch_mesh_infos(const hcm_mesh_rec *recs, const Counters *ctr, uint32_t persistent, uint32_t rec_cap,
                             const int32_t *chunk_pos, hcm_mesh_info *out, hcm_mesh_info *out2, uint32_t *n,
                             hipStream_t stream);
struct CullCounts { // zero between launches
	uint32_t kept[2], done;
};
// out_counts: opaque and transparent draws
hipError_t launch_cull(const hcm_mesh_info *infos, uint32_t n, const CullParams &cp, hcm_draw_cmd *opaque,
                       hcm_draw_cmd *transparent, CullCounts *counts, uint32_t *out_counts, hipStream_t stream);
// Launchers (hcm_light.hip)
hipError_t launch_light_prep(const LightParams &p, hipStream_t stream);
hipError_t launch_light(const LightParams &p, int grid, hipStream_t stream);
int light_lds_bytes();

// Context internals the serving loop needs (hcm_api.cpp)
struct CtxInfo {
	const DevReg *reg;          // in device memory
	const MeshTables *tables;   // likewise
	uint32_t raw_front;
	int n_cu;
	uint32_t threads;
	uint32_t grid;              // persistent grid for `threads`
	uint32_t threads_few;       // workgroup size of launches of at most n_cu jobs
	const uint8_t *light_info;  // [65536] for the light rebuild
	const uint8_t *light_info_host; // the same table in host memory
};
int ctx_info(hcm_ctx *ctx, uint32_t threads, CtxInfo *out);

} // namespace hcm
