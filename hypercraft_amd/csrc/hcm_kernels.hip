// hcm_kernels.hip -- gfx950 chunk-meshing kernels.
//
// One workgroup meshes one 16^3 chunk at a time; a persistent workgroup takes chunk jobs from work
// queues (one per XCD, then the others') until they are empty. Per chunk:
//   1. staging: one thread per 18-voxel x-row of the 18^3 halo loads the row from its chunk slots with
//      vector loads and writes one LDS word per voxel: light byte, direct/indirect light-pass bits,
//      a 2-bit face class per face (empty / opaque / transparent / liquid), custom-mesh and flow bits
//      and the texture row. A chunk without a custom mesh whose halo holds a single block value (whose
//      opposite faces hide each other) or only opaque cubes, or none of whose own voxels has a face, has
//      no quads and stops here; so does one
//      with no visible face after step 3's visibility masks.
//   2. liquid-flow cells take their per-cell face textures (the reference's m_dynamic_block_textures).
//   3. faces, per (axis, slice, direction) task, each a 16x16 mask:
//      - visibility, bit-parallel: one lane per x-row of blocks has their face classes as bit planes (made
//        while the row is staged), so BlockTexture::Show is a few logic operations per row and axis (texture
//        codes are compared only for transparent against transparent);
//      - face words: visible faces are numbered densely in the reference's scan order and one lane per
//        face evaluates light4_init; the face word is Light4 plus texture code and pass;
//      - link masks: each face is compared with its right and lower neighbours, giving the
//        equal-to-right, equal-to-below and transparent-pass masks.
//   4. greedy merge: one lane per task replays the reference's merge row by row on the bit masks:
//      the quads starting in a row are the row's uncovered visible runs split where the face word
//      changes; each extends downward while every column of it continues (equal and uncovered).
//   5. ballots over blocks of 64 faces and a scan of the blocks' counts give every quad its index in its
//      pass; one atomic per chunk and list allocates its output range; one lane per face that starts a quad
//      writes it as packed BlockVertex words and u16 indices (custom meshes: one lane per vertex), with the
//      reference's 65,532-vertex mesh split, per-mesh AABBs and mesh order.
// All arithmetic is integer. References are to client/include/client/BlockMeshAlgo.hpp unless noted.
#include <hip/hip_runtime.h>

#include "hcm_device.h"

namespace hcm {

constexpr int kHalo = 18;
constexpr int kHaloVox = kHalo * kHalo * kHalo;
constexpr int kHaloRows = kHalo * kHalo;
// A task is the 16 x 16 faces of one axis, layer of owning blocks and direction, in the reference's order
// (axis, then slice, then direction): t = 32 axis + 2 layer + (1 for the + faces), the - faces of layer l
// lying in slice l and its + faces in slice l + 1. (The reference's 3 x 17 x 2 also scans the + faces of
// slice 0 and the - faces of slice 16, which the chunk owns none of.)
constexpr int kTasks = 96;
__host__ __device__ constexpr int task_axis(int t) { return t >> 5; }
__host__ __device__ constexpr int task_layer(int t) { return (t >> 1) & 15; }
__host__ __device__ constexpr int task_plus(int t) { return t & 1; }
constexpr int kMaskRows = kTasks * 16;
constexpr int kUnits = kMaskRows / 4; // a unit is four mask rows, 64 faces
constexpr uint32_t kSplitQuads = 16383u; // a BlockMesh holds at most 65,532 vertices (:273-279, :397-403)
constexpr int kMaxMeshPerPass = 8;

// Halo layout: x fastest, then z, then y -- the chunk-local order x + 16 * (z + 16 * y) with a 1-voxel rim.
constexpr int kSX = 1, kSZ = kHalo, kSY = kHalo * kHalo;
__host__ __device__ constexpr int axis_stride(int a) { return a == 0 ? kSX : (a == 1 ? kSY : kSZ); }
// Mask axes per slice axis (BlockAlgo.hpp:70-81 with the YZX swizzle): x -> (U=y, V=z), y -> (U=z, V=x),
// z -> (U=y, V=x).

// The light4_init cell pattern (kLookup3v, :75-108). Vertex k of face F reads, in the plane of the front
// cell, a side cell c0 offset along plane axis Q, the corner cell c1 offset along P and Q, and a side cell
// c2 offset along P; (P, Q) = (y, z) for x faces, (x, z) for y faces, (x, y) for z faces. The signs along
// (P, Q) are (-,-), (+,-), (+,+), (-,+) for faces 0, 3, 4 ("winding a") and (-,-), (-,+), (+,+), (+,-) for
// faces 1, 2, 5. The static_assert below checks this against the reference's literal table.
__host__ __device__ constexpr int plane_p(int F) { return (F >> 1) == 0 ? 1 : 0; }
__host__ __device__ constexpr int plane_q(int F) { return (F >> 1) == 2 ? 1 : 2; }
__host__ __device__ constexpr bool winding_a(int F) { return F == 0 || F == 3 || F == 4; }
__host__ __device__ constexpr int corner_sp(int F, int k) {
	return k == 0 ? -1 : (k == 2 ? 1 : (k == 1 ? (winding_a(F) ? 1 : -1) : (winding_a(F) ? -1 : 1)));
}
__host__ __device__ constexpr int corner_sq(int F, int k) {
	return k == 0 ? -1 : (k == 2 ? 1 : (k == 1 ? (winding_a(F) ? -1 : 1) : (winding_a(F) ? 1 : -1)));
}
__host__ __device__ constexpr int normal_sign(int F) { return (F & 1) ? -1 : 1; }
__host__ __device__ constexpr int corner_comp(int F, int k, int b, int axis) {
	return (axis == (F >> 1) ? normal_sign(F) : 0) + (axis == plane_p(F) && b >= 1 ? corner_sp(F, k) : 0) +
	       (axis == plane_q(F) && b <= 1 ? corner_sq(F, k) : 0);
}

namespace check {
// kLookup3v exactly as the reference lists it (:75-108).
constexpr int8_t kLookup3v[6][4][3][3] = {
    {{{1, 0, -1}, {1, -1, -1}, {1, -1, 0}}, {{1, 0, -1}, {1, 1, -1}, {1, 1, 0}}, {{1, 0, 1}, {1, 1, 1}, {1, 1, 0}},
     {{1, 0, 1}, {1, -1, 1}, {1, -1, 0}}},
    {{{-1, 0, -1}, {-1, -1, -1}, {-1, -1, 0}}, {{-1, 0, 1}, {-1, -1, 1}, {-1, -1, 0}},
     {{-1, 0, 1}, {-1, 1, 1}, {-1, 1, 0}}, {{-1, 0, -1}, {-1, 1, -1}, {-1, 1, 0}}},
    {{{0, 1, -1}, {-1, 1, -1}, {-1, 1, 0}}, {{0, 1, 1}, {-1, 1, 1}, {-1, 1, 0}}, {{0, 1, 1}, {1, 1, 1}, {1, 1, 0}},
     {{0, 1, -1}, {1, 1, -1}, {1, 1, 0}}},
    {{{0, -1, -1}, {-1, -1, -1}, {-1, -1, 0}}, {{0, -1, -1}, {1, -1, -1}, {1, -1, 0}},
     {{0, -1, 1}, {1, -1, 1}, {1, -1, 0}}, {{0, -1, 1}, {-1, -1, 1}, {-1, -1, 0}}},
    {{{0, -1, 1}, {-1, -1, 1}, {-1, 0, 1}}, {{0, -1, 1}, {1, -1, 1}, {1, 0, 1}}, {{0, 1, 1}, {1, 1, 1}, {1, 0, 1}},
     {{0, 1, 1}, {-1, 1, 1}, {-1, 0, 1}}},
    {{{0, -1, -1}, {-1, -1, -1}, {-1, 0, -1}}, {{0, 1, -1}, {-1, 1, -1}, {-1, 0, -1}},
     {{0, 1, -1}, {1, 1, -1}, {1, 0, -1}}, {{0, -1, -1}, {1, -1, -1}, {1, 0, -1}}}};
constexpr bool corner_table_matches() {
	for (int F = 0; F < 6; ++F)
		for (int k = 0; k < 4; ++k)
			for (int b = 0; b < 3; ++b)
				for (int a = 0; a < 3; ++a)
					if (corner_comp(F, k, b, a) != kLookup3v[F][k][b][a])
						return false;
	return true;
}
static_assert(corner_table_matches(), "light4 cell pattern must equal kLookup3v");
} // namespace check

__device__ __forceinline__ int slot27(int x, int y, int z) {
	// CmpXYZ2NeighbourIndex (common/include/common/Position.hpp:138-145): L(-1) = 1, L(0) = 2, L(1) = 0
	int cx = x < 0 ? -1 : (x >= 16 ? 1 : 0), cy = y < 0 ? -1 : (y >= 16 ? 1 : 0), cz = z < 0 ? -1 : (z >= 16 ? 1 : 0);
	return ((cx + 2) % 3) * 9 + ((cy + 2) % 3) * 3 + (cz + 2) % 3;
}
// slot27's y and z terms for the halo row (hy, hz) = (y + 1, z + 1): a halo coordinate h contributes 1 at
// h = 0 (-1), 2 at h = 1 .. 16 (0) and 0 at h = 17 (16), two bits per h in kSlotTerm.
constexpr uint64_t slot_term_table() {
	uint64_t c = 0;
	for (int h = 0; h < 18; ++h)
		c |= uint64_t(h == 0 ? 1 : (h == 17 ? 0 : 2)) << (2 * h);
	return c;
}
constexpr uint64_t kSlotTerm = slot_term_table();
static_assert(kSlotTerm == 0x2aaaaaaa9ull, "slot27 halo-coordinate terms");
__device__ __forceinline__ int slot27_yz(int hy, int hz) {
	return 3 * int((kSlotTerm >> (2 * hy)) & 3u) + int((kSlotTerm >> (2 * hz)) & 3u);
}
__device__ __forceinline__ uint32_t local16(int x, int y, int z) {
	return uint32_t(x & 15) + 16u * (uint32_t(z & 15) + 16u * uint32_t(y & 15));
}
__device__ __forceinline__ int hidx(int x, int y, int z) { return (x + 1) * kSX + (y + 1) * kSY + (z + 1) * kSZ; }

template <int NT> struct Smem {
	// Entries of the face-word stage; the tasks of a chunk with more visible faces are taken in several groups. 1,344
	// keeps the 256-thread workgroup's LDS within three per CU (static_assert below). A 512-thread one has the CU
	// to itself by its registers, and 64 KB to itself in an LDS instruction's offset: 2,496. One random
	// chunk of 7,700 quads took 65.2 us in groups of 1,344, 60.5 so.
	static constexpr int kListCap = NT >= 512 ? 2496 : 1344;
	static_assert(kListCap % 64 == 0 && kListCap / 64 <= 64, "whole blocks of faces, one lane each");
	// A group but the last holds more than kListCap - 256 faces (a task has at most 256), of 24,576 at most.
	static constexpr int kMaxGroups = kTasks * 256 / (kListCap - 255) + 2;
	uint32_t vox[kHaloVox];
	union {
		struct {
			// a mask row of 16 faces per task and row, row 16 t + u: visible faces; equal-to-right faces, then
			// the faces where a quad starts; equal-to-below faces, then the uncovered visible ones
			alignas(16) uint16_t ne[kMaskRows];
			alignas(16) uint16_t eh[kMaskRows];
			alignas(16) uint16_t ev[kMaskRows];
			union {
				uint2 key[kListCap]; // face words of the current group of tasks, in dense order
				struct {             // until the visibility masks are made: the halo rows' face classes as bit planes
					uint4 planes[kHaloRows];  // of the y faces, then the z faces (row_planes)
					uint32_t vis_x[256], tt_x[256]; // per chunk row: its visible x faces and those to compare
				};
			};
		};
		struct { // while a packed halo is staged (a row per thread): its bytes
			alignas(16) uint16_t blocks[NT >= kHaloRows ? HCM_HALO_BLOCKS : 8];
			alignas(8) uint8_t light[NT >= kHaloRows ? HCM_HALO_LIGHT : 8];
		} halo;
	};
	alignas(16) uint16_t own[kListCap]; // per face of the group: 1 + its unit where one begins, else 0; then its descriptor
	uint16_t upre[kUnits + 2]; // visible faces before each unit (the dense face order; at most 24,576), and in all
	uint32_t bcnt[64];         // per 64 faces of the group: quads that start there, opaque | transparent << 16
	uint2 grp[kMaxGroups];     // per group of tasks: its first task, and the quads of the groups before it
	alignas(16) MeshTables tables;
	uint32_t custom_bits[128]; // in-chunk cells with a custom mesh
	uint32_t aabb[2][kMaxMeshPerPass][6];
	uint32_t events[16][2];
	uint32_t scan_w[NT / 64][4]; // per wavefront: its totals of block_excl_sums
	uint32_t slots[27];
	uint32_t job, flags, n_events;
	uint32_t wave_ref[NT / 64];
	uint32_t pool_base, mesh_base;
	JobClaims claims;
};

constexpr uint32_t kFlagNonUniform = 1u, kFlagCustom = 2u, kFlagFlow = 4u;
// kFlagMixed: some halo voxel is not an opaque cube (opaque class on all six faces, no custom or flow
// mesh); kFlagInnerFaces: some chunk voxel has a non-empty face class or a custom or flow mesh. A chunk
// without either has no visible face: BlockTexture::Show never shows an empty face, nor an opaque face
// against an opaque one (texture/include/texture/BlockTexture.hpp:68-76).
constexpr uint32_t kFlagMixed = 8u, kFlagInnerFaces = 16u;
constexpr uint32_t kVoxShape = 0xfff00000u | kTmplMesh | kTmplFlow; // the face classes and the mesh and flow bits
constexpr uint32_t kVoxOpaqueCube = 0x555u << kVoxClassShift; // opaque on all six faces

// ------------------------------------------------------------------------------------------------
// small helpers
// ------------------------------------------------------------------------------------------------
__device__ __forceinline__ uint32_t vox_pid(uint32_t vox) { return (vox >> kVoxPidShift) & kVoxPidMask; }

template <int NT> __device__ __forceinline__ uint32_t row_code(const Smem<NT> &s, uint32_t pid, int face) {
	const uint2 r = s.tables.rows[pid];
	const uint32_t w = face < 4 ? r.x : r.y;
	return (w >> (8 * (face & 3))) & 0xffu;
}

// Texture row of a block value: from LDS for most ids, from the full table for meta-dependent ones.
template <int NT> __device__ __forceinline__ uint32_t block_pid(const MeshParams &p, const Smem<NT> &s, uint32_t b) {
	const uint2 q = s.tables.tmpl_id[b & 0xffu];
	return q.x & kTmplMeta ? p.reg->pid_of[b] : vox_pid(q.y);
}

// AO of a light4_init vertex (:126-130) by side, corner and side cell direct-pass bits and the front cell's:
// two bits per index d0 | d1 << 1 | d2 << 2 | pass3 << 3, 0 when both side cells or the corner and front
// cells block, else 3 minus the number of blocking cells.
constexpr uint32_t ao_table() {
	uint32_t t = 0;
	for (uint32_t i = 0; i < 16; ++i) {
		const int d0 = i & 1, d1 = (i >> 1) & 1, d2 = (i >> 2) & 1, p = (i >> 3) & 1;
		const int a = 3 - !d0 - !d1 - !d2 - !p;
		t |= ((!d0 && !d2) || (!d1 && !p) || a < 0 ? 0u : uint32_t(a)) << (2 * i);
	}
	return t;
}
constexpr uint32_t kAoTable = ao_table();
static_assert(kAoTable == 0xe9849040u, "AO table");
constexpr uint32_t rotate_left(uint32_t v, int n) { return n ? v << n | v >> (32 - n) : v; }

// A cell's word in a light4_init sum when it passes indirect light (:132-161). Voxel words have no light where their
// block does not pass it, so that words are added as they are, unless the registry has such a block in front of
// visible faces (kRaw), whose light counts there.
template <bool kRaw> __device__ __forceinline__ uint32_t lpass(uint32_t c) {
	return kRaw ? c & (uint32_t(int32_t(c << (31 - kVoxIndirectBit)) >> 31) | ~kVoxLight) : c;
}

// Sum of one vertex of light4_init (:114-162), without branches, from its side cells a and b, corner cell c and f, the
// sum of the front cell and a: the corner counts when a side cell passes indirect light.
__device__ __forceinline__ uint32_t light_sum(uint32_t a, uint32_t c, uint32_t b, uint32_t f) {
	return f + b + (c & uint32_t(int32_t((a | b) << (31 - kVoxIndirectBit)) >> 31));
}

// light4_init (:48-163) for the face whose front cell is at byte f of vox. P and Q: the byte strides of its plane's axes
// in the order of its winding, so that its vertices 0 to 3 have the corner cells (-,-), (+,-), (+,+) and (-,+) and the
// side cells along each axis. Returns the packed Light4, a vertex in 14 bits as a vertex word holds it from
// bit 16 on: vertex 0 | vertex 1 << 14 in x, vertex 2 | vertex 3 << 14 in y.
//
// Dense chunks issue most of their instructions here. Sums of whole words (no masks), averages by LDS look-ups at the
// sums' fields and AO by a table rotated by the cells' direct-pass bits, which each word has at the four places its cell
// may take: the loop around it is 174 VALU instructions per 64 faces, where masked sums with reciprocals made it 247.
// 2,304 chunks of random blocks took 724 us so, now 659; 768 plant chunks 30.7 and 30.1.
template <bool kRaw, int NT> __device__ __forceinline__ uint2 light4(const Smem<NT> &s, int f, int P, int Q) {
	const char *vox = reinterpret_cast<const char *>(s.vox);
	const auto cell = [vox](int at) { return *reinterpret_cast<const uint32_t *>(vox + at); };
	const int fm = f - P, fp = f + P;
	const uint32_t F = cell(f);
	const uint32_t qm = lpass<kRaw>(cell(f - Q)), qp = lpass<kRaw>(cell(f + Q));
	const uint32_t pm = lpass<kRaw>(cell(fm)), pp = lpass<kRaw>(cell(fp));
	const uint32_t c0 = lpass<kRaw>(cell(fm - Q)), c1 = lpass<kRaw>(cell(fp - Q));
	const uint32_t c2 = lpass<kRaw>(cell(fp + Q)), c3 = lpass<kRaw>(cell(fm + Q));
	const uint32_t front = F & ~kVoxIndirect; // counted always, as the 1 of count - 1
	const uint32_t fqm = front + qm, fqp = front + qp;
	const uint32_t s0 = light_sum(qm, c0, pm, fqm), s1 = light_sum(qm, c1, pp, fqm);
	const uint32_t s2 = light_sum(qp, c2, pp, fqp), s3 = light_sum(qp, c3, pm, fqp);
	const auto vertex = [&s](uint32_t sum) {
		return uint32_t(s.tables.sun_of[(sum >> kVoxSunBit) & 0xffu]) | uint32_t(s.tables.torch_of[(sum >> (kVoxTorchBit - 2)) & 0xffu]) << 8;
	};
	uint32_t x = vertex(s0) | vertex(s1) << 14, y = vertex(s2) | vertex(s3) << 14;
	// AO: bits 1 to 4 of a word, of which bit 0 is zero, rotate the table by the two bits of each cell's flag
	const auto direct = [](uint32_t bit, uint32_t a, uint32_t b) { return (a & bit) | (b & ~bit); };
	const uint32_t dqm = direct(2u, qm, F), dqp = direct(2u, qp, F);
	const auto ao = [&](uint32_t dq, uint32_t c, uint32_t b, uint32_t table) {
		return __builtin_amdgcn_alignbit(table, table, direct(8u, b, direct(4u, c, dq)));
	};
	constexpr uint32_t table1 = rotate_left(kAoTable, 14);
	x = direct(3u << 14, ao(dqm, c1, pp, table1), direct(3u, ao(dqm, c0, pm, kAoTable), x));
	y = direct(3u << 14, ao(dqp, c3, pm, table1), direct(3u, ao(dqp, c2, pp, kAoTable), y));
	return make_uint2(x, y);
}

// The same for face `face` of the block at halo index self. Winding a (faces 0, 3 and 4) has the plane axes in order.
template <bool kRaw, int NT> __device__ __forceinline__ uint2 light4_of(const Smem<NT> &s, int face, int self) {
	const int a = face >> 1;
	const int sn = a == 0 ? kSX : (a == 1 ? kSY : kSZ);
	const int sp = a == 0 ? kSY : kSX, sq = a == 2 ? kSY : kSZ;
	const bool wa = face == 0 || face == 3 || face == 4;
	return light4<kRaw>(s, 4 * (self + ((face & 1) ? -sn : sn)), 4 * (wa ? sp : sq), 4 * (wa ? sq : sp));
}

__device__ __forceinline__ uint32_t l4_at(uint2 l, int k, int bit) { return (k < 2 ? l.x : l.y) >> (14 * (k & 1) + bit); }
__device__ __forceinline__ uint32_t l4_ao(uint2 l, int k) { return l4_at(l, k, 0) & 3u; }
__device__ __forceinline__ uint32_t l4_sun(uint2 l, int k) { return l4_at(l, k, 2) & 63u; }
__device__ __forceinline__ uint32_t l4_torch(uint2 l, int k) { return l4_at(l, k, 8) & 63u; }

// Light4::GetFlip (:38-43): sunlight and AO only.
__device__ __forceinline__ bool l4_flip(uint2 l) {
	const uint2 more = make_uint2(l.x + (4u | 4u << 14), l.y + (4u | 4u << 14)); // sunlight + 1 (at most 61)
	const auto product = [&](int k) { return l4_ao(l, k) * l4_sun(more, k) + l4_sun(more, k); };
	return abs(int(product(0) - product(2))) < abs(int(product(1) - product(3)));
}

__device__ __forceinline__ uint64_t ballot64(bool b) { return __ballot(b); }

// Minima of the 16-bit halves of two words.
__device__ __forceinline__ uint32_t min_halves(uint32_t a, uint32_t b) {
	typedef uint16_t halves __attribute__((vector_size(4)));
	const halves x = __builtin_bit_cast(halves, a), y = __builtin_bit_cast(halves, b);
	return __builtin_bit_cast(uint32_t, x < y ? x : y);
}

// The minima over the wavefront with DPP lane moves (no LDS): swaps within quads, the half-row
// and row mirrors leave every lane of a 16-lane row with the row's result, then the row broadcasts of
// lanes 15 and 31 fold the rows into lane 63. Lanes a move does not write keep the identity.
__device__ __forceinline__ uint32_t wave_min_halves(uint32_t v) {
	v = min_halves(v, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0xb1, 0xf, 0xf, false));  // quad_perm 1,0,3,2
	v = min_halves(v, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0x4e, 0xf, 0xf, false));  // quad_perm 2,3,0,1
	v = min_halves(v, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0x141, 0xf, 0xf, false)); // row_half_mirror
	v = min_halves(v, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0x140, 0xf, 0xf, false)); // row_mirror
	v = min_halves(v, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0x142, 0xa, 0xf, false)); // row_bcast:15
	v = min_halves(v, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, 0x143, 0xc, 0xf, false)); // row_bcast:31
	return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// ------------------------------------------------------------------------------------------------
// block-wide exclusive scan of three 32-bit counters (every thread reads s.scan_w after the barrier; the
// next write to it is a later chunk's, after several more barriers)
// ------------------------------------------------------------------------------------------------
// Inclusive prefix sum over the wavefront by DPP: shifts by 1, 2, 4 and 8 lanes within each row of 16,
// then the last lane of row 0 into row 1 (and of row 2 into row 3), then lane 31 into rows 2 and 3.
__device__ __forceinline__ uint32_t wave_incl_sum(uint32_t v) {
	v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, true); // row_shr:1
	v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, true); // row_shr:2
	v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, true); // row_shr:4
	v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, true); // row_shr:8
	v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, true); // row_bcast:15
	v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, true); // row_bcast:31
	return v;
}

// Exclusive prefix sums over the workgroup of three 32-bit values per thread, and their totals, with one
// barrier.
template <int NT>
__device__ __forceinline__ void block_excl_sums(Smem<NT> &s, uint32_t v[3], uint32_t tot[3]) {
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	uint32_t inc[3];
#pragma unroll
	for (int i = 0; i < 3; ++i)
		inc[i] = wave_incl_sum(v[i]);
	if (lane == 63) {
#pragma unroll
		for (int i = 0; i < 3; ++i)
			s.scan_w[wave][i] = inc[i];
	}
	__syncthreads();
#pragma unroll
	for (int i = 0; i < 3; ++i) {
		uint32_t before = 0, all = 0;
#pragma unroll
		for (int w = 0; w < NT / 64; ++w) {
			const uint32_t x = s.scan_w[w][i];
			before += w < wave ? x : 0u;
			all += x;
		}
		v[i] = before + inc[i] - v[i];
		tot[i] = all;
	}
}

// ------------------------------------------------------------------------------------------------
// liquid flow (block/block/public/Liquid.hpp:151-302)
// ------------------------------------------------------------------------------------------------
struct Flow {
	uint32_t h;        // corner heights h0 | h1 << 8 | h2 << 16 | h3 << 24 (0 1 / 2 3 over x, z)
	uint32_t liq_side; // bit per neighbour 1, 3, 4, 6 (back, left, right, front) that is a liquid
};

__device__ __forceinline__ uint32_t flow_h(const Flow &f, int i) { return (f.h >> (8 * i)) & 0xffu; }

// Where a job's blocks are in global memory: the store's slots, or its packed halo.
struct JobBlocks {
	const uint16_t *store;  // p.blocks
	const uint32_t *slots;  // s.slots
	const uint16_t *halo;   // null: the store
	__device__ __forceinline__ uint16_t at(int x, int y, int z) const {
		if (halo)
			return halo[(x + 2) + 20 * ((z + 2) + 20 * (y + 1))];
		return store[(size_t)slots[slot27(x, y, z)] * HCM_CHUNK_VOXELS + local16(x, y, z)];
	}
};

// get_nei_height (:164-169) as a signed integer: the reference returns it as int8_t, so a flow level's
// uint8_t height max(meta * 2, 1) wraps to [-128, 127].
__device__ __forceinline__ int flow_nei_height(uint32_t b, uint32_t src_id, uint32_t flow_id) {
	const uint32_t id = b & 0xffu, meta = b >> 8;
	if (id == src_id)
		return 16;
	if (id == flow_id) {
		const uint32_t h = (meta * 2u > 1u ? meta * 2u : 1u) & 0xffu;
		return h >= 128u ? int(h) - 256 : int(h);
	}
	return id != 0 ? -1 : 0; // WaterTrait::IsObstacle: id != kAir (block/block/public/Water.hpp:13)
}

// get_vh (:181-186): the signed maximum as uint8_t, or 0 when three of the four are empty (height 0)
__device__ __forceinline__ uint32_t flow_vh(int nb, int a, int b, int c) {
	const int m = max(max(nb, a), max(b, c));
	const uint32_t mx = uint32_t(m) & 0xffu;
	const int zeros = int(nb == 0) + int(a == 0) + int(b == 0) + int(c == 0);
	return (mx != 16u && zeros >= 3) ? 0u : mx;
}

__device__ __forceinline__ Flow flow_heights(const MeshParams &p, const JobBlocks &blocks, int x, int y, int z,
                                          uint32_t nb_height) {
	const uint32_t src = p.reg->src_id, fid = p.reg->flow_id;
	// neighbours (:291-300): 0 (-1,-1) 1 (0,-1) 2 (1,-1) 3 (-1,0) 4 (1,0) 5 (-1,1) 6 (0,1) 7 (1,1) in (x, z)
	const uint32_t b0 = blocks.at(x - 1, y, z - 1), b1 = blocks.at(x, y, z - 1);
	const uint32_t b2 = blocks.at(x + 1, y, z - 1), b3 = blocks.at(x - 1, y, z);
	const uint32_t b4 = blocks.at(x + 1, y, z), b5 = blocks.at(x - 1, y, z + 1);
	const uint32_t b6 = blocks.at(x, y, z + 1), b7 = blocks.at(x + 1, y, z + 1);
	const int n0 = flow_nei_height(b0, src, fid), n1 = flow_nei_height(b1, src, fid);
	const int n2 = flow_nei_height(b2, src, fid), n3 = flow_nei_height(b3, src, fid);
	const int n4 = flow_nei_height(b4, src, fid), n5 = flow_nei_height(b5, src, fid);
	const int n6 = flow_nei_height(b6, src, fid), n7 = flow_nei_height(b7, src, fid);
	const int nb = int(nb_height);
	Flow f;
	f.h = flow_vh(nb, n0, n1, n3) | flow_vh(nb, n1, n2, n4) << 8 | flow_vh(nb, n3, n5, n6) << 16 |
	      flow_vh(nb, n4, n6, n7) << 24;
	auto liq = [&](uint32_t b) { return ((b & 0xffu) == src || (b & 0xffu) == fid) ? 1u : 0u; };
	f.liq_side = liq(b1) | liq(b3) << 1 | liq(b4) << 2 | liq(b6) << 3;
	return f;
}

__device__ __forceinline__ bool flow_all_full(const Flow &f) { return f.h == 0x10101010u; }

// Emitted faces of a flow cell, in order: top, left, right, back, front (:193-274). Returns a 5-bit set.
__device__ __forceinline__ uint32_t flow_face_set(const Flow &f) {
	if (flow_all_full(f))
		return 0;
	const uint32_t h0 = flow_h(f, 0), h1 = flow_h(f, 1), h2 = flow_h(f, 2), h3 = flow_h(f, 3);
	const bool lf = h0 == 16 && h2 == 16, le = h0 == 0 && h2 == 0;
	const bool rf = h1 == 16 && h3 == 16, re = h1 == 0 && h3 == 0;
	const bool ff = h2 == 16 && h3 == 16, fe = h2 == 0 && h3 == 0;
	const bool bf = h0 == 16 && h1 == 16, be = h0 == 0 && h1 == 0;
	uint32_t set = 1u;
	if (!lf && !le && !(f.liq_side & 2u))
		set |= 2u;
	if (!rf && !re && !(f.liq_side & 4u))
		set |= 4u;
	if (!bf && !be && !(f.liq_side & 1u))
		set |= 8u;
	if (!ff && !fe && !(f.liq_side & 8u))
		set |= 16u;
	return set;
}

// Dynamic texture pattern of a flow cell: 16 = all six faces liquid; otherwise bits right, left, front,
// back full (:193-197, :275-280).
__device__ __forceinline__ uint32_t flow_pattern(const Flow &f) {
	if (flow_all_full(f))
		return 16u;
	const uint32_t h0 = flow_h(f, 0), h1 = flow_h(f, 1), h2 = flow_h(f, 2), h3 = flow_h(f, 3);
	return uint32_t(h1 == 16 && h3 == 16) | (uint32_t(h0 == 16 && h2 == 16) << 1) |
	       (uint32_t(h2 == 16 && h3 == 16) << 2) | (uint32_t(h0 == 16 && h1 == 16) << 3);
}

__device__ __forceinline__ hcm_mesh_vertex fv(uint32_t x, uint32_t y, uint32_t z) {
	hcm_mesh_vertex v;
	v.x = uint8_t(x), v.y = uint8_t(y), v.z = uint8_t(z), v.ao = 4;
	return v;
}

// The kind-th face (0 top, 1 left, 2 right, 3 back, 4 front) of a flow cell (:198-274).
__device__ hcm_mesh_face flow_face(const Flow &f, int kind, uint16_t tex) {
	const uint32_t h0 = flow_h(f, 0), h1 = flow_h(f, 1), h2 = flow_h(f, 2), h3 = flow_h(f, 3);
	hcm_mesh_face m;
	m.pad = 0, m.pad2 = 0, m.texture = tex;
	switch (kind) {
	case 0:
		m.axis = 1, m.light_face = 2;
		m.v[0] = fv(0, h0, 0), m.v[1] = fv(0, h2, 16), m.v[2] = fv(16, h3, 16), m.v[3] = fv(16, h1, 0);
		break;
	case 1:
		m.axis = 0, m.light_face = 1;
		m.v[0] = fv(0, h0, 0), m.v[1] = fv(0, 0, 0), m.v[2] = fv(0, 0, 16), m.v[3] = fv(0, h2, 16);
		break;
	case 2:
		m.axis = 0, m.light_face = 0;
		m.v[0] = fv(16, 0, 0), m.v[1] = fv(16, h1, 0), m.v[2] = fv(16, h3, 16), m.v[3] = fv(16, 0, 16);
		break;
	case 3:
		m.axis = 2, m.light_face = 5;
		m.v[0] = fv(0, 0, 0), m.v[1] = fv(0, h0, 0), m.v[2] = fv(16, h1, 0), m.v[3] = fv(16, 0, 0);
		break;
	default:
		m.axis = 2, m.light_face = 4;
		m.v[0] = fv(0, h2, 16), m.v[1] = fv(0, 0, 16), m.v[2] = fv(16, 0, 16), m.v[3] = fv(16, h3, 16);
		break;
	}
	m.render_face = m.light_face;
	return m;
}

// ------------------------------------------------------------------------------------------------
// custom meshes (:198-306)
// ------------------------------------------------------------------------------------------------
struct CustomCell {
	uint32_t count; // faces emitted
	uint32_t trans; // bit j: face j goes to the transparent pass
	uint32_t mesh;  // registry mesh index
	uint32_t flow;  // 1 if liquid flow
	Flow fl;
	uint32_t flow_set; // liquid flow: emitted face kinds
};

template <int NT>
__device__ __forceinline__ CustomCell custom_cell(const MeshParams &p, const Smem<NT> &s, const JobBlocks &blocks, int cell) {
	const int x = cell & 15, z = (cell >> 4) & 15, y = cell >> 8;
	// the voxel word has the block's row but for flow cells, whose words took a row of face textures
	uint32_t pid = vox_pid(s.vox[hidx(x, y, z)]);
	if (pid >= p.reg->flow_pid_base)
		pid = block_pid(p, s, blocks.at(x, y, z));
	CustomCell c;
	c.mesh = s.tables.rows[pid].y >> 24;
	c.flow = (s.tables.pid_vox[pid].x & kTmplFlow) ? 1u : 0u;
	c.trans = 0;
	c.flow_set = 0;
	c.fl.h = 0, c.fl.liq_side = 0;
	const uint32_t sum = p.reg->mesh_sums[c.mesh]; // (one load: the faces' textures and flags would be two per face)
	if (c.flow) {
		c.fl = flow_heights(p, blocks, x, y, z, p.reg->meshes[c.mesh].flow_height);
		c.flow_set = flow_face_set(c.fl);
		c.count = __popc(c.flow_set);
		if (p.reg->flow_trans)
			c.trans = (1u << c.count) - 1u;
	} else {
		c.count = sum & 0x1fu;
		c.trans = sum >> 16;
	}
	return c;
}

// The custom-mesh cells among this thread's 4096 / NT.
template <int NT> __device__ __forceinline__ uint32_t custom_cells(const Smem<NT> &s) {
	constexpr int n = HCM_CHUNK_VOXELS / NT;
	static_assert(n <= 32 && 32 % n == 0, "a thread's cells in one word");
	const uint32_t at = threadIdx.x * n;
	return (s.custom_bits[at >> 5] >> (at & 31)) & uint32_t((1ull << n) - 1ull);
}

__device__ __forceinline__ hcm_mesh_face custom_face(const MeshParams &p, const CustomCell &c, int j) {
	if (!c.flow)
		return p.reg->meshes[c.mesh].faces[j];
	uint32_t set = c.flow_set;
	for (int i = 0; i < j; ++i)
		set &= set - 1u;
	return flow_face(c.fl, __ffs(set) - 1, uint16_t(p.reg->flow_tex));
}

// ------------------------------------------------------------------------------------------------
// writing one quad
// ------------------------------------------------------------------------------------------------
__device__ __forceinline__ void put_indices(uint32_t *ip, uint32_t base, bool flip) {
	// index patterns: flip (0,1,2, 0,2,3) (:440-446) -- also the custom-mesh pattern (:295-301) --
	// and no flip (1,2,3, 0,1,3) (:453-459)
	const uint32_t two = base | base << 16; // at most 65,532 each: no carry
	ip[0] = two + (flip ? 0u | 1u << 16 : 1u | 2u << 16);
	ip[1] = two + (flip ? 2u | 0u << 16 : 3u | 0u << 16);
	ip[2] = two + (flip ? 2u | 3u << 16 : 1u | 3u << 16);
}

// BlockVertex word 1 (client/include/client/BlockVertex.hpp:13-14)
__device__ __forceinline__ uint32_t vword1(uint16_t tex, uint32_t face, uint32_t ao, uint32_t sun, uint32_t torch) {
	return ((uint32_t)(tex & 0x1fffu) - 1u) | ((uint32_t)(tex >> 13) << 10) | (face << 13) | (ao << 16) | (sun << 18) |
	       (torch << 24);
}

// The box of a pass, over words of vertices (x, y, z in 10 bits each): the lowest x, y and z and the lowest complements
// of the highest, in the upper bits of six 16-bit halves, whose lower bits are of no account; all of them are minima,
// of all ones where there is none.
struct Box {
	uint32_t lo_xy, hi_xy, z;
};
__device__ __forceinline__ uint32_t low_high(uint32_t low, uint32_t high) { return (low & 0xffffu) | (high & 0xffff0000u); }
// The box of the vertex words lo and hi.
__device__ __forceinline__ Box word_box(uint32_t lo, uint32_t hi) {
	return {low_high(lo << 6, lo << 12), low_high(~hi << 6, ~hi << 12), low_high(lo >> 14, ~hi << 2)};
}
__device__ __forceinline__ void box_min(Box &b, const Box &a, uint32_t m) {
	b.lo_xy = min_halves(b.lo_xy, a.lo_xy | m), b.hi_xy = min_halves(b.hi_xy, a.hi_xy | m), b.z = min_halves(b.z, a.z | m);
}
__device__ __forceinline__ Box wave_box(const Box &b) {
	return {wave_min_halves(b.lo_xy), wave_min_halves(b.hi_xy), wave_min_halves(b.z)};
}

template <int NT> __device__ __forceinline__ void aabb_merge(Smem<NT> &s, int pass, int k, const Box &b) {
	uint32_t *a = s.aabb[pass][k];
	atomicMin(&a[0], (b.lo_xy >> 6) & 0x3ffu);
	atomicMin(&a[1], b.lo_xy >> 22);
	atomicMin(&a[2], (b.z >> 6) & 0x3ffu);
	atomicMax(&a[3], ~(b.hi_xy >> 6) & 0x3ffu);
	atomicMax(&a[4], ~b.hi_xy >> 22);
	atomicMax(&a[5], ~b.z >> 22);
}

// Regular quad at the face at desc (task, row u, column v0), width w along V, height h along U (:357-460), with the
// face word of its origin face (Light4 and texture code), to quad i of the chunk, whose pool range starts at verts
// and idx. Returns its box.
template <int NT>
__device__ __forceinline__ Box emit_quad(const Smem<NT> &s, uint32_t desc, uint32_t w, uint32_t h, uint2 word, uint4 *verts,
                                         uint32_t *idx, uint32_t i, uint32_t vbase) {
	const int t = (desc >> 8) & 127, A = task_axis(t), plus = task_plus(t);
	const uint32_t u = (desc >> 4) & 15, v0 = desc & 15;
	// a vertex word has x, y and z (1/16 units, at most 256) in 10-bit fields: the origin's word and the packed
	// vectors along U and V, with no carry between fields
	const uint32_t at_u = A == 1 ? 24 : 14, at_v = A == 0 ? 24 : 4, at_a = 42 - at_u - at_v;
	const uint32_t base = uint32_t(task_layer(t) + plus) << at_a | u << at_u | v0 << at_v | uint32_t(A) << 30;
	const uint32_t pu = h << at_u, pv = w << at_v;
	// quad vectors (:383-390): (U+1)%3 == V holds for the x and y axes
	const bool height_first = (plus == 0) != (A != 2);
	const uint32_t second = base + (height_first ? pu : pv), opposite = base + pu + pv, fourth = base + (height_first ? pv : pu);
	// BlockVertex word 1 (client/include/client/BlockVertex.hpp:13-14): texture, face, and the vertex's light
	const uint32_t code = (word.x >> 28) | ((word.y >> 24) & 0x70u);
	const uint32_t common = (s.tables.codes[code] & kCodeVertex) | uint32_t(2 * A + (plus ^ 1)) << 13;
	constexpr uint32_t kLight = 0x3fff0000u;
	uint4 *vp = verts + 2 * (size_t)i;
	vp[0] = make_uint4(base, common | (word.x << 16 & kLight), second, common | (word.x << 2 & kLight));
	vp[1] = make_uint4(opposite, common | (word.y << 16 & kLight), fourth, common | (word.y << 2 & kLight));
	put_indices(idx + 3 * (size_t)i, vbase, l4_flip(word));
	return word_box(base, opposite);
}

// light4_interpolate (:165-196): trilinear in 1/16 steps, rounded up, for two values of at most 63 in the
// half-words of each corner word. The corners' plane (du, dv) stays within 16 bits (63 * 256); the last step, between
// the planes (dw), is in 32.
typedef uint16_t halves __attribute__((vector_size(4)));
__device__ __forceinline__ halves lerp16(halves a, halves b, uint32_t t) {
	const halves s = {uint16_t(16u - t), uint16_t(16u - t)}, u = {uint16_t(t), uint16_t(t)};
	return a * s + b * u;
}
__device__ __forceinline__ halves as_halves(uint32_t v) {
	const halves h = {uint16_t(v), uint16_t(v >> 16)};
	return h;
}
struct Interp {
	uint32_t first, second;
};
__device__ __forceinline__ uint32_t interp32(const uint32_t l[4], const uint32_t h[4], int shift, uint32_t du, uint32_t dv,
                                             uint32_t dw) {
	const auto v = [shift](uint32_t w) { return (w >> shift) & 0xffffu; };
	const auto lerp = [](uint32_t a, uint32_t b, uint32_t t) { return a * (16u - t) + b * t; };
	const uint32_t lo = lerp(lerp(v(l[0]), v(l[1]), du), lerp(v(l[3]), v(l[2]), du), dv);
	const uint32_t hi = lerp(lerp(v(h[0]), v(h[1]), du), lerp(v(h[3]), v(h[2]), du), dv);
	const uint32_t sum = lerp(lo, hi, dw);
	return sum / 4096u + (sum % 4096u ? 1u : 0u);
}
__device__ __forceinline__ Interp interp(const uint32_t l[4], const uint32_t h[4], uint32_t du, uint32_t dv, uint32_t dw) {
	if (du > 16u || dv > 16u) // a vertex outside its block: in 32 bits throughout, which wrap as the reference's do
		return {interp32(l, h, 0, du, dv, dw), interp32(l, h, 16, du, dv, dw)};
	const halves lo = lerp16(lerp16(as_halves(l[0]), as_halves(l[1]), du), lerp16(as_halves(l[3]), as_halves(l[2]), du), dv);
	const halves hi = lerp16(lerp16(as_halves(h[0]), as_halves(h[1]), du), lerp16(as_halves(h[3]), as_halves(h[2]), du), dv);
	const uint32_t a = uint32_t(lo[0]) * (16u - dw) + uint32_t(hi[0]) * dw, b = uint32_t(lo[1]) * (16u - dw) + uint32_t(hi[1]) * dw;
	return {(a + 4095u) >> 12, (b + 4095u) >> 12};
}

// Vertex k of custom quad desc (cell | face << 12), to quad `slot` of the pool. Returns its word, which is its box. A chunk has few custom quads, so their time
// is the length of one's chain of loads and operations: four lanes share a quad's vertices, the face counts and passes
// come from one word per mesh, and light is interpolated two values at a time. 768 chunks of terrain with plants
// took 47.7 us with a lane per quad and two loads per face, 31.9 so; one such chunk from host memory 41.4 and 33.3.
template <bool kRaw, int NT>
__device__ __forceinline__ uint32_t emit_custom(const MeshParams &p, Smem<NT> &s, const JobBlocks &blocks, uint32_t desc,
                                                uint32_t k, uint32_t slot, uint32_t vbase) {
	const int cell = desc & 4095, j = (desc >> 12) & 15;
	const int x = cell & 15, z = (cell >> 4) & 15, y = cell >> 8;
	const CustomCell c = custom_cell(p, s, blocks, cell);
	const hcm_mesh_face f = custom_face(p, c, j);
	const int lf = f.light_face, la = lf >> 1, sg = (lf & 1) ? -1 : 1;
	const int pos = hidx(x, y, z);
	// low: the face of the cell behind; high: this cell's own face if the next cell passes light (:259-267)
	const uint2 lo4 = light4_of<kRaw>(s, lf, pos - sg * axis_stride(la));
	const uint2 hi4 = (s.vox[pos + sg * axis_stride(la)] & kVoxIndirect) ? light4_of<kRaw>(s, lf, pos) : lo4;
	int ua = (la + 1) % 3, va = (la + 2) % 3;
	if (lf & 1) {
		const int tmp = ua;
		ua = va, va = tmp;
	}
	const hcm_mesh_vertex v = k == 0 ? f.v[0] : (k == 1 ? f.v[1] : (k == 2 ? f.v[2] : f.v[3]));
	const uint32_t vx = v.x, vy = v.y, vz = v.z;
	auto pick = [&](int a) { return a == 0 ? vx : (a == 1 ? vy : vz); };
	const uint32_t at = ((uint32_t(x) << 4) + vx) | ((uint32_t(y) << 4) + vy) << 10 | ((uint32_t(z) << 4) + vz) << 20;
	const uint32_t du = pick(ua), dv = pick(va);
	uint32_t dw = min(pick(la), 16u);
	if (lf & 1)
		dw = 16u - dw;
	uint32_t l[4], h[4];
#pragma unroll
	for (int i = 0; i < 4; ++i)
		l[i] = l4_sun(lo4, i) | l4_torch(lo4, i) << 16, h[i] = l4_sun(hi4, i) | l4_torch(hi4, i) << 16;
	const Interp light = interp(l, h, du, dv, dw);
	uint32_t ao = v.ao;
	if (ao == 4) {
#pragma unroll
		for (int i = 0; i < 4; ++i)
			l[i] = l4_ao(lo4, i), h[i] = l4_ao(hi4, i);
		ao = interp(l, h, du, dv, dw).first & 0xffu;
	}
	p.pool_verts[4 * (size_t)slot + k] =
	    make_uint2(at | (uint32_t(f.axis) << 30), vword1(f.texture, f.render_face, ao, light.first & 0xffu, light.second & 0xffu));
	if (k == 0)
		put_indices(reinterpret_cast<uint32_t *>(p.pool_idx) + 3 * (size_t)slot, vbase, true);
	return at;
}

// ------------------------------------------------------------------------------------------------
// visibility: one lane per x-row of blocks, its faces as bit planes
// ------------------------------------------------------------------------------------------------
// BlockTexture::Show (texture/include/texture/BlockTexture.hpp:68-76) on the 2-bit face classes
// (empty 0, opaque 1, transparent 2, liquid 3):
//   opaque self:      visible unless the other face is opaque,
//   transparent self: visible if the other is empty or liquid, or transparent with another texture,
//   liquid self:      visible if the other is empty.
// A row's 16 blocks are 16 bits, so the rule is a few logic operations for a whole row, and both directions
// of an axis share them: the + direction in the low half-word, the - direction in the high one.
__host__ __device__ constexpr uint32_t show_planes(uint32_t s0, uint32_t s1, uint32_t o0, uint32_t o1) {
	return (s0 & ~s1 & ~(o0 & ~o1)) | (s1 & ~s0 & ~(o0 ^ o1)) | (s0 & s1 & ~(o0 | o1));
}
// Transparent against transparent, which also needs the textures.
__host__ __device__ constexpr uint32_t tt_planes(uint32_t s0, uint32_t s1, uint32_t o0, uint32_t o1) {
	return s1 & ~s0 & o1 & ~o0;
}
namespace check {
constexpr bool show_matches() {
	for (uint32_t self = 0; self < 4; ++self)
		for (uint32_t other = 0; other < 4; ++other) {
			const bool want = self == 1 ? other != 1 : self == 2 ? (other == 0 || other == 3) : self == 3 ? other == 0 : false;
			if ((show_planes(self & 1, self >> 1, other & 1, other >> 1) & 1u) != uint32_t(want) ||
			    (tt_planes(self & 1, self >> 1, other & 1, other >> 1) & 1u) != uint32_t(self == 2 && other == 2))
				return false;
		}
	return true;
}
static_assert(show_matches(), "Show on face classes");
} // namespace check

// Bytes of (hi, lo) by selector: selector byte 0-3 takes that byte of lo, 4-7 of hi, 12 is zero.
__device__ __forceinline__ uint32_t byte_perm(uint32_t hi, uint32_t lo, uint32_t sel) {
	return __builtin_amdgcn_perm(hi, lo, sel);
}

// The class bits of 16 blocks' templates as planes, two per word: p0[a] holds class bit 0 and p1[a] class
// bit 1 of the blocks' + faces along axis a in the low half-word (bit i: block i) and of their - faces in
// the high one. The templates' upper half-words, two to a register, are an 8 x 8 bit matrix per byte;
// three exchange steps transpose all four at once: 62 VALU instructions a row of 16 blocks, where one
// shift-and-or per class bit and block would be 192. The phase is bound by instruction issue: with one lane
// per column of an axis and two ballots per slice the 4,096-chunk cave batch issued 45.5 M instructions in
// 100.8 us, with the planes 39.4 M in 89.0 us.
__device__ __forceinline__ void row_planes(const uint32_t tm[16], uint32_t p0[3], uint32_t p1[3]) {
	static_assert(kVoxClassShift == 20, "class bits 4 .. 15 of the template's upper half-word");
	uint32_t r[8];
#pragma unroll
	for (int i = 0; i < 8; ++i)
		r[i] = byte_perm(tm[i + 8], tm[i], 0x07060302u);
	exchange_bits<4>(r);
	exchange_bits<2>(r);
	exchange_bits<1>(r);
	// r[k]: bit k of every block's four bytes; block i < 8 in bit i of bytes 0 (class bits 0-3 in bits 4-7)
	// and 1 (class bits 4-11), block i + 8 in bit i of bytes 2 and 3
	p0[0] = byte_perm(r[6], r[4], 0x06040200u), p1[0] = byte_perm(r[7], r[5], 0x06040200u);
	p0[1] = byte_perm(r[2], r[0], 0x07050301u), p1[1] = byte_perm(r[3], r[1], 0x07050301u);
	p0[2] = byte_perm(r[6], r[4], 0x07050301u), p1[2] = byte_perm(r[7], r[5], 0x07050301u);
}

// A halo row's planes (first template words tm[0 .. 17] of x = -1 .. 16) to where the rows beside it read them; for a
// row of the chunk also its visible x faces, which need no other row.
template <int NT> __device__ __forceinline__ void put_planes(Smem<NT> &s, int hy, int hz, const uint32_t tm[18]) {
	uint32_t p0[3], p1[3];
	row_planes(tm + 1, p0, p1);
	s.planes[hy * kHalo + hz] = make_uint4(p0[1], p1[1], p0[2], p1[2]);
	if ((unsigned)(hy - 1) < 16u && (unsigned)(hz - 1) < 16u) {
		// + faces meet the - face of the block at x + 1, - faces the + face of the one at x - 1
		constexpr int cp = kVoxClassShift, cm = kVoxClassShift + 2; // the rim blocks' + and - class bits
		const uint32_t o0 = (p0[0] >> 17) | (p0[0] << 17) | ((tm[17] >> (cm - 15)) & 0x8000u) | ((tm[0] >> (cp - 16)) & 0x10000u);
		const uint32_t o1 = (p1[0] >> 17) | (p1[0] << 17) | ((tm[17] >> (cm - 14)) & 0x8000u) | ((tm[0] >> (cp - 15)) & 0x10000u);
		const int row = (hy - 1) * 16 + hz - 1;
		s.vis_x[row] = show_planes(p0[0], p1[0], o0, o1);
		s.tt_x[row] = tt_planes(p0[0], p1[0], o0, o1);
	}
}

// Transparent faces of a row against transparent ones (bits tt, both directions along axis A), which show
// when the two texture codes differ. cell: halo index of the row's first block.
template <int NT> __device__ uint32_t show_textures(const Smem<NT> &s, uint32_t tt, int A, int cell) {
	uint32_t vis = 0;
	while (tt) {
		const uint32_t bit = __ffs(tt) - 1;
		tt &= tt - 1u;
		const int self = cell + int(bit & 15u), other = self + (bit < 16 ? axis_stride(A) : -axis_stride(A));
		const int f = 2 * A + int(bit >> 4);
		if (row_code(s, vox_pid(s.vox[self]), f) != row_code(s, vox_pid(s.vox[other]), f ^ 1))
			vis |= 1u << bit;
	}
	return vis;
}

// One step of a 16 x 16 bit transposition over 16 lanes, for both half-words: bits and lanes whose index
// differs in d change places. m: the half-words' bits without d, complemented in the lanes with d.
__device__ __forceinline__ uint32_t transpose_step(uint32_t v, uint32_t other, uint32_t m, bool has, int d) {
	const uint32_t moved = has ? other >> d : other << d;
	return (v & m) | (moved & ~m);
}

// The tasks' masks from the planes, one lane per row (y, z) of the chunk; every mask row is written. The y
// and z tasks' rows run along x as the planes do; the x tasks' rows run along z, so the 16 rows of a y are
// transposed over 16 lanes first.
template <int NT> __device__ __forceinline__ void visibility_row(Smem<NT> &s, int row) {
	const int y = row >> 4, z = row & 15, h = (y + 1) * kHalo + z + 1, cell = h * kHalo + 1;
	const uint4 p = s.planes[h];
	const uint4 yp = s.planes[h + kHalo], ym = s.planes[h - kHalo], zp = s.planes[h + 1], zm = s.planes[h - 1];
	// the other face of the + direction is the next row's - face (high half-word), of the - direction the
	// previous row's + face (low half-word)
	constexpr uint32_t kOther = 0x01000706u;
	const uint32_t y0 = byte_perm(yp.x, ym.x, kOther), y1 = byte_perm(yp.y, ym.y, kOther);
	const uint32_t z0 = byte_perm(zp.z, zm.z, kOther), z1 = byte_perm(zp.w, zm.w, kOther);
	uint32_t vx = s.vis_x[row], vy = show_planes(p.x, p.y, y0, y1), vz = show_planes(p.z, p.w, z0, z1);
	const uint32_t tx = s.tt_x[row], ty = tt_planes(p.x, p.y, y0, y1), tz = tt_planes(p.z, p.w, z0, z1);
	if (tx | ty | tz) {
		vx |= show_textures(s, tx, 0, cell);
		vy |= show_textures(s, ty, 1, cell);
		vz |= show_textures(s, tz, 2, cell);
	}
	s.ne[16 * (32 + 2 * y + 1) + z] = uint16_t(vy);
	s.ne[16 * (32 + 2 * y) + z] = uint16_t(vy >> 16);
	s.ne[16 * (64 + 2 * z + 1) + y] = uint16_t(vz);
	s.ne[16 * (64 + 2 * z) + y] = uint16_t(vz >> 16);
	// lanes 8, 4, 2 and 1 apart within a row of 16: row_ror:8, half-row mirror of the quads mirrored, and
	// quad_perm 2,3,0,1 and 1,0,3,2
	uint32_t o = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)vx, 0x128, 0xf, 0xf, true);
	vx = transpose_step(vx, o, z & 8 ? 0xff00ff00u : 0x00ff00ffu, z & 8, 8);
	o = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)vx, 0x1b, 0xf, 0xf, true);
	o = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)o, 0x141, 0xf, 0xf, true);
	vx = transpose_step(vx, o, z & 4 ? 0xf0f0f0f0u : 0x0f0f0f0fu, z & 4, 4);
	o = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)vx, 0x4e, 0xf, 0xf, true);
	vx = transpose_step(vx, o, z & 2 ? 0xccccccccu : 0x33333333u, z & 2, 2);
	o = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)vx, 0xb1, 0xf, 0xf, true);
	vx = transpose_step(vx, o, z & 1 ? 0xaaaaaaaau : 0x55555555u, z & 1, 1);
	s.ne[16 * (2 * z + 1) + y] = uint16_t(vx);
	s.ne[16 * (2 * z) + y] = uint16_t(vx >> 16);
}

// ------------------------------------------------------------------------------------------------
// visible faces, numbered densely
// ------------------------------------------------------------------------------------------------
// A face's descriptor is its bit among all mask rows: task << 8 | row << 4 | column, with kDescTrans when it
// goes to the transparent pass.
constexpr uint32_t kDescTrans = 0x8000u;
static_assert(kTasks * 256 <= (int)kDescTrans, "descriptors of 15 bits");

// Running maximum over the wavefront, as wave_incl_sum.
__device__ __forceinline__ uint32_t wave_incl_max(uint32_t v) {
	v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, true));
	v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, true));
	v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, true));
	v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, true));
	v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, true));
	v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, true));
	return v;
}

// Units per thread of the numbering: 192 threads hold two each (128 threads: three).
template <int NT> constexpr int kUnitsPerThread = NT >= 192 ? 2 : 3;

// Numbers the visible faces, task by task and row by row, as the reference scans them: every unit's faces
// before it into s.upre. first: the faces before this thread's units; cnt: those in each. One barrier; s.upre
// is complete after the caller's next one. Returns the number of faces.
template <int NT> __device__ __forceinline__ uint32_t number_faces(Smem<NT> &s, uint32_t &first, uint32_t cnt[3]) {
	constexpr int U = kUnitsPerThread<NT>;
	const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
	uint32_t c = 0;
	cnt[0] = cnt[1] = cnt[2] = 0;
	if (tid < kUnits / U) {
		const uint64_t *rows = reinterpret_cast<const uint64_t *>(s.ne) + tid * U;
#pragma unroll
		for (int k = 0; k < U; ++k)
			c += cnt[k] = __popcll(rows[k]);
	}
	const uint32_t inc = wave_incl_sum(c);
	if (lane == 63)
		s.scan_w[wave][0] = inc;
	__syncthreads();
	uint32_t before = inc - c, all = 0;
#pragma unroll
	for (int w = 0; w < (kUnits / U + 63) / 64; ++w) {
		const uint32_t x = s.scan_w[w][0];
		before += w < wave ? x : 0u;
		all += x;
	}
	first = before;
	if (tid < kUnits / U) {
		uint32_t at = before;
#pragma unroll
		for (int k = 0; k < U; ++k) {
			s.upre[tid * U + k] = uint16_t(at);
			at += cnt[k];
		}
	}
	if (tid == 0)
		s.upre[kUnits] = uint16_t(all);
	return all;
}

// Marks the units of the tasks [t0, t1) at their first faces in s.own (all zero before), and again at the
// first face of a block of 64 where a unit continues into it, so that the unit of every face is the running
// maximum of the marks over the lanes of its block.
template <int NT>
__device__ __forceinline__ void mark_units(Smem<NT> &s, int t0, int t1, uint32_t g0, uint32_t first, const uint32_t cnt[3]) {
	constexpr int U = kUnitsPerThread<NT>;
	uint32_t p = first - g0;
#pragma unroll
	for (int k = 0; k < U; ++k) {
		const int q = (int)threadIdx.x * U + k;
		if (cnt[k] && q >= 4 * t0 && q < 4 * t1) {
			const uint32_t next = (p + 63u) & ~63u; // the first block that begins at or after p
			s.own[p] = uint16_t(q + 1);
			if (next < p + cnt[k])
				s.own[next] = uint16_t(q + 1);
		}
		p += cnt[k];
	}
}

// Position of the n-th set bit (from 0) of the 64-bit word (hi, lo).
__device__ __forceinline__ uint32_t nth_bit(uint32_t lo, uint32_t hi, uint32_t n) {
	uint32_t c = __popc(lo);
	bool up = n >= c;
	uint32_t w = up ? hi : lo, pos = up ? 32u : 0u;
	n -= up ? c : 0u;
#pragma unroll
	for (int h = 16; h >= 1; h >>= 1) {
		c = __popc(w & ((1u << h) - 1u));
		up = n >= c;
		n -= up ? c : 0u;
		w = up ? w >> h : w;
		pos += up ? uint32_t(h) : 0u;
	}
	return pos;
}

// The descriptor of face i of the group (dense index g0 + i); every lane of the wavefront comes here.
template <int NT> __device__ __forceinline__ uint32_t face_desc(const Smem<NT> &s, uint32_t i, uint32_t g0) {
	const uint32_t q = max(wave_incl_max(s.own[i]), 1u) - 1u;
	const uint2 rows = reinterpret_cast<const uint2 *>(s.ne)[q];
	return (q << 6) + nth_bit(rows.x, rows.y, g0 + i - s.upre[q]);
}

// Word of a visible face: Light4 (light4_init, :48-163) in the low 28 bits of x and y, the texture code in the upper
// four of x and bits 28-30 of y and the transparent-pass flag in bit 31. Faces merge only if their words are equal
// (Light4::operator==, :44, and the texture compare, :367-368). The code's upper three bits and the flag come from
// the table of codes as they lie in the word.
template <bool kRaw, int NT> __device__ __forceinline__ uint2 face_word(const Smem<NT> &s, uint32_t desc) {
	const int t = desc >> 8, u = (desc >> 4) & 15, v = desc & 15;
	const int A = task_axis(t), inv = task_plus(t) ^ 1;
	// byte strides along the mask's axes and the task's: 1, 18 and 324 voxels
	constexpr int all = 4 * (kSX + kSY + kSZ);
	const int su = A == 1 ? 4 * kSZ : 4 * kSY, sv = A == 0 ? 4 * kSZ : 4 * kSX, sa = all - su - sv;
	const int self = all + task_layer(t) * sa + u * su + v * sv;
	const bool u_first = inv == int(A == 2); // the winding's first axis (kLookup3v) is U
	const uint2 l = light4<kRaw>(s, self + (inv ? -sa : sa), u_first ? su : sv, u_first ? sv : su);
	const uint32_t pid = vox_pid(*reinterpret_cast<const uint32_t *>(reinterpret_cast<const char *>(s.vox) + self));
	const uint32_t tc = row_code(s, pid, 2 * A + inv);
	return make_uint2(l.x | tc << 28, l.y | (s.tables.codes[tc] & ~kCodeLow));
}

// Equal-to-right and equal-to-below bits of the visible face with dense index i (local to the group): its
// right and lower neighbours, when visible, are at i + 1 and after the rest of row u and the start of row
// u + 1 in the dense order.
template <int NT> __device__ __forceinline__ void face_links(Smem<NT> &s, uint32_t i, uint32_t desc) {
	const uint32_t r = (desc >> 4) & 0x7ffu, u = r & 15, v = desc & 15;
	// the neighbours' words are read whether or not the neighbours are visible (positions clamped into the
	// stage) and compared as whole words, so that only the rare atomics sit behind branches
	const uint32_t ne_u = s.ne[r], ne_d = uint32_t(s.ne[min(r + 1, uint32_t(kMaskRows - 1))]) & (0u - uint32_t(u < 15));
	const uint2 w = s.key[i];
	const uint32_t bit = 1u << (v + 16 * (u & 1));
	const uint32_t ir = min(i + 1, uint32_t(s.kListCap - 1));
	const uint32_t id = min(i + 1 + __popc(ne_u >> (v + 1)) + __popc(ne_d & ((1u << v) - 1u)), uint32_t(s.kListCap - 1));
	const uint2 right = s.key[ir], d = s.key[id];
	const bool eq_r = v < 15 && ((ne_u >> (v + 1)) & 1u) && ((right.x ^ w.x) | (right.y ^ w.y)) == 0;
	const bool eq_d = ((ne_d >> v) & 1u) && ((d.x ^ w.x) | (d.y ^ w.y)) == 0;
	if (eq_r)
		atomicOr(reinterpret_cast<uint32_t *>(&s.eh[r & ~1u]), bit);
	if (eq_d)
		atomicOr(reinterpret_cast<uint32_t *>(&s.ev[r & ~1u]), bit);
}

// ------------------------------------------------------------------------------------------------
// greedy merge of one task (:357-476), one lane per task
// ------------------------------------------------------------------------------------------------
// The reference scans rows u ascending and cells v ascending; at an uncovered visible cell it grows the
// quad along V while the next cell has an equal face word and is uncovered, then along U while every
// cell of the next row's segment is equal and uncovered, and marks the covered cells. The quads that start
// in row u are therefore exactly the maximal runs of uncovered visible cells split wherever the face word
// changes, and each run's height depends only on the rows below. Here a row's runs are found with bit
// operations and all of them are extended downward together.
// Moves marked bits from v to v - 1 (spread_down) or v - 1 to v (spread_up) while v is in `link`, i.e.
// while v continues the run of v - 1: it reaches a run's start from any of its cells, and vice versa.
__device__ __forceinline__ uint32_t spread_down(uint32_t d, uint32_t link) {
	uint32_t m = link;
	d |= (d & m) >> 1;
	m &= m >> 1;
	d |= (d & (m << 1)) >> 2;
	m &= m >> 2;
	d |= (d & (m << 3)) >> 4;
	m &= m >> 4;
	d |= (d & (m << 7)) >> 8;
	return d;
}
__device__ __forceinline__ uint32_t spread_up(uint32_t f, uint32_t link) {
	uint32_t m = link;
	f |= (f << 1) & m;
	m &= m << 1;
	f |= (f << 2) & m;
	m &= m << 2;
	f |= (f << 4) & m;
	m &= m << 4;
	f |= (f << 8) & m;
	return f;
}

// One task: its quad starts into eh and its uncovered visible cells into ev, in place of the link masks.
template <int NT> __device__ __forceinline__ void greedy_merge(Smem<NT> &s, int t) {
	// coverage of the rows below the current one by quads of earlier rows, and the equal-to-below masks,
	// held in registers as windows that shift up by one row per step (window row k = row u + k)
	uint32_t cov[8], ev[8];
	const uint16_t *nes = s.ne + 16 * t;
	uint16_t *ehs = s.eh + 16 * t, *evs = s.ev + 16 * t;
#pragma unroll
	for (int k = 0; k < 8; ++k) {
		cov[k] = 0;
		ev[k] = reinterpret_cast<const uint32_t *>(evs)[k];
	}
	// a row's masks are read one step ahead, so that their LDS latency overlaps the previous row's work
	uint32_t ne_n = nes[0], eh_n = ehs[0];
#pragma unroll 1
	for (int u = 0; u < 16; ++u) {
		const uint32_t ne = ne_n, eh = eh_n;
		if (u < 15) // row u + 1 is not written before this step writes row u
			ne_n = nes[u + 1], eh_n = ehs[u + 1];
		const uint32_t S = ne & ~(cov[0] & 0xffffu); // uncovered visible cells of row u
		const uint32_t link = S & ((S & eh) << 1);   // v continues the run of v - 1
		const uint32_t starts = S & ~link;
		// row u's results replace its (already read) inputs; ev's rows are in registers
		evs[u] = uint16_t(S);
		ehs[u] = uint16_t(starts);
		if (__ballot(S != 0)) { // branches for the whole wavefront: per-lane ones cost more in execution masks
			uint32_t alive = starts, cols = S;
#pragma unroll
			for (int k = 1; k <= 16; ++k) {
				// row u + k, if it exists: every column of a surviving run must continue into it
				if (!__ballot(alive != 0))
					break;
				uint32_t ok = 0; // rows past 15 read as empty from the shifted windows
				if (k < 16) {
					const uint32_t evr = (ev[(k - 1) >> 1] >> (16 * ((k - 1) & 1))) & 0xffffu;
					const uint32_t cvr = (cov[k >> 1] >> (16 * (k & 1))) & 0xffffu;
					ok = evr & ~cvr;
				}
				const uint32_t bad = cols & ~ok;
				if (bad) {
					const uint32_t dead = spread_down(bad, link) & alive;
					alive &= ~dead;
					cols &= ~spread_up(dead, link);
				}
				if (k < 16)
					cov[k >> 1] |= cols << (16 * (k & 1));
			}
		}
		// shift the windows up by one row
#pragma unroll
		for (int k = 0; k < 8; ++k) {
			const uint32_t nc = k < 7 ? cov[k + 1] : 0u, nv = k < 7 ? ev[k + 1] : 0u;
			cov[k] = (cov[k] >> 16) | (nc << 16);
			ev[k] = (ev[k] >> 16) | (nv << 16);
		}
	}
}

// The quad starts of one task into eh, and its uncovered visible cells into ev, in place of the link masks.
// A task whose equal neighbouring faces are all side by side (no equal-to-below bit) has one quad per
// run of equal faces along V: a visible face starts one unless it continues its left neighbour, and no
// cell is covered from above. One whose equal faces are all above each other (no equal-to-right bit)
// has one quad per run along U: a face starts one unless it continues the face above, and the cells
// below a start are covered by its quad. With neither, every visible face is a 1 x 1 quad. These follow
// from the masks directly (rows are 16-bit fields of the 64-bit words, row u + 4 q at bit 16 u, and a
// row's equal-to-right bit 15 is never set). Tasks with both are merged row by row.
template <int NT> __device__ __forceinline__ void quad_starts(Smem<NT> &s, int t) {
	uint64_t *eh64 = reinterpret_cast<uint64_t *>(s.eh + 16 * t), *ev64 = reinterpret_cast<uint64_t *>(s.ev + 16 * t);
	const uint64_t *ne64 = reinterpret_cast<const uint64_t *>(s.ne + 16 * t);
	uint64_t eh[4], ev[4], anyh = 0, anyv = 0;
#pragma unroll
	for (int q = 0; q < 4; ++q) {
		eh[q] = eh64[q], ev[q] = ev64[q];
		anyh |= eh[q], anyv |= ev[q];
	}
	if (anyh && anyv) {
		greedy_merge(s, t);
		return;
	}
#pragma unroll
	for (int q = 0; q < 4; ++q) {
		const uint64_t ne = ne64[q];
		// equal-to-below bits of the row above each row: the word shifted up one row, with the last
		// row of the previous word
		const uint64_t above = (ev[q] << 16) | (q > 0 ? ev[q - 1] >> 48 : 0ull);
		const uint64_t st = ne & ~(eh[q] << 1) & ~above;
		ev64[q] = anyv ? st : ne;
		eh64[q] = st;
	}
}

// ------------------------------------------------------------------------------------------------
// emission of one quad
// ------------------------------------------------------------------------------------------------
// The end of the longest run of tasks from t0 whose visible faces fit the face-word stage (one task, at
// most 256 faces, always fits). Every wavefront counts the tasks that end within it, two per lane (a search by one
// thread and a barrier took 0.8 us for each of a dense chunk's groups).
template <int NT> __device__ __forceinline__ int group_end(const Smem<NT> &s, int t0, uint32_t n_faces) {
	const uint32_t limit = uint32_t(s.upre[4 * t0]) + (uint32_t)s.kListCap;
	if (n_faces <= limit) // the rest fits (the usual case)
		return kTasks;
	static_assert(kTasks <= 128, "two tasks per lane");
	const int lane = threadIdx.x & 63, high = min(64 + lane, kTasks - 1);
	const bool in0 = s.upre[4 * (lane + 1)] <= limit, in1 = (s.upre[4 * (high + 1)] <= limit) & (64 + lane < kTasks);
	return __builtin_amdgcn_readfirstlane(__popcll(ballot64(in0)) + __popcll(ballot64(in1)));
}

// Where quad i of a pass goes: the base vertex of its mesh, the mesh of the pass (mk) and its index in that mesh (mj). The reference reads the 16-bit vertex count before splitting, so the first
// quad of a continuation mesh keeps base 65,532 (:273-279, :397-403).
__device__ __forceinline__ void quad_place(uint32_t i, uint32_t &vbase, uint32_t &mk, uint32_t &mj) {
	mk = i / kSplitQuads;
	mj = i - mk * kSplitQuads;
	vbase = (mj == 0 && mk > 0) ? 65532u : 4u * mj;
}

// A quad's box into the lane's box of the first mesh of its pass: the other pass's box takes the empty box, which
// changes nothing, and the transparent pass's box is left alone in chunks without transparent quads (any_tr, the same
// in every lane).
__device__ __forceinline__ void box_add(Box box[2], uint32_t pass, const Box &b, bool any_tr = true) {
	const uint32_t m = 0u - pass; // all ones for the transparent pass
	box_min(box[0], b, m);
	if (any_tr)
		box_min(box[1], b, ~m);
}

// A written quad's box into its mesh's AABB (per lane for the first mesh of a pass, LDS atomics for the
// others) and, when it starts a continuation mesh, a split event at its emission position epos.
template <int NT>
__device__ __forceinline__ void quad_done(Smem<NT> &s, uint32_t pass, uint32_t mk, uint32_t mj, uint32_t epos, const Box &b,
                                          Box box[2]) {
	if (mk == 0)
		box_add(box, pass, b);
	else
		aabb_merge(s, pass, mk, b);
	if (mj == 0 && mk > 0) { // a split happened right before this quad (:397-403)
		const uint32_t ev = atomicAdd(&s.n_events, 1u);
		if (ev < 16) {
			s.events[ev][0] = epos;
			s.events[ev][1] = (pass << 16) | (mk - 1u);
		}
	}
}

// Whether a quad starts at the face at desc.
template <int NT> __device__ __forceinline__ bool starts_quad(const Smem<NT> &s, uint32_t desc) {
	return (s.eh[(desc >> 4) & 0x7ffu] >> (desc & 15)) & 1u;
}

// Lanes below this one in a ballot.
__device__ __forceinline__ uint32_t lanes_below(uint64_t ballot) {
	return __builtin_amdgcn_mbcnt_hi(uint32_t(ballot >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(ballot), 0u));
}

// The quad that starts at the visible face at desc with face word `word`, quad i of its pass. Per
// task, ne still holds the visible cells, eh the quad starts and ev the uncovered visible cells S; the
// covered cells are C = ne & ~S. A quad from (u, v0) spans S's run from v0 to the next start along V, and
// covers rows u .. u + h - 1 of its columns, so below it column v0 is in C exactly for rows u + 1 ..
// u + h - 1: the cell under its last row is either not covered or starts a quad. split: some pass of the
// chunk has more than kSplitQuads quads; else every quad is in the first mesh of its pass. epos: the quads
// emitted before it, for a split.
template <int NT>
__device__ __forceinline__ void emit_face(Smem<NT> &s, uint32_t desc, uint2 word, uint32_t i, uint32_t epos, uint32_t n0,
                                          uint4 *verts, uint32_t *idx, Box box[2], bool any_tr, bool split) {
	const uint32_t r = (desc >> 4) & 0x7ffu, tr = desc >> 15;
	const int u = r & 15, v = desc & 15;
	const uint32_t link = uint32_t(s.ev[r] & ~s.eh[r]);
	const int w = __ffs(~(link >> (v + 1)));
	// most quads are one row high: the covered cells of the row below are tested before the loop (row 15
	// has none; its index is clamped so that the load needs no branch)
	const uint32_t rb = min(r + 1, uint32_t(kMaskRows - 1));
	const uint32_t cov_below = uint32_t(s.ne[rb] & ~s.ev[rb]) & (0u - uint32_t(u < 15));
	int h = 1;
	if ((cov_below >> v) & 1u) {
		h = 2;
#pragma unroll 1
		for (int k = 2; u + k < 16 && ((uint32_t(s.ne[r + k] & ~s.ev[r + k]) >> v) & 1u); ++k)
			++h;
	}
	uint32_t vbase = 4u * i, mk = 0, mj = i;
	if (split)
		quad_place(i, vbase, mk, mj);
	const Box b = emit_quad(s, desc, w, h, word, verts, idx, (tr ? n0 : 0u) + i, vbase);
	if (split)
		quad_done(s, tr, mk, mj, epos, b, box);
	else
		box_add(box, tr, b, any_tr);
}

// ------------------------------------------------------------------------------------------------
// one chunk
// ------------------------------------------------------------------------------------------------
// Per-chunk LDS state a job starts from (the slot list is loaded with the job).
template <int NT> __device__ __forceinline__ void chunk_init(Smem<NT> &s) {
	const int tid = threadIdx.x;
	for (int i = tid; i < 128; i += NT)
		s.custom_bits[i] = 0;
	if (tid < 2 * kMaxMeshPerPass * 6) {
		uint32_t *a = &s.aabb[0][0][0];
		a[tid] = (tid % 6) < 3 ? 0xffffffffu : 0u; // AABB<uint32_t>{}: min = max(), max = min() (dep/AABB.hpp:11)
	}
	if (tid == 0)
		s.n_events = 0, s.flags = 0;
}

// A packed halo (include/hcm.h, HCM_HALO_BLOCKS / HCM_HALO_LIGHT) into LDS as it is, in whole 16-byte loads
// where it is aligned (its job's place keeps the alignment of the first: 14,400 and 5,832 bytes a halo), so that
// each of its lines is read once also where it lies in host memory.
template <int NT> __device__ __forceinline__ void load_halo(const MeshParams &p, Smem<NT> &s, uint32_t job) {
	const uint16_t *b = p.halo_in + (size_t)job * HCM_HALO_BLOCKS;
	const uint8_t *l = p.halo_in_light + (size_t)job * HCM_HALO_LIGHT;
	const int tid = threadIdx.x;
	if (((uintptr_t(b) & 15u) | (uintptr_t(l) & 7u)) == 0) {
		constexpr int nb = HCM_HALO_BLOCKS * 2 / 16, nl = HCM_HALO_LIGHT / 8, kb = (nb + NT - 1) / NT, kl = (nl + NT - 1) / NT;
		static_assert(nb * 16 == HCM_HALO_BLOCKS * 2 && nl * 8 == HCM_HALO_LIGHT, "whole words");
		uint4 vb[kb];
		uint2 vl[kl];
#pragma unroll
		for (int k = 0; k < kb; ++k)
			vb[k] = reinterpret_cast<const uint4 *>(b)[min(tid + k * NT, nb - 1)];
#pragma unroll
		for (int k = 0; k < kl; ++k)
			vl[k] = reinterpret_cast<const uint2 *>(l)[min(tid + k * NT, nl - 1)];
#pragma unroll
		for (int k = 0; k < kb; ++k)
			if (tid + k * NT < nb)
				reinterpret_cast<uint4 *>(s.halo.blocks)[tid + k * NT] = vb[k];
#pragma unroll
		for (int k = 0; k < kl; ++k)
			if (tid + k * NT < nl)
				reinterpret_cast<uint2 *>(s.halo.light)[tid + k * NT] = vl[k];
	} else {
		for (int i = tid; i < HCM_HALO_BLOCKS; i += NT)
			s.halo.blocks[i] = b[i];
		for (int i = tid; i < HCM_HALO_LIGHT; i += NT)
			s.halo.light[i] = l[i];
	}
}

// One halo row of 18 voxels: blocks at x = -1, 0 .. 15 (two per word) and 16, light bytes from x = -1 on.
struct HaloRow {
	uint32_t bw[8], bl, br, lw[5];
};
template <int NT> __device__ __forceinline__ HaloRow halo_row(const Smem<NT> &s, int row) {
	// the packed halo's blocks reach from x = -2 to 17: 20 per row, ten words that start at an even word
	const int hz = row % kHalo, hy = row / kHalo;
	const uint2 *hb = reinterpret_cast<const uint2 *>(s.halo.blocks + 20 * (hz + 1 + 20 * hy));
	const uint16_t *hl = reinterpret_cast<const uint16_t *>(s.halo.light + kHalo * row);
	HaloRow r;
	uint32_t d[10];
#pragma unroll
	for (int k = 0; k < 5; ++k) {
		const uint2 w = hb[k];
		d[2 * k] = w.x, d[2 * k + 1] = w.y;
	}
	r.bl = d[0] >> 16, r.br = d[9] & 0xffffu;
#pragma unroll
	for (int k = 0; k < 8; ++k)
		r.bw[k] = d[k + 1];
#pragma unroll
	for (int k = 0; k < 5; ++k)
		r.lw[k] = hl[2 * k] | (k < 4 ? uint32_t(hl[2 * k + 1]) << 16 : 0u);
	return r;
}

// The words and descriptors of a group of n faces to the workgroup's part of p.kept, from its face g0 on, and back; a
// thread reads what it wrote, all of it on its way at once.
template <int NT> __device__ __forceinline__ void store_kept(const MeshParams &p, const Smem<NT> &s, uint32_t g0, uint32_t n) {
	uint2 *words = reinterpret_cast<uint2 *>(p.kept + blockIdx.x * kKeptBytes);
	uint16_t *desc = reinterpret_cast<uint16_t *>(words + kKeptFaces);
#pragma unroll 1
	for (uint32_t i = threadIdx.x; i < n; i += NT)
		words[g0 + i] = s.key[i], desc[g0 + i] = s.own[i];
}
template <int NT> __device__ __forceinline__ void load_kept(const MeshParams &p, Smem<NT> &s, uint32_t g0, uint32_t n) {
	const uint2 *words = reinterpret_cast<const uint2 *>(p.kept + blockIdx.x * kKeptBytes);
	const uint16_t *desc = reinterpret_cast<const uint16_t *>(words + kKeptFaces);
	constexpr int kSteps = (Smem<NT>::kListCap + NT - 1) / NT;
	uint2 w[kSteps];
	uint16_t d[kSteps];
#pragma unroll
	for (int k = 0; k < kSteps; ++k) {
		const uint32_t i = g0 + min(uint32_t(threadIdx.x + k * NT), n - 1);
		w[k] = words[i], d[k] = desc[i];
	}
#pragma unroll
	for (int k = 0; k < kSteps; ++k)
		if (uint32_t(threadIdx.x + k * NT) < n)
			s.key[threadIdx.x + k * NT] = w[k], s.own[threadIdx.x + k * NT] = d[k];
}

// One job; s.slots and the state of chunk_init are in place (a barrier after them).
template <bool kRaw, int NT> __device__ __forceinline__ void mesh_chunk(const MeshParams &p, Smem<NT> &s, uint32_t job) {
	const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
	constexpr int CPT = HCM_CHUNK_VOXELS / NT; // custom cells per thread

	// 1. halo staging: one thread per x-row (hy, hz) of 18 voxels. A voxel's word is its light fields and
	// the template its block id's byte looks up in LDS (the full table only for the few ids whose meta byte
	// changes the texture row); the row's flags come from an AND and an OR over its templates and from
	// comparing packed block pairs, the custom-mesh cells only when some template has a mesh.
	uint32_t my_flags = 0, wave_ref = 0xffffffffu;
	const JobBlocks blocks{p.blocks, s.slots, p.halo_in ? p.halo_in + (size_t)job * HCM_HALO_BLOCKS : nullptr};
	HaloRow given; // a packed halo's row: one per thread, all read before the first is staged over them
	if constexpr (NT >= kHaloRows)
		if (p.halo_in) {
			load_halo(p, s, job);
			__syncthreads();
			if (tid < kHaloRows)
				given = halo_row(s, tid);
			__syncthreads();
		}
	for (int row = tid; row < kHaloRows; row += NT) {
		const int hz = row % kHalo, hy = row / kHalo, y = hy - 1, z = hz - 1;
		uint32_t bw[8], bl, br, lw[5];
		if (NT >= kHaloRows && p.halo_in) {
			bl = given.bl, br = given.br;
#pragma unroll
			for (int k = 0; k < 8; ++k)
				bw[k] = given.bw[k];
#pragma unroll
			for (int k = 0; k < 5; ++k)
				lw[k] = given.lw[k];
		} else {
			const size_t lrow = 16u * (uint32_t(z & 15) + 16u * uint32_t(y & 15));
			const int syz = slot27_yz(hy, hz); // slot27(x, y, z) = 9 * (x term) + syz: 18 at x = 0, 9 at -1, 0 at 16
			const size_t cm = (size_t)s.slots[18 + syz] * HCM_CHUNK_VOXELS + lrow;
			const size_t cl = (size_t)s.slots[9 + syz] * HCM_CHUNK_VOXELS + lrow + 15;
			const size_t cr = (size_t)s.slots[syz] * HCM_CHUNK_VOXELS + lrow;
			const uint4 b0 = *reinterpret_cast<const uint4 *>(p.blocks + cm);
			const uint4 b1 = *reinterpret_cast<const uint4 *>(p.blocks + cm + 8);
			bw[0] = b0.x, bw[1] = b0.y, bw[2] = b0.z, bw[3] = b0.w, bw[4] = b1.x, bw[5] = b1.y, bw[6] = b1.z, bw[7] = b1.w;
			bl = p.blocks[cl], br = p.blocks[cr];
			if (p.halo_light) { // the job's rebuilt light, one 20-byte record per halo x-row
				const uint32_t *hl = reinterpret_cast<const uint32_t *>(p.halo_light + (size_t)job * kLightJobBytes +
				                                                        row * kLightRowBytes);
#pragma unroll
				for (int k = 0; k < 5; ++k)
					lw[k] = hl[k];
			} else { // the same layout from the store: x = -1 in byte 0, x = 0 .. 15 in bytes 1 .. 16, x = 16 in 17
				const uint4 lm = *reinterpret_cast<const uint4 *>(p.light + cm);
				const uint32_t ll = p.light[cl], lr = p.light[cr];
				lw[0] = ll | (lm.x << 8);
				lw[1] = (lm.x >> 24) | (lm.y << 8);
				lw[2] = (lm.y >> 24) | (lm.z << 8);
				lw[3] = (lm.z >> 24) | (lm.w << 8);
				lw[4] = (lm.w >> 24) | (lr << 8);
			}
		}
		// one reference value per wavefront (its first row's first voxel): a halo of one block value has
		// every voxel equal to it and all wavefronts' references equal
		const uint32_t v0 = __builtin_amdgcn_readfirstlane(bl);
		if (row < NT)
			wave_ref = v0;
		const uint32_t ref2 = wave_ref | (wave_ref << 16);
		uint32_t diff = (bl ^ wave_ref) | (br ^ wave_ref);
#pragma unroll
		for (int k = 0; k < 8; ++k)
			diff |= bw[k] ^ ref2;
		const bool nonuniform = diff != 0;
		uint32_t tm[18], words[18];
#pragma unroll
		for (int x = 0; x < 18; ++x) {
			const uint32_t b = x == 0 ? bl : (x == 17 ? br : bw[(x - 1) >> 1] >> (16 * ((x - 1) & 1)));
			const uint2 q = s.tables.tmpl_id[b & 0xffu];
			tm[x] = q.x, words[x] = q.y;
		}
		uint32_t any_meta = 0;
#pragma unroll
		for (int x = 0; x < 18; ++x)
			any_meta |= tm[x];
		if (any_meta & kTmplMeta) { // ids whose texture row depends on the meta byte
			// every voxel's row from the full table (any 16-bit value indexes it), issued as one batch of
			// loads and then one of LDS lookups, so the row waits once on memory and not once per voxel
			uint32_t full[18];
#pragma unroll
			for (int x = 0; x < 18; ++x) {
				const uint32_t b = x == 0 ? bl : (x == 17 ? br : (bw[(x - 1) >> 1] >> (16 * ((x - 1) & 1))) & 0xffffu);
				full[x] = p.reg->pid_of[b];
			}
#pragma unroll
			for (int x = 0; x < 18; ++x) {
				const uint2 v = s.tables.pid_vox[full[x]];
				words[x] = tm[x] & kTmplMeta ? v.y : words[x];
				tm[x] = tm[x] & kTmplMeta ? v.x : tm[x];
			}
		}
		uint32_t and_all = ~0u, or_inner = 0;
		uint32_t *dst = s.vox + row * kHalo;
		static_assert(kVoxSunBit == 8 && kVoxTorchBit == 16, "light in the low nibbles of two bytes");
#pragma unroll
		for (int x = 0; x < 18; ++x) {
			const uint32_t w = lw[x >> 2], k = x & 3; // light bytes are sun | torch << 4
			const uint32_t light = byte_perm((w >> 4) & 0x0f0f0f0fu, w & 0x0f0f0f0fu, 0x0c04000cu + 0x010100u * k);
			dst[x] = (light & tm[x]) | words[x];
			and_all &= tm[x];
			if (x >= 1 && x <= 16)
				or_inner |= tm[x];
		}
		put_planes(s, hy, hz, tm);
		const uint32_t or_all = or_inner | tm[0] | tm[17];
		const bool inside_yz = (unsigned)y < 16u && (unsigned)z < 16u;
		// every voxel an opaque cube: the shape bits that the cube has set are set in all, the others in none
		const bool mixed = (and_all & kVoxShape & kVoxOpaqueCube) != (kVoxShape & kVoxOpaqueCube) ||
		                   (or_all & kVoxShape & ~kVoxOpaqueCube) != 0;
		if (nonuniform)
			my_flags |= kFlagNonUniform;
		if (mixed)
			my_flags |= kFlagMixed;
		if (inside_yz && (or_inner & kVoxShape))
			my_flags |= kFlagInnerFaces;
		if (or_all & kTmplFlow)
			my_flags |= kFlagFlow;
		if (inside_yz && (or_inner & kTmplMesh)) {
			uint32_t mesh_bits = 0;
#pragma unroll
			for (int x = 0; x < 16; ++x)
				mesh_bits |= ((tm[x + 1] / kTmplMesh) & 1u) << x;
			const uint32_t cell0 = 16u * (uint32_t(z) + 16u * uint32_t(y));
			atomicOr(&s.custom_bits[cell0 >> 5], mesh_bits << (cell0 & 31));
			my_flags |= kFlagCustom;
		}
	}
	// the wavefront's flags, bit by bit (kFlagNonUniform .. kFlagInnerFaces), then one lane's LDS atomic:
	// an atomic from every lane with a different value is expanded into a scalar loop over the lanes
	uint32_t wave_flags = 0;
#pragma unroll
	for (int b = 0; b < 5; ++b)
		wave_flags |= ballot64((my_flags >> b) & 1u) ? 1u << b : 0u;
	if (lane == 0) {
		if (wave_flags)
			atomicOr(&s.flags, wave_flags);
		s.wave_ref[wave] = wave_ref; // 0xffffffff: the wavefront staged no row
	}
	__syncthreads();
	uint32_t flags = s.flags;
#pragma unroll
	for (int w = 1; w < NT / 64; ++w)
		if (s.wave_ref[w] != 0xffffffffu && s.wave_ref[w] != s.wave_ref[0])
			flags |= kFlagNonUniform;

	// one block value everywhere hides every face when the block's opposite textures do not show to each
	// other (true of every registered block; a registry may define one whose do)
	const bool uniform_hidden =
	    !(flags & kFlagNonUniform) && !(s.tables.rows[block_pid(p, s, s.wave_ref[0])].y & kRowSelfShow);
	if (!(flags & kFlagCustom) && (uniform_hidden || !(flags & kFlagMixed) || !(flags & kFlagInnerFaces))) {
		// one block value everywhere whose faces hide each other, opaque cubes only, or no chunk voxel
		// with a face: no quads
		if (tid == 0)
			p.results[job] = hcm_job_result{HCM_OK, 0u, 0u, 0u};
		return;
	}

	// 2. liquid-flow cells take the flow mesh's face textures (:221-236)
	if (flags & kFlagFlow) {
		constexpr uint32_t kKeep = kVoxLight | kVoxDirect;
		for (int i = tid; i < kHaloVox; i += NT) {
			if (!(s.vox[i] & kVoxFlow)) // each thread rewrites only its own cells
				continue;
			const int hx = i % kHalo, rest = i / kHalo, hz = rest % kHalo, hy = rest / kHalo;
			const uint32_t pid = vox_pid(s.vox[i]);
			const uint32_t mesh = s.tables.rows[pid].y >> 24;
			const Flow f = flow_heights(p, blocks, hx - 1, hy - 1, hz - 1, p.reg->meshes[mesh].flow_height);
			const uint32_t tmpl = s.tables.pid_vox[p.reg->flow_pid_base + flow_pattern(f)].y;
			s.vox[i] = (s.vox[i] & kKeep) | (tmpl & ~kKeep);
		}
		__syncthreads();
		// their rows' planes again
		for (int row = tid; row < kHaloRows; row += NT) {
			uint32_t w[18];
#pragma unroll
			for (int x = 0; x < 18; ++x)
				w[x] = s.tables.pid_vox[vox_pid(s.vox[row * kHalo + x])].x;
			put_planes(s, row / kHalo, row % kHalo, w);
		}
		__syncthreads();
	}

	// 3. faces: visibility masks, then the dense numbering of the visible faces. The link masks start empty, and
	// so do the marks of the numbering.
	for (int row = tid; row < 256; row += NT)
		visibility_row(s, row);
	for (int i = tid; i < kMaskRows / 8; i += NT) {
		reinterpret_cast<uint4 *>(s.eh)[i] = make_uint4(0, 0, 0, 0);
		reinterpret_cast<uint4 *>(s.ev)[i] = make_uint4(0, 0, 0, 0);
	}
	for (int i = tid; i < s.kListCap / 8; i += NT)
		reinterpret_cast<uint4 *>(s.own)[i] = make_uint4(0, 0, 0, 0);
	__syncthreads();
	uint32_t first, cnt[3];
	const uint32_t n_faces = number_faces(s, first, cnt);
	if (n_faces == 0 && !(flags & kFlagCustom)) { // no visible face and no custom mesh: no quads
		if (tid == 0)
			p.results[job] = hcm_job_result{HCM_OK, 0u, 0u, 0u};
		return;
	}

	// custom faces per thread range of cells, and their prefix sums
	uint32_t c_o = 0, c_t = 0, cust0 = 0, cust1 = 0;
	uint64_t cust_pre = 0;
	if (flags & kFlagCustom) {
		for (uint32_t bits = custom_cells(s); bits; bits &= bits - 1) {
			const CustomCell c = custom_cell(p, s, blocks, tid * CPT + __ffs(bits) - 1);
			const uint32_t nt = __popc(c.trans);
			c_t += nt;
			c_o += c.count - nt;
		}
		__syncthreads(); // scan_w is read by number_faces
		uint32_t scan[3] = {c_o, c_t, 0}, tot[3];
		block_excl_sums(s, scan, tot);
		cust_pre = (uint64_t)scan[0] | ((uint64_t)scan[1] << 32);
		cust0 = tot[0], cust1 = tot[1];
	}

	// 4. groups of tasks whose visible faces fit the stage, twice: first every group's faces, links and quads
	// (one group but in dense chunks), which gives the chunk's quad counts; then, from the last group, whose
	// words are still in the stage, the emission, for which an earlier group's words are read back from the
	// workgroup's part of p.kept, or computed again where that is not given or too small. A
	// quad's place in its pass is its start's among the faces, counted by ballots over blocks of 64 faces.
	const uint32_t wave_u = __builtin_amdgcn_readfirstlane(wave);
	uint32_t base_o = cust0, base_t = cust1;       // quads of each pass before the group
	uint32_t n0 = 0, n1 = 0, nm0 = 0, nm1 = 0;      // the chunk's quads and meshes per pass
	uint32_t pool_base = 0;
	uint4 *verts = nullptr;  // the chunk's range of the pool
	uint32_t *idx = nullptr;
	// AABB<uint32_t>::Merge (dep/AABB.hpp:52-59) of the first mesh of each pass per lane, reduced at the end; later
	// meshes of a pass (past 16,383 quads) by LDS atomics
	Box box[2] = {{~0u, ~0u, ~0u}, {~0u, ~0u, ~0u}};
	bool any_tr = false, split = false, collect = true;
	uint32_t n_saved = 0, next_saved = 0, g0 = 0; // groups before the last; the next to emit; the group's first face
	int t0 = 0;
#pragma unroll 1
	for (bool again = false;; again = true) {
		int t1 = kTasks;
		uint32_t n = n_faces;
		bool loaded = false;
		if (again || n_faces > (uint32_t)s.kListCap) {
			__syncthreads(); // s.upre is complete; the last group's descriptors are read
			t1 = group_end(s, t0, n_faces);
			const uint32_t end = __builtin_amdgcn_readfirstlane(s.upre[4 * t1]);
			n = end - g0;
			if (!collect && p.kept && end <= kKeptFaces) {
				load_kept(p, s, g0, n);
				loaded = true;
			} else if (again) {
				for (int i = tid; i < s.kListCap / 8; i += NT)
					reinterpret_cast<uint4 *>(s.own)[i] = make_uint4(0, 0, 0, 0);
				__syncthreads();
			}
		}
		if (!loaded) {
			mark_units(s, t0, t1, g0, first, cnt);
			__syncthreads();
			// face words
#pragma unroll 1
			for (uint32_t b = wave_u; b * 64 < n; b += NT / 64) {
				const uint32_t i = 64 * b + lane, desc = face_desc(s, i, g0);
				if (i < n) {
					const uint2 word = face_word<kRaw>(s, desc);
					s.key[i] = word;
					s.own[i] = uint16_t(desc | (word.y >> 31 ? kDescTrans : 0u));
				}
			}
		}
		__syncthreads();
		if (collect) {
#pragma unroll 1
			for (uint32_t i = tid; i < n; i += NT)
				face_links(s, i, s.own[i]);
			__syncthreads();
			if (t0 + tid < t1)
				quad_starts(s, t0 + tid);
			__syncthreads();
		}
		// quads that start in each block of 64 faces, and before each block in the group (lane b: block b)
#pragma unroll 1
		for (uint32_t b = wave_u; b * 64 < n; b += NT / 64) {
			const uint32_t i = 64 * b + lane, desc = s.own[i];
			const bool st = (i < n) & starts_quad(s, desc), tr = desc >> 15;
			const uint32_t c = (uint32_t)__popcll(ballot64(st & !tr)) | (uint32_t)__popcll(ballot64(st & tr)) << 16;
			if (lane == 0)
				s.bcnt[b] = c;
		}
		__syncthreads();
		const uint32_t c = (uint32_t)lane * 64 < n ? s.bcnt[lane] : 0u, inc = wave_incl_sum(c), ex = inc - c;
		if (collect) {
			const uint32_t tot = (uint32_t)__builtin_amdgcn_readlane((int)inc, 63);
			n0 = base_o + (tot & 0xffffu), n1 = base_t + (tot >> 16);
			if (t1 < kTasks) { // the group waits for the others' counts
				if (p.kept && g0 + n <= kKeptFaces)
					store_kept(p, s, g0, n);
				if (tid == 0)
					s.grp[n_saved] = make_uint2(uint32_t(t0) | base_o << 8, base_t);
				++n_saved;
				base_o = n0, base_t = n1;
				t0 = t1;
				g0 += n;
				continue;
			}
			// 5. allocation: the chunk's output is [pool_base, +n0) opaque and [+n0, +n0+n1) transparent, custom
			// quads first in each pass; the quad range and the mesh records by one atomic each, issued by two
			// lanes of one instruction so that both are in flight together
			const uint32_t total = n0 + n1;
			if (total == 0) {
				if (tid == 0)
					p.results[job] = hcm_job_result{HCM_OK, 0u, 0u, 0u};
				return;
			}
			nm0 = (n0 + kSplitQuads - 1) / kSplitQuads, nm1 = (n1 + kSplitQuads - 1) / kSplitQuads;
			// (a launch of one job has the pool to itself)
			if (tid < 2) {
				const uint32_t base = p.alone ? 0u : atomicAdd(tid == 0 ? &p.ctr->pool_cursor : &p.ctr->mesh_cursor, tid == 0 ? total : nm0 + nm1);
				if (tid == 0)
					s.pool_base = base;
				else
					s.mesh_base = base;
			}
			__syncthreads();
			pool_base = __builtin_amdgcn_readfirstlane(s.pool_base);
			verts = reinterpret_cast<uint4 *>(p.pool_verts) + 2 * (size_t)pool_base;
			idx = reinterpret_cast<uint32_t *>(p.pool_idx) + 3 * (size_t)pool_base;
			if ((uint64_t)pool_base + total > p.pool_cap || (uint64_t)s.mesh_base + nm0 + nm1 > p.rec_cap) {
				if (tid == 0)
					p.results[job] = hcm_job_result{(int32_t)HCM_ERR_POOL_FULL, 0u, 0u, total};
				return;
			}
			any_tr = n1 != 0;
			split = n0 > kSplitQuads || n1 > kSplitQuads;
			collect = false;
		}
		// 6. emission: one lane per visible face, a quad per face that starts one
#pragma unroll 1
		for (uint32_t b = wave_u; b * 64 < n; b += NT / 64) {
			const uint32_t i = 64 * b + lane, desc = s.own[i];
			const bool st = (i < n) & starts_quad(s, desc), tr = desc >> 15;
			const uint64_t opaque = ballot64(st & !tr), trans = ballot64(st & tr);
			const uint32_t before = (uint32_t)__builtin_amdgcn_readlane((int)ex, (int)b);
			if (st) {
				const uint32_t io = base_o + (before & 0xffffu) + lanes_below(opaque);
				const uint32_t it = base_t + (before >> 16) + lanes_below(trans);
				emit_face(s, desc, s.key[i], tr ? it : io, io + it, n0, verts, idx, box, any_tr, split);
			}
		}
		if (next_saved == n_saved)
			break;
		const uint2 saved = s.grp[next_saved++];
		t0 = int(saved.x & 0xffu), base_o = saved.x >> 8, base_t = saved.y;
		g0 = s.upre[4 * t0];
	}
	// custom quads, after the regular ones (their positions in the output are fixed by the prefix sums): in
	// windows of the face-word stage, the threads list their cells' quads (cells in YZX order, faces in
	// mesh order, each thread its range of cells), then one lane per listed quad writes it
	if (flags & kFlagCustom) {
		const uint32_t n_cust = cust0 + cust1;
#pragma unroll 1
		for (uint32_t w0 = 0; w0 < n_cust; w0 += s.kListCap) {
			__syncthreads(); // key is free: the regular quads and the previous window are written
			const uint32_t w1 = w0 + s.kListCap;
			uint32_t io = (uint32_t)cust_pre, it = (uint32_t)(cust_pre >> 32);
			if (io + it < w1 && io + it + c_o + c_t > w0) {
				for (uint32_t bits = custom_cells(s); bits && io + it < w1; bits &= bits - 1) {
					const int cell = tid * CPT + __ffs(bits) - 1;
					const CustomCell c = custom_cell(p, s, blocks, cell);
					for (uint32_t j = 0; j < c.count; ++j) {
						const uint32_t tr = (c.trans >> j) & 1u, g = io + it, i = tr ? it++ : io++;
						if (g >= w0 && g < w1)
							s.key[g - w0] = make_uint2(uint32_t(cell) | (j << 12) | (tr << 31), i);
					}
				}
			}
			__syncthreads();
			const uint32_t n = min(n_cust - w0, (uint32_t)s.kListCap);
			for (uint32_t v = tid; v < 4 * n; v += NT) { // a lane per vertex
				const uint32_t e = v >> 2;
				const uint2 ent = s.key[e];
				const uint32_t tr = ent.x >> 31;
				uint32_t vbase, mk, mj;
				quad_place(ent.y, vbase, mk, mj);
				const uint32_t slot = pool_base + (tr ? n0 : 0u) + ent.y;
				const uint32_t at = emit_custom<kRaw>(p, s, blocks, ent.x & 0xffffu, v & 3, slot, vbase);
				quad_done(s, tr, mk, (v & 3) ? ~0u : mj, w0 + e, word_box(at, at), box); // (a split is one lane's to note)
			}
		}
	}

	// the passes' boxes over the wavefront (a pass without quads is skipped: its boxes are empty)
	if (n0) {
		const Box b = wave_box(box[0]);
		if (lane == 0)
			aabb_merge(s, 0, 0, b);
	}
	if (n1) {
		const Box b = wave_box(box[1]);
		if (lane == 0)
			aabb_merge(s, 1, 0, b);
	}
	__syncthreads();

	// 7. mesh records in the reference's order: split meshes by time, then opaque, then transparent
	if (tid == 0) {
		const uint32_t ne = min(s.n_events, 16u);
		for (uint32_t a = 1; a < ne; ++a) // insertion sort by emission position
			for (uint32_t b = a; b > 0 && s.events[b - 1][0] > s.events[b][0]; --b) {
				const uint32_t e0 = s.events[b][0], e1 = s.events[b][1];
				s.events[b][0] = s.events[b - 1][0], s.events[b][1] = s.events[b - 1][1];
				s.events[b - 1][0] = e0, s.events[b - 1][1] = e1;
			}
		const uint32_t mbase = s.mesh_base;
		uint32_t m = 0;
		auto put = [&](uint32_t pass, uint32_t k) {
			const uint32_t n_p = pass ? n1 : n0;
			hcm_mesh_rec r;
			for (int a = 0; a < 6; ++a)
				r.aabb[a] = s.aabb[pass][k][a];
			r.first_quad = pool_base + (pass ? n0 : 0u) + k * kSplitQuads;
			r.quad_count = min(kSplitQuads, n_p - k * kSplitQuads);
			r.job = job;
			r.transparent = pass;
			p.recs[mbase + m++] = r;
		};
		for (uint32_t e = 0; e < ne; ++e)
			put(s.events[e][1] >> 16, s.events[e][1] & 0xffffu);
		if (nm0)
			put(0, nm0 - 1);
		if (nm1)
			put(1, nm1 - 1);
		p.results[job] = hcm_job_result{HCM_OK, mbase, m, n0 + n1};
	}
}

template <int NT, bool kRaw> __global__ __launch_bounds__(NT, NT >= 512 ? 2 : 3) void mesh_kernel(MeshParams p) {
	__shared__ Smem<NT> s;
	if (threadIdx.x == 0) // (only this lane uses it)
		s.claims.init(p.n_jobs);
	const int lane = threadIdx.x & 63;
	const uint32_t given = p.job_base + blockIdx.x; // per-chunk launches: the workgroup's one job
	for (uint32_t i = threadIdx.x; i < sizeof(MeshTables) / 16; i += NT)
		reinterpret_cast<uint4 *>(&s.tables)[i] = reinterpret_cast<const uint4 *>(p.tables)[i];
	for (;;) {
		// wavefront 0 claims the next job and loads its slot list while the others set up its LDS state
		if (threadIdx.x < 64) {
			uint32_t job = ~0u;
			if (lane == 0) {
				job = p.persistent ? s.claims.next(p.ctr) : given;
				s.job = job;
			}
			job = (uint32_t)__builtin_amdgcn_readfirstlane((int)job);
			if (job < p.n_jobs && lane < 27 && !p.halo_in)
				s.slots[lane] = p.nbr[27 * (size_t)job + lane];
		}
		chunk_init(s);
		__syncthreads();
		const uint32_t job = s.job;
		if (job >= p.n_jobs)
			break;
		mesh_chunk<kRaw>(p, s, job);
		if (!p.persistent)
			break;
		__syncthreads();
	}
	// every claim and allocation of this workgroup precedes its increment of `done`, so the last
	// workgroup to increment it sees final totals and may clear the counters for the next run. They are
	// atomics that have returned, and nothing else of this workgroup is read before the launch ends: no fence, which
	// would write back the XCD's L2 once per workgroup (the cave batch 95.0 -> 86.2 us without, 1,000 random chunks
	// 258 -> 230 us).
	if (p.self_reset && threadIdx.x == 0) {
		claims_returned();
		if (atomicAdd(&p.ctr->done, 1u) == gridDim.x - 1) {
			p.ctr->total_quads = atomicAdd(&p.ctr->pool_cursor, 0u);
			p.ctr->total_meshes = atomicAdd(&p.ctr->mesh_cursor, 0u);
			for (uint32_t q = 0; q < kQueues; ++q)
				p.ctr->queue[q].v = 0;
			p.ctr->dry.v = 0;
			p.ctr->pool_cursor = 0;
			p.ctr->mesh_cursor = 0;
			p.ctr->done = 0;
		}
	}
}

__global__ void reset_kernel(Counters *ctr) {
	if (threadIdx.x == 0) {
		for (uint32_t q = 0; q < kQueues; ++q)
			ctr->queue[q].v = 0;
		ctr->dry.v = 0;
		ctr->pool_cursor = 0;
		ctr->mesh_cursor = 0;
		ctr->done = 0;
	}
}

// Applies voxel edits in order of their index; edits to one voxel within a launch are resolved by the
// host, which keeps only the last one. An edit with local >= 4096 sets sunlight height local - 4096 of
// its slot to the low byte of `block` (heights may be null when no such edit is sent).
__global__ void edit_kernel(uint16_t *blocks, uint8_t *light, int8_t *heights, const VoxelEdit *edits, uint32_t n) {
	const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i < n) {
		const VoxelEdit e = edits[i];
		if (e.local >= HCM_CHUNK_VOXELS) {
			heights[(size_t)e.slot * 256 + (e.local - HCM_CHUNK_VOXELS)] = int8_t(uint8_t(e.block));
			return;
		}
		const size_t g = (size_t)e.slot * HCM_CHUNK_VOXELS + e.local;
		blocks[g] = uint16_t(e.block);
		light[g] = uint8_t(e.light);
	}
}

hipError_t launch_edits(uint16_t *blocks, uint8_t *light, int8_t *heights, const VoxelEdit *edits, uint32_t n,
                        hipStream_t stream) {
	if (n == 0)
		return hipSuccess;
	hipLaunchKernelGGL(edit_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, blocks, light, heights, edits, n);
	return hipGetLastError();
}

// Copies staged chunk uploads into their store slots, one workgroup per chunk: move k copies staged
// chunk moves[k].x to slot moves[k].y -- its 4096 blocks, and its 4096 light bytes or its 256 sunlight
// heights, whichever staging array is given.
__global__ void upload_scatter_kernel(const uint4 *sblocks, const uint4 *slight, const uint4 *sheights,
                                      const uint2 *moves, uint4 *blocks, uint4 *light, uint4 *heights) {
	const uint2 m = moves[blockIdx.x];
	const uint32_t t = threadIdx.x;
	constexpr uint32_t kB = HCM_CHUNK_VOXELS * 2 / 16, kL = HCM_CHUNK_VOXELS / 16, kH = 256 / 16;
	blocks[(size_t)m.y * kB + t] = sblocks[(size_t)m.x * kB + t];
	blocks[(size_t)m.y * kB + 256 + t] = sblocks[(size_t)m.x * kB + 256 + t];
	if (slight)
		light[(size_t)m.y * kL + t] = slight[(size_t)m.x * kL + t];
	if (sheights && t < kH)
		heights[(size_t)m.y * kH + t] = sheights[(size_t)m.x * kH + t];
}
static_assert(HCM_CHUNK_VOXELS * 2 / 16 == 512 && HCM_CHUNK_VOXELS / 16 == 256, "one 256-thread workgroup per chunk");

hipError_t launch_upload_scatter(const uint16_t *sblocks, const uint8_t *slight, const int8_t *sheights,
                                 const uint2 *moves, uint32_t n, uint16_t *blocks, uint8_t *light, int8_t *heights,
                                 hipStream_t stream) {
	if (n == 0)
		return hipSuccess;
	hipLaunchKernelGGL(upload_scatter_kernel, dim3(n), dim3(256), 0, stream, reinterpret_cast<const uint4 *>(sblocks),
	                   reinterpret_cast<const uint4 *>(slight), reinterpret_cast<const uint4 *>(sheights), moves,
	                   reinterpret_cast<uint4 *>(blocks), reinterpret_cast<uint4 *>(light),
	                   reinterpret_cast<uint4 *>(heights));
	return hipGetLastError();
}

// n words of type T from src to dst by the whole grid.
template <typename T> __device__ __forceinline__ void copy_words(void *dst, const void *src, size_t n) {
	for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
		reinterpret_cast<T *>(dst)[i] = reinterpret_cast<const T *>(src)[i];
}

// Bound by the link to the host (56 GB/s): 64 KB of results and 120 KB of records of 4,096 jobs take about 7 us
// with the launch, where three copies and two synchronisations took about 75.
__global__ __launch_bounds__(256) void export_kernel(ExportParams p) {
	uint32_t quads = p.given_quads, meshes = 0;
	if (p.ctr) {
		quads = p.persistent ? p.ctr->total_quads : p.ctr->pool_cursor;
		meshes = p.persistent ? p.ctr->total_meshes : p.ctr->mesh_cursor;
	}
	if (p.out_totals && blockIdx.x == 0 && threadIdx.x == 0)
		p.out_totals[0] = quads, p.out_totals[1] = meshes;
	if (p.results)
		copy_words<uint4>(p.out_results, p.results, p.n_jobs);
	if (p.recs)
		copy_words<uint2>(p.out_recs, p.recs, (size_t)min(meshes, p.rec_cap) * (sizeof(hcm_mesh_rec) / sizeof(uint2)));
	if (p.verts && quads <= p.quad_cap) {
		copy_words<uint4>(p.out_verts, p.verts, 2 * (size_t)quads);
		copy_words<uint32_t>(p.out_idx, p.idx, 3 * (size_t)quads);
	}
}
static_assert(sizeof(hcm_job_result) == sizeof(uint4) && sizeof(hcm_mesh_rec) % sizeof(uint2) == 0, "whole words");

hipError_t launch_export(const ExportParams &p, hipStream_t stream) {
	const int grid = p.verts ? 256 : 64;
	hipLaunchKernelGGL(export_kernel, dim3(grid), dim3(256), 0, stream, p);
	return hipGetLastError();
}

hipError_t launch_reset(Counters *ctr, hipStream_t stream) {
	hipLaunchKernelGGL(reset_kernel, dim3(1), dim3(64), 0, stream, ctr);
	return hipGetLastError();
}

hipError_t launch_mesh(const MeshParams &p, int threads, int grid, hipStream_t stream) {
	if (p.halo_in && threads < kHaloRows) // packed halos are staged one row per thread
		return hipErrorInvalidValue;
	const auto launch = [&](auto plain, auto raw) {
		hipLaunchKernelGGL((p.raw_front ? raw : plain), dim3(grid), dim3(threads), 0, stream, p);
	};
	switch (threads) {
	case 128:
		launch(mesh_kernel<128, false>, mesh_kernel<128, true>);
		break;
	case 256:
		launch(mesh_kernel<256, false>, mesh_kernel<256, true>);
		break;
	case 512:
		launch(mesh_kernel<512, false>, mesh_kernel<512, true>);
		break;
	default:
		return hipErrorInvalidValue;
	}
	return hipGetLastError();
}

// gfx950 allocates a CU's 160 KB of LDS in 1,280-byte blocks: three 256-thread workgroups per CU need
// at most 42 blocks each (a 54,208-byte build ran at two per CU).
static_assert(sizeof(Smem<256>) <= 42 * 1280, "three 256-thread workgroups per CU");

int mesh_lds_bytes(int threads) {
	switch (threads) {
	case 128:
		return (int)sizeof(Smem<128>);
	case 256:
		return (int)sizeof(Smem<256>);
	case 512:
		return (int)sizeof(Smem<512>);
	default:
		return 0;
	}
}

} // namespace hcm
