// What the serving loop (hcm_serve.cpp) enqueues on which stream, over the CPU stand-ins of stub_hip and
// serve_stub_device.cpp: this file compiles the loop with its runtime calls and launches recorded. Batches end only while
// the gate is open, so that requests can be held back until one batch takes them all. Exit status 0 when all holds.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <condition_variable>
#include <cstdio>
#include <map>
#include <mutex>
#include <thread>
#include <vector>

#include "hcm_internal.h"

namespace rec {

struct Scatter {
	hipStream_t stream;
	const void *blocks, *light, *heights;
	std::vector<uint32_t> slots;
};
struct Copy {
	hipStream_t stream;
	const void *dst, *src;
};
std::mutex mu;
std::map<const char *, size_t> pinned; // begin -> bytes
std::vector<Scatter> scatters;
std::vector<Copy> copies;
std::vector<hipStream_t> exports, syncs; // exports: of a chunk's quads, not of a batch's results
std::atomic<bool> gate{true};

bool is_pinned(const void *p) {
	std::lock_guard<std::mutex> lk(mu);
	auto it = pinned.upper_bound((const char *)p);
	return it != pinned.begin() && (const char *)p < std::prev(it)->first + std::prev(it)->second;
}
void clear() {
	std::lock_guard<std::mutex> lk(mu);
	scatters.clear(), copies.clear(), exports.clear(), syncs.clear();
}
hipError_t host_malloc(void **p, size_t n) {
	const hipError_t e = hipHostMalloc(p, n);
	std::lock_guard<std::mutex> lk(mu);
	pinned[(const char *)*p] = n;
	return e;
}
hipError_t memcpy_async(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t st) {
	{
		std::lock_guard<std::mutex> lk(mu);
		copies.push_back(Copy{st, d, s});
	}
	return hipMemcpyAsync(d, s, n, k, st);
}
hipError_t stream_synchronize(hipStream_t s) {
	std::lock_guard<std::mutex> lk(mu);
	syncs.push_back(s);
	return hipSuccess;
}
hipError_t event_query(hipEvent_t) { return gate ? hipSuccess : hipErrorNotReady; }

} // namespace rec

#define launch_upload_scatter stub_upload_scatter
#define launch_export stub_export
#include "serve_stub_device.cpp"
#undef launch_upload_scatter
#undef launch_export

namespace hcm {

hipError_t launch_upload_scatter(const uint16_t *sblocks, const uint8_t *slight, const int8_t *sheights,
                                 const uint2 *moves, uint32_t n, uint16_t *blocks, uint8_t *light, int8_t *heights,
                                 hipStream_t st) {
	if (n) {
		rec::Scatter s{st, sblocks, slight, sheights, {}};
		for (uint32_t i = 0; i < n; ++i)
			s.slots.push_back(moves[i].y);
		std::lock_guard<std::mutex> lk(rec::mu);
		rec::scatters.push_back(s);
	}
	return stub_upload_scatter(sblocks, slight, sheights, moves, n, blocks, light, heights, st);
}
hipError_t launch_export(const ExportParams &p, hipStream_t st) {
	if (!p.ctr) {
		std::lock_guard<std::mutex> lk(rec::mu);
		rec::exports.push_back(st);
	}
	return stub_export(p, st);
}

} // namespace hcm

#define hipHostMalloc rec::host_malloc
#define hipMemcpyAsync rec::memcpy_async
#define hipStreamSynchronize rec::stream_synchronize
#define hipEventQuery rec::event_query
#include "hcm_serve.cpp"

static int g_fail = 0;
#define CHECK(c)                                                                                                   \
	do {                                                                                                           \
		if (!(c)) {                                                                                                \
			std::fprintf(stderr, "check failed at %s:%d: %s\n", __FILE__, __LINE__, #c);                           \
			++g_fail;                                                                                              \
		}                                                                                                          \
	} while (0)

struct World { // 3 x 3 x 3 chunks: one that is meshed
	hcm_server *s = nullptr;
	uint32_t mode;
	explicit World(uint32_t light_mode) : mode(light_mode) {
		hcm_server_config cfg{};
		cfg.max_chunks = 64, cfg.max_batch = 64, cfg.max_inflight = 1, cfg.pool_quads = 1u << 12, cfg.light_mode = mode;
		int ctx = 0;
		CHECK(hcm_server_create(reinterpret_cast<hcm_ctx *>(&ctx), &cfg, &s) == HCM_OK);
		for (int k = 0; k < 27; ++k)
			load(k / 9 - 1, k / 3 % 3 - 1, k % 3 - 1, 1);
		CHECK(hcm_server_drain(s) == HCM_OK);
		rec::clear();
	}
	~World() { hcm_server_destroy(s); }
	void load(int x, int y, int z, uint16_t block) {
		const std::vector<uint16_t> b(HCM_CHUNK_VOXELS, block);
		const std::vector<uint8_t> l(HCM_CHUNK_VOXELS, 15);
		const std::vector<int8_t> h(256, 3);
		CHECK((mode == HCM_LIGHT_REBUILD ? hcm_server_load_sunlit(s, x, y, z, b.data(), h.data(), 0)
		                                 : hcm_server_load(s, x, y, z, b.data(), l.data(), 0)) == HCM_OK);
	}
	void wait_uploads(size_t n) { // until the scheduler has taken in requests that leave n uploads pending
		for (;;) {
			{
				std::lock_guard<std::mutex> lk(s->world_mu);
				if (s->uploads.size() == n && s->any_busy())
					return;
			}
			std::this_thread::sleep_for(std::chrono::microseconds(100));
		}
	}
	uint32_t center_block() {
		std::vector<uint32_t> v(2 << 10);
		std::vector<uint16_t> i(1 << 10);
		hcm_mesh_desc m[4];
		hcm_host_result out{};
		out.vertices = reinterpret_cast<uint32_t(*)[2]>(v.data()), out.vertex_capacity = 1 << 10;
		out.indices = i.data(), out.index_capacity = 1 << 10, out.meshes = m, out.mesh_capacity = 4;
		CHECK(hcm_server_chunk_mesh(s, 0, 0, 0, &out) == HCM_OK && out.vertex_count);
		return v[0] & 0xffffu;
	}
};

// A chunk is read back on a stream of its own, without waiting for uploads or batches, and not at all when the caller's
// buffers are too small.
static void check_read_back(uint32_t mode) {
	World w(mode);
	std::vector<uint32_t> v(2 << 10);
	std::vector<uint16_t> i(1 << 10);
	hcm_mesh_desc m[4];
	hcm_host_result out{};
	out.vertices = reinterpret_cast<uint32_t(*)[2]>(v.data()), out.vertex_capacity = 3;
	out.indices = i.data(), out.index_capacity = 1 << 10, out.meshes = m, out.mesh_capacity = 4;
	const uint32_t quads = hcm::toy_quads(std::vector<uint16_t>(HCM_CHUNK_VOXELS, 1).data());
	CHECK(hcm_server_chunk_mesh(w.s, 0, 0, 0, &out) == HCM_ERR_CAPACITY);
	CHECK(out.vertex_count == 4 * quads && out.index_count == 6 * quads && out.mesh_count == 1);
	CHECK(rec::exports.empty() && rec::syncs.empty());
	CHECK(w.center_block() == 1);
	CHECK(rec::exports.size() == 1 && rec::syncs == rec::exports);
	CHECK(rec::exports[0] != w.s->s_copy && rec::exports[0] != w.s->s_comp);
}

// A chunk that is loaded again and again before a batch takes the loads: the last one counts, and no launch writes a slot
// twice (its workgroups run in any order).
static void check_repeated_loads(uint32_t mode) {
	World w(mode);
	rec::gate = false;
	w.load(0, 0, 0, 2); // goes ahead alone; the others gather behind it
	w.wait_uploads(0);
	for (uint16_t block : {3, 4, 5}) {
		w.load(0, 0, 0, block);
		w.load(0, 1, 0, block);
		w.load(5, 5, 5, block); // the first of these is a first load
	}
	w.wait_uploads(9);
	rec::clear();
	rec::gate = true;
	CHECK(hcm_server_drain(w.s) == HCM_OK);
	size_t n = 0;
	for (rec::Scatter &s : rec::scatters) {
		n += s.slots.size();
		std::sort(s.slots.begin(), s.slots.end());
		CHECK(std::adjacent_find(s.slots.begin(), s.slots.end()) == s.slots.end());
	}
	CHECK(n == 4); // three chunks, one of them also for the first time
	CHECK(w.center_block() == 5);
}

int main() {
	for (uint32_t mode : {HCM_LIGHT_STORE, HCM_LIGHT_REBUILD})
		check_read_back(mode), check_repeated_loads(mode);
	if (g_fail)
		return 1;
	std::printf("serve_streams_check: all checks passed\n");
	return 0;
}
