// hcm_device.h -- device code that several of the gfx950 kernels use.
#pragma once

#include "hcm_internal.h"

namespace hcm {

// One step of four 8 x 8 bit transpositions (one per byte) over eight words: bits and words whose index
// differs in D change places. (A template argument: the steps in a loop were not unrolled.)
template <int D> __device__ __forceinline__ void exchange_bits(uint32_t r[8]) {
	constexpr uint32_t m = D == 4 ? 0x0f0f0f0fu : (D == 2 ? 0x33333333u : 0x55555555u); // bits without D
#pragma unroll
	for (int i = 0; i < 8; ++i)
		if (!(i & D)) {
			const uint32_t a = r[i], b = r[i + D];
			r[i] = (a & m) | ((b << D) & ~m);
			r[i + D] = ((a >> D) & m) | (b & ~m);
		}
}

// The jobs of one workgroup of a persistent launch, by one lane. It lies in LDS: in registers, everything that follows
// from the numbers of jobs and workgroups was computed ahead of the loop over jobs and spilled (281
// moves from spilled scalars in the mesh kernel, 144 so: 4,096 cave chunks 77.1 us, 75.9 so).
struct JobClaims {
	uint32_t n_jobs, block, grid, tried, first;
	__device__ void init(uint32_t n) { n_jobs = n, block = blockIdx.x, grid = gridDim.x, tried = 0, first = 1; }
	__device__ uint32_t part(uint32_t q) const { return uint32_t(uint64_t(q) * n_jobs / kQueues); }
	// The next job, or ~0. A part is left for the next one once its counter has passed its end; whoever finds
	// that out first sets its bit in `dry`, so that a workgroup that runs out of its own part's jobs reads one
	// word instead of failing a claim in every other part: eight failed claims of 768 workgroups, one after
	// another, were 26 us of every launch, that of one job too (a 37-chunk batch: 57 us).
	__device__ uint32_t next(Counters *ctr) {
		const uint32_t home = block % kQueues, turn = block / kQueues;
		if (grid >= n_jobs) { // one job each: parts as long as the XCDs have workgroups, and no claims
			const uint32_t len = n_jobs / kQueues, more = n_jobs % kQueues; // the first `more` parts hold one more
			const bool mine = first && turn < len + (home < more ? 1u : 0u);
			first = 0;
			return mine ? home * len + min(home, more) + turn : ~0u;
		}
		if (first) {
			first = 0;
			const uint32_t job = part(home) + turn;
			if (job < part(home + 1))
				return job;
		}
		uint32_t dry = 0;
		for (; tried < kQueues; ++tried) {
			const uint32_t q = (home + tried) % kQueues, lo = part(q), len = part(q + 1) - lo;
			const uint32_t given = (grid - q + kQueues - 1) / kQueues; // its workgroups
			if (given >= len || ((dry >> q) & 1u))
				continue;
			const uint32_t k = given + atomicAdd(&ctr->queue[q].v, 1u);
			if (k < len)
				return lo + k;
			if (k == len)
				atomicOr(&ctr->dry.v, 1u << q); // (awaited by claims_returned)
			dry = atomicOr(&ctr->dry.v, 0u);
		}
		return ~0u;
	}
};

// Waits until every atomic that this wavefront has issued on the counters has been performed, before the workgroup counts
// as done and the last one clears them: JobClaims::next discards the result of the one that marks a part as dry, and a
// mark that landed after the clearing would keep the next launch's workgroups from the jobs of that part. (The wait
// instead of a use of the results in next(), by which 4,096 cave chunks took 77.4 us instead of 74.8.)
__device__ __forceinline__ void claims_returned() { __builtin_amdgcn_s_waitcnt(0); }

} // namespace hcm
