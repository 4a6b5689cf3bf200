/*
 * host_report.h -- how a kernel tells the host that it is done without a
 * stream synchronisation: its last workgroup writes to host memory, where the
 * caller polls (a launch and its wait take 6.5 us so, 11.5 us with
 * hipStreamSynchronize; a device-to-host copy of the results adds 3 us more).
 */
#ifndef NEMOSIM_HOST_REPORT_H
#define NEMOSIM_HOST_REPORT_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "step_abi.h"

namespace {

/* Stores to the caller's host memory: written through, so that s_waitcnt waits
 * until they are there */
template<typename V>
__device__ inline void st_host(V* p, V v)
{
	__hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

/* Counts the workgroup as finished, once its stores have landed. True in one
 * thread of the launch's last one. Two levels of counters, each in a line of
 * its own: one shared by hundreds of workgroups takes 10 ns for each. They
 * return to zero for the next launch. Called by whole workgroups. */
__device__ inline bool last_block(uint32_t* done, uint32_t block, uint32_t blocks)
{
	__builtin_amdgcn_s_waitcnt(0);
	__syncthreads();
	auto zero = [](uint32_t* c) {   /* there for a launch on another stream, too */
		__hip_atomic_store(c, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
		__builtin_amdgcn_s_waitcnt(0);
	};
	if(threadIdx.x == 0) {
		const uint32_t groups = min(blocks, NEMO_DONE_GROUPS);
		const uint32_t g = block % groups;
		const uint32_t mine = (blocks - g + groups - 1u) / groups;
		uint32_t* c = done + 32u * (g + 1u);
		if(atomicAdd(c, 1u) + 1u == mine) {
			zero(c);
			if(atomicAdd(done, 1u) + 1u == groups) {
				zero(done);
				return true;
			}
		}
	}
	return false;
}

__device__ inline void report_done(const DoneReport& r, uint32_t block, uint32_t blocks)
{
	if(last_block(r.done, block, blocks)) st_host(r.seen, r.sequence);
}

} // namespace

#endif
