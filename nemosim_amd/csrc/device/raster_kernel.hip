/*
 * raster_kernel.hip -- the fired neurons of a run, from its bit raster to
 * counts per cycle and lists of user indices (the form nemo_step reports,
 * src/nemo/FiringBuffer.cpp, for every cycle of a run).
 *
 * What bounds it: for long runs the ids, which leave over PCIe and are copied
 * into the caller's buffer (6 MB for 1000 cycles of 200k neurons at 8 Hz, 0.45
 * ms; the raster itself, 25 MB, is read in 10 us); for short ones the launches
 * and the wait. The kernels report to host memory, where the caller polls, and
 * the second follows the first without the host. Decoded on the host, with the
 * whole raster copied back and walked bit by bit, 200k x 1000 cycles took 26.8
 * ms per nemosim_amd.Simulation.read_fired(), 50k x 1000 6.7 ms.
 */
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "host_report.h"
#include "step_abi.h"

namespace {

constexpr uint32_t BLOCK = 256u;
constexpr uint32_t WAVES = BLOCK / 64u;

/* word w with the bits of neurons >= n cleared */
__device__ inline uint64_t fired_word(const uint64_t* row, uint32_t w, uint32_t words, uint32_t n)
{
	if(w >= words || w * 64u >= n) return 0ull;
	const uint64_t b = row[w];
	const uint32_t left = n - w * 64u;
	return left >= 64u ? b : b & ((1ull << left) - 1ull);
}

/* One block per cycle: counts[t] = fired neurons of cycle t (host memory).
 * With offs the last block to finish also writes the exclusive prefix of the
 * counts there. */
__global__ void __launch_bounds__(BLOCK) raster_count_kernel(const uint64_t* raster, uint32_t words, uint32_t n,
		uint32_t* counts, uint32_t* devCounts, uint64_t* offs, DoneReport report)
{
	__shared__ uint64_t wsum[WAVES];
	__shared__ bool last;
	const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
	const uint64_t* row = raster + size_t(blockIdx.x) * words;
	uint32_t c = 0;
	for(uint32_t w = tid; w < words; w += BLOCK) {
		c += uint32_t(__popcll(fired_word(row, w, words, n)));
	}
	for(uint32_t d = 32; d >= 1; d >>= 1) c += __shfl_down(c, d, 64);
	if(lane == 0u) wsum[wave] = c;
	__syncthreads();
	if(tid == 0) {
		for(uint32_t k = 1; k < WAVES; ++k) c += uint32_t(wsum[k]);
		st_host(counts + blockIdx.x, c);
		if(offs) __hip_atomic_store(devCounts + blockIdx.x, c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
	}
	const bool l = last_block(report.done, blockIdx.x, gridDim.x);
	if(tid == 0) last = l;
	__syncthreads();
	if(!last) return;   /* block-uniform */
	if(offs) {
		/* each thread a contiguous share of the cycles */
		const uint32_t share = (gridDim.x + BLOCK - 1u) / BLOCK;
		const uint32_t t0 = min(gridDim.x, tid * share), t1 = min(gridDim.x, t0 + share);
		auto count = [&](uint32_t t) {
			return __hip_atomic_load(devCounts + t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
		};
		uint64_t mine = 0;
		for(uint32_t t = t0; t < t1; ++t) mine += count(t);
		uint64_t x = mine;
		for(uint32_t d = 1; d < 64u; d <<= 1) {
			const uint64_t y = __shfl_up((unsigned long long) x, d, 64);
			if(lane >= d) x += y;
		}
		if(lane == 63u) wsum[wave] = x;
		__syncthreads();
		x -= mine;
		for(uint32_t k = 0; k < wave; ++k) x += wsum[k];
		for(uint32_t t = t0; t < t1; ++t) {
			offs[t] = x;
			x += count(t);
		}
	}
	if(tid == 0) st_host(report.seen, report.sequence);
}

/* One block per cycle. The cycle's ids have positions offs[t], offs[t]+1, ...
 * in the run's list; those in [lo, hi) go to out[position - lo]. Each pass
 * takes 256 words, ranks their bits by a block scan and lists them in LDS, so
 * that the writes to host memory are whole lines whatever the firing rate:
 * written by the lanes that find them they are 4-byte PCIe writes once words
 * hold several bits. */
__global__ void __launch_bounds__(BLOCK) raster_ids_kernel(const uint64_t* raster, uint32_t words, uint32_t n,
		const uint64_t* offs, uint64_t lo, uint64_t hi, const uint32_t* ids, uint32_t first, uint32_t* out,
		DoneReport report)
{
	__shared__ uint16_t list[BLOCK * 64u];
	__shared__ uint32_t wsum[WAVES];
	const uint32_t lane = threadIdx.x & 63u;
	const uint32_t wave = threadIdx.x >> 6;
	const uint64_t* row = raster + size_t(blockIdx.x) * words;
	uint64_t pos = offs[blockIdx.x];
	for(uint32_t w0 = 0; w0 < words && pos < hi; w0 += BLOCK) {   /* block-uniform */
		uint64_t b = fired_word(row, w0 + threadIdx.x, words, n);
		const uint32_t c = uint32_t(__popcll(b));
		uint32_t x = c;
		for(uint32_t d = 1; d < 64u; d <<= 1) {
			const uint32_t y = __shfl_up(x, d, 64);
			if(lane >= d) x += y;
		}
		if(lane == 63u) wsum[wave] = x;
		__syncthreads();
		uint32_t before = 0, total = 0;
		for(uint32_t k = 0; k < WAVES; ++k) {
			before += (k < wave) ? wsum[k] : 0u;
			total += wsum[k];
		}
		uint32_t at = before + x - c;
		while(b) {
			list[at++] = uint16_t(threadIdx.x * 64u + uint32_t(__ffsll((unsigned long long) b) - 1));
			b &= b - 1ull;
		}
		__syncthreads();
		for(uint32_t i = threadIdx.x; i < total; i += BLOCK) {
			const uint64_t p = pos + i;
			if(p >= lo && p < hi) {
				const uint32_t l = w0 * 64u + list[i];
				st_host(out + (p - lo), ids ? ids[l] : first + l);
			}
		}
		__syncthreads();   /* the list and the sums are written again by the next pass */
		pos += total;
	}
	report_done(report, blockIdx.x, gridDim.x);
}

__global__ void peek_kernel(const uint32_t* src, uint32_t* out, DoneReport report)
{
	st_host(out, *src);
	__builtin_amdgcn_s_waitcnt(0);
	st_host(report.seen, report.sequence);
}

} // namespace

extern "C" {

int nemo_dev_raster_count(const uint64_t* raster, uint32_t words, uint32_t n, uint32_t cycles, uint32_t* counts,
		uint32_t* devCounts, uint64_t* offs, const DoneReport* report, void* stream)
{
	hipLaunchKernelGGL(raster_count_kernel, dim3(cycles), dim3(BLOCK), 0, static_cast<hipStream_t>(stream),
			raster, words, n, counts, devCounts, offs, *report);
	return int(hipGetLastError());
}

int nemo_dev_raster_ids(const uint64_t* raster, uint32_t words, uint32_t n, uint32_t cycles, const uint64_t* offs,
		uint64_t lo, uint64_t hi, const uint32_t* ids, uint32_t first, uint32_t* out, const DoneReport* report,
		void* stream)
{
	hipLaunchKernelGGL(raster_ids_kernel, dim3(cycles), dim3(BLOCK), 0, static_cast<hipStream_t>(stream),
			raster, words, n, offs, lo, hi, ids, first, out, *report);
	return int(hipGetLastError());
}

int nemo_dev_peek(const uint32_t* src, uint32_t* out, const DoneReport* report, void* stream)
{
	hipLaunchKernelGGL(peek_kernel, dim3(1), dim3(1), 0, static_cast<hipStream_t>(stream), src, out, *report);
	return int(hipGetLastError());
}

} // extern "C"
