/*
 * raster_kernel.hip -- the fired neurons of a run, from its bit raster to
 * counts per cycle and lists of user indices (the form nemo_step reports,
 * src/nemo/FiringBuffer.cpp, for every cycle of a run).
 *
 * What bounds it: the raster is read once per call (25 MB for 1000 cycles of
 * 200k neurons, ~10 us), the ids leave over PCIe, and the host copies them
 * into the caller's buffer. Decoded on the host, with the whole raster copied
 * back and walked bit by bit, 200k x 1000 cycles took 26.8 ms per
 * nemosim_amd.Simulation.read_fired(), 50k x 1000 6.7 ms.
 */
#include <hip/hip_runtime.h>
#include <stdint.h>

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

/* one block per cycle: counts[t] = fired neurons of cycle t (host memory) */
__global__ void __launch_bounds__(BLOCK) raster_count_kernel(const uint64_t* raster, uint32_t words, uint32_t n,
		uint32_t* counts)
{
	__shared__ uint32_t wsum[WAVES];
	const uint64_t* row = raster + size_t(blockIdx.x) * words;
	uint32_t c = 0;
	for(uint32_t w = threadIdx.x; w < words; w += BLOCK) {
		c += uint32_t(__popcll(fired_word(row, w, words, n)));
	}
	for(uint32_t d = 32; d >= 1; d >>= 1) c += __shfl_down(c, d, 64);
	if((threadIdx.x & 63u) == 0u) wsum[threadIdx.x >> 6] = c;
	__syncthreads();
	if(threadIdx.x == 0) {
		for(uint32_t k = 1; k < WAVES; ++k) c += wsum[k];
		counts[blockIdx.x] = c;
	}
}

/* One block per cycle. The cycle's ids have positions offs[t], offs[t]+1, ...
 * in the run's list; those in [lo, hi) go to out[position - lo]. Each pass
 * takes 256 words, ranks their bits by a block scan and lists them in LDS, so
 * that the writes to host memory are whole lines whatever the firing rate:
 * written by the lanes that find them they are 4-byte PCIe writes once words
 * hold several bits. */
__global__ void __launch_bounds__(BLOCK) raster_ids_kernel(const uint64_t* raster, uint32_t words, uint32_t n,
		const uint64_t* offs, uint64_t lo, uint64_t hi, const uint32_t* ids, uint32_t first, uint32_t* out)
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
				out[p - lo] = ids ? ids[l] : first + l;
			}
		}
		__syncthreads();   /* the list and the sums are written again by the next pass */
		pos += total;
	}
}

} // namespace

extern "C" {

int nemo_dev_raster_count(const uint64_t* raster, uint32_t words, uint32_t n, uint32_t cycles, uint32_t* counts,
		void* stream)
{
	if(cycles == 0) return 0;
	hipLaunchKernelGGL(raster_count_kernel, dim3(cycles), dim3(BLOCK), 0, static_cast<hipStream_t>(stream),
			raster, words, n, counts);
	return int(hipGetLastError());
}

int nemo_dev_raster_ids(const uint64_t* raster, uint32_t words, uint32_t n, uint32_t cycles, const uint64_t* offs,
		uint64_t lo, uint64_t hi, const uint32_t* ids, uint32_t first, uint32_t* out, void* stream)
{
	if(cycles == 0 || lo >= hi) return 0;
	hipLaunchKernelGGL(raster_ids_kernel, dim3(cycles), dim3(BLOCK), 0, static_cast<hipStream_t>(stream),
			raster, words, n, offs, lo, hi, ids, first, out);
	return int(hipGetLastError());
}

} // extern "C"
