/*
 * cycle_kernel.hip -- one cycle of a network the fused kernel holds
 * (step_kernel.hip), without its fixed cost: that kernel restores and saves
 * the whole ring of pending current around its cycles (2 x 32 MB at 100k
 * neurons and 20 delays), and its workgroups wait for each other once per
 * cycle. A single nemo_step pays all of it for one cycle.
 *
 * Here each workgroup takes 256 neurons, reads and clears their entries of the
 * cycle's ring slot in memory, updates them, and adds the synapses of those
 * that fired into the slots t+1 .. t+D with global atomics. The ring in memory
 * has D+1 slots (slot of cycle t: t mod (D+1)), so that none of them is slot
 * t, which other workgroups may still be reading: a cycle is one launch, with
 * nothing to wait for. Networks with STDP (whose fired lists and reverse rows
 * of past cycles the fused kernel keeps) and with sums that may leave int32
 * (whose overflow its LDS atomics detect) run on the fused kernel.
 *
 * The last workgroup to finish says so in host memory, where the caller polls:
 * a stream synchronisation takes 5 us more, its two timing events 4 us, each
 * copy of results 3 us.
 *
 * What bounds it: the launch and the chain ring slot -> update -> row bounds ->
 * records -> atomics; at high rates the atomics (about 23e9 per second).
 */
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "host_report.h"
#include "models.h"
#include "step_abi.h"

using namespace nemo_dev;

namespace {

constexpr uint32_t BLOCK = 256u;
/* Neurons per workgroup: 64 while that leaves all workgroups resident at once
 * (all four waves deliver what the one wave's neurons fire), 256 beyond */
constexpr uint32_t SMALL = 65536u;
constexpr uint32_t MAX_ROW = 5u;      /* bounds of a row per lane read ahead: P < 320 */
constexpr uint32_t WAVES = BLOCK / 64u;
constexpr uint32_t OFF_MASK_DEFER = (1u << 28) - 1u;   /* bits 28..31 of off[]: delay-1 records */

__host__ __device__ inline uint32_t neurons_per_block(uint32_t neurons)
{
	return neurons <= SMALL ? 64u : BLOCK;
}

/* Dynamic LDS: a source's bucket bounds for each wave. 64 KB is what a launch
 * takes without asking for more; 4 KB are for the kernel's own variables. */
constexpr uint32_t LDS_DYNAMIC = 60u * 1024u;

__host__ inline uint64_t dynamic_lds(uint32_t P)
{
	return uint64_t(WAVES) * (uint64_t(P) + 1u) * 4u;
}

/* the end of the launch, and the report */
__device__ inline void finish_cycle(const CycleArgs& ca)
{
	if(last_block(ca.done, blockIdx.x, gridDim.x)) {
		st_host(&ca.report->end, (uint64_t) wall_clock64());
		__builtin_amdgcn_s_waitcnt(0);
		st_host(&ca.report->sequence, ca.sequence);
	}
}

template<bool IZO>
__global__ void __launch_bounds__(BLOCK) nemo_cycle_kernel(const NetDev nd, const CycleArgs ca)
{
	constexpr int NP = IZO ? 5 : MAX_PARAM;
	constexpr int NS = IZO ? 2 : MAX_STATE;
	extern __shared__ uint32_t rows[];          /* [WAVES][P+1] bucket bounds of a wave's source */
	__shared__ float ext[BLOCK];
	__shared__ uint32_t fst[BLOCK / 32u];
	__shared__ uint32_t list[BLOCK];
	__shared__ uint32_t wfired[WAVES];
	__shared__ uint64_t wmask[WAVES];
	const uint32_t tid = threadIdx.x;
	const uint32_t lane = tid & 63u;
	const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	const uint32_t n = nd.n, T = nd.T, P = nd.P, R = nd.D + 1u;
	const uint32_t nb = neurons_per_block(P * T);
	const uint32_t first = blockIdx.x * nb;
	const uint32_t l = tid < nb ? first + tid : ~0u;
	const uint32_t p = (first + wave * 64u) / T;   /* T is a multiple of 64: one partition per wave */
	const uint32_t tl = l - p * T;
	if(l == 0) st_host(&ca.report->start, (uint64_t) wall_clock64());

	/* the cycle's stimulus */
	const bool stim = ca.nf > 0u || ca.ni > 0u;
	if(stim) {
		ext[tid] = 0.0f;
		if(tid < BLOCK / 32u) fst[tid] = 0u;
		__syncthreads();
		static_assert(NEMO_CYCLE_STIM <= BLOCK, "a thread per entry");
		if(tid < ca.nf) {
			const uint32_t x = ca.fidx[tid] - first;
			if(x < nb) atomicOr(&fst[x >> 5], 1u << (x & 31u));
		}
		if(tid < ca.ni) {   /* one entry per neuron */
			const uint32_t x = ca.iidx[tid] - first;
			if(x < nb) ext[x] = ca.ival[tid];
		}
		__syncthreads();
	}

	bool fired = false;
	if(l < n) {
		int32_t* pe = nd.ring + (size_t(p) * 2u * R + ca.slot) * T + tl;
		int32_t* pi = pe + size_t(R) * T;
		const int32_t e = *pe, i = *pi;
		float prm[NP], st[NS];
#pragma unroll
		for(int q = 0; q < NP; ++q) prm[q] = nd.param[size_t(q) * n + l];
#pragma unroll
		for(int q = 0; q < NS; ++q) st[q] = nd.state[size_t(q) * n + l];
		Rng r;
#pragma unroll
		for(int q = 0; q < 4; ++q) r.s[q] = nd.rng[size_t(q) * n + l];
		const uint64_t recent = nd.recent[l];
		const float cx = stim ? ext[tid] : 0.0f;
		const bool fs = stim && ((fst[tid >> 5] >> (tid & 31u)) & 1u) != 0u;
		*pe = 0;
		*pi = 0;
		if(IZO) {
			fired = izhikevich(prm, st, r, fx20_to_float(e), fx20_to_float(i), cx, fs);
		} else {
			fired = update_neuron(nd.model[l], prm, st, r, fx20_to_float(e), fx20_to_float(i), cx, fs);
		}
#pragma unroll
		for(int q = 0; q < NS; ++q) nd.state[size_t(q) * n + l] = st[q];
#pragma unroll
		for(int q = 0; q < 4; ++q) nd.rng[size_t(q) * n + l] = r.s[q];
		nd.recent[l] = (recent << 1) | (fired ? 1ull : 0ull);
	}

	const uint64_t mask = __ballot(fired);
	if(lane == 0) {
		const uint32_t word = l >> 6;
		if(word < nd.words) {
			nd.raster[word] = mask;
		}
		wmask[wave] = mask;
		wfired[wave] = uint32_t(__popcll(mask));
	}
	__syncthreads();
	/* the workgroup's words to the host in one write: over PCIe, and for the
	 * host's cache, four of 8 bytes cost four times as much (step() of 100k x 100
	 * 38 -> 33 us, 200k x 100 56 -> 43) */
	if(tid < nb / 64u && first / 64u + tid < nd.words) st_host(ca.hostRow + first / 64u + tid, wmask[tid]);
	uint32_t before = 0, total = 0;
#pragma unroll
	for(uint32_t w = 0; w < WAVES; ++w) {
		before += (w < wave) ? wfired[w] : 0u;
		total += wfired[w];
	}
	if(total == 0u) {   /* block-uniform */
		finish_cycle(ca);
		return;
	}
	if(fired) {
		const uint64_t below = lane ? (mask & (~0ull >> (64u - lane))) : 0ull;
		list[before + uint32_t(__popcll(below))] = l;
	}
	__syncthreads();

	/* delivery: the (source, chunk of 256 records) items of the workgroup, dealt
	 * to its waves in turn, four records per lane. A record's target is within
	 * its partition, found by a search of the source's bucket bounds; bounds
	 * and records are read together. */
	const uint32_t offMask = (nd.flags & NEMO_NET_DEFER) ? OFF_MASK_DEFER : ~0u;
	const uint2* syn = reinterpret_cast<const uint2*>(nd.syn);
	uint32_t* row = rows + wave * (P + 1u);
	const uint32_t top = P > 1u ? 1u << (31u - uint32_t(__builtin_clz(P - 1u))) : 0u;
	uint32_t turn = 0;
	for(uint32_t j0 = 0; j0 < total; j0 += 64u) {
		uint32_t ra = 0, rb = 0;     /* rows of 64 sources, one per lane */
		if(j0 + lane < total) {
			const uint32_t* o = nd.off + size_t(list[j0 + lane]) * (P + 1u);
			ra = o[0] & offMask;
			rb = o[P] & offMask;
		}
		const uint32_t cnt = min(64u, total - j0);
		for(uint32_t j = 0; j < cnt; ++j) {
			const uint32_t a = uint32_t(__builtin_amdgcn_readlane(int(ra), int(j)));
			const uint32_t b = uint32_t(__builtin_amdgcn_readlane(int(rb), int(j)));
			bool have = false;       /* the bounds of this source are in LDS */
			for(uint32_t c = a; c < b; c += 256u, ++turn) {   /* wave-uniform */
				if((turn & 3u) != wave) continue;
				uint2 rec[4];
				uint32_t q[4];
#pragma unroll
				for(uint32_t u = 0; u < 4u; ++u) {
					const uint32_t x = c + 64u * u + lane;
					rec[u] = (x < b) ? syn[x] : make_uint2(0u, 0u);
					q[u] = 0u;
				}
				if(!have) {
					const uint32_t* o = nd.off + size_t(list[j0 + j]) * (P + 1u);
					uint32_t v[MAX_ROW];
#pragma unroll
					for(uint32_t k = 0; k < MAX_ROW; ++k) v[k] = (64u * k + lane <= P) ? o[64u * k + lane] : 0u;
#pragma unroll
					for(uint32_t k = 0; k < MAX_ROW; ++k) {
						if(64u * k + lane <= P) row[64u * k + lane] = v[k] & offMask;
					}
					for(uint32_t i = 64u * MAX_ROW + lane; i <= P; i += 64u) row[i] = o[i] & offMask;
					have = true;
				}
				__builtin_amdgcn_wave_barrier();   /* a wave's LDS operations complete in order */
				for(uint32_t s = top; s; s >>= 1) {   /* the last q with row[q] <= x */
#pragma unroll
					for(uint32_t u = 0; u < 4u; ++u) {
						const uint32_t m = q[u] + s;
						if(m < P && row[m] <= c + 64u * u + lane) q[u] = m;
					}
				}
				__builtin_amdgcn_wave_barrier();   /* the row is written again */
#pragma unroll
				for(uint32_t u = 0; u < 4u; ++u) {
					if(c + 64u * u + lane < b) {
						const int32_t w = int32_t(rec[u].y);
						uint32_t sl = ca.slot + (rec[u].x >> 16);
						sl = (sl >= R) ? sl - R : sl;
						const uint32_t plane = (w >= 0) ? 0u : R;
						atomicAdd(nd.ring + (size_t(q[u]) * 2u * R + plane + sl) * T + (rec[u].x & 0xffffu), w);
					}
				}
			}
		}
	}
	finish_cycle(ca);
}

__global__ void __launch_bounds__(BLOCK) longest_row_kernel(const uint32_t* off, uint32_t stride, uint32_t n, uint32_t mask,
		uint32_t* max, uint32_t* done, uint32_t* out)
{
	uint32_t most = 0;
	for(uint32_t i = blockIdx.x * BLOCK + threadIdx.x; i < n; i += gridDim.x * BLOCK) {
		const uint32_t a = off[size_t(i) * stride] & mask, b = off[(size_t(i) + 1u) * stride] & mask;
		most = b - a > most ? b - a : most;
	}
	for(uint32_t d = 32; d >= 1; d >>= 1) {
		const uint32_t x = __shfl_down(most, d, 64);
		most = x > most ? x : most;
	}
	if((threadIdx.x & 63u) == 0u) atomicMax(max, most);
	if(last_block(done, blockIdx.x, gridDim.x)) {
		st_host(out, __hip_atomic_load(max, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
	}
}

} // namespace

extern "C" {

int nemo_dev_longest_row(const uint32_t* off, uint32_t stride, uint32_t n, uint32_t mask, uint32_t* max, uint32_t* done,
		uint32_t* out, void* stream)
{
	const uint32_t blocks = n > 256u * BLOCK ? 256u : (n + BLOCK - 1u) / BLOCK;
	hipLaunchKernelGGL(longest_row_kernel, dim3(blocks), dim3(BLOCK), 0, static_cast<hipStream_t>(stream),
			off, stride, n, mask, max, done, out);
	return int(hipGetLastError());
}

uint32_t nemo_dev_cycle_block_neurons(uint32_t P, uint32_t T)
{
	return neurons_per_block(P * T);
}

int nemo_dev_cycle_fits(uint32_t P)
{
	return dynamic_lds(P) <= LDS_DYNAMIC ? 1 : 0;
}

int nemo_dev_cycle(const NetDev* nd, const CycleArgs* ca, void* stream)
{
	if(!nemo_dev_cycle_fits(nd->P)) return int(hipErrorInvalidValue);
	const uint32_t nb = neurons_per_block(nd->P * nd->T);
	const uint32_t blocks = (nd->P * nd->T + nb - 1u) / nb;
	const uint32_t lds = uint32_t(dynamic_lds(nd->P));
	auto kernel = (nd->flags & NEMO_NET_IZHIKEVICH_ONLY) ? &nemo_cycle_kernel<true> : &nemo_cycle_kernel<false>;
	hipLaunchKernelGGL(kernel, dim3(blocks), dim3(BLOCK), lds, static_cast<hipStream_t>(stream), *nd, *ca);
	return int(hipGetLastError());
}

} // extern "C"
