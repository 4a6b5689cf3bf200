/*
 * Kuramoto.hip -- HIP plugin for Kuramoto phase oscillators
 * (lib<Kuramoto>.so, ABI in include/nemo_hip_plugin.h).
 *
 * The model of src/nemo/cpu/plugins/Kuramoto.cpp:85-123: each cycle, the
 * phase theta of an oscillator with natural frequency f moves by one
 * fourth-order Runge-Kutta step of
 *     d theta / dt = f + sum_j w_j sin(theta_j - theta),
 * where theta_j is the phase of source j at cycle t - (delay_j - 1), held
 * fixed over the four stages, and the result is wrapped into [0, 2*pi).
 * The arithmetic is the reference CPU plugin's, operation for operation, in
 * IEEE single precision without contraction (sums in reverse-matrix order,
 * the host C library's sinf restated in csrc/device/libm_f32.h, fmodf exact),
 * so the phases agree bit for bit with the CPU backend.
 *
 * A workgroup takes a tile of consecutive oscillators, whose rows of the
 * reverse matrix are contiguous: its threads evaluate the tile's coupling
 * terms into LDS, then a lane, or a row of 16, per oscillator adds its row's
 * terms in order.
 * Phase history: plane c mod 32 of the state holds the phase
 * of cycle c (the descriptor's history=32).
 */
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../csrc/device/libm_f32.h"
#include "nemo_hip_plugin.h"

namespace {

constexpr unsigned HISTORY = 32u;   /* history= of Kuramoto.ini */

constexpr unsigned THREADS = 256u;
constexpr unsigned TILE_OSC = 64u;            /* oscillators of a tile: at least a lane each in the sums */
/* A tile's rows in LDS start at multiples of 4 floats (16-byte reads), and at
 * least 65 zeros follow each: the sums run in steps of 64 terms, and adding
 * +0 leaves a sum that started from +0 as it is. */
constexpr unsigned STEP = 64u;
constexpr unsigned ROW_GAP = STEP + 4u;
constexpr unsigned RESIDENT = 1024u;          /* workgroups on the chip at once: 4 per compute unit */

/* couplings of a tile whose threads hold PER each, and its floats in LDS (the
 * sums read up to a step further) */
template<unsigned PER> struct Tile {
	static constexpr unsigned couplings = THREADS * PER;
	static constexpr unsigned half = PER > 9u ? 4u : 8u;   /* 16-byte reads per half step of the sums */
	static constexpr unsigned lds = couplings + ROW_GAP * TILE_OSC + STEP;
};

/* how much further row j starts in LDS than its first coupling's number
 * within the tile, off */
__device__ inline unsigned row_shift(unsigned off, unsigned j)
{
	return ((off + ROW_GAP * j) & ~3u) - off;
}

typedef float Quad __attribute__((ext_vector_type(4)));
#if defined(__HIP_DEVICE_COMPILE__)
typedef const volatile __attribute__((address_space(3))) Quad* LdsQuads;   /* volatile generic reads are flat ones */
#else
typedef const volatile Quad* LdsQuads;
#endif

/* s + row[0] + ... + row[len-1], each addition rounded to float, in that
 * order (the reference's sequential sum); the row is followed by zeros up to
 * the next multiple of STEP terms. The chain of dependent adds bounds a long
 * row (4.5 cycles each), so half a step is read while the half before is
 * added. The reads are volatile and the sum passes through empty asm between
 * them: left alone, the compiler gathers the reads at their use, and every
 * step waits for LDS (13 cycles a term). H: 16-byte reads per half step. */
template<unsigned H>
__device__ inline float ordered_sum(float s, const float* row, unsigned len)
{
	LdsQuads r4 = (LdsQuads) row;
	Quad a[H], b[H];
#pragma unroll
	for(unsigned q = 0; q < H; ++q) a[q] = r4[q];
	for(unsigned i = 0; i < len; i += 8u * H) {
#pragma unroll
		for(unsigned q = 0; q < H; ++q) b[q] = r4[H + q];
		asm volatile("" : "+v"(s));
#pragma unroll
		for(unsigned q = 0; q < H; ++q) {
			s = s + a[q].x;
			s = s + a[q].y;
			s = s + a[q].z;
			s = s + a[q].w;
		}
		asm volatile("" : "+v"(s));
		r4 += 2u * H;
#pragma unroll
		for(unsigned q = 0; q < H; ++q) a[q] = r4[q];
		asm volatile("" : "+v"(s));
#pragma unroll
		for(unsigned q = 0; q < H; ++q) {
			s = s + b[q].x;
			s = s + b[q].y;
			s = s + b[q].z;
			s = s + b[q].w;
		}
		asm volatile("" : "+v"(s));
	}
	return s;
}

/* The same by 16 lanes (a DPP row), all of which have the sum: they read a step
 * of 64 terms at once, 4 each, and every add takes its term from the lane that
 * has it. So a read of LDS goes with 64 adds instead of 4, and a term takes 6.3
 * cycles of a 1000-term row instead of 8.9 (4.8 without the loop around it). In assembly since
 * the compiler waits between DPP adds for the operand that is not moved, too;
 * the moved ones are not written here, and what may have written them, or the
 * lanes in use, just before is waited for at the start. */
#define ADD_LANE(L) \
	"v_add_f32_dpp %0, %1, %0 row_newbcast:" #L " row_mask:0xf bank_mask:0xf\n" \
	"v_add_f32_dpp %0, %2, %0 row_newbcast:" #L " row_mask:0xf bank_mask:0xf\n" \
	"v_add_f32_dpp %0, %3, %0 row_newbcast:" #L " row_mask:0xf bank_mask:0xf\n" \
	"v_add_f32_dpp %0, %4, %0 row_newbcast:" #L " row_mask:0xf bank_mask:0xf\n"

__device__ inline float ordered_sum_row(float s, const float* row, unsigned len, unsigned lane)
{
#if defined(__HIP_DEVICE_COMPILE__)
	LdsQuads r4 = (LdsQuads) row + lane;
	Quad v = r4[0];
	for(unsigned i = 0; i < len; i += STEP) {
		r4 += STEP / 4u;
		const Quad next = r4[0];
		asm volatile("s_nop 4\n"
				ADD_LANE(0) ADD_LANE(1) ADD_LANE(2) ADD_LANE(3) ADD_LANE(4) ADD_LANE(5) ADD_LANE(6) ADD_LANE(7)
				ADD_LANE(8) ADD_LANE(9) ADD_LANE(10) ADD_LANE(11) ADD_LANE(12) ADD_LANE(13) ADD_LANE(14) ADD_LANE(15)
				: "+v"(s) : "v"(v.x), "v"(v.y), "v"(v.z), "v"(v.w));
		v = next;
	}
#else
	(void) row; (void) len; (void) lane;
#endif
	return s;
}
#undef ADD_LANE

/* Where a workgroup's share starts if work is shared by couplings: the first of
 * the n oscillators whose rows, counted with OSC_COST couplings for each
 * oscillator, start at `target` or later. By one wave, in rounds of 64 probes. */
constexpr unsigned OSC_COST = 16u;

__device__ inline unsigned share_start(const uint32_t* rstart, unsigned n, uint64_t target, unsigned lane)
{
	const uint32_t first = rstart[0];
	unsigned lo = 0, hi = n;
	while(lo < hi) {   /* wave-uniform; the answer is in lo .. hi */
		const unsigned step = (hi - lo + 63u) / 64u;
		const unsigned o = lo + (lane + 1u) * step - 1u;
		const bool before = o < hi && uint64_t(rstart[o] - first) + uint64_t(OSC_COST) * o < target;
		const unsigned cnt = unsigned(__popcll(__ballot(before)));
		hi = min(hi, lo + (cnt + 1u) * step - 1u);
		lo += cnt * step;
	}
	return lo;
}

/* One workgroup per `per` consecutive oscillators, or, SHARED, per `quota`
 * couplings: with rows of very different lengths next to each other (hubs)
 * a workgroup of `per` would have many long rows, one after the other. Tiles of them whose rows
 * hold at most TILE = 256 PER couplings together are done one after the other (one tile,
 * unless rows are uneven); a row longer than TILE is a tile of its own and is
 * read in pieces, again for each stage, where the others stay in registers
 * over the four stages.
 *
 * What bounds it: with few and long rows the chains of dependent adds, 4
 * stages x row length x 4.5 cycles, so that as many of them as possible run at
 * once; with many oscillators the reads of the sources' phases (random, 32
 * planes) and the sines (about 30 instructions each). One cycle, with the
 * plugin step's other kernels (about 10 us), before (one wave per oscillator,
 * which evaluated 64 couplings at a time, every lane repeating the sum) and
 * now: 1000 oscillators x 1000 couplings 65 -> 28 us (33 with a lane's sums
 * alone), 4000 x 1000 101 -> 57, 2000 x 2500 182 -> 113, 3000 x 300 36 -> 21,
 * 20000 x 100 48 -> 31, 50000 x 100 99 -> 75. */
template<unsigned PER, bool SHARED = false>
__global__ void __launch_bounds__(256, 4) kuramoto_update_kernel(unsigned start, unsigned end, unsigned per,
		uint64_t quota, unsigned cycle, const float* freq, float* state, size_t hstride, const uint32_t* rstart,
		const uint32_t* src, const uint32_t* dly, const float* w)
{
	constexpr unsigned TILE = Tile<PER>::couplings;
	struct Row { float x; uint32_t shift; };  /* the stage's phase; row_shift */
	__shared__ __align__(16) float term[Tile<PER>::lds];
	__shared__ uint32_t rs[TILE_OSC + 1u];    /* row starts of the block's remaining oscillators */
	__shared__ Row rows[TILE_OSC];
	const unsigned tid = threadIdx.x;
	const float* phase0 = state + size_t(cycle % HISTORY) * hstride;
	float* phase1 = state + size_t((cycle + 1u) % HISTORY) * hstride;
	unsigned last = min(end - start, (blockIdx.x + 1u) * per);
	unsigned o = blockIdx.x * per;
	if(SHARED) {
		__shared__ unsigned share[2];
		const unsigned wave = tid >> 6;
		if(wave < 2u) {
			const unsigned at = share_start(rstart + start, end - start, quota * (blockIdx.x + wave), tid & 63u);
			if((tid & 63u) == 0u) share[wave] = at;
		}
		__syncthreads();
		o = share[0];
		last = share[1];
	}
	while(o < last) {   /* block-uniform */
		const unsigned left = min(last - o, TILE_OSC);
		if(tid <= left) rs[tid] = rstart[start + o + tid];
		__syncthreads();
		const uint32_t r0 = rs[0];
		unsigned nb = left;                                     /* oscillators of the tile */
		while(nb > 1u && rs[nb] - r0 > TILE) --nb;
		const uint32_t total = rs[nb] - r0;                     /* couplings of the tile */
		const uint32_t pieces = total <= TILE ? 1u : (total + TILE - 1u) / TILE;   /* > 1: one oscillator */
		const uint32_t used = min(TILE, total) + ROW_GAP * nb + STEP;   /* of `term` */
		for(unsigned i = tid; i < used; i += THREADS) term[i] = 0.0f;
		float f = 0.0f, theta = 0.0f, k0 = 0.0f, k1 = 0.0f, k2 = 0.0f, k3 = 0.0f;
		/* the lane of an oscillator, or with few of them the row of 16 lanes */
		const bool byRow = nb <= THREADS / 16u;
		const unsigned own = byRow ? tid / 16u : tid;
		const bool owner = own < nb;
		if(owner) {
			f = freq[o + own];
			theta = phase0[o + own];
			rows[own] = Row{theta, row_shift(rs[own] - r0, own)};
		}
		float sp[PER], wt[PER];
		uint32_t osc[(PER + 3u) / 4u];                          /* oscillators of the couplings, 8 bits each */
		for(unsigned stage = 0; stage < 4u; ++stage) {
			float s = 0.0f;
			for(uint32_t pc = 0; pc < pieces; ++pc) {
				const uint32_t base = pc * TILE;
				const uint32_t cnt = min(TILE, total - base);
				if(stage == 0u || pieces > 1u) {
#pragma unroll
					for(unsigned k = 0; k < PER; ++k) {
						const uint32_t i = k * THREADS + tid;
						if(k % 4u == 0u) osc[k / 4u] = 0u;
						sp[k] = 0.0f;
						wt[k] = 0.0f;
						if(i < cnt) {
							const uint32_t r = r0 + base + i;
							/* phase of the source at cycle t - (delay - 1) */
							const unsigned plane = (cycle - (dly[r] - 1u)) % HISTORY;
							sp[k] = state[size_t(plane) * hstride + (src[r] - start)];
							wt[k] = w[r];
							unsigned lo = 0, hi = nb;
							while(hi - lo > 1u) {
								const unsigned mid = (lo + hi) >> 1;
								if(rs[mid] <= r) lo = mid; else hi = mid;
							}
							osc[k / 4u] |= lo << (8u * (k % 4u));
						}
					}
				}
				__syncthreads();   /* the stage's phases are in `rows`; the last sums have read `term` */
				if(pieces > 1u && tid < STEP) term[cnt + tid] = 0.0f;   /* a shorter piece than the one before */
#pragma unroll
				for(unsigned k = 0; k < PER; ++k) {
					const uint32_t i = k * THREADS + tid;
					if(k * THREADS >= cnt) break;   /* block-uniform */
					if(i < cnt) {
						/* w * sin(theta_source - x), rounded to float (src/nemo/cpu/plugins/Kuramoto.cpp:18-29) */
						const Row row = rows[(osc[k / 4u] >> (8u * (k % 4u))) & 0xffu];
						term[i + row.shift] = wt[k] * nemo_libm::sinf_glibc(sp[k] - row.x);
					}
				}
				__syncthreads();
				if(owner) {
					const bool whole = pieces == 1u;
					const float* row = term + (whole ? rs[own] - r0 + rows[own].shift : 0u);
					const unsigned len = whole ? rs[own + 1u] - rs[own] : cnt;
					if(byRow) s = ordered_sum_row(s, row, len, tid & 15u);
					else s = ordered_sum<Tile<PER>::half>(s, row, len);
				}
			}
			if(owner) {
				const float k = f + s;
				if(stage == 0u) { k0 = k; rows[own].x = theta + k * 0.5f; }
				else if(stage == 1u) { k1 = k; rows[own].x = theta + k * 0.5f; }
				else if(stage == 2u) { k2 = k; rows[own].x = theta + k; }
				else { k3 = k; }
			}
		}
		if(owner) {
			const float next = theta + (k0 + 2.0f * k1 + 2.0f * k2 + k3) / 6.0f;
			phase1[o + own] = nemo_libm::kuramoto_wrap(next);
		}
		o += nb;
		__syncthreads();   /* rs, rows and term are written again by the next tile */
	}
}

/* Couplings per thread and oscillators per workgroup. A tile holds as many
 * oscillators as fit on average, with room for three standard deviations of
 * random rows, and the workgroups are whole rounds of RESIDENT. The smallest
 * tile with which all of them run at once is taken (fewer instructions and
 * registers: see the figures at the kernel); where none is large enough, the
 * middle one, in several rounds. */
struct Plan {
	unsigned per, threadCouplings;
	uint64_t quota;     /* couplings per workgroup; 0: `per` oscillators each */
	unsigned blocks;
};

Plan plan(unsigned n, const nemo_hip_rcm* rcm)
{
	const double avg = rcm->targets ? double(rcm->synapses) / double(rcm->targets) : 0.0;
	auto fit = [&](unsigned couplings) {
		unsigned b = TILE_OSC;
		while(b > 0u && double(b) * avg + 3.0 * __builtin_sqrt(double(b) * avg) > double(couplings)) --b;
		return b;
	};
	auto spread = [&](unsigned b) {
		const unsigned rounds = (n + RESIDENT * b - 1u) / (RESIDENT * b);
		return (n + RESIDENT * rounds - 1u) / (RESIDENT * rounds);
	};
	Plan p = { 1u, 18u, 0u, 0u };
	const unsigned mid = fit(THREADS * 9u);
	if(mid > 0u) p = Plan{ spread(mid), 9u, 0u, 0u };
	const unsigned sizes[3] = { 3u, 9u, 18u };
	for(unsigned c : sizes) {
		const unsigned b = fit(THREADS * c);
		if(b > 0u && n <= RESIDENT * b) {
			p = Plan{ spread(b), c, 0u, 0u };
			break;
		}
	}
	p.blocks = (n + p.per - 1u) / p.per;
	/* Shared by couplings where the longest rows, next to each other, could make
	 * a workgroup's share several tiles, and are several times the average, as
	 * those of random networks are not: two or three rounds of reads more before the
	 * first tile, two thirds of a tile per workgroup on average. 20000 x 30 with 20
	 * neighbours of 15000 couplings each: 4311 us per cycle in shares of 20
	 * oscillators, 240 so. */
	const uint64_t longest = rcm->longest;
	if(p.per > 1u && double(longest) > 4.0 * avg && longest * p.per > 2u * THREADS * p.threadCouplings) {
		const uint64_t work = uint64_t(rcm->synapses) + uint64_t(OSC_COST) * n + 1u;
		const uint64_t most = THREADS * 9u * 2u / 3u;
		p.threadCouplings = 9u;
		p.blocks = unsigned(RESIDENT * ((work + RESIDENT * most - 1u) / (RESIDENT * most)));
		p.quota = (work + p.blocks - 1u) / p.blocks;
	}
	return p;
}

/* src/nemo/cpu/plugins/Kuramoto.cpp:133-152: the planes of cycles -1 .. -31
 * from the initial phase in plane 0, running the uncoupled model backwards */
__global__ void kuramoto_init_kernel(unsigned n, const float* freq, float* state, size_t hstride)
{
	const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
	if(i >= n) {
		return;
	}
	const float f = freq[i];
	for(unsigned t = 0; t + 1u < HISTORY; ++t) {
		const float p0 = state[size_t((0u - t) % HISTORY) * hstride + i];
		state[size_t((0u - (t + 1u)) % HISTORY) * hstride + i] = nemo_libm::kuramoto_wrap(p0 - f);
	}
}

} // namespace

extern "C" __attribute__((visibility("default")))
int hip_update_neurons(void* stream, unsigned cycle, unsigned start, unsigned end,
		float* param, size_t paramStride, float* state, size_t stateHistoryStride, size_t stateVarStride,
		uint32_t* rng, size_t rngStride, const uint32_t* fstim,
		const float* currentE, const float* currentI, const float* currentExt,
		uint64_t* recentFiring, uint32_t* fired, const nemo_hip_rcm* rcm)
{
	/* no synaptic current, no firing, no RNG (src/nemo/cpu/plugins/Kuramoto.cpp:85-99) */
	(void) paramStride; (void) stateVarStride; (void) rng; (void) rngStride; (void) fstim;
	(void) currentE; (void) currentI; (void) currentExt; (void) recentFiring; (void) fired;
	if(end <= start) return 0;
	if(!rcm || !rcm->start || (rcm->synapses && (!rcm->source || !rcm->delay || !rcm->weight))) {
		return int(hipErrorInvalidValue);   /* the descriptor asks for sources, delays and weights */
	}
	const unsigned n = end - start;
	const Plan pl = plan(n, rcm);
	auto kernel = pl.quota ? &kuramoto_update_kernel<9u, true> : pl.threadCouplings == 3u ? &kuramoto_update_kernel<3u>
		: pl.threadCouplings == 9u ? &kuramoto_update_kernel<9u> : &kuramoto_update_kernel<18u>;
	hipLaunchKernelGGL(kernel, dim3(pl.blocks), dim3(THREADS), 0,
			static_cast<hipStream_t>(stream), start, end, pl.per, pl.quota, cycle, param, state, stateHistoryStride,
			rcm->start, rcm->source, rcm->delay, rcm->weight);
	return int(hipGetLastError());
}

extern "C" __attribute__((visibility("default")))
int hip_init_neurons(void* stream, unsigned start, unsigned end,
		float* param, size_t paramStride, float* state, size_t stateHistoryStride, size_t stateVarStride,
		uint32_t* rng, size_t rngStride)
{
	(void) paramStride; (void) stateVarStride; (void) rng; (void) rngStride;
	if(end <= start) return 0;
	const unsigned n = end - start;
	hipLaunchKernelGGL(kuramoto_init_kernel, dim3((n + 255u) / 256u), dim3(256), 0,
			static_cast<hipStream_t>(stream), n, param, state, stateHistoryStride);
	return int(hipGetLastError());
}

[[maybe_unused]] static hip_update_neurons_t* const check_update = &hip_update_neurons;
[[maybe_unused]] static hip_init_neurons_t* const check_init = &hip_init_neurons;
