/*
 * plugin_step.hip -- the step as kernels launched every cycle, for what the
 * fused persistent kernel (step_kernel.hip) cannot run:
 *
 *   - models that exist as a plugin: gather, the plugin's hip_update_neurons,
 *     scatter, STDP (the structure of NeMo's CUDA step,
 *     src/nemo/cuda/Simulation.cpp:336-430);
 *   - networks of built-in models beyond its range (more neurons or longer
 *     delays than the chip's LDS holds): one kernel that updates, lists the
 *     fired neurons and delivers their spikes, and STDP.
 *
 * Pending current lives in a global ring of accumulators acc[2][R][n] (E, I);
 * spikes are added with global atomics at fire time into slot (t + delay) mod
 * R. They are int64, so that sums equal NeMo's int64 sums exactly
 * (src/nemo/cpu/Simulation.cpp:292-307) and are clamped at conversion
 * (src/nemo/fixedpoint.cpp:41-49), or int32 where the host has proven that no
 * sum can leave that range, which is the same sums.
 *
 * Forward records here carry the absolute target: {target | (delay-1) << 26,
 * Q11.20 weight}; a source's synapses are syn[off[s] .. off[s+1]).
 */
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "models.h"
#include "plugin_abi.h"

using namespace nemo_dev;

namespace {

__device__ inline float sat_to_float(long long v)
{
	if(v > 2147483647ll) v = 2147483647ll;
	if(v < -2147483648ll) v = -2147483648ll;
	return float(int32_t(v)) / 1048576.0f;
}

__device__ inline float acc_to_float(long long v) { return sat_to_float(v); }
__device__ inline float acc_to_float(int32_t v) { return fx20_to_float(v); }

__device__ inline void acc_add(long long* p, int32_t w)
{
	atomicAdd(reinterpret_cast<unsigned long long*>(p), (unsigned long long)(long long) w);
}

__device__ inline void acc_add(int32_t* p, int32_t w) { atomicAdd(p, w); }

/* Start of cycle, plugins: convert and clear this cycle's ring slot, clear the
 * external current, forced-firing bits and the cycle's fired bits. */
__global__ void pm_begin_kernel(PluginStepDev s, uint32_t k)
{
	const uint64_t t = s.cycle0 + k;
	const uint32_t slot = uint32_t(t % s.R);
	long long* acc = static_cast<long long*>(s.acc);
	long long* accE = acc + size_t(slot) * s.n;
	long long* accI = acc + size_t(s.R + slot) * s.n;
	uint32_t* fired = s.raster + size_t(k) * s.words32;
	const size_t stride = size_t(gridDim.x) * blockDim.x;
	for(size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < s.n; i += stride) {
		s.curE[i] = sat_to_float(accE[i]);
		s.curI[i] = sat_to_float(accI[i]);
		accE[i] = 0;
		accI[i] = 0;
		s.curX[i] = 0.0f;
	}
	for(size_t w = size_t(blockIdx.x) * blockDim.x + threadIdx.x; w < s.words32; w += stride) {
		s.fstim[w] = 0u;
		fired[w] = 0u;
	}
}

/* Stimulus of cycle k (deduplicated by the host) */
__global__ void pm_stimulus_kernel(PluginStepDev s, uint32_t k)
{
	const size_t stride = size_t(gridDim.x) * blockDim.x;
	const size_t tid = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
	if(s.fs_ptr) {
		for(size_t e = s.fs_ptr[k] + tid; e < s.fs_ptr[k + 1]; e += stride) {
			uint32_t i = s.fs_idx[e];
			atomicOr(&s.fstim[i >> 5], 1u << (i & 31u));
		}
	}
	if(s.is_ptr) {
		for(size_t e = s.is_ptr[k] + tid; e < s.is_ptr[k + 1]; e += stride) {
			s.curX[s.is_idx[e]] = s.is_val[e];
		}
	}
}

/* The rows of up to 64 fired sources into ring slots (base + d) mod R, by the
 * four waves of a workgroup. Lane l has the bounds ra, rb of a row if bit l of
 * `rows` is set (the same in all four waves); chunk c of 256 synapses of the
 * j-th row goes to wave (c + j) mod 4, four records per lane. The records of
 * the wave's next chunk are loaded before this one's are added: a load waits
 * for the atomics issued before it. Returns the synapses of the chunks this
 * wave did (wave-uniform). */
template<typename ACC>
__device__ inline uint32_t deliver_rows(const PluginStepDev& s, uint32_t ra, uint32_t rb, uint64_t rows,
		uint32_t base, uint32_t wave, uint32_t lane)
{
	ACC* acc = static_cast<ACC*>(s.acc);
	const uint2* syn = reinterpret_cast<const uint2*>(s.syn);
	uint32_t ev = 0, j = 0, c = 0, b = 0;   /* the chunk and its row's end */
	auto next = [&]() {   /* c >= b: none left */
		c += 1024u;
		while(c >= b && rows) {   /* wave-uniform */
			const int l = __builtin_ctzll(rows);
			rows &= rows - 1ull;
			b = uint32_t(__builtin_amdgcn_readlane(int(rb), l));
			c = uint32_t(__builtin_amdgcn_readlane(int(ra), l)) + 256u * ((wave - j) & 3u);
			++j;
		}
	};
	auto load = [&](uint2 (&rec)[4]) {
#pragma unroll
		for(uint32_t i = 0; i < 4u; ++i) {
			const uint32_t q = c + 64u * i + lane;
			rec[i] = (q < b) ? syn[q] : make_uint2(0u, 0u);
		}
	};
	next();
	uint2 rec[4];
	load(rec);
	while(c < b) {   /* wave-uniform */
		const uint32_t c0 = c, b0 = b;
		next();
		uint2 ahead[4];
		load(ahead);
#pragma unroll
		for(uint32_t i = 0; i < 4u; ++i) {
			if(c0 + 64u * i + lane < b0) {
				const int32_t w = int32_t(rec[i].y);
				uint32_t sl = base + (rec[i].x >> 26) + 1u;
				sl = (sl >= s.R) ? sl - s.R : sl;
				const uint32_t plane = (w >= 0) ? 0u : s.R;
				acc_add(acc + size_t(plane + sl) * s.n + (rec[i].x & 0x3ffffffu), w);
			}
			rec[i] = ahead[i];
		}
		ev += min(256u, b0 - c0);
	}
	return ev;
}

/* The wave's ev into one of NEMO_PM_PARTS counters, which the host adds up. A
 * single one, and a shared list of the fired neurons, serialise the atomics of
 * all workgroups (compaction and scatter of 150k synapses: 28 us a cycle with
 * them, 19 without). */
__device__ inline void count_events(unsigned long long* part, uint32_t ev, uint32_t wave, uint32_t lane)
{
	if(lane == 0 && ev) {
		atomicAdd(part + size_t((blockIdx.x * 4u + wave) % NEMO_PM_PARTS) * 16u, (unsigned long long) ev);
	}
}

/* Plugins, and built-in networks with long rows: the spikes of cycle k.
 * Workgroup g of G takes the pieces g, g + G, g + 2G, ... of 1 << plog
 * neighbouring neurons, a neuron per lane, so that all workgroups have sources
 * whatever fires: neurons that fire together are often neighbours. Every wave
 * reads the fired bits and the rows' bounds for itself, so nothing is listed and
 * nothing waited for.
 *
 * What bounds it: with few spikes the launch; with many the atomics. Per cycle
 * of the plugin step, with a wave per fired source of a list in memory, with a
 * workgroup per 2048 neurons, and now: 2000 x 1000 IF_curr_exp_noise at 333 Hz
 * 48, 1504, 44 us; 12000 x 550 140, 1062, 111; Izhikevich at 8 Hz 2000 x 1000
 * 20, 41, 13, 20000 x 1000 24, 57, 18, 200000 x 100 28, 25, 19. */
template<typename ACC>
__global__ void __launch_bounds__(256) pm_scatter_kernel(PluginStepDev s, uint32_t k, uint32_t plog)
{
	const uint32_t lane = threadIdx.x & 63u;
	const uint32_t wave = threadIdx.x >> 6;
	const uint32_t G = gridDim.x;
	const uint32_t* fired = s.raster + size_t(k) * s.words32;
	const uint32_t base = uint32_t((s.cycle0 + k) % s.R);
	uint32_t ev = 0;
	for(uint32_t p0 = blockIdx.x; (p0 << plog) < s.n; p0 += G * (64u >> plog)) {   /* block-uniform */
		const uint32_t i = ((p0 + (lane >> plog) * G) << plog) + (lane & ((1u << plog) - 1u));
		const bool f = i < s.n && ((fired[i >> 5] >> (i & 31u)) & 1u) != 0u;
		const uint32_t ra = f ? s.off[i] : 0u, rb = f ? s.off[i + 1u] : 0u;
		ev += deliver_rows<ACC>(s, ra, rb, __ballot(f), base, wave, lane);
	}
	count_events(s.part, ev, wave, lane);
}

/* Built-in models: one cycle of 256 neurons per workgroup, 16 pieces of 16
 * neighbours that lie a grid apart: neurons that fire together are often
 * neighbours, and a compute unit adds about 0.4 synapses per ns. The two pieces
 * of 32 neurons, whose values are one line of memory in each array, go to
 * workgroups b and b + 8, which run on one XCD: its L2 reads the line once. With
 * 256 forced neighbours, 270k x 300, a cycle takes 50 us so, 60 with pieces of
 * 32, 46 with pieces of 8 (but 9 % more without them), and 230 with 256
 * neighbours in a workgroup; 270k x 300 on the plugins' sequence as it was 66.
 * Reads and clears
 * the cycle's ring slot, updates the neurons (models.h), writes their raster
 * words, lists the fired ones in LDS and delivers them at once into slots t+1
 * .. t+D, none of which is slot t of a ring of D+1: other workgroups may still
 * be reading it. So a cycle is one launch where plugins need three. Without
 * DELIVER the delivery is left to pm_scatter_kernel: for networks with long rows
 * next to each other.
 *
 * What bounds it: the neurons' parameters, state and ring slot (about 90 bytes
 * each) and the chain slot -> update -> row bounds -> records -> atomics; with
 * many spikes the atomics. Per cycle, against the plugins' sequence as it was
 * (begin, update, compact, scatter): 300k x 100 37 -> 13.4 us, 300k x 50 35 ->
 * 9.9, 300k x 30 IF_curr_exp_noise 67 -> 13, 300k x 50 with STDP 56 -> 18. */
template<typename ACC, bool IZO, bool DELIVER>
__global__ void __launch_bounds__(256) pm_cycle_kernel(PluginStepDev s, uint32_t k, int stim)
{
	constexpr int NP = IZO ? 5 : MAX_PARAM;
	constexpr int NS = IZO ? 2 : MAX_STATE;
	__shared__ uint32_t list[256];
	__shared__ uint32_t wfired[4];
	const uint32_t lane = threadIdx.x & 63u;
	const uint32_t wave = threadIdx.x >> 6;
	const uint32_t n = s.n;
	/* line of 32 neurons, and its half: see above */
	const uint32_t line = ((threadIdx.x >> 4) * (gridDim.x >> 4) + (blockIdx.x >> 4)) * 8u + (blockIdx.x & 7u);
	const uint32_t piece = line * 2u + ((blockIdx.x >> 3) & 1u);
	const uint32_t l = piece * 16u + (lane & 15u);
	const uint32_t slot = uint32_t((s.cycle0 + k) % s.R);
	bool fired = false;
	if(l < n) {
		ACC* acc = static_cast<ACC*>(s.acc);
		ACC* pe = acc + size_t(slot) * n + l;
		ACC* pi = acc + size_t(s.R + slot) * n + l;
		const ACC e = *pe, i = *pi;
		float p[NP], st[NS];
#pragma unroll
		for(int q = 0; q < NP; ++q) p[q] = s.param[size_t(q) * n + l];
#pragma unroll
		for(int q = 0; q < NS; ++q) st[q] = s.state[size_t(q) * n + l];
		Rng r;
#pragma unroll
		for(int q = 0; q < 4; ++q) r.s[q] = s.rng[size_t(q) * n + l];
		const uint64_t recent = s.recent[l];
		float x = 0.0f;
		bool fs = false;
		if(stim) {
			x = s.curX[l];
			fs = ((s.fstim[l >> 5] >> (l & 31u)) & 1u) != 0u;
			s.curX[l] = 0.0f;
		}
		*pe = 0;
		*pi = 0;
		if(IZO) {
			fired = izhikevich(p, st, r, acc_to_float(e), acc_to_float(i), x, fs);
		} else {
			fired = update_neuron(s.model[l], p, st, r, acc_to_float(e), acc_to_float(i), x, fs);
		}
#pragma unroll
		for(int q = 0; q < NS; ++q) s.state[size_t(q) * n + l] = st[q];
#pragma unroll
		for(int q = 0; q < 4; ++q) s.rng[size_t(q) * n + l] = r.s[q];
		s.recent[l] = (recent << 1) | (fired ? 1ull : 0ull);
	}
	const uint64_t mask = __ballot(fired);
	if(lane == 0) wfired[wave] = uint32_t(__popcll(mask));
	if((lane & 15u) == 0u && line < s.words32) {
		reinterpret_cast<uint16_t*>(s.raster + size_t(k) * s.words32)[piece] = uint16_t(mask >> lane);
		/* every lane of the wave has read its bit */
		if(stim) reinterpret_cast<uint16_t*>(s.fstim)[piece] = 0u;
	}
	if(!DELIVER) return;
	__syncthreads();
	uint32_t before = 0, total = 0;
#pragma unroll
	for(uint32_t w = 0; w < 4u; ++w) {
		before += (w < wave) ? wfired[w] : 0u;
		total += wfired[w];
	}
	if(total == 0u) return;   /* block-uniform */
	if(fired) {
		const uint64_t below = lane ? (mask & (~0ull >> (64u - lane))) : 0ull;
		list[before + uint32_t(__popcll(below))] = l;
	}
	__syncthreads();
	uint32_t ev = 0;
	for(uint32_t j = 0; j < total; j += 64u) {   /* block-uniform */
		const uint32_t cnt = min(64u, total - j);
		uint32_t ra = 0, rb = 0;
		if(lane < cnt) {
			ra = s.off[list[j + lane]];
			rb = s.off[list[j + lane] + 1u];
		}
		ev += deliver_rows<ACC>(s, ra, rb, ~0ull >> (64u - cnt), slot, wave, lane);
	}
	count_events(s.part, ev, wave, lane);
}

/* STDP: targets whose history has bit postLen set walk their plastic
 * in-synapses (src/nemo/ConnectivityMatrix.cpp:193-227). Wave w of W looks at
 * the pieces w, w + W, w + 2W, ... of 1 << plog neighbouring targets, 64 targets
 * at a time, and walks the rows of those that qualify: neighbours, which often
 * fire together, are not one wave's.
 *
 * What bounds it: with few qualifying targets the launch and the read of the
 * histories; with many the random reads of the sources' histories. Per cycle of
 * the plugin step, with a wave per target, with a wave per 64 neighbours, and
 * now: IF_curr_exp_noise at 333 Hz 1000 x 300 28, 102, 24 us, 12000 x 300 114,
 * 222, 86; Izhikevich at 8 Hz 20000 x 300 27, 29, 23. */
__global__ void __launch_bounds__(256) pm_stdp_kernel(PluginStepDev s, uint32_t plog)
{
	const StdpParams& sp = *reinterpret_cast<const StdpParams*>(s.stdp);
	const uint32_t lane = threadIdx.x & 63u;
	const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
	const uint32_t nwaves = (gridDim.x * blockDim.x) >> 6;
	for(uint32_t p0 = wave; (p0 << plog) < s.n; p0 += nwaves * (64u >> plog)) {   /* wave-uniform */
		const uint32_t tl = ((p0 + (lane >> plog) * nwaves) << plog) + (lane & ((1u << plog) - 1u));
		const bool has = tl < s.n && ((s.recent[tl] >> sp.postLen) & 1ull) != 0ull;
		const uint32_t ra = has ? s.rcm_start[tl] : 0u, rb = has ? s.rcm_start[tl + 1u] : 0u;
		for(uint64_t todo = __ballot(has); todo; todo &= todo - 1ull) {
			const int l = __builtin_ctzll(todo);
			const uint32_t r1 = uint32_t(__builtin_amdgcn_readlane(int(rb), l));
			for(uint32_t r = uint32_t(__builtin_amdgcn_readlane(int(ra), l)) + lane; r < r1; r += 64u) {
				const uint32_t sd = s.rcm_sd[r];
				const uint64_t pre = s.recent[sd & 0x3ffffffu] >> ((sd >> 26) + 1u);
				const int32_t wd = stdp_weight_change(sp, pre);
				if(wd != 0) {
					s.rcm_acc[r] = int32_t(uint32_t(s.rcm_acc[r]) + uint32_t(wd));
				}
			}
		}
	}
}

/* After weights change (applyStdp): rebuild the ring from the firing
 * history, since NeMo reads a weight when the spike arrives
 * (src/nemo/cpu/Simulation.cpp:258-307). The ring has been zeroed; a spike
 * fired at cycle0-1-k with delay d > k is still pending and lands in slot
 * (cycle0-1-k+d) mod R. One wave per source with pending spikes. */
template<typename ACC>
__global__ void pm_replay_kernel(PluginStepDev s)
{
	ACC* acc = static_cast<ACC*>(s.acc);
	const uint32_t lane = threadIdx.x & 63u;
	const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
	const uint32_t nwaves = (gridDim.x * blockDim.x) >> 6;
	const uint64_t pend = (s.D >= 64u) ? ~0ull : ((1ull << s.D) - 1ull);
	const uint32_t last = uint32_t((s.cycle0 + s.R - 1u) % s.R);
	for(uint32_t src = wave; src < s.n; src += nwaves) {
		const uint64_t h = s.recent[src] & pend;
		if(!h) continue;
		const uint32_t a = s.off[src], b = s.off[src + 1];
		for(uint32_t q = a + lane; q < b; q += 64u) {
			const uint32_t x = s.syn[2 * size_t(q)];
			const int32_t w = int32_t(s.syn[2 * size_t(q) + 1]);
			const uint32_t tgt = x & 0x3ffffffu;
			const uint32_t d = (x >> 26) + 1u;
			const uint32_t plane = (w >= 0) ? 0u : s.R;
			uint64_t hb = h & ((d >= 64u) ? ~0ull : ((1ull << d) - 1ull));
			while(hb) {
				const uint32_t kk = uint32_t(__builtin_ctzll(hb));
				hb &= hb - 1ull;
				const uint32_t sl = (last + d - kk) % s.R;
				acc_add(acc + size_t(plane + sl) * s.n + tgt, w);
			}
		}
	}
}

template<typename ACC, bool IZO>
void launch_cycle(const PluginStepDev* s, uint32_t k, int stim, int deliver, hipStream_t stream)
{
	auto kernel = deliver ? &pm_cycle_kernel<ACC, IZO, true> : &pm_cycle_kernel<ACC, IZO, false>;
	hipLaunchKernelGGL(kernel, dim3((s->words32 + 127u) / 128u * 16u), dim3(256), 0, stream, *s, k, stim);
}

unsigned grid(size_t n, unsigned block, unsigned cap)
{
	size_t g = (n + block - 1) / block;
	if(g < 1) g = 1;
	if(g > cap) g = cap;
	return unsigned(g);
}

} // namespace

extern "C" {

int nemo_dev_pm_begin(const PluginStepDev* s, uint32_t k, void* stream)
{
	hipLaunchKernelGGL(pm_begin_kernel, dim3(grid(s->n, 256, 2048)), dim3(256), 0,
			static_cast<hipStream_t>(stream), *s, k);
	return int(hipGetLastError());
}

int nemo_dev_pm_stimulus(const PluginStepDev* s, uint32_t k, uint32_t entries, void* stream)
{
	if(entries == 0) return 0;
	hipLaunchKernelGGL(pm_stimulus_kernel, dim3(grid(entries, 256, 256)), dim3(256), 0,
			static_cast<hipStream_t>(stream), *s, k);
	return int(hipGetLastError());
}

int nemo_dev_pm_scatter(const PluginStepDev* s, uint32_t k, int narrow, int longRows, void* stream)
{
	/* 8 neurons per workgroup while that leaves the chip room; a workgroup each
	 * costs networks that fire little or not at all. Where all lanes have one in
	 * pieces of 8, which read one word of fired bits (500k oscillators x 10, per
	 * cycle 122 -> 120 us; 200k x 100 at 8 Hz 19 -> 17) */
	const bool large = s->n > 64u * NEMO_PM_SCATTER_BLOCKS && !longRows;
	auto kernel = narrow ? &pm_scatter_kernel<int32_t> : &pm_scatter_kernel<long long>;
	hipLaunchKernelGGL(kernel, dim3(grid(s->n, 8, NEMO_PM_SCATTER_BLOCKS)), dim3(256), 0,
			static_cast<hipStream_t>(stream), *s, k, large ? 3u : 0u);
	return int(hipGetLastError());
}

int nemo_dev_pm_replay(const PluginStepDev* s, int narrow, void* stream)
{
	if(narrow) {
		hipLaunchKernelGGL(pm_replay_kernel<int32_t>, dim3(2048), dim3(256), 0, static_cast<hipStream_t>(stream), *s);
	} else {
		hipLaunchKernelGGL(pm_replay_kernel<long long>, dim3(2048), dim3(256), 0, static_cast<hipStream_t>(stream), *s);
	}
	return int(hipGetLastError());
}

int nemo_dev_pm_cycle(const PluginStepDev* s, uint32_t k, int stim, int narrow, int izhikevichOnly, int deliver,
		void* stream)
{
	hipStream_t st = static_cast<hipStream_t>(stream);
	if(narrow) {
		if(izhikevichOnly) launch_cycle<int32_t, true>(s, k, stim, deliver, st);
		else launch_cycle<int32_t, false>(s, k, stim, deliver, st);
	} else {
		if(izhikevichOnly) launch_cycle<long long, true>(s, k, stim, deliver, st);
		else launch_cycle<long long, false>(s, k, stim, deliver, st);
	}
	return int(hipGetLastError());
}

int nemo_dev_pm_stdp(const PluginStepDev* s, void* stream)
{
	/* a wave per target up to 4096, then per up to 64; where every lane has one
	 * in pieces of 8, whose histories are one line of memory (300k x 50 per cycle
	 * 18.2 us, 19.6 in pieces of one) */
	const bool large = s->n / 64u > 4096u;
	const size_t waves = s->n < 4096u ? s->n : (large ? (s->n + 63u) / 64u : 4096u);
	hipLaunchKernelGGL(pm_stdp_kernel, dim3(grid(waves, 4, 4096)), dim3(256), 0,
			static_cast<hipStream_t>(stream), *s, large ? 3u : 0u);
	return int(hipGetLastError());
}

} // extern "C"
