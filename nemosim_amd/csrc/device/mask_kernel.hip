/*
 * mask_kernel.hip -- the persistent step: the fused kernel of step_kernel.hip
 * with another exchange between partitions, and with far waves, which deliver
 * the previous cycle's records of delays >= 2, and STDP beside the neurons'.
 *
 * There, a partition publishes a list of its fired neurons and a count, and
 * the others read the counts, then the entries, then each source's bucket
 * bounds, then its records: four dependent round trips, behind a barrier for
 * the list's positions and one for the counts. Here every wave publishes its
 * 64 fired bits as they are, two words of 32 bits with the cycle's number in
 * the upper half, as soon as it has them; every wave of every workgroup polls
 * its share of the network's words and delivers the sources it finds there.
 * That is one round trip less, two barriers a cycle instead of three, and no
 * search for a source's partition. Each workgroup reads n/32 words a cycle
 * whatever fires (50 KB at 200k neurons), which costs a wave up to eight loads
 * that are in flight together; how the words are shared is at Deal.
 *
 * What bounds it: the latency of the chain update -> words -> bounds -> delay-1
 * records of one cycle; no unit is busy. From 200k neurons on, with few waves
 * left over, the requests for bounds and records. Per cycle, lists, words with
 * the far records on the neurons' waves, on far waves, and dealt: 1k x 100 4.5,
 * 3.5, 2.6, 2.5 us; 10k x 313 5.6, 4.6, 3.5, 3.4; 60k x 300 6.3, 5.7, 4.6, 4.4;
 * 100k x 100 7.6, 6.3, 5.4, 5.3; 200k x 1000 13.8, 12.9, 12.6, 12.7; 12k x 550
 * IF_curr_exp_noise at 333 Hz 57, 49, 37, 37. 48 networks of 1k-20k batched, 200
 * cycles, 3.96 -> 3.1 ms (3 launches, with far waves where all of one's networks
 * fit with them). With STDP, 3k x 300 10.9 -> 3.4 us, 10k x 300 10.5 -> 4.3, 50k x
 * 1000 17.4 -> 10.2 (see stdp_waves).
 *
 * Without STDP two buffers of words are enough: a wave publishes cycle t+1 after its own
 * reads of cycle t, and a workgroup publishes t+2 only once its waves have
 * seen every word of t+1.
 */
#include <algorithm>

#include "step_device.h"

namespace {

constexpr uint32_t LIST = 128u;      /* sources a wave lists in LDS at a time (16 bits: from its first word on) */

constexpr uint32_t CHUNK = 64u;      /* synapses per STDP work item (one per lane of a wave) */

/* The words that a wave polls. Neurons that fire together are often neighbours,
 * and with contiguous shares one wave delivers all of them. So the words are
 * dealt to the waves in turn, one at a time while a wave has up to 64, in pieces
 * of 8 (64 bytes) beyond; there among four waves, since a wave delivers once all
 * its words have come, and with words from all partitions it waits for the last
 * of them. The kernels for batches and for saturating networks (ANY) decide so
 * for each network, and deal to more than 8 waves by pieces, too (32 networks in
 * partitions of 512 to 960, 200 cycles: 2.64 ms one at a time, 2.39). Per cycle
 * with 1000 forced neighbours, contiguous and dealt: 5k x 1000 97, 51 us (lists
 * 66), 50k x 300 43, 29 (32), 200k x 100 59, 35 (37), with STDP 20k x 300 58, 42
 * (48); without them 1k x 100 2.7, 2.5, 10k x 313 3.6, 3.4, 60k x 300 4.5, 4.4,
 * 200k x 300 8.6, 8.8 (9.0 dealt to all waves), 200k x 1000 and 50k x 1000 with
 * STDP 1 and 3 % less, 1k x 100 IF_curr_exp_noise at 333 Hz 2 % more. */
template<uint32_t WORDS, bool ANY, bool IZO>
struct Deal {
	uint32_t waves, begin, end;   /* of the wave's group; begin: its own first word */
	uint32_t plog;                /* ANY: of either kind */
	__device__ inline uint32_t piece() const { return ANY ? plog : WORDS == 1u ? 0u : 3u; }
	__device__ inline Deal(uint32_t wave, uint32_t nwaves, uint32_t W)
	{
		const bool few = ANY ? W <= 64u * nwaves && nwaves <= 8u : WORDS == 1u;
		plog = few ? 0u : 3u;
		const uint32_t group = few ? 16u : 4u;
		const uint32_t g0 = wave & ~(group - 1u), g1 = min(g0 + group, nwaves);
		waves = g1 - g0;
		end = wave >= nwaves ? 0u : g1 == nwaves ? W : (W * g1 / nwaves) & ~15u;   /* waves beyond: no words */
		begin = ((W * g0 / nwaves) & ~15u) + ((wave - g0) << piece());
	}
	/* the first of the wave's words from the j-th on, j a multiple of 64; how much
	 * further a lane's own is, and the (j+k)-th, k < 64 WORDS */
	__device__ inline uint32_t first(uint32_t j) const { return begin + j * waves; }
	__device__ inline uint32_t further(uint32_t lane) const
	{
		return (__umul24(lane >> piece(), waves) << piece()) | (lane & ((1u << piece()) - 1u));
	}
	__device__ inline uint32_t word(uint32_t j, uint32_t k) const
	{
		/* the Izhikevich kernels are slower with the shorter product (60k x 300
		 * 4.4 -> 4.6 us), the others 3 % faster */
		if(IZO) return first((j + k) & ~63u) + further(k & 63u);
		if(WORDS == 1u) return first(j) + further(k);
		return first(j) + __umul24(k & ~63u, waves) + further(k & 63u);
	}
};

/* The neurons that fired in an earlier cycle, whose words are complete, of the
 * words dealt to a wave: f(valid, neuron) for whole waves. */
template<uint32_t WORDS, bool ANY, bool IZO, typename F>
__device__ inline void each_fired(const NEMO_GLOBAL uint64_t* words, uint32_t tag, const Deal<WORDS, ANY, IZO>& deal,
		uint16_t* list, uint32_t lane, F f)
{
	const uint32_t mine = deal.further(lane);
	for(uint32_t c0 = 0; deal.first(c0) < deal.end; c0 += 64u * WORDS) {   /* wave-uniform */
		uint32_t v[WORDS], pos[WORDS];
#pragma unroll
		for(uint32_t i = 0; i < WORDS; ++i) {
			const uint32_t w = deal.first(c0 + 64u * i) + mine;
			const uint64_t e = w < deal.end ? ld_agent(words + w) : 0ull;
			v[i] = w < deal.end && uint32_t(e >> 32) == tag ? uint32_t(e) : 0u;
		}
		uint32_t total = 0;
#pragma unroll
		for(uint32_t i = 0; i < WORDS; ++i) {
			const uint32_t c = uint32_t(__popc(v[i]));
			const uint32_t x = wave_scan(c);
			pos[i] = total + x - c;
			total += uint32_t(__builtin_amdgcn_readlane(int(x), 63));
		}
		for(uint32_t l0 = 0; l0 < total; l0 += LIST) {   /* wave-uniform */
#pragma unroll
			for(uint32_t i = 0; i < WORDS; ++i) {
				uint32_t b = v[i];
				for(uint32_t at = pos[i]; b; ++at) {
					if(at - l0 < LIST) list[at - l0] = uint16_t((64u * i + lane) * 32u + uint32_t(__builtin_ctz(b)));
					b &= b - 1u;
				}
			}
			__builtin_amdgcn_wave_barrier();   /* a wave's LDS operations complete in order */
			const uint32_t n = min(LIST, total - l0);
			for(uint32_t h = 0; h < n; h += 64u) {   /* wave-uniform */
				const bool ok = h + lane < n;
				const uint32_t e = ok ? list[h + lane] : 0u;
				f(ok, deal.word(c0, e >> 5) * 32u + (e & 31u));
			}
			__builtin_amdgcn_wave_barrier();   /* the list is written again */
		}
	}
}

/* stdp_weight_change of models.h without branches, so that the chunks that a
 * wave has in flight overlap (with them a chunk took about 1000 cycles, most of
 * them waits for LDS). Per region (potentiation, depression) the closest
 * arrival before and after the target's firing and their distances; the closer
 * one's table entry, none if there is none or they are equally close. m: the
 * regions' masks over h >> postLen and over h << (64 - postLen). h: the
 * source's firing history as it arrived at the target. */
struct StdpMasks { uint64_t pre[2], post[2]; };

__device__ inline int32_t stdp_change(const StdpMasks& m, uint32_t postLen, const int32_t* fn, uint64_t h)
{
	const uint64_t hp = h >> postLen, hq = h << (64u - postLen);   /* postLen: 1..63 */
	uint32_t w = 0;
#pragma unroll
	for(uint32_t i = 0; i < 2u; ++i) {
		const uint64_t a = hp & m.pre[i], b = hq & m.post[i];
		const uint32_t da = a ? uint32_t(__builtin_ctzll(a)) : 64u;
		const uint32_t db = b ? uint32_t(__builtin_clzll(b)) : 64u;
		const int32_t v = fn[min(da, 63u) < db ? da : 64u + min(db, 63u)];   /* fnPre, then fnPost */
		w += da == db ? 0u : uint32_t(v);
	}
	return int32_t(w);
}

/* Lanes per source: as many as cover a bucket in one pass, fewer (down to
 * glog2) where that would take more rounds than are in flight together */
template<bool SAT, bool IZO>
__device__ inline uint32_t lanes_for(const NetDev& nd, uint32_t nsrc)
{
	uint32_t g = nd.glogFew;
	while(g > nd.glog2 && pass_rounds(nsrc, g) > DeliverRounds<SAT, IZO>::value) --g;
	return g;
}

/* ---- STDP (src/nemo/ConnectivityMatrix.cpp:193-227), on waves of its own that
 * have no neurons. The targets of cycle t fired in cycle t-postLen; their rows
 * of plastic in-synapses are cut into chunks of CHUNK, and chunk c of target x
 * belongs to partition (x + c) mod P, always: no other workgroup of the launch
 * adds to it, so its XCD's cache can (shares made equal by the targets'
 * position in the cycle's list had to add at the memory side, 50k x 1000 19.1
 * us per cycle against 18.2 then). The chunks are listed in cycle t and
 * accumulated in cycle t+1: then every word of cycle t has been seen, and
 * behind a wave's word of cycle t are its neurons' histories up to t-1, stored
 * a cycle earlier, so no wave waits for its stores. The history without cycle
 * t's spikes is enough: they arrive a cycle later at the earliest; its oldest
 * bit would have been shifted out. Histories are kept for 4 cycles: a
 * partition reads those of t-1 in t+1, when another may be storing t+2's.
 * Words are kept for postLen+3: if there are more chunks than a list holds it
 * is left, and each wave accumulates the targets that it finds in its words,
 * in t+1.
 *
 * What bounds it: the histories, 8 bytes each from anywhere (400k a cycle at
 * 50k x 1000 and 8 Hz, 3.6 us), and the latency of the chain records, history,
 * table, add. On waves of its own it runs beside the exchange and the delivery:
 * done by the neurons' waves, where those wait for words, a cycle took 17.3 us
 * (50k x 1000) and 6.3 (3k x 300) instead of 11.9 and 3.6. */
struct StdpLds {
	StdpParams* table;
	uint2* work;          /* [2][NEMO_MASK_STDP_CAP] {row index, length}, by cycle parity */
	uint32_t* count;      /* [2] */
	StdpMasks* masks;
	uint32_t* records;    /* [2][stdpCache][CHUNK] reverse records of the first chunks */
};

/* K: chunks of a wave whose loads are in flight together */
template<bool SAT, bool IZO, uint32_t WORDS, bool ANY, uint32_t K>
__device__ inline void stdp_waves(const NetDev& nd, uint32_t p, uint32_t wave, uint32_t nwaves, uint32_t lane,
		const StdpLds& l, uint16_t* list)
{
	const uint32_t P = nd.P, R = nd.flRing, n_total = nd.n, cache = nd.stdpCache;
	const uint32_t postLen = uint32_t(l.table->postLen);
	const uint32_t W = P * (nd.T >> 5);
	const Deal<WORDS, ANY, IZO> deal(wave, nwaves, W);
	const NEMO_GLOBAL uint32_t* rsd = glb(nd.rcm_sd);
	NEMO_GLOBAL int32_t* racc = glb(nd.rcm_acc);
	const StdpMasks m = *l.masks;
	/* the first `count` of K chunks, one synapse per lane: the sources'
	 * histories, the weight changes, the adds */
	auto chunks = [&](const NEMO_GLOBAL uint64_t* h, const uint32_t* r, const uint32_t* len, const uint32_t* sd,
			uint32_t count) {
		uint64_t hh[K];
		int32_t wd[K];
#pragma unroll
		for(uint32_t i = 0; i < K; ++i) {
			hh[i] = 0ull;
			if(i < count) hh[i] = ld_agent(h + (sd[i] & 0x3ffffffu));
		}
#pragma unroll
		for(uint32_t i = 0; i < K; ++i) {
			wd[i] = stdp_change(m, postLen, l.table->fnPre, (hh[i] & (~0ull >> 1)) >> (sd[i] >> 26));
		}
#pragma unroll
		for(uint32_t i = 0; i < K; ++i) {
			if(i < count && lane < len[i] && wd[i] != 0) {
				(void) __hip_atomic_fetch_add(racc + r[i] + lane, wd[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
			}
		}
	};
	/* a lane's target: the bounds of its row, and its first chunk (or a number
	 * beyond the last) of this partition */
	struct Row { uint32_t begin, len, ch; };
	auto row_of = [&](bool ok, uint32_t x) {
		Row r = {0u, 0u, (p + P - x % P) % P};
		if(ok) {
			r.begin = glb(nd.rcm_start)[x];
			r.len = glb(nd.rcm_start)[x + 1u] - r.begin;
		}
		return r;
	};
	/* the list of cycle tc, whose words are in slot tslot */
	auto accumulate = [&](uint32_t tc, uint32_t tslot) {
		const uint32_t par = tc & 1u, total = l.count[par];
		const NEMO_GLOBAL uint64_t* h = glb(nd.rfg) + size_t((tc - 1u) & 3u) * n_total;
		const uint2* work = l.work + par * NEMO_MASK_STDP_CAP;
		const uint32_t* rec = l.records + par * cache * CHUNK;
		if(total <= NEMO_MASK_STDP_CAP) {
			for(uint32_t c0 = wave; c0 < total; c0 += K * nwaves) {   /* wave-uniform */
				uint32_t r[K], len[K], sd[K], count = 0;
#pragma unroll
				for(uint32_t i = 0; i < K; ++i) {
					const uint32_t c = min(c0 + i * nwaves, total - 1u);
					const uint2 ck = work[c];
					r[i] = __builtin_amdgcn_readfirstlane(ck.x);
					len[i] = __builtin_amdgcn_readfirstlane(ck.y);
					count += c0 + i * nwaves < total ? 1u : 0u;
					if(c < cache) sd[i] = rec[c * CHUNK + lane];
					else sd[i] = rsd[r[i] + min(lane, len[i] - 1u)];
				}
				chunks(h, r, len, sd, count);
			}
			return;
		}
		const uint32_t s = tslot >= postLen ? tslot - postLen : tslot + R - postLen;
		each_fired<WORDS, ANY, IZO>(glb(nd.mk) + size_t(s) * nemo_mask_words(W), tc - postLen, deal, list, lane, [&](bool ok, uint32_t x) {
			const Row row = row_of(ok, x);
			uint32_t ch = row.ch;
			while(__any(ch * CHUNK < row.len)) {   /* wave-uniform */
				const uint32_t mr = row.begin + ch * CHUNK;
				const uint32_t ml = ch * CHUNK < row.len ? min(CHUNK, row.len - ch * CHUNK) : 0u;
				for(uint64_t b = __ballot(ml != 0u); b; ) {
					uint32_t r[K], len[K], sd[K], count = 0;
#pragma unroll
					for(uint32_t i = 0; i < K; ++i) {
						const int src = __builtin_ctzll(b | 1ull << 63);
						r[i] = uint32_t(__builtin_amdgcn_readlane(int(mr), src));
						len[i] = uint32_t(__builtin_amdgcn_readlane(int(ml), src));
						sd[i] = 0u;
						if(b) sd[i] = rsd[r[i] + min(lane, len[i] - 1u)];
						count += b ? 1u : 0u;
						b &= b - 1ull;
					}
					chunks(h, r, len, sd, count);
				}
				ch += P;
			}
		});
	};
	uint32_t wslot = uint32_t(nd.cycle0 % R);
	for(uint32_t k = 0; k < nd.nsteps; ++k) {
		const uint64_t t = nd.cycle0 + k;
		const uint32_t tag = uint32_t(t), par = tag & 1u;
		if(wave == 0u && lane == 0u) l.count[par] = 0u;   /* the last list of this parity is done */
		__syncthreads();
		if(SAT) __syncthreads();
		if(k > 0u) accumulate(tag - 1u, wslot ? wslot - 1u : R - 1u);
		/* this cycle's chunks; the records of the first `cache` go to LDS */
		if(t >= postLen) {
			const uint32_t s = wslot >= postLen ? wslot - postLen : wslot + R - postLen;
			each_fired<WORDS, ANY, IZO>(glb(nd.mk) + size_t(s) * nemo_mask_words(W), tag - postLen, deal, list, lane, [&](bool ok, uint32_t x) {
				const Row row = row_of(ok, x);
				uint32_t ch = row.ch;
				while(__any(ch * CHUNK < row.len)) {   /* wave-uniform */
					const bool has = ch * CHUNK < row.len;
					const uint32_t r = row.begin + ch * CHUNK;
					const uint32_t len = has ? min(CHUNK, row.len - ch * CHUNK) : 0u;
					uint32_t at = ~0u;
					if(has) {
						at = atomicAdd(l.count + par, 1u);
						if(at < NEMO_MASK_STDP_CAP) l.work[par * NEMO_MASK_STDP_CAP + at] = make_uint2(r, len);
					}
					for(uint64_t b = __ballot(has && at < cache); b; b &= b - 1ull) {
						const int src = __builtin_ctzll(b);
						const uint32_t as = uint32_t(__builtin_amdgcn_readlane(int(at), src));
						const uint32_t rs = uint32_t(__builtin_amdgcn_readlane(int(r), src));
						const uint32_t ls = uint32_t(__builtin_amdgcn_readlane(int(len), src));   /* >= 1 */
						__builtin_amdgcn_global_load_lds((NEMO_GLOBAL void*)(rsd + rs + min(lane, ls - 1u)),
								(NEMO_LDS void*)(l.records + (par * cache + as) * CHUNK), 4, 0, 0);
					}
					ch += P;
				}
			});
		}
		__builtin_amdgcn_s_waitcnt(0);   /* the staged records are in LDS */
		__syncthreads();
		wslot = wslot + 1u == R ? 0u : wslot + 1u;
	}
	if(nd.nsteps > 0u) accumulate(uint32_t(nd.cycle0) + nd.nsteps - 1u, wslot ? wslot - 1u : R - 1u);
}

/* The far list of a cycle (ranges [x, y) of records, relative to ring slot
 * base) by nw waves, wave w taking a contiguous share */
template<bool SAT, bool IZO>
__device__ inline void deliver_far(const NetDev& nd, const uint2* far, uint32_t count, uint32_t w, uint32_t nw,
		uint32_t lane, uint32_t base, const NEMO_GLOBAL uint2* syn, int32_t* ringE, int32_t* ringI, uint32_t* ovf)
{
	const uint32_t share = (count + nw - 1u) / nw;
	const uint32_t j0 = min(count, w * share), j1 = min(count, j0 + share);
	for(uint32_t jb = j0; jb < j1; jb += 128u) {   /* wave-uniform */
		const uint32_t nsrc = min(128u, j1 - jb);
		const uint2 e0 = lane < nsrc ? far[jb + lane] : make_uint2(0u, 0u);
		const uint2 e1 = 64u + lane < nsrc ? far[jb + 64u + lane] : make_uint2(0u, 0u);
		deliver_ranges<SAT, IZO>(e0.x, e0.y, e1.x, e1.y, nsrc, lanes_for<SAT, IZO>(nd, nsrc), lane, base, syn,
				ringE, ringI, ovf, nd.D, nd.T, nd.T >> 5);
	}
}

/* WORDS: words a lane polls together. A wave whose share of the words takes
 * more than 64 WORDS of them goes through the rest of the cycle's chain once
 * per 64 WORDS, and every word costs instructions whether it is there or not
 * (10k x 100: 4.0 us a cycle with 4, 4.5 with 8; 200k x 100: 9.0 with 4, 8.4
 * with 8), so the host picks the smallest of 1, 4 and 8 that covers the share. */
template<bool SAT, bool IZO, uint32_t WORDS, bool STDP, bool ANY>
__device__ __forceinline__ void run_masked(const NetDev& nd, uint32_t p)
{
	constexpr int NP = IZO ? 5 : MAX_PARAM;
	constexpr int NS = IZO ? 2 : MAX_STATE;
	constexpr uint32_t PAIRS = (WORDS + 1u) / 2u;   /* words joined to 64 bits */
	extern __shared__ __align__(16) uint8_t lds[];

	const uint32_t T = nd.T, D = nd.D, P = nd.P;
	const uint32_t n_total = nd.n;
	const uint32_t tid = threadIdx.x;
	const uint32_t nthreads = blockDim.x;
	const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);   /* wave-uniform, in a scalar register */
	const uint32_t lane = tid & 63u;
	const uint32_t nwaves = nthreads >> 6;
	const uint32_t nw = T >> 6;                 /* waves that have neurons; the rest (batches) only keep the barriers */
	const uint32_t n = p * T + tid;
	const bool active = (tid < T) && (n < n_total);
	const uint32_t fwords = T >> 5;

	/* LDS: see nemo_mask_lds_bytes */
	int32_t* ringE = reinterpret_cast<int32_t*>(lds);
	int32_t* ringI = ringE + D * T;
	float* ext = reinterpret_cast<float*>(ringI + D * T);
	uint32_t* fst = reinterpret_cast<uint32_t*>(ext + T);
	uint32_t* ovf = fst + fwords;                                      /* [2][D][T/32] when SAT */
	uint16_t* list = reinterpret_cast<uint16_t*>(ovf + (SAT ? 2u * D * fwords : 0u)) + wave * LIST;
	/* with STDP (nemo_mask_stdp_lds_bytes), lists by cycle parity */
	const uint32_t R = STDP ? nd.flRing : 2u;          /* cycles of words kept */
	const uint32_t nsw = STDP ? nd.stdpWaves : 0u;
	StdpLds stdpLds;
	uint8_t* area = reinterpret_cast<uint8_t*>(ovf + (SAT ? 2u * D * fwords : 0u)) + (nw + nsw) * LIST * 2u;
	stdpLds.table = reinterpret_cast<StdpParams*>(area);
	stdpLds.work = reinterpret_cast<uint2*>(area + NEMO_STDP_LDS_BYTES);
	stdpLds.count = reinterpret_cast<uint32_t*>(stdpLds.work + 2u * NEMO_MASK_STDP_CAP);
	stdpLds.masks = reinterpret_cast<StdpMasks*>(stdpLds.count + 4);
	stdpLds.records = stdpLds.count + 16;
	/* With far waves: two far lists, by cycle parity. The neurons' waves of
	 * cycle t leave the ranges of delays >= 2 there, which the far waves
	 * deliver in cycle t+1, none of them into slot t+1. */
	const uint32_t nfw = nd.farWaves, fcap = nd.farCap;
	uint2* far = reinterpret_cast<uint2*>(STDP ? reinterpret_cast<uint8_t*>(stdpLds.records + 2u * nd.stdpCache * CHUNK) : area);
	uint32_t* farAsked = reinterpret_cast<uint32_t*>(far + 2u * fcap);   /* [2] */
	uint32_t* farLen = farAsked + 2;                                     /* [2] */
	if(nfw && tid < 2u) farAsked[tid] = farLen[tid] = 0u;
	const bool defer = (nd.flags & NEMO_NET_DEFER) != 0u;
	const uint32_t offMask = defer ? ((1u << OFF_NEAR_SHIFT) - 1u) : ~0u;
	const NEMO_GLOBAL uint2* syn = glb(reinterpret_cast<const uint2*>(nd.syn));
	const NEMO_GLOBAL uint32_t* off = glb(nd.off);

	/* as in step_kernel.hip: workgroups started, first start (diagnostics) */
	if(tid == 0) {
		atomicAdd(nd.status - 1, 1u);
		atomicMin(reinterpret_cast<unsigned long long*>(nd.status + 7), (unsigned long long) wall_clock64());
	}

	int32_t* gring = nd.ring + size_t(p) * 2u * (D + 1u) * T;
	const bool replay = STDP && (nd.flags & NEMO_NET_REPLAY) != 0u;
	if(replay) {
		for(uint32_t i = tid; i < 2u * D * T; i += nthreads) ringE[i] = 0;
	} else {
		ring_restore(gring, ringE, T, D, nd.cycle0, wave, nwaves, lane);
	}
	if(SAT) {
		for(uint32_t i = tid; i < 2u * D * fwords; i += nthreads) ovf[i] = 0u;
	}
	if(tid < T) ext[tid] = 0.0f;
	if(tid < fwords) fst[tid] = 0u;
	if(replay) {
		__syncthreads();
		ring_replay<SAT>(nd, p, syn, off, offMask, ringE, ringI, ovf, fwords, wave, nwaves, lane);
	}

	/* neuron registers */
	int model = 0;
	float prm[NP];
	float st[NS];
	Rng rng;
	uint64_t recent = 0;
#pragma unroll
	for(int k = 0; k < NP; ++k) prm[k] = 0.0f;
#pragma unroll
	for(int k = 0; k < NS; ++k) st[k] = 0.0f;
	rng.s[0] = rng.s[1] = rng.s[2] = rng.s[3] = 0u;
	if(active) {
		model = nd.model[n];
#pragma unroll
		for(int k = 0; k < NP; ++k) prm[k] = nd.param[size_t(k) * n_total + n];
#pragma unroll
		for(int k = 0; k < NS; ++k) st[k] = nd.state[size_t(k) * n_total + n];
#pragma unroll
		for(int k = 0; k < 4; ++k) rng.s[k] = nd.rng[size_t(k) * n_total + n];
		recent = nd.recent[n];
	}
	unsigned long long events = 0;
	/* deferred delivery: this wave's far ranges (delays >= 2) of the previous
	 * cycle's sources, one per lane, kn of them (wave-uniform) */
	uint32_t ka0 = 0, kb0 = 0, ka1 = 0, kb1 = 0, kn = 0;
	auto lanes = [&](uint32_t nsrc) { return lanes_for<SAT, IZO>(nd, nsrc); };
	/* the Gaussian input of Izhikevich networks is drawn a cycle ahead */
	float noise = 0.0f;
	if(IZO && active && nd.nsteps > 0u && prm[IZ_SIGMA] != 0.0f) {
		noise = prm[IZ_SIGMA] * nrand(rng);
	}
	const uint32_t W = P * fwords;
	const Deal<WORDS, ANY, IZO> deal(wave, nw, W);
	const uint32_t myFurther = deal.further(lane);
	uint32_t wslot = uint32_t(nd.cycle0 % R);               /* cycle mod R */
	if(STDP) {
		/* the tables to LDS: they are read for every plastic synapse */
		const NEMO_GLOBAL StdpParams* sp = glb(static_cast<const StdpParams*>(nd.stdp));
		const NEMO_GLOBAL uint32_t* src = glb(static_cast<const uint32_t*>(nd.stdp));
		uint32_t* dst = reinterpret_cast<uint32_t*>(stdpLds.table);
		for(uint32_t i = tid; i < uint32_t(sizeof(StdpParams) / 4u); i += nthreads) dst[i] = src[i];
		if(tid < 2u) {
			stdpLds.count[tid] = 0u;
			const uint64_t region = tid ? sp->depression : sp->potentiation;
			stdpLds.masks->pre[tid] = (region & sp->prePost) >> sp->postLen;
			stdpLds.masks->post[tid] = (region & sp->postPre) << (64 - sp->postLen);
		}
	}

	/* Stimulus is put into LDS a cycle ahead: the schedule's bounds of the next
	 * cycle are in registers, its first entries are loaded after the publish
	 * and stored before the cycle's last barrier; the update that reads them
	 * clears them. */
	const bool sched = nd.fs_ptr != nullptr;
	const uint32_t sthreads = STDP || nfw ? T : nthreads;   /* threads that take entries */
	const bool takes = tid < sthreads;
	uint32_t fb = 0, fe = 0, ib = 0, ie = 0;    /* bounds of the next cycle's entries */
	const uint32_t lo = p * T;
	auto force = [&](uint32_t idx) {
		const uint32_t l = idx - lo;
		if(l < T) atomicOr(&fst[l >> 5], 1u << (l & 31u));
	};
	auto drive = [&](uint32_t idx, float v) {
		const uint32_t l = idx - lo;
		if(l < T) ext[l] = v;
	};
	__syncthreads();
	if(sched && nd.nsteps > 0u) {
		const uint32_t f0 = glb(nd.fs_ptr)[0], i0 = glb(nd.is_ptr)[0];
		fb = glb(nd.fs_ptr)[1];
		ib = glb(nd.is_ptr)[1];
		for(uint32_t e = f0 + tid; e < fb; e += nthreads) force(glb(nd.fs_idx)[e]);
		for(uint32_t e = i0 + tid; e < ib; e += nthreads) drive(glb(nd.is_idx)[e], glb(nd.is_val)[e]);
		if(nd.nsteps > 1u) {
			fe = glb(nd.fs_ptr)[2];
			ie = glb(nd.is_ptr)[2];
		}
	}
	uint32_t slotK = uint32_t(nd.cycle0 % D);
	__syncthreads();

	const bool learns = STDP && wave >= nw && wave < nw + nsw;   /* its barriers are those of this loop */
	if(learns) stdp_waves<SAT, IZO, WORDS, ANY, IZO ? 8u : 4u>(nd, p, wave - nw, nsw, lane, stdpLds, list);
	const bool carries = nfw && wave >= nw + nsw && wave < nw + nsw + nfw;
	if(carries) {
		uint32_t prev = slotK;   /* slot of the cycle before */
		for(uint32_t k = 0; k < nd.nsteps; ++k) {
			const uint32_t par = uint32_t(nd.cycle0 + k) & 1u;
			prev = prev ? prev - 1u : D - 1u;
			__syncthreads();
			if(SAT) __syncthreads();
			if(k > 0u) {
				deliver_far<SAT, IZO>(nd, far + (par ^ 1u) * fcap, farLen[par ^ 1u], wave - nw - nsw, nfw, lane, prev, syn,
						ringE, ringI, ovf);
			}
			__syncthreads();
			prev = prev + 2u >= D ? prev + 2u - D : prev + 2u;
		}
	}
	const uint32_t nsteps = learns || carries ? 0u : nd.nsteps;
	for(uint32_t k = 0; k < nsteps; ++k) {
		const uint64_t t = nd.cycle0 + k;
		const uint32_t tag = uint32_t(t);
		const uint32_t slot = slotK;
		slotK = (slotK + 1u == D) ? 0u : slotK + 1u;
		const bool drawn = !(IZO && active && k + 1u < nd.nsteps && prm[IZ_SIGMA] != 0.0f);
		NEMO_GLOBAL uint64_t* words = glb(nd.mk) + size_t(wslot) * nemo_mask_words(W);

		/* ---- 1. neuron update */
		bool fired = false;
		if(active) {
			const uint32_t r = slot * T + tid;
			int32_t e = ringE[r];
			int32_t i = ringI[r];
			if(SAT) {
				const uint32_t bit = 1u << (tid & 31u);
				if(ovf[slot * fwords + (tid >> 5)] & bit) e = INT32_MAX;
				if(ovf[(D + slot) * fwords + (tid >> 5)] & bit) i = INT32_MIN;
			}
			ringE[r] = 0;
			ringI[r] = 0;
			float cx = 0.0f;
			bool fs = false;
			if(sched) {
				cx = ext[tid];
				fs = ((fst[tid >> 5] >> (tid & 31u)) & 1u) != 0u;
				ext[tid] = 0.0f;
			}
			if(IZO) {
				fired = izhikevich_drawn(prm, st, noise, fx20_to_float(e), fx20_to_float(i), cx, fs);
			} else {
				fired = update_neuron(model, prm, st, rng, fx20_to_float(e), fx20_to_float(i), cx, fs);
			}
			recent = (recent << 1) | (fired ? 1ull : 0ull);
			if(STDP) st_agent(glb(nd.rfg) + size_t(tag & 3u) * n_total + n, recent);
		}

		if(nfw && tid == 0u) farAsked[tag & 1u] = farLen[tag & 1u] = 0u;   /* the last list of this parity is done */

		/* ---- 2. publish the wave's fired bits; the raster */
		const uint64_t mask = __ballot(fired);
		if(wave < nw) {
			if(lane < 2u) {
				st_agent(words + p * fwords + wave * 2u + lane,
						(uint64_t(tag) << 32) | uint64_t(uint32_t(mask >> (32u * lane))));
				/* the wave's forced-firing bits have been read */
				if(sched) fst[wave * 2u + lane] = 0u;
			}
			if(lane == 0u) {
				glb(nd.raster)[size_t(k) * nd.words + p * (T >> 6) + wave] = mask;
			}
		}
		/* every wave has read its slot before records of delay D, or the
		 * next stimulus, are added */
		__syncthreads();
		if(SAT) {
			/* the slot just consumed starts empty for cycle t + D */
			for(uint32_t w = tid; w < fwords; w += nthreads) {
				ovf[slot * fwords + w] = 0u;
				ovf[(D + slot) * fwords + w] = 0u;
			}
			__syncthreads();
		}

		/* the next cycle's first stimulus entries, and the bounds of the one after */
		uint32_t fx = ~0u, ix = ~0u, fnext = 0, inext = 0;
		float iv = 0.0f;
		if(sched) {
			if(takes && fb + tid < fe) fx = glb(nd.fs_idx)[fb + tid];
			if(takes && ib + tid < ie) {
				ix = glb(nd.is_idx)[ib + tid];
				iv = glb(nd.is_val)[ib + tid];
			}
			if(k + 2u < nd.nsteps) {
				fnext = glb(nd.fs_ptr)[k + 3u];
				inext = glb(nd.is_ptr)[k + 3u];
			}
		}

		/* the next cycle's Gaussian input, while the words are under way */
		if(!drawn) {
			noise = prm[IZ_SIGMA] * nrand(rng);
		}

		/* ---- deferred records (delays >= 2) of the previous cycle's spikes */
		if(kn) {
			deliver_ranges<SAT, IZO>(ka0, kb0, ka1, kb1, kn, lanes(kn), lane, (slot + D - 1u) % D, syn,
					ringE, ringI, ovf, D, T, fwords);
			kn = 0;
		}

		/* ---- 3. this wave's words of every partition; 4. delivery of the
		 * sources in them */
		bool first = true;
		for(uint32_t c0 = 0; deal.first(c0) < deal.end; c0 += 64u * WORDS) {   /* wave-uniform */
			uint32_t mine = myFurther;
			if(SAT) {   /* found again each time: no register left to keep it in over the cycle */
				mine = lane;
				asm volatile("" : "+v"(mine));
				mine = deal.further(mine);
			}
			uint64_t m[PAIRS];
			uint32_t pos[PAIRS];
			uint32_t pending = 0;
#pragma unroll
			for(uint32_t i = 0; i < PAIRS; ++i) m[i] = 0ull;
#pragma unroll
			for(uint32_t i = 0; i < WORDS; ++i) {
				if(deal.first(c0 + 64u * i) + mine < deal.end) pending |= 1u << i;
			}
			uint32_t spins = 0;
			while(pending) {
				uint64_t v[WORDS];
#pragma unroll
				for(uint32_t i = 0; i < WORDS; ++i) {
					v[i] = 0ull;
					if(deal.first(c0 + 64u * i) < deal.end) {   /* wave-uniform */
						/* a byte offset from a scalar address */
						if((pending >> i) & 1u) v[i] = ld_agent(reinterpret_cast<const NEMO_GLOBAL uint64_t*>(
								reinterpret_cast<const NEMO_GLOBAL uint8_t*>(words + deal.first(c0 + 64u * i)) + mine * 8u));
					}
				}
#pragma unroll
				for(uint32_t i = 0; i < WORDS; ++i) {
					if(((pending >> i) & 1u) && uint32_t(v[i] >> 32) == tag) {
						m[i / 2u] |= uint64_t(uint32_t(v[i])) << (32u * (i & 1u));
						pending &= ~(1u << i);
					}
				}
				if(!pending) break;
				/* bounded, as gather_counts in step_kernel.hip */
				if((++spins & 15u) == 0u) {
					if(ld_agent(glb(nd.status)) != 0u) break;
					if(spins > nd.spinLimit) {
						report_timeout(nd.status, NEMO_STATUS_BARRIER_TIMEOUT, tag, p,
								deal.word(c0, 64u * uint32_t(__builtin_ctz(pending)) + lane) / fwords);
						break;
					}
				}
			}
			uint32_t total = 0;
#pragma unroll
			for(uint32_t i = 0; i < PAIRS; ++i) {
				pos[i] = 0u;
				if(deal.first(c0 + 128u * i) < deal.end) {   /* wave-uniform */
					const uint32_t c = uint32_t(__popcll(m[i]));
					const uint32_t x = wave_scan(c);
					pos[i] = total + x - c;
					total += uint32_t(__builtin_amdgcn_readlane(int(x), 63));
				}
			}
			/* The sources, up to LIST at a time, in LDS so that one lane takes
			 * each: every lane writes its own bits. More than one list (dense
			 * firing): word by word, so that a list's bits are spread over
			 * more lanes. */
			const bool dense = total > LIST;
			uint32_t word = 0, cur = 0, cpos = 0, ctotal = 0, cdone = 0;   /* dense: the word being listed */
			for(uint32_t left = total; left > 0u; ) {   /* wave-uniform */
				uint32_t nsrc = total;
				if(!dense) {
#pragma unroll
					for(uint32_t i = 0; i < PAIRS; ++i) {
						while(m[i]) {
							const uint32_t x = uint32_t(__builtin_ctzll(m[i]));
							list[pos[i]++] = uint16_t((128u * i + 64u * (x >> 5) + lane) * 32u + (x & 31u));
							m[i] &= m[i] - 1ull;
						}
					}
				} else {
					nsrc = 0u;
					while(nsrc < LIST && nsrc < left) {
						while(cdone == ctotal) {   /* the next word that has bits */
#pragma unroll
							for(uint32_t i = 0; i < PAIRS; ++i) {
								if(word >> 1 == i) cur = (word & 1u) ? uint32_t(m[i] >> 32) : uint32_t(m[i]);
							}
							word += 1u;
							const uint32_t c = uint32_t(__popc(cur));
							const uint32_t x = wave_scan(c);
							cpos = x - c;
							ctotal = uint32_t(__builtin_amdgcn_readlane(int(x), 63));
							cdone = 0u;
						}
						const uint32_t take = min(LIST - nsrc, ctotal - cdone);
						while(cur && cpos < cdone + take) {
							list[nsrc + cpos - cdone] = uint16_t((64u * (word - 1u) + lane) * 32u + uint32_t(__builtin_ctz(cur)));
							cur &= cur - 1u;
							cpos += 1u;
						}
						nsrc += take;
						cdone += take;
					}
				}
				left -= nsrc;
				__builtin_amdgcn_wave_barrier();   /* a wave's LDS operations complete in order */
				const bool v0 = lane < nsrc;
				const bool v1 = 64u + lane < nsrc;
				uint32_t a0 = 0, b0r = 0, a1 = 0, b1r = 0;
				if(v0) {
					const uint32_t e = list[lane];
					const NEMO_GLOBAL uint32_t* o = off + size_t(deal.word(c0, e >> 5) * 32u + (e & 31u)) * (P + 1u) + p;
					a0 = ld_off(o);
					b0r = ld_off(o + 1) & offMask;
				}
				if(v1) {
					const uint32_t e = list[64u + lane];
					const NEMO_GLOBAL uint32_t* o = off + size_t(deal.word(c0, e >> 5) * 32u + (e & 31u)) * (P + 1u) + p;
					a1 = ld_off(o);
					b1r = ld_off(o + 1) & offMask;
				}
				__builtin_amdgcn_wave_barrier();   /* the list is written again */
				const uint32_t n0 = a0 >> OFF_NEAR_SHIFT, n1 = a1 >> OFF_NEAR_SHIFT;
				a0 &= offMask;
				a1 &= offMask;
				events += (b0r - a0) + (b1r - a1);
				/* places in the far list. Once a wave asks for more than are
				 * left, no wave gets any more in this cycle, so the places
				 * given are the first farLen of the list, without gaps. */
				uint32_t at = ~0u;
				if(defer && nfw) {
					if(lane == 0u) {
						at = atomicAdd(farAsked + (tag & 1u), nsrc);
						if(at + nsrc > fcap) at = ~0u;
						else atomicAdd(farLen + (tag & 1u), nsrc);
					}
					at = uint32_t(__builtin_amdgcn_readfirstlane(int(at)));
				}
				if(defer && (nfw ? at != ~0u : first)) {
					/* the records of delay 1 (first in each bucket, their count
					 * in the top bits of its start) now, the rest in the next
					 * cycle while its words are under way */
					const uint32_t mx = max(n0, n1);
					const uint32_t sl = (slot + 1u >= D) ? slot + 1u - D : slot + 1u;
					for(uint32_t i = 0; i < mx; i += 2u) {
						const bool ok00 = i < n0, ok01 = i + 1u < n0, ok10 = i < n1, ok11 = i + 1u < n1;
						const uint2 r00 = ld_rec(syn, ok00 ? a0 + i : 0u);
						const uint2 r01 = ld_rec(syn, ok01 ? a0 + i + 1u : 0u);
						const uint2 r10 = ld_rec(syn, ok10 ? a1 + i : 0u);
						const uint2 r11 = ld_rec(syn, ok11 ? a1 + i + 1u : 0u);
						if(ok00) ring_add<SAT>(ringE, ringI, ovf, D, T, fwords, sl, r00.x & 0xffffu, int32_t(r00.y));
						if(ok01) ring_add<SAT>(ringE, ringI, ovf, D, T, fwords, sl, r01.x & 0xffffu, int32_t(r01.y));
						if(ok10) ring_add<SAT>(ringE, ringI, ovf, D, T, fwords, sl, r10.x & 0xffffu, int32_t(r10.y));
						if(ok11) ring_add<SAT>(ringE, ringI, ovf, D, T, fwords, sl, r11.x & 0xffffu, int32_t(r11.y));
					}
					if(nfw) {
						uint2* f = far + (tag & 1u) * fcap + at;
						if(v0) f[lane] = make_uint2(a0 + n0, b0r);
						if(v1) f[64u + lane] = make_uint2(a1 + n1, b1r);
					} else {
						ka0 = a0 + n0;
						kb0 = b0r;
						ka1 = a1 + n1;
						kb1 = b1r;
						kn = nsrc;
						first = false;
					}
				} else {
					deliver_ranges<SAT, IZO>(a0, b0r, a1, b1r, nsrc, lanes(nsrc), lane, slot, syn,
							ringE, ringI, ovf, D, T, fwords);
				}
			}
		}

		if(sched) {
			if(fx != ~0u) force(fx);
			if(ix != ~0u) drive(ix, iv);
			if(takes) {
				for(uint32_t e = fb + sthreads + tid; e < fe; e += sthreads) force(glb(nd.fs_idx)[e]);
				for(uint32_t e = ib + sthreads + tid; e < ie; e += sthreads) drive(glb(nd.is_idx)[e], glb(nd.is_val)[e]);
			}
			fb = fe;
			ib = ie;
			fe = k + 2u < nd.nsteps ? fnext : fe;
			ie = k + 2u < nd.nsteps ? inext : ie;
		}
		if(STDP) __builtin_amdgcn_s_waitcnt(0);   /* this cycle's histories are out */
		__syncthreads();
		wslot = wslot + 1u == R ? 0u : wslot + 1u;
	}

	/* ---- the last cycle's deferred records */
	if(nfw && nd.nsteps > 0u) {
		const uint64_t tc = nd.cycle0 + nd.nsteps - 1u;
		deliver_far<SAT, IZO>(nd, far + (uint32_t(tc) & 1u) * fcap, farLen[uint32_t(tc) & 1u], wave, nwaves, lane,
				uint32_t(tc % D), syn, ringE, ringI, ovf);
	}
	if(kn) {
		deliver_ranges<SAT, IZO>(ka0, kb0, ka1, kb1, kn, lanes(kn), lane,
				uint32_t((nd.cycle0 + nd.nsteps - 1u) % D), syn, ringE, ringI, ovf, D, T, fwords);
	}
	__syncthreads();

	/* ---- save state and the ring for the next launch */
	if(active) {
#pragma unroll
		for(int k = 0; k < NS; ++k) nd.state[size_t(k) * n_total + n] = st[k];
#pragma unroll
		for(int k = 0; k < 4; ++k) nd.rng[size_t(k) * n_total + n] = rng.s[k];
		nd.recent[n] = recent;
	}
	ring_save<SAT>(gring, ringE, ovf, T, D, nd.cycle0 + nd.nsteps, wave, nwaves, lane);
	for(uint32_t d = 32; d >= 1; d >>= 1) {
		events += __shfl_down(events, d, 64);
	}
	if(lane == 0 && events) {
		atomicAdd(nd.events, events);
	}
	__syncthreads();
	if(tid == 0) {
		atomicMax(reinterpret_cast<unsigned long long*>(nd.status + 9), (unsigned long long) wall_clock64());
	}
}

} // namespace

template<bool SAT, bool IZO, bool STDP>
__global__ void __launch_bounds__(1024)
nemo_mask_kernel(const NetDev* __restrict__ nets, const WorkItem* __restrict__ work)
{
	const WorkItem wi = work[blockIdx.x];
	const NetDev nd = nets[wi.net];
	run_masked<SAT, IZO, 4u, STDP, true>(nd, wi.part);
}

/* one network per launch: the descriptor as a kernel argument */
template<bool SAT, bool IZO, uint32_t WORDS, bool STDP>
__global__ void __launch_bounds__(1024)
nemo_mask_kernel_single(const NetDev nd, const WorkItem* __restrict__ work)
{
	run_masked<SAT, IZO, WORDS, STDP, SAT>(nd, work[blockIdx.x].part);
}

namespace {

template<bool SAT, bool IZO, bool STDP>
const void* mask_kernel(uint32_t words)
{
	if(words == 0u) return reinterpret_cast<const void*>(&nemo_mask_kernel<SAT, IZO, STDP>);
	/* saturating networks, whose atomics take more registers, always 4; with
	 * STDP at most 4 */
	if(!SAT && words <= 64u) return reinterpret_cast<const void*>(&nemo_mask_kernel_single<SAT, IZO, SAT ? 4u : 1u, STDP>);
	if(!SAT && !STDP && words > 256u) {
		return reinterpret_cast<const void*>(&nemo_mask_kernel_single<SAT, IZO, SAT || STDP ? 4u : 8u, STDP>);
	}
	return reinterpret_cast<const void*>(&nemo_mask_kernel_single<SAT, IZO, 4u, STDP>);
}

template<bool STDP>
const void* mask_kernel_variant(uint32_t variant, uint32_t words)
{
	switch(variant & 3u) {
	case 0: return mask_kernel<false, false, STDP>(words);
	case 1: return mask_kernel<true, false, STDP>(words);
	case 2: return mask_kernel<false, true, STDP>(words);
	default: return mask_kernel<true, true, STDP>(words);
	}
}

} // namespace

extern "C" {

const void* nemo_dev_mask_kernel(uint32_t variant, uint32_t words)
{
	return (variant & 8u) ? mask_kernel_variant<true>(variant, words) : mask_kernel_variant<false>(variant, words);
}

} // extern "C"
