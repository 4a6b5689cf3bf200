/*
 * step_device.h -- device code the persistent step kernels share
 * (step_kernel.hip, mask_kernel.hip): wave-level sums, device-scope accesses,
 * the LDS ring of pending current and the delivery of synapse records into it.
 */
#ifndef NEMOSIM_STEP_DEVICE_H
#define NEMOSIM_STEP_DEVICE_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "models.h"
#include "step_abi.h"

namespace {

using namespace nemo_dev;

/* Inclusive sum over the lanes of a wave by DPP moves (a scan by shuffles
 * waits for LDS six times: four of them took 0.7 us of a cycle's exchange).
 * Every lane must be active. */
__device__ inline uint32_t wave_scan(uint32_t x)
{
	int v = int(x);
	v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);   /* row_shr:1 */
	v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);   /* row_shr:2 */
	v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);   /* row_shr:4 */
	v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);   /* row_shr:8 */
	v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);   /* row_bcast:15 into rows 1, 3 */
	v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);   /* row_bcast:31 into rows 2, 3 */
	return uint32_t(v);
}

/* Cross-workgroup data (fired lists, their tagged counts, the STDP firing
 * history) is exchanged with agent-scope relaxed atomic loads and stores.
 * On gfx950 these are sc1 accesses, coherent across the XCDs' L2s, so no L2
 * write-back or invalidate is needed. A writer drains its stores
 * (s_waitcnt; __syncthreads alone waits only for LDS traffic) before
 * publishing the count that names them. */
#if defined(__HIP_DEVICE_COMPILE__)
#define NEMO_GLOBAL __attribute__((address_space(1)))
#define NEMO_LDS __attribute__((address_space(3)))
#else
#define NEMO_GLOBAL   /* host pass: the kernels are only parsed there */
#define NEMO_LDS
#endif

/* The network's arrays as global-address-space pointers. Pointers read from
 * the network descriptor are generic, and generic (flat) accesses also count
 * against the LDS wait counter, so every LDS wait would also wait for all
 * outstanding memory loads; global accesses keep the two independent. */
template<typename V>
__device__ inline NEMO_GLOBAL V* glb(V* p)
{
	return (NEMO_GLOBAL V*) p;
}

template<typename V>
__device__ inline void st_agent(NEMO_GLOBAL V* p, V v)
{
	__hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template<typename V>
__device__ inline V ld_agent(const NEMO_GLOBAL V* p)
{
	return __hip_atomic_load(const_cast<NEMO_GLOBAL V*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

/* device-coherent add (two's-complement wrap, as NeMo's int32 accumulator) */
__device__ inline void add_agent(NEMO_GLOBAL int32_t* p, int32_t v)
{
	(void) __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

/* Flags a timed-out wait in the status word; the first one also records
 * where it happened (control block words 4..7, see step_abi.h). */
__device__ inline void report_timeout(uint32_t* status, uint32_t kind, uint32_t cycle, uint32_t part,
		uint32_t awaited)
{
	const uint32_t old = atomicOr(status, kind);
	if(old == 0u) {
		status[3] = cycle;
		status[4] = part;
		status[5] = awaited;
		status[6] = ld_agent(glb(status - 1));
	}
}

/* Loads of a synapse record and of a bucket bound in the delivery loops */
__device__ inline uint2 ld_rec(const NEMO_GLOBAL uint2* syn, uint32_t q)
{
	return syn[q];
}

__device__ inline uint32_t ld_off(const NEMO_GLOBAL uint32_t* o)
{
	return *o;
}

/* With deferred delivery the bucket start off[s][p] carries, in its top
 * 4 bits, the number of delay-1 records at the head of the bucket. */
constexpr uint32_t OFF_NEAR_SHIFT = 28u;

/* Delivery rounds whose record loads are issued together (fewer with the
 * saturating accumulation, whose returning atomics need more registers),
 * and records per lane per round (lane i of a group reads records i and i+G) */
/* rounds of record loads in flight per batch: fewer where the variant has
 * fewer registers left (saturating accumulation; any model, 10 parameters
 * and 4 state variables per neuron) */
template<bool SAT, bool IZO> struct DeliverRounds { static constexpr uint32_t value = SAT ? 4u : (IZO ? 6u : 5u); };
constexpr uint32_t DELIVER_KPL = 2u;

/* Add a Q11.20 weight into ring slot sl of local target tl: the excitatory
 * plane for w >= 0, the inhibitory plane otherwise (as the CPU's split,
 * src/nemo/cpu/Simulation.cpp:299). In saturating mode the returning atomic
 * detects the first partial sum to leave int32 and sets a sticky bit. */
template<bool SAT>
__device__ inline void ring_add(int32_t* ringE, int32_t* ringI, uint32_t* ovf, uint32_t D, uint32_t T,
		uint32_t fwords, uint32_t sl, uint32_t tl, int32_t w)
{
	int32_t* acc = (w >= 0) ? ringE : ringI;
	if(SAT) {
		int32_t old = __hip_atomic_fetch_add(&acc[sl * T + tl], w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
		int64_t sum = int64_t(old) + int64_t(w);
		if(sum > int64_t(INT32_MAX) || sum < int64_t(INT32_MIN)) {
			uint32_t plane = (w >= 0) ? 0u : D;
			atomicOr(&ovf[(plane + sl) * fwords + (tl >> 5)], 1u << (tl & 31u));
		}
	} else {
		__hip_atomic_fetch_add(&acc[sl * T + tl], w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
	}
}

/* One pass of record delivery for up to 128 sources held one per lane
 * (a0/b0 for sources 0..63, a1/b1 for 64..127 of the batch): groups of
 * G = 2^glog lanes share one source, lane i of a group reads records i and
 * i+G of its bucket, so a load instruction touches a few cache lines
 * instead of 64; DELIVER_RU rounds of record loads are issued before their
 * LDS atomics. Rounds [rbeg, rend) of the pass_rounds(nsrc) are done here,
 * so a pass can be split; records from 2G on are left to the caller. */
__device__ inline uint32_t pass_rounds(uint32_t nsrc, uint32_t glog)
{
	return (nsrc + (64u >> glog) - 1u) >> (6u - glog);
}

template<bool SAT, bool IZO>
__device__ inline void deliver_pass(uint32_t a0, uint32_t b0, uint32_t a1, uint32_t b1, uint32_t nsrc,
		uint32_t glog, uint32_t lane, uint32_t base, const NEMO_GLOBAL uint2* syn,
		int32_t* ringE, int32_t* ringI, uint32_t* ovf, uint32_t D, uint32_t T, uint32_t fwords,
		uint32_t rbeg, uint32_t rend)
{
	const uint32_t G = 1u << glog;
	const uint32_t NG = 64u >> glog;                 /* sources per round */
	const uint32_t grp = lane >> glog;
	const uint32_t gl = lane & (G - 1u);
	const uint32_t rounds = rend;
	constexpr uint32_t DELIVER_RU = DeliverRounds<SAT, IZO>::value;
	for(uint32_t r0 = rbeg; r0 < rounds; r0 += DELIVER_RU) {    /* wave-uniform */
		uint2 rec[DELIVER_RU][DELIVER_KPL];
		uint32_t ok = 0;
#pragma unroll
		for(uint32_t u = 0; u < DELIVER_RU; ++u) {
			const uint32_t k = (r0 + u) * NG + grp;      /* source within the batch */
			const bool hi = ((r0 + u) * NG) >= 64u;     /* wave-uniform */
			const uint32_t ak = __shfl(hi ? a1 : a0, int(k & 63u), 64);
			const uint32_t bk = __shfl(hi ? b1 : b0, int(k & 63u), 64);
			const bool live = (r0 + u < rounds) && (k < nsrc);
#pragma unroll
			for(uint32_t i = 0; i < DELIVER_KPL; ++i) {
				const uint32_t q = ak + gl + i * G;
				const bool valid = live && (q < bk);
				/* the first load of a round is issued by every lane (record 0
				 * stands in for absent ones); the later ones only when some
				 * lane of the wave has a record there: buckets rarely reach
				 * past G records, and the vector memory unit's time goes by
				 * load instructions, not by the records they carry */
				if(i == 0 || __any(valid)) {   /* wave-uniform */
					rec[u][i] = ld_rec(syn, valid ? q : 0u);
				} else {
					rec[u][i] = make_uint2(0u, 0u);
				}
				ok |= uint32_t(valid) << (u * DELIVER_KPL + i);
			}
		}
#pragma unroll
		for(uint32_t u = 0; u < DELIVER_RU; ++u) {
#pragma unroll
			for(uint32_t i = 0; i < DELIVER_KPL; ++i) {
				if((ok >> (u * DELIVER_KPL + i)) & 1u) {
					const uint2 r = rec[u][i];
					uint32_t sl = base + (r.x >> 16);
					sl = (sl >= D) ? sl - D : sl;
					ring_add<SAT>(ringE, ringI, ovf, D, T, fwords, sl, r.x & 0xffffu, int32_t(r.y));
				}
			}
		}
	}
}

/* Delivers the records [a, b) of up to 128 sources held one per lane into
 * the ring, relative to base slot `base`. The first pass takes up to 2G
 * records of every bucket. The remainders of longer buckets are then packed
 * into the first lanes (each lane pushes its range to the lane of its rank
 * among the long ones) and delivered by further passes, so a long bucket
 * costs one more round of loads for the whole wave, not one per bucket.
 * All lanes of the wave must call it together (nsrc is wave-uniform). */
template<bool SAT, bool IZO>
__device__ inline void deliver_ranges(uint32_t a0, uint32_t b0, uint32_t a1, uint32_t b1, uint32_t nsrc,
		uint32_t glog, uint32_t lane, uint32_t base, const NEMO_GLOBAL uint2* syn,
		int32_t* ringE, int32_t* ringI, uint32_t* ovf, uint32_t D, uint32_t T, uint32_t fwords)
{
	const uint32_t covered = DELIVER_KPL << glog;   /* records per bucket taken by a pass */
	if(lane >= nsrc) { a0 = b0 = 0u; }
	if(64u + lane >= nsrc) { a1 = b1 = 0u; }
	for(;;) {
		deliver_pass<SAT, IZO>(a0, b0, a1, b1, nsrc, glog, lane, base, syn, ringE, ringI, ovf, D, T, fwords,
				0u, pass_rounds(nsrc, glog));
		/* what the pass left */
		a0 = (b0 - a0 > covered) ? a0 + covered : b0;
		a1 = (b1 - a1 > covered) ? a1 + covered : b1;
		const uint64_t m0 = __ballot(a0 < b0);
		const uint64_t m1 = __ballot(a1 < b1);
		const uint32_t n0 = uint32_t(__popcll(m0));
		const uint32_t nl = n0 + uint32_t(__popcll(m1));
		if(nl == 0u) {
			return;
		}
		if(nl > 63u) {
			/* too many to pack into one register: another pass as they are */
			nsrc = 128u;
			continue;
		}
		/* pack: a long source goes to the lane of its rank; the others to
		 * lane 63, which no rank reaches */
		const uint32_t below = uint32_t(__popcll(m0 & ((1ull << lane) - 1ull)));
		const uint32_t below1 = uint32_t(__popcll(m1 & ((1ull << lane) - 1ull)));
		const int dst0 = int(((a0 < b0) ? below : 63u) * 4u);
		const int dst1 = int(((a1 < b1) ? n0 + below1 : 63u) * 4u);
		const uint32_t pa0 = uint32_t(__builtin_amdgcn_ds_permute(dst0, int(a0)));
		const uint32_t pb0 = uint32_t(__builtin_amdgcn_ds_permute(dst0, int(b0)));
		const uint32_t pa1 = uint32_t(__builtin_amdgcn_ds_permute(dst1, int(a1)));
		const uint32_t pb1 = uint32_t(__builtin_amdgcn_ds_permute(dst1, int(b1)));
		a0 = (lane < n0) ? pa0 : pa1;
		b0 = (lane < n0) ? pb0 : pb1;
		if(lane >= nl) { a0 = b0 = 0u; }
		a1 = b1 = 0u;
		nsrc = nl;
	}
}

/* Row r (plane E for r < D, then I; LDS slot r mod D) of the LDS ring as a row
 * of the ring in memory, whose planes have D+1 slots. s0 and m0 are the slots
 * of the first pending cycle in each. */
__device__ inline uint32_t ring_row(uint32_t r, uint32_t D, uint32_t s0, uint32_t m0)
{
	const uint32_t plane = r >= D ? 1u : 0u;
	const uint32_t sl = r - plane * D;
	uint32_t m = m0 + (sl >= s0 ? sl - s0 : sl + D - s0);
	m = m >= D + 1u ? m - (D + 1u) : m;
	return plane * (D + 1u) + m;
}

/* The LDS ring (excitatory plane, then inhibitory) from the ring in memory,
 * slot by slot: LDS slot t mod D of the input of cycle t is slot t mod (D+1)
 * there (which cycle_kernel.hip needs). Up to 1 KB per wave instruction
 * straight into LDS (16 bytes per lane), every load in flight at once; the
 * caller's barrier follows. */
__device__ inline void ring_restore(const int32_t* gring, int32_t* ringE, uint32_t T, uint32_t D, uint64_t cycle,
		uint32_t wave, uint32_t nwaves, uint32_t lane)
{
	const uint32_t s0 = uint32_t(cycle % D), m0 = uint32_t(cycle % (D + 1u));
	for(uint32_t r = wave; r < 2u * D; r += nwaves) {   /* wave-uniform */
		const int32_t* src = gring + size_t(ring_row(r, D, s0, m0)) * T;
		for(uint32_t c = 0; c < T; c += 256u) {
			if(c + lane * 4u < T) {
				__builtin_amdgcn_global_load_lds((NEMO_GLOBAL void*)(src + c + lane * 4u),
						(NEMO_LDS void*)(ringE + r * T + c), 16, 0, 0);
			}
		}
	}
	__builtin_amdgcn_s_waitcnt(0);
}

/* The ring in memory from the LDS ring at the end of a launch, with sticky
 * overflow bits folded into the values; the slot of no pending cycle, that of
 * cycle + D, starts empty. */
template<bool SAT>
__device__ inline void ring_save(int32_t* gring, const int32_t* ringE, const uint32_t* ovf, uint32_t T, uint32_t D,
		uint64_t cycle, uint32_t wave, uint32_t nwaves, uint32_t lane)
{
	const uint32_t fwords = T >> 5;
	const uint32_t s0 = uint32_t(cycle % D), m0 = uint32_t(cycle % (D + 1u));
	for(uint32_t r = wave; r < 2u * D; r += nwaves) {   /* wave-uniform; 16 bytes per lane */
		NEMO_GLOBAL int4* dst = glb(reinterpret_cast<int4*>(gring + size_t(ring_row(r, D, s0, m0)) * T));
		const int4* src = reinterpret_cast<const int4*>(ringE + r * T);
		for(uint32_t c = lane; c < T / 4u; c += 64u) {
			int4 v = src[c];
			if(SAT) {
				const uint32_t o = ovf[r * fwords + (c >> 3)] >> (4u * (c & 7u));
				const int32_t lim = r < D ? INT32_MAX : INT32_MIN;
				if(o & 1u) v.x = lim;
				if(o & 2u) v.y = lim;
				if(o & 4u) v.z = lim;
				if(o & 8u) v.w = lim;
			}
			dst[c] = v;
		}
	}
	const uint32_t e0 = m0 ? m0 - 1u : D;
	for(uint32_t c = wave * 64u + lane; c < T; c += nwaves * 64u) {
		gring[size_t(e0) * T + c] = 0;
		gring[size_t(D + 1u + e0) * T + c] = 0;
	}
}

/* The ring of pending current from the firing history, when weights changed
 * (applyStdp) since it was filled. NeMo reads a weight when the spike arrives
 * (src/nemo/cpu/Simulation.cpp:258-307): every spike fired at cycle0-1-k whose
 * synapse delay d > k has not arrived yet and lands in slot (cycle0-1-k+d) mod
 * D, with the current weight. The ring is zero before. A wave reads the
 * histories of 256 sources at a time and the bucket bounds of those
 * that fired, all loads in flight together; then 1 << glog2 lanes share a
 * source's records. One lane per source took 0.67 ms a launch for 50k neurons x
 * 1000 and 0.15 ms for 3k x 300. */
template<bool SAT>
__device__ inline void ring_replay(const NetDev& nd, uint32_t p, const NEMO_GLOBAL uint2* syn,
		const NEMO_GLOBAL uint32_t* off, uint32_t offMask, int32_t* ringE, int32_t* ringI, uint32_t* ovf,
		uint32_t fwords, uint32_t wave, uint32_t nwaves, uint32_t lane)
{
	constexpr uint32_t REPLAY_U = 4u;   /* groups of 64 sources */
	const uint32_t D = nd.D, T = nd.T, P = nd.P, glog = nd.glog2;
	const uint32_t G = 1u << glog, NG = 64u >> glog;
	const uint32_t grp = lane >> glog, gl = lane & (G - 1u);
	const uint64_t pend = (D >= 64u) ? ~0ull : ((1ull << D) - 1ull);
	const uint32_t last = uint32_t((nd.cycle0 + D - 1u) % D);    /* slot of cycle0-1 */
	for(uint32_t s0 = wave * 64u * REPLAY_U; s0 < nd.n; s0 += nwaves * 64u * REPLAY_U) {   /* wave-uniform */
		uint64_t h[REPLAY_U];
		uint32_t a[REPLAY_U], b[REPLAY_U];
#pragma unroll
		for(uint32_t u = 0; u < REPLAY_U; ++u) {
			const uint32_t s = s0 + 64u * u + lane;
			h[u] = (s < nd.n) ? glb(nd.recent)[s] & pend : 0ull;
		}
#pragma unroll
		for(uint32_t u = 0; u < REPLAY_U; ++u) {
			a[u] = b[u] = 0u;
			if(h[u]) {
				const NEMO_GLOBAL uint32_t* o = off + size_t(s0 + 64u * u + lane) * (P + 1u) + p;
				a[u] = ld_off(o) & offMask;
				b[u] = ld_off(o + 1) & offMask;
			}
		}
#pragma unroll
		for(uint32_t u = 0; u < REPLAY_U; ++u) {
			/* the sources with records to the front lanes */
			const bool has = a[u] < b[u];
			const uint64_t m = __ballot(has);
			const uint32_t cnt = uint32_t(__popcll(m));
			if(cnt == 0u) continue;   /* wave-uniform */
			const uint64_t below = (1ull << lane) - 1ull;
			const int dst = int((has ? uint32_t(__popcll(m & below)) : cnt + uint32_t(__popcll(~m & below))) * 4u);
			const uint32_t pa = uint32_t(__builtin_amdgcn_ds_permute(dst, int(a[u])));
			const uint32_t pb = uint32_t(__builtin_amdgcn_ds_permute(dst, int(b[u])));
			const uint32_t h0 = uint32_t(__builtin_amdgcn_ds_permute(dst, int(uint32_t(h[u]))));
			const uint32_t h1 = uint32_t(__builtin_amdgcn_ds_permute(dst, int(uint32_t(h[u] >> 32))));
			for(uint32_t k0 = 0; k0 < cnt; k0 += NG) {   /* wave-uniform */
				const uint32_t k = k0 + grp;
				const uint32_t ak = __shfl(pa, int(k & 63u), 64);
				const uint32_t bk = __shfl(pb, int(k & 63u), 64);
				const uint64_t hk = (uint64_t(uint32_t(__shfl(h1, int(k & 63u), 64))) << 32)
					| uint32_t(__shfl(h0, int(k & 63u), 64));
				const uint32_t end = k < cnt ? bk : ak;
				for(uint32_t q = ak + gl; __any(q < end); q += 2u * G) {   /* wave-uniform */
					const bool ok0 = q < end, ok1 = q + G < end;
					const uint2 r0 = ld_rec(syn, ok0 ? q : 0u);
					const uint2 r1 = ld_rec(syn, ok1 ? q + G : 0u);
					auto arrive = [&](const uint2& rec) {
						const uint32_t d = rec.x >> 16;
						uint64_t hb = hk & ((d >= 64u) ? ~0ull : ((1ull << d) - 1ull));
						while(hb) {
							const uint32_t kk = uint32_t(__builtin_ctzll(hb));
							hb &= hb - 1ull;
							ring_add<SAT>(ringE, ringI, ovf, D, T, fwords, (last + d - kk) % D, rec.x & 0xffffu,
									int32_t(rec.y));
						}
					};
					if(ok0) arrive(r0);
					if(ok1) arrive(r1);
				}
			}
		}
	}
}

} // namespace

#endif
