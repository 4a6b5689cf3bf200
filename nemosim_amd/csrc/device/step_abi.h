/*
 * step_abi.h -- plain-old-data structures shared by the C++ host code and
 * the HIP kernels (the internal C-ABI between them). No HIP types appear
 * here, so the host side compiles against it with any C++ compiler.
 */
#ifndef NEMOSIM_STEP_ABI_H
#define NEMOSIM_STEP_ABI_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* Bits of NetDev.flags */
#define NEMO_NET_STDP      1u   /* accumulate STDP this launch */
#define NEMO_NET_SATURATE  2u   /* accumulators may leave the int32 range */
#define NEMO_NET_REPLAY    4u   /* weights changed since the ring was filled:
                                 * rebuild it from the firing history */
#define NEMO_NET_IZHIKEVICH_ONLY 16u  /* every neuron is an Izhikevich neuron */
#define NEMO_NET_DEFER     8u   /* delay-1 records first in each bucket, their
                                 * count in bits 28..31 of off[]; records of
                                 * delay >= 2 are delivered one cycle later */
#define NEMO_NET_PREF_RING 32u  /* STDP: prefixes of the fired counts of the last
                                 * postLen cycles kept in LDS */

#define NEMO_NET_MASKS 64u      /* fired bits exchanged as words (mask_kernel.hip) */

/* Bits of the per-network status word */
#define NEMO_STATUS_BARRIER_TIMEOUT 1u   /* a fired count never arrived */
#define NEMO_STATUS_ENTRY_TIMEOUT   2u   /* a fired-list entry never arrived */

/* The per-network control block (16 words): [0] workgroups started, [1]
 * status, [2..3] delivered-synapse count, and, for the first timeout,
 * [4] cycle, [5] waiting partition, [6] awaited partition, [7] workgroups
 * started by then; [8..9] the earliest start and [10..11] the latest end
 * of its workgroups on the device wall clock, all-ones and zero before a
 * launch. */
#define NEMO_CTL_WORDS 16u

/*
 * One simulated network as seen by the step kernel. Neurons use
 * simulation-local indices 0..n-1; partition p owns neurons [p*T, p*T+T).
 * All arrays are device pointers.
 */
typedef struct NetDev {
	uint32_t n;          /* neurons */
	uint32_t P;          /* partitions (workgroups) */
	uint32_t T;          /* neurons per partition, multiple of 64, <= 1024 */
	uint32_t D;          /* delay-ring depth = maximum delay (1..64) */
	uint32_t words;      /* 64-bit raster words per step = P*T/64 */
	uint32_t flags;      /* NEMO_NET_* */
	uint32_t nsteps;     /* steps this network runs in the current launch */
	uint32_t spinLimit;  /* barrier spin bound (iterations) */
	uint32_t glog2;      /* log2 of the lanes that share one fired source in delivery (0..6) */
	uint32_t glogFew;    /* the same where a wave has few fired sources (NEMO_NET_MASKS; >= glog2) */
	uint32_t flRing;     /* fired lists and counts, or fired words, kept for this many cycles (buffer t mod flRing) */
	uint32_t stdpCache;  /* STDP chunks whose reverse records are staged in LDS (64 words each) */
	uint32_t stdpWaves;  /* waves for STDP after those of the neurons (NEMO_NET_MASKS) */
	uint32_t farWaves;   /* with NEMO_NET_MASKS and NEMO_NET_DEFER: waves after those that deliver the previous
	                      * cycle's far records (0: the neurons' waves do) */
	uint32_t exWaves;    /* with NEMO_NET_DEFER: waves of a workgroup that run the exchange and the
	                      * delay-1 delivery while the others deliver the previous cycle's far
	                      * records (0: every wave does both, one after the other) */
	uint32_t farCap;     /* fired sources per cycle whose far ranges fit the LDS far list (multiple
	                      * of 64; with exWaves or farWaves) */
	uint64_t cycle0;     /* cycle count at the start of the launch */

	const uint8_t* model;     /* [n] model id */
	float* param;             /* [MAX_PARAM][n] */
	float* state;             /* [MAX_STATE][n] */
	uint32_t* rng;            /* [4][n] */
	uint64_t* recent;         /* [n] firing history, bit 0 = last cycle */
	int32_t* ring;            /* [P][2][D+1][T] pending current between launches: slot t mod (D+1) for
	                           * the input of cycle t, the slot of no pending cycle zero */

	/* forward matrix: synapses of source s bucketed by target partition;
	 * partition p's bucket is syn[off[s*(P+1)+p] .. off[s*(P+1)+p+1]).
	 * Record = {target - p*T | delay << 16, Q11.20 weight}. */
	const uint32_t* off;
	uint32_t* syn;            /* [2 * synapses] */

	/* per-step exchange between the network's workgroups, double-buffered
	 * by cycle parity */
	uint64_t* fl;             /* [flRing][P][T] fired neurons of each partition, (cycle << 32) | neuron */
	uint64_t* fc;             /* [flRing][P] (cycle << 32) | fired count; starts all-ones */
	uint64_t* mk;             /* [flRing][nemo_mask_words(P*T/32)] (cycle << 32) | 32 fired bits; starts all-ones (NEMO_NET_MASKS) */
	uint64_t* rfg;            /* [2][n], with NEMO_NET_MASKS [4][n], firing history by cycle (STDP only) */
	uint32_t* status;         /* NEMO_STATUS_* */
	unsigned long long* events; /* delivered-synapse counter */

	/* reverse matrix of plastic synapses (STDP) */
	const uint32_t* rcm_start;   /* [n+1] */
	const uint32_t* rcm_sd;      /* source | (delay-1) << 26 */
	const uint32_t* rcm_fwd;     /* index of the synapse record */
	int32_t* rcm_acc;            /* accumulated weight change */
	const void* stdp;            /* StdpParams */
	uint64_t* srow;              /* [flRing][P][T] reverse row {start, length} of each fired
	                              * neuron, at its fired-list position (STDP only) */

	/* stimulus of this launch, CSR over steps (sim-local indices); NULL if none */
	const uint32_t* fs_ptr;
	const uint32_t* fs_idx;
	const uint32_t* is_ptr;
	const uint32_t* is_idx;
	const float* is_val;

	uint64_t* raster;         /* [nsteps][words] fired bits */
} NetDev;

/* One cycle by cycle_kernel.hip: its stimulus (one current per neuron) and its
 * report */
#define NEMO_CYCLE_STIM 64u
#define NEMO_DONE_GROUPS 16u   /* first-level counters of finished workgroups */

/* what the last workgroup of a launch writes to host memory: the device wall
 * clock at its start and end, then the launch's number */
typedef struct CycleReport {
	uint64_t start, end;
	uint32_t ctl[8];          /* the control block's first words (nemo_dev_step_report) */
	uint64_t sequence;
} CycleReport;

typedef struct CycleArgs {
	uint32_t slot;            /* cycle0 mod (D+1) */
	uint32_t nf, ni;
	uint64_t* hostRow;        /* the cycle's raster words in host memory too */
	CycleReport* report;      /* host memory */
	uint64_t sequence;
	uint32_t* done;           /* [1 + NEMO_DONE_GROUPS][32] counters, zero between launches */
	uint32_t fidx[NEMO_CYCLE_STIM];
	uint32_t iidx[NEMO_CYCLE_STIM];
	float ival[NEMO_CYCLE_STIM];
} CycleArgs;

/* blockIdx -> (network, partition) */
typedef struct WorkItem {
	uint32_t net;
	uint32_t part;
} WorkItem;

/* Kernel launchers (nemosim_amd/csrc/device/step_kernel.hip). They return a
 * hipError_t value as int and take a hipStream_t as void*. */
/* Step-kernel variants: bit 0 = saturating accumulation (NEMO_NET_SATURATE),
 * bit 1 = Izhikevich-only network (NEMO_NET_IZHIKEVICH_ONLY), bit 2 = fired
 * bits exchanged as words (NEMO_NET_MASKS, mask_kernel.hip), bit 3 = STDP
 * there. All networks of one launch must be of the launch's variant. */
static inline uint32_t nemo_step_variant(uint32_t flags)
{
	return ((flags & NEMO_NET_SATURATE) ? 1u : 0u) | ((flags & NEMO_NET_IZHIKEVICH_ONLY) ? 2u : 0u)
		| ((flags & NEMO_NET_MASKS) ? 4u : 0u)
		| ((flags & (NEMO_NET_MASKS | NEMO_NET_STDP)) == (NEMO_NET_MASKS | NEMO_NET_STDP) ? 8u : 0u);
}
/* The kernel of mask_kernel.hip for a variant: for one network whose waves
 * take up to `words` words each, or for batches (words = 0) */
const void* nemo_dev_mask_kernel(uint32_t variant, uint32_t words);
int nemo_dev_step_launch(const NetDev* nets_dev, const WorkItem* work_dev, uint32_t nblocks,
		uint32_t blockDim, uint32_t ldsBytes, uint32_t variant, void* stream);
/* One network: the descriptor is passed by value (nd_host is read at the
 * call), the work table maps blocks to its partitions. */
int nemo_dev_step_launch_one(const NetDev* nd_host, const WorkItem* work_dev, uint32_t nblocks,
		uint32_t blockDim, uint32_t ldsBytes, uint32_t variant, void* stream);
/* One cycle of a network without STDP whose sums stay within int32 */
int nemo_dev_cycle(const NetDev* nd_host, const CycleArgs* ca, void* stream);
/* whether the bucket bounds of P partitions fit its LDS */
int nemo_dev_cycle_fits(uint32_t P);
/* *out (host memory) = the most synapses of a source, whose rows start at
 * off[i * stride] & mask; max: a zero word, done: counters as in CycleArgs */
int nemo_dev_longest_row(const uint32_t* off, uint32_t stride, uint32_t n, uint32_t mask, uint32_t* max, uint32_t* done,
		uint32_t* out, void* stream);
/* neurons of one of its workgroups, a power of two */
uint32_t nemo_dev_cycle_block_neurons(uint32_t P, uint32_t T);
/* The end of a launch of one network, after its step kernel on the stream: its
 * control block to host memory, then the report; the clock words start anew. */
int nemo_dev_step_report(uint32_t* ctl, CycleReport* report, uint64_t sequence, void* stream);
/* Workgroups that the device holds at once: of the batched launch's kernel, or
 * with P partitions of T neurons (P > 0) of that and of the one that a launch of
 * such a network alone takes, whichever are fewer. */
int nemo_dev_step_max_blocks(uint32_t blockDim, uint32_t ldsBytes, uint32_t variant, uint32_t P, uint32_t T,
		uint32_t* maxBlocks);
/* Batched step as an instantiated HIP graph (clear -> persistent step ->
 * collect); collect_dev receives [nnets][16] words: the first 12 words of
 * each network's control block, the last four of them the first start and
 * the last end of its workgroups on the device wall clock (64-bit each; the
 * graph initialises them before the step kernel). The graph reads
 * nets_dev/work_dev at replay time. */
int nemo_dev_batch_graph_create(const NetDev* nets_dev, uint32_t nnets, const WorkItem* work_dev,
		uint32_t nblocks, uint32_t blockDim, uint32_t ldsBytes, uint32_t variant, uint32_t* collect_dev,
		void** exec_out);
int nemo_dev_graph_launch(void* exec, void* stream);
int nemo_dev_graph_destroy(void* exec);
/* The allocation-free run's scratch array: 4-byte words, one array per
 * device. nemo_dev_static_scratch gives its device address on the current
 * device (looked up once per device with hipGetSymbolAddress). The caller
 * holds the library's device lock. */
#define NEMO_STATIC_SCRATCH_WORDS (1u << 20)
int nemo_dev_static_scratch(void** ptr);
int nemo_dev_apply_stdp(uint32_t* syn, const uint32_t* rcm_fwd, int32_t* rcm_acc, size_t nr,
		const void* stdp_dev, int32_t fx_reward, void* stream);
int nemo_dev_fill_u32(uint32_t* p, uint32_t value, size_t n, void* stream);
int nemo_dev_fill_u64(uint64_t* p, uint64_t value, size_t n, void* stream);
/* Where a kernel says that it is done: its last workgroup writes `sequence`
 * to *seen in host memory, which the caller polls. done: counters of finished
 * workgroups, zero between launches. */
typedef struct DoneReport {
	uint64_t* seen;
	uint64_t sequence;
	uint32_t* done;           /* [1 + NEMO_DONE_GROUPS][32] */
} DoneReport;

/* The raster of a run (rows of `words` 64-bit words, one per cycle) as fired
 * counts and ids (csrc/device/raster_kernel.hip). counts and out are host
 * memory the device can reach (pinned), offs is device memory: its first call
 * writes counts[t] and, with offs, the positions offs[t] of the cycles' ids in
 * the run's list. The second writes the ids with positions in [lo, hi) to
 * out[position - lo], as ids[local index], or first + local index where ids is
 * NULL. Both report. */
int nemo_dev_raster_count(const uint64_t* raster, uint32_t words, uint32_t n, uint32_t cycles, uint32_t* counts,
		uint32_t* devCounts, uint64_t* offs, const DoneReport* report, void* stream);
int nemo_dev_raster_ids(const uint64_t* raster, uint32_t words, uint32_t n, uint32_t cycles, const uint64_t* offs,
		uint64_t lo, uint64_t hi, const uint32_t* ids, uint32_t first, uint32_t* out, const DoneReport* report,
		void* stream);
/* *out (host memory) = the 4-byte word at src, then the report */
int nemo_dev_peek(const uint32_t* src, uint32_t* out, const DoneReport* report, void* stream);
/* Evaluates the device math pieces on inputs in[] (for tests):
 * kind 0 = logf_glibc(in), 1 = sinf_rng(in), 2 = kuramoto_wrap(in), 3 = sinf_glibc(in) */
int nemo_dev_eval_libm(int kind, const float* in_dev, float* out_dev, size_t n, void* stream);
int nemo_dev_nrand_seq(const uint32_t* state4_dev, float* out_dev, size_t n, void* stream);

/* Bytes of LDS the STDP tables take (the StdpParams of models.h, rounded) */
#define NEMO_STDP_LDS_BYTES 576u
/* Entries of a workgroup's per-cycle STDP work list (64-synapse chunks), and
 * of each of mask_kernel.hip's two */
#define NEMO_STDP_WORK_CAP 1024u
#define NEMO_MASK_STDP_CAP 512u

/* LDS bytes the step kernel needs for partitions of T neurons, ring depth D,
 * P partitions. Optional STDP areas follow, in this order, when the host
 * finds room for them: stdpCache x 256 bytes of staged reverse records, then
 * with NEMO_NET_PREF_RING postLen x ((P+1) rounded up to 64) x 4 bytes.
 * With exchange waves the far list follows: NEMO_FAR_LDS_BYTES(farCap). */
/* far list: [2][farCap] range starts, [2][farCap] range ends, two counts
 * and the exchange waves' flag */
#define NEMO_FAR_LDS_BYTES(cap) (16u * (cap) + 16u)

static inline uint32_t nemo_step_lds_bytes(uint32_t T, uint32_t D, uint32_t P, int saturate, int stdp)
{
	uint32_t b = 0;
	b += 2u * D * T * 4u;          /* ringE, ringI */
	b += T * 4u;                   /* external current / STDP target list */
	b += (T / 32u) * 4u;           /* forced-firing bits */
	b += ((P + 1u + 63u) & ~63u) * 4u; /* partition prefix */
	b += 64u * 4u;                 /* wave sums / scratch */
	if(saturate) {
		b += 2u * D * (T / 32u) * 4u;  /* overflow bits */
	}
	if(stdp) {
		b += NEMO_STDP_LDS_BYTES;      /* STDP tables */
		b += NEMO_STDP_WORK_CAP * 8u + 64u;  /* STDP work list and its counters */
		b += ((P + 1u + 63u) & ~63u) * 4u;   /* prefix of the counts of the targets' cycle */
	}
	return b;
}

/* words between cycles in NetDev.mk: whole lines of memory */
#ifdef __HIPCC__
__host__ __device__
#endif
static inline uint32_t nemo_mask_words(uint32_t words) { return (words + 15u) & ~15u; }

/* LDS bytes of mask_kernel.hip: the ring, external current, forced-firing
 * bits, overflow bits and 128 16-bit sources per wave */
static inline uint32_t nemo_mask_lds_bytes(uint32_t T, uint32_t D, int saturate)
{
	return 2u * D * T * 4u + T * 4u + (T / 32u) * 4u + (saturate ? 2u * D * (T / 32u) * 4u : 0u) + (T / 64u) * 256u;
}

/* and with farWaves: two far lists (by cycle parity) of cap ranges, and their
 * lengths, at the end */
#define NEMO_MASK_FAR_LDS_BYTES(cap) (16u * (cap) + 16u)

/* with STDP: the sources of its waves, the tables, two work lists (by
 * cycle parity) and their lengths, and the staged reverse records of both */
static inline uint32_t nemo_mask_stdp_lds_bytes(uint32_t waves, uint32_t cache)
{
	return waves * 256u + NEMO_STDP_LDS_BYTES + 2u * NEMO_MASK_STDP_CAP * 8u + 64u + 2u * cache * 256u;
}

#ifdef __cplusplus
}
#endif

#endif
