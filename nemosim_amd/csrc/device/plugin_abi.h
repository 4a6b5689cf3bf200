/*
 * plugin_abi.h -- POD descriptor of one network for the per-cycle step
 * kernels in plugin_step.hip (plugins, and built-in models beyond the fused
 * kernel's range), shared by host C++ and HIP.
 */
#ifndef NEMOSIM_PLUGIN_ABI_H
#define NEMOSIM_PLUGIN_ABI_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

typedef struct PluginStepDev {
	uint32_t n;            /* neurons */
	uint32_t D;            /* maximum delay */
	uint32_t words32;      /* 32-bit raster words per cycle (even: whole 64-bit words) */
	uint32_t R;            /* ring depth: D with plugins; D + 1 for built-in models, whose spikes are
	                        * delivered while other neurons still read the cycle's slot */
	uint64_t cycle0;       /* cycle at the start of the run */

	void* acc;             /* [2][R][n] pending E (plane 0) and I (plane 1) current, Q11.20: int64;
	                        * int32 for built-in models where no sum can leave that range */
	float* curE;           /* [n] this cycle's input, converted */
	float* curI;
	float* curX;           /* [n] external current */
	uint32_t* fstim;       /* [words32] forced-firing bits */
	uint32_t* raster;      /* [cycles][words32] fired bits; the plugin's `fired` row */
	const uint32_t* off;   /* [n+1] synapses of source s: syn[off[s] .. off[s+1]) */
	const uint32_t* syn;   /* records {target | (delay-1) << 26, Q11.20 weight} */
	uint64_t* recent;      /* [n] firing history */
	unsigned long long* part;   /* [NEMO_PM_PARTS][16] delivered synapses, in the first word of each line */

	/* built-in models */
	const uint8_t* model;  /* [n] */
	const float* param;    /* [MAX_PARAM][n] */
	float* state;          /* [MAX_STATE][n] */
	uint32_t* rng;         /* [4][n] */

	const uint32_t* rcm_start;
	const uint32_t* rcm_sd;
	int32_t* rcm_acc;
	const void* stdp;

	const uint32_t* fs_ptr;
	const uint32_t* fs_idx;
	const uint32_t* is_ptr;
	const uint32_t* is_idx;
	const float* is_val;
} PluginStepDev;

int nemo_dev_pm_begin(const PluginStepDev* s, uint32_t k, void* stream);
int nemo_dev_pm_stimulus(const PluginStepDev* s, uint32_t k, uint32_t entries, void* stream);
/* narrow: int32 accumulators; longRows: neighbours with long rows */
int nemo_dev_pm_scatter(const PluginStepDev* s, uint32_t k, int narrow, int longRows, void* stream);
int nemo_dev_pm_stdp(const PluginStepDev* s, void* stream);
/* rebuilds the zeroed ring */
int nemo_dev_pm_replay(const PluginStepDev* s, int narrow, void* stream);
/* one cycle of built-in models; stim: the cycle's stimulus is in fstim and
 * curX, which are cleared; deliver: with its spikes, otherwise nemo_dev_pm_scatter follows */
int nemo_dev_pm_cycle(const PluginStepDev* s, uint32_t k, int stim, int narrow, int izhikevichOnly, int deliver,
		void* stream);
#define NEMO_PM_SCATTER_BLOCKS 2048u
#define NEMO_PM_PARTS 64u

#ifdef __cplusplus
}
#endif

#endif
