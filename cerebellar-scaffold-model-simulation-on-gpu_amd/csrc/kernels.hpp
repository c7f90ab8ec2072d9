// kernels.hpp -- launchers of the gfx950 kernels (kernels.hip) used by the engine.
#pragma once
#include <hip/hip_runtime.h>

#include "model.hpp"

namespace sc {

#define HIP_TRY(x)                                                                                   \
    do {                                                                                             \
        hipError_t e_ = (x);                                                                         \
        if (e_ != hipSuccess)                                                                        \
            return fail(SCAFFOLD_ERR_HIP, "%s: %s (%s:%d)", #x, hipGetErrorString(e_), __FILE__, __LINE__); \
    } while (0)

// Device work of one step: blocks and the descriptor arrays they index.
struct DevWork {
    ScLayout layout{};
    int n_blocks = 0;
    const ScLaneTask *lanes = nullptr;
    const ScStimTask *stims = nullptr;
    const ScTeamTask *teams = nullptr;
    bool idx16 = false;  // some descriptor holds 16-bit column offsets
    bool nontemporal = false;  // synapse streams loaded as nontemporal (networks beyond the L2)
    std::vector<ScTeamTask> h_teams;  // host copies: the team descriptors as uploaded, the staging plan
    std::vector<ScStage> h_stages;
    const ScStage *stages = nullptr;  // per block: spike windows staged in LDS (nullptr: none)
    int n_staged = 0;                 // blocks with staged windows
    int max_groups = 0;               // most 64-neuron groups of one instance (statistics grid)
    std::vector<ScPlastic> plastic;   // plasticity rules, applied in order after each step
    const ScPlastic *d_plastic = nullptr;  // the rules on the device (window-count blocks of the step kernel)
    unsigned int *end_done = nullptr;      // arrival counters of the run-end kernel (zero between launches): 2, and
                                           // one per instance of a batch
    ScHostStats host{};                    // places of the statistics' copies (one network)
    const ScHostStats *hosts = nullptr;    // per instance of a batch, on the device
};

// Output spike train of a run's last T steps: n_out output neurons at device bits
// bits[0..n_out), written T x n_out bytes, row-major by step, to out.
struct ScOut {
    const int32_t *bits = nullptr;
    uint8_t *out = nullptr;
    int T = 0, n_out = 0;
    ScSignal sig{};  // once it is there (the run's end only)
};

// All launchers are asynchronous on stream s.  `single` != nullptr selects the
// kernels that take one instance by value; otherwise instances come from `insts`.
void launch_step(hipStream_t s, const ScInstance *single, const ScInstance *insts, const DevWork &w, int k);
// The end of a run of K steps, one launch (plus a zeroing launch when a ring row
// spans several statistics chunks): per-population counts and synaptic events of
// the run's rows, the output spike train of its last out->T steps when out is set
// (one instance only), then the statistics' copies in host memory (signalled by
// `stats`) and the advance of every instance's step counters by K.
void launch_run_end(hipStream_t s, const ScInstance *single, ScInstance *insts, int n_inst, const DevWork &w, int K,
                    const ScOut *out, const ScSignal &stats, unsigned int *run_done = nullptr);
// The batch rows of an instance table, before a batch's first step after other calls.
void launch_batch_rows(hipStream_t s, ScInstance *insts, int n_inst);
// The stimulus descriptors dst[0..n) := src[0..n) (host memory, read by the call).
void launch_set_stims(hipStream_t s, ScStim *dst, const ScStim *src, int n);
// Blocks of a resident run that the current device holds at once, and the run (one
// network, no plasticity rules).  launch_run_end follows with run_done = r.done.
int run_capacity(bool idx16, int *blocks, int *n_cus = nullptr);  // and the device's CUs
void launch_run(hipStream_t s, const ScInstance &I, const DevWork &w, const ScRun &r);
void launch_set_ctl(hipStream_t s, ScCtl *ctl, int64_t n, int64_t m, int row);
void launch_init_params(hipStream_t s, const ScInstance *di, int n_threads, uint64_t seed, uint64_t off);
// Ids [first, first + len) of the fired-neuron list of one ring row and its length.
void launch_fired(hipStream_t s, const uint64_t *row, int n_groups, const ScGroup *groups, int32_t *out, int first,
                  int len, int32_t *count, const ScSignal &sig);
void launch_copy(hipStream_t s, const void *src, void *dst, int64_t n16, int grid);
// Output spike train: T steps from ring row row0 (wrapping at R), one byte per
// (step, output neuron), output neurons at device bits bits[0..n_out).
void launch_out_train(hipStream_t s, const uint64_t *ring, int Wr, int R, int row0, int T, const int32_t *bits,
                      int n_out, uint8_t *out);
void launch_zero_g(hipStream_t s, ScState *st, int n);
// State of n > 0 neurons from reference id r0 on into mapped host memory: potentials,
// conductances and counters, with room for cap (even) neurons each.  `done`: a zeroed
// counter (left zero).
void launch_state(hipStream_t s, const ScInstance &I, int r0, int n, int cap, void *out, unsigned int *done,
                  const ScSignal &sig);
// out[i] = val[vidx[i]] for n > 0 synapses, out in mapped host memory; `done` as above.
void launch_multipliers(hipStream_t s, const float *val, const uint32_t *vidx, int n, float *out, unsigned int *done,
                        const ScSignal &sig);
// The plasticity rules of one network after step k of a run (single instance).
void launch_plastic(hipStream_t s, const ScInstance &I, const DevWork &w, int k);

}  // namespace sc
