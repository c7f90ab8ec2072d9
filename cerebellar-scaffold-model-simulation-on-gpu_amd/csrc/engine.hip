// engine.hip -- device-side engine: HBM layout upload, lowering of the planner's
// work list to kernel descriptors, step runs (direct or hipGraph replays),
// queries and batches of instances.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

#include "kernels.hpp"
#include "recorder.hpp"

namespace sc {

// Bit ranges one task reads (per lane slice, or per incoming projection of a team
// neuron) and the 64-byte segments its gathers touch: the input of the staging
// plan.  lo > hi: the slice / projection reads nothing.
// Events a function creates for its own timing, destroyed on every path out of it.
struct LocalEvents {
    std::vector<hipEvent_t> ev;
    LocalEvents() = default;
    LocalEvents(const LocalEvents &) = delete;
    LocalEvents &operator=(const LocalEvents &) = delete;
    ~LocalEvents()
    {
        for (hipEvent_t x : ev) (void)hipEventDestroy(x);
    }
    int make(hipEvent_t *out)
    {
        *out = nullptr;
        HIP_TRY(hipEventCreate(out));
        ev.push_back(*out);
        return SCAFFOLD_OK;
    }
};

struct TaskWin {
    int n = 0;
    int32_t delay[SC_MAX_IN] = {}, pre[SC_MAX_IN] = {};
    uint32_t lo[SC_MAX_IN] = {}, hi[SC_MAX_IN] = {};
    int64_t segs = 0;
    int64_t qsegs[SC_MAX_IN] = {};  // segments of each slice / projection
    bool partial = false;           // a team in the 16-bit form: its projections can be staged one by one
};

// Optional timing of the step kernels inside the runs: a pair of events recorded
// on the engine's stream around the step kernels of every run piece (direct
// launches, or one replay of a graph that holds the step kernels only, the
// statistics and counter advance of the piece following it as direct launches).
struct KTimer {
    bool on = false;
    int every = 1;                 // time one run in `every` (the runs counted in `seq`)
    int64_t seq = 0;
    std::vector<hipEvent_t> pool;  // pairs
    size_t used = 0;
    std::vector<int> piece_k;      // step launches of each measured piece
    double ms = 0.0;
    int64_t launches = 0;
};

// The captured graphs of an engine or a batch, one per use: a whole run (step
// kernels, then the run's end), a whole run whose end also gathers the output
// train, and the step kernels alone (timed runs).  Each is captured on first use
// and again when the run length or the output train changes.
struct RunGraphs {
    enum { RUN, RUN_OUT, STEPS, N };
    struct Slot {
        hipGraphExec_t exec = nullptr;
        int chunk = 0;
        ScOut out;
    } slot[N];
    void destroy()
    {
        for (Slot &x : slot) {
            if (x.exec) (void)hipGraphExecDestroy(x.exec);
            x.exec = nullptr;
        }
    }
};

// Resident runs of an engine (k_run): what its launches share.
struct RunSync {
    const ScDeps *deps = nullptr;        // per block; nullptr: the network's runs launch a kernel per step
    unsigned long long *tags = nullptr;  // progress of each block, SC_TAG_WORDS apart
    uint32_t *done = nullptr;
    uint32_t *failed_h = nullptr, *failed_hd = nullptr;  // host word a given-up run sets, and its device address
    int max_steps = 0;                   // longest run whose rows the ring holds beside those it reads
    int polls = 0;                       // most polls of one wait
    int cus = 0;                         // compute units of the device
    int64_t launched = 0, given_up = 0;  // runs so far (engine_run_counts)
};

// Mapped host memory that kernels of one engine hand results over in (its calls are
// one after another, so it holds one result at a time).  `ready` is the sequence
// number of the last result that is complete (ScSignal).  The data's size follows the
// network's (16 bytes a neuron, within bounds): pinning costs 1.5 ms a megabyte when
// the network is set up; larger results are handed over in parts.
constexpr size_t kHandLeast = 64 << 10, kHandMost = 1 << 20;
constexpr unsigned long long kNoSignal = ~0ull;
struct HandOff {
    uint32_t run_failed;  // a resident run was given up
    int32_t count;
    unsigned long long ready;
    unsigned long long pad_[6];
};
static_assert(sizeof(HandOff) == 64, "the data starts on a line of its own");

struct Engine {
    hipStream_t stream = nullptr;
    int device = 0;
    RunSync run;
    std::vector<void *> allocs;
    int64_t bytes = 0;
    ScInstance hi{};
    ScInstance *di = nullptr;
    DevWork w;
    // host copies of the lowered work (batches concatenate them)
    std::vector<ScLaneTask> h_lanes;
    std::vector<ScStimTask> h_stims;
    std::vector<ScTeamTask> h_teams;
    std::vector<int> h_team_t;  // team width (wavefronts) of each team task
    std::vector<int> h_team_b;  // its width in a batch
    std::vector<TaskWin> h_lane_win, h_team_win;
    ScStim *stims = nullptr;
    int n_stims = 0;
    int n_pops = 0;
    int32_t *scratch = nullptr;  // the static scratch on this engine's device (no-allocation queries)
    std::vector<int32_t> dev_to_ref;
    int Ndev = 0, total_ref = 0;
    RunGraphs graphs;
    KTimer kt;
    // output spike train: device bits of the OUTPUT neurons, T_out x n_out bytes in
    // mapped pinned memory
    const int32_t *out_bits = nullptr;
    uint8_t *out_h = nullptr;
    uint8_t *out_hd = nullptr;      // the device's address of out_h
    int n_out = 0, T_out = 0;
    size_t out_bytes = 0;  // the train's bytes in out_h, in whole 64-byte lines
    HandOff *hand = nullptr, *hand_d = nullptr;  // behind them, and the device's address of it
    uint8_t *data = nullptr, *data_d = nullptr;  // behind that: hand_bytes of data
    size_t hand_bytes = 0;
    unsigned long long seq = 0;  // of the last signal asked for
    uint64_t moved = 0;   // what has moved the step counters (runs, jumps of the step count), for batches
    bool queued = false;  // work of a call that returned may still be on the stream (new rates, the end of a run)
    // the statistics of the last run are in host memory once this signal is in
    // (kNoSignal: once the stream is idle)
    unsigned long long stats_seq = 0;
    const int32_t *counts_h = nullptr;  // R x n_pops, R, n_pops + 1: the host copies
    const unsigned long long *events_h = nullptr, *totals_h = nullptr;
    // plastic projections: multiplier array and per-synapse index, for read-back
    struct PlasticView {
        int proj;
        const float *val;
        const uint32_t *vidx;  // on the device
        int64_t n;
    };
    std::vector<PlasticView> plastic_views;
};

// Static scratch of scaffold_get_fired_noalloc: word 0 receives the fired count,
// words SC_SCRATCH_IDS .. the ids (256-byte aligned).  One copy per GPU, held
// until the process ends; its device address is looked up once per device with
// hipGetSymbolAddress (in host code the array's name is not a device address).
static __device__ __align__(256) int32_t scratch[SC_SCRATCH_IDS + SC_FIRED_NOALLOC_MAX];
static constexpr int kMaxDevices = 64;
static int32_t *g_scratch[kMaxDevices] = {};
static std::mutex g_scratch_mu;

// The scratch address on the current device (looked up on first use per device).
static int scratch_on_current_device(int32_t **out)
{
    int dev = 0;
    HIP_TRY(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) return fail(SCAFFOLD_ERR_CAPACITY, "device %d beyond the scratch table", dev);
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch[dev]) {
        void *p = nullptr;
        HIP_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        g_scratch[dev] = static_cast<int32_t *>(p);
    }
    *out = g_scratch[dev];
    return SCAFFOLD_OK;
}

template <typename T>
static int dalloc(std::vector<void *> &allocs, int64_t *bytes, T **p, size_t count, bool clear = true)
{
    size_t b = sizeof(T) * (count ? count : 1);
    void *q = nullptr;
    HIP_TRY(hipMalloc(&q, b));
    allocs.push_back(q);
    if (clear) HIP_TRY(hipMemset(q, 0, b));
    if (bytes) *bytes += (int64_t)b;
    *p = static_cast<T *>(q);
    return SCAFFOLD_OK;
}

template <typename T>
static int dupload(std::vector<void *> &allocs, int64_t *bytes, T **p, const std::vector<T> &v)
{
    int rc = dalloc(allocs, bytes, p, v.size(), v.empty());
    if (rc) return rc;
    if (!v.empty()) HIP_TRY(hipMemcpy(*p, v.data(), sizeof(T) * v.size(), hipMemcpyHostToDevice));
    return SCAFFOLD_OK;
}

static int check_device()
{
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n < 1) return fail(SCAFFOLD_ERR_NO_DEVICE, "no HIP device visible");
    hipDeviceProp_t prop;
    HIP_TRY(hipGetDeviceProperties(&prop, 0));
    if (strncmp(prop.gcnArchName, "gfx950", 6) != 0)
        return fail(SCAFFOLD_ERR_NO_DEVICE, "device 0 is %s; this library is built for gfx950", prop.gcnArchName);
    return SCAFFOLD_OK;
}

static int wbytes_of(int wprec) { return wprec == SC_W_F32 ? 4 : wprec == SC_W_BF16 ? 2 : wprec == SC_W_FP8 ? 1 : 0; }

// Block layout of the step kernel: team neurons by team width (widest first, so
// the longest rows start earliest), then lane groups, then stimulus groups, then
// the plasticity rules' window-count groups, 16 wavefronts per block.  `team_t` lists the team width of every team descriptor,
// widest first.
static ScLayout make_layout(const std::vector<int> &team_t, int n_lanes, int n_stims, int n_hist, int lane_per,
                            int stim_per, int *n_blocks)
{
    ScLayout L{};
    L.lane_per = lane_per;
    L.stim_per = stim_per;
    int blocks = 0;
    size_t i = 0;
    for (int c = 0; c < SC_CLASS_LANE; ++c) {
        const int t = SC_MAX_TEAM >> c, per = 1 << c;
        size_t j = i;
        while (j < team_t.size() && team_t[j] == t) ++j;
        L.cls_task0[c] = (int)i;
        L.cls_ntask[c] = (int)(j - i);
        blocks += (L.cls_ntask[c] + per - 1) / per;
        L.cls_end[c] = blocks;
        i = j;
    }
    L.cls_ntask[SC_CLASS_LANE] = n_lanes;
    blocks += (n_lanes + lane_per - 1) / lane_per;
    L.cls_end[SC_CLASS_LANE] = blocks;
    L.cls_ntask[SC_CLASS_STIM] = n_stims;
    blocks += (n_stims + stim_per - 1) / stim_per;
    L.cls_end[SC_CLASS_STIM] = blocks;
    L.cls_ntask[SC_CLASS_HIST] = n_hist;
    blocks += (n_hist + SC_BLOCK / SC_WAVE - 1) / (SC_BLOCK / SC_WAVE);
    L.cls_end[SC_CLASS_HIST] = blocks;
    *n_blocks = blocks;
    return L;
}

// Staging plan: for every block of lane groups or team neurons, the windows of
// ring-row words its tasks read, one per (instance, delay, presynaptic
// population) spanning the union of their bit ranges.  A block stages all its
// windows when they fit the LDS budget and hold at most `ratio` words per
// 64-byte segment its gathers would touch (ratio 8: the copy touches at most
// half the segments the gathers would, words / 16 <= segments / 2).  When they
// do not, a block of team neurons in the 16-bit form (whose chunks name their
// projection) stages the windows that pay most -- most segments per word, each
// within the ratio -- while they fit, and its other projections read the ring
// in memory (their ScTeamIn.lds is SC_LDS_GLOBAL).  The slices and projections
// of a staged window carry the LDS word that stands for word 0 of its ring row.
static std::vector<ScStage> plan_stages(const ScLayout &L, int n_blocks, std::vector<ScLaneTask> &lanes,
                                        const std::vector<TaskWin> &lane_win, std::vector<ScTeamTask> &teams,
                                        const std::vector<TaskWin> &team_win, int ratio, int *n_staged)
{
    constexpr int MAXK = 4 * SC_MAX_WIN;  // candidate windows per block
    std::vector<ScStage> st((size_t)n_blocks);
    *n_staged = 0;
    for (int c = 0; c <= SC_CLASS_LANE; ++c) {
        const bool lane = c == SC_CLASS_LANE;
        const int b0 = c ? L.cls_end[c - 1] : 0;
        for (int b = b0; b < L.cls_end[c]; ++b) {
            const int bi = b - b0, per = lane ? L.lane_per : 1 << c;
            const int first = (lane ? 0 : L.cls_task0[c]) + bi * per;
            const int count = std::min(per, L.cls_ntask[c] - bi * per);
            ScWin wins[MAXK];
            int32_t pre_of[MAXK];
            uint32_t lo_of[MAXK], hi_of[MAXK];
            int64_t seg_of[MAXK];
            int nw = 0;
            bool ok = true, partial = !lane;
            int64_t segs = 0;
            auto key_of = [&](int inst, int delay, int pre) {
                for (int i = 0; i < nw; ++i)
                    if (wins[i].inst == inst && wins[i].delay == delay && pre_of[i] == pre) return i;
                return -1;
            };
            for (int i = 0; i < count && ok; ++i) {
                const TaskWin &W = lane ? lane_win[first + i] : team_win[first + i];
                const int inst = lane ? lanes[first + i].inst : teams[first + i].inst;
                segs += W.segs;
                partial = partial && W.partial;
                for (int r = 0; r < W.n && ok; ++r) {
                    if (W.lo[r] > W.hi[r]) continue;
                    int kx = key_of(inst, W.delay[r], W.pre[r]);
                    if (kx < 0) {
                        if (nw == MAXK) { ok = false; break; }
                        kx = nw++;
                        wins[kx] = ScWin{inst, W.delay[r], 0, 0, 0, 0};
                        pre_of[kx] = W.pre[r];
                        lo_of[kx] = W.lo[r];
                        hi_of[kx] = W.hi[r];
                        seg_of[kx] = 0;
                    }
                    lo_of[kx] = std::min(lo_of[kx], W.lo[r]);
                    hi_of[kx] = std::max(hi_of[kx], W.hi[r]);
                    seg_of[kx] += W.qsegs[r];
                }
            }
            if (!ok || nw == 0) continue;
            int64_t total = 4;  // LDS words 0..3: zero (padding entries read word 0)
            for (int i = 0; i < nw; ++i) {  // whole 16-byte vectors: rows are 16-byte aligned
                wins[i].w0 = (int32_t)((lo_of[i] >> 5) & ~3u);
                wins[i].nw = (int32_t)((((hi_of[i] >> 5) + 4) & ~3u) - (uint32_t)wins[i].w0);
                total += wins[i].nw;
            }
            bool chosen[MAXK] = {};
            int n_chosen = 0;
            if (nw <= SC_MAX_WIN && total <= SC_WIN_WORDS && total <= (int64_t)ratio * segs) {
                for (int i = 0; i < nw; ++i) chosen[i] = true;
                n_chosen = nw;
            } else if (partial) {
                int order[MAXK];
                for (int i = 0; i < nw; ++i) order[i] = i;
                std::sort(order, order + nw, [&](int x, int y) {  // most segments per word first
                    return seg_of[x] * wins[y].nw > seg_of[y] * wins[x].nw;
                });
                int64_t words = 4;
                for (int k = 0; k < nw && n_chosen < SC_MAX_WIN; ++k) {
                    const int i = order[k];
                    if (wins[i].nw > (int64_t)ratio * seg_of[i] || words + wins[i].nw > SC_WIN_WORDS) continue;
                    chosen[i] = true;
                    words += wins[i].nw;
                    ++n_chosen;
                }
            }
            if (n_chosen == 0) continue;
            ScStage &S = st[(size_t)b];
            int64_t off = 4;
            for (int i = 0; i < nw; ++i) {
                if (!chosen[i]) continue;
                wins[i].off = (int32_t)off;
                off += wins[i].nw;
                S.w[S.n++] = wins[i];
            }
            for (int i = 0; i < count; ++i) {
                const TaskWin &W = lane ? lane_win[first + i] : team_win[first + i];
                const int inst = lane ? lanes[first + i].inst : teams[first + i].inst;
                for (int r = 0; r < W.n; ++r) {
                    const int kx = W.lo[r] > W.hi[r] ? -1 : key_of(inst, W.delay[r], W.pre[r]);
                    const int32_t lds = kx < 0 ? 0 : chosen[kx] ? wins[kx].off - wins[kx].w0 : SC_LDS_GLOBAL;
                    if (lane) lanes[first + i].sl[r].lds = lds;
                    else teams[first + i].in[r].lds = lds;
                }
            }
            ++*n_staged;
        }
    }
    return st;
}

// The wait tables of a network's resident runs (one per block): which blocks own the
// presynaptic neurons of each projection a block reads, from the bit ranges of its
// tasks (neurons of a population are assigned to tasks, and tasks to blocks, in
// ascending order, so a bit range belongs to a range of blocks).  Entries past the
// table's size widen the last one of their kind: waiting for more blocks, or for a
// later step of them, is always allowed.
static std::vector<ScDeps> plan_deps(const ScLayout &L, int n_blocks, int Ndev, const std::vector<ScLaneTask> &lanes,
                                     const std::vector<TaskWin> &lane_win, const std::vector<ScTeamTask> &teams,
                                     const std::vector<TaskWin> &team_win, const std::vector<ScStimTask> &stims,
                                     const std::vector<ScStage> &stages)
{
    std::vector<int32_t> owner((size_t)Ndev, -1);  // block of each device neuron
    struct Part { int first, count; };
    auto part_of = [&](int c, int b) {
        const int bi = b - (c ? L.cls_end[c - 1] : 0);
        const int per = c == SC_CLASS_LANE ? L.lane_per : c == SC_CLASS_STIM ? L.stim_per : 1 << c;
        return Part{(c < SC_CLASS_LANE ? L.cls_task0[c] : 0) + bi * per, std::min(per, L.cls_ntask[c] - bi * per)};
    };
    for (int c = 0; c <= SC_CLASS_STIM; ++c)
        for (int b = c ? L.cls_end[c - 1] : 0; b < L.cls_end[c]; ++b) {
            const Part p = part_of(c, b);
            for (int i = p.first; i < p.first + p.count; ++i) {
                if (c < SC_CLASS_LANE) { owner[teams[i].group * SC_WAVE + teams[i].bit] = b; continue; }
                const int g = c == SC_CLASS_LANE ? lanes[i].group : stims[i].group;
                const int nv = c == SC_CLASS_LANE ? lanes[i].nvalid : stims[i].nvalid;
                for (int l = 0; l < nv; ++l) owner[g * SC_WAVE + l] = b;
            }
        }
    std::vector<ScDeps> deps((size_t)n_blocks);
    for (int c = 0; c <= SC_CLASS_LANE; ++c)
        for (int b = c ? L.cls_end[c - 1] : 0; b < L.cls_end[c]; ++b) {
            const bool lane = c == SC_CLASS_LANE;
            const Part p = part_of(c, b);
            std::vector<ScDep> kind[2];  // longer delays, one-step delays of team neurons
            if (!lane) {
                int lo = n_blocks, hi = -1;
                for (int i = p.first; i < p.first + p.count; ++i) {
                    const int o = owner[teams[i].group * SC_WAVE];
                    lo = std::min(lo, o);
                    hi = std::max(hi, o);
                }
                kind[0].push_back(ScDep{lo, hi - lo + 1, SC_DEP_ONCE, 0, 0, 0, 0, 0});
            }
            for (int i = p.first; i < p.first + p.count; ++i) {
                const TaskWin &W = lane ? lane_win[i] : team_win[i];
                for (int r = 0; r < W.n; ++r) {
                    if (W.lo[r] > W.hi[r]) continue;
                    const int b0 = owner[W.lo[r]], b1 = owner[W.hi[r]];
                    std::vector<ScDep> &v = kind[!lane && W.delay[r] < 2];
                    bool in = false;
                    for (ScDep &x : v) {
                        // ranges of one delay that overlap or touch are one entry
                        if (x.delay != W.delay[r] || b0 > x.b0 + x.cnt || b1 + 1 < x.b0) continue;
                        const int e = std::max(x.b0 + x.cnt, b1 + 1);
                        x.b0 = std::min(x.b0, b0);
                        x.cnt = e - x.b0;
                        in = true;
                        break;
                    }
                    if (!in) v.push_back(ScDep{b0, b1 - b0 + 1, W.delay[r], 0, 0, 0, 0, 0});
                }
            }
            ScDeps &D = deps[(size_t)b];
            for (int k = 0; k < 2; ++k) {
                const int most = SC_MAX_DEP / 2;
                for (size_t i = 0; i < kind[k].size(); ++i) {
                    const ScDep &x = kind[k][i];
                    if ((int)i < most) { D.e[D.n++] = x; continue; }
                    ScDep &y = D.e[D.n - 1];
                    const int e = std::max(y.b0 + y.cnt, x.b0 + x.cnt);
                    y.b0 = std::min(y.b0, x.b0);
                    y.cnt = e - y.b0;
                    y.delay = std::min(y.delay, x.delay);
                }
                if (k == 0) D.n_early = D.n;
            }
            // mail: every one-step entry names team blocks of one width that hold whole
            // ranges of one population's neurons, and the block's one-step windows are
            // staged, one per entry
            D.mail = !lane && D.n > D.n_early && kind[1].size() <= SC_MAX_DEP / 2;
            int n_late_win = 0;
            for (int w = 0; w < (stages.empty() ? 0 : stages[b].n); ++w) n_late_win += stages[b].w[w].delay < 2;
            if (n_late_win != D.n - D.n_early) D.mail = 0;
            std::vector<char> taken(SC_MAX_WIN, 0);
            for (int i = D.n_early; i < D.n && D.mail; ++i) {
                ScDep &x = D.e[i];
                int cls = -1;
                for (int j = 0; j < x.cnt && D.mail; ++j) {
                    int cj = 0;
                    while (x.b0 + j >= L.cls_end[cj]) ++cj;
                    if (j == 0) cls = cj;
                    D.mail = cj == cls && cj < SC_CLASS_LANE;
                    if (!D.mail) break;
                    const Part q = part_of(cj, x.b0 + j);
                    for (int n = q.first; n < q.first + q.count && D.mail; ++n) {
                        const int bit = teams[n].group * SC_WAVE + teams[n].bit;
                        if (j == 0 && n == q.first) {
                            x.bit0 = bit;
                            x.per = 1 << cj;
                            D.mail = x.bit0 % x.per == 0;
                        }
                        D.mail = D.mail && bit == x.bit0 + j * x.per + (n - q.first);
                    }
                }
                if (!D.mail) break;
                D.mail = 0;
                const int lo = x.bit0 >> 5, hi = (x.bit0 + x.cnt * x.per - 1) >> 5;
                for (int w = 0; w < stages[b].n; ++w) {
                    const ScWin &win = stages[b].w[w];
                    if (win.delay >= 2 || taken[w] || win.w0 + win.nw <= lo || win.w0 > hi) continue;
                    taken[w] = 1;
                    D.mail = 1;
                    x.w0 = win.w0;
                    x.w1 = win.w0 + win.nw;
                    x.lds = win.off - win.w0;
                    break;
                }
            }
            int n_mail = 0;
            for (int i = D.n_early; i < D.n; ++i) n_mail += D.e[i].cnt;
            if (n_mail > SC_MAIL_MOST) D.mail = 0;
            // every projection of the block's teams with a one-step delay is staged
            for (int i = p.first; i < p.first + p.count && D.mail; ++i)
                for (int r = 0; r < team_win[i].n; ++r)
                    if (team_win[i].delay[r] < 2 && teams[i].in[r].lds == SC_LDS_GLOBAL) D.mail = 0;
        }
    return deps;
}

static int upload_work(std::vector<void *> &allocs, int64_t *bytes, DevWork &w, const std::vector<int> &team_t,
                       std::vector<ScLaneTask> lanes, const std::vector<ScStimTask> &stims,
                       std::vector<ScTeamTask> teams, const std::vector<TaskWin> &lane_win,
                       const std::vector<TaskWin> &team_win, bool stage, int ratio, int n_hist,
                       int most_blocks, int n_inst)
{
    for (size_t i = 1; i < team_t.size(); ++i)
        if (team_t[i] > team_t[i - 1]) return fail(SCAFFOLD_ERR_STATE, "team descriptors not ordered by width");
    if (lane_win.size() != lanes.size() || team_win.size() != teams.size())
        return fail(SCAFFOLD_ERR_STATE, "staging ranges do not match the descriptors");
    int rc;
    ScLaneTask *l;
    ScStimTask *s;
    ScTeamTask *t;
    w.layout = make_layout(team_t, (int)lanes.size(), (int)stims.size(), n_hist, SC_LANE_PER_BLOCK, SC_STIM_PER_BLOCK,
                           &w.n_blocks);
    // a network that leaves CUs idle is cut into smaller blocks of lane and stimulus
    // groups (the neuron update and the Philox draws keep the vector units of their
    // CU busy), as small as still fit the chip at once
    for (int per = 4; per < SC_LANE_PER_BLOCK && w.n_blocks < most_blocks; per *= 2) {
        int n = 0;
        const ScLayout l = make_layout(team_t, (int)lanes.size(), (int)stims.size(), n_hist, per, per, &n);
        if (n > most_blocks) continue;
        w.layout = l;
        w.n_blocks = n;
        break;
    }
    int n_staged = 0;
    std::vector<ScStage> st;
    if (stage) st = plan_stages(w.layout, w.n_blocks, lanes, lane_win, teams, team_win, ratio, &n_staged);
    w.stages = nullptr;
    w.h_stages = st;
    w.n_staged = n_staged;
    if (n_staged > 0) {
        ScStage *ds;
        if ((rc = dupload(allocs, bytes, &ds, st))) return rc;
        w.stages = ds;
    }
    if ((rc = dupload(allocs, bytes, &l, lanes))) return rc;
    if ((rc = dupload(allocs, bytes, &s, stims))) return rc;
    if ((rc = dupload(allocs, bytes, &t, teams))) return rc;
    w.h_teams = teams;  // with the staging plan's LDS words
    w.lanes = l;
    w.stims = s;
    w.teams = t;
    if ((rc = dalloc(allocs, bytes, &w.end_done, (size_t)2 + n_inst))) return rc;  // zeroed
    w.idx16 = false;
    for (const ScLaneTask &x : lanes) w.idx16 = w.idx16 || x.idx16;
    for (const ScTeamTask &x : teams) w.idx16 = w.idx16 || x.hdr;
    return SCAFFOLD_OK;
}

// Sets up resident runs where the network allows them: the option is on, no
// plasticity rule (its update kernel runs between steps), a grid that the device
// holds at once, and a ring with room for at least SC_RUN_MIN new rows beside those
// the steps read.
static int engine_plan_run(Engine *e, const Plan &P)
{
    if (!P.resident || !e->w.plastic.empty() || e->w.n_blocks <= 0) return SCAFFOLD_OK;
    if ((int64_t)P.Wr * P.R >= (int64_t)1 << 30) return SCAFFOLD_OK;  // ring words are counted in 32 bits
    e->run.max_steps = P.R - P.max_delay - 2;
    if (e->run.max_steps < SC_RUN_MIN) return SCAFFOLD_OK;
    int rc, most = 0;
    if ((rc = run_capacity(e->w.idx16, &most, &e->run.cus))) return rc;
    if (e->w.n_blocks > most) return SCAFFOLD_OK;
    e->run.failed_h = &e->hand->run_failed;
    e->run.failed_hd = &e->hand_d->run_failed;
    // (the count of finished blocks has a line of its own after the blocks' lines)
    if ((rc = dalloc(e->allocs, &e->bytes, &e->run.tags, (size_t)(e->w.n_blocks + 1) * SC_TAG_WORDS))) return rc;  // zeroed
    e->run.done = reinterpret_cast<uint32_t *>(e->run.tags + (size_t)e->w.n_blocks * SC_TAG_WORDS);
    ScDeps *d;
    if ((rc = dupload(e->allocs, &e->bytes, &d,
                      plan_deps(e->w.layout, e->w.n_blocks, e->Ndev, e->h_lanes, e->h_lane_win, e->w.h_teams,
                                e->h_team_win, e->h_stims, e->w.h_stages))))
        return rc;
    e->run.deps = d;
    e->run.polls = P.run_polls;
    return SCAFFOLD_OK;
}

int engine_create(Engine **out, Plan &P)
{
    int rc = check_device();
    if (rc) return rc;
    Engine *e = new Engine();
    *out = nullptr;
    auto bail = [&](int code) { engine_destroy(e); return code; };
    auto &A = e->allocs;
    int64_t *B = &e->bytes;
    if (hipGetDevice(&e->device) != hipSuccess || e->device < 0 || e->device >= kMaxDevices)
        return bail(fail(SCAFFOLD_ERR_CAPACITY, "device %d beyond the table of calls", e->device));
    if (hipStreamCreateWithFlags(&e->stream, hipStreamNonBlocking) != hipSuccess)
        return bail(fail(SCAFFOLD_ERR_HIP, "hipStreamCreate failed"));
    ScInstance &I = e->hi;
    I.R = P.R;
    I.Wr = P.Wr;
    I.n_groups = P.n_groups;
    I.n_pops = (int)P.pops.size();
    I.n_stims = (int)P.stims.size();
    I.Ndev = P.Ndev;
    e->n_pops = I.n_pops;
    e->Ndev = P.Ndev;
    e->total_ref = P.total_ref;
    e->dev_to_ref = P.dev_to_ref;
    if ((rc = dalloc(A, B, &I.st, P.Ndev))) return bail(rc);
    // 16 bytes of slack: a staged window's last 16-byte load may run past the last row
    if ((rc = dalloc(A, B, &I.ring, (size_t)P.R * P.Wr + 2))) return bail(rc);
    if ((rc = dalloc(A, B, &I.counts, (size_t)P.R * I.n_pops))) return bail(rc);
    if ((rc = dalloc(A, B, &I.events, (size_t)P.R))) return bail(rc);
    if ((rc = dalloc(A, B, &I.totals, (size_t)I.n_pops + 1))) return bail(rc);
    ScGroup *groups;
    if ((rc = dupload(A, B, &groups, P.groups))) return bail(rc);
    I.groups = groups;
    ScPop *pops;
    if ((rc = dupload(A, B, &pops, P.pops))) return bail(rc);
    I.pops = pops;
    if ((rc = dupload(A, B, &e->stims, P.stims))) return bail(rc);
    I.stims = e->stims;
    e->n_stims = (int)P.stims.size();
    int32_t *ss, *se;
    if ((rc = dupload(A, B, &ss, P.stim_s))) return bail(rc);
    if ((rc = dupload(A, B, &se, P.stim_e))) return bail(rc);
    I.stim_s = ss;
    I.stim_e = se;
    uint32_t *od;
    if ((rc = dupload(A, B, &od, P.outdeg))) return bail(rc);
    I.outdeg = od;
    ScCtl *ctl;
    if ((rc = dalloc(A, B, &ctl, 1))) return bail(rc);
    I.ctl = ctl;

    // synapse streams: sliced-ELL slices of lane-mode projections
    std::vector<const uint8_t *> pcol(P.projs.size(), nullptr);  // 32-bit words or 16-bit offsets
    std::vector<const uint32_t *> phdr(P.projs.size(), nullptr);
    std::vector<const uint8_t *> pval(P.projs.size(), nullptr);
    for (size_t pi = 0; pi < P.projs.size(); ++pi) {
        if (P.projs[pi].mode != SC_MODE_LANE) continue;
        HostProjArrays &H = P.parr[pi];
        if (H.idx16) {
            uint16_t *c16;
            uint32_t *h;
            if ((rc = dupload(A, B, &c16, H.col16))) return bail(rc);
            if ((rc = dupload(A, B, &h, H.hdr))) return bail(rc);
            pcol[pi] = reinterpret_cast<const uint8_t *>(c16);
            phdr[pi] = h;
        } else {
            uint32_t *col;
            if ((rc = dupload(A, B, &col, H.col))) return bail(rc);
            pcol[pi] = reinterpret_cast<const uint8_t *>(col);
        }
        if (!H.val.empty()) {
            uint8_t *val;
            if ((rc = dupload(A, B, &val, H.val))) return bail(rc);
            pval[pi] = val;
        }
        std::vector<uint32_t>().swap(H.col);  // now on the device only
        std::vector<uint16_t>().swap(H.col16);
        std::vector<uint32_t>().swap(H.hdr);
        std::vector<uint8_t>().swap(H.val);
    }
    // merged rows of team-mode populations
    std::vector<const uint8_t *> tcol(P.teams.size(), nullptr);
    std::vector<const uint32_t *> thdr(P.teams.size(), nullptr);
    std::vector<const uint8_t *> tval(P.teams.size(), nullptr);
    std::vector<const uint32_t *> tgrp(P.teams.size(), nullptr);
    for (size_t ti = 0; ti < P.teams.size(); ++ti) {
        TeamPop &T = P.teams[ti];
        if (!T.grp.empty()) {
            uint32_t *g;
            if ((rc = dupload(A, B, &g, T.grp))) return bail(rc);
            tgrp[ti] = g;
        }
        if (T.idx16) {
            uint16_t *c16;
            uint32_t *h;
            if ((rc = dupload(A, B, &c16, T.col16))) return bail(rc);
            if ((rc = dupload(A, B, &h, T.hdr))) return bail(rc);
            tcol[ti] = reinterpret_cast<const uint8_t *>(c16);
            thdr[ti] = h;
        } else {
            uint32_t *col;
            if ((rc = dupload(A, B, &col, T.col))) return bail(rc);
            tcol[ti] = reinterpret_cast<const uint8_t *>(col);
        }
        if (!T.val.empty()) {
            uint8_t *val;
            if ((rc = dupload(A, B, &val, T.val))) return bail(rc);
            tval[ti] = val;
        }
        std::vector<uint32_t>().swap(T.col);
        std::vector<uint16_t>().swap(T.col16);
        std::vector<uint32_t>().swap(T.hdr);
        std::vector<uint8_t>().swap(T.val);
        std::vector<uint32_t>().swap(T.grp);
    }

    // lower the planner's work list to descriptors with absolute pointers
    for (const ScTask &t : P.tasks) {
        if (t.kind == SC_TASK_ROW) {
            const int pop = t.proj, j = t.post;
            const TeamPop &T = P.teams[P.team_of[pop]];
            const ScPop &pp = P.pops[pop];
            ScTeamTask d{};
            const int ti = P.team_of[pop];
            // 32-bit form: row_ptr counts entries; 16-bit form: 8-entry chunks (16 bytes
            // of offsets, one header word and 8 multipliers each)
            const int64_t e0 = T.idx16 ? T.row_ptr[j] * 8 : T.row_ptr[j];
            d.col = tcol[ti] + e0 * (T.idx16 ? 2 : 4);
            d.hdr = thdr[ti] ? thdr[ti] + T.row_ptr[j] : nullptr;
            d.val = tval[ti] ? tval[ti] + e0 * wbytes_of(T.wprec) : nullptr;
            d.group = t.group;
            d.bit = j % SC_WAVE;
            d.pop = pop;
            d.n_in = pp.n_in;
            d.wprec = T.wprec;
            // 16-bit form: the padded group length; 32-bit: the synapse count
            d.len = T.idx16 ? (int)(T.row_ptr[j + 1] - T.row_ptr[j])  // chunks
                            : 0;
            for (int q = 0; q < pp.n_in && !T.idx16; ++q) d.len = std::max(d.len, T.seg_end[(size_t)j * pp.n_in + q]);
            d.len_e = T.len_e[j];
            d.n_grp_e = T.grp_e[j];
            d.n_grp = (int)(T.grp_ptr[j + 1] - T.grp_ptr[j]);
            d.grp = d.n_grp ? tgrp[ti] + 4 * T.grp_ptr[j] : nullptr;
            TaskWin tw;
            tw.n = pp.n_in;
            tw.segs = T.row_seg[j];
            tw.partial = T.idx16;
            for (int q = 0; q < pp.n_in; ++q) {
                const ScProj &sp = P.projs[pp.in_proj[q]];
                tw.delay[q] = sp.delay;
                tw.pre[q] = sp.pre_pop;
                tw.qsegs[q] = T.q_seg[(size_t)j * pp.n_in + q];
                tw.lo[q] = T.q_lo[(size_t)j * pp.n_in + q];
                tw.hi[q] = T.q_hi[(size_t)j * pp.n_in + q];
                d.in[q].delay = sp.delay;
                d.in[q].exc = sp.exc;
                d.in[q].W = sp.W;
                d.in[q].scale = sp.scale * sp.sum_scale;  // exact: scale is a power of two
            }
            e->h_teams.push_back(d);
            e->h_team_t.push_back(T.team_waves);
            e->h_team_b.push_back(T.batch_waves);
            e->h_team_win.push_back(tw);
        } else if (t.kind == SC_TASK_LANE) {
            const ScGroup &G = P.groups[t.group];
            const ScPop &pp = P.pops[G.pop];
            const int gi = t.group - pp.group_base;
            ScLaneTask l{};
            TaskWin tw;
            l.wp = SC_W_UNIT;
            l.group = t.group;
            l.pop = G.pop;
            l.nvalid = G.nvalid;
            for (int q = 0; q < pp.n_in; ++q) {
                const int pi = pp.in_proj[q];
                const ScProj &sp = P.projs[pi];
                const HostProjArrays &H = P.parr[pi];
                tw.delay[l.n_sl] = sp.delay;
                tw.pre[l.n_sl] = sp.pre_pop;
                tw.lo[l.n_sl] = H.sl_lo[gi];
                tw.hi[l.n_sl] = H.sl_hi[gi];
                tw.segs += H.sl_seg[gi];
                tw.qsegs[l.n_sl] = H.sl_seg[gi];
                tw.n = l.n_sl + 1;
                ScSlice &s = l.sl[l.n_sl++];
                const int64_t off = H.sell_off[gi];
                s.col = H.idx16 ? pcol[pi] + H.sell_off16[gi] * 4 : pcol[pi] + off * 4;
                s.hdr = H.idx16 ? phdr[pi] + H.sell_off16[gi] / SC_WAVE : nullptr;
                l.idx16 = H.idx16 ? 1 : 0;
                s.val = pval[pi] ? pval[pi] + off * wbytes_of(sp.wprec) : nullptr;
                s.width = H.sell_w[gi];
                s.delay = sp.delay;
                s.wprec = sp.wprec;
                s.exc = sp.exc;
                s.W = sp.W;
                s.scale = sp.scale * sp.sum_scale;  // exact: scale is a power of two
                if (s.val) l.wp = sp.wprec;
            }
            e->h_lanes.push_back(l);
            e->h_lane_win.push_back(tw);
        } else {
            const ScGroup &G = P.groups[t.group];
            ScStimTask s{};
            s.group = t.group;
            s.pop = G.pop;
            s.nvalid = G.nvalid;
            e->h_stims.push_back(s);
        }
    }
    int n_hist = 0;  // window-count groups of the plasticity rules
    for (const PlasticPlan &X : P.plastic) {
        const int groups = (P.pops[P.projs[X.rule.target].pre_pop].num + SC_WAVE - 1) / SC_WAVE;
        n_hist += (groups + SC_HIST_GROUPS - 1) / SC_HIST_GROUPS;  // wavefronts of the window-count class
    }
    int most_blocks = 0;
    if ((rc = run_capacity(P.index_bits == 16, &most_blocks))) return bail(rc);
    if ((rc = upload_work(A, B, e->w, e->h_team_t, e->h_lanes, e->h_stims, e->h_teams, e->h_lane_win, e->h_team_win,
                          P.stage != 0, P.stage_ratio, n_hist, most_blocks, 0)))
        return bail(rc);
    // plasticity rules: per-synapse arrays; the multipliers they update are the
    // f32 arrays of the target's lane slices or merged rows
    e->w.plastic.clear();
    for (const PlasticPlan &X : P.plastic) {
        ScPlastic d{};
        uint32_t *pre, *vidx, *cb;
        int32_t *ct;
        if ((rc = dupload(A, B, &pre, X.pre))) return bail(rc);
        if ((rc = dupload(A, B, &vidx, X.vidx))) return bail(rc);
        if ((rc = dupload(A, B, &cb, X.ch_begin))) return bail(rc);
        if ((rc = dupload(A, B, &ct, X.ch_trig))) return bail(rc);
        const uint8_t *v = X.team ? tval[X.owner] : pval[X.owner];
        if (!v && !X.pre.empty()) return bail(fail(SCAFFOLD_ERR_STATE, "plastic projection without multipliers"));
        const ScPop &pp = P.pops[P.projs[X.rule.target].pre_pop];
        uint8_t *hist;
        if ((rc = dalloc(A, B, &hist, (size_t)(pp.num + SC_WAVE - 1) / SC_WAVE * SC_WAVE))) return bail(rc);
        d.hist = hist;
        d.pre_group0 = pp.group_base;
        d.pre_groups = (pp.num + SC_WAVE - 1) / SC_WAVE;
        d.pre = pre;
        d.vidx = vidx;
        d.ch_begin = cb;
        d.ch_trig = ct;
        d.val = const_cast<float *>(reinterpret_cast<const float *>(v));
        d.packed = X.packed ? 1 : 0;
        d.n_syn = X.packed ? (uint32_t)X.pre.size() : 0u;
        d.n_chunks = (int32_t)(X.packed ? (X.pre.size() + SC_WAVE - 1) / SC_WAVE : X.ch_trig.size());
        d.skip_quiet = X.skip_quiet ? 1 : 0;
        d.rule = X.rule.rule;
        d.delay = X.delay;
        d.t_delay = X.t_delay;
        d.window = X.rule.window;
        d.present = (int32_t)(X.rule.present & 15u);
        d.grid_exp = X.grid_exp;
        for (int c = 0; c < 4; ++c) {
            d.coef[c] = X.rule.coef[c];
            d.ac[c] = X.rule.ac[c];
            d.aa[c] = X.rule.aa[c];
            d.ab[c] = X.rule.ab[c];
        }
        d.affine = (int32_t)(X.rule.affine & 15u);
        e->w.plastic.push_back(d);
        e->plastic_views.push_back(Engine::PlasticView{X.rule.target, d.val, vidx, (int64_t)X.vidx.size()});
    }
    if (!e->w.plastic.empty()) {
        ScPlastic *dp;
        if ((rc = dupload(A, B, &dp, e->w.plastic))) return bail(rc);
        e->w.d_plastic = dp;
    }
    e->w.max_groups = P.n_groups;
    e->w.nontemporal = P.nontemporal;
    if ((rc = scratch_on_current_device(&e->scratch))) return bail(rc);
    // output spike train (T_out steps x n_out neurons)
    e->n_out = P.n_output;
    e->T_out = std::max(1, P.T_out);
    {
        int32_t *ob;
        if ((rc = dupload(A, B, &ob, P.out_bits))) return bail(rc);
        e->out_bits = ob;
        // the gather writes the train straight into mapped pinned memory (no separate
        // device-to-host copy); the hand-off buffer of the queries lies behind it
        e->out_bytes = ((size_t)e->T_out * (size_t)std::max(1, e->n_out) + 63) / 64 * 64;
        void *dp = nullptr;
        e->hand_bytes = std::min(kHandMost, std::max(kHandLeast, (size_t)P.Ndev * 16));  // whole lines
        const size_t stat_bytes = ((size_t)P.R + I.n_pops + 1) * 8 + (size_t)P.R * I.n_pops * 4;
        if (hipHostMalloc(reinterpret_cast<void **>(&e->out_h),
                          e->out_bytes + sizeof(HandOff) + e->hand_bytes + stat_bytes,
                          hipHostMallocMapped) != hipSuccess)
            return bail(fail(SCAFFOLD_ERR_HIP, "hipHostMalloc of the hand-off memory failed"));
        if (hipHostGetDevicePointer(&dp, e->out_h, 0) != hipSuccess || !dp)
            return bail(fail(SCAFFOLD_ERR_HIP, "no device address for the hand-off memory"));
        e->out_hd = static_cast<uint8_t *>(dp);
        memset(e->out_h, 0, e->out_bytes + sizeof(HandOff));
        e->hand = reinterpret_cast<HandOff *>(e->out_h + e->out_bytes);
        e->hand_d = reinterpret_cast<HandOff *>(e->out_hd + e->out_bytes);
        e->data = reinterpret_cast<uint8_t *>(e->hand + 1);
        e->data_d = reinterpret_cast<uint8_t *>(e->hand_d + 1);
        // the statistics' copies close it
        const size_t n64 = (size_t)P.R + I.n_pops + 1;
        auto *st = reinterpret_cast<unsigned long long *>(e->data + e->hand_bytes);
        memset(st, 0, stat_bytes);
        e->events_h = st;
        e->totals_h = st + P.R;
        e->counts_h = reinterpret_cast<const int32_t *>(st + n64);
        st = reinterpret_cast<unsigned long long *>(e->data_d + e->hand_bytes);
        e->w.host = ScHostStats{reinterpret_cast<int32_t *>(st + n64), st, st + P.R};
    }
    if ((rc = engine_plan_run(e, P))) return bail(rc);
    std::vector<ScInstance> one{I};
    if ((rc = dupload(A, B, &e->di, one))) return bail(rc);
    *out = e;
    return SCAFFOLD_OK;
}

// Resident runs that a call of n steps is cut into, of about `chunk` steps each and
// equally long (0: none, a launch per step).  A remainder too short for a call of its own
// goes to the other runs where the ring has room, so 26 steps at a chunk of 25 are one
// run.  A run below SC_RUN_LEAST steps is slower than its steps one by one.
static int resident_runs(int n, int chunk, int max_steps, int n_blocks)
{
    int runs = (n + chunk - 1) / chunk;
    if (runs > 1 && n - (runs - 1) * chunk < SC_RUN_MIN && (n + runs - 2) / (runs - 1) <= max_steps) --runs;
    return n >= SC_RUN_MIN && n / runs >= SC_RUN_LEAST(n_blocks) ? runs : 0;
}

// The calls under way on a device and what they hold of it.  Resident runs of two streams
// side by side could each hold CUs the other's blocks need, so a call's runs are resident
// only if its blocks fit beside those of every other call under way; a call returns when
// its resident runs are done, so those that run together always fit together.  A call
// that launches step by step waits for nobody; its kernels, two blocks to a CU, count
// half.  Blocks are counted in whole 32nds: the hardware deals them out to 8 XCDs and 4
// shader engines each in turn.  Two networks on two threads, us a window of 25 steps: 9.9k
// cells (96 blocks counted) 98 by single steps, 145 with runs one after another, 72 side
// by side; 24k cells (224) 104, 146, 96.  96.7k cells beside 24k ones whose runs hold
// their CUs: 29k steps a second, 82k this way.
static std::mutex g_share_mu;
static int g_share[kMaxDevices] = {};

struct ChipShare {
    int dev, held = 0;
    int n_runs = 0;  // resident runs of the call (0: a launch per step)
    // A call whose kernels have n_blocks blocks and whose steps would be `runs` resident
    // runs (0: cannot be) on a device of `cus` CUs.
    ChipShare(int device, int n_blocks, int runs, int cus) : dev(device)
    {
        const auto counted = [](int n) { return (n + 31) / 32 * 32; };
        std::lock_guard<std::mutex> lock(g_share_mu);
        // (alone, the grid fits: engine_plan_run)
        if (g_share[dev] == 0 || g_share[dev] + counted(n_blocks) <= cus) n_runs = runs;
        held = n_runs ? counted(n_blocks) : counted((n_blocks + 1) / 2);
        g_share[dev] += held;
    }
    ~ChipShare()
    {
        std::lock_guard<std::mutex> lock(g_share_mu);
        g_share[dev] -= held;
    }
    ChipShare(const ChipShare &) = delete;
    ChipShare &operator=(const ChipShare &) = delete;
};

// The share of a call of n_steps steps on engine e; `resident`: its runs may be.
static ChipShare share_for(const Engine *e, int n_steps, int chunk, bool resident)
{
    const int most = e->run.max_steps;
    return ChipShare(e->device, e->w.n_blocks,
                     resident && e->run.deps ? resident_runs(n_steps, std::min(chunk, most), most, e->w.n_blocks) : 0,
                     e->run.cus);
}

void engine_destroy(Engine *e)
{
    if (!e) return;
    if (e->stream) (void)hipStreamSynchronize(e->stream);
    e->graphs.destroy();
    for (void *p : e->allocs) (void)hipFree(p);
    if (e->out_h) (void)hipHostFree(e->out_h);
    for (hipEvent_t x : e->kt.pool) (void)hipEventDestroy(x);
    if (e->stream) (void)hipStreamDestroy(e->stream);
    delete e;
}

int64_t engine_device_bytes(Engine *e) { return e ? e->bytes : 0; }

void engine_blocks(Engine *e, int *n_blocks, int *n_staged)
{
    *n_blocks = e ? e->w.n_blocks : 0;
    *n_staged = e ? e->w.n_staged : 0;
}

void engine_run_counts(Engine *e, int64_t *launched, int64_t *given_up)
{
    if (launched) *launched = e ? e->run.launched : 0;
    if (given_up) *given_up = e ? e->run.given_up : 0;
}

int engine_sync(Engine *e)
{
    HIP_TRY(hipStreamSynchronize(e->stream));
    return SCAFFOLD_OK;
}

int engine_init_params(Engine *e, uint64_t seed, int64_t call_index)
{
    launch_init_params(e->stream, e->di, std::max(e->Ndev, e->hi.Wr), seed, (uint64_t)call_index);
    HIP_TRY(hipGetLastError());
    return engine_sync(e);
}

int engine_zero_g(Engine *e)
{
    launch_zero_g(e->stream, e->hi.st, e->Ndev);
    HIP_TRY(hipGetLastError());
    return engine_sync(e);
}

// Start the next run at step n.  The ring row of step n is cleared: every word of
// it is rewritten during step n, and team-mode words are assembled by atomicOr.
int engine_set_ctl(Engine *e, int64_t n, int64_t m)
{
    ++e->moved;
    const int row = (int)(((n % e->hi.R) + e->hi.R) % e->hi.R);
    HIP_TRY(hipMemsetAsync(e->hi.ring + (size_t)row * e->hi.Wr, 0, sizeof(uint64_t) * e->hi.Wr, e->stream));
    launch_set_ctl(e->stream, e->hi.ctl, n, m, row);
    HIP_TRY(hipGetLastError());
    return engine_sync(e);
}

int engine_upload_stims(Engine *e, const std::vector<ScStim> &stims)
{
    if ((int)stims.size() != e->n_stims) return fail(SCAFFOLD_ERR_STATE, "stimulus table size changed");
    if (stims.empty()) return SCAFFOLD_OK;
    // a launch takes 8 descriptors and 3-4 us of the caller's time, a copy 16 us whatever
    // their number: new rates and a one-step exchange take 27 against 36 us with 24 stimuli,
    // 47 against 36 with 64, 489 against 97 with 1024.  The copy need not wait: every
    // step of a call that has returned is done, and nothing after a run's steps reads these
    if (stims.size() > SC_STIMS_BY_LAUNCH) {
        HIP_TRY(hipMemcpy(e->stims, stims.data(), sizeof(ScStim) * stims.size(), hipMemcpyHostToDevice));
        return SCAFFOLD_OK;
    }
    e->queued = true;
    launch_set_stims(e->stream, e->stims, stims.data(), (int)stims.size());
    HIP_TRY(hipGetLastError());
    return SCAFFOLD_OK;
}

// Steps in runs of at most `chunk` (< ring rows, so the end of a run still finds
// every row of the run): the step kernels (and the plasticity kernels after
// each), then the run's end (statistics, the output train when the run is the
// last of a hand-off, the counter advance).  Runs are launched directly; with the
// `graph` option full runs replay a captured hipGraph (batches always do).
static void launch_step_kernels(hipStream_t s, const ScInstance *single, const ScInstance *insts, const DevWork &w,
                                int K)
{
    for (int k = 0; k < K; ++k) {
        launch_step(s, single, insts, w, k);
        if (single) launch_plastic(s, *single, w, k);
    }
}

static void launch_end(hipStream_t s, const ScInstance *single, ScInstance *insts, int n_inst, const DevWork &w,
                       int K, const ScOut *out, const ScSignal &stats = ScSignal{}, const RunSync *res = nullptr)
{
    launch_run_end(s, single, insts, n_inst, w, K, out, stats, res ? res->done : nullptr);
}

static bool same_out(const ScOut &a, const ScOut &b)
{
    return a.bits == b.bits && a.out == b.out && a.T == b.T && a.n_out == b.n_out;
}

// Captures `chunk` steps as a graph: the step kernels, and with `end` the run's
// end as well (with the output train when out is set).
static hipError_t capture_run(hipStream_t s, hipGraphExec_t *gexec, const ScInstance *single, ScInstance *insts,
                              int n_inst, const DevWork &w, int chunk, bool end, const ScOut *out)
{
    hipGraph_t g = nullptr;
    hipError_t err = hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal);
    if (err != hipSuccess) return err;
    launch_step_kernels(s, single, insts, w, chunk);
    if (end) launch_end(s, single, insts, n_inst, w, chunk, out);
    err = hipStreamEndCapture(s, &g);
    if (err == hipSuccess) err = hipGraphInstantiate(gexec, g, nullptr, nullptr, 0);
    if (g) (void)hipGraphDestroy(g);
    if (err != hipSuccess) *gexec = nullptr;
    return err;
}

// The graph `which` of G for runs of `chunk` steps, captured on first use.
static int graph_for(hipStream_t s, RunGraphs &G, int which, const ScInstance *single, ScInstance *insts,
                     int n_inst, const DevWork &w, int chunk, const ScOut *out, hipGraphExec_t *ge)
{
    RunGraphs::Slot &x = G.slot[which];
    const ScOut o = out ? *out : ScOut{};
    if (!x.exec || x.chunk != chunk || !same_out(x.out, o)) {
        if (x.exec) (void)hipGraphExecDestroy(x.exec);
        x.exec = nullptr;
        hipError_t err = capture_run(s, &x.exec, single, insts, n_inst, w, chunk, which != RunGraphs::STEPS, out);
        if (err != hipSuccess) return fail(SCAFFOLD_ERR_HIP, "graph capture: %s", hipGetErrorString(err));
        x.chunk = chunk;
        x.out = o;
    }
    *ge = x.exec;
    return SCAFFOLD_OK;
}

// The next pair of timer events (created on first use).
static int timer_pair(KTimer *kt, int K, hipEvent_t *a, hipEvent_t *b)
{
    while (kt->used + 2 > kt->pool.size()) {
        hipEvent_t x;
        HIP_TRY(hipEventCreate(&x));
        kt->pool.push_back(x);
    }
    *a = kt->pool[kt->used];
    *b = kt->pool[kt->used + 1];
    kt->used += 2;
    kt->piece_k.push_back(K);
    return SCAFFOLD_OK;
}

// The next signal of the engine's stream.
static ScSignal hand_signal(Engine *e) { return ScSignal{&e->hand_d->ready, ++e->seq}; }

// Waits until signal `seq` is in.  The host reads the word for about as long as short
// work takes (a read of the word is seen 3-8 us sooner than the runtime's wait returns), then
// leaves the wait to the runtime, which also reports what went wrong on the stream.
static int hand_wait(Engine *e, unsigned long long seq)
{
    if (seq == kNoSignal) {
        HIP_TRY(hipStreamSynchronize(e->stream));
        return SCAFFOLD_OK;
    }
    const auto arrived = [&] { return __atomic_load_n(&e->hand->ready, __ATOMIC_ACQUIRE) >= seq; };
    const auto t0 = std::chrono::steady_clock::now();
    while (!arrived()) {
        for (int i = 0; i < 64 && !arrived(); ++i) __builtin_ia32_pause();
        if (std::chrono::steady_clock::now() - t0 > std::chrono::milliseconds(2)) break;
    }
    if (!arrived()) HIP_TRY(hipStreamSynchronize(e->stream));
    return SCAFFOLD_OK;
}

// n_steps steps in runs: graph replays of `chunk` steps, then direct launches for
// the rest (every run direct without graphs).  With the timer on, each run's step
// kernels lie between two events and its end is launched after them.  `out`: the
// output train of the last out->T steps, gathered by the last run's end when that
// run holds them all (*out_taken then set; otherwise the caller gathers it).
// `n_runs`: the steps are that many resident runs (0: a launch per step).
// `e` (one instance): the end of its last run, if
// launched directly, signals the train (*train_seq; 0: no signal) and then the run's
// statistics (e->stats_seq), so a caller that waits for the train alone does not wait
// for the statistics.
static int run_steps(hipStream_t s, RunGraphs &G, const ScInstance *single, ScInstance *insts, int n_inst,
                     const DevWork &w, int n_steps, int use_graph, int chunk, KTimer *kt = nullptr,
                     Engine *e = nullptr, const ScOut *out = nullptr, bool *out_taken = nullptr,
                     unsigned long long *train_seq = nullptr, int n_runs = 0)
{
    if (out_taken) *out_taken = false;
    if (train_seq) *train_seq = 0;
    if (n_steps <= 0) return SCAFFOLD_OK;
    if (e) {
        e->queued = true;
        ++e->moved;
    }
    const bool timer = kt && kt->on;
    const RunSync *res = n_runs ? &e->run : nullptr;
    // steps of the last run
    const int last_k = res ? n_steps / n_runs : n_steps % chunk ? n_steps % chunk : chunk;
    const ScOut *last_out = out && out->out && out->T > 0 && out->T <= last_k ? out : nullptr;
    int done = 0;
    while (done < n_steps) {
        const int left = n_steps - done, K = res ? (left + n_runs - 1) / n_runs : std::min(chunk, left);
        if (res) --n_runs;
        const bool last = done + K == n_steps;
        const ScOut *o = last ? last_out : nullptr;
        const bool graph = use_graph && K == chunk;
        const bool timed = timer && kt->seq++ % kt->every == 0;  // one run in kt->every
        hipEvent_t a = nullptr, b = nullptr;
        if (timed) {
            int rc = timer_pair(kt, K, &a, &b);
            if (rc) return rc;
            HIP_TRY(hipEventRecord(a, s));
        }
        if (graph) {
            hipGraphExec_t ge = nullptr;
            const int which = timed ? RunGraphs::STEPS : o ? RunGraphs::RUN_OUT : RunGraphs::RUN;
            int rc = graph_for(s, G, which, single, insts, n_inst, w, chunk, which == RunGraphs::RUN_OUT ? o : nullptr,
                               &ge);
            if (rc) return rc;
            HIP_TRY(hipGraphLaunch(ge, s));
        } else if (res) {
            launch_run(s, *single, w, ScRun{res->deps, res->tags, res->done, res->failed_hd, K, res->polls});
            ++e->run.launched;
        } else {
            launch_step_kernels(s, single, insts, w, K);
        }
        if (timed) HIP_TRY(hipEventRecord(b, s));
        if (timed || !graph) {
            ScOut train = o ? *o : ScOut{};
            ScSignal stats{};
            if (e && last) {
                if (o && train_seq) {
                    train.sig = hand_signal(e);
                    *train_seq = train.sig.seq;
                }
                stats = hand_signal(e);
                e->stats_seq = stats.seq;
            }
            launch_end(s, single, insts, n_inst, w, K, o ? &train : nullptr, stats, res);
        } else if (e && last) {
            e->stats_seq = kNoSignal;
        }
        HIP_TRY(hipGetLastError());
        done += K;
    }
    if (out_taken) *out_taken = last_out != nullptr;
    return SCAFFOLD_OK;
}

static int chunk_for(int graph_steps, int R) { return std::max(1, std::min(graph_steps, R - 1)); }

// After a resident run was given up (its blocks were not on the device together in
// time, e.g. beside another process's): nothing of it or of the runs behind it was
// stored or counted.  Launches their steps again, a kernel per step, as all later
// ones of this engine will be.  *ms_per_step: what they took.
static int engine_recover(Engine *e, int graph_steps, double *ms_per_step)
{
    LocalEvents L;
    hipEvent_t a, b;
    int rc = L.make(&a);
    if (!rc) rc = L.make(&b);
    if (rc) return rc;
    HIP_TRY(hipStreamSynchronize(e->stream));
    ScCtl c;
    HIP_TRY(hipMemcpy(&c, e->hi.ctl, sizeof(c), hipMemcpyDeviceToHost));
    const int steps = c.skipped;
    c.failed = c.skipped = 0;
    HIP_TRY(hipMemcpy(e->hi.ctl, &c, sizeof(c), hipMemcpyHostToDevice));
    HIP_TRY(hipMemset(e->run.done, 0, sizeof(uint32_t)));
    HIP_TRY(hipMemset(e->hi.ring + (size_t)c.row * e->hi.Wr, 0, sizeof(uint64_t) * e->hi.Wr));
    HIP_TRY(hipDeviceSynchronize());  // the fills above, before the engine's (non-blocking) stream goes on
    *e->run.failed_h = 0u;
    e->run.deps = nullptr;
    ++e->run.given_up;
    HIP_TRY(hipEventRecord(a, e->stream));
    rc = run_steps(e->stream, e->graphs, &e->hi, e->di, 1, e->w, steps, 0, chunk_for(graph_steps, e->hi.R));
    if (rc) return rc;
    HIP_TRY(hipEventRecord(b, e->stream));
    HIP_TRY(hipStreamSynchronize(e->stream));
    float ms = 0.f;
    HIP_TRY(hipEventElapsedTime(&ms, a, b));
    if (ms_per_step) *ms_per_step = ms / std::max(1, steps);
    return SCAFFOLD_OK;
}

// Waits for signal `upto` (kNoSignal: for the engine's stream), then adds what the
// step-kernel timer measured.  *recovered: a resident run was given up and its steps
// were launched again, in *ms_per_step each; the timer leaves that call out (its events
// lie around runs that ended early).
static int engine_finish(Engine *e, int graph_steps, unsigned long long upto, bool *recovered = nullptr,
                         double *ms_per_step = nullptr)
{
    int rc = hand_wait(e, upto);
    if (rc) return rc;
    const bool failed = __atomic_load_n(&e->hand->run_failed, __ATOMIC_ACQUIRE) != 0;
    KTimer &kt = e->kt;
    float x = 0.f;
    for (size_t i = 0; i < kt.piece_k.size(); ++i) {
        HIP_TRY(hipEventSynchronize(kt.pool[2 * i + 1]));
        if (failed) continue;
        HIP_TRY(hipEventElapsedTime(&x, kt.pool[2 * i], kt.pool[2 * i + 1]));
        kt.ms += x;
        kt.launches += kt.piece_k[i];
    }
    kt.piece_k.clear();
    kt.used = 0;
    if (recovered) *recovered = failed;
    return failed ? engine_recover(e, graph_steps, ms_per_step) : (int)SCAFFOLD_OK;
}

int engine_run(Engine *e, int n_steps, int use_graph, int graph_steps)
{
    const int chunk = chunk_for(graph_steps, e->hi.R);
    const ChipShare share = share_for(e, n_steps, chunk, !use_graph);
    int rc = run_steps(e->stream, e->graphs, &e->hi, e->di, 1, e->w, n_steps, use_graph, chunk, &e->kt, e, nullptr,
                       nullptr, nullptr, share.n_runs);
    if (rc) return rc;
    return engine_finish(e, graph_steps, e->stats_seq);
}

int engine_run_output(Engine *e, int n_steps, int use_graph, int graph_steps, int64_t first_out_step,
                      const uint8_t **train, Recorder *rec, int rec_T, int64_t step0)
{
    const int chunk = chunk_for(graph_steps, e->hi.R);
    const ChipShare share = share_for(e, n_steps, chunk, !use_graph && !rec);
    int rc = SCAFFOLD_OK;
    // the train of steps [first_out_step, first_out_step + T_out) is gathered by
    // the end of the call's last run when the window closes the call and that run
    // holds all of it; otherwise by a launch of its own after the runs
    ScOut out;
    out.bits = e->out_bits;
    out.out = e->out_hd;
    out.T = e->T_out;
    out.n_out = e->n_out;
    const bool closes = train && out.T * out.n_out > 0 && first_out_step + out.T == step0 + n_steps;
    const int R = e->hi.R;
    const int row0 = (int)(((first_out_step % R) + R) % R);
    // the call returns once the train is in host memory (written there by the gather
    // itself), not after the last run's statistics
    bool taken = false;
    unsigned long long early = 0;
    if (!rec) {
        rc = run_steps(e->stream, e->graphs, &e->hi, e->di, 1, e->w, n_steps, use_graph, chunk, &e->kt,
                       e, closes ? &out : nullptr, &taken, &early, share.n_runs);
        if (rc) return rc;
    }
    for (int done = 0; rec && done < n_steps;) {
        const int64_t s = step0 + done;
        const int K = (int)std::min<int64_t>(n_steps - done, (s / rec_T + 1) * rec_T - s);
        if ((rc = recorder_before(rec, e->stream, s + K))) return rc;
        rc = run_steps(e->stream, e->graphs, &e->hi, e->di, 1, e->w, K, use_graph, chunk, &e->kt,
                       e, closes && done + K == n_steps ? &out : nullptr, &taken, &early);
        if (rc) return rc;
        if ((s + K) % rec_T == 0 && (rc = recorder_window(rec, e->stream, e->hi.ring, s + K))) return rc;
        done += K;
    }
    if (train) {
        if (!taken) {
            launch_out_train(e->stream, e->hi.ring, e->hi.Wr, R, row0, e->T_out, e->out_bits, e->n_out, out.out);
            HIP_TRY(hipGetLastError());
        }
        *train = e->out_h;  // complete once engine_finish has waited for its signal or the stream
    }
    bool recovered = false;
    const unsigned long long upto = !train ? e->stats_seq : early ? early : kNoSignal;
    if ((rc = engine_finish(e, graph_steps, upto, &recovered))) return rc;
    if (train && recovered) {  // the train of the steps launched again
        launch_out_train(e->stream, e->hi.ring, e->hi.Wr, R, row0, e->T_out, e->out_bits, e->n_out, out.out);
        HIP_TRY(hipGetLastError());
        HIP_TRY(hipStreamSynchronize(e->stream));
    }
    return SCAFFOLD_OK;
}

int engine_record_sync(Engine *e, Recorder *rec)
{
    return rec ? recorder_wait_all(rec, e->stream) : SCAFFOLD_OK;
}

int engine_timer(Engine *e, int on, double *ms, int64_t *launches)
{
    if (on >= 0) {
        e->kt.on = on != 0;
        if (on) { e->kt.ms = 0.0; e->kt.launches = 0; e->kt.every = on; e->kt.seq = 0; }
    }
    if (ms) *ms = e->kt.ms;
    if (launches) *launches = e->kt.launches;
    return SCAFFOLD_OK;
}

int engine_time(Engine *e, int n_steps, int use_graph, int graph_steps, double *ms_total, double *ms_kernel_mean)
{
    LocalEvents L;
    hipEvent_t a, b;
    int rc = L.make(&a);
    if (!rc) rc = L.make(&b);
    if (rc) return rc;
    const int chunk = chunk_for(graph_steps, e->hi.R);
    const ChipShare share = share_for(e, n_steps, chunk, !use_graph && !ms_kernel_mean);
    if (!ms_kernel_mean) {
        HIP_TRY(hipEventRecord(a, e->stream));
        rc = run_steps(e->stream, e->graphs, &e->hi, e->di, 1, e->w, n_steps, use_graph, chunk, &e->kt, e, nullptr,
                       nullptr, nullptr, share.n_runs);
        if (rc) return rc;
        HIP_TRY(hipEventRecord(b, e->stream));
    } else {
        ++e->moved;
        // direct launches; one event pair brackets each run of back-to-back step
        // kernels, so the mean is per step kernel without per-launch event overhead
        std::vector<hipEvent_t> ev;
        HIP_TRY(hipEventRecord(a, e->stream));
        int done = 0;
        while (done < n_steps) {
            const int K = std::min(chunk, n_steps - done);
            hipEvent_t s0, s1;
            rc = L.make(&s0);
            if (!rc) rc = L.make(&s1);
            if (rc) return rc;
            ev.push_back(s0);
            ev.push_back(s1);
            HIP_TRY(hipEventRecord(s0, e->stream));
            for (int k = 0; k < K; ++k) {
                launch_step(e->stream, &e->hi, e->di, e->w, k);
                launch_plastic(e->stream, e->hi, e->w, k);
            }
            HIP_TRY(hipEventRecord(s1, e->stream));
            launch_end(e->stream, &e->hi, e->di, 1, e->w, K, nullptr);
            done += K;
        }
        HIP_TRY(hipEventRecord(b, e->stream));
        HIP_TRY(hipEventSynchronize(b));
        double sum = 0.0;
        for (size_t i = 0; i < ev.size(); i += 2) {
            float x = 0.f;
            HIP_TRY(hipEventElapsedTime(&x, ev[i], ev[i + 1]));
            sum += x;
        }
        *ms_kernel_mean = sum / n_steps;
    }
    HIP_TRY(hipEventSynchronize(b));
    float ms = 0.f;
    HIP_TRY(hipEventElapsedTime(&ms, a, b));
    bool recovered = false;
    double ms_per_step = 0.0;
    rc = engine_finish(e, graph_steps, kNoSignal, &recovered, &ms_per_step);  // (the step-kernel timer's events, too)
    // a given-up run says nothing about the steps: those launched again do
    if (ms_total) *ms_total = recovered ? ms_per_step * n_steps : ms;
    return rc;
}

int engine_set_state(Engine *e, const float *V, const float *g, const int32_t *refr)
{
    HIP_TRY(hipStreamSynchronize(e->stream));
    const size_t N = (size_t)e->Ndev;
    std::vector<ScState> hs(N);
    HIP_TRY(hipMemcpy(hs.data(), e->hi.st, sizeof(ScState) * N, hipMemcpyDeviceToHost));
    for (size_t d = 0; d < N; ++d) {
        const int r = e->dev_to_ref[d];
        if (r < 0) continue;
        if (V) hs[d].V = V[r];
        if (g) { hs[d].g_exc = g[2 * (size_t)r]; hs[d].g_inh = g[2 * (size_t)r + 1]; }
        if (refr) hs[d].refr = refr[r];
    }
    HIP_TRY(hipMemcpy(e->hi.st, hs.data(), sizeof(ScState) * N, hipMemcpyHostToDevice));
    return SCAFFOLD_OK;
}

int engine_get_ring_row(Engine *e, int row, uint64_t *words)
{
    HIP_TRY(hipStreamSynchronize(e->stream));
    HIP_TRY(hipMemcpy(words, e->hi.ring + (size_t)row * e->hi.Wr, sizeof(uint64_t) * e->hi.Wr, hipMemcpyDeviceToHost));
    return SCAFFOLD_OK;
}

int engine_get_counts(Engine *e, int row, int32_t *counts, unsigned long long *events)
{
    int rc = hand_wait(e, e->stats_seq);
    if (rc) return rc;
    if (counts) memcpy(counts, e->counts_h + (size_t)row * e->n_pops, sizeof(int32_t) * e->n_pops);
    if (events) *events = e->events_h[row];
    return SCAFFOLD_OK;
}

int engine_get_totals(Engine *e, unsigned long long *totals)
{
    int rc = hand_wait(e, e->stats_seq);
    if (rc) return rc;
    memcpy(totals, e->totals_h, sizeof(unsigned long long) * (e->n_pops + 1));
    return SCAFFOLD_OK;
}

// A result that is handed over in parts: launch(c) queues the kernel that writes chunk c
// into part c % parts of the hand-off buffer and asks for one signal; copy(c) takes it out.
// Chunks are copied while the next ones come; for results above kCopyAlone bytes a few
// threads share the copying, which the page faults of newly allocated arrays bound.
constexpr int kParts = 4, kCopyThreads = 4;
constexpr size_t kCopyAlone = 2 << 20;

template <typename Launch, typename Copy>
static int hand_parts(Engine *e, int n_chunks, int parts, size_t bytes, const Launch &launch, const Copy &copy)
{
    const unsigned long long seq0 = e->seq + 1;  // signal of chunk c: seq0 + c
    int launched = 0;
    const auto launch_next = [&] {
        launch(launched++);
        return hipGetLastError();
    };
    while (launched < std::min(parts, n_chunks)) HIP_TRY(launch_next());
    const auto alone = [&](int c) {
        for (; c < n_chunks; ++c) {
            int rc = hand_wait(e, seq0 + c);
            if (rc) return rc;
            copy(c);
            if (launched < n_chunks) HIP_TRY(launch_next());
        }
        return (int)SCAFFOLD_OK;
    };
    if (bytes < kCopyAlone || parts < kParts) return alone(0);
    // chunks are taken in order; copied[p]: chunks that left part p
    std::atomic<int> next{0}, copied[kParts] = {};
    std::atomic<bool> stop{false};
    const auto arrived = [&](int c) { return __atomic_load_n(&e->hand->ready, __ATOMIC_ACQUIRE) >= seq0 + c; };
    const auto work = [&] {
        for (int c = next++; c < n_chunks; c = next++) {
            for (int i = 0; !arrived(c); ++i) {
                if (stop) return;
                if (i < 4096) __builtin_ia32_pause();
                else std::this_thread::yield();
            }
            copy(c);
            copied[c % kParts].fetch_add(1);
        }
    };
    std::thread helpers[kCopyThreads];
    int n_helpers = 0;
    try {
        for (; n_helpers < kCopyThreads; ++n_helpers) helpers[n_helpers] = std::thread(work);
    } catch (...) {  // no more threads: the ones that started do
    }
    if (!n_helpers) return alone(0);
    hipError_t err = hipSuccess;
    while (err == hipSuccess && launched < n_chunks) {
        for (int i = 1; err == hipSuccess && copied[launched % kParts] < launched / kParts; ++i) {
            __builtin_ia32_pause();
            if ((i & 0xFFFFF) == 0 && (err = hipStreamQuery(e->stream)) == hipErrorNotReady) err = hipSuccess;
        }
        if (err == hipSuccess) err = launch_next();
    }
    if (err == hipSuccess) err = hipStreamSynchronize(e->stream);
    if (err != hipSuccess) stop = true;
    for (int i = 0; i < n_helpers; ++i) helpers[i].join();
    if (err != hipSuccess) return fail(SCAFFOLD_ERR_HIP, "hand-over in parts: %s", hipGetErrorString(err));
    return SCAFFOLD_OK;
}

// The state in reference order, which a kernel brings it into.  One copy of the records,
// reordered by the host, took 4.0 ms at 1.55M neurons; 1.5 ms this way.
int engine_get_state(Engine *e, float *V, float *g, int32_t *refr)
{
    const int N = e->total_ref;
    if (N <= 0) return SCAFFOLD_OK;
    // (the buffer holds at least 4096 neurons, and all of a network of up to 65536)
    const int room = (int)(e->hand_bytes / sizeof(ScState)), parts = N <= std::min(room, 16384) ? 1 : kParts;
    const int cap = parts == 1 ? (N + 1) & ~1 : room / kParts & ~1, n_chunks = (N + cap - 1) / cap;
    const size_t part_bytes = (size_t)cap * sizeof(ScState);
    const auto launch = [&](int c) {
        launch_state(e->stream, e->hi, c * cap, std::min(cap, N - c * cap), cap, e->data_d + (c % parts) * part_bytes,
                     e->w.end_done, hand_signal(e));
    };
    const auto copy = [&](int c) {
        const size_t r0 = (size_t)c * cap, n = std::min((size_t)cap, (size_t)N - r0);
        const float *from = reinterpret_cast<const float *>(e->data + (c % parts) * part_bytes);
        if (V) memcpy(V + r0, from, n * sizeof(float));
        if (g) memcpy(g + 2 * r0, from + cap, 2 * n * sizeof(float));
        if (refr) memcpy(refr + r0, from + 3 * (size_t)cap, n * sizeof(int32_t));
    };
    return hand_parts(e, n_chunks, parts, (size_t)N * sizeof(ScState), launch, copy);
}

// The multipliers of a plastic projection in source order, handed over like the state.
// -1: `proj` is not plastic.
int engine_read_plastic(Engine *e, int proj, float *out)
{
    for (const Engine::PlasticView &v : e->plastic_views) {
        if (v.proj != proj) continue;
        const int64_t cap = (int64_t)(e->hand_bytes / kParts / sizeof(float)), n_chunks = (v.n + cap - 1) / cap;
        const auto launch = [&](int c) {
            launch_multipliers(e->stream, v.val, v.vidx + c * cap, (int)std::min(cap, v.n - c * cap),
                               reinterpret_cast<float *>(e->data_d) + (c % kParts) * cap, e->w.end_done, hand_signal(e));
        };
        const auto copy = [&](int c) {
            memcpy(out + c * cap, reinterpret_cast<const float *>(e->data) + (c % kParts) * cap,
                   sizeof(float) * (size_t)std::min(cap, v.n - c * cap));
        };
        return hand_parts(e, (int)n_chunks, kParts, (size_t)v.n * sizeof(float), launch, copy);
    }
    return -1;
}

int engine_get_fired(Engine *e, int row, int32_t *ids, int32_t cap, int32_t *n)
{
    const int32_t most = (int32_t)(e->hand_bytes / sizeof(int32_t));  // ids handed over at a time
    int32_t first = 0;
    do {
        const int32_t len = std::min(most, std::max(cap, 0) - first);
        const ScSignal sig = hand_signal(e);
        launch_fired(e->stream, e->hi.ring + (size_t)row * e->hi.Wr, e->hi.n_groups, e->hi.groups,
                     reinterpret_cast<int32_t *>(e->data_d), first, len, &e->hand_d->count, sig);
        HIP_TRY(hipGetLastError());
        int rc = hand_wait(e, sig.seq);
        if (rc) return rc;
        *n = e->hand->count;
        const int32_t k = std::min(len, *n - first);
        if (k > 0) memcpy(ids + first, e->data, sizeof(int32_t) * (size_t)k);
        first += len;
    } while (first < std::min(cap, *n));
    return SCAFFOLD_OK;
}

// engine_get_fired through the static scratch of the engine's device: the compaction
// writes its count and ids there, then both are copied out.
int engine_get_fired_noalloc(Engine *e, int row, int32_t *ids, int32_t cap, int32_t *n)
{
    if (cap < 0 || cap > SC_FIRED_NOALLOC_MAX)
        return fail(SCAFFOLD_ERR_CAPACITY, "cap %d: the static scratch holds at most %d ids", cap, SC_FIRED_NOALLOC_MAX);
    int32_t *count = e->scratch, *out = e->scratch + SC_SCRATCH_IDS;
    launch_fired(e->stream, e->hi.ring + (size_t)row * e->hi.Wr, e->hi.n_groups, e->hi.groups, out, 0, cap, count,
                 ScSignal{});
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(e->stream));
    HIP_TRY(hipMemcpy(n, count, sizeof(int32_t), hipMemcpyDeviceToHost));
    const int32_t k = std::min(cap, *n);
    if (k > 0) HIP_TRY(hipMemcpy(ids, out, sizeof(int32_t) * (size_t)k, hipMemcpyDeviceToHost));
    return SCAFFOLD_OK;
}

int engine_copy_probe(int64_t bytes, int iters, double *ms)
{
    int rc = check_device();
    if (rc) return rc;
    const int64_t n = std::max<int64_t>(1, bytes / 16);
    struct Buffers {
        void *a = nullptr, *b = nullptr;
        ~Buffers()
        {
            (void)hipFree(a);
            (void)hipFree(b);
        }
    } B;
    void *&a = B.a, *&b = B.b;
    HIP_TRY(hipMalloc(&a, n * 16));
    HIP_TRY(hipMalloc(&b, n * 16));
    HIP_TRY(hipMemset(a, 1, n * 16));
    LocalEvents L;
    hipEvent_t e0, e1;
    rc = L.make(&e0);
    if (!rc) rc = L.make(&e1);
    if (rc) return rc;
    const int grid = (int)std::min<int64_t>((n + 255) / 256, 256 * 64);
    launch_copy(nullptr, a, b, n, grid);
    HIP_TRY(hipEventRecord(e0));
    for (int i = 0; i < iters; ++i) launch_copy(nullptr, a, b, n, grid);
    HIP_TRY(hipEventRecord(e1));
    HIP_TRY(hipEventSynchronize(e1));
    float t = 0.f;
    HIP_TRY(hipEventElapsedTime(&t, e0, e1));
    *ms = t / iters;
    return SCAFFOLD_OK;
}

// ---------------------------------------------------------------------- batching
// Independent instances of uneven size advance together: the descriptors of all
// instances (each naming its instance) form one step kernel per exchange step.
struct Batch {
    hipStream_t stream = nullptr;
    std::vector<void *> allocs;
    std::vector<Engine *> engines;
    std::vector<uint64_t> moved;  // of each engine, after the batch's own last run (its rows are in the table)
    ScInstance *di = nullptr;
    int n_inst = 0;
    int min_R = 0;
    DevWork w;
    RunGraphs graphs;
};

void batch_destroy(Batch *b)
{
    if (!b) return;
    if (b->stream) (void)hipStreamSynchronize(b->stream);
    b->graphs.destroy();
    for (void *p : b->allocs) (void)hipFree(p);
    if (b->stream) (void)hipStreamDestroy(b->stream);
    delete b;
}

int batch_build(Batch **out, std::vector<Engine *> &engines, const std::vector<const Plan *> &plans)
{
    int stage = 1;  // staged only if every instance allows it
    for (const Plan *p : plans) stage = stage && p->stage;
    // nontemporal streams when the instances' streams together exceed 64 MB, or
    // when every instance's own plan loads them so
    int64_t algo = 0;
    bool nt_all = true;
    for (const Plan *p : plans) {
        algo += p->algo_bytes;
        nt_all = nt_all && p->nontemporal;
    }
    *out = nullptr;
    Batch *b = new Batch();
    auto bail = [&](int code) { batch_destroy(b); return code; };
    if (hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking) != hipSuccess)
        return bail(fail(SCAFFOLD_ERR_HIP, "hipStreamCreate failed"));
    std::vector<ScInstance> insts;
    std::vector<ScHostStats> stats;
    std::vector<ScLaneTask> lanes;
    std::vector<ScStimTask> stims;
    struct TeamEntry {
        int width;  // wavefronts
        size_t win; // index of its ranges in team_win_u
        ScTeamTask t;
    };
    std::vector<TeamEntry> teams;
    std::vector<TaskWin> lane_win, team_win_u;
    b->min_R = 1 << 30;
    for (size_t i = 0; i < engines.size(); ++i) {
        const Engine *e = engines[i];
        b->engines.push_back(engines[i]);
        b->moved.push_back(~0ull);
        insts.push_back(e->hi);
        stats.push_back(e->w.host);
        b->min_R = std::min(b->min_R, e->hi.R);
        for (ScLaneTask t : e->h_lanes) { t.inst = (int)i; lanes.push_back(t); }
        lane_win.insert(lane_win.end(), e->h_lane_win.begin(), e->h_lane_win.end());
        for (ScStimTask t : e->h_stims) { t.inst = (int)i; stims.push_back(t); }
        for (size_t j = 0; j < e->h_teams.size(); ++j) {
            ScTeamTask t = e->h_teams[j];
            t.inst = (int)i;
            teams.push_back({e->h_team_b[j], team_win_u.size(), t});
            team_win_u.push_back(e->h_team_win[j]);
        }
    }
    std::stable_sort(teams.begin(), teams.end(), [](const TeamEntry &x, const TeamEntry &y) { return x.width > y.width; });
    std::vector<ScTeamTask> tt;
    std::vector<int> tw;
    std::vector<TaskWin> team_win;
    for (const TeamEntry &p : teams) {
        tw.push_back(p.width);
        team_win.push_back(team_win_u[p.win]);
        tt.push_back(p.t);
    }
    int rc;
    if ((rc = dupload(b->allocs, nullptr, &b->di, insts))) return bail(rc);
    ScHostStats *hosts;
    if ((rc = dupload(b->allocs, nullptr, &hosts, stats))) return bail(rc);
    b->w.hosts = hosts;
    if ((rc = upload_work(b->allocs, nullptr, b->w, tw, lanes, stims, tt, lane_win, team_win, stage != 0,
                          plans[0]->stage_ratio, 0, 0, (int)insts.size())))
        return bail(rc);
    for (const ScInstance &x : insts) b->w.max_groups = std::max(b->w.max_groups, x.n_groups);
    b->w.nontemporal = nt_all || algo > ((int64_t)64 << 20);
    b->n_inst = (int)insts.size();
    *out = b;
    return SCAFFOLD_OK;
}

int batch_run(Batch *b, int n_steps, int graph_steps, double *ms)
{
    LocalEvents L;
    hipEvent_t e0, e1;
    int rc = L.make(&e0);
    if (!rc) rc = L.make(&e1);
    if (rc) return rc;
    const ChipShare share(b->engines[0]->device, b->w.n_blocks, 0, 0);
    // what calls on the networks themselves left queued: new rates, the end of a run
    for (Engine *e : b->engines) {
        if (!e->queued) continue;
        HIP_TRY(hipStreamSynchronize(e->stream));
        e->queued = false;
    }
    HIP_TRY(hipEventRecord(e0, b->stream));
    bool moved = false;
    for (size_t i = 0; i < b->engines.size(); ++i)
        if (b->engines[i]->moved++ != b->moved[i]) moved = true;
    if (moved) launch_batch_rows(b->stream, b->di, b->n_inst);
    rc = run_steps(b->stream, b->graphs, nullptr, b->di, b->n_inst, b->w, n_steps, 1,
                   chunk_for(graph_steps, b->min_R));
    if (rc) return rc;
    HIP_TRY(hipEventRecord(e1, b->stream));
    HIP_TRY(hipEventSynchronize(e1));
    float t = 0.f;
    HIP_TRY(hipEventElapsedTime(&t, e0, e1));
    if (ms) *ms = t;
    for (size_t i = 0; i < b->engines.size(); ++i) b->moved[i] = b->engines[i]->moved;
    return SCAFFOLD_OK;
}

}  // namespace sc
