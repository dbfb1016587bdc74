// Internal: the per-cluster context behind abyss_ctx_t, shared by the
// single-cluster runtime (regf_runtime.hip) and the ensemble / serving
// runtime (regf_ensemble.hip).  Not part of the public ABI.
#pragma once
#include "../../include/abyss_regf.h"
#include "regf_internal.h"

struct abyss_ctx_s {
    int device = -1;
    hipStream_t stream = nullptr;
    bool own_stream = true;   // false: the stream belongs to an ensemble
    int cu_count = 0;
    int cap = ABYSS_NUM_NEIGHBOR_MAX;
    int precision = ABYSS_PREC_CHECKED;
    int force_ipl = 0, force_splits = 0, force_unroll = 0, force_jl = 0;
    int force_tile = 0, force_wpb = 0;   // lanes-per-target shape (0: automatic)
    bool batch_member = false;   // an ensemble's cluster: lane-group plans only
    unsigned long long scratch_limit = 2ull << 30;   // split-j scratch bound

    // j-set: device SoA [x|y|z|vx|vy|vz|m|rnb2] (stride n) + FP32 mass
    int n = 0;
    size_t j_bytes = 0;
    char *d_j = nullptr;
    char *h_j = nullptr;  // pinned staging, same layout
    abyss::JState js{};

    // targets and outputs
    int nt = 0;
    bool counts_valid = false;   // d_nnb holds the counts of the current targets
    size_t t_capacity = 0;  // targets the output buffers can hold
    // Work on the stream that may not have finished and uses host staging or
    // the target and output buffers: a target list's way to the device or a
    // launch (busy_tgt), the list kernels (busy_irr), a state update
    // (busy_upd).  ctx_wait clears them.  A call that only needs one of these
    // buffers need not wait for an upload or a prediction before it.
    bool busy_tgt = false, busy_irr = false, busy_upd = false;
    // no caller can put work of its own on the stream (the drop-in calls'
    // context), so the flags tell all there is
    bool closed = false;
    // A caller's capture has recorded work of this context, which it may
    // replay at any time between calls: calls then keep to the buffers and the
    // waits that such work can rely on (ctx_launch_force, ctx_set_targets).
    bool captured = false;
    // ... has recorded a prediction, so the j-set may change with no call
    bool predict_recorded = false;
    int *d_tgt = nullptr, *h_tgt = nullptr;
    // h_tgt is mapped, coherent pinned memory; h_tgt_dev is its device
    // address.  `tgt` is the target array the kernels read: h_tgt_dev for
    // small blocks (no copy), d_tgt otherwise.
    const int *h_tgt_dev = nullptr, *tgt = nullptr;
    // per-target results (device block and pinned host mirror, same
    // layout): acc [nt][3] | adot [nt][3] | nnb [nt] | pad to 256 B | list
    // rows [nt][cap]; the pointers below are views of d_out / h_out for the
    // current nt (the host mirror holds the rows that fit one copy, or those
    // that a query's last kernels write there)
    char *d_out = nullptr, *h_out = nullptr;
    size_t h_row_bytes = 0;   // list rows h_out has room for
    double *d_acc = nullptr, *d_adot = nullptr;
    int *d_nnb = nullptr, *d_list = nullptr;
    double *h_res = nullptr;  // acc then adot
    int *h_nnb = nullptr, *h_rows = nullptr;
    // h_out is mapped, coherent pinned memory; the last kernels of small
    // launches also write the results there (device view `mirror`; for one
    // split it is where the views above point), and mirror_valid tells fetch
    // that no copy is needed
    char *h_out_dev = nullptr;
    abyss::FinalMirror mirror{};
    bool mirror_valid = false;
    int *h_list = nullptr;    // mapped pinned rows of larger results
    int *h_list_dev = nullptr;   // their device address
    size_t h_list_bytes = 0;
    // one event per chunk of a large fetch
    static constexpr int kFetchChunks = 16;
    hipEvent_t fev[kFetchChunks] = {};
    // list rows under way on `side`, beside the recomputation of checked
    // precision, to the fetch that follows the launch (set by the launch)
    hipStream_t side = nullptr;
    hipEvent_t sums_ev = nullptr;
    bool rows_sent = false, side_busy = false;
    int rows_chunks = 0, rows_width = 0, rows_overflowed = 0;
    size_t rows_bytes = 0;

    // device-resident particle state (regf_state.hip): SoA x,v,a,adot (3n
    // each), t, m, r2 (n each); staging for incremental updates
    double *d_state = nullptr, *h_state = nullptr;
    size_t state_bytes = 0;
    int state_n = 0;
    char *h_upd = nullptr, *h_upd_dev = nullptr;
    size_t upd_bytes = 0;

    // resident neighbour lists (regf_irregular.hip): [nnb: n ints, padded
    // to 64][list: n rows of cap ints], row = particle index; filled after
    // each launch while keep_lists is on
    bool keep_lists = false;
    char *d_rlists = nullptr;
    size_t rlist_bytes = 0;
    int rlist_n = 0;
    // inputs and results of the list kernels: device copy of the inputs, and
    // mapped pinned staging (device address h_irr_dev) of both
    char *d_irr = nullptr, *h_irr = nullptr, *h_irr_dev = nullptr;
    size_t d_irr_bytes = 0, irr_bytes = 0;
    // 64-byte AoS copy of the j-set {x,y,z,vx,vy,vz,m,0} for the list
    // gathers (one cache line per neighbour instead of seven); rebuilt when
    // jset_version (bumped by every upload / predict) has moved on
    char *d_aos = nullptr;
    size_t aos_bytes = 0;
    long long jset_version = 0, aos_version = -1;
    // start-up derivatives (regf_derivs.hip): records, split partials,
    // targets, results; pinned targets + results; radius results
    char *d_drv = nullptr, *h_drv = nullptr;
    size_t drv_bytes = 0, h_drv_bytes = 0;
    char *d_rad = nullptr;
    size_t rad_bytes = 0;

    // split-j scratch
    size_t scratch_bytes = 0;
    char *d_scratch = nullptr;
    abyss::QueryOut part{};

    // checked precision: device block of spread [t][2] | spread partials
    // [S][t][2] | counters [2] | flagged positions [t] | their j-indices [t];
    // the recomputation's split partials; pinned readback of the count
    char *d_chk = nullptr;
    size_t chk_bytes = 0;
    float *chk_spread = nullptr, *chk_pspread = nullptr;
    int *chk_counters = nullptr, *chk_fq = nullptr, *chk_fi = nullptr;
    char *d_rchk = nullptr;
    size_t rchk_bytes = 0;
    int *h_chk = nullptr;       // pinned, mapped: [0] flagged-count readback,
                                // [1] the count a device-read recomputation reports
    int *h_chk_dev = nullptr;   // device address of h_chk
    double check_tol = 1.0e-6;
    int n_rechecked = 0;        // targets recomputed by the last launch
    bool recheck_pending = false;   // n_rechecked is h_chk[1] once the stream drains
    bool spread_valid = false;  // chk_spread holds the last launch's spread

    abyss::Plan plan{};
    bool plan_valid = false;

    // counters (ProfileDevice); t_grav_ms is the legacy entry points'
    // wall-clock time in CalculateAccelerationOnDevice
    long long n_send = 0, n_grav = 0, sum_ni = 0;
    double interactions = 0.0, t_grav_ms = 0.0;

    // force-kernel timing (abyss_ctx_set_kernel_timing): an event pair
    // around the force kernel of every launch, in a ring that is read when
    // it fills and at sync
    static constexpr int kTimingRing = 64;
    bool ktiming = false;
    hipEvent_t kev[2 * kTimingRing] = {};
    int kev_used = 0;
    double kforce_ms = 0.0;
    long long klaunches = 0;

    char detail[512] = {0};
};


namespace abyss {
// 64-byte AoS record of the j-set for the list gathers.
struct __align__(64) JRec {
    double x, y, z, vx, vy, vz, m, pad;
};
// Up to this many targets the list kernels read their targets (and a regular
// step its dt and a_old) from mapped host memory instead of a device copy: a
// copy is 3 us before the kernel can start (N = 65536, one target: 19.1 us
// with it, 16.2 without), but in place every workgroup's 16 bytes are a read
// over the link of their own; at 16384 targets the two are even (72 to 75 us).
constexpr int kMappedListTargets = 16384;

// Creates a context that issues all its work on `stream` (owned by the
// caller) instead of a stream of its own.
int ctx_create_on_stream(int device, int cap, hipStream_t stream, abyss_ctx_t *out);
// abyss_ctx_fetch with the device->host work issued on `st` (which must not
// race with a launch writing this context's outputs).
int ctx_fetch_on_stream(abyss_ctx_t c, hipStream_t st, double *acc, double *adot, int *nnb,
                        int *list);
// Device bytes a context holds (j-set, targets, outputs, scratch).
unsigned long long ctx_device_bytes(abyss_ctx_t c);
// abyss_ctx_launch without keeping the resident lists (force kernels only).
// to_host: a fetch follows, so blocks of up to kQueryMirrorTargets targets
// also write their results to mapped host memory, small ones only there.
int ctx_launch_force(abyss_ctx_t c, bool to_host = false);
// After a launch: copies its neighbour rows into the resident per-particle
// lists when they are enabled (no-op otherwise).
int keep_launch_lists(abyss_ctx_t c);
// Checked precision: the spread / flag buffers for nt targets and S splits.
int ctx_ensure_check(abyss_ctx_t c, int nt, int S);
// abyss_ctx_set_targets that waits for the context's stream always, only for
// work that uses the target list or the outputs (a synchronous call's own
// step), or not at all (the caller guarantees that no launch using this
// context is in flight: an ensemble member whose last batch has finished).
enum class TargetWait { kStream, kUse, kNone };
int ctx_set_targets(abyss_ctx_t c, int nt, const int *targets, TargetWait wait);
// Waits for the context's stream.
int ctx_wait(abyss_ctx_t c);
// Whether a caller's capture is recording the context's stream.
int ctx_capturing(abyss_ctx_t c, bool *capturing);
// ABYSS_ERR_HIP under such a capture: for a call that waits for the stream, but
// not before it has enqueued work or changed what the context holds.
int refuse_capture(abyss_ctx_t c);
}  // namespace abyss
