// MTTKRP over the per-mode chunk-ordered nonzero streams (host side; kernels
// in mttkrp_kernels.hpp) and the process-wide tunables.
//
// Layout: the nonzeros of each ALTO chunk (2^chunk_log2 consecutive nonzeros
// in ALTO order) are stored, per target mode, sorted by that mode's row
// (stable), as packed coordinates + value; with the fiber layout by row and
// fiber row.  A lane group of G lanes (a power of two; E columns of the rank
// per lane) walks a contiguous range of the stream: batches of G nonzeros are
// loaded coalesced and decoded (one per lane) and their fields broadcast
// through DPP or readlane; the Hadamard product of the input factor rows is
// formed with one vector load per lane and row; contributions are summed in
// registers while the output row stays the same.  When it changes, the sums
// change places in LDS, so that hardware FP atomics go to consecutive columns,
// and a workgroup's last rows are combined before they are flushed.  (Mappings
// 0 and 1 of launch_mttkrp broadcast through LDS permutes and flush each
// group's rows directly.)
// Workgroups are mapped XCD-aware: the 8 XCDs each walk one contiguous eighth
// of the stream so that each XCD's L2 holds the factor rows of its region.
//
// Reference semantics: mttkrp_alto_par / mttkrp_alto_da_mem_pull
// (include/alto.hpp:617-623, :1227-1318).
#include "mttkrp_kernels.hpp"

namespace alto {

// Nonzeros walked by one lane group of the kernels that flush every group's
// rows by itself (Phi, the strided MTTKRP lanes, hot-row streams):
// ALTO_TUNE_SEG when set, else a power of two in [512, 4096] sized so that a
// launch has about 2^21 threads (G lanes per group), doubled for FP32
// accumulation.  Long segments cut the flushes -- and with them the atomic
// traffic on heavily used output rows -- while enough groups remain to fill
// the chip.
static int g_seg = 0;
int tuned_seg(uint64_t nnz, int G, int acc_bytes)
{
    if (g_seg > 0) return g_seg;
    if (nnz < (4ull << 20)) {
        // below 4M nonzeros a launch is latency-bound: short segments give
        // more lane groups.  Measured optimum on MI355X from 10K to 4M
        // nonzeros (3-5 modes, ranks 8-64, FP64 and FP32): ~0.16 sqrt(nnz)
        // nonzeros per group, as a power of two from 16
        const double target = 0.16 * sqrt((double)nnz);
        int seg = 16;
        while (seg < 256 && seg * 1.5 < target) seg <<= 1;
        return seg;
    }
    // large tensors: about 2^21 threads per launch (flushes cost more than
    // the lost parallelism), twice as long segments with FP32 accumulation
    const uint64_t want = (nnz * (uint64_t)G >> 21) * (acc_bytes < 8 ? 2 : 1);
    int seg = 512;
    while (seg < 4096 && (uint64_t)seg * 3 / 2 < want) seg <<= 1;
    return seg;
}

// Nonzeros walked by one lane group (G lanes) of the vector-lane MTTKRP kernels,
// whose workgroups combine their groups' last rows before they flush
// (flush_last_rows), so that a segment need not be long for the heavy rows'
// sake.  A group walks its segment in steps that each wait for their gathers;
// the shorter it is, the more wavefronts hide that.  About 4096 wavefronts
// (four per SIMD) are enough, more only add flushes: nnz G / 2^18 nonzeros,
// the largest power of two below two thirds of that, between
//  - 8, or G / 2 (a workgroup of few wide groups combines little: rank 64,
//    60K nonzeros: 17 us at 8, 13.4 at 16 and 32) and
//  - 32 (G <= 4), 64, or 128 (G >= 32): a workgroup then covers one to four
//    thousand nonzeros, and the heavy rows' atomics no longer show.
// All-mode averages at 16, 32, 64, 128, 256: FP64 rank 16, 200K nonzeros 11.3,
// 12.6, 17.6, 26.5, 44 us; 1000^3, 1M, rank 16 17.3, 17.6, 18.1, 22.6, 36 us; 4
// modes, 3M, rank 16 50, 50, 54, 59, 83; 20M, rank 32 448, 427, 435, 454, 482;
// rank 64 840, 689, 652, 643, 650; 76.9M, rank 32 1267, 1223, 1195, 1250, 1269;
// FP32 4 modes, 3M, rank 32 57, 56, 60, 70, 98; BF16 rank 64, 8M 167 (32), 173,
// 204, 263; 100M 2056 (32), 1967, 1954, 2007.
int lane_seg(uint64_t nnz, int G)
{
    if (g_seg > 0) return g_seg;
    const int lo = G / 2 > 8 ? G / 2 : 8;
    const int hi = G <= 4 ? 32 : G >= 32 ? 128 : 64;
    const uint64_t want = nnz * (uint64_t)G >> 18;
    int seg = lo;
    while (seg < hi && (uint64_t)seg * 3 < want) seg <<= 1;
    return seg;
}
static int g_chunk = 0;
static int g_nt = 0;
// lane mapping of the MTTKRP kernel; -1 = per element type
static int g_variant = -1;
static int g_graphs = 0;
static int g_hot = 0;
static int g_hot_block = 512;
static int g_hot_lds = 32768;
static int g_narrow_max = -1;  // -1: per element type (lane_cols)
static int g_narrow_small = 1;
// Phi kernel: 0 = runtime batch loop with LDS permutes, 1 = compile-time
// batch with DPP broadcasts (5% faster on the 120M-count CP-APR workload)
static int g_phi_variant = 1;
int phi_variant() { return g_phi_variant; }
// Fiber layout of the mode streams (tensors from 4M nonzeros, 3 or more
// modes): fibers of at least g_fiber_min nonzeros are walked with the
// fiber-mode factor row held in registers.  g_fibers = number of fiber
// modes per stream (0 = off; 2: the nonzeros outside the first mode's
// fibers are searched for fibers of a second mode -- measured slower on the
// 76.9M-nonzero rank-32 tensor: all-mode FP64 4.48 -> 4.53 ms, FP32 3.27 ->
// 3.65 ms, although it moves ~10% of the nonzeros into fibers)
static int g_fibers = 1;
// 3 (FP32 all-mode MTTKRP of the 76.9M-nonzero rank-32 tensor 3.27 ms
// against 3.44 at 4; FP64 equal within noise)
static int g_fiber_min = 3;
static int g_fiber_chunk = 30;
static uint64_t g_fiber_min_nnz = 4ull << 20;
static int g_fiber_rule = 0;  // fiber mode: 0 = the other mode with the fewest rows, 1 = the most
int fiber_rule() { return g_fiber_rule; }
int fiber_settings(int* min_len, int* chunk_log2, uint64_t* min_nnz)
{
    *min_len = g_fiber_min;
    *chunk_log2 = g_fiber_chunk;
    *min_nnz = g_fiber_min_nnz;
    return g_fibers;
}
// deterministic-order MTTKRP / Phi (fixed summation order, no float atomics)
static int g_det = 0;
int det_enabled() { return g_det; }
// CP-APR: products of the other modes' rows kept per nonzero across a
// mode's inner iterations (when they fit)
static int g_apr_pi_cache = 1;
int apr_pi_cache_enabled() { return g_apr_pi_cache; }
int graphs_enabled() { return g_graphs; }
// lockstep CP-ALS: the sessions' mode updates and fits in batched launches
static int g_lockstep_dense = 1;
int lockstep_dense_batch_enabled() { return g_lockstep_dense; }
// lockstep CP-ALS: repeated iterations replayed as a HIP graph
static int g_lockstep_graphs = 0;
int lockstep_graphs_enabled() { return g_lockstep_graphs; }
// FP32 / BF16 CP-ALS: Grams and row solves on FP64 MFMA
static int g_dense_f64 = 1;
int dense_f64_enabled() { return g_dense_f64; }
// server: small jobs iterated in lockstep groups
static uint64_t g_serve_lock_nnz = 0;
static int g_serve_lock_sessions = 64;
void serve_lockstep_settings(uint64_t* max_nnz, int* max_sessions)
{
    *max_nnz = g_serve_lock_nnz;
    *max_sessions = g_serve_lock_sessions;
}
int hot_rows_enabled() { return g_hot; }
int tuned_chunk_log2() { return g_chunk; }
int set_chunk(int v)
{
    if (v < 0 || v > 31) return ALTO_ERR_ARG;
    g_chunk = v;
    return ALTO_OK;
}
int set_seg(int v)
{
    if (v < 0 || v > (1 << 20)) return ALTO_ERR_ARG;
    g_seg = v;
    return ALTO_OK;
}

// ------------------------------------------------------------------ host side
// factor row offsets (row * rank) are carried as 32-bit values
int check_offsets(const alto_tensor* t, int R)
{
    for (int m = 0; m < t->nmode; ++m)
        if (t->dims[m] * (uint64_t)R >= (1ull << 32)) {
            set_error("mode %d: dims*rank = %llu exceeds 2^32 (32-bit row offsets)", m,
                      (unsigned long long)(t->dims[m] * (uint64_t)R));
            return ALTO_ERR_UNSUPPORTED;
        }
    return ALTO_OK;
}

static size_t elem_bytes(int precision) { return precision == ALTO_PREC_F64 ? 8 : precision == ALTO_PREC_F32 ? 4 : 2; }

// Stream layout for MTTKRPs of rank R in `precision`: per-mode streams,
// rank-ordered factor buffers and, with hot rows on, each stream grouped by
// hot pattern for the LDS budget.  A no-op once in place (so it may run
// inside a graph capture after a first call outside it).
int mttkrp_prepare(alto_tensor* t, int R, int precision, hipStream_t s)
{
    ALTO_TRY(check_offsets(t, R));
    ALTO_TRY(prepare_mode_streams(t, precision == ALTO_PREC_F64, precision != ALTO_PREC_F64, s));
    const size_t eb = elem_bytes(precision);
    ALTO_TRY(reserve_rank_copies(t, (uint64_t)R, eb, s));
    const int no = t->nmode - 1;
    const int v = g_variant >= 0 ? g_variant : 2;
    const uint64_t lane_bytes = precision == ALTO_PREC_BF16 ? 8 : 16;
    if (!g_hot || v != 2 || no < 1 || no > 2 || ((uint64_t)R * eb) % lane_bytes != 0) return ALTO_OK;
    for (int m = 0; m < t->nmode; ++m) {
        if (!t->ms[m].ranked) continue;
        int want[ALTO_MAXN - 1] = {0};
        bool any = false;
        int o = 0;
        for (int q = 0; q < t->nmode; ++q) {
            if (q == m) continue;
            uint64_t rows = (uint64_t)g_hot_lds / no / ((uint64_t)R * eb);
            if (rows > t->dims[q]) rows = t->dims[q];
            want[o] = (int)rows;
            any = any || rows > 0;
            ++o;
        }
        if (!any) continue;
        bool same = t->ms[m].split != 0;
        for (int q = 0; q < no && same; ++q) same = t->ms[m].hot_k[q] == want[q];
        if (!same) ALTO_TRY(split_stream(t, m, want, s));
    }
    return ALTO_OK;
}

// variant >= -1: that lane mapping (and `seg` as given), for the autotuner;
// -2: the process-wide knobs, else the tensor's tuned shape, else defaults
static int mttkrp_device_shape(alto_tensor* t, int mode, int R, const void* const* U, void* out, int precision,
                               int accumulate, hipStream_t s, int seg, int variant)
{
    if (mode < 0 || mode >= t->nmode || R < 1 || R > 128) {
        set_error("mttkrp: mode %d / rank %d out of range (rank 1..128)", mode, R);
        return ALTO_ERR_ARG;
    }
    ALTO_TRY(mttkrp_prepare(t, R, precision, s));
    uint64_t nout = t->dims[mode] * (uint64_t)R;
    if (g_det) {
        if (!accumulate) ALTO_TRY(fill_zero((double*)out, nout, s));
        return mttkrp_det_device(t, mode, R, U, (double*)out, precision, s);
    }
    MttkrpTune k;
    k.variant = variant >= -1 ? variant : g_variant;
    if (variant == -2 && seg <= 0 && g_seg == 0 && g_variant < 0) {  // shape from the autotuner, if it ran
        for (const auto& c : t->tuned)
            if (c.mode == mode && c.rank == R && c.precision == precision) {
                k.variant = c.variant;
                seg = c.seg;
                break;
            }
    }
    k.nt = g_nt;
    k.hot_block = g_hot_block;
    k.hot_lds = g_hot_lds;
    k.narrow_max = g_narrow_max;
    k.narrow_small = g_narrow_small;
    if (precision == ALTO_PREC_F64) {
        if (!accumulate) ALTO_TRY(fill_zero((double*)out, nout, s));
        return launch_mttkrp_f64(t, mode, R, (const double* const*)U, t->ms[mode].val64.as<double>(), (double*)out, seg,
                                 k, s);
    }
    // FP32 / BF16: products and row sums in FP32 registers, flushed into an
    // FP64 output (FP32 atomics summing thousands of row partials lost
    // ~5e-4 of the heavy rows of a 200M-nonzero Zipf(1.2) tensor)
    if (!accumulate) ALTO_TRY(fill_zero((double*)out, nout, s));
    if (precision == ALTO_PREC_F32)
        return launch_mttkrp_f32(t, mode, R, (const float* const*)U, t->ms[mode].val32.as<float>(), (double*)out, seg,
                                 k, s);
    if (precision == ALTO_PREC_BF16)
        return launch_mttkrp_bf16(t, mode, R, (const bf16_t* const*)U, t->ms[mode].val32.as<float>(), (double*)out,
                                  seg, k, s);
    set_error("mttkrp: unknown precision %d", precision);
    return ALTO_ERR_ARG;
}

int mttkrp_device(alto_tensor* t, int mode, int R, const void* const* U, void* out, int precision, int accumulate,
                  hipStream_t s, int seg)
{
    return mttkrp_device_shape(t, mode, R, U, out, precision, accumulate, s, seg, -2);
}

// the segment length that lane mapping v takes by itself for this tensor and mode
template <typename FT, typename VT>
static int own_seg(const alto_tensor* t, int mode, int R, const void* const* U, int v)
{
    if (v == 2) {
        StreamArgs<FT, VT, double> a;
        fill_stream_args(t, mode, R, 0, a);
        for (int m = 0; m < t->nmode; ++m)
            if (m != mode) a.Uo[a.nother++] = (const FT*)U[m];
        MttkrpTune k;
        k.narrow_max = g_narrow_max;
        k.narrow_small = g_narrow_small;
        int G = 0, E = 0;
        if (vector_lane_shape(t, mode, R, a, k, G, E)) return lane_seg(t->nnz, G);
    }
    return tuned_seg(t->nnz, group_lanes(R), (int)sizeof(VT));  // (32-bit values are summed in 32 bits)
}

}  // namespace alto

using namespace alto;

extern "C" {

int alto_tune_set(int param, int value)
{
    if (param == ALTO_TUNE_SEG) return set_seg(value);
    if (param == ALTO_TUNE_CHUNK_LOG2) return set_chunk(value);
    if (param == ALTO_TUNE_NARROW_RANK) {
        if (value < -1 || value > 128) return ALTO_ERR_ARG;
        g_narrow_max = value;
        return ALTO_OK;
    }
    if (param == ALTO_TUNE_HOT_ROWS) {
        g_hot = value ? 1 : 0;
        return ALTO_OK;
    }
    if (param == ALTO_TUNE_HOT_BLOCK) {
        if (value != 256 && value != 512 && value != 1024) return ALTO_ERR_ARG;
        g_hot_block = value;
        return ALTO_OK;
    }
    if (param == ALTO_TUNE_HOT_LDS) {
        if (value < 0 || value > 160 * 1024) return ALTO_ERR_ARG;
        g_hot_lds = value;
        return ALTO_OK;
    }
    if (param == ALTO_TUNE_GRAPHS) {
        g_graphs = value ? 1 : 0;
        return ALTO_OK;
    }
    if (param == ALTO_TUNE_MTTKRP_VARIANT) {
        if (value < -1 || value > 2) return ALTO_ERR_ARG;
        g_variant = value;
        return ALTO_OK;
    }
    if (param == ALTO_TUNE_NARROW_SMALL) {
        g_narrow_small = value ? 1 : 0;
        return ALTO_OK;
    }
    if (param == ALTO_TUNE_PHI_VARIANT) {
        if (value < 0 || value > 2) return ALTO_ERR_ARG;
        g_phi_variant = value;
        return ALTO_OK;
    }
    if (param == ALTO_TUNE_FIBERS) {
        if (value < 0 || value > 2) return ALTO_ERR_ARG;
        g_fibers = value;
        return ALTO_OK;
    }
    if (param == ALTO_TUNE_DETERMINISTIC) {
        g_det = value ? 1 : 0;
        return ALTO_OK;
    }
    if (param == ALTO_TUNE_DENSE_F64) {
        g_dense_f64 = value ? 1 : 0;
        return ALTO_OK;
    }
    if (param == ALTO_TUNE_SERVE_LOCKSTEP_NNZ) {
        if (value < 0) return ALTO_ERR_ARG;
        g_serve_lock_nnz = (uint64_t)value;
        return ALTO_OK;
    }
    if (param == ALTO_TUNE_SERVE_LOCKSTEP_SESSIONS) {
        if (value < 1 || value > 4096) return ALTO_ERR_ARG;
        g_serve_lock_sessions = value;
        return ALTO_OK;
    }
    if (param == ALTO_TUNE_LOCKSTEP_GRAPHS) {
        g_lockstep_graphs = value ? 1 : 0;
        return ALTO_OK;
    }
    if (param == ALTO_TUNE_LOCKSTEP_DENSE_BATCH) {
        g_lockstep_dense = value ? 1 : 0;
        return ALTO_OK;
    }
    if (param == ALTO_TUNE_APR_PI_CACHE) {
        g_apr_pi_cache = value ? 1 : 0;
        return ALTO_OK;
    }
    if (param == ALTO_TUNE_FIBER_MIN) {
        if (value < 2 || value > (1 << 20)) return ALTO_ERR_ARG;
        g_fiber_min = value;
        return ALTO_OK;
    }
    if (param == ALTO_TUNE_FIBER_CHUNK_LOG2) {
        if (value < 10 || value > 31) return ALTO_ERR_ARG;
        g_fiber_chunk = value;
        return ALTO_OK;
    }
    if (param == ALTO_TUNE_FIBER_MODE_RULE) {
        if (value < 0 || value > 1) return ALTO_ERR_ARG;
        g_fiber_rule = value;
        return ALTO_OK;
    }
    if (param == ALTO_TUNE_FIBER_MIN_NNZ) {
        if (value < 0) return ALTO_ERR_ARG;
        g_fiber_min_nnz = (uint64_t)value;
        return ALTO_OK;
    }
    if (param == ALTO_TUNE_NONTEMPORAL) {
        g_nt = value ? 1 : 0;
        return ALTO_OK;
    }
    set_error("alto_tune_set: unknown parameter %d", param);
    return ALTO_ERR_ARG;
}

int alto_mttkrp_autotune(alto_tensor_t* t, uint64_t rank, int precision, const void* const* factors, void* out,
                         int reps, alto_stream_t stream, alto_tune_entry_t* result)
{
    if (!t || !factors || !out || rank < 1 || rank > 128 || reps < 1) {
        set_error("alto_mttkrp_autotune: invalid argument");
        return ALTO_ERR_ARG;
    }
    hipStream_t s = (hipStream_t)stream;
    const int R = (int)rank;
    static const int variants[] = {2, 0, 1};
    static const int segs[] = {16, 32, 64, 128, 256, 512, 1024, 2048, 4096};
    hipEvent_t e0 = nullptr, e1 = nullptr;
    HIP_TRY(hipEventCreate(&e0));
    HIP_TRY(hipEventCreate(&e1));
    int st = ALTO_OK;
    // times `reps` accumulating launches of one shape (variant -1 / seg 0:
    // the defaults, without any tuned entry)
    auto time_cfg = [&](int mode, int v, int sg, double* ms) -> int {
        // warm-up first (it also prepares the streams)
        int r = mttkrp_device_shape(t, mode, R, factors, out, precision, 1, s, sg, v);
        if (r == ALTO_OK && hipEventRecord(e0, s) != hipSuccess) r = ALTO_ERR_HIP;
        for (int k = 0; k < reps && r == ALTO_OK; ++k)
            r = mttkrp_device_shape(t, mode, R, factors, out, precision, 1, s, sg, v);
        if (r == ALTO_OK && hipEventRecord(e1, s) != hipSuccess) r = ALTO_ERR_HIP;
        if (r == ALTO_OK && hipEventSynchronize(e1) != hipSuccess) r = ALTO_ERR_HIP;
        float f = 0;
        if (r == ALTO_OK && hipEventElapsedTime(&f, e0, e1) != hipSuccess) r = ALTO_ERR_HIP;
        *ms = (double)f / reps;
        return r;
    };
    // the defaults must not pick up an earlier tuned entry for this case
    std::vector<alto_tensor::Tuned> keep;
    for (const auto& c : t->tuned)
        if (!(c.rank == R && c.precision == precision)) keep.push_back(c);
    t->tuned = keep;
    for (int mode = 0; mode < t->nmode && st == ALTO_OK; ++mode) {
        double def_ms = 0, best_ms = 0;
        st = time_cfg(mode, -2, 0, &def_ms);
        int bv = -1, bs = 0;
        best_ms = def_ms;
        // segment lengths within 4x of what the mapping takes by itself (the
        // others measured slower on every tensor tried, up to 10x on large ones)
        for (int v : variants) {
            const int h = precision == ALTO_PREC_F64   ? own_seg<double, double>(t, mode, R, factors, v)
                          : precision == ALTO_PREC_F32 ? own_seg<float, float>(t, mode, R, factors, v)
                                                       : own_seg<bf16_t, float>(t, mode, R, factors, v);
            for (int sg : segs) {
                if (sg * 4 < h || sg > h * 4) continue;
                if (st != ALTO_OK) break;
                double ms = 0;
                st = time_cfg(mode, v, sg, &ms);
                if (st == ALTO_OK && ms < best_ms) {
                    best_ms = ms;
                    bv = v;
                    bs = sg;
                }
            }
        }
        if (st != ALTO_OK) break;
        if (bv >= 0) t->tuned.push_back({mode, R, precision, bv, bs});
        if (result) {
            result[mode].mode = mode;
            result[mode].variant = bv;
            result[mode].seg = bs;
            result[mode].ms = best_ms;
            result[mode].default_ms = def_ms;
        }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    return st;
}

int alto_mttkrp(alto_tensor_t* t, int mode, uint64_t rank, const void* const* factors, void* out, int precision,
                int accumulate, alto_stream_t stream)
{
    if (!t || !factors || !out) {
        set_error("alto_mttkrp: null argument");
        return ALTO_ERR_ARG;
    }
    ALTO_TRY(mttkrp_device(t, mode, (int)rank, factors, out, precision, accumulate, (hipStream_t)stream, 0));
    return t->note_use((hipStream_t)stream);
}

int alto_mttkrp_batched(int njobs, alto_tensor_t* const* tensors, const int* modes, uint64_t rank,
                        const void* const* const* factors, void* const* outs, int precision, int accumulate,
                        alto_stream_t stream)
{
    ALTO_TRY(alto::mttkrp_batched_impl(njobs, tensors, modes, rank, factors, outs, precision, accumulate,
                                       (hipStream_t)stream));
    for (int i = 0; i < njobs; ++i) {
        bool seen = false;  // one event per tensor listed several times
        for (int k = 0; k < i && !seen; ++k) seen = tensors[k] == tensors[i];
        if (!seen) ALTO_TRY(tensors[i]->note_use((hipStream_t)stream));
    }
    return ALTO_OK;
}

}  // extern "C"

namespace alto {

// alto_mttkrp_batched without the tensors' use events (for callers that
// synchronize the stream themselves, such as lockstep CP-ALS)
int mttkrp_batched_impl(int njobs, alto_tensor_t* const* tensors, const int* modes, uint64_t rank,
                        const void* const* const* factors, void* const* outs, int precision, int accumulate,
                        hipStream_t s)
{
    if (njobs < 0 || (njobs > 0 && (!tensors || !modes || !factors || !outs))) {
        set_error("alto_mttkrp_batched: null argument");
        return ALTO_ERR_ARG;
    }
    if (precision != ALTO_PREC_F64 && precision != ALTO_PREC_F32 && precision != ALTO_PREC_BF16) {
        set_error("alto_mttkrp_batched: unknown precision %d", precision);
        return ALTO_ERR_ARG;
    }
    const int R = (int)rank;
    for (int i = 0; i < njobs; ++i) {
        alto_tensor* t = tensors[i];
        if (!t || !factors[i] || !outs[i]) {
            set_error("alto_mttkrp_batched: null argument in job %d", i);
            return ALTO_ERR_ARG;
        }
        if (modes[i] < 0 || modes[i] >= t->nmode || rank < 1 || rank > 128) {
            set_error("alto_mttkrp_batched: job %d: mode %d / rank %llu out of range (rank 1..128)", i, modes[i],
                      (unsigned long long)rank);
            return ALTO_ERR_ARG;
        }
        for (int m = 0; m < t->nmode; ++m)
            if (!factors[i][m]) {
                set_error("alto_mttkrp_batched: job %d: null factor %d", i, m);
                return ALTO_ERR_ARG;
            }
    }
    if (g_det) {  // one deterministic MTTKRP per job
        for (int i = 0; i < njobs; ++i)
            ALTO_TRY(mttkrp_device(tensors[i], modes[i], R, factors[i], outs[i], precision, accumulate, s, 0));
        return ALTO_OK;
    }
    MttkrpTune k;
    k.variant = g_variant;
    k.nt = g_nt;
    k.hot_block = g_hot_block;
    k.hot_lds = g_hot_lds;
    k.narrow_max = g_narrow_max;
    k.narrow_small = g_narrow_small;
    std::vector<const void*> vals(njobs);
    for (int i = 0; i < njobs; ++i) {
        alto_tensor* t = tensors[i];
        ALTO_TRY(mttkrp_prepare(t, R, precision, s));
        const uint64_t nout = t->dims[modes[i]] * (uint64_t)R;
        if (precision == ALTO_PREC_F64) {
            vals[i] = t->ms[modes[i]].val64.as<double>();
            if (!accumulate) ALTO_TRY(fill_zero((double*)outs[i], nout, s));
        } else {
            vals[i] = t->ms[modes[i]].val32.as<float>();
            if (!accumulate) ALTO_TRY(fill_zero((double*)outs[i], nout, s));
        }
    }
    if (njobs == 0) return ALTO_OK;
    if (precision == ALTO_PREC_F64)
        return launch_mttkrp_batch_f64(njobs, tensors, modes, R, (const double* const* const*)factors,
                                       (const double* const*)vals.data(), (double* const*)outs, g_seg, k, s);
    if (precision == ALTO_PREC_F32)
        return launch_mttkrp_batch_f32(njobs, tensors, modes, R, (const float* const* const*)factors,
                                       (const float* const*)vals.data(), (double* const*)outs, g_seg, k, s);
    return launch_mttkrp_batch_bf16(njobs, tensors, modes, R, (const bf16_t* const* const*)factors,
                                    (const float* const*)vals.data(), (double* const*)outs, g_seg, k, s);
}

}  // namespace alto
