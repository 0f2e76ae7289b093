// CP-APR Phi with one nonzero per lane and the rank's columns in registers
// (ranks 2 to 16), over the per-mode nonzero streams (layout: mttkrp.hip).
//
// Reference semantics: CalculatePhi_alto_par (include/apr.hpp:295-303,
// :383-501); the products kept per nonzero are its PRE mode
// (include/apr.hpp:1049-1097, 1128-1165).
#include "mttkrp_kernels.hpp"
#include "phi_cols.hpp"

namespace alto {

namespace {

constexpr uint32_t NO_ROW = 0xffffffffu;

// the value DPP control C brings from another lane, 0 where there is none
template <int C, int ROWS = 0xf> __device__ __forceinline__ double dpp_f64(double v)
{
    const uint64_t u = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, C, ROWS, 0xf, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), C, ROWS, 0xf, false);
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}
constexpr int ROW_SHR1 = 0x111, ROW_SHR2 = 0x112, ROW_SHR4 = 0x114, ROW_SHR8 = 0x118;
constexpr int ROW_BCAST15 = 0x142, ROW_BCAST31 = 0x143;  // into rows 1, 3 and into rows 2, 3

__device__ __forceinline__ double lane63(double v)
{
    const uint64_t u = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)u, 63), hi = __builtin_amdgcn_readlane((uint32_t)(u >> 32), 63);
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

// Phi: per nonzero pi = prod_{m != n} U_m[row_m,:], d = <B[row,:], pi>,
// contribution (x / max(d, eps)) * pi into row `row`.
//
// A wavefront takes blocks of 64 consecutive nonzeros, one per lane, each
// lane holding its nonzero's columns as P pairs (an odd rank's last pair is
// the row's last two columns, its first one a duplicate that the dot product
// leaves out).  Against lane groups per nonzero (k_phi_b) the dot product
// needs no cross-lane sums and the division is done once per nonzero instead
// of once per lane: that arithmetic, not the memory, bounded k_phi_b.
// A block whose nonzeros share one output row adds into per-lane
// accumulators, which are summed over the lanes when the row changes;
// a mixed block is summed by a segmented scan over its runs of equal rows,
// and each run is flushed.
//
// PIM 1 / 2: the products pi are stored into / read from Pc, pair by pair in
// blocks of 64 nonzeros (pair p of block b: doubles [(b np + p) 128, + 128)),
// so that every access is 1 KB of consecutive memory per wavefront: the
// stored form is bound by HBM.  PIM 0 / 1 gather the factor rows with
// (R + 1) / 2 lanes per row, 16 bytes each, and turn the products of 64
// nonzeros around in LDS.
template <int P, int PW, int PIM>
__global__ void __launch_bounds__(256)
    k_phi_cols(StreamArgs<double, double, double> a, const double* __restrict__ B, double eps, double* __restrict__ Pc,
               uint64_t nblk, uint32_t per)
{
    constexpr int TS = 2 * P + 1;  // odd: the lanes' rows start in different banks
    __shared__ double s_tile[4 * 64 * TS];
    __shared__ uint32_t s_rows[4][64];
    const uint64_t block = xcd_block(a.nblocks_real);
    if (block == ~0ull) return;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    double* tile = s_tile + wave * 64 * TS;
    const uint64_t b0 = (block * 4 + wave) * per;
    if (b0 >= nblk) return;
    const uint64_t b1 = b0 + per < nblk ? b0 + per : nblk;
    constexpr int np = P;  // (R + 1) / 2
    const int R = a.rank;
    const bool odd = R & 1;
    // gather lanes: row `sub` of each step, column pair `gp`
    const int rps = 64 / np;  // rows per step
    const int sub = lane / np, gp = lane - sub * np;
    const bool gathers = sub < rps;
    const int gcb = min(2 * gp, R - 2);
    // flush lanes: run `fsub` of each step, column `fcol`
    const int fps = 64 / R, fsub = lane / R, fcol = lane - fsub * R;
    const int fat = fcol + (odd && fcol == R - 1 ? 1 : 0);  // the column's place among the pairs
    auto to_tile = [&](double (&x)[P][2], int r) {
#pragma unroll
        for (int p = 0; p < P; ++p)
            {
                tile[r * TS + 2 * p] = x[p][0];
                tile[r * TS + 2 * p + 1] = x[p][1];
            }
    };
    // out[row, :] += the sum of x over the wavefront's lanes
    auto flush_acc = [&](uint32_t row, const double (&x)[P][2]) {
        double mine = 0;  // lane c: column c
#pragma unroll
        for (int p = 0; p < P; ++p) {
            const int cb = min(2 * p, R - 2);
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                double t = x[p][q];
                t += dpp_f64<ROW_SHR1>(t);
                t += dpp_f64<ROW_SHR2>(t);
                t += dpp_f64<ROW_SHR4>(t);
                t += dpp_f64<ROW_SHR8>(t);
                t += dpp_f64<ROW_BCAST15, 0xa>(t);
                t += dpp_f64<ROW_BCAST31, 0xc>(t);
                t = lane63(t);
                mine = lane == cb + q ? t : mine;
            }
        }
        if (lane < R) atomic_add_hw(&a.out[(uint64_t)row * R + lane], mine);
    };

    double acc[P][2];
#pragma unroll
    for (int p = 0; p < P; ++p) acc[p][0] = acc[p][1] = 0;
    uint32_t cur = NO_ROW;  // the row acc belongs to (uniform)

    uint64_t kn[PW];
    double vn;
    {
        const uint64_t i = b0 * 64 + lane, ii = i < a.nnz ? i : a.nnz - 1;
#pragma unroll
        for (int w = 0; w < PW; ++w) kn[w] = a.pk[ii * PW + w];
        vn = a.val[ii];
    }
    for (uint64_t b = b0; b < b1; ++b) {
        // lanes past the end repeat the last nonzero and add nothing
        const bool valid = b * 64 + lane < a.nnz;
        uint64_t k[PW];
#pragma unroll
        for (int w = 0; w < PW; ++w) k[w] = kn[w];
        const double v = vn;
        const uint32_t row = (uint32_t)field<PW>(k, a.offn, a.bitsn);
        double pi[P][2];
        if constexpr (PIM == 2) {
            const double* src = Pc + b * np * 128 + 2 * lane;
#pragma unroll
            for (int p = 0; p < P; ++p)
                VecLoad<double, 2>::load(src + p * 128, pi[p]);
        }
        // the model row (runs of equal rows read the same lines)
        double bm[P][2];
        const double* br = B + (uint64_t)row * R;
#pragma unroll
        for (int p = 0; p < P; ++p)
            VecLoad<double, 2>::load(br + min(2 * p, R - 2), bm[p]);
        if (b + 1 < b1) {  // the next block's nonzeros
            const uint64_t i = (b + 1) * 64 + lane, ii = i < a.nnz ? i : a.nnz - 1;
#pragma unroll
            for (int w = 0; w < PW; ++w) kn[w] = a.pk[ii * PW + w];
            vn = a.val[ii];
        }
        if constexpr (PIM != 2) {
            uint32_t off[ALTO_MAXN - 1];
#pragma unroll
            for (int o = 0; o < ALTO_MAXN - 1; ++o)
                off[o] = o < a.nother ? (uint32_t)(field<PW>(k, a.offo[o], a.bitso[o]) * (uint64_t)R) : 0u;
            // GS steps' gathers are issued together (more at once only lower
            // the occupancy; five pairs: six steps in two goes)
            constexpr int GS = P == 5 ? 3 : 2;
#pragma unroll 1  // (unrolled, the loads of all steps would take too many registers)
            for (int r0 = 0; r0 < 64; r0 += GS * rps) {
                double x[GS][2];
                uint32_t f[GS][ALTO_MAXN - 1];
#pragma unroll
                for (int g = 0; g < GS; ++g)
#pragma unroll
                    for (int o = 0; o < ALTO_MAXN - 1; ++o)
                        f[g][o] = o < a.nother ? (uint32_t)__shfl((int)off[o], (r0 + g * rps + sub) & 63) : 0u;
                double y[ALTO_MAXN - 1][GS][2];
#pragma unroll
                for (int o = 0; o < ALTO_MAXN - 1; ++o)
                    if (o < a.nother) {  // uniform
#pragma unroll
                        for (int g = 0; g < GS; ++g) VecLoad<double, 2>::load(a.Uo[o] + f[g][o] + gcb, y[o][g]);
                    }
#pragma unroll
                for (int g = 0; g < GS; ++g) x[g][0] = x[g][1] = 1.0;
#pragma unroll
                for (int o = 0; o < ALTO_MAXN - 1; ++o)
                    if (o < a.nother) {
#pragma unroll
                        for (int g = 0; g < GS; ++g) {
                            x[g][0] *= y[o][g][0];
                            x[g][1] *= y[o][g][1];
                        }
                    }
#pragma unroll
                for (int g = 0; g < GS; ++g) {
                    const int r = r0 + g * rps + sub;
                    if (gathers && r < 64) {
                        tile[r * TS + 2 * gp] = x[g][0];
                        tile[r * TS + 2 * gp + 1] = x[g][1];
                    }
                }
            }
            // one wavefront's LDS accesses keep their order
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int p = 0; p < P; ++p)
                {
                    pi[p][0] = tile[lane * TS + 2 * p];
                    pi[p][1] = tile[lane * TS + 2 * p + 1];
                }
            __builtin_amdgcn_wave_barrier();
            if constexpr (PIM == 1) {
                double* dst = Pc + b * np * 128 + 2 * lane;
#pragma unroll
                for (int p = 0; p < P; ++p)
                    *reinterpret_cast<v2f64*>(dst + p * 128) = v2f64{pi[p][0], pi[p][1]};
            }
        }
        double d = 0;
#pragma unroll
        for (int p = 0; p < P; ++p)
            {
                const double x = bm[p][0] * pi[p][0];
                d += odd && p == np - 1 ? 0.0 : x;
                d += bm[p][1] * pi[p][1];
            }
        const double w = v / fmax(d, eps);
#pragma unroll
        for (int p = 0; p < P; ++p) {
            pi[p][0] = valid ? pi[p][0] * w : 0.0;
            pi[p][1] = valid ? pi[p][1] * w : 0.0;
        }
        const uint32_t row0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)row);
        if (__all(row == row0)) {
            if (row0 != cur) {
                if (cur != NO_ROW) flush_acc(cur, acc);
                cur = row0;
#pragma unroll
                for (int p = 0; p < P; ++p) acc[p][0] = acc[p][1] = 0;
            }
#pragma unroll
            for (int p = 0; p < P; ++p) {
                acc[p][0] += pi[p][0];
                acc[p][1] += pi[p][1];
            }
            continue;
        }
        if (cur != NO_ROW) {
            flush_acc(cur, acc);
            cur = NO_ROW;
        }
        const uint32_t before = (uint32_t)__shfl_up((int)row, 1);
        const uint64_t heads = __ballot(lane == 0 || before != row);
        const int start = 63 - __builtin_clzll(heads & ((2ull << lane) - 1));  // my run's first lane
        const int left = min(lane - start, lane & 15);  // run lanes to the left in this row of 16
#define SCAN_(C, ROWS, COND)                                \
    do {                                                    \
        double y[P][2];                                     \
        _Pragma("unroll") for (int p = 0; p < P; ++p)       \
        {                                                   \
            y[p][0] = dpp_f64<C, ROWS>(pi[p][0]);           \
            y[p][1] = dpp_f64<C, ROWS>(pi[p][1]);           \
        }                                                   \
        if (COND) {                                         \
            _Pragma("unroll") for (int p = 0; p < P; ++p)   \
            {                                               \
                pi[p][0] += y[p][0];                        \
                pi[p][1] += y[p][1];                        \
            }                                               \
        }                                                   \
    } while (0)
        SCAN_(ROW_SHR1, 0xf, left >= 1);
        SCAN_(ROW_SHR2, 0xf, left >= 2);
        SCAN_(ROW_SHR4, 0xf, left >= 4);
        SCAN_(ROW_SHR8, 0xf, left >= 8);
        SCAN_(ROW_BCAST15, 0xa, (lane & 16) && start < (lane & 48));
        SCAN_(ROW_BCAST31, 0xc, (lane & 32) && start < 32);
#undef SCAN_
        // the runs' sums are in their last lanes; they are flushed through LDS
        // with a run's columns in consecutive lanes, so that an atomic
        // instruction covers whole rows
        const int run = __popcll(heads & ((2ull << lane) - 1)) - 1, runs = __popcll(heads);
        if (lane == 63 || ((heads >> lane) >> 1) & 1) {
            s_rows[wave][run] = row;
            to_tile(pi, run);
        }
        __builtin_amdgcn_wave_barrier();
        for (int r0 = 0; r0 < runs; r0 += fps) {
            const int r = r0 + fsub;
            if (fsub < fps && r < runs)
                atomic_add_hw(&a.out[(uint64_t)s_rows[wave][r] * R + fcol], tile[r * TS + fat]);
        }
        __builtin_amdgcn_wave_barrier();
    }
    if (cur != NO_ROW) flush_acc(cur, acc);
}

}  // namespace

// 20M nonzeros, 4 modes, a mode's ten inner iterations per call: rank 5 465 ->
// 310 us, rank 10 633 -> 463, rank 12 662 -> 542, rank 16 730 -> 653, above
// rank 16 the columns no longer fit the registers (rank 24: 618 -> 770);
// without the products kept, rank 5 773 -> 598, rank 10 868 -> 830, rank 12
// 903 -> 1069.  3M nonzeros, rank 7: 107 -> 51 us; 3M nonzeros on 900,000 rows
// (three to a row), rank 10: 247 -> 146.
bool phi_cols_rank(int R, int pim) { return R >= 2 && R <= (pim ? 16 : 10); }

uint64_t phi_cols_cache(uint64_t nnz, int R) { return (nnz + 63) / 64 * 64 * (uint64_t)((R + 1) / 2 * 2); }

int launch_phi_cols(StreamArgs<double, double, double>& a, int pw, const double* B, double eps, double* pc, int pim,
                    hipStream_t s)
{
    const uint64_t nblk = (a.nnz + 63) / 64;
    // blocks per wavefront: a flush per wavefront against enough of them
    uint64_t per = nblk >> 14;
    per = per < 1 ? 1 : per > 32 ? 32 : per;
    const uint64_t blocks = (nblk + 4 * per - 1) / (4 * per);
    a.nblocks_real = blocks;
    const dim3 grid((unsigned)((blocks + 7) / 8 * 8));
#define PC_(P_, PW_, M_) \
    hipLaunchKernelGGL((k_phi_cols<P_, PW_, M_>), grid, dim3(256), 0, s, a, B, eps, pc, nblk, (uint32_t)per)
#define PCM_(P_, PW_)                 \
    do {                              \
        if (pim == 2) PC_(P_, PW_, 2); \
        else if (pim == 1) PC_(P_, PW_, 1); \
        else PC_(P_, PW_, 0);         \
    } while (0)
#define PCP_(P_)                      \
    do {                              \
        if (pw == 1) PCM_(P_, 1);     \
        else PCM_(P_, 2);             \
    } while (0)
    switch ((a.rank + 1) / 2) {
    case 1: PCP_(1); break;
    case 2: PCP_(2); break;
    case 3: PCP_(3); break;
    case 4: PCP_(4); break;
    case 5: PCP_(5); break;
    case 6: PCP_(6); break;
    case 7: PCP_(7); break;
    default: PCP_(8); break;
    }
#undef PCP_
#undef PCM_
#undef PC_
    HIP_TRY(hipGetLastError());
    return ALTO_OK;
}

}  // namespace alto
