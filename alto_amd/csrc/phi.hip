// CP-APR Phi over the per-mode nonzero streams (layout: mttkrp.hip).
//
// Reference semantics: CalculatePhi_alto_par (include/apr.hpp:295-303,
// :383-501).
#include "mttkrp_kernels.hpp"
#include "phi_cols.hpp"

namespace alto {

// Phi: per nonzero pi = prod_{m != n} U_m[row_m,:], d = <B[row,:], pi>,
// contribution (x / max(d, eps)) * pi.
template <int G, int E, int PW, int J>
__global__ void __launch_bounds__(256) k_phi(StreamArgs<double, double, double> a, const double* __restrict__ B, double eps)
{
    const int lane = threadIdx.x & 63;
    const int gl = lane & (G - 1);
    const uint64_t block = xcd_block(a.nblocks_real);
    if (block == ~0ull) return;
    const uint64_t group = (block * 256 + threadIdx.x) / G;
    const uint64_t s = group * a.seg;
    if (s >= a.nnz) return;
    const uint64_t e = s + a.seg < a.nnz ? s + a.seg : a.nnz;
    const int R = a.rank;
    const int nother = a.nother;

    double acc[E];
#pragma unroll
    for (int q = 0; q < E; ++q) acc[q] = 0;
    uint32_t cur = 0xffffffffu;
    for (uint64_t p = s; p < e; p += G) {
        uint32_t offs[ALTO_MAXN - 1];
        uint32_t rown = 0;
        double myv = 0;
        {
            uint64_t k[PW];
            if (p + gl < e) {
#pragma unroll
                for (int w = 0; w < PW; ++w) k[w] = a.pk[(p + gl) * PW + w];
                myv = a.val[p + gl];
            } else {
#pragma unroll
                for (int w = 0; w < PW; ++w) k[w] = 0;
            }
#pragma unroll
            for (int o = 0; o < ALTO_MAXN - 1; ++o)
                offs[o] = o < nother ? (uint32_t)(field<PW>(k, a.offo[o], a.bitso[o]) * (uint64_t)R) : 0u;
            rown = (uint32_t)field<PW>(k, a.offn, a.bitsn);
        }
        const int cnt = (int)(e - p < (uint64_t)G ? e - p : (uint64_t)G);
        for (int j0 = 0; j0 < cnt; j0 += J) {
            double pi[J][E], b[J][E], v[J];
            uint32_t rj[J];
#pragma unroll
            for (int jj = 0; jj < J; ++jj) {
                const int j = j0 + jj < cnt ? j0 + jj : cnt - 1;
                rj[jj] = (uint32_t)__shfl((int)rown, j, G);
                v[jj] = shfl_val(myv, j, G);
                load_cols<double, double, G, E>(B + (uint64_t)rj[jj] * R, gl, R, b[jj]);
#pragma unroll
                for (int q = 0; q < E; ++q) pi[jj][q] = 1.0;
            }
#pragma unroll
            for (int o = 0; o < ALTO_MAXN - 1; ++o) {
                if (o < nother) {
                    const double* __restrict__ U = a.Uo[o];
#pragma unroll
                    for (int jj = 0; jj < J; ++jj) {
                        const int j = j0 + jj < cnt ? j0 + jj : cnt - 1;
                        const uint32_t off = (uint32_t)__shfl((int)offs[o], j, G);
                        double x[E];
                        load_cols<double, double, G, E>(U + off, gl, R, x);
#pragma unroll
                        for (int q = 0; q < E; ++q) pi[jj][q] *= x[q];
                    }
                }
            }
#pragma unroll
            for (int jj = 0; jj < J; ++jj) {
                double d = 0;
#pragma unroll
                for (int q = 0; q < E; ++q) d += b[jj][q] * pi[jj][q];
                d = group_sum<G>(d);
                const double w = v[jj] / fmax(d, eps);
                if (j0 + jj < cnt) {
                    if (rj[jj] != cur) {
                        if (cur != 0xffffffffu) flush_row<double, double, G, E>(a.out, cur, R, gl, acc);
                        cur = rj[jj];
#pragma unroll
                        for (int q = 0; q < E; ++q) acc[q] = 0;
                    }
#pragma unroll
                    for (int q = 0; q < E; ++q) acc[q] += w * pi[jj][q];
                }
            }
        }
    }
    if (cur != 0xffffffffu) flush_row<double, double, G, E>(a.out, cur, R, gl, acc);
}

// The same sum with the batch loop unrolled at compile time: each lane
// decodes one nonzero of a batch of G, and the group takes each nonzero's
// row offsets and value from the decoding lane through DPP / readlane
// broadcasts (no LDS permutes); the NO other modes' gathers of J = 4
// nonzeros are issued back to back, and the next batch is loaded behind the
// first gathers.  Lanes still read strided 8-byte columns (16-byte lanes
// raise the register count past the point where occupancy pays for them;
// holding this kernel to 128 VGPRs for a fourth wave per SIMD measured
// slower too).
// PIM: the products pi of the other modes' rows are computed from the
// factors (0), computed and stored per nonzero into Pc in stream order (1),
// or read back from Pc (2): within CP-APR's inner iterations of one mode the
// other factors do not change, so the later iterations stream pi instead of
// gathering NO rows per nonzero (the reference's precomputed rows,
// include/apr.hpp:1049-1097 and 1128-1165).
template <int G, int E, int PW, int NO, int PIM>
__global__ void __launch_bounds__(256)
    k_phi_b(StreamArgs<double, double, double> a, const double* __restrict__ B, double eps, double* __restrict__ Pc)
{
    constexpr int J = G < 4 ? G : 4;
    const int lane = threadIdx.x & 63;
    const int gl = lane & (G - 1);
    const uint64_t block = xcd_block(a.nblocks_real);
    if (block == ~0ull) return;
    const uint64_t group = (block * 256 + threadIdx.x) / G;
    const uint64_t s = group * a.seg;
    if (s >= a.nnz) return;
    const uint64_t e = s + a.seg < a.nnz ? s + a.seg : a.nnz;
    const int R = a.rank;

    double acc[E], b_last[E];
#pragma unroll
    for (int q = 0; q < E; ++q) acc[q] = b_last[q] = 0;
    uint32_t cur = 0xffffffffu;
    uint32_t b_row = 0xffffffffu;  // the model row b_last holds (this group's)
    // this lane's nonzero of the next batch (past the segment: row 0 of
    // every mode, value 0 -- valid memory, never accumulated)
    uint64_t kn[PW];
    double vn = 0;
#pragma unroll
    for (int w = 0; w < PW; ++w) kn[w] = 0;
    if (s + gl < e) {
#pragma unroll
        for (int w = 0; w < PW; ++w) kn[w] = a.pk[(s + gl) * PW + w];
        vn = a.val[s + gl];
    }
    for (uint64_t p = s; p < e; p += G) {
        uint32_t offs[NO];
#pragma unroll
        for (int o = 0; o < NO; ++o) offs[o] = (uint32_t)(field<PW>(kn, a.offo[o], a.bitso[o]) * (uint64_t)R);
        const uint32_t rown = (uint32_t)field<PW>(kn, a.offn, a.bitsn);
        const double myv = vn;
        const int cnt = (int)(e - p < (uint64_t)G ? e - p : (uint64_t)G);
        static_for<0, G / J>([&](auto bi) {
            constexpr int j0 = decltype(bi)::value * J;
            if (j0 >= cnt) return;
            double pi[J][E], b[J][E], v[J];
            uint32_t rj[J];
            static_for<0, J>([&](auto ji) {
                constexpr int jj = decltype(ji)::value;
                rj[jj] = bcast32<G, j0 + jj>(rown);
                v[jj] = bcast_val<G, j0 + jj>(myv);
#pragma unroll
                for (int q = 0; q < E; ++q) pi[jj][q] = 1.0;
            });
            // the model row only at the positions where some group's row
            // changes: a wave-uniform branch, so every lane loads (groups
            // whose row did not change reload the row they hold), and the
            // stream's runs of one row skip the load
            double rb[J][E];
            uint32_t ldm = 0;  // positions loaded (uniform)
#pragma unroll
            for (int jj = 0; jj < J; ++jj) {
                const bool head = jj == 0 ? rj[0] != b_row : rj[jj] != rj[jj - 1];
                if (__any(head)) {
                    load_cols<double, double, G, E>(B + (uint64_t)rj[jj] * R, gl, R, rb[jj]);
                    ldm |= 1u << jj;
                }
            }
            // the mask reaches the selection below through an opaque copy, so
            // that the selection is not folded into the branches above
            asm volatile("" : "+s"(ldm));
            if constexpr (PIM == 2) {
#pragma unroll
                for (int jj = 0; jj < J; ++jj) {
                    const uint64_t i = p + j0 + jj < e ? p + j0 + jj : e - 1;
#pragma unroll
                    for (int q = 0; q < E; ++q) {
                        const int c = gl + q * G;
                        pi[jj][q] = c < R ? Pc[i * R + c] : 0.0;
                    }
                }
            } else {
                static_for<0, NO>([&](auto oi) {
                    constexpr int o = decltype(oi)::value;
                    const double* __restrict__ U = a.Uo[o];
                    static_for<0, J>([&](auto ji) {
                        constexpr int jj = decltype(ji)::value;
                        const uint32_t off = bcast32<G, j0 + jj>(offs[o]);
                        double x[E];
                        load_cols<double, double, G, E>(U + off, gl, R, x);
#pragma unroll
                        for (int q = 0; q < E; ++q) pi[jj][q] *= x[q];
                    });
                });
            }
            if constexpr (PIM == 1) {
#pragma unroll
                for (int jj = 0; jj < J; ++jj)
                    if (j0 + jj < cnt)
#pragma unroll
                        for (int q = 0; q < E; ++q) {
                            const int c = gl + q * G;
                            if (c < R) Pc[(p + j0 + jj) * R + c] = pi[jj][q];
                        }
            }
            if constexpr (j0 == 0) {
                const uint64_t i = p + G + gl;
                vn = 0;
#pragma unroll
                for (int w = 0; w < PW; ++w) kn[w] = 0;
                if (i < e) {
#pragma unroll
                    for (int w = 0; w < PW; ++w) kn[w] = a.pk[i * PW + w];
                    vn = a.val[i];
                }
            }
            // each position's model row is that of the last load at or before it
#pragma unroll
            for (int jj = 0; jj < J; ++jj) {
                const bool use = (ldm >> jj) & 1u;
#pragma unroll
                for (int q = 0; q < E; ++q) {
                    b_last[q] = use ? rb[jj][q] : b_last[q];
                    b[jj][q] = b_last[q];
                }
            }
            b_row = rj[J - 1];
#pragma unroll
            for (int jj = 0; jj < J; ++jj) {
                double d = 0;
#pragma unroll
                for (int q = 0; q < E; ++q) d += b[jj][q] * pi[jj][q];
                d = group_sum<G>(d);
                const double w = v[jj] / fmax(d, eps);
                if (j0 + jj < cnt) {
                    if (rj[jj] != cur) {
                        if (cur != 0xffffffffu) flush_row<double, double, G, E>(a.out, cur, R, gl, acc);
                        cur = rj[jj];
#pragma unroll
                        for (int q = 0; q < E; ++q) acc[q] = 0;
                    }
#pragma unroll
                    for (int q = 0; q < E; ++q) acc[q] += w * pi[jj][q];
                }
            }
        });
    }
    if (cur != 0xffffffffu) flush_row<double, double, G, E>(a.out, cur, R, gl, acc);
}

// Phi with 16-byte lanes (the k_mttkrp16 lane mapping): lane gl of a group
// of G holds columns 2 gl and 2 gl + 1, so every factor row (the model row
// B[row] and the NO other modes' rows) arrives with one 16-byte load per
// lane, half the gather instructions of the strided 8-byte lanes.  Needs an
// even rank and 16-byte aligned factors (rows of 16 R / 2 bytes).  Per
// nonzero: Pi = the product of the other rows, d = <B[row], Pi> summed over
// the group, and Pi x / max(d, eps) added into the row's run.  The model
// row is loaded only where the row changes inside a block of J nonzeros or
// from the previous block, with the decision uniform over the wave (the
// stream is ordered by row inside each chunk, so long runs skip most
// model-row loads).  PIM as in k_phi_b: 0 gather the other rows, 1 gather
// and store their products per nonzero into Pc, 2 read the products back
// (one 16-byte load per lane instead of NO).
template <int G, int PW, int NO, int PIM>
__global__ void __launch_bounds__(256)
    k_phi16(StreamArgs<double, double, double> a, const double* __restrict__ Bm, double eps, double* __restrict__ Pc)
{
    constexpr int E = 2;
    constexpr int NS = G < 4 ? 4 / G : 1;
    constexpr int BB = G * NS;
    constexpr int J = 4;
    const uint64_t block = xcd_block(a.nblocks_real);
    if (block == ~0ull) return;
    const int lane = threadIdx.x & 63;
    const int gl = lane & (G - 1);
    const uint64_t group = (block * 256 + threadIdx.x) / G;
    const uint64_t s = group * a.seg;
    if (s >= a.nnz) return;
    const uint64_t e = s + a.seg < a.nnz ? s + a.seg : a.nnz;
    const int R = a.rank;
    const int c0 = gl * E < R ? gl * E : 0;
    const bool inr = gl * E < R;

    double acc[E], blast[E];
#pragma unroll
    for (int q = 0; q < E; ++q) acc[q] = blast[q] = 0;
    uint32_t cur = 0xffffffffu;
    uint32_t prev_r = 0xffffffffu;  // row whose model row blast holds

    uint64_t kn[NS][PW];
    double vn[NS];
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        const uint64_t i = s + k * G + gl;
        vn[k] = 0;
#pragma unroll
        for (int w = 0; w < PW; ++w) kn[k][w] = 0;
        if (i < e) {
#pragma unroll
            for (int w = 0; w < PW; ++w) kn[k][w] = a.pk[i * PW + w];
            vn[k] = a.val[i];
        }
    }
    for (uint64_t p = s; p < e; p += BB) {
        uint32_t offs[NS][NO];
        uint32_t rown[NS];
        double myv[NS];
#pragma unroll
        for (int k = 0; k < NS; ++k) {
            myv[k] = vn[k];
#pragma unroll
            for (int o = 0; o < NO; ++o) offs[k][o] = (uint32_t)(field<PW>(kn[k], a.offo[o], a.bitso[o]) * (uint64_t)R);
            rown[k] = (uint32_t)field<PW>(kn[k], a.offn, a.bitsn);
        }
        const int cnt = (int)(e - p < (uint64_t)BB ? e - p : (uint64_t)BB);
        static_for<0, BB / J>([&](auto bi) {
            constexpr int j0 = decltype(bi)::value * J;
            if (j0 >= cnt) return;
            double pi[J][E], v[J];
            uint32_t rj[J];
            static_for<0, J>([&](auto ji) {
                constexpr int jj = decltype(ji)::value;
                constexpr int slot = (j0 + jj) / G, src = (j0 + jj) % G;
                rj[jj] = bcast32<G, src>(rown[slot]);
                v[jj] = bcast_val<G, src>(myv[slot]);
#pragma unroll
                for (int q = 0; q < E; ++q) pi[jj][q] = 1.0;
            });
            if constexpr (PIM == 2) {
                // lanes past the rank read the row's first pair (never used)
#pragma unroll
                for (int jj = 0; jj < J; ++jj) {
                    const uint64_t i = p + j0 + jj < e ? p + j0 + jj : e - 1;
                    VecLoad<double, E>::load(Pc + i * R + c0, pi[jj]);
                }
            } else {
                static_for<0, NO>([&](auto oi) {
                    constexpr int o = decltype(oi)::value;
                    const double* __restrict__ U = a.Uo[o];
                    static_for<0, J>([&](auto ji) {
                        constexpr int jj = decltype(ji)::value;
                        constexpr int slot = (j0 + jj) / G, src = (j0 + jj) % G;
                        const uint32_t off = bcast32<G, src>(offs[slot][o]);
                        double x[E];
                        VecLoad<double, E>::load(U + off + c0, x);
#pragma unroll
                        for (int q = 0; q < E; ++q) pi[jj][q] *= x[q];
                    });
                });
            }
            if constexpr (PIM == 1) {
#pragma unroll
                for (int jj = 0; jj < J; ++jj)
                    if (inr && j0 + jj < cnt)
                        *reinterpret_cast<v2f64*>(Pc + (p + j0 + jj) * R + c0) = v2f64{pi[jj][0], pi[jj][1]};
            }
            // model rows where the row changes (uniform over the wave)
            double br[J][E];
            uint32_t ldm = 0;
#pragma unroll
            for (int jj = 0; jj < J; ++jj) {
                const bool chg = jj == 0 ? rj[0] != prev_r : rj[jj] != rj[jj - 1];
                if (__any(chg)) {
                    VecLoad<double, E>::load(Bm + (uint64_t)rj[jj] * R + c0, br[jj]);
                    ldm |= 1u << jj;
                }
            }
            // the mask reaches the selection below through an opaque copy, so
            // that the selection is not folded into the branches above
            asm volatile("" : "+s"(ldm));
            if constexpr (j0 == 0) {
#pragma unroll
                for (int k = 0; k < NS; ++k) {
                    const uint64_t i = p + BB + k * G + gl;
                    vn[k] = 0;
#pragma unroll
                    for (int w = 0; w < PW; ++w) kn[k][w] = 0;
                    if (i < e) {
#pragma unroll
                        for (int w = 0; w < PW; ++w) kn[k][w] = a.pk[i * PW + w];
                        vn[k] = a.val[i];
                    }
                }
            }
#pragma unroll
            for (int jj = 0; jj < J; ++jj) {
                const bool use = (ldm >> jj) & 1u;
                double d = 0;
#pragma unroll
                for (int q = 0; q < E; ++q) {
                    blast[q] = use ? br[jj][q] : blast[q];
                    d += (inr ? blast[q] : 0.0) * pi[jj][q];
                }
                d = group_sum<G>(d);
                const double w = v[jj] / fmax(d, eps);
                if (j0 + jj < cnt) {
                    if (rj[jj] != cur) {
                        if (cur != 0xffffffffu) flush_row<double, double, G, E, true>(a.out, cur, R, gl, acc);
                        cur = rj[jj];
#pragma unroll
                        for (int q = 0; q < E; ++q) acc[q] = 0;
                    }
#pragma unroll
                    for (int q = 0; q < E; ++q) acc[q] += w * pi[jj][q];
                }
            }
            prev_r = rj[J - 1];
        });
    }
    if (cur != 0xffffffffu) flush_row<double, double, G, E, true>(a.out, cur, R, gl, acc);
}

// ------------------------------------------------------------------ host side
// doubles of a product cache that fits whichever kernel `variant` picks
uint64_t phi_cache_doubles(uint64_t nnz, int R, int variant)
{
    return variant == 1 && phi_cols_rank(R, 1) ? phi_cols_cache(nnz, R) : nnz * (uint64_t)R;
}

int phi_device(alto_tensor* t, int mode, int R, const double* const* U, double* phi, double eps, hipStream_t s, int seg)
{
    return phi_device_cached(t, mode, R, U, phi, eps, s, seg, nullptr, 0, phi_variant());
}

// pim: 0 = no cache; 1 = store the products of the other modes' rows per
// nonzero into pc (phi_cache_doubles of them); 2 = read them from pc (stored
// by a pim 1 call for the same mode, factors and variant)
int phi_device_cached(alto_tensor* t, int mode, int R, const double* const* U, double* phi, double eps, hipStream_t s,
                      int seg, double* pc, int pim, int variant)
{
    if (mode < 0 || mode >= t->nmode || R < 1 || R > 128) {
        set_error("phi: mode %d / rank %d out of range (rank 1..128)", mode, R);
        return ALTO_ERR_ARG;
    }
    ALTO_TRY(check_offsets(t, R));
    ALTO_TRY(prepare_mode_streams(t, 1, 0, s));
    if (seg <= 0) seg = tuned_seg(t->nnz, group_lanes(R), 8);
    ALTO_TRY(fill_zero(phi, t->dims[mode] * (uint64_t)R, s));
    ALTO_TRY(reserve_rank_copies(t, (uint64_t)R, 8, s));
    if (det_enabled()) return phi_det_device(t, mode, R, U, phi, eps, s);
    StreamArgs<double, double, double> a;
    fill_stream_args(t, mode, R, seg, a);
    ALTO_TRY(set_factors(t, mode, U, a, s));
    a.val = t->ms[mode].val64.as<double>();
    a.out = phi;
    if (variant == 1 && phi_cols_rank(R, pim)) return launch_phi_cols(a, t->pack.pw, U[mode], eps, pc, pim, s);
    dim3 grid = stream_grid(t->nnz, seg, group_lanes(R), a);
    bool al16 = R % 2 == 0 && ((uintptr_t)U[mode] & 15) == 0;
    for (int o = 0; o < a.nother; ++o) al16 = al16 && ((uintptr_t)a.Uo[o] & 15) == 0;
    if (variant == 2 && al16 && (!pim || ((uintptr_t)pc & 15) == 0)) {
        const int no = t->nmode - 1;
#define PHI16_P_(N_, P_) hipLaunchKernelGGL((k_phi16<G, PW, N_, P_>), grid, dim3(256), 0, s, a, U[mode], eps, pc)
#define PHI16_NO_(N_)                      \
    do {                                   \
        if (pim == 1) PHI16_P_(N_, 1);     \
        else if (pim == 2) PHI16_P_(N_, 2); \
        else PHI16_P_(N_, 0);              \
    } while (0)
        RANK_DISPATCH(R, t->pack.pw, {
            if (no == 1) PHI16_NO_(1);
            else if (no == 2) PHI16_NO_(2);
            else if (no == 3) PHI16_NO_(3);
            else PHI16_NO_(4);
        });
#undef PHI16_NO_
#undef PHI16_P_
    } else if (variant >= 1 || pim) {
        const int no = t->nmode - 1;
#define PHI_NO_(N_)                                                                                              \
    do {                                                                                                         \
        if (pim == 1) hipLaunchKernelGGL((k_phi_b<G, E, PW, N_, 1>), grid, dim3(256), 0, s, a, U[mode], eps, pc); \
        else if (pim == 2)                                                                                       \
            hipLaunchKernelGGL((k_phi_b<G, E, PW, N_, 2>), grid, dim3(256), 0, s, a, U[mode], eps, pc);          \
        else hipLaunchKernelGGL((k_phi_b<G, E, PW, N_, 0>), grid, dim3(256), 0, s, a, U[mode], eps, pc);          \
    } while (0)
        RANK_DISPATCH(R, t->pack.pw, {
            if (no == 1) PHI_NO_(1);
            else if (no == 2) PHI_NO_(2);
            else if (no == 3) PHI_NO_(3);
            else PHI_NO_(4);
        });
#undef PHI_NO_
    } else {
        RANK_DISPATCH(R, t->pack.pw,
                      { hipLaunchKernelGGL((k_phi<G, E, PW, 4>), grid, dim3(256), 0, s, a, U[mode], eps); });
    }
    HIP_TRY(hipGetLastError());
    return ALTO_OK;
}

}  // namespace alto

using namespace alto;

extern "C" {

int alto_phi(alto_tensor_t* t, int mode, uint64_t rank, const double* const* factors, double* phi, double eps_div_zero,
             alto_stream_t stream)
{
    if (!t || !factors || !phi) {
        set_error("alto_phi: null argument");
        return ALTO_ERR_ARG;
    }
    ALTO_TRY(phi_device(t, mode, (int)rank, factors, phi, eps_div_zero, (hipStream_t)stream, 0));
    return t->note_use((hipStream_t)stream);
}

}  // extern "C"
