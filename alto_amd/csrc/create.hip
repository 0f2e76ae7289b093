// ALTO format construction on gfx950: linearization (bit deposit) and
// delinearization (bit extract) as byte-LUT bit permutations, the sort by key
// (sort.hip), line-balanced partition pointers, partition intervals,
// conflict-resolution (CR) bits, and the per-mode chunk-ordered nonzero streams
// consumed by MTTKRP / Phi.
//
// Reference behaviour followed: create_alto (include/alto.hpp:108-294),
// setup_packed_alto (:669-770), sort_alto (:772-803), prtn_alto (:805-1028).
#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <map>
#include <memory>
#include <mutex>

#include "alto_internal.hpp"
#include "kernels_common.hpp"
#include "sort.hpp"

namespace alto {

// ------------------------------------------------------------------ errors
static thread_local std::string g_err;

void set_error(const char* fmt, ...)
{
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    g_err = buf;
}

void set_error_hip(hipError_t e, const char* what)
{
    set_error("%s failed: %s", what, hipGetErrorString(e));
}

const char* last_error() { return g_err.c_str(); }

// Caching device allocator: freed blocks are kept per device in power-of-two
// size classes and reused, so concurrent jobs never call hipFree (which
// synchronizes the device) on their hot path.  alto_device_trim returns the
// cache to the runtime.
namespace {
struct Pool {
    std::mutex mu;
    std::multimap<size_t, void*> free_blocks[64];  // per device: class bytes -> ptr
    size_t cached[64] = {0};
    size_t in_use[64] = {0};
};
Pool& pool()
{
    static Pool* p = new Pool();
    return *p;
}
size_t size_class(size_t n)
{
    if (n <= 256) return 256;
    size_t c = 256;
    while (c < n) c <<= 1;
    return c;
}
}  // namespace

int DevBuf::alloc(size_t n)
{
    release();
    if (n == 0) n = 8;
    int dev = 0;
    HIP_TRY(hipGetDevice(&dev));
    const size_t cls = size_class(n);
    Pool& P = pool();
    {
        std::lock_guard<std::mutex> g(P.mu);
        auto& fb = P.free_blocks[dev & 63];
        auto it = fb.find(cls);
        if (it != fb.end()) {
            p = it->second;
            fb.erase(it);
            P.cached[dev & 63] -= cls;
            P.in_use[dev & 63] += cls;
            bytes = n;
            cap = cls;
            device = dev;
            return ALTO_OK;
        }
    }
    hipError_t e = hipMalloc(&p, cls);
    if (e == hipErrorOutOfMemory) {  // give the cache back and retry once
        (void)hipGetLastError();
        alto_device_trim();
        e = hipMalloc(&p, cls);
    }
    if (e != hipSuccess) {
        p = nullptr;
        set_error("hipMalloc(%zu bytes) failed: %s", cls, hipGetErrorString(e));
        (void)hipGetLastError();
        return e == hipErrorOutOfMemory ? ALTO_ERR_OOM : ALTO_ERR_HIP;
    }
    {
        std::lock_guard<std::mutex> g(P.mu);
        P.in_use[dev & 63] += cls;
    }
    bytes = n;
    cap = cls;
    device = dev;
    return ALTO_OK;
}

void DevBuf::release()
{
    if (p) {
        Pool& P = pool();
        std::lock_guard<std::mutex> g(P.mu);
        P.free_blocks[device & 63].emplace(cap, p);
        P.cached[device & 63] += cap;
        P.in_use[device & 63] -= cap;
    }
    p = nullptr;
    bytes = 0;
    cap = 0;
}

size_t pool_in_use(int dev)
{
    Pool& P = pool();
    std::lock_guard<std::mutex> g(P.mu);
    return P.in_use[dev & 63];
}

}  // namespace alto

int alto_tensor::note_use(hipStream_t s)
{
    std::lock_guard<std::mutex> g(use_mu);
    hipEvent_t e = nullptr;
    for (auto& u : uses)
        if (u.first == s) e = u.second;
    if (!e) {
        HIP_TRY(hipEventCreateWithFlags(&e, hipEventDisableTiming));
        uses.emplace_back(s, e);
    }
    HIP_TRY(hipEventRecord(e, s));
    return ALTO_OK;
}

int alto_tensor::wait_uses()
{
    std::lock_guard<std::mutex> g(use_mu);
    for (auto& u : uses) HIP_TRY(hipEventSynchronize(u.second));
    return ALTO_OK;
}

alto_tensor::~alto_tensor()
{
    for (auto& u : uses) {
        (void)hipEventSynchronize(u.second);
        (void)hipEventDestroy(u.second);
    }
}

namespace alto {

// ------------------------------------------------------------------ masks
// setup_packed_alto(at, LSB_FIRST, SHORT_FIRST): modes ordered by bit count
// (stable), one bit per still-active mode per level, LSB first.
int compute_masks(int nmode, const uint64_t* dims, int W, uint64_t* masks, uint64_t* alto_mask)
{
    int mode[ALTO_MAXN], bits[ALTO_MAXN], total = 0, maxb = 0;
    for (int n = 0; n < nmode; ++n) {
        uint64_t d = dims[n] - 1;
        mode[n] = n;
        bits[n] = d ? 64 - __builtin_clzll(d) : 0;
        total += bits[n];
        maxb = std::max(maxb, bits[n]);
    }
    if (total > 64 * W) return -1;
    std::stable_sort(mode, mode + nmode, [&](int a, int b) { return bits[a] < bits[b]; });
    memset(masks, 0, sizeof(uint64_t) * nmode * W);
    int shift = 0;
    for (int level = 0; level < maxb; ++level)
        for (int k = 0; k < nmode; ++k)
            if (level < bits[mode[k]]) {
                masks[mode[k] * W + (shift >> 6)] |= 1ull << (shift & 63);
                ++shift;
            }
    for (int w = 0; w < W; ++w) {
        alto_mask[w] = 0;
        for (int n = 0; n < nmode; ++n) alto_mask[w] |= masks[n * W + w];
    }
    return total;
}

// Packed layout: mode n at bit offset sum_{m<n} bits[m].  The key->packed
// map is a bit permutation: the j-th set bit of mask_n goes to off[n]+j.
int build_luts(alto_tensor* t, hipStream_t s)
{
    PackLayout& L = t->pack;
    L.nmode = t->nmode;
    int off = 0;
    int keypos_of[128];   // packed bit -> key bit
    for (int n = 0; n < t->nmode; ++n) {
        L.off[n] = off;
        int j = 0;
        for (int q = 0; q < 64 * t->W; ++q)
            if ((t->masks[n * t->W + (q >> 6)] >> (q & 63)) & 1) keypos_of[off + j++] = q;
        L.bits[n] = j;
        off += j;
    }
    L.pw = off > 64 ? 2 : 1;
    int packpos_of[128];
    for (int q = 0; q < 128; ++q) packpos_of[q] = -1;
    for (int p = 0; p < off; ++p) packpos_of[keypos_of[p]] = p;

    const int nbits = off;
    auto fill = [nbits, s](BitPermLut& lut, int in_w, int out_w, const int* map /* in bit -> out bit or -1 */) -> int {
        lut.in_words = in_w;
        lut.out_words = out_w;
        lut.nb = std::min(in_w * 8, (nbits + 7) / 8);
        lut.host.assign((size_t)in_w * 8 * 256 * out_w, 0);
        for (int b = 0; b < in_w * 8; ++b)
            for (int v = 0; v < 256; ++v) {
                uint64_t* e = &lut.host[((size_t)b * 256 + v) * out_w];
                for (int i = 0; i < 8; ++i) {
                    if (!((v >> i) & 1)) continue;
                    int o = map[b * 8 + i];
                    if (o >= 0) e[o >> 6] |= 1ull << (o & 63);
                }
            }
        ALTO_TRY(lut.dev.alloc(lut.host.size() * 8));
        // (the table stays in `host`; the caller waits)
        HIP_TRY(hipMemcpyAsync(lut.dev.p, lut.host.data(), lut.host.size() * 8, hipMemcpyHostToDevice, s));
        return ALTO_OK;
    };
    int map_delin[128], map_lin[128];
    for (int q = 0; q < 128; ++q) map_delin[q] = q < 64 * t->W ? packpos_of[q] : -1;
    for (int p = 0; p < 128; ++p) map_lin[p] = p < off ? keypos_of[p] : -1;
    ALTO_TRY(fill(t->delin, t->W, L.pw, map_delin));
    ALTO_TRY(fill(t->lin, L.pw, t->W, map_lin));
    return ALTO_OK;
}

// ------------------------------------------------------------------ kernels
// Byte-LUT bit permutation: out = OR_b lut[b][byte_b(in)], b < nb (the bytes
// that can carry index bits).  The table is staged in LDS when it fits.
template <int IW, int OW>
__device__ inline void lut_apply(const uint64_t* __restrict__ lut, int nb, const uint64_t (&in)[IW], uint64_t (&out)[OW])
{
#pragma unroll
    for (int w = 0; w < OW; ++w) out[w] = 0;
#pragma unroll
    for (int b = 0; b < IW * 8; ++b) {
        if (b < nb) {
            unsigned v = (unsigned)(in[b >> 3] >> ((b & 7) * 8)) & 0xffu;
            const uint64_t* e = lut + ((size_t)b * 256 + v) * OW;
#pragma unroll
            for (int w = 0; w < OW; ++w) out[w] |= e[w];
        }
    }
}

struct LutRef {
    const uint64_t* g;  // device table
    int nb;             // input bytes covered
    int lds;            // staged in LDS?
};

template <int OW>
__device__ inline const uint64_t* stage_lut(uint64_t* s_lut, LutRef L)
{
    if (!L.lds) return L.g;
    const int n = L.nb * 256 * OW;
    for (int i = threadIdx.x; i < n; i += blockDim.x) s_lut[i] = L.g[i];
    __syncthreads();
    return s_lut;
}

struct CoordPtrs {
    const uint64_t* c[ALTO_MAXN];
};

struct DimArr {
    uint64_t d[ALTO_MAXN];
};

// linearize (include/alto.hpp:184-204): pack the coordinates, then permute
// the packed bits into ALTO key order.  Coordinates must lie inside dims (the
// reference asserts it in CreateSparseTensor, src/sptensor.cpp:276-281); a
// violation sets *bad.
template <int PW, int W>
__global__ void __launch_bounds__(256) k_linearize(CoordPtrs cp, int nmode, DimArr dims, PackLayout L, LutRef g_lut,
                                                   uint64_t n, uint64_t* __restrict__ keys, int* __restrict__ bad)
{
    extern __shared__ uint64_t s_lut[];
    const uint64_t* lut = stage_lut<W>(s_lut, g_lut);
    int out = 0;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        uint64_t pk[PW];
#pragma unroll
        for (int w = 0; w < PW; ++w) pk[w] = 0;
        for (int m = 0; m < nmode; ++m) {
            uint64_t c = cp.c[m][i];
            out |= c >= dims.d[m];
            int o = L.off[m];
            if (PW == 1) {
                pk[0] |= c << o;
            } else {
                if (o < 64) {
                    pk[0] |= c << o;
                    if (o > 0) pk[PW - 1] |= c >> (64 - o);
                } else {
                    pk[PW - 1] |= c << (o - 64);
                }
            }
        }
        uint64_t k[W];
        lut_apply<PW, W>(lut, g_lut.nb, pk, k);
#pragma unroll
        for (int w = 0; w < W; ++w) keys[i * W + w] = k[w];
    }
    if (out) atomicOr(bad, 1);
}

// generic bit permutation of an array of keys (pdep / pext of all modes)
template <int IW, int OW>
__global__ void __launch_bounds__(256) k_bitperm(const uint64_t* __restrict__ in, LutRef g_lut,
                                                 uint64_t n, uint64_t* __restrict__ out)
{
    extern __shared__ uint64_t s_lut[];
    const uint64_t* lut = stage_lut<OW>(s_lut, g_lut);
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        uint64_t a[IW], b[OW];
#pragma unroll
        for (int w = 0; w < IW; ++w) a[w] = in[i * IW + w];
        lut_apply<IW, OW>(lut, g_lut.nb, a, b);
#pragma unroll
        for (int w = 0; w < OW; ++w) out[i * OW + w] = b[w];
    }
}

// delinearize all modes: keys -> coordinates (nmode x n)
template <int W, int PW>
__global__ void __launch_bounds__(256) k_delin_coords(const uint64_t* __restrict__ keys, LutRef g_lut,
                                                      PackLayout L, uint64_t n, uint64_t* __restrict__ coords)
{
    extern __shared__ uint64_t s_lut[];
    const uint64_t* lut = stage_lut<PW>(s_lut, g_lut);
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        uint64_t k[W], pk[PW];
#pragma unroll
        for (int w = 0; w < W; ++w) k[w] = keys[i * W + w];
        lut_apply<W, PW>(lut, g_lut.nb, k, pk);
        for (int m = 0; m < L.nmode; ++m) coords[(uint64_t)m * n + i] = field<PW>(pk, L.off[m], L.bits[m]);
    }
}

// packed coords -> coordinates (used by alto_pdep_keys inputs is the reverse)
template <int PW, int W>
__global__ void __launch_bounds__(256) k_pack_lin(const uint64_t* __restrict__ coords, PackLayout L, LutRef g_lut,
                                                  uint64_t n, uint64_t* __restrict__ keys)
{
    extern __shared__ uint64_t s_lut[];
    const uint64_t* lut = stage_lut<W>(s_lut, g_lut);
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        uint64_t pk[PW];
#pragma unroll
        for (int w = 0; w < PW; ++w) pk[w] = 0;
        for (int m = 0; m < L.nmode; ++m) {
            uint64_t c = coords[(uint64_t)m * n + i];
            int o = L.off[m];
            if (PW == 1) pk[0] |= c << o;
            else if (o < 64) {
                pk[0] |= c << o;
                if (o > 0) pk[PW - 1] |= c >> (64 - o);
            } else pk[PW - 1] |= c << (o - 64);
        }
        uint64_t k[W];
        lut_apply<PW, W>(lut, g_lut.nb, pk, k);
#pragma unroll
        for (int w = 0; w < W; ++w) keys[i * W + w] = k[w];
    }
}

static int grid_for(uint64_t n, int threads = 256, int max_blocks = 4096)
{
    uint64_t b = (n + threads - 1) / threads;
    if (b < 1) b = 1;
    if (b > (uint64_t)max_blocks) b = max_blocks;
    return (int)b;
}

static LutRef lutref(const BitPermLut& L)
{
    LutRef r;
    r.g = L.dev.as<uint64_t>();
    r.nb = L.nb;
    r.lds = (size_t)L.nb * 256 * L.out_words * 8 <= 48 * 1024;
    return r;
}
static size_t lut_smem(const BitPermLut& L)
{
    size_t b = (size_t)L.nb * 256 * L.out_words * 8;
    return b <= 48 * 1024 ? b : 0;
}

// ------------------------------------------------------------------ post-sort
// values in ALTO order, cast to ValType
__global__ void k_gather_vals(const double* __restrict__ in, const uint32_t* __restrict__ perm, uint64_t n, int val_u64,
                              double* __restrict__ out)
{
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        const double v = in[perm[i]];
        out[i] = val_u64 ? (double)(unsigned long long)v : v;
    }
}

// [first row, last row] before any nonzero: dims[n] and 0 (the reference's
// empty partition)
__global__ void k_intervals_init(DimArr dims, int nmode, uint64_t n, unsigned long long* __restrict__ iv)
{
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        iv[i] = (i & 1) ? 0ull : (unsigned long long)dims.d[(i >> 1) % nmode];
}

// partition intervals (include/alto.hpp:874-899): per (partition, mode) the
// [min, max] row; partition p holds [p*per, min((p+1)*per, nnz)).  A workgroup
// takes slices of up to IV_SLICE nonzeros of one partition, each thread keeps
// its minima and maxima in registers, and a slice ends in one pair of global
// atomics per mode and wavefront: bound by reading the keys (20M nonzeros,
// 3 modes: 1600 us with two LDS atomics per nonzero and mode before).
constexpr uint64_t IV_SLICE = 8192;
template <int W, int PW>
__global__ void __launch_bounds__(256) k_intervals(const uint64_t* __restrict__ keys, LutRef g_lut,
                                                   PackLayout L, uint64_t n, uint64_t per, uint64_t slices,
                                                   uint64_t nitems, unsigned long long* __restrict__ iv)
{
    extern __shared__ uint64_t s_lut[];
    const uint64_t* lut = stage_lut<PW>(s_lut, g_lut);
    for (uint64_t it = blockIdx.x; it < nitems; it += gridDim.x) {
        const uint64_t p = it / slices;
        const uint64_t b = p * per + (it - p * slices) * IV_SLICE;
        uint64_t e = b + IV_SLICE < (p + 1) * per ? b + IV_SLICE : (p + 1) * per;
        if (e > n) e = n;
        if (b >= e) continue;
        unsigned long long lo[ALTO_MAXN], hi[ALTO_MAXN];
#pragma unroll
        for (int m = 0; m < ALTO_MAXN; ++m) {
            lo[m] = ~0ull;
            hi[m] = 0;
        }
        for (uint64_t i = b + threadIdx.x; i < e; i += 256) {
            uint64_t k[W], pk[PW];
#pragma unroll
            for (int w = 0; w < W; ++w) k[w] = keys[i * W + w];
            lut_apply<W, PW>(lut, g_lut.nb, k, pk);
#pragma unroll
            for (int m = 0; m < ALTO_MAXN; ++m) {
                if (m < L.nmode) {
                    const unsigned long long r = field<PW>(pk, L.off[m], L.bits[m]);
                    lo[m] = r < lo[m] ? r : lo[m];
                    hi[m] = r > hi[m] ? r : hi[m];
                }
            }
        }
#pragma unroll
        for (int m = 0; m < ALTO_MAXN; ++m) {
            if (m < L.nmode) {
#pragma unroll
                for (int o = 32; o > 0; o >>= 1) {
                    const unsigned long long a = __shfl_xor(lo[m], o), c = __shfl_xor(hi[m], o);
                    lo[m] = a < lo[m] ? a : lo[m];
                    hi[m] = c > hi[m] ? c : hi[m];
                }
                if ((threadIdx.x & 63) == 0 && lo[m] != ~0ull) {
                    atomicMin(&iv[(p * L.nmode + m) * 2], lo[m]);
                    atomicMax(&iv[(p * L.nmode + m) * 2 + 1], hi[m]);
                }
            }
        }
    }
}

// CR ownership (include/alto.hpp:970-1020): rows reached from more than one
// partition get the mode's CR bit in every one of their keys.
template <int W, int PW>
__global__ void __launch_bounds__(256) k_cr_owner(const uint64_t* __restrict__ keys, LutRef g_lut,
                                                  PackLayout L, int mode, uint64_t n, uint64_t per, int* __restrict__ lo,
                                                  int* __restrict__ hi)
{
    extern __shared__ uint64_t s_lut[];
    const uint64_t* lut = stage_lut<PW>(s_lut, g_lut);
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        uint64_t k[W], pk[PW];
#pragma unroll
        for (int w = 0; w < W; ++w) k[w] = keys[i * W + w];
        lut_apply<W, PW>(lut, g_lut.nb, k, pk);
        uint64_t r = field<PW>(pk, L.off[mode], L.bits[mode]);
        const int p = (int)(i / per);
        // most updates change nothing (many nonzeros per row and partition):
        // read before issuing the atomic
        if (lo[r] > p) atomicMin(&lo[r], p);
        if (hi[r] < p) atomicMax(&hi[r], p);
    }
}

template <int W, int PW>
__global__ void __launch_bounds__(256) k_cr_set(uint64_t* __restrict__ keys, LutRef g_lut, PackLayout L,
                                                int mode, uint64_t n, const int* __restrict__ lo, const int* __restrict__ hi,
                                                uint64_t cm0, uint64_t cm1)
{
    extern __shared__ uint64_t s_lut[];
    const uint64_t* lut = stage_lut<PW>(s_lut, g_lut);
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        uint64_t k[W], pk[PW];
#pragma unroll
        for (int w = 0; w < W; ++w) k[w] = keys[i * W + w];
        lut_apply<W, PW>(lut, g_lut.nb, k, pk);
        uint64_t r = field<PW>(pk, L.off[mode], L.bits[mode]);
        if (lo[r] != hi[r]) {
            keys[i * W] = k[0] | cm0;
            if (W == 2) keys[i * W + W - 1] = k[W - 1] | cm1;
        }
    }
}

__global__ void k_fill_i32(int* __restrict__ a, uint64_t n, int v)
{
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) a[i] = v;
}

// rows of one mode in ALTO order, as sort keys
template <int W, int PW>
__global__ void __launch_bounds__(256) k_mode_key(const uint64_t* __restrict__ keys, LutRef g_lut, PackLayout L, int mode,
                                                  uint64_t n, uint64_t* __restrict__ ck)
{
    extern __shared__ uint64_t s_lut[];
    const uint64_t* lut = stage_lut<PW>(s_lut, g_lut);
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        uint64_t k[W], pk[PW];
#pragma unroll
        for (int w = 0; w < W; ++w) k[w] = keys[i * W + w];
        lut_apply<W, PW>(lut, g_lut.nb, k, pk);
        ck[i] = field<PW>(pk, L.off[mode], L.bits[mode]);
    }
}

// Packed coordinates and value of each nonzero side by side, in ALTO order:
// every mode's stream is gathered from these records (one access per nonzero
// where keys and values apart would take two, and the key's bits are permuted
// once instead of twice per mode).
template <int W, int PW>
__global__ void __launch_bounds__(256) k_records(const uint64_t* __restrict__ keys, const double* __restrict__ vals,
                                                 LutRef g_lut, uint64_t n, uint64_t* __restrict__ rec)
{
    extern __shared__ uint64_t s_lut[];
    const uint64_t* lut = stage_lut<PW>(s_lut, g_lut);
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        uint64_t k[W], pk[PW];
#pragma unroll
        for (int w = 0; w < W; ++w) k[w] = keys[i * W + w];
        lut_apply<W, PW>(lut, g_lut.nb, k, pk);
#pragma unroll
        for (int w = 0; w < PW; ++w) rec[i * (PW + 1) + w] = pk[w];
        rec[i * (PW + 1) + PW] = (uint64_t)__double_as_longlong(vals[i]);
    }
}

// Where the streams' nonzeros come from, by ALTO position: the records, or (when
// the records' memory is not there) the keys and values themselves.
template <int PW_>
struct FromRecords {
    static constexpr int PW = PW_;
    const uint64_t* rec;
    __device__ __forceinline__ void coords(uint64_t i, uint64_t (&pk)[PW]) const
    {
#pragma unroll
        for (int w = 0; w < PW; ++w) pk[w] = rec[i * (PW + 1) + w];
    }
    __device__ __forceinline__ double value(uint64_t i) const
    {
        return __longlong_as_double((long long)rec[i * (PW + 1) + PW]);
    }
};
template <int W, int PW_>
struct FromKeys {
    static constexpr int PW = PW_;
    const uint64_t* keys;
    const double* vals;
    const uint64_t* lut;
    int nb;
    __device__ __forceinline__ void coords(uint64_t i, uint64_t (&pk)[PW]) const
    {
        uint64_t k[W];
#pragma unroll
        for (int w = 0; w < W; ++w) k[w] = keys[i * W + w];
        lut_apply<W, PW>(lut, nb, k, pk);
    }
    __device__ __forceinline__ double value(uint64_t i) const { return vals[i]; }
};

// Sort key of a mode's stream: (chunk, row of `mode`, row of `amode`) of the
// nonzero at ALTO position idx[j] (j itself when idx is null; the positions
// are then left to the sort), without the last field when amode < 0.
template <typename K, typename S>
__global__ void __launch_bounds__(256) k_stream_key(S from, PackLayout L, int mode, int amode, int chunk_log2,
                                                    uint64_t n, const uint32_t* __restrict__ idx, K* __restrict__ ck,
                                                    uint32_t* __restrict__ pay)
{
    constexpr int PW = S::PW;
    const int ba = amode >= 0 ? L.bits[amode] : 0, bn = L.bits[mode];
    for (uint64_t j = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; j < n; j += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t i = idx ? idx[j] : j;
        uint64_t pk[PW];
        from.coords(i, pk);
        uint64_t k = ((i >> chunk_log2) << bn) | field<PW>(pk, L.off[mode], bn);
        if (amode >= 0) k = (k << ba) | field<PW>(pk, L.off[amode], ba);
        ck[j] = (K)k;
        if (idx) pay[j] = (uint32_t)i;
    }
}

// where a stream's nonzeros go
struct StreamOut {
    uint64_t* pk;
    double* v64;
    float* v32;
};

template <typename S>
__device__ inline void put_nonzero(const S& from, uint64_t src, uint64_t dst, const StreamOut& o)
{
    constexpr int PW = S::PW;
    uint64_t pk[PW];
    from.coords(src, pk);
    const double v = from.value(src);
#pragma unroll
    for (int w = 0; w < PW; ++w) o.pk[dst * PW + w] = pk[w];
    if (o.v64) o.v64[dst] = v;
    if (o.v32) o.v32[dst] = (float)v;
}

template <typename S>
__global__ void __launch_bounds__(256) k_mode_gather(S from, const uint32_t* __restrict__ perm, uint64_t n, StreamOut o)
{
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        put_nonzero(from, perm[i], i, o);
}

// ------------------------------------------------------------------ fiber layout
// Whether sorted position i lies in a run (fiber) of at least `min_len` equal
// keys: its equal neighbours to the left and to the right, each found by
// bisection (the keys are sorted, so equality ends once).
template <typename K>
__device__ inline bool fiber_long(const K* __restrict__ ck, uint64_t n, uint64_t i, uint32_t min_len, uint32_t top)
{
    const K k = ck[i];
    const uint32_t want = min_len - 1;
    uint32_t l = 0, r = 0;
    for (uint32_t st = top; st; st >>= 1)
        if (l + st <= want && i >= l + st && ck[i - l - st] == k) l += st;
    for (uint32_t st = top; st; st >>= 1)
        if (l + r + st <= want && i + r + st < n && ck[i + r + st] == k) r += st;
    return l + r >= want;
}

// The stable split of the sorted nonzeros into those of long fibers and the
// others: counts per tile, and (after their scan) the nonzeros put at their
// places -- as positions in perm when it is given, else gathered into the
// stream.  A tile is FS_ROUNDS rounds of 256 consecutive positions.
constexpr int FS_ROUNDS = 8;
constexpr int FS_TILE = 256 * FS_ROUNDS;

template <typename K>
__global__ void __launch_bounds__(256) k_fiber_count(const K* __restrict__ ck, uint64_t n, uint32_t min_len, uint32_t top,
                                                     uint32_t* __restrict__ cnt)
{
    __shared__ uint32_t s_wave[4];
    uint32_t c = 0;
#pragma unroll
    for (int j = 0; j < FS_ROUNDS; ++j) {
        const uint64_t i = (uint64_t)blockIdx.x * FS_TILE + j * 256 + threadIdx.x;
        c += (uint32_t)__popcll(__ballot(i < n && fiber_long(ck, n, i, min_len, top)));
    }
    if ((threadIdx.x & 63) == 0) s_wave[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0) cnt[blockIdx.x] = s_wave[0] + s_wave[1] + s_wave[2] + s_wave[3];
}

template <typename K, typename S>
__global__ void __launch_bounds__(256) k_fiber_place(const K* __restrict__ ck, const uint32_t* __restrict__ pay, uint64_t n,
                                                     uint32_t min_len, uint32_t top, const uint32_t* __restrict__ cnt,
                                                     const uint32_t* __restrict__ nlong, uint32_t* __restrict__ perm,
                                                     S from, StreamOut o)
{
    __shared__ uint32_t s_cnt[FS_ROUNDS * 4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t in = 0;  // bit j: round j's position is in a long fiber
    uint32_t below[FS_ROUNDS];
#pragma unroll
    for (int j = 0; j < FS_ROUNDS; ++j) {
        const uint64_t i = (uint64_t)blockIdx.x * FS_TILE + j * 256 + threadIdx.x;
        const bool lg = i < n && fiber_long(ck, n, i, min_len, top);
        const uint64_t b = __ballot(lg);
        below[j] = (uint32_t)__popcll(b & ((1ull << lane) - 1));
        if (lg) in |= 1u << j;
        if (lane == 0) s_cnt[j * 4 + wave] = (uint32_t)__popcll(b);
    }
    __syncthreads();
    uint32_t run = cnt[blockIdx.x];
    const uint64_t nl = nlong[0];
#pragma unroll
    for (int j = 0; j < FS_ROUNDS; ++j) {
        uint32_t before = 0, sum = 0;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            if (w < wave) before += s_cnt[j * 4 + w];
            sum += s_cnt[j * 4 + w];
        }
        const uint64_t i = (uint64_t)blockIdx.x * FS_TILE + j * 256 + threadIdx.x;
        if (i < n) {
            const uint64_t p = run + before + below[j];  // long nonzeros ahead of i
            const uint64_t dst = (in >> j) & 1 ? p : nl + (i - p);
            if (perm) perm[dst] = pay[i];
            else put_nonzero(from, pay[i], dst, o);
        }
        run += sum;
    }
}

#define DISPATCH_WPW(W_, PW_, ...)                                              \
    do {                                                                        \
        if ((W_) == 1 && (PW_) == 1) { constexpr int W = 1, PW = 1; __VA_ARGS__; } \
        else if ((W_) == 2 && (PW_) == 1) { constexpr int W = 2, PW = 1; __VA_ARGS__; } \
        else { constexpr int W = 2, PW = 2; __VA_ARGS__; }                      \
    } while (0)

int delinearize_all(const alto_tensor* t, uint64_t* coords, hipStream_t s)
{
    DISPATCH_WPW(t->W, t->pack.pw, {
        hipLaunchKernelGGL((k_delin_coords<W, PW>), dim3(grid_for(t->nnz)), dim3(256), lut_smem(t->delin), s,
                           t->key.as<uint64_t>(), lutref(t->delin), t->pack, t->nnz, coords);
    });
    HIP_TRY(hipGetLastError());
    return ALTO_OK;
}

// ------------------------------------------------------- row frequency ranks
// Nonzeros per row of mode m, from stream m (inside each chunk the rows are
// contiguous): each run adds (end - start) through two wrapping additions.
template <int PW>
__global__ void __launch_bounds__(256) k_row_counts(const uint64_t* __restrict__ pk, uint64_t n, int off, int bits,
                                                    int chunk_log2, uint32_t* __restrict__ cnt)
{
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        uint64_t k[PW], kp[PW], kn[PW];
#pragma unroll
        for (int w = 0; w < PW; ++w) k[w] = pk[i * PW + w];
        const uint64_t r = field<PW>(k, off, bits);
        bool start = i == 0, end = i + 1 == n;
        if (!start) {
#pragma unroll
            for (int w = 0; w < PW; ++w) kp[w] = pk[(i - 1) * PW + w];
            start = field<PW>(kp, off, bits) != r || (i >> chunk_log2) != ((i - 1) >> chunk_log2);
        }
        if (!end) {
#pragma unroll
            for (int w = 0; w < PW; ++w) kn[w] = pk[(i + 1) * PW + w];
            end = field<PW>(kn, off, bits) != r || (i >> chunk_log2) != ((i + 1) >> chunk_log2);
        }
        if (start) atomicAdd(&cnt[r], 0u - (uint32_t)i);
        if (end) atomicAdd(&cnt[r], (uint32_t)(i + 1));
    }
}

__global__ void k_rank_keys(const uint32_t* __restrict__ cnt, uint64_t d, int bits, uint64_t* __restrict__ keys)
{
    for (uint64_t r = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; r < d; r += (uint64_t)gridDim.x * blockDim.x)
        keys[r] = ((uint64_t)(0xffffffffu - cnt[r]) << bits) | r;
}

__global__ void k_rank_scatter(const uint32_t* __restrict__ pay, uint64_t d, uint32_t* __restrict__ rank_row,
                               uint32_t* __restrict__ row_rank)
{
    for (uint64_t k = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; k < d; k += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t r = pay[k];
        rank_row[k] = r;
        row_rank[r] = (uint32_t)k;
    }
}

struct RankTabs {
    const uint32_t* row_rank[ALTO_MAXN];
};

// rewrite the other modes' fields of one stream from rows to ranks
template <int PW>
__global__ void __launch_bounds__(256) k_stream_rank(uint64_t* __restrict__ pk, uint64_t n, PackLayout L, int mode,
                                                     RankTabs T)
{
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        uint64_t k[PW];
#pragma unroll
        for (int w = 0; w < PW; ++w) k[w] = pk[i * PW + w];
        for (int o = 0; o < L.nmode; ++o) {
            if (o == mode || L.bits[o] == 0) continue;
            set_field<PW>(k, L.off[o], L.bits[o], T.row_rank[o][field<PW>(k, L.off[o], L.bits[o])]);
        }
#pragma unroll
        for (int w = 0; w < PW; ++w) pk[i * PW + w] = k[w];
    }
}

// rank tables from the (row-ordered) streams, then every unranked stream
// rewritten; streams must all exist
static int rank_streams(alto_tensor* t, hipStream_t s)
{
    const uint64_t n = t->nnz;
    for (int m = 0; m < t->nmode; ++m) {
        if (t->rank_row[m].p) continue;
        const uint64_t d = t->dims[m];
        DevBuf cnt, keys, pay, rank_row, row_rank;  // (the tensor gets the tables when they are written)
        SortSpace sp;
        const Drain drain{s};
        ALTO_TRY(cnt.alloc(d * 4));
        ALTO_TRY(keys.alloc(d * 8));
        ALTO_TRY(pay.alloc(d * 4));
        ALTO_TRY(rank_row.alloc(d * 4));
        ALTO_TRY(row_rank.alloc(d * 4));
        ALTO_TRY(fill_zero(cnt.as<uint32_t>(), d, s));
        RANK_DISPATCH_PW(t->pack.pw, {
            hipLaunchKernelGGL((k_row_counts<PW>), dim3(grid_for(n)), dim3(256), 0, s, t->ms[m].pk.as<uint64_t>(), n,
                               t->pack.off[m], t->pack.bits[m], t->ms[m].chunk_log2, cnt.as<uint32_t>());
        });
        hipLaunchKernelGGL(k_rank_keys, dim3(grid_for(d)), dim3(256), 0, s, cnt.as<uint32_t>(), d, t->pack.bits[m],
                           keys.as<uint64_t>());
        HIP_TRY(hipGetLastError());
        ALTO_TRY(sort_pairs<uint64_t>(keys, pay, true, d, 32 + t->pack.bits[m], sp, s));
        hipLaunchKernelGGL(k_rank_scatter, dim3(grid_for(d)), dim3(256), 0, s, pay.as<uint32_t>(), d,
                           rank_row.as<uint32_t>(), row_rank.as<uint32_t>());
        HIP_TRY(hipGetLastError());
        HIP_TRY(hipStreamSynchronize(s));
        t->rank_row[m].swap(rank_row);
        t->row_rank[m].swap(row_rank);
    }
    RankTabs T;
    for (int m = 0; m < ALTO_MAXN; ++m) T.row_rank[m] = m < t->nmode ? t->row_rank[m].as<uint32_t>() : nullptr;
    for (int m = 0; m < t->nmode; ++m) {
        ModeStream& M = t->ms[m];
        if (M.ranked) continue;
        RANK_DISPATCH_PW(t->pack.pw, {
            hipLaunchKernelGGL((k_stream_rank<PW>), dim3(grid_for(n)), dim3(256), 0, s, M.pk.as<uint64_t>(), n,
                               t->pack, m, T);
        });
        HIP_TRY(hipGetLastError());
        M.ranked = 1;
    }
    return ALTO_OK;
}

int reserve_rank_copies(alto_tensor* t, uint64_t rank, size_t elem_bytes, hipStream_t s)
{
    bool ranked = false;
    for (int m = 0; m < t->nmode; ++m) ranked = ranked || t->ms[m].ranked;
    if (!ranked) return ALTO_OK;
    bool drained = false;
    for (int m = 0; m < t->nmode; ++m) {
        const size_t need = t->dims[m] * rank * elem_bytes + 64;
        if (t->pcopy[m].bytes >= need) continue;
        if (!drained) {  // the old copy goes back to the shared cache
            HIP_TRY(hipStreamSynchronize(s));
            ALTO_TRY(t->wait_uses());
            drained = true;
        }
        t->pcopy[m].release();
        ALTO_TRY(t->pcopy[m].alloc(need));
    }
    return ALTO_OK;
}

// ------------------------------------------------------- hot-pattern split
struct HotK {
    int k[ALTO_MAXN - 1];
};

// sort key of the split: (pattern, chunk, row); the stream is ranked, so the
// other modes' fields are ranks
template <int PW>
__global__ void __launch_bounds__(256) k_split_key(const uint64_t* __restrict__ pk, uint64_t n, PackLayout L, int mode,
                                                   HotK hk, int chunk_log2, int cbits, uint64_t* __restrict__ ck,
                                                   unsigned int* __restrict__ pat_count)
{
    __shared__ unsigned int s_cnt[16];
    if (threadIdx.x < 16) s_cnt[threadIdx.x] = 0;
    __syncthreads();
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        uint64_t k[PW];
#pragma unroll
        for (int w = 0; w < PW; ++w) k[w] = pk[i * PW + w];
        uint64_t pat = 0;
        int o = 0;
        for (int m = 0; m < L.nmode; ++m) {
            if (m == mode) continue;
            if (field<PW>(k, L.off[m], L.bits[m]) < (uint64_t)hk.k[o]) pat |= 1ull << o;
            ++o;
        }
        const uint64_t r = field<PW>(k, L.off[mode], L.bits[mode]);
        ck[i] = (((pat << cbits) | (i >> chunk_log2)) << L.bits[mode]) | r;
        atomicAdd(&s_cnt[pat], 1u);
    }
    __syncthreads();
    if (threadIdx.x < 16 && s_cnt[threadIdx.x]) atomicAdd(&pat_count[threadIdx.x], s_cnt[threadIdx.x]);
}

template <int PW>
__global__ void __launch_bounds__(256) k_split_gather(const uint64_t* __restrict__ pk, const double* __restrict__ v64,
                                                      const float* __restrict__ v32, const uint32_t* __restrict__ perm,
                                                      uint64_t n, uint64_t* __restrict__ pk_out,
                                                      double* __restrict__ v64_out, float* __restrict__ v32_out)
{
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t src = perm[i];
#pragma unroll
        for (int w = 0; w < PW; ++w) pk_out[i * PW + w] = pk[src * PW + w];
        if (v64) v64_out[i] = v64[src];
        if (v32) v32_out[i] = v32[src];
    }
}

// Groups a ranked stream by hot pattern (see ModeStream); hot_k[o] = rows of
// the o-th other mode counted as hot.  Synchronous on `s`.
int split_stream(alto_tensor* t, int mode, const int* hot_k, hipStream_t s)
{
    ModeStream& M = t->ms[mode];
    if (!M.ranked) {
        set_error("split_stream: stream %d is not ranked", mode);
        return ALTO_ERR_UNSUPPORTED;
    }
    const int no = t->nmode - 1;
    const uint64_t n = t->nnz;
    const int npat = 1 << no;  // at most 16 (five modes)
    uint64_t nchunks = (n + (1ull << M.chunk_log2) - 1) >> M.chunk_log2;
    int cbits = 0;
    while ((1ull << cbits) < nchunks) ++cbits;
    const int bits = no + cbits + t->pack.bits[mode];
    if (bits > 64) {
        set_error("split_stream: sort key of %d bits", bits);
        return ALTO_ERR_UNSUPPORTED;
    }
    HotK hk;
    for (int o = 0; o < ALTO_MAXN - 1; ++o) hk.k[o] = o < no ? hot_k[o] : 0;
    DevBuf ck, pay, cnt, pk2, v64, v32;
    SortSpace sp;
    const Drain drain{s};
    ALTO_TRY(ck.alloc(n * 8));
    ALTO_TRY(pay.alloc(n * 4));
    ALTO_TRY(cnt.alloc(64 * 4));
    ALTO_TRY(fill_zero(cnt.as<uint32_t>(), 64, s));
    ALTO_TRY(pk2.alloc(n * t->pack.pw * 8));
    if (M.val64.p) ALTO_TRY(v64.alloc(n * 8));
    if (M.val32.p) ALTO_TRY(v32.alloc(n * 4));
    RANK_DISPATCH_PW(t->pack.pw, {
        hipLaunchKernelGGL((k_split_key<PW>), dim3(grid_for(n)), dim3(256), 0, s, M.pk.as<uint64_t>(), n, t->pack, mode,
                           hk, M.chunk_log2, cbits, ck.as<uint64_t>(), cnt.as<unsigned int>());
    });
    HIP_TRY(hipGetLastError());
    ALTO_TRY(sort_pairs<uint64_t>(ck, pay, true, n, bits, sp, s));
    RANK_DISPATCH_PW(t->pack.pw, {
        hipLaunchKernelGGL((k_split_gather<PW>), dim3(grid_for(n)), dim3(256), 0, s, M.pk.as<uint64_t>(),
                           M.val64.as<double>(), M.val32.as<float>(), pay.as<uint32_t>(), n, pk2.as<uint64_t>(),
                           v64.as<double>(), v32.as<float>());
    });
    HIP_TRY(hipGetLastError());
    uint32_t hc[64];
    HIP_TRY(hipMemcpyAsync(hc, cnt.p, sizeof(hc), hipMemcpyDeviceToHost, s));
    HIP_TRY(hipStreamSynchronize(s));
    M.pk.swap(pk2);
    if (M.val64.p) M.val64.swap(v64);
    if (M.val32.p) M.val32.swap(v32);
    M.pat_start.assign(npat + 1, 0);
    for (int p = 0; p < npat; ++p) M.pat_start[p + 1] = M.pat_start[p] + hc[p];
    for (int o = 0; o < ALTO_MAXN - 1; ++o) M.hot_k[o] = hk.k[o];
    M.split = 1;
    return ALTO_OK;
}

// Ranked streams need every mode's rows below 2^32 (32-bit ranks) and a sort
// key of 32 count bits + row bits.
static bool rank_applicable(const alto_tensor* t)
{
    if (!hot_rows_enabled() || t->nmode < 2) return false;
    for (int m = 0; m < t->nmode; ++m)
        if (t->pack.bits[m] > 32) return false;
    return true;
}

// the order a mode's stream should have with the current settings
struct StreamLayout {
    int chunk_log2, fib_mode, fib_mode2, fib_min;
};
static StreamLayout wanted_layout(const alto_tensor* t, int m, int ranked)
{
    StreamLayout L{t->chunk_log2, -1, -1, 0};
    if (det_enabled()) {  // one chunk: each row's nonzeros contiguous
        L.chunk_log2 = 63;
        return L;
    }
    int fmin = 0, fchunk = 0;
    uint64_t fnnz = 0;
    const int tiers = fiber_settings(&fmin, &fchunk, &fnnz);
    if (ranked || !tiers || t->nmode < 3 || t->nnz < fnnz) return L;
    const uint64_t nch = (t->nnz + (1ull << fchunk) - 1) >> fchunk;
    int cb = 0;
    while ((1ull << cb) < nch) ++cb;
    // the fiber modes: the other modes with the fewest (rule 1: most) rows,
    // in that order, whose sort keys fit 64 bits
    const int most = fiber_rule();
    int pick[2] = {-1, -1};
    for (int k = 0; k < tiers; ++k) {
        int a = -1;
        for (int q = 0; q < t->nmode; ++q) {
            if (q == m || q == pick[0] || cb + t->pack.bits[m] + t->pack.bits[q] > 64) continue;
            if (a < 0 || (most ? t->dims[q] > t->dims[a] : t->dims[q] < t->dims[a])) a = q;
        }
        pick[k] = a;
        if (a < 0) break;
    }
    if (pick[0] < 0) return L;
    L.chunk_log2 = fchunk;
    L.fib_mode = pick[0];
    L.fib_mode2 = pick[1];
    L.fib_min = fmin;
    return L;
}

static int chunk_bits(uint64_t n, int chunk_log2)
{
    const uint64_t nch = chunk_log2 >= 63 ? 1 : (n + (1ull << chunk_log2) - 1) >> chunk_log2;
    int cb = 0;
    while ((1ull << cb) < nch) ++cb;
    return cb;
}

// Buffers shared by the orderings of a tensor's modes (all sized for nnz; ck
// and sort.keys, which change places in the sorts, both for the widest key)
struct OrderSpace {
    DevBuf rec, ck, pay, cnt, nl, perm;
    SortSpace sort;
    int hold_keys(uint64_t n, size_t key_bytes) const
    {
        if (ck.bytes >= n * key_bytes && pay.bytes >= n * 4) return ALTO_OK;
        set_error("mode streams: %zu bytes for %llu sort keys of %zu", ck.bytes, (unsigned long long)n, key_bytes);
        return ALTO_ERR_ARG;
    }
};

// f(the source of the tensor's nonzeros)
template <typename F>
static void with_source(const alto_tensor* t, const OrderSpace& w, F&& f)
{
    if (w.rec.p) {
        const uint64_t* rec = w.rec.as<uint64_t>();
        if (t->pack.pw == 1) f(FromRecords<1>{rec});
        else f(FromRecords<2>{rec});
    } else {
        DISPATCH_WPW(t->W, t->pack.pw, {
            f((FromKeys<W, PW>{t->key.as<uint64_t>(), t->vals.as<double>(), t->delin.dev.as<uint64_t>(), t->delin.nb}));
        });
    }
}

// bits of the widest sort key of stream m in layout L
static int stream_key_bits(const alto_tensor* t, int m, const StreamLayout& L)
{
    int a = 0;  // of the fiber mode's row
    if (L.fib_mode >= 0) a = t->pack.bits[L.fib_mode];
    if (L.fib_mode2 >= 0) a = std::max(a, t->pack.bits[L.fib_mode2]);
    return chunk_bits(t->nnz, L.chunk_log2) + t->pack.bits[m] + a;
}

// One fiber split: the nonzeros at ALTO positions idx[0, n) (0..n-1 when
// idx is null) ordered by (chunk, row_m, row_a) and split stably into the
// nonzeros of fibers of at least `min_len` and the others; their ALTO
// positions in that order go to perm[0, n), or without perm the nonzeros
// themselves to `o`.  The length of the first part goes to *nl_dev.
// Keys of up to 32 bits are sorted as such: two thirds of the bytes per pass.
template <typename K>
static int fiber_split(alto_tensor* t, int m, int amode, int chunk_log2, int bits, uint32_t min_len, const uint32_t* idx,
                       uint64_t n, OrderSpace& w, uint32_t* nl_dev, uint32_t* perm, const StreamOut& o, hipStream_t s)
{
    ALTO_TRY(w.hold_keys(n, sizeof(K)));
    with_source(t, w, [&](auto from) {
        hipLaunchKernelGGL((k_stream_key<K, decltype(from)>), dim3(grid_for(n)), dim3(256), 0, s, from, t->pack, m, amode,
                           chunk_log2, n, idx, w.ck.as<K>(), w.pay.as<uint32_t>());
    });
    HIP_TRY(hipGetLastError());
    ALTO_TRY(sort_pairs<K>(w.ck, w.pay, idx == nullptr, n, bits, w.sort, s));
    uint32_t top = 1;
    while (top * 2 <= min_len - 1) top *= 2;
    const uint64_t nt = (n + FS_TILE - 1) / FS_TILE;
    hipLaunchKernelGGL(k_fiber_count<K>, dim3((unsigned)nt), dim3(256), 0, s, w.ck.as<K>(), n, min_len, top,
                       w.cnt.as<uint32_t>());
    HIP_TRY(hipGetLastError());
    ALTO_TRY(scan_rows(w.cnt.as<uint32_t>(), 1, nt, nl_dev, s));
    with_source(t, w, [&](auto from) {
        hipLaunchKernelGGL((k_fiber_place<K, decltype(from)>), dim3((unsigned)nt), dim3(256), 0, s, w.ck.as<K>(),
                           w.pay.as<uint32_t>(), n, min_len, top, w.cnt.as<uint32_t>(), nl_dev, perm, from, o);
    });
    HIP_TRY(hipGetLastError());
    return ALTO_OK;
}

static int fiber_split_any(alto_tensor* t, int m, int amode, int chunk_log2, uint32_t min_len, const uint32_t* idx,
                           uint64_t n, OrderSpace& w, uint32_t* nl_dev, uint32_t* perm, const StreamOut& o,
                           hipStream_t s)
{
    const int bits = chunk_bits(t->nnz, chunk_log2) + t->pack.bits[m] + t->pack.bits[amode];
    return bits <= 32 ? fiber_split<uint32_t>(t, m, amode, chunk_log2, bits, min_len, idx, n, w, nl_dev, perm, o, s)
                      : fiber_split<uint64_t>(t, m, amode, chunk_log2, bits, min_len, idx, n, w, nl_dev, perm, o, s);
}

// Orders the nonzeros of stream m by (chunk, row_m, row_a), long fibers first
// and the others after them, and writes the stream; with a second fiber mode
// b the others are ordered by (chunk, row_m, row_b) and split again.  The
// lengths of the fiber parts go to nl_dev[0] and nl_dev[1] (the latter is
// left alone without a second fiber part).
static int fiber_order(alto_tensor* t, int m, const StreamLayout& L, OrderSpace& w, uint32_t* nl_dev, const StreamOut& o,
                       hipStream_t s)
{
    const uint64_t n = t->nnz;
    if (L.fib_mode2 < 0)
        return fiber_split_any(t, m, L.fib_mode, L.chunk_log2, (uint32_t)L.fib_min, nullptr, n, w, nl_dev, nullptr, o, s);
    uint32_t* perm = w.perm.as<uint32_t>();
    ALTO_TRY(fiber_split_any(t, m, L.fib_mode, L.chunk_log2, (uint32_t)L.fib_min, nullptr, n, w, nl_dev, perm, o, s));
    uint32_t nlong = 0;
    HIP_TRY(hipMemcpyAsync(&nlong, nl_dev, 4, hipMemcpyDeviceToHost, s));
    HIP_TRY(hipStreamSynchronize(s));
    if (nlong < n)  // the short part [nlong, n) of perm holds the ALTO positions it orders
        ALTO_TRY(fiber_split_any(t, m, L.fib_mode2, L.chunk_log2, (uint32_t)L.fib_min, perm + nlong, n - nlong, w,
                                 nl_dev + 1, perm + nlong, o, s));
    with_source(t, w, [&](auto from) {
        hipLaunchKernelGGL((k_mode_gather<decltype(from)>), dim3(grid_for(n)), dim3(256), 0, s, from, perm, n, o);
    });
    HIP_TRY(hipGetLastError());
    return ALTO_OK;
}

// The stream of mode m ordered by (chunk, row) into `o`
template <typename K>
static int row_order(alto_tensor* t, int m, int chunk_log2, int bits, OrderSpace& w, const StreamOut& o, hipStream_t s)
{
    const uint64_t n = t->nnz;
    ALTO_TRY(w.hold_keys(n, sizeof(K)));
    with_source(t, w, [&](auto from) {
        hipLaunchKernelGGL((k_stream_key<K, decltype(from)>), dim3(grid_for(n)), dim3(256), 0, s, from, t->pack, m, -1,
                           chunk_log2, n, nullptr, w.ck.as<K>(), nullptr);
    });
    HIP_TRY(hipGetLastError());
    ALTO_TRY(sort_pairs<K>(w.ck, w.pay, true, n, bits, w.sort, s));
    with_source(t, w, [&](auto from) {
        hipLaunchKernelGGL((k_mode_gather<decltype(from)>), dim3(grid_for(n)), dim3(256), 0, s, from,
                           w.pay.as<uint32_t>(), n, o);
    });
    HIP_TRY(hipGetLastError());
    return ALTO_OK;
}

// What a call that leaves early takes back: the arrays that it allocated and did
// not write, and whole streams that it was writing (bit m: stream m), so that the
// next call builds them
struct StreamsInWork {
    alto_tensor* t;
    int fresh64 = 0, fresh32 = 0, writing = 0;
    ~StreamsInWork()
    {
        for (int m = 0; m < t->nmode; ++m) {
            ModeStream& M = t->ms[m];
            if ((writing >> m) & 1) {
                M.pk.release();
                M.chunk_log2 = -1;
            }
            if (((writing | fresh64) >> m) & 1) M.val64.release();
            if (((writing | fresh32) >> m) & 1) M.val32.release();
        }
    }
};

// Writes every stream that lacks its coordinates or a value array, in the layout
// want[m].  Beside the streams this takes, per nonzero, 24 bytes for the sorts
// (16 where all keys have up to 32 bits, 4 more for a second fiber mode) and 16
// or (two-word coordinates) 24 for the records; when those last do not fit, the
// streams are gathered without records.  The streams' own arrays come first, so
// that the records are what gives way.
static int build_streams(alto_tensor* t, const StreamLayout* want, int need64, int need32, hipStream_t s)
{
    const uint64_t n = t->nnz;
    StreamsInWork work{t};
    OrderSpace w;
    const Drain drain{s};
    int modes = 0, key_bits = 0;
    bool second = false;
    for (int m = 0; m < t->nmode; ++m) {
        ModeStream& M = t->ms[m];
        if (M.pk.p && (!need64 || M.val64.p) && (!need32 || M.val32.p)) continue;
        modes |= 1 << m;
        if (!M.pk.p) {
            work.writing |= 1 << m;
            ALTO_TRY(M.pk.alloc(n * t->pack.pw * 8));
        }
        if (need64 && !M.val64.p) {
            work.fresh64 |= 1 << m;
            ALTO_TRY(M.val64.alloc(n * 8));
        }
        if (need32 && !M.val32.p) {
            work.fresh32 |= 1 << m;
            ALTO_TRY(M.val32.alloc(n * 4));
        }
        key_bits = std::max(key_bits, stream_key_bits(t, m, want[m]));
        second = second || want[m].fib_mode2 >= 0;
    }
    const size_t key_bytes = key_bits <= 32 ? 4 : 8;
    ALTO_TRY(w.ck.alloc(n * key_bytes));
    ALTO_TRY(w.pay.alloc(n * 4));
    ALTO_TRY(reserve_sort(n, key_bytes, w.sort));
    if (second) ALTO_TRY(w.perm.alloc(n * 4));
    ALTO_TRY(w.cnt.alloc((n + FS_TILE - 1) / FS_TILE * 4));
    ALTO_TRY(w.nl.alloc(ALTO_MAXN * 2 * 4));
    const int st = w.rec.alloc(n * (t->pack.pw + 1) * 8);
    if (st != ALTO_OK && st != ALTO_ERR_OOM) return st;
    ALTO_TRY(fill_zero(w.nl.as<uint32_t>(), ALTO_MAXN * 2, s));
    if (w.rec.p)
        DISPATCH_WPW(t->W, t->pack.pw, {
            hipLaunchKernelGGL((k_records<W, PW>), dim3(grid_for(n)), dim3(256), lut_smem(t->delin), s,
                               t->key.as<uint64_t>(), t->vals.as<double>(), lutref(t->delin), n, w.rec.as<uint64_t>());
        });
    HIP_TRY(hipGetLastError());
    int fibers = 0;  // modes ordered by fibers here
    for (int m = 0; m < t->nmode; ++m) {
        if (!((modes >> m) & 1)) continue;
        ModeStream& M = t->ms[m];
        work.writing |= 1 << m;
        M.ranked = 0;
        M.split = 0;
        M.pat_start.clear();
        // the stream is rewritten in its base order: every value array it
        // has is rewritten with it
        const StreamOut o{M.pk.as<uint64_t>(), M.val64.as<double>(), M.val32.as<float>()};
        const StreamLayout& L = want[m];
        if (L.fib_mode >= 0) {
            ALTO_TRY(fiber_order(t, m, L, w, w.nl.as<uint32_t>() + 2 * m, o, s));
            fibers |= 1 << m;
        } else {
            const int bits = stream_key_bits(t, m, L);
            if (bits <= 32) ALTO_TRY(row_order<uint32_t>(t, m, L.chunk_log2, bits, w, o, s));
            else ALTO_TRY(row_order<uint64_t>(t, m, L.chunk_log2, bits, w, o, s));
        }
        M.chunk_log2 = L.chunk_log2;
        M.fib_mode = L.fib_mode;
        M.fib_mode2 = L.fib_mode2;
        M.fib_min = L.fib_min;
        M.nlong = M.nlong2 = 0;
    }
    if (fibers) {
        uint32_t nl[ALTO_MAXN * 2];
        HIP_TRY(hipMemcpyAsync(nl, w.nl.p, sizeof nl, hipMemcpyDeviceToHost, s));
        HIP_TRY(hipStreamSynchronize(s));
        for (int m = 0; m < t->nmode; ++m)
            if ((fibers >> m) & 1) {
                t->ms[m].nlong = nl[2 * m];
                t->ms[m].nlong2 = nl[2 * m + 1];
            }
    }
    work.fresh64 = work.fresh32 = work.writing = 0;
    return ALTO_OK;
}

int prepare_mode_streams(alto_tensor* t, int need64, int need32, hipStream_t s)
{
    const int want_chunk = tuned_chunk_log2();
    if (want_chunk > 0 && want_chunk != t->chunk_log2) t->chunk_log2 = want_chunk;
    const int ranked = det_enabled() ? 0 : (int)rank_applicable(t);
    StreamLayout want[ALTO_MAXN];
    bool any = false, reorder = false;
    for (int m = 0; m < t->nmode; ++m) {
        const ModeStream& M = t->ms[m];
        want[m] = wanted_layout(t, m, ranked);
        if (M.chunk_log2 != want[m].chunk_log2 || M.ranked != ranked || M.fib_mode != want[m].fib_mode ||
            M.fib_mode2 != want[m].fib_mode2 || M.fib_min != want[m].fib_min)
            reorder = true;
        if ((need64 && !M.val64.p) || (need32 && !M.val32.p) || !M.pk.p) any = true;
    }
    if (!any && !reorder) return ALTO_OK;
    // buffers go back to the shared cache: drain work that may still read them
    HIP_TRY(hipStreamSynchronize(s));
    ALTO_TRY(t->wait_uses());
    for (int m = 0; m < t->nmode; ++m) {
        ModeStream& M = t->ms[m];
        if (M.chunk_log2 != want[m].chunk_log2 || M.ranked != ranked || M.fib_mode != want[m].fib_mode ||
            M.fib_mode2 != want[m].fib_mode2 || M.fib_min != want[m].fib_min) {
            M.pk.release();
            M.val64.release();
            M.val32.release();
            M.ranked = 0;
            M.split = 0;
            M.pat_start.clear();
            M.fib_mode = M.fib_mode2 = -1;
            M.fib_min = 0;
            M.nlong = M.nlong2 = 0;
        }
    }
    ALTO_TRY(build_streams(t, want, need64, need32, s));
    if (rank_applicable(t)) ALTO_TRY(rank_streams(t, s));
    HIP_TRY(hipStreamSynchronize(s));
    return ALTO_OK;
}

static int create_impl(int nmode, const uint64_t* dims, uint64_t nnz, const uint64_t* const* cidx,
                       const double* vals, int ptr_kind, int val_kind, int lit_bits, int nprtn, hipStream_t s,
                       alto_tensor** out)
{
    if (nmode < 1 || nmode > ALTO_MAXN || !dims || !cidx || !vals || !out || nprtn < 1 || nnz < 1) {
        set_error("alto_tensor_create: invalid argument");
        return ALTO_ERR_ARG;
    }
    if (nnz >= (1ull << 32)) {
        set_error("alto_tensor_create: nnz must be below 2^32");
        return ALTO_ERR_UNSUPPORTED;
    }
    for (int m = 0; m < nmode; ++m)
        if (dims[m] < 1) {
            set_error("alto_tensor_create: dims must be >= 1");
            return ALTO_ERR_ARG;
        }
    alto_tensor* t = new alto_tensor();
    std::unique_ptr<alto_tensor> guard(t);
    t->nmode = nmode;
    t->nnz = nnz;
    t->nprtn = nprtn;
    t->val_kind = val_kind;
    HIP_TRY(hipGetDevice(&t->device));
    for (int m = 0; m < nmode; ++m) t->dims[m] = dims[m];
    int total = 0;
    for (int m = 0; m < nmode; ++m) total += dims[m] > 1 ? 64 - __builtin_clzll(dims[m] - 1) : 0;
    if (lit_bits == 0) lit_bits = total <= 64 ? 64 : 128;
    if (lit_bits != 64 && lit_bits != 128) {
        set_error("lit_bits must be 64 or 128");
        return ALTO_ERR_ARG;
    }
    t->W = lit_bits / 64;
    t->alto_bits = compute_masks(nmode, dims, t->W, t->masks, t->alto_mask);
    if (t->alto_bits < 0) {
        set_error("alto_tensor_create: %d index bits exceed the %d-bit ALTO mask", total, lit_bits);
        return ALTO_ERR_ARG;
    }
    // the tensor's own buffers (guard) and every temporary here are released
    // only after the stream has drained: the allocator hands freed blocks to
    // other streams
    DevBuf dcoord[ALTO_MAXN], dvals, pay, bad, iv, lo, hi;
    SortSpace sp;
    const Drain drain{s};
    ALTO_TRY(build_luts(t, s));

    // inputs to device
    CoordPtrs cp = {};
    const double* dv = vals;
    if (ptr_kind == ALTO_PTR_HOST) {
        for (int m = 0; m < nmode; ++m) {
            ALTO_TRY(dcoord[m].alloc(nnz * 8));
            HIP_TRY(hipMemcpyAsync(dcoord[m].p, cidx[m], nnz * 8, hipMemcpyHostToDevice, s));
            cp.c[m] = dcoord[m].as<uint64_t>();
        }
        ALTO_TRY(dvals.alloc(nnz * 8));
        HIP_TRY(hipMemcpyAsync(dvals.p, vals, nnz * 8, hipMemcpyHostToDevice, s));
        dv = dvals.as<double>();
    } else {
        for (int m = 0; m < nmode; ++m) cp.c[m] = cidx[m];
    }

    ALTO_TRY(t->key.alloc(nnz * t->W * 8));
    ALTO_TRY(t->vals.alloc(nnz * 8));
    ALTO_TRY(pay.alloc(nnz * 4));
    ALTO_TRY(bad.alloc(4));
    ALTO_TRY(fill_zero(bad.as<int>(), 1, s));
    DimArr da = {};
    for (int m = 0; m < nmode; ++m) da.d[m] = dims[m];
    DISPATCH_WPW(t->W, t->pack.pw, {
        hipLaunchKernelGGL((k_linearize<PW, W>), dim3(grid_for(nnz)), dim3(256), lut_smem(t->lin), s, cp, nmode, da,
                           t->pack, lutref(t->lin), nnz, t->key.as<uint64_t>(), bad.as<int>());
    });
    HIP_TRY(hipGetLastError());
    // sort_alto: by the ALTO key (unique after duplicate merging; stable otherwise)
    if (t->W == 1) ALTO_TRY(sort_pairs<uint64_t>(t->key, pay, true, nnz, t->alto_bits, sp, s));
    else ALTO_TRY(sort_pairs<Key128>(t->key, pay, true, nnz, t->alto_bits, sp, s));
    hipLaunchKernelGGL(k_gather_vals, dim3(grid_for(nnz)), dim3(256), 0, s, dv, pay.as<uint32_t>(), nnz,
                       val_kind == ALTO_VAL_U64, t->vals.as<double>());
    HIP_TRY(hipGetLastError());

    // oidx flag (include/alto.hpp:250-258)
    for (int m = 0; m < nmode; ++m)
        if (nnz / dims[m] <= 4) t->is_oidx = 1;

    // prtn_alto: pointers (closed form) and intervals
    uint64_t per = (nnz + nprtn - 1) / nprtn;
    t->prtn_ptr.assign(nprtn + 1, 0);
    for (int p = 0; p < nprtn; ++p) t->prtn_ptr[p + 1] = std::min<uint64_t>((uint64_t)(p + 1) * per, nnz);
    {
        const uint64_t niv = (uint64_t)nprtn * nmode * 2;
        ALTO_TRY(iv.alloc(niv * 8));
        hipLaunchKernelGGL(k_intervals_init, dim3(grid_for(niv)), dim3(256), 0, s, da, nmode, niv,
                           iv.as<unsigned long long>());
        const uint64_t slices = (per + IV_SLICE - 1) / IV_SLICE, nitems = (uint64_t)nprtn * slices;
        DISPATCH_WPW(t->W, t->pack.pw, {
            hipLaunchKernelGGL((k_intervals<W, PW>), dim3((unsigned)std::min<uint64_t>(nitems, 4096)), dim3(256),
                               lut_smem(t->delin), s, t->key.as<uint64_t>(), lutref(t->delin), t->pack, nnz, per,
                               slices, nitems, iv.as<unsigned long long>());
        });
        HIP_TRY(hipGetLastError());
        t->intervals.assign(niv, 0);
        int hbad = 0;
        HIP_TRY(hipMemcpyAsync(&hbad, bad.p, 4, hipMemcpyDeviceToHost, s));
        HIP_TRY(hipMemcpyAsync(t->intervals.data(), iv.p, niv * 8, hipMemcpyDeviceToHost, s));
        HIP_TRY(hipStreamSynchronize(s));
        if (hbad) {  // nothing so far used a row as an index
            set_error("alto_tensor_create: a coordinate is outside dims");
            return ALTO_ERR_ARG;
        }
    }

    // CR bits (include/alto.hpp:930-1027)
    int free_bits = 64 * t->W - t->alto_bits;
    for (int m = 0; m < nmode; ++m) {
        if (nnz / dims[m] <= 4 && free_bits) {
            int pos = 64 * t->W - free_bits;
            t->cr_masks[m * t->W + (pos >> 6)] = 1ull << (pos & 63);
            t->alto_cr_mask[pos >> 6] |= 1ull << (pos & 63);
            --free_bits;
        }
    }
    for (int m = 0; m < nmode; ++m) {
        uint64_t cm0 = t->cr_masks[m * t->W], cm1 = t->W == 2 ? t->cr_masks[m * t->W + 1] : 0;
        // with one partition no row is shared, so no key gets the bit
        if (!(cm0 | cm1) || nprtn == 1) continue;
        ALTO_TRY(lo.alloc(dims[m] * 4));
        ALTO_TRY(hi.alloc(dims[m] * 4));
        hipLaunchKernelGGL(k_fill_i32, dim3(grid_for(dims[m])), dim3(256), 0, s, lo.as<int>(), dims[m], nprtn);
        hipLaunchKernelGGL(k_fill_i32, dim3(grid_for(dims[m])), dim3(256), 0, s, hi.as<int>(), dims[m], -1);
        DISPATCH_WPW(t->W, t->pack.pw, {
            hipLaunchKernelGGL((k_cr_owner<W, PW>), dim3(grid_for(nnz)), dim3(256), lut_smem(t->delin), s, t->key.as<uint64_t>(),
                               lutref(t->delin), t->pack, m, nnz, per, lo.as<int>(), hi.as<int>());
            hipLaunchKernelGGL((k_cr_set<W, PW>), dim3(grid_for(nnz)), dim3(256), lut_smem(t->delin), s, t->key.as<uint64_t>(),
                               lutref(t->delin), t->pack, m, nnz, lo.as<int>(), hi.as<int>(), cm0, cm1);
        });
        HIP_TRY(hipGetLastError());
        HIP_TRY(hipStreamSynchronize(s));
    }
    *out = guard.release();
    return ALTO_OK;
}

}  // namespace alto

using namespace alto;

extern "C" {

const char* alto_last_error(void) { return alto::last_error(); }
const char* alto_version(void) { return "alto-mi355x 0.1.2"; }

int alto_tensor_create(int nmodes, const uint64_t* dims, uint64_t nnz, const uint64_t* const* cidx,
                       const double* vals, int ptr_kind, int val_kind, int lit_bits, int nprtn,
                       alto_stream_t stream, alto_tensor_t** out)
{
    return create_impl(nmodes, dims, nnz, cidx, vals, ptr_kind, val_kind, lit_bits, nprtn, (hipStream_t)stream, out);
}

int alto_tensor_destroy(alto_tensor_t* t)
{
    if (!t) return ALTO_OK;
    const int st = t->wait_uses();  // kernels of asynchronous calls may still read the buffers
    delete t;
    return st;
}

int alto_tensor_info(const alto_tensor_t* t, alto_tensor_info_t* info)
{
    if (!t || !info) {
        set_error("alto_tensor_info: null argument");
        return ALTO_ERR_ARG;
    }
    memset(info, 0, sizeof(*info));
    info->nmodes = t->nmode;
    info->lit_words = t->W;
    info->alto_bits = t->alto_bits;
    info->nprtn = t->nprtn;
    info->is_oidx = t->is_oidx;
    info->val_kind = t->val_kind;
    info->nnz = t->nnz;
    for (int m = 0; m < t->nmode; ++m) info->dims[m] = t->dims[m];
    memcpy(info->mode_masks, t->masks, sizeof(t->masks));
    memcpy(info->alto_mask, t->alto_mask, sizeof(t->alto_mask));
    memcpy(info->cr_masks, t->cr_masks, sizeof(t->cr_masks));
    memcpy(info->alto_cr_mask, t->alto_cr_mask, sizeof(t->alto_cr_mask));
    uint64_t b = t->key.bytes + t->vals.bytes + t->lin.dev.bytes + t->delin.dev.bytes;
    for (int m = 0; m < t->nmode; ++m) b += t->ms[m].pk.bytes + t->ms[m].val64.bytes + t->ms[m].val32.bytes;
    info->device_bytes = b;
    return ALTO_OK;
}

int alto_tensor_export(const alto_tensor_t* t, uint64_t* idx, double* vals, uint64_t* prtn_ptr, uint64_t* intervals)
{
    if (!t) {
        set_error("alto_tensor_export: null tensor");
        return ALTO_ERR_ARG;
    }
    if (idx) HIP_TRY(hipMemcpy(idx, t->key.p, t->nnz * t->W * 8, hipMemcpyDeviceToHost));
    if (vals) HIP_TRY(hipMemcpy(vals, t->vals.p, t->nnz * 8, hipMemcpyDeviceToHost));
    if (prtn_ptr) memcpy(prtn_ptr, t->prtn_ptr.data(), (t->nprtn + 1) * 8);
    if (intervals) memcpy(intervals, t->intervals.data(), t->intervals.size() * 8);
    return ALTO_OK;
}

int alto_tensor_delinearize(const alto_tensor_t* t, uint64_t* coords)
{
    if (!t || !coords) {
        set_error("alto_tensor_delinearize: null argument");
        return ALTO_ERR_ARG;
    }
    DevBuf c;
    ALTO_TRY(c.alloc(t->nnz * t->nmode * 8));
    ALTO_TRY(delinearize_all(t, c.as<uint64_t>(), 0));
    HIP_TRY(hipMemcpy(coords, c.p, t->nnz * t->nmode * 8, hipMemcpyDeviceToHost));
    return ALTO_OK;
}

int alto_tensor_export_oidx(const alto_tensor_t* t, int mode, uint64_t* oidx)
{
    if (!t || !oidx || mode < 0 || mode >= t->nmode) {
        set_error("alto_tensor_export_oidx: invalid argument");
        return ALTO_ERR_ARG;
    }
    uint64_t n = t->nnz;
    DevBuf ck, pay;
    SortSpace sp;
    const Drain drain{nullptr};
    ALTO_TRY(ck.alloc(n * 8));
    ALTO_TRY(pay.alloc(n * 4));
    // a plain stable sort by row
    DISPATCH_WPW(t->W, t->pack.pw, {
        hipLaunchKernelGGL((k_mode_key<W, PW>), dim3(grid_for(n)), dim3(256), lut_smem(t->delin), 0, t->key.as<uint64_t>(),
                           lutref(t->delin), t->pack, mode, n, ck.as<uint64_t>());
    });
    HIP_TRY(hipGetLastError());
    ALTO_TRY(sort_pairs<uint64_t>(ck, pay, true, n, t->pack.bits[mode], sp, 0));
    std::vector<uint32_t> h(n);
    HIP_TRY(hipMemcpy(h.data(), pay.p, n * 4, hipMemcpyDeviceToHost));
    for (uint64_t i = 0; i < n; ++i) oidx[i] = h[i];
    return ALTO_OK;
}

int alto_pdep_keys(const alto_tensor_t* t, const uint64_t* coords, uint64_t n, uint64_t* keys, alto_stream_t stream)
{
    if (!t || !coords || !keys) {
        set_error("alto_pdep_keys: null argument");
        return ALTO_ERR_ARG;
    }
    hipStream_t s = (hipStream_t)stream;
    DISPATCH_WPW(t->W, t->pack.pw, {
        hipLaunchKernelGGL((k_pack_lin<PW, W>), dim3(grid_for(n)), dim3(256), lut_smem(t->lin), s, coords, t->pack,
                           lutref(t->lin), n, keys);
    });
    HIP_TRY(hipGetLastError());
    return const_cast<alto_tensor*>(t)->note_use(s);
}

int alto_pext_keys(const alto_tensor_t* t, const uint64_t* keys, uint64_t n, uint64_t* coords, alto_stream_t stream)
{
    if (!t || !coords || !keys) {
        set_error("alto_pext_keys: null argument");
        return ALTO_ERR_ARG;
    }
    hipStream_t s = (hipStream_t)stream;
    DISPATCH_WPW(t->W, t->pack.pw, {
        hipLaunchKernelGGL((k_delin_coords<W, PW>), dim3(grid_for(n)), dim3(256), lut_smem(t->delin), s, keys,
                           lutref(t->delin), t->pack, n, coords);
    });
    HIP_TRY(hipGetLastError());
    return const_cast<alto_tensor*>(t)->note_use(s);
}

int alto_device_malloc(void** p, uint64_t bytes)
{
    HIP_TRY(hipMalloc(p, bytes ? bytes : 8));
    return ALTO_OK;
}
int alto_device_free(void* p)
{
    HIP_TRY(hipFree(p));
    return ALTO_OK;
}
int alto_memcpy_h2d(void* dst, const void* src, uint64_t bytes)
{
    HIP_TRY(hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice));
    return ALTO_OK;
}
int alto_memcpy_d2h(void* dst, const void* src, uint64_t bytes)
{
    HIP_TRY(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost));
    return ALTO_OK;
}
int alto_memcpy_d2d(void* dst, const void* src, uint64_t bytes, alto_stream_t stream)
{
    HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, (hipStream_t)stream));
    return ALTO_OK;
}
int alto_device_trim(void)
{
    int dev = 0;
    HIP_TRY(hipGetDevice(&dev));
    Pool& P = pool();
    std::lock_guard<std::mutex> g(P.mu);
    for (auto& kv : P.free_blocks[dev & 63]) (void)hipFree(kv.second);
    P.free_blocks[dev & 63].clear();
    P.cached[dev & 63] = 0;
    return ALTO_OK;
}

int alto_device_synchronize(void)
{
    HIP_TRY(hipDeviceSynchronize());
    return ALTO_OK;
}

}  // extern "C"
