// Stable LSD radix sort of (key, 32-bit position) pairs for wave64: the order
// of the ALTO format (sort_alto, include/alto.hpp:772-803) and of the
// per-mode streams.
//
// A pass over one digit of up to 8 bits is three launches: digit counts per
// tile, a scan of each digit's counts over the tiles, and the scatter.  Bound:
// HBM -- per element a pass reads the key for the counts and reads and writes
// key and position for the scatter.  What that bound needs is that the scatter
// writes in runs: a tile's pairs are put in digit order in LDS first, so that
// a wavefront writes ~16 consecutive elements per digit instead of 64 single
// ones at 64 places, and the ranking synchronises the workgroup once per tile
// and not three times per 256 keys (each wavefront counts its digits in LDS
// of its own).
#include "sort.hpp"

#include <algorithm>

#include "kernels_common.hpp"

namespace alto {

namespace {

constexpr int RS_THREADS = 256;
constexpr int RS_WAVES = RS_THREADS / 64;

__device__ inline unsigned digit_of(uint32_t k, int shift, unsigned mask) { return (k >> shift) & mask; }
__device__ inline unsigned digit_of(uint64_t k, int shift, unsigned mask) { return (unsigned)(k >> shift) & mask; }
__device__ inline unsigned digit_of(Key128 k, int shift, unsigned mask)
{
    if (shift >= 64) return (unsigned)(k.hi >> (shift - 64)) & mask;
    if (shift == 0) return (unsigned)k.lo & mask;
    return (unsigned)((k.lo >> shift) | (k.hi << (64 - shift))) & mask;
}

// lanes of the wavefront that hold the same digit
__device__ inline uint64_t match_digit(unsigned d, unsigned mask, bool valid)
{
    uint64_t m = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
        if ((mask >> b) == 0) break;  // uniform
        const bool bit = (d >> b) & 1;
        const uint64_t bb = __ballot(bit);
        m &= bit ? bb : ~bb;
    }
    return m;
}

// exclusive scan over the workgroup's threads; *all = the sum
template <int WAVES>
__device__ inline uint32_t block_scan(uint32_t v, uint32_t* s_wave, uint32_t* all)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = __shfl_up(x, o);
        if (lane >= o) x += y;
    }
    if (lane == 63) s_wave[wave] = x;
    __syncthreads();
    uint32_t before = 0, sum = 0;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
        if (w < wave) before += s_wave[w];
        sum += s_wave[w];
    }
    __syncthreads();
    *all = sum;
    return before + x - v;
}

template <typename K, int ITEMS>
__global__ void __launch_bounds__(RS_THREADS) k_rs_hist(const K* __restrict__ keys, uint64_t n, int shift,
                                                        unsigned mask, uint32_t* __restrict__ hist, uint32_t ntiles)
{
    __shared__ uint32_t h[RS_WAVES][256];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
#pragma unroll
    for (int w = 0; w < RS_WAVES; ++w) h[w][t] = 0;
    __syncthreads();
    const uint64_t base = (uint64_t)blockIdx.x * (RS_THREADS * ITEMS) + t;
    unsigned d[ITEMS];
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
        const uint64_t i = base + (uint64_t)j * RS_THREADS;
        d[j] = i < n ? digit_of(keys[i], shift, mask) : 256u;
    }
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
        // nearly sorted digits (the high ones of ordered input) would queue
        // 64 additions on one counter
        const unsigned d0 = (unsigned)__builtin_amdgcn_readfirstlane((int)d[j]);
        if (__all(d[j] == d0)) {
            if (lane == 0 && d0 < 256u) atomicAdd(&h[wave][d0], 64u);
        } else if (d[j] < 256u) {
            atomicAdd(&h[wave][d[j]], 1u);
        }
    }
    __syncthreads();
    uint32_t c = 0;
#pragma unroll
    for (int w = 0; w < RS_WAVES; ++w) c += h[w][t];
    if ((unsigned)t <= mask) hist[(size_t)t * ntiles + blockIdx.x] = c;
}

// one workgroup per row
constexpr int SCAN_THREADS = 1024;
constexpr int SCAN_ITEMS = 4;
__global__ void __launch_bounds__(SCAN_THREADS) k_scan_rows(uint32_t* __restrict__ a, uint64_t m,
                                                            uint32_t* __restrict__ total)
{
    __shared__ uint32_t s_wave[SCAN_THREADS / 64];
    uint32_t* row = a + (uint64_t)blockIdx.x * m;
    uint32_t carry = 0;
    for (uint64_t base = 0; base < m; base += SCAN_THREADS * SCAN_ITEMS) {
        const uint64_t i0 = base + (uint64_t)threadIdx.x * SCAN_ITEMS;
        uint32_t v[SCAN_ITEMS], sum = 0;
#pragma unroll
        for (int q = 0; q < SCAN_ITEMS; ++q) {
            v[q] = i0 + q < m ? row[i0 + q] : 0u;
            sum += v[q];
        }
        uint32_t all;
        uint32_t run = carry + block_scan<SCAN_THREADS / 64>(sum, s_wave, &all);
#pragma unroll
        for (int q = 0; q < SCAN_ITEMS; ++q) {
            if (i0 + q < m) row[i0 + q] = run;
            run += v[q];
        }
        carry += all;
    }
    if (threadIdx.x == 0) total[blockIdx.x] = carry;
}

// hist: per digit, the exclusive scan of the tiles' counts; total: each
// digit's count.  A wavefront's keys are ITEMS consecutive runs of 64, ranked
// run by run, so that equal digits keep their order.
template <typename K, int ITEMS>
__global__ void __launch_bounds__(RS_THREADS) k_rs_scatter(const K* __restrict__ keys, const uint32_t* __restrict__ pay,
                                                           uint64_t n, int shift, unsigned mask,
                                                           const uint32_t* __restrict__ hist,
                                                           const uint32_t* __restrict__ total, uint32_t ntiles,
                                                           K* __restrict__ keys_out, uint32_t* __restrict__ pay_out)
{
    constexpr int TILE = RS_THREADS * ITEMS;
    __shared__ __align__(16) unsigned char s_buf[TILE * sizeof(K)];  // keys, then positions
    __shared__ uint32_t s_cnt[RS_WAVES][256];
    __shared__ uint32_t s_off[256];
    __shared__ uint32_t s_wave[RS_WAVES];
    K* s_key = reinterpret_cast<K*>(s_buf);
    uint32_t* s_pay = reinterpret_cast<uint32_t*>(s_buf);
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
#pragma unroll
    for (int w = 0; w < RS_WAVES; ++w) s_cnt[w][t] = 0;
    const uint64_t tile = (uint64_t)blockIdx.x * TILE;
    const uint64_t first = tile + (uint64_t)wave * (64 * ITEMS) + lane;
    K key[ITEMS];
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
        const uint64_t i = first + j * 64;
        if (i < n) key[j] = keys[i];
        else key[j] = K{};
    }
    __syncthreads();
    uint32_t pos[ITEMS];
    const uint64_t lt = (1ull << lane) - 1;
    volatile uint32_t* cnt = s_cnt[wave];  // this wavefront's own: LDS keeps its order
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
        const bool valid = first + j * 64 < n;
        const unsigned d = digit_of(key[j], shift, mask);
        const uint64_t m = match_digit(d, mask, valid);
        const uint32_t before = cnt[d];
        const uint32_t r = (uint32_t)__popcll(m & lt);
        if (valid && r == 0) cnt[d] = before + (uint32_t)__popcll(m);
        pos[j] = before + r;
    }
    __syncthreads();
    // thread t: digit t.  Its start in the tile, its place in the output, and
    // each wavefront's offset
    {
        uint32_t c[RS_WAVES], sum = 0, all;
#pragma unroll
        for (int w = 0; w < RS_WAVES; ++w) {
            c[w] = s_cnt[w][t];
            sum += c[w];
        }
        const bool has = (unsigned)t <= mask;
        const uint32_t start = block_scan<RS_WAVES>(sum, s_wave, &all);
        const uint32_t below = block_scan<RS_WAVES>(has ? total[t] : 0u, s_wave, &all);
        s_off[t] = below + (has ? hist[(size_t)t * ntiles + blockIdx.x] : 0u) - start;
        uint32_t run = start;
#pragma unroll
        for (int w = 0; w < RS_WAVES; ++w) {
            s_cnt[w][t] = run;
            run += c[w];
        }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
        if (first + j * 64 < n) {
            pos[j] += s_cnt[wave][digit_of(key[j], shift, mask)];
            s_key[pos[j]] = key[j];
        }
    }
    uint32_t p[ITEMS];
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
        const uint64_t i = first + j * 64;
        p[j] = pay ? (i < n ? pay[i] : 0u) : (uint32_t)i;
    }
    __syncthreads();
    const uint32_t count = (uint32_t)(n - tile < (uint64_t)TILE ? n - tile : (uint64_t)TILE);
    uint32_t dst[ITEMS];
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
        const uint32_t q = j * RS_THREADS + t;
        dst[j] = 0;
        if (q < count) {
            const K k = s_key[q];
            dst[j] = s_off[digit_of(k, shift, mask)] + q;
            keys_out[dst[j]] = k;
        }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < ITEMS; ++j)
        if (first + j * 64 < n) s_pay[pos[j]] = p[j];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
        const uint32_t q = j * RS_THREADS + t;
        if (q < count) pay_out[dst[j]] = s_pay[q];
    }
}

__global__ void k_iota(uint32_t* __restrict__ p, uint64_t n)
{
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        p[i] = (uint32_t)i;
}

// A buffer that grows goes back to the cache shared by all streams: only after
// the work that may still use it
int grow(DevBuf& b, size_t bytes, hipStream_t s)
{
    if (b.bytes >= bytes) return ALTO_OK;
    if (b.p) HIP_TRY(hipStreamSynchronize(s));
    return b.alloc(bytes);
}

template <typename K, int ITEMS>
int sort_passes(DevBuf& keys, DevBuf& pay, bool identity, uint64_t n, int bits, SortSpace& sp, hipStream_t s)
{
    const uint64_t ntiles = (n + RS_THREADS * ITEMS - 1) / (RS_THREADS * ITEMS);
    ALTO_TRY(grow(sp.hist, 256 * ntiles * 4, s));
    ALTO_TRY(grow(sp.total, 256 * 4, s));
    const int passes = (bits + 7) / 8;
    for (int p = 0, shift = 0; p < passes; ++p) {
        const int w = (bits - shift + passes - p - 1) / (passes - p);  // digits of equal width
        const unsigned mask = (1u << w) - 1;
        const uint32_t* pin = identity && p == 0 ? nullptr : pay.as<uint32_t>();
        hipLaunchKernelGGL((k_rs_hist<K, ITEMS>), dim3((unsigned)ntiles), dim3(RS_THREADS), 0, s, keys.as<K>(), n, shift,
                           mask, sp.hist.as<uint32_t>(), (uint32_t)ntiles);
        ALTO_TRY(scan_rows(sp.hist.as<uint32_t>(), mask + 1, ntiles, sp.total.as<uint32_t>(), s));
        hipLaunchKernelGGL((k_rs_scatter<K, ITEMS>), dim3((unsigned)ntiles), dim3(RS_THREADS), 0, s, keys.as<K>(), pin,
                           n, shift, mask, sp.hist.as<uint32_t>(), sp.total.as<uint32_t>(), (uint32_t)ntiles,
                           sp.keys.as<K>(), sp.pay.as<uint32_t>());
        HIP_TRY(hipGetLastError());
        keys.swap(sp.keys);
        pay.swap(sp.pay);
        shift += w;
    }
    return ALTO_OK;
}

}  // namespace

int scan_rows(uint32_t* a, uint64_t rows, uint64_t m, uint32_t* total, hipStream_t s)
{
    hipLaunchKernelGGL(k_scan_rows, dim3((unsigned)rows), dim3(SCAN_THREADS), 0, s, a, m, total);
    HIP_TRY(hipGetLastError());
    return ALTO_OK;
}

// small inputs: shorter tiles, so that more workgroups share them
constexpr uint64_t SMALL = 1ull << 20;

int reserve_sort(uint64_t n, size_t key_bytes, SortSpace& sp)
{
    // (a part of n pairs may be a small input with more tiles than all of them)
    const uint64_t tiles = std::max((std::min(n, SMALL) + RS_THREADS * 4 - 1) / (RS_THREADS * 4),
                                    (n + RS_THREADS * 16 - 1) / (RS_THREADS * 16));
    ALTO_TRY(sp.keys.alloc(n * key_bytes));
    ALTO_TRY(sp.pay.alloc(n * 4));
    ALTO_TRY(sp.hist.alloc(256 * tiles * 4));
    return sp.total.alloc(256 * 4);
}

template <typename K>
int sort_pairs(DevBuf& keys, DevBuf& pay, bool identity, uint64_t n, int bits, SortSpace& sp, hipStream_t s)
{
    if (bits > 8 * (int)sizeof(K)) {
        set_error("radix sort: %d key bits exceed the %d-bit key", bits, 8 * (int)sizeof(K));
        return ALTO_ERR_UNSUPPORTED;
    }
    if (n >= (1ull << 32)) {
        set_error("radix sort supports fewer than 2^32 nonzeros");
        return ALTO_ERR_UNSUPPORTED;
    }
    // (the passes swap the halves, so what a shared space holds depends on the
    // sorts before this one)
    if (keys.bytes < n * sizeof(K) || pay.bytes < n * 4) {
        set_error("radix sort: %zu bytes of keys and %zu of positions for %llu pairs", keys.bytes, pay.bytes,
                  (unsigned long long)n);
        return ALTO_ERR_ARG;
    }
    if (n <= 1 || bits <= 0) {
        if (identity && n) {
            hipLaunchKernelGGL(k_iota, dim3((unsigned)std::min<uint64_t>((n + 255) / 256, 4096)), dim3(256), 0, s,
                               pay.as<uint32_t>(), n);
            HIP_TRY(hipGetLastError());
        }
        return ALTO_OK;
    }
    ALTO_TRY(grow(sp.keys, n * sizeof(K), s));
    ALTO_TRY(grow(sp.pay, n * 4, s));
    return n < SMALL ? sort_passes<K, 4>(keys, pay, identity, n, bits, sp, s)
                     : sort_passes<K, 16>(keys, pay, identity, n, bits, sp, s);
}
template int sort_pairs<uint32_t>(DevBuf&, DevBuf&, bool, uint64_t, int, SortSpace&, hipStream_t);
template int sort_pairs<uint64_t>(DevBuf&, DevBuf&, bool, uint64_t, int, SortSpace&, hipStream_t);
template int sort_pairs<Key128>(DevBuf&, DevBuf&, bool, uint64_t, int, SortSpace&, hipStream_t);

}  // namespace alto
