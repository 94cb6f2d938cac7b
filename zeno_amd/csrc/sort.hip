// Stable LSD radix sort for gfx950 (wave64).
//
// The partition step of the reference (ZSPartitionForZSParticles,
// projects/CuLagrange/mpm/MPMPipeline.cu:75-84) inserts block keys into a
// hash table; its exclusive scans (MPMPipeline.cu:210) and the zpc
// radix_sort_pair used for Morton ordering (projects/CUDA/Structures.hpp:430)
// are the library calls these kernels replace.  Here particles are binned by a
// stable sort of (block key, index), so the particle order and block list are
// deterministic and equal to std::stable_sort by key.
//
// 8-bit digits, tiles of 2048 keys (256 threads x 8 rounds); a pass is
//   hist    per-tile digit counts;
//   rows    (more than kFewTiles tiles) one workgroup per digit: exclusive prefix of the
//           digit's counts over the tiles, in place, and its total;
//   scatter stable in-tile ranks from wave ballots (8 ballots match the digit
//           across the 64 lanes).  A wave ranks 512 consecutive keys against its own
//           counts in LDS, so the rounds need no barrier; keys are then staged in LDS
//           in digit order so each digit run is written out with consecutive addresses.
//           The digits' bases are the scan of their totals, made by every workgroup; of
//           few tiles it also sums the counts itself.
// A launch here is mostly latency: 3,264 keys took 20 us a pass in five launches, now 9 in
// two; 1,048,583 keys 35 us, now 23 in three.
#include "zmpm_internal.h"

namespace zmpm {

namespace {

constexpr int kThreads = 256;
constexpr int kItems = 8;
constexpr int kChunk = kThreads * kItems;  // 2048
constexpr int kRadix = 256;
static_assert(kChunk == kSortChunk && kRadix == kSortRadix, "radix_scratch_bound's tile and digit sizes");

// LDS accesses of one wave before this come before those after it.
__device__ __forceinline__ void wave_order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t x, int lane) {
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        uint32_t y = __shfl_up(x, off, 64);
        if (lane >= off) x += y;
    }
    return x;
}

// Exclusive scan of one value per thread over a 256-thread block; returns the
// exclusive prefix and writes the block total to *total.
__device__ __forceinline__ uint32_t block_excl_scan256(uint32_t v, uint32_t *s_wave, uint32_t *total) {
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    uint32_t inc = wave_incl_scan(v, lane);
    if (lane == 63) s_wave[w] = inc;
    __syncthreads();
    uint32_t pre = 0, tot = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        uint32_t s = s_wave[k];
        pre += (k < w) ? s : 0u;
        tot += s;
    }
    __syncthreads();
    *total = tot;
    return pre + inc - v;
}

__global__ void __launch_bounds__(kThreads) k_fill(uint32_t *p, uint32_t value, int64_t n) {
    for (int64_t i = blockIdx.x * (int64_t)kThreads + threadIdx.x; i < n; i += (int64_t)gridDim.x * kThreads)
        p[i] = value;
}

// Summing the counts of up to 64 tiles in the scatter costs at most four batches of loads, less than a
// launch; the counts are then tile-major, so that the digits' threads read them together.
constexpr int64_t kFewTiles = 64;

template <bool FEW>
__global__ void __launch_bounds__(kThreads) k_rs_hist(const uint32_t *keys, int64_t n, int shift, uint32_t dmask,
                                                      uint32_t *hist, int64_t ntiles) {
    __shared__ uint32_t h[kRadix];
    const int t = threadIdx.x;
    h[t] = 0;
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * kChunk;
#pragma unroll
    for (int r = 0; r < kItems; ++r) {
        int64_t e = base + r * kThreads + t;
        if (e < n) atomicAdd(&h[(keys[e] >> shift) & dmask], 1u);
    }
    __syncthreads();
    hist[FEW ? (int64_t)blockIdx.x * kRadix + t : (int64_t)t * ntiles + blockIdx.x] = h[t];
}

// Workgroup = digit: its row of counts -> exclusive prefix in place; totals[digit] = the sum.
__global__ void __launch_bounds__(kThreads) k_rs_rows(uint32_t *hist, int64_t ntiles, uint32_t *totals) {
    __shared__ uint32_t s_wave[4];
    uint32_t *row = hist + (int64_t)blockIdx.x * ntiles;
    uint32_t carry = 0;
    for (int64_t b = 0; b < ntiles; b += kChunk) {
        const int64_t base = b + (int64_t)threadIdx.x * kItems;
        uint32_t v[kItems], sum = 0, tot;
#pragma unroll
        for (int k = 0; k < kItems; ++k) {
            v[k] = base + k < ntiles ? row[base + k] : 0u;
            sum += v[k];
        }
        uint32_t pre = carry + block_excl_scan256(sum, s_wave, &tot);
#pragma unroll
        for (int k = 0; k < kItems; ++k) {
            if (base + k < ntiles) row[base + k] = pre;
            pre += v[k];
        }
        carry += tot;
    }
    if (threadIdx.x == 0) totals[blockIdx.x] = carry;
}

template <bool FEW>
__global__ void __launch_bounds__(kThreads) k_rs_scatter(const uint32_t *keys_in, const uint32_t *vals_in, int64_t n,
                                                         int shift, uint32_t dmask, const uint32_t *hist,
                                                         const uint32_t *totals, int64_t ntiles, uint32_t *keys_out,
                                                         uint32_t *vals_out, uint32_t *inv_out) {
    __shared__ uint32_t s_keys[kChunk];
    __shared__ uint32_t s_vals[kChunk];
    __shared__ uint32_t s_wcnt[4][kRadix];
    __shared__ uint32_t s_start[kRadix];  // the digit's first slot in the tile
    __shared__ uint32_t s_base[kRadix];   // its first output position, less that slot
    __shared__ uint32_t s_wave[2][4];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int64_t tile = blockIdx.x, base = tile * kChunk;
    uint32_t key[kItems], val[kItems], rank[kItems];
#pragma unroll
    for (int r = 0; r < kItems; ++r) {
        const int64_t e = base + (w * kItems + r) * 64 + lane;
        key[r] = e < n ? keys_in[e] : 0u;
        val[r] = e < n ? (vals_in ? vals_in[e] : (uint32_t)e) : 0u;
    }
    // this thread's digit: keys of the tiles before this one, and of all
    uint32_t before = 0, total = 0;
    if (FEW) {
#pragma unroll 16
        for (int64_t j = 0; j < ntiles; ++j) {
            const uint32_t c = hist[j * kRadix + t];
            total += c;
            before += j < tile ? c : 0u;
        }
    } else {
        before = hist[(int64_t)t * ntiles + tile];
        total = totals[t];
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) s_wcnt[w][k * 64 + lane] = 0u;
    wave_order();
    const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
#pragma unroll
    for (int r = 0; r < kItems; ++r) {
        const bool valid = base + (w * kItems + r) * 64 + lane < n;
        const uint32_t d = (key[r] >> shift) & dmask;
        uint64_t m = __ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const bool bit = (d >> b) & 1u;
            const uint64_t bb = __ballot(bit);
            m &= bit ? bb : ~bb;
        }
        const uint32_t below = (uint32_t)__popcll(m & lt_mask), count = s_wcnt[w][d];
        rank[r] = count + below;
        wave_order();
        if (valid && below == 0) s_wcnt[w][d] = count + (uint32_t)__popcll(m);
        wave_order();
    }
    __syncthreads();
    // counts -> the waves' prefixes; the tile's digit starts; the digits' bases
    uint32_t c = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const uint32_t x = s_wcnt[k][t];
        s_wcnt[k][t] = c;
        c += x;
    }
    uint32_t all;
    const uint32_t start = block_excl_scan256(c, s_wave[0], &all);
    const uint32_t first = block_excl_scan256(total, s_wave[1], &all);
    s_start[t] = start;
    s_base[t] = first + before - start;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kItems; ++r) {
        if (base + (w * kItems + r) * 64 + lane < n) {
            const uint32_t d = (key[r] >> shift) & dmask;
            const uint32_t slot = s_start[d] + s_wcnt[w][d] + rank[r];
            s_keys[slot] = key[r];
            s_vals[slot] = val[r];
        }
    }
    __syncthreads();
    const int64_t tile_n = (n - base) < kChunk ? (n - base) : kChunk;
    for (int s = t; s < tile_n; s += kThreads) {
        const uint32_t k = s_keys[s], v = s_vals[s];
        const uint32_t pos = s_base[(k >> shift) & dmask] + (uint32_t)s;
        keys_out[pos] = k;
        vals_out[pos] = v;
        if (inv_out) inv_out[v] = pos;
    }
}

inline int64_t div_up(int64_t a, int64_t b) { return (a + b - 1) / b; }
inline size_t align256(size_t b) { return (b + 255) & ~size_t(255); }

}  // namespace

void fill_u32(uint32_t *p, uint32_t value, int64_t n, hipStream_t s) {
    if (n <= 0) return;
    int64_t blocks = div_up(n, kThreads);
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(k_fill, dim3((unsigned)blocks), dim3(kThreads), 0, s, p, value, n);
}

size_t radix_scratch_bytes(int64_t n) { return radix_scratch_bound(n); }

void radix_sort_pairs(const uint32_t *keys_in, const uint32_t *vals_in, int64_t n, int bit_lo, int bit_hi,
                      uint32_t *keys_out, uint32_t *vals_out, uint32_t *inv_out, void *scratch, hipStream_t s) {
    if (n <= 0) return;
    const int64_t ntiles = div_up(n, kChunk);
    char *p = (char *)scratch;
    uint32_t *tk = (uint32_t *)p;
    p += align256(sizeof(uint32_t) * (size_t)n);
    uint32_t *tv = (uint32_t *)p;
    p += align256(sizeof(uint32_t) * (size_t)n);
    uint32_t *hist = (uint32_t *)p;
    p += align256(sizeof(uint32_t) * (size_t)(ntiles * kRadix));
    uint32_t *totals = (uint32_t *)p;
    int passes = (bit_hi - bit_lo + 7) / 8;
    if (passes < 1) passes = 1;
    // the passes alternate between the scratch pair and the outputs, so that the last one
    // writes the outputs: pass k writes the outputs when passes - 1 - k is even
    for (int pass = 0; pass < passes; ++pass) {
        const bool to_out = ((passes - 1 - pass) & 1) == 0;
        const uint32_t *ksrc = pass == 0 ? keys_in : (to_out ? tk : keys_out);
        const uint32_t *vsrc = pass == 0 ? vals_in : (to_out ? tv : vals_out);
        const bool last = pass == passes - 1;
        uint32_t *kdst = to_out ? keys_out : tk;
        uint32_t *vdst = to_out ? vals_out : tv;
        const int shift = bit_lo + 8 * pass;
        const int bits = bit_hi - shift < 8 ? bit_hi - shift : 8;
        const uint32_t dmask = bits <= 0 ? 0u : ((1u << bits) - 1u);
        const dim3 g((unsigned)ntiles), wg(kThreads);
        uint32_t *inv = last ? inv_out : nullptr;
        if (ntiles <= kFewTiles) {
            hipLaunchKernelGGL(k_rs_hist<true>, g, wg, 0, s, ksrc, n, shift, dmask, hist, ntiles);
            hipLaunchKernelGGL(k_rs_scatter<true>, g, wg, 0, s, ksrc, vsrc, n, shift, dmask, (const uint32_t *)hist,
                               (const uint32_t *)nullptr, ntiles, kdst, vdst, inv);
        } else {
            hipLaunchKernelGGL(k_rs_hist<false>, g, wg, 0, s, ksrc, n, shift, dmask, hist, ntiles);
            hipLaunchKernelGGL(k_rs_rows, dim3(kRadix), wg, 0, s, hist, ntiles, totals);
            hipLaunchKernelGGL(k_rs_scatter<false>, g, wg, 0, s, ksrc, vsrc, n, shift, dmask, (const uint32_t *)hist,
                               (const uint32_t *)totals, ntiles, kdst, vdst, inv);
        }
    }
}

}  // namespace zmpm
