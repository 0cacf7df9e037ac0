// sort.hip - stable LSD radix sort_by_key for uint32 keys/values (gfx950).
//
// Replaces thrust::sort_by_key of sortParticles (DamBreak.Core/fluidSystem.cu:94-99).
// Stability is what makes the reference's permutation reproducible: index
// starts as the identity every step, so the expected result is exactly the
// stable argsort of the hash.
//
// One pass per digit (8 bits; 9 or 10 where that saves a pass), three launches
// per pass up to 2^17 counts, else four or five (reduce-then-scan):
//   rs_hist      per-tile digit histogram, written digit-major so that
//   scan         one exclusive scan gives every (digit, tile) its global base
//   rs_scatter   stable in-tile ranking with wave64 ballots (one a bit give
//                the mask of lanes holding the same digit), a local sort of
//                the tile in LDS, then coalesced runs written per digit.
// No inter-workgroup waiting anywhere, so no launch order assumptions.
#include "common.hpp"
#include "kernels.hpp"
#include "scan_device.hpp"

#include <mutex>
#include <string>
#include <type_traits>

namespace cmag {

constexpr int RS_NT = 256;
// keys per thread: 16 (4096-key tiles) for large sorts; 4 (1024-key tiles) up
// to RS_SMALL_N keys, where a pass is a handful of tiles and the in-tile
// ranking rounds, not bandwidth, set its duration
constexpr int RS_ITEMS = 16;
constexpr int RS_ITEMS_SMALL = 4;
constexpr uint32_t RS_SMALL_N = 1u << 18;
// Digits of 9 or 10 bits: keys of 17 to 20 bits take two passes instead of three,
// and end where they began, without the copy back: five to seven launches less
// of 4.6 us each.  Up to this many keys, where launches count; larger sorts keep
// 8 bits, whose runs of a tile's keys are longer.
constexpr uint32_t RS_WIDE_MAX = 1u << 21;
static int digit_bits(uint32_t n, int key_bits) {
    if (n > RS_WIDE_MAX || key_bits <= 16 || key_bits > 20) return 8;
    return key_bits <= 18 ? 9 : 10;
}
constexpr int SCAN_NT = 256;
constexpr int SCAN_ITEMS = 16;
constexpr int SCAN_TILE = SCAN_NT * SCAN_ITEMS;

// lanes of this wave whose digit equals mine (among valid lanes)
template <int BITS>
__device__ __forceinline__ uint64_t match_digit(uint32_t d, bool valid) {
    uint64_t m = __ballot(valid);
#pragma unroll
    for (int b = 0; b < BITS; ++b) {
        uint32_t bit = (d >> b) & 1u;
        uint64_t bb = __ballot(bit);
        m &= bit ? bb : ~bb;
    }
    return m;
}

// ---- exclusive scan of a uint32 array -------------------------------------
// the block total of one tile; each thread sums SCAN_ITEMS consecutive
// elements, as 16-byte words when vec and they lie inside len
__global__ __launch_bounds__(SCAN_NT) void scan_reduce_kernel(const uint32_t* __restrict__ in, size_t len,
                                                               uint32_t* __restrict__ partial, bool vec) {
    __shared__ uint32_t lds[SCAN_NT / 64];
    const size_t base = (size_t)blockIdx.x * SCAN_TILE + (size_t)threadIdx.x * SCAN_ITEMS;
    uint32_t sum = 0;
    if (vec && base + SCAN_ITEMS <= len) {
#pragma unroll
        for (int q = 0; q < SCAN_ITEMS / 4; ++q) {
            const uint4 x = *reinterpret_cast<const uint4*>(in + base + 4 * q);
            sum += (x.x + x.y) + (x.z + x.w);
        }
    } else {
#pragma unroll
        for (int k = 0; k < SCAN_ITEMS; ++k) sum += (base + k < len) ? in[base + k] : 0u;
    }
    uint32_t tot;
    block_exclusive_scan<SCAN_NT>(sum, lds, &tot);
    if (threadIdx.x == 0) partial[blockIdx.x] = tot;
}

// each thread owns SCAN_ITEMS consecutive elements, read and written as
// 16-byte words when vec (all pointers 16-byte aligned) and the thread's
// elements lie inside len; `carry` (may be null) holds the exclusive base of
// every block.  An in-place scan of a plain array is allowed: every thread
// reads its own elements before the block barrier and writes them after it.
__global__ __launch_bounds__(SCAN_NT) void scan_down_kernel(const uint32_t* in, uint32_t* out, size_t len,
                                                             const uint32_t* __restrict__ carry, bool vec) {
    static_assert(SCAN_ITEMS % 4 == 0, "16-byte words per thread");
    __shared__ uint32_t lds[SCAN_NT / 64];
    const size_t base = (size_t)blockIdx.x * SCAN_TILE + (size_t)threadIdx.x * SCAN_ITEMS;
    const bool whole = vec && base + SCAN_ITEMS <= len;
    uint32_t v[SCAN_ITEMS];
    if (whole) {
#pragma unroll
        for (int q = 0; q < SCAN_ITEMS / 4; ++q) {
            const uint4 x = *reinterpret_cast<const uint4*>(in + base + 4 * q);
            v[4 * q] = x.x; v[4 * q + 1] = x.y; v[4 * q + 2] = x.z; v[4 * q + 3] = x.w;
        }
    } else {
#pragma unroll
        for (int k = 0; k < SCAN_ITEMS; ++k) v[k] = (base + k < len) ? in[base + k] : 0u;
    }
    uint32_t sum = 0;
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; ++k) sum += v[k];
    uint32_t tot;
    uint32_t run = block_exclusive_scan<SCAN_NT>(sum, lds, &tot);
    if (carry) run += carry[blockIdx.x];
    uint32_t o[SCAN_ITEMS];
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; ++k) {
        o[k] = run;
        run += v[k];
    }
    if (whole) {
#pragma unroll
        for (int q = 0; q < SCAN_ITEMS / 4; ++q)
            *reinterpret_cast<uint4*>(out + base + 4 * q) = make_uint4(o[4 * q], o[4 * q + 1], o[4 * q + 2], o[4 * q + 3]);
    } else {
#pragma unroll
        for (int k = 0; k < SCAN_ITEMS; ++k)
            if (base + k < len) out[base + k] = o[k];
    }
}

// The whole scan in one launch, for up to SCAN_FRONT_TILES tiles: a workgroup sums
// what is in front of its tile itself (in 16-byte words, at most 28 a thread).
// The other two or three launches cost 4.6 us each; in and out are distinct and
// 16-byte aligned.
constexpr int SCAN_FRONT_NT = 1024;
constexpr size_t SCAN_FRONT_TILE = (size_t)SCAN_FRONT_NT * SCAN_ITEMS;
constexpr size_t SCAN_FRONT_TILES = 8;
__global__ __launch_bounds__(SCAN_FRONT_NT) void scan_front_kernel(const uint32_t* __restrict__ in,
                                                                   uint32_t* __restrict__ out, size_t len) {
    __shared__ uint32_t lds[SCAN_FRONT_NT / 64];
    const uint4* w = reinterpret_cast<const uint4*>(in);
    const size_t words = (size_t)blockIdx.x * (SCAN_FRONT_TILE / 4);
    uint32_t sum = 0, carry;
#pragma unroll 4
    for (size_t q = threadIdx.x; q < words; q += SCAN_FRONT_NT) {
        const uint4 x = w[q];
        sum += (x.x + x.y) + (x.z + x.w);
    }
    (void)block_exclusive_scan<SCAN_FRONT_NT>(sum, lds, &carry);
    const size_t base = (size_t)blockIdx.x * SCAN_FRONT_TILE + (size_t)threadIdx.x * SCAN_ITEMS;
    const bool whole = base + SCAN_ITEMS <= len;
    uint32_t v[SCAN_ITEMS];
    if (whole) {
#pragma unroll
        for (int q = 0; q < SCAN_ITEMS / 4; ++q) {
            const uint4 x = *reinterpret_cast<const uint4*>(in + base + 4 * q);
            v[4 * q] = x.x; v[4 * q + 1] = x.y; v[4 * q + 2] = x.z; v[4 * q + 3] = x.w;
        }
    } else {
#pragma unroll
        for (int k = 0; k < SCAN_ITEMS; ++k) v[k] = base + k < len ? in[base + k] : 0u;
    }
    sum = 0;
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; ++k) sum += v[k];
    uint32_t tot;
    uint32_t run = carry + block_exclusive_scan<SCAN_FRONT_NT>(sum, lds, &tot);
    uint32_t o[SCAN_ITEMS];
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; ++k) {
        o[k] = run;
        run += v[k];
    }
    if (whole) {
#pragma unroll
        for (int q = 0; q < SCAN_ITEMS / 4; ++q)
            *reinterpret_cast<uint4*>(out + base + 4 * q) = make_uint4(o[4 * q], o[4 * q + 1], o[4 * q + 2], o[4 * q + 3]);
    } else {
#pragma unroll
        for (int k = 0; k < SCAN_ITEMS; ++k)
            if (base + k < len) out[base + k] = o[k];
    }
}

size_t scan_levels_words(size_t len) {
    size_t words = 0;
    while (len > (size_t)SCAN_TILE) {
        len = (len + SCAN_TILE - 1) / SCAN_TILE;
        words += len;
    }
    return words;
}

// out = exclusive_scan(in) (in place allowed); workspace holds scan_levels_words(len) words
int exclusive_scan_u32(const uint32_t* in, uint32_t* out, size_t len, uint32_t* ws, hipStream_t s) {
    if (len == 0) return CMAG_OK;
    const bool vec = ((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out)) & 15u) == 0;
    if (len <= (size_t)SCAN_TILE) {
        hipLaunchKernelGGL(scan_down_kernel, dim3(1), dim3(SCAN_NT), 0, s, in, out, len, (const uint32_t*)nullptr,
                           vec);
        return check_launch("scan_down_kernel");
    }
    if (vec && in != out && len <= SCAN_FRONT_TILES * SCAN_FRONT_TILE) {
        hipLaunchKernelGGL(scan_front_kernel, dim3((uint32_t)((len + SCAN_FRONT_TILE - 1) / SCAN_FRONT_TILE)),
                           dim3(SCAN_FRONT_NT), 0, s, in, out, len);
        return check_launch("scan_front_kernel");
    }
    size_t blocks = (len + SCAN_TILE - 1) / SCAN_TILE;
    uint32_t* partial = ws;
    hipLaunchKernelGGL(scan_reduce_kernel, dim3((uint32_t)blocks), dim3(SCAN_NT), 0, s, in, len, partial, vec);
    CMAG_TRY(check_launch("scan_reduce_kernel"));
    // scan the partials in place (recursively for very long inputs)
    CMAG_TRY(exclusive_scan_u32(partial, partial, blocks, ws + blocks, s));
    hipLaunchKernelGGL(scan_down_kernel, dim3((uint32_t)blocks), dim3(SCAN_NT), 0, s, in, out, len,
                       (const uint32_t*)partial, vec);
    return check_launch("scan_down_kernel");
}

// ---- radix passes ----------------------------------------------------------
// per-tile digit counts: each wave counts into its own LDS histogram, and the
// block adds the wave histograms.  Keys in particle order are spatially
// coherent, so neighbouring lanes often share a digit: only the first lane of
// each run of equal digits adds, the run's length (lanes of one bin in
// different runs are serialised by the LDS atomics)
template <int ITEMS, int BITS>
__global__ __launch_bounds__(RS_NT) void rs_hist_kernel(const uint32_t* __restrict__ keys, uint32_t n,
                                                         int shift, uint32_t* __restrict__ counts,
                                                         uint32_t numTiles) {
    constexpr int NW = RS_NT / 64;
    constexpr uint32_t DIGITS = 1u << BITS;
    __shared__ uint32_t hist[NW][DIGITS];
    const int tid = threadIdx.x, w = tid >> 6;
#pragma unroll
    for (int k = 0; k < NW; ++k)
        for (uint32_t g = tid; g < DIGITS; g += RS_NT) hist[k][g] = 0;
    __syncthreads();
    const uint32_t base = blockIdx.x * (uint32_t)(RS_NT * ITEMS);
    uint32_t d[ITEMS];
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        const uint32_t idx = base + k * RS_NT + tid;
        d[k] = idx < n ? (keys[idx] >> shift) & (DIGITS - 1u) : DIGITS;
    }
    const int lane = __lane_id();
    const uint64_t above = lane == 63 ? 0ull : (~0ull << (lane + 1));
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        const uint32_t prev = __shfl_up(d[k], 1);
        const bool head = lane == 0 || prev != d[k];
        const uint64_t heads = __ballot(head);
        const uint64_t later = heads & above;
        const uint32_t next = later ? (uint32_t)(__ffsll((unsigned long long)later) - 1) : 64u;
        if (head && d[k] < DIGITS) atomicAdd(&hist[w][d[k]], next - (uint32_t)lane);
    }
    __syncthreads();
#pragma unroll
    for (uint32_t g = tid; g < DIGITS; g += RS_NT) {
        uint32_t c = 0;
#pragma unroll
        for (int k = 0; k < NW; ++k) c += hist[k][g];
        counts[(size_t)g * numTiles + blockIdx.x] = c;
    }
}

// Stable scatter of one tile: wave w ranks its own contiguous chunk of 64 *
// ITEMS keys in rounds of 64 (a key's rank is the number of keys of its digit
// before it in the chunk: earlier rounds, kept in the wave's LDS digit counts,
// plus lower lanes of its round), the waves' counts are turned into per-wave
// digit offsets, and the tile is reordered by digit in LDS and written out
// run by run.  Wave chunks, rounds and lanes follow the input order, so equal
// digits keep their order.
template <int ITEMS, int BITS>
__global__ __launch_bounds__(RS_NT) void rs_scatter_kernel(
    const uint32_t* __restrict__ keys_in, const uint32_t* __restrict__ vals_in,
    uint32_t* __restrict__ keys_out, uint32_t* __restrict__ vals_out, uint32_t n, int shift,
    const uint32_t* __restrict__ counts, const uint32_t* __restrict__ offsets, uint32_t numTiles) {
    constexpr int NW = RS_NT / 64;
    constexpr uint32_t TILE = RS_NT * ITEMS;
    constexpr uint32_t CHUNK = 64 * ITEMS;
    constexpr uint32_t DIGITS = 1u << BITS;
    constexpr int PER = DIGITS / RS_NT;  // digits per thread, next to each other
    __shared__ uint32_t s_keys[TILE];
    __shared__ uint32_t s_vals[TILE];
    __shared__ uint32_t s_base[DIGITS];
    __shared__ uint32_t s_start[DIGITS];
    __shared__ uint32_t s_wcnt[NW][DIGITS];
    __shared__ uint32_t s_scan[NW];

    const int tid = threadIdx.x, lane = __lane_id(), w = tid / 64;
    const uint32_t tile = blockIdx.x;
    const uint32_t base = tile * TILE;
    const uint32_t cnt = min(TILE, n - base);
    const uint32_t wbase = base + (uint32_t)w * CHUNK;

    uint32_t rk[ITEMS], rv[ITEMS];
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        const uint32_t idx = wbase + k * 64 + lane;
        rk[k] = idx < n ? keys_in[idx] : 0u;
        rv[k] = idx < n ? vals_in[idx] : 0u;
    }
#pragma unroll
    for (int ww = 0; ww < NW; ++ww)
        for (uint32_t g = tid; g < DIGITS; g += RS_NT) s_wcnt[ww][g] = 0;
    uint32_t c[PER], sum = 0;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const uint32_t g = tid * PER + j;
        c[j] = counts[(size_t)g * numTiles + tile];
        s_base[g] = offsets[(size_t)g * numTiles + tile];
        sum += c[j];
    }
    uint32_t tot;
    uint32_t at = block_exclusive_scan<RS_NT>(sum, s_scan, &tot);
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        s_start[tid * PER + j] = at;
        at += c[j];
    }
    __syncthreads();

    const uint64_t lt_mask = (lane == 0) ? 0ull : ((~0ull) >> (64 - lane));
    uint32_t rank[ITEMS];
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        const bool valid = wbase + k * 64 + lane < n;
        const uint32_t dg = (rk[k] >> shift) & (DIGITS - 1u);
        const uint64_t m = match_digit<BITS>(dg, valid);
        // LDS operations of one wave take effect in program order: every lane
        // reads its digit's count before the round's leaders advance it
        const uint32_t before = s_wcnt[w][dg];
        rank[k] = before + (uint32_t)__popcll(m & lt_mask);
        if (valid && (__ffsll((unsigned long long)m) - 1) == lane) s_wcnt[w][dg] = before + (uint32_t)__popcll(m);
    }
    __syncthreads();
#pragma unroll
    for (uint32_t g = tid; g < DIGITS; g += RS_NT) {
        uint32_t run = 0;
#pragma unroll
        for (int ww = 0; ww < NW; ++ww) {
            const uint32_t x = s_wcnt[ww][g];
            s_wcnt[ww][g] = run;
            run += x;
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        if (wbase + k * 64 + lane < n) {
            const uint32_t dg = (rk[k] >> shift) & (DIGITS - 1u);
            const uint32_t p = s_start[dg] + s_wcnt[w][dg] + rank[k];
            s_keys[p] = rk[k];
            s_vals[p] = rv[k];
        }
    }
    __syncthreads();

#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        const uint32_t p = k * RS_NT + tid;
        if (p < cnt) {
            const uint32_t key = s_keys[p];
            const uint32_t dg = (key >> shift) & (DIGITS - 1u);
            const uint32_t dst = s_base[dg] + (p - s_start[dg]);
            keys_out[dst] = key;
            vals_out[dst] = s_vals[p];
        }
    }
}

__global__ __launch_bounds__(256) void copy_u32_kernel(uint32_t* __restrict__ dst,
                                                        const uint32_t* __restrict__ src, size_t n) {
    size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) dst[i] = src[i];
}

int launch_copy_u32(uint32_t* dst, const uint32_t* src, size_t n, hipStream_t s) {
    if (n == 0) return CMAG_OK;
    uint32_t blocks = (uint32_t)std::min<size_t>((n + 255) / 256, 16384);
    hipLaunchKernelGGL(copy_u32_kernel, dim3(blocks), dim3(256), 0, s, dst, src, n);
    return check_launch("copy_u32_kernel");
}

static uint32_t tile_keys(uint32_t n) { return RS_NT * (n <= RS_SMALL_N ? RS_ITEMS_SMALL : RS_ITEMS); }
static uint32_t num_tiles(uint32_t n) { return (uint32_t)(((uint64_t)n + tile_keys(n) - 1) / tile_keys(n)); }

static size_t workspace_bytes_of(uint32_t n, int bits) {
    size_t len = ((size_t)1 << bits) * num_tiles(n);
    size_t words = 2 * len + scan_levels_words(len);
    return (words * sizeof(uint32_t) + 255) & ~(size_t)255;
}

size_t radix_sort_workspace_bytes(uint32_t n) { return workspace_bytes_of(n, 8); }

template <int ITEMS, int BITS>
static int radix_pass(const uint32_t* kin, const uint32_t* vin, uint32_t* kout, uint32_t* vout, uint32_t n, int shift,
                      uint32_t* workspace, hipStream_t s) {
    const uint32_t tiles = num_tiles(n);
    const size_t len = ((size_t)1 << BITS) * tiles;
    uint32_t *counts = workspace, *offsets = counts + len, *scan_ws = offsets + len;
    hipLaunchKernelGGL((rs_hist_kernel<ITEMS, BITS>), dim3(tiles), dim3(RS_NT), 0, s, kin, n, shift, counts, tiles);
    CMAG_TRY(check_launch("rs_hist_kernel"));
    CMAG_TRY(exclusive_scan_u32(counts, offsets, len, scan_ws, s));
    hipLaunchKernelGGL((rs_scatter_kernel<ITEMS, BITS>), dim3(tiles), dim3(RS_NT), 0, s, kin, vin, kout, vout, n, shift,
                       counts, offsets, tiles);
    return check_launch("rs_scatter_kernel");
}

int radix_sort_pairs(uint32_t* keys, uint32_t* vals, uint32_t* alt_keys, uint32_t* alt_vals,
                     uint32_t n, int key_bits, void* workspace, size_t workspace_bytes,
                     bool* result_in_alt, hipStream_t s) {
    *result_in_alt = false;
    if (key_bits < 0 || key_bits > 32) return fail(CMAG_E_INVALID, "key_bits outside [0,32]");
    if (n < 2 || key_bits == 0) return CMAG_OK;
    if (workspace_bytes < radix_sort_workspace_bytes(n))
        return fail(CMAG_E_SIZE, "radix sort workspace too small");
    // a workspace that holds the tables of 8-bit digits only is enough
    int bits = digit_bits(n, key_bits);
    if (workspace_bytes < workspace_bytes_of(n, bits)) bits = 8;
    const bool small = n <= RS_SMALL_N;
    uint32_t* ws = static_cast<uint32_t*>(workspace);
    uint32_t *kin = keys, *vin = vals, *kout = alt_keys, *vout = alt_vals;
    for (int shift = 0; shift < key_bits; shift += bits) {
        auto pass = [&](auto b) {
            constexpr int B = decltype(b)::value;
            return small ? radix_pass<RS_ITEMS_SMALL, B>(kin, vin, kout, vout, n, shift, ws, s)
                         : radix_pass<RS_ITEMS, B>(kin, vin, kout, vout, n, shift, ws, s);
        };
        CMAG_TRY(bits == 8   ? pass(std::integral_constant<int, 8>{})
                 : bits == 9 ? pass(std::integral_constant<int, 9>{})
                             : pass(std::integral_constant<int, 10>{}));
        std::swap(kin, kout);
        std::swap(vin, vout);
        *result_in_alt = !*result_in_alt;
    }
    return CMAG_OK;
}

// ---- scratch for callers that cannot allocate ------------------------------
// cmag_sort_by_key_noalloc keeps cmag_sort_by_key's scratch (alternate keys and
// values, then the per-tile digit tables) in this file-scope array, sized for
// CMAG_SORT_NOALLOC_MAX_KEYS keys.  Every GPU the library runs on holds its own
// copy until the process ends.  On the host the array's name is a stand-in, not
// a device address: host code only ever uses the address hipGetSymbolAddress
// returns for the current device, fetched once per device.
constexpr uint32_t NOALLOC_MAX_KEYS = CMAG_SORT_NOALLOC_MAX_KEYS;
static_assert(NOALLOC_MAX_KEYS > RS_SMALL_N && NOALLOC_MAX_KEYS % (RS_NT * RS_ITEMS) == 0,
              "the no-allocation limit sits in the large-tile regime, on a whole tile");

constexpr size_t round256(size_t b) { return (b + 255) & ~(size_t)255; }

constexpr size_t scan_levels_words_c(size_t len) {
    size_t words = 0;
    while (len > (size_t)SCAN_TILE) {
        len = (len + SCAN_TILE - 1) / SCAN_TILE;
        words += len;
    }
    return words;
}

// cmag_sort_scratch_bytes at a key count in the large-tile regime; the
// small-tile regime (n <= RS_SMALL_N) needs less than it does at the limit
constexpr size_t sort_scratch_bytes_large(size_t n) {
    return round256(n * 2 * sizeof(uint32_t)) +
           round256((2 * 256 * (n / (RS_NT * RS_ITEMS)) + scan_levels_words_c(256 * (n / (RS_NT * RS_ITEMS)))) *
                    sizeof(uint32_t));
}
constexpr size_t NOALLOC_BYTES = sort_scratch_bytes_large(NOALLOC_MAX_KEYS);
static_assert(sort_scratch_bytes_large(NOALLOC_MAX_KEYS) >=
                  round256((size_t)RS_SMALL_N * 8) +
                      round256((2 * 256 * (RS_SMALL_N / (RS_NT * RS_ITEMS_SMALL)) +
                                scan_levels_words_c(256 * (RS_SMALL_N / (RS_NT * RS_ITEMS_SMALL)))) *
                               sizeof(uint32_t)),
              "the array covers the small-tile regime too");

static __device__ __align__(256) unsigned char scratch[NOALLOC_BYTES];

constexpr int NOALLOC_MAX_DEVICES = 64;
static std::mutex noalloc_mu;
static void* noalloc_ptr[NOALLOC_MAX_DEVICES] = {};

// device address of `scratch` on the current device
static int noalloc_scratch(void** out) {
    int dev = -1;
    CMAG_HIP_TRY(hipGetDevice(&dev));
    if (dev < 0 || dev >= NOALLOC_MAX_DEVICES) return fail(CMAG_E_INVALID, "device ordinal beyond 63");
    std::lock_guard<std::mutex> lock(noalloc_mu);
    if (!noalloc_ptr[dev]) {
        void* p = nullptr;
        CMAG_HIP_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (!p) return fail(CMAG_E_HIP, "hipGetSymbolAddress returned a null address for the sort scratch");
        noalloc_ptr[dev] = p;
    }
    *out = noalloc_ptr[dev];
    return CMAG_OK;
}

}  // namespace cmag

using namespace cmag;

extern "C" {

static size_t sort_pairs_bytes(uint32_t n) { return ((size_t)n * 2 * sizeof(uint32_t) + 255) & ~(size_t)255; }
// the least a sort takes (8-bit digits); cmag_sort_scratch_bytes names what it runs fastest with
static size_t sort_least_bytes(uint32_t n) { return sort_pairs_bytes(n) + radix_sort_workspace_bytes(n); }

size_t cmag_sort_scratch_bytes(uint32_t n, int key_bits) {
    return sort_pairs_bytes(n) + workspace_bytes_of(n, digit_bits(n, key_bits));
}

int cmag_sort_by_key(uint32_t* keys, uint32_t* vals, uint32_t n, int key_bits, void* scratch,
                     size_t scratch_bytes, cmag_stream_t stream) {
    if (n && (!keys || !vals)) return fail(CMAG_E_INVALID, "cmag_sort_by_key: null pointer");
    if (n < 2 || key_bits == 0) return CMAG_OK;
    if (!scratch || scratch_bytes < sort_least_bytes(n))
        return fail(CMAG_E_SIZE, "cmag_sort_by_key: scratch smaller than cmag_sort_scratch_bytes");
    hipStream_t s = as_stream(stream);
    uint32_t* alt_keys = static_cast<uint32_t*>(scratch);
    uint32_t* alt_vals = alt_keys + n;
    const size_t pairs = sort_pairs_bytes(n);
    void* ws = static_cast<char*>(scratch) + pairs;
    bool in_alt = false;
    CMAG_TRY(radix_sort_pairs(keys, vals, alt_keys, alt_vals, n, key_bits, ws,
                              scratch_bytes - pairs, &in_alt, s));
    if (in_alt) {
        CMAG_TRY(launch_copy_u32(keys, alt_keys, n, s));
        CMAG_TRY(launch_copy_u32(vals, alt_vals, n, s));
    }
    return CMAG_OK;
}

size_t cmag_sort_noalloc_scratch_bytes(void) { return NOALLOC_BYTES; }

int cmag_sort_by_key_noalloc(uint32_t* keys, uint32_t* vals, uint32_t n, int key_bits, cmag_stream_t stream) {
    if (n && (!keys || !vals)) return fail(CMAG_E_INVALID, "cmag_sort_by_key_noalloc: null pointer");
    if (n > NOALLOC_MAX_KEYS)
        return fail(CMAG_E_SIZE, "cmag_sort_by_key_noalloc: n = " + std::to_string(n) +
                                     " keys is above the limit of " + std::to_string(NOALLOC_MAX_KEYS) +
                                     " (CMAG_SORT_NOALLOC_MAX_KEYS); use cmag_sort_by_key with a scratch buffer");
    if (n < 2 || key_bits == 0) return CMAG_OK;
    if (sort_least_bytes(n) > NOALLOC_BYTES)
        return fail(CMAG_E_SIZE, "cmag_sort_by_key_noalloc: scratch array smaller than the sort needs");
    void* ws = nullptr;
    CMAG_TRY(noalloc_scratch(&ws));
    return cmag_sort_by_key(keys, vals, n, key_bits, ws, NOALLOC_BYTES, stream);
}

}  // extern "C"
