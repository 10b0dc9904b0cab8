// primitives.hip — device-wide scan, LSD radix sort and the deterministic
// reduction behind the compute shim's sort_by_key / sort /
// reduce_sum (compute/include/compute/{sort,reduction}.hpp).
#include <vector>

#include "dy_internal.hpp"

namespace dy {

// ---------------------------------------------------------------------------
// Exclusive scan
// ---------------------------------------------------------------------------
constexpr uint32_t kScanThreads = 1024;
constexpr uint32_t kScanItems = 8;
constexpr uint32_t kScanTile = kScanThreads * kScanItems;  // one workgroup pass
constexpr size_t kScanSingleMax = 1u << 16;

// One workgroup scans up to kScanSingleMax values: every tile's values are
// loaded before the first tile is scanned (one memory latency for the whole
// input), then the tiles are scanned in order with a running carry.
// `total` (may be null) receives the sum.
__global__ __launch_bounds__(kScanThreads) void scan_one_block(const uint32_t *__restrict__ in,
                                                               uint32_t *__restrict__ out, uint32_t n,
                                                               uint32_t *__restrict__ total) {
    constexpr uint32_t kMaxTiles = static_cast<uint32_t>(kScanSingleMax / kScanTile);
    __shared__ uint32_t tile[kScanTile];
    __shared__ uint32_t wsum[17];
    const uint32_t t = threadIdx.x;
    const uint32_t ntiles = (n + kScanTile - 1u) / kScanTile;
    uint32_t in_v[kMaxTiles][kScanItems];
#pragma unroll
    for (uint32_t b = 0; b < kMaxTiles; ++b)
#pragma unroll
        for (uint32_t j = 0; j < kScanItems; ++j) {
            const uint32_t idx = b * kScanTile + j * kScanThreads + t;
            in_v[b][j] = idx < n ? in[idx] : 0u;
        }
    uint32_t carry = 0;
#pragma unroll
    for (uint32_t b = 0; b < kMaxTiles; ++b) {
        if (b >= ntiles) break;
        const uint32_t base = b * kScanTile;
#pragma unroll
        for (uint32_t j = 0; j < kScanItems; ++j) tile[j * kScanThreads + t] = in_v[b][j];
        __syncthreads();
        uint32_t v[kScanItems], sum = 0;
#pragma unroll
        for (uint32_t j = 0; j < kScanItems; ++j) { v[j] = tile[t * kScanItems + j]; sum += v[j]; }
        uint32_t btotal;
        uint32_t run = carry + block_exclusive_scan(sum, wsum, btotal);
#pragma unroll
        for (uint32_t j = 0; j < kScanItems; ++j) { tile[t * kScanItems + j] = run; run += v[j]; }
        __syncthreads();
#pragma unroll
        for (uint32_t j = 0; j < kScanItems; ++j) {
            const uint32_t idx = base + j * kScanThreads + t;
            if (idx < n) out[idx] = tile[j * kScanThreads + t];
        }
        carry += btotal;
        __syncthreads();
    }
    if (t == 0 && total) *total = carry;
}

// One workgroup, values staged in LDS (one pad word per 32, so that a
// thread's contiguous run falls on distinct banks): thread t scans the run
// [t*K, t*K + K) serially, one workgroup scan of the 1 024 run sums gives each
// run's base — four workgroup barriers in all, against several per 8 192-value
// tile in scan_one_block.  Up to kScanLdsMax values.
constexpr uint32_t kScanLdsMax = kScanThreads * 36u;  // 36 864 values, 148.5 KiB with padding

__global__ __launch_bounds__(kScanThreads) void scan_lds(const uint32_t *__restrict__ in, uint32_t *__restrict__ out,
                                                         uint32_t n, uint32_t *__restrict__ total) {
    __shared__ uint32_t buf[kScanLdsMax + kScanLdsMax / 32u];
    __shared__ uint32_t wsum[17];
    const uint32_t t = threadIdx.x;
    const uint32_t k_run = (n + kScanThreads - 1u) / kScanThreads;  // values per thread (<= 36)
    const uint32_t padded = k_run * kScanThreads;
    for (uint32_t i0 = 0; i0 < padded; i0 += 8u * kScanThreads) {  // coalesced, eight loads in flight
        uint32_t v[8];
#pragma unroll
        for (uint32_t k = 0; k < 8u; ++k) {
            const uint32_t i = i0 + k * kScanThreads + t;
            v[k] = i < n ? in[i] : 0u;
        }
#pragma unroll
        for (uint32_t k = 0; k < 8u; ++k) {
            const uint32_t i = i0 + k * kScanThreads + t;
            if (i < padded) buf[i + (i >> 5)] = v[k];
        }
    }
    __syncthreads();
    const uint32_t r0 = t * k_run;
    uint32_t sum = 0;
    for (uint32_t k = 0; k < k_run; ++k) {
        const uint32_t i = r0 + k;
        sum += buf[i + (i >> 5)];
    }
    uint32_t all = 0;
    uint32_t run = block_exclusive_scan(sum, wsum, all);
    for (uint32_t k = 0; k < k_run; ++k) {
        const uint32_t i = r0 + k, j = i + (i >> 5);
        const uint32_t v = buf[j];
        buf[j] = run;
        run += v;
    }
    __syncthreads();
    for (uint32_t i = t; i < n; i += kScanThreads) out[i] = buf[i + (i >> 5)];
    if (t == 0 && total) *total = all;
}

constexpr uint32_t kMbThreads = 256;
constexpr uint32_t kMbItems = 8;
constexpr uint32_t kMbTile = kMbThreads * kMbItems;

__global__ __launch_bounds__(kMbThreads) void scan_tile_sums(const uint32_t *__restrict__ in, uint32_t n,
                                                             uint32_t *__restrict__ sums) {
    __shared__ uint32_t red[kMbThreads / 64];
    const uint32_t base = blockIdx.x * kMbTile;
    uint32_t s = 0;
#pragma unroll
    for (uint32_t j = 0; j < kMbItems; ++j) {
        const uint32_t idx = base + j * kMbThreads + threadIdx.x;
        if (idx < n) s += in[idx];
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) s += __shfl_xor(s, d, 64);
    if (lane_id() == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t t = 0;
        for (uint32_t w = 0; w < kMbThreads / 64; ++w) t += red[w];
        sums[blockIdx.x] = t;
    }
}

__global__ __launch_bounds__(kMbThreads) void scan_tiles(const uint32_t *__restrict__ in,
                                                         uint32_t *__restrict__ out, uint32_t n,
                                                         const uint32_t *__restrict__ offs) {
    __shared__ uint32_t tile[kMbTile];
    __shared__ uint32_t wsum[17];
    const uint32_t base = blockIdx.x * kMbTile, t = threadIdx.x;
#pragma unroll
    for (uint32_t j = 0; j < kMbItems; ++j) {
        const uint32_t idx = base + j * kMbThreads + t;
        tile[j * kMbThreads + t] = idx < n ? in[idx] : 0u;
    }
    __syncthreads();
    uint32_t v[kMbItems], sum = 0;
#pragma unroll
    for (uint32_t j = 0; j < kMbItems; ++j) { v[j] = tile[t * kMbItems + j]; sum += v[j]; }
    uint32_t btotal;
    uint32_t run = offs[blockIdx.x] + block_exclusive_scan(sum, wsum, btotal);
#pragma unroll
    for (uint32_t j = 0; j < kMbItems; ++j) { tile[t * kMbItems + j] = run; run += v[j]; }
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < kMbItems; ++j) {
        const uint32_t idx = base + j * kMbThreads + t;
        if (idx < n) out[idx] = tile[j * kMbThreads + t];
    }
}

__global__ __launch_bounds__(64) void clear_words_kernel(uint32_t *__restrict__ p, uint32_t n) {
    for (uint32_t i = threadIdx.x; i < n; i += 64u) p[i] = 0u;
}

int clear_words(hipStream_t s, uint32_t *p, uint32_t n) {
    if (n == 0) return DY_OK;
    clear_words_kernel<<<1, 64, 0, s>>>(p, n);
    DY_LAUNCH_CHECK();
    return DY_OK;
}

size_t scan_tmp_words(size_t n) {
    const size_t nb = (n + kMbTile - 1) / kMbTile;
    return 2 * nb + 2;
}

int scan_exclusive(hipStream_t s, const uint32_t *in, uint32_t *out, size_t n, uint32_t *d_total,
                   uint32_t *tmp) {
    if (n == 0) {
        if (d_total) DY_TRY(hipMemsetAsync(d_total, 0, sizeof(uint32_t), s));
        return DY_OK;
    }
    if (n > 0xffffffffu) return DY_ERR_INVALID_ARG;
    if (n <= kScanLdsMax) {
        scan_lds<<<1, kScanThreads, 0, s>>>(in, out, static_cast<uint32_t>(n), d_total);
        DY_LAUNCH_CHECK();
        return DY_OK;
    }
    if (n <= kScanSingleMax) {
        scan_one_block<<<1, kScanThreads, 0, s>>>(in, out, static_cast<uint32_t>(n), d_total);
        DY_LAUNCH_CHECK();
        return DY_OK;
    }
    const uint32_t nb = ceil_div(static_cast<uint32_t>(n), kMbTile);
    uint32_t *sums = tmp, *offs = tmp + nb;
    scan_tile_sums<<<nb, kMbThreads, 0, s>>>(in, static_cast<uint32_t>(n), sums);
    DY_LAUNCH_CHECK();
    scan_one_block<<<1, kScanThreads, 0, s>>>(sums, offs, nb, d_total);
    DY_LAUNCH_CHECK();
    scan_tiles<<<nb, kMbThreads, 0, s>>>(in, out, static_cast<uint32_t>(n), offs);
    DY_LAUNCH_CHECK();
    return DY_OK;
}

// ---------------------------------------------------------------------------
// Stable LSD radix sort, 8-bit digits.
//
// Up to kSortTile keys: sort_block, one workgroup, the keys in registers and
// exchanged through LDS between the passes (bound by its barriers and ballots;
// 1 000 u64 keys with values 50 -> 20 us a call, 8 192 147 -> 69 us, against a
// workgroup that kept them in global memory).  The tiled sort of 8 193 keys
// takes 133 us (a dozen launches), so the line lies at what one workgroup's
// LDS holds.
//
// More: sort_hist counts every digit of every key once, sort_plan turns the
// counts into each pass's digit starts, and sort_pass runs once per digit over
// tiles of kSortTile keys: a tile ranks its keys, publishes its digit counts,
// sums the counts of the tiles before it (decoupled look-back) and writes its
// keys, ordered in LDS, to one run per digit.  A pass moves each key and value
// once in and once out, the least an LSD pass can.  u64 keys with values:
// 100 003 1 596 -> 153 us, 1 000 003 17 300 -> 210 us, 8 000 001 141 000 ->
// 795 us (one workgroup on one CU before).  Tiles of 8 192: half as many
// look-back steps as with 4 096, and 1M keys still give 123 of them.  A pass
// whose digit is the same in every key (the high bytes of small keys) moves
// nothing; which buffer holds the keys then follows from the plan, and
// sort_finish copies them back if they ended in the scratch buffer.  Tiles
// take their numbers from a ticket, so every tile that one waits for is
// running already: the waits end whatever else the device runs.
// ---------------------------------------------------------------------------
constexpr uint32_t kSortThreads = 1024;
constexpr uint32_t kSortWaves = kSortThreads / 64;
constexpr uint32_t kSortItems = 8;
constexpr uint32_t kSortTile = kSortThreads * kSortItems;
constexpr uint32_t kSortHistMax = 256;  // workgroups (rows of counts) of sort_hist
constexpr uint32_t kSortPeek = 8;       // status words a look-back thread reads at a time

template <typename K>
__device__ __forceinline__ uint32_t digit_of(K k, uint32_t pass) {
    return static_cast<uint32_t>(k >> (8u * pass)) & 0xffu;
}

// Ranks one key per lane among the wavefront's keys of the same digit: `cnt`
// is the wavefront's digit counters in LDS, advanced by the keys ranked.
// Lanes without a key (valid false) take no part.
__device__ __forceinline__ uint32_t rank_in_wave(uint32_t d, bool valid, uint32_t *cnt, uint64_t lt_mask) {
    uint64_t peers = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
        const bool set = (d >> b) & 1u;
        const uint64_t bal = __ballot(set);
        peers &= set ? bal : ~bal;
    }
    const uint32_t pre = static_cast<uint32_t>(__popcll(peers & lt_mask));
    // a wavefront's LDS operations execute in program order; the fences hold the compiler to it
    const uint32_t c = valid ? cnt[d] : 0u;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (valid && pre == 0) cnt[d] = c + static_cast<uint32_t>(__popcll(peers));
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    return c + pre;
}

// Shared memory of a tile: keys and values by place in the tile, the
// wavefronts' digit counters (then each digit's keys in earlier wavefronts).
template <typename K, uint32_t ITEMS>
struct SortTile {
    K key[kSortThreads * ITEMS];
    uint32_t val[kSortThreads * ITEMS];
    uint32_t wcnt[kSortWaves][256];
    uint32_t start[256];  // digit's first place in the tile
    uint32_t wsum[17];
};

// Ranks the tile's keys on digit `pass`: place[j] becomes the place in the
// tile of the key in slot (wave, j, lane); returns the tile's count of digit t
// (threads t < 256).  Element order is (wave, item, lane).
template <typename K, uint32_t ITEMS>
__device__ __forceinline__ uint32_t rank_tile(SortTile<K, ITEMS> &S, const K (&kk)[ITEMS], uint32_t pass,
                                              uint32_t n_tile, uint32_t (&place)[ITEMS]) {
    const uint32_t t = threadIdx.x, lane = lane_id(), wave = t >> 6;
    const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    for (uint32_t i = t; i < kSortWaves * 256u; i += kSortThreads) (&S.wcnt[0][0])[i] = 0u;
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < ITEMS; ++j) {
        const bool valid = wave * (64u * ITEMS) + j * 64u + lane < n_tile;
        place[j] = rank_in_wave(digit_of(kk[j], pass), valid, S.wcnt[wave], lt_mask);
    }
    __syncthreads();
    uint32_t count = 0;
    if (t < 256u) {
#pragma unroll
        for (uint32_t w = 0; w < kSortWaves; ++w) {
            const uint32_t c = S.wcnt[w][t];
            S.wcnt[w][t] = count;
            count += c;
        }
    }
    uint32_t all;
    const uint32_t st = block_exclusive_scan(t < 256u ? count : 0u, S.wsum, all);
    if (t < 256u) S.start[t] = st;
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < ITEMS; ++j) {
        const uint32_t d = digit_of(kk[j], pass);
        place[j] += S.start[d] + S.wcnt[wave][d];
    }
    return count;
}

// ITEMS keys a thread: the launch takes the least power of two that holds n.
template <typename K, bool HAS_V, uint32_t ITEMS>
__global__ __launch_bounds__(kSortThreads) void sort_block(K *__restrict__ keys, uint32_t *__restrict__ vals,
                                                           uint32_t n) {
    __shared__ SortTile<K, ITEMS> S;
    const uint32_t lane = lane_id(), wave = threadIdx.x >> 6;
    K kk[ITEMS];
    uint32_t vv[ITEMS], place[ITEMS];
#pragma unroll
    for (uint32_t j = 0; j < ITEMS; ++j) {
        const uint32_t i = wave * (64u * ITEMS) + j * 64u + lane;
        kk[j] = i < n ? keys[i] : K(0);
        vv[j] = (HAS_V && i < n) ? vals[i] : 0u;
    }
    for (uint32_t pass = 0; pass < sizeof(K); ++pass) {
        (void)rank_tile(S, kk, pass, n, place);
#pragma unroll
        for (uint32_t j = 0; j < ITEMS; ++j) {
            const uint32_t i = wave * (64u * ITEMS) + j * 64u + lane;
            if (i < n) {
                S.key[place[j]] = kk[j];
                if (HAS_V) S.val[place[j]] = vv[j];
            }
        }
        __syncthreads();
#pragma unroll
        for (uint32_t j = 0; j < ITEMS; ++j) {
            const uint32_t i = wave * (64u * ITEMS) + j * 64u + lane;
            if (i < n) {
                kk[j] = S.key[i];
                if (HAS_V) vv[j] = S.val[i];
            }
        }
    }
#pragma unroll
    for (uint32_t j = 0; j < ITEMS; ++j) {
        const uint32_t i = wave * (64u * ITEMS) + j * 64u + lane;
        if (i < n) {
            keys[i] = kk[j];
            if (HAS_V) vals[i] = vv[j];
        }
    }
}

// Words the larger sort keeps beside its buffers: the plan (per pass: 256
// digit starts, then one "moves nothing" flag per pass), the tickets, the
// rows of digit counts, and two halves of status words (tile x digit), used
// by alternate passes.
struct SortWork {
    uint32_t *start;    // [passes][256]
    uint32_t *trivial;  // [8]
    uint32_t *ticket;   // [8]
    uint32_t *hist;     // [passes][rows][256]
    uint64_t *status[2];  // [tiles][256]: 0 = not there yet, kSortAgg | count, kSortPre | count of this and earlier tiles
    uint32_t rows, tiles;
};
constexpr uint64_t kSortAgg = 1ull << 62, kSortPre = 2ull << 62, kSortCount = kSortAgg - 1ull;

template <typename K>
__global__ __launch_bounds__(256) void sort_hist(const K *__restrict__ keys, uint32_t n, SortWork W) {
    constexpr uint32_t P = sizeof(K);
    __shared__ uint32_t h[P][256];
    const uint32_t t = threadIdx.x;
#pragma unroll
    for (uint32_t p = 0; p < P; ++p) h[p][t] = 0u;
    if (blockIdx.x == 0 && t < 8u) W.ticket[t] = 0u;
    for (size_t i = static_cast<size_t>(blockIdx.x) * 256u + t; i < static_cast<size_t>(W.tiles) * 256u;
         i += static_cast<size_t>(gridDim.x) * 256u)
        W.status[0][i] = 0ull;
    __syncthreads();
    // every wavefront makes the same number of rounds; a digit that is the
    // same in all its lanes costs one atomic
    constexpr uint32_t kAhead = 8;  // keys in flight a thread
    const size_t stride = static_cast<size_t>(gridDim.x) * 256u * kAhead;
    for (size_t b = static_cast<size_t>(blockIdx.x) * 256u * kAhead; b < n; b += stride) {
        K k[kAhead];
#pragma unroll
        for (uint32_t j = 0; j < kAhead; ++j) k[j] = b + j * 256u + t < n ? keys[b + j * 256u + t] : K(0);
#pragma unroll
        for (uint32_t j = 0; j < kAhead; ++j) {
            const bool valid = b + j * 256u + t < n;
            const uint64_t m = __ballot(valid);
            if (m == 0ull) continue;
            const uint32_t lead = static_cast<uint32_t>(__builtin_ctzll(m));
#pragma unroll
            for (uint32_t p = 0; p < P; ++p) {
                const uint32_t d = digit_of(k[j], p);
                const uint32_t d0 = __shfl(d, static_cast<int>(lead), 64);
                if (__ballot(valid && d != d0) == 0ull) {
                    if (lane_id() == lead) atomicAdd(&h[p][d0], static_cast<uint32_t>(__popcll(m)));
                } else if (valid) {
                    atomicAdd(&h[p][d], 1u);
                }
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (uint32_t p = 0; p < P; ++p)
        W.hist[(static_cast<size_t>(p) * W.rows + blockIdx.x) * 256u + t] = h[p][t];
}

// One workgroup per pass: the digits' first places.
__global__ __launch_bounds__(1024) void sort_plan(uint32_t n, SortWork W) {
    __shared__ uint32_t part[4][256];
    __shared__ uint32_t wsum[17];
    const uint32_t t = threadIdx.x, d = t & 255u, g = t >> 8;
    const uint32_t *h = W.hist + static_cast<size_t>(blockIdx.x) * W.rows * 256u;
    uint32_t sum = 0;
#pragma unroll 8
    for (uint32_t r = g; r < W.rows; r += 4u) sum += h[static_cast<size_t>(r) * 256u + d];
    part[g][d] = sum;
    __syncthreads();
    uint32_t total = 0;
    if (t < 256u) total = part[0][t] + part[1][t] + part[2][t] + part[3][t];
    uint32_t all;
    const uint32_t st = block_exclusive_scan(total, wsum, all);
    if (t < 256u) {
        W.start[blockIdx.x * 256u + t] = st;
        const uint64_t full = __ballot(total == n);
        if (lane_id() == 0) part[0][t >> 6] = full ? 1u : 0u;
    }
    __syncthreads();
    if (t == 0) W.trivial[blockIdx.x] = part[0][0] | part[0][1] | part[0][2] | part[0][3];
}

// Passes before `pass` that moved the keys: odd means they are in the scratch buffer.
__device__ __forceinline__ uint32_t sort_moves(const SortWork &W, uint32_t pass) {
    uint32_t moves = 0;
    for (uint32_t p = 0; p < pass; ++p) moves += W.trivial[p] ? 0u : 1u;
    return moves;
}

template <typename K, bool HAS_V>
__global__ __launch_bounds__(kSortThreads) void sort_pass(K *k0, uint32_t *v0, K *k1, uint32_t *v1, uint32_t n,
                                                          uint32_t pass, SortWork W) {
    __shared__ SortTile<K, kSortItems> S;
    __shared__ uint32_t s_tile;
    __shared__ uint64_t s_sum[kSortThreads / 256][256];
    __shared__ uint32_t s_found[kSortThreads / 256][256], s_open;
    constexpr uint32_t G = kSortThreads / 256;  // look-back threads per digit
    const uint32_t t = threadIdx.x, lane = lane_id(), wave = t >> 6;
    uint64_t *status = W.status[pass & 1u], *next = W.status[(pass + 1u) & 1u];
    for (uint32_t i = blockIdx.x * 256u + t; t < 256u && i < W.tiles * 256u; i += gridDim.x * 256u) next[i] = 0ull;
    if (W.trivial[pass]) return;
    const bool back = sort_moves(W, pass) & 1u;
    const K *sk = back ? k1 : k0;
    const uint32_t *sv = back ? v1 : v0;
    K *dk = back ? k0 : k1;
    uint32_t *dv = back ? v0 : v1;
    if (t == 0) s_tile = atomicAdd(&W.ticket[pass], 1u);
    __syncthreads();
    const uint32_t tile = s_tile;
    const uint32_t base = tile * kSortTile;
    const uint32_t n_tile = n - base < kSortTile ? n - base : kSortTile;
    K kk[kSortItems];
    uint32_t vv[kSortItems], place[kSortItems];
#pragma unroll
    for (uint32_t j = 0; j < kSortItems; ++j) {
        const uint32_t i = wave * (64u * kSortItems) + j * 64u + lane;
        kk[j] = i < n_tile ? sk[base + i] : K(0);
        vv[j] = (HAS_V && i < n_tile) ? sv[base + i] : 0u;
    }
    const uint32_t count = rank_tile(S, kk, pass, n_tile, place);
    if (t < 256u)
        __hip_atomic_store(&status[static_cast<size_t>(tile) * 256u + t], (tile ? kSortAgg : kSortPre) | count,
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
    for (uint32_t j = 0; j < kSortItems; ++j) {
        const uint32_t i = wave * (64u * kSortItems) + j * 64u + lane;
        if (i < n_tile) {
            S.key[place[j]] = kk[j];
            if (HAS_V) S.val[place[j]] = vv[j];
        }
    }
    __syncthreads();
    // Look-back: thread (g, d) sums digit d over kSortPeek of the G * kSortPeek
    // tiles before `hi`, nearest first, up to one that has its running count.
    const uint32_t d = t & 255u, g = t >> 8;
    uint64_t before = 0;
    bool open = tile > 0;  // this digit's running count not met yet (kept by g == 0)
    for (uint32_t hi = tile; hi > 0;) {
        uint64_t sum = 0;
        uint32_t found = 0;
        uint64_t w[kSortPeek];
#pragma unroll
        for (uint32_t j = 0; j < kSortPeek; ++j) {
            const uint32_t off = g * kSortPeek + j + 1u;
            w[j] = off <= hi ? __hip_atomic_load(&status[static_cast<size_t>(hi - off) * 256u + d], __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT)
                             : kSortPre;
        }
#pragma unroll
        for (uint32_t j = 0; j < kSortPeek; ++j) {
            if (found) continue;
            const uint32_t off = g * kSortPeek + j + 1u;
            while (w[j] == 0ull) {
                __builtin_amdgcn_s_sleep(1);
                w[j] = __hip_atomic_load(&status[static_cast<size_t>(hi - off) * 256u + d], __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
            }
            sum += w[j] & kSortCount;
            found = (w[j] & kSortPre) ? 1u : 0u;
        }
        s_sum[g][d] = sum;
        s_found[g][d] = found;
        if (t == 0) s_open = 0u;
        __syncthreads();
        if (g == 0 && open) {
            for (uint32_t q = 0; q < G && open; ++q) {
                before += s_sum[q][d];
                open = s_found[q][d] == 0u;
            }
        }
        if (g == 0 && __ballot(open) && lane == 0) s_open = 1u;
        __syncthreads();
        const bool more = s_open != 0u;
        __syncthreads();
        if (!more) break;
        hi -= hi < G * kSortPeek ? hi : G * kSortPeek;
    }
    if (t < 256u) {
        if (tile)
            __hip_atomic_store(&status[static_cast<size_t>(tile) * 256u + t], kSortPre | (before + count),
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        // destination of the key at place i of the tile, digit t: start + i (modulo 2^32)
        S.start[t] = W.start[pass * 256u + t] + static_cast<uint32_t>(before) - S.start[t];
    }
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < kSortItems; ++j) {
        const uint32_t i = j * kSortThreads + t;
        if (i < n_tile) {
            const K k = S.key[i];
            const uint32_t pos = S.start[digit_of(k, pass)] + i;
            dk[pos] = k;
            if (HAS_V) dv[pos] = S.val[i];
        }
    }
}

template <typename K, bool HAS_V>
__global__ __launch_bounds__(256) void sort_finish(K *__restrict__ k0, uint32_t *__restrict__ v0,
                                                   const K *__restrict__ k1, const uint32_t *__restrict__ v1,
                                                   uint32_t n, SortWork W) {
    if ((sort_moves(W, sizeof(K)) & 1u) == 0u) return;
    const size_t stride = static_cast<size_t>(gridDim.x) * 256u;
    for (size_t i = static_cast<size_t>(blockIdx.x) * 256u + threadIdx.x; i < n; i += stride) {
        k0[i] = k1[i];
        if (HAS_V) v0[i] = v1[i];
    }
}

// Bytes of scratch a sort of n keys needs (0: none), and its parts.
template <typename K, bool HAS_V>
static size_t sort_layout(size_t n, uint8_t *p, K **k1, uint32_t **v1, SortWork *W) {
    if (n <= kSortTile) return 0;
    size_t o = 0;
    auto take = [&](size_t bytes) {
        uint8_t *q = p ? p + o : nullptr;
        o += (bytes + 255u) & ~static_cast<size_t>(255u);
        return q;
    };
    W->tiles = static_cast<uint32_t>((n + kSortTile - 1u) / kSortTile);
    const size_t rows = (n + 4095u) / 4096u;
    W->rows = static_cast<uint32_t>(rows < kSortHistMax ? rows : kSortHistMax);
    *k1 = reinterpret_cast<K *>(take(n * sizeof(K)));
    *v1 = HAS_V ? reinterpret_cast<uint32_t *>(take(n * sizeof(uint32_t))) : nullptr;
    W->start = reinterpret_cast<uint32_t *>(take(sizeof(K) * 256u * 4u));
    W->trivial = reinterpret_cast<uint32_t *>(take(64u));
    W->ticket = W->trivial + 8;
    W->hist = reinterpret_cast<uint32_t *>(take(sizeof(K) * W->rows * 256u * 4u));
    for (auto &s : W->status) s = reinterpret_cast<uint64_t *>(take(static_cast<size_t>(W->tiles) * 256u * 8u));
    return o;
}

template <typename K, bool HAS_V>
static int radix_sort_t(hipStream_t s, K *k0, uint32_t *v0, size_t n) {
    if (n <= 1) return DY_OK;
    if (n > 0xffffffffu) return DY_ERR_INVALID_ARG;
    const uint32_t m = static_cast<uint32_t>(n);
    if (n <= kSortTile) {
        if (m <= kSortThreads) sort_block<K, HAS_V, 1><<<1, kSortThreads, 0, s>>>(k0, v0, m);
        else if (m <= 2u * kSortThreads) sort_block<K, HAS_V, 2><<<1, kSortThreads, 0, s>>>(k0, v0, m);
        else if (m <= 4u * kSortThreads) sort_block<K, HAS_V, 4><<<1, kSortThreads, 0, s>>>(k0, v0, m);
        else sort_block<K, HAS_V, 8><<<1, kSortThreads, 0, s>>>(k0, v0, m);
        DY_LAUNCH_CHECK();
        return DY_OK;
    }
    SortWork W{};
    K *k1 = nullptr;
    uint32_t *v1 = nullptr;
    uint8_t *p = nullptr;
    DY_TRY(hipMallocAsync(reinterpret_cast<void **>(&p), sort_layout<K, HAS_V>(n, nullptr, &k1, &v1, &W), s));
    (void)sort_layout<K, HAS_V>(n, p, &k1, &v1, &W);
    sort_hist<K><<<W.rows, 256, 0, s>>>(k0, m, W);
    sort_plan<<<sizeof(K), 1024, 0, s>>>(m, W);
    for (uint32_t pass = 0; pass < sizeof(K); ++pass)
        sort_pass<K, HAS_V><<<W.tiles, kSortThreads, 0, s>>>(k0, v0, k1, v1, m, pass, W);
    const uint32_t blocks = ceil_div(m, 1024u);
    sort_finish<K, HAS_V><<<blocks < 2048u ? blocks : 2048u, 256, 0, s>>>(k0, v0, k1, v1, m, W);
    const hipError_t launched = hipGetLastError();
    DY_TRY(hipFreeAsync(p, s));
    return static_cast<int>(launched);
}

// ---------------------------------------------------------------------------
// Deterministic sum: 256-wide halving tree per workgroup, partials merged on
// the host in index order (compute/include/compute/reduction.hpp:22-62).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void reduce_sum_partials(const float *__restrict__ d, size_t n,
                                                           float *__restrict__ partial) {
    __shared__ float sm[256];
    const size_t gid = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x;
    const uint32_t lid = threadIdx.x;
    sm[lid] = gid < n ? d[gid] : 0.f;
    __syncthreads();
    for (uint32_t st = 128; st > 0; st >>= 1) {
        if (lid < st) sm[lid] += sm[lid + st];
        __syncthreads();
    }
    if (lid == 0) partial[blockIdx.x] = sm[0];
}

}  // namespace dy

using namespace dy;

namespace {
template <typename K>
static int sort_api(dy_stream_t s, K *keys, uint32_t *vals, size_t n) {
    if (n <= 1) return DY_OK;
    if (!keys) return DY_ERR_INVALID_ARG;
    return vals ? radix_sort_t<K, true>(hs(s), keys, vals, n) : radix_sort_t<K, false>(hs(s), keys, vals, n);
}

}  // namespace

extern "C" {

int dy_scan_exclusive_u32(dy_stream_t s, const uint32_t *d_in, uint32_t *d_out, size_t n, uint32_t *d_total) {
    if ((n && (!d_in || !d_out))) return DY_ERR_INVALID_ARG;
    uint32_t *tmp = nullptr;
    if (n > kScanSingleMax) DY_TRY(hipMallocAsync(reinterpret_cast<void **>(&tmp),
                                                  scan_tmp_words(n) * sizeof(uint32_t), hs(s)));
    const int st = scan_exclusive(hs(s), d_in, d_out, n, d_total, tmp);
    if (tmp) DY_TRY(hipFreeAsync(tmp, hs(s)));
    return st;
}

int dy_sort_by_key_u64_u32(dy_stream_t s, uint64_t *keys, uint32_t *vals, size_t n) {
    if (n > 1 && !vals) return DY_ERR_INVALID_ARG;
    return sort_api<uint64_t>(s, keys, vals, n);
}
int dy_sort_by_key_u32_u32(dy_stream_t s, uint32_t *keys, uint32_t *vals, size_t n) {
    if (n > 1 && !vals) return DY_ERR_INVALID_ARG;
    return sort_api<uint32_t>(s, keys, vals, n);
}
int dy_sort_u32(dy_stream_t s, uint32_t *keys, size_t n) { return sort_api<uint32_t>(s, keys, nullptr, n); }
int dy_sort_u64(dy_stream_t s, uint64_t *keys, size_t n) { return sort_api<uint64_t>(s, keys, nullptr, n); }

int dy_reduce_sum_f32(dy_stream_t s, const float *d_data, size_t n, float *out) {
    if (!out) return DY_ERR_INVALID_ARG;
    *out = 0.f;
    if (n == 0) return DY_OK;
    if (!d_data) return DY_ERR_INVALID_ARG;
    const size_t groups = (n + 255) / 256;
    float *d_part = nullptr;
    DY_TRY(hipMallocAsync(reinterpret_cast<void **>(&d_part), groups * sizeof(float), hs(s)));
    reduce_sum_partials<<<static_cast<uint32_t>(groups), 256, 0, hs(s)>>>(d_data, n, d_part);
    DY_LAUNCH_CHECK();
    std::vector<float> h(groups);
    DY_TRY(hipMemcpyAsync(h.data(), d_part, groups * sizeof(float), hipMemcpyDeviceToHost, hs(s)));
    DY_TRY(hipFreeAsync(d_part, hs(s)));
    DY_TRY(hipStreamSynchronize(hs(s)));
    float r = 0.f;
    for (size_t i = 0; i < groups; ++i) r += h[i];
    *out = r;
    return DY_OK;
}

}  // extern "C"
