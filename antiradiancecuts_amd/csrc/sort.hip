// Stable LSD radix sort of (uint32 key, int32 value) pairs for the LBVH key
// sort (replaces thrust::sort_by_key, bvh.cu:795-807 / 888-894).
//
// One pass per 8-bit digit, three kernels per pass (two over few tiles), over
// tiles of kSortTile keys:
//   hist    — each 512-thread block counts the digits of its tile; lanes
//             with equal digits are found with 8 wave ballots, so only one
//             lane per (wave, digit) touches LDS.
//   scan    — one block per digit turns its row of tile counts into an
//             exclusive prefix and records the digit total.
//   scatter — each block sorts its tile by the digit in LDS, then writes it
//             out: the tile's keys of one digit go to one contiguous run of
//             the output, so consecutive threads write consecutive
//             addresses.  A key's place in its digit's run: keys of that
//             digit in earlier waves + earlier in its wave + in earlier
//             lanes (ballot match), so equal digits keep their input order
//             and the sort is stable.  With the tile's keys read a round of
//             512 at a time, three barriers each and two scans of 16, the
//             scatter of 1M pairs took 15.4 us and of 131071 11.4, 10.4 and 6.2 here.
#include "arc_internal.hpp"

namespace {

constexpr int kThreads = 512;
constexpr int kWaves = kThreads / 64;
constexpr int kTile = arc::kSortTile;
constexpr int kItems = kTile / kThreads;
constexpr int kRadix = arc::kSortRadix;
constexpr int kScanThreads = 512;
static_assert(kTile % kThreads == 0 && 2 * kRadix == kThreads, "sort tile shape");

// Up to this many tiles the scatter adds the tiles' counts up itself, a row of
// 256 per tile, instead of a scan kernel between: tiles loads per digit and
// block against a launch.  Builds over random points, with the sums and with
// the scan: 5000 points 68 us and 78, 65536 78 and 87, 131072 (64 tiles) 88 and
// 92, 196608 97 and 98, 262144 105 and 103, 1M 221 and 174.
constexpr int kFewTiles = 64;

__device__ inline uint64_t match_digit(uint64_t active, uint32_t digit) {
    uint64_t m = active;
#pragma unroll
    for (int b = 0; b < 8; ++b) {
        const bool bit = (digit >> b) & 1u;
        const uint64_t bb = __ballot(bit);
        m &= bit ? bb : ~bb;
    }
    return m;
}

template <bool kFew>
__global__ __launch_bounds__(kThreads) void k_hist(const uint32_t* __restrict__ keys, int n, int shift,
                                                   uint32_t* __restrict__ counts, int num_tiles) {
    __shared__ uint32_t h[kRadix];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    if (tid < kRadix) h[tid] = 0;
    __syncthreads();
    const int base = blockIdx.x * kTile;
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
        const int idx = base + j * kThreads + tid;
        const bool valid = idx < n;
        const uint32_t digit = valid ? (keys[idx] >> shift) & 0xffu : 0u;
        const uint64_t m = match_digit(__ballot(valid), digit);
        const uint64_t lower = m & ((1ull << lane) - 1ull);
        if (valid && lower == 0ull) atomicAdd(&h[digit], (uint32_t)__popcll(m));
    }
    __syncthreads();
    if (tid < kRadix) counts[kFew ? (size_t)blockIdx.x * kRadix + tid : (size_t)tid * num_tiles + blockIdx.x] = h[tid];
}

// Exclusive scan of one value per thread over the first kRadix threads (whole
// waves; all the block's threads call it).  sums: one word per wave of them.
__device__ inline uint32_t radix_exclusive_scan(uint32_t v, uint32_t* sums) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t x = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t u = __shfl_up(x, off);
        if (lane >= off) x += u;
    }
    if (lane == 63 && wave < kRadix / 64) sums[wave] = x;
    __syncthreads();
    uint32_t before = 0;
    for (int w = 0; w < min(wave, kRadix / 64); ++w) before += sums[w];
    return before + x - v;
}

// Thread tid's digit tid % kRadix in every second tile from tid / kRadix on:
// the digit's keys in those before `tile` and in all of them.  Sixteen loads
// are in flight at a time.
__device__ inline void sum_tiles(const uint32_t* __restrict__ counts, int tile, int num_tiles, uint32_t& before,
                                 uint32_t& all) {
    const int d = threadIdx.x % kRadix;
    before = all = 0;
    for (int t0 = threadIdx.x / kRadix; t0 < num_tiles; t0 += 32) {
        uint32_t c[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) c[j] = t0 + 2 * j < num_tiles ? counts[(size_t)(t0 + 2 * j) * kRadix + d] : 0u;
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            all += c[j];
            before += t0 + 2 * j < tile ? c[j] : 0u;
        }
    }
}

// Block d scans row d of the digit-major count table (exclusive, in place)
// and writes the digit's total count.  Bound by latency: the scan is in
// registers per wave and one barrier per 512 tiles joins the waves (with a
// scan in LDS of 16 barriers per 256 tiles a build over 1M points took 173.6
// us, 168.2 here).
__global__ __launch_bounds__(kScanThreads) void k_scan_digit(uint32_t* __restrict__ counts, int num_tiles,
                                                            uint32_t* __restrict__ totals) {
    __shared__ uint32_t sums[2][kScanThreads / 64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    uint32_t* row = counts + (size_t)blockIdx.x * num_tiles;
    uint32_t run = 0;
    for (int base = 0, k = 0; base < num_tiles; base += kScanThreads, k ^= 1) {
        const int t = base + tid;
        const uint32_t v = t < num_tiles ? row[t] : 0u;
        uint32_t x = v;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const uint32_t u = __shfl_up(x, off);
            if (lane >= off) x += u;
        }
        if (lane == 63) sums[k][wave] = x;
        __syncthreads();  // two sets of sums: the next round's writes are a barrier behind this one's reads
        uint32_t before = 0, all = 0;
#pragma unroll
        for (int w = 0; w < kScanThreads / 64; ++w) {
            const uint32_t c = sums[k][w];
            before += w < wave ? c : 0u;
            all += c;
        }
        if (t < num_tiles) row[t] = run + before + x - v;
        run += all;
    }
    if (tid == 0) totals[blockIdx.x] = run;
}

// kFew: offsets are k_hist's counts, a row per tile; else the scanned table, a
// row per digit, and totals.
template <bool kFew>
__global__ __launch_bounds__(kThreads) void k_scatter(const uint32_t* __restrict__ keys_in,
                                                      const int* __restrict__ vals_in,
                                                      uint32_t* __restrict__ keys_out,
                                                      int* __restrict__ vals_out, int n, int shift,
                                                      const uint32_t* __restrict__ offsets,
                                                      const uint32_t* __restrict__ totals, int num_tiles) {
    __shared__ uint32_t s_keys[kTile];
    __shared__ int s_vals[kTile];
    __shared__ uint32_t out_start[kRadix];      // output place of a digit's keys minus their place in the tile
    __shared__ uint32_t wcount[kWaves][kRadix];  // keys of each digit per wave, then where the wave's start in the tile
    __shared__ uint32_t sums[2][kRadix / 64];
    __shared__ uint2 odd[kFew ? kRadix : 1];  // the second half's sums of sum_tiles
    const int tid = threadIdx.x;
    const int wave = tid >> 6;
    const int lane = tid & 63;
    const int tile = blockIdx.x;
    const int base = tile * kTile;
    const int tile_n = min(kTile, n - base);
    // 1. the tile sorted by digit into LDS, stably: a wave's keys are kItems
    // times 64 consecutive ones, all read before the first is ranked, and
    // ranked within the wave without a barrier
    const int first = wave * 64 * kItems + lane;
    uint32_t key[kItems], rank[kItems];
    int val[kItems];
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
        const int i = first + 64 * j;
        key[j] = i < tile_n ? keys_in[base + i] : 0u;
        val[j] = i < tile_n ? vals_in[base + i] : 0;
    }
    uint32_t off = 0, total = 0;
    if constexpr (kFew) {
        sum_tiles(offsets, tile, num_tiles, off, total);
        if (tid >= kRadix) odd[tid - kRadix] = make_uint2(off, total);
    } else if (tid < kRadix) {
        // the tile's place within each digit (the scanned count table)
        off = offsets[(size_t)tid * num_tiles + tile];
        total = totals[tid];
    }
    for (int d = lane; d < kRadix; d += 64) wcount[wave][d] = 0;
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
        const bool valid = first + 64 * j < tile_n;
        const uint32_t digit = (key[j] >> shift) & 0xffu;
        const uint64_t m = match_digit(__ballot(valid), digit);
        const uint64_t lower = m & ((1ull << lane) - 1ull);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        const uint32_t before = wcount[wave][digit];
        rank[j] = before + (uint32_t)__popcll(lower);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (valid && lower == 0ull) wcount[wave][digit] = before + (uint32_t)__popcll(m);
    }
    __syncthreads();
    uint32_t mine = 0, count[kWaves];
    if (tid < kRadix) {
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            count[w] = wcount[w][tid];
            mine += count[w];
        }
        if constexpr (kFew) {
            off += odd[tid].x;
            total += odd[tid].y;
        }
    }
    const uint32_t digit_base = radix_exclusive_scan(total, sums[0]);
    const uint32_t local = radix_exclusive_scan(mine, sums[1]);
    if (tid < kRadix) {
        out_start[tid] = digit_base + off - local;
        uint32_t at = local;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            wcount[w][tid] = at;
            at += count[w];
        }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
        if (first + 64 * j >= tile_n) continue;
        const uint32_t pos = wcount[wave][(key[j] >> shift) & 0xffu] + rank[j];
        s_keys[pos] = key[j];
        s_vals[pos] = val[j];
    }
    __syncthreads();
    // 2. out in LDS order: consecutive threads, consecutive places of one run
    for (int i = tid; i < tile_n; i += kThreads) {
        const uint32_t key = s_keys[i];
        const uint32_t digit = (key >> shift) & 0xffu;
        const uint32_t pos = out_start[digit] + (uint32_t)i;
        keys_out[pos] = key;
        vals_out[pos] = s_vals[i];
    }
}

}  // namespace

namespace arc {

int sort_pairs(arc_ctx* ctx, SortScratch& s, uint32_t* keys, int* vals, int n, int key_bits) {
    if (n <= 1) return ARC_OK;
    const int num_tiles = (n + kTile - 1) / kTile;
    ARC_TRY(ensure(ctx, s.keys_alt, sizeof(uint32_t) * (size_t)n));
    ARC_TRY(ensure(ctx, s.vals_alt, sizeof(int) * (size_t)n));
    ARC_TRY(ensure(ctx, s.counts, sizeof(uint32_t) * sort_counts_size((size_t)n)));
    const int passes = (key_bits + 7) / 8;
    uint32_t* kin = keys;
    int* vin = vals;
    uint32_t* kout = s.keys_alt.as<uint32_t>();
    int* vout = s.vals_alt.as<int>();
    uint32_t* counts = s.counts.as<uint32_t>();
    uint32_t* totals = counts + (size_t)kRadix * num_tiles;
    for (int p = 0; p < passes; ++p) {
        const int shift = 8 * p;
        if (num_tiles <= kFewTiles) {
            hipLaunchKernelGGL(k_hist<true>, dim3(num_tiles), dim3(kThreads), 0, ctx->stream, kin, n, shift,
                               counts, num_tiles);
            hipLaunchKernelGGL(k_scatter<true>, dim3(num_tiles), dim3(kThreads), 0, ctx->stream, kin, vin,
                               kout, vout, n, shift, counts, totals, num_tiles);
        } else {
            hipLaunchKernelGGL(k_hist<false>, dim3(num_tiles), dim3(kThreads), 0, ctx->stream, kin, n, shift,
                               counts, num_tiles);
            hipLaunchKernelGGL(k_scan_digit, dim3(kRadix), dim3(kScanThreads), 0, ctx->stream, counts, num_tiles,
                               totals);
            hipLaunchKernelGGL(k_scatter<false>, dim3(num_tiles), dim3(kThreads), 0, ctx->stream, kin, vin,
                               kout, vout, n, shift, counts, totals, num_tiles);
        }
        ARC_LAUNCHED(ctx);
        std::swap(kin, kout);
        std::swap(vin, vout);
    }
    if (kin != keys) {  // odd number of passes: copy the result back
        ARC_HIP(ctx, hipMemcpyAsync(keys, kin, sizeof(uint32_t) * (size_t)n, hipMemcpyDeviceToDevice,
                                    ctx->stream));
        ARC_HIP(ctx, hipMemcpyAsync(vals, vin, sizeof(int) * (size_t)n, hipMemcpyDeviceToDevice,
                                    ctx->stream));
    }
    return ARC_OK;
}

}  // namespace arc
