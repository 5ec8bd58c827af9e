// Stable LSD radix sort of (uint32 key, int32 value) pairs for the LBVH key
// sort (replaces thrust::sort_by_key, bvh.cu:795-807 / 888-894).
//
// One pass per 8-bit digit, three kernels per pass, over tiles of
// kSortTile keys:
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
constexpr int kScanThreads = 256;
static_assert(kTile % kThreads == 0 && kRadix <= kThreads, "sort tile shape");

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
    if (tid < kRadix) counts[(size_t)tid * num_tiles + blockIdx.x] = h[tid];
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

// Block d scans row d of the digit-major count table (exclusive, in place)
// and writes the digit's total count.
__global__ __launch_bounds__(kScanThreads) void k_scan_digit(uint32_t* __restrict__ counts, int num_tiles,
                                                            uint32_t* __restrict__ totals) {
    __shared__ uint32_t sh[kScanThreads];
    const int tid = threadIdx.x;
    uint32_t* row = counts + (size_t)blockIdx.x * num_tiles;
    uint32_t run = 0;
    for (int base = 0; base < num_tiles; base += kScanThreads) {
        const int t = base + tid;
        const uint32_t v = t < num_tiles ? row[t] : 0u;
        sh[tid] = v;
        __syncthreads();
        for (int off = 1; off < kScanThreads; off <<= 1) {
            const uint32_t u = tid >= off ? sh[tid - off] : 0u;
            __syncthreads();
            sh[tid] += u;
            __syncthreads();
        }
        if (t < num_tiles) row[t] = run + sh[tid] - v;
        run += sh[kScanThreads - 1];
        __syncthreads();
    }
    if (tid == 0) totals[blockIdx.x] = run;
}

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
    if (tid < kRadix) {
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
        hipLaunchKernelGGL(k_hist, dim3(num_tiles), dim3(kThreads), 0, ctx->stream, kin, n, shift,
                           counts, num_tiles);
        hipLaunchKernelGGL(k_scan_digit, dim3(kRadix), dim3(kScanThreads), 0, ctx->stream, counts, num_tiles,
                           totals);
        hipLaunchKernelGGL(k_scatter, dim3(num_tiles), dim3(kThreads), 0, ctx->stream, kin, vin,
                           kout, vout, n, shift, counts, totals, num_tiles);
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
