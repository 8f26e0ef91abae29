// radix_sort.hpp -- hand-written LSD radix sort of records on the device, 8-bit digits.
//
// One pass = three launches: k_rs_hist (digit counts of every 2048-record tile, stored
// digit-major), k_rs_scan (exclusive prefix sums of each digit's counts and their totals: with
// the totals of the digits below, where each (digit, tile) starts in the output), k_rs_scatter
// (stable scatter of each tile).  In the scatter, wave w of a tile owns records
// [w * 512, (w + 1) * 512) taken 64 at a time in order; a record's rank among the equal digits
// of its wave is the wave's running count of that digit (LDS) plus the lanes below it with the
// same digit (eight ballots); per-wave prefix sums then place the waves' runs one after another.
// Every pass is stable, so the passes together sort by the digits of the last pass first, ties
// keeping the input order.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <stdexcept>
#include <string>

namespace ifgf
{
namespace radix
{
constexpr int THREADS = 256; // four waves
constexpr int ITEMS = 8;     // records per lane
constexpr int WAVE_SEG = 64 * ITEMS;
constexpr int TILE = THREADS * ITEMS;

// Dig: a functor giving the 8-bit digit (0..255) of a record for the current pass
template <class Rec, class Dig>
__global__ __launch_bounds__(THREADS) void k_rs_hist(const Rec* __restrict__ in, int64_t n,
                                                    Dig dig, uint32_t* __restrict__ counts,
                                                    int nblk)
{
    __shared__ uint32_t h[256];
    h[threadIdx.x] = 0;
    __syncthreads();
    const int64_t base = int64_t(blockIdx.x) * TILE;
    for (int r = 0; r < ITEMS; r++)
    {
        const int64_t i = base + int64_t(r) * THREADS + threadIdx.x;
        if (i < n)
            atomicAdd(&h[dig(in[i])], 1u);
    }
    __syncthreads();
    counts[int64_t(threadIdx.x) * nblk + blockIdx.x] = h[threadIdx.x];
}

// Exclusive prefix sum of v over the workgroup's 256 threads; *total = the sum over all of them.
// s: 4 words of LDS.
__device__ __forceinline__ uint32_t block_scan(uint32_t v, uint32_t* s, uint32_t* total)
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint32_t x = v;
    for (int off = 1; off < 64; off <<= 1)
    {
        const uint32_t y = uint32_t(__shfl_up(int(x), off));
        if (lane >= off)
            x += y;
    }
    __syncthreads();
    if (lane == 63)
        s[w] = x;
    __syncthreads();
    uint32_t base = 0, all = 0;
    for (int k = 0; k < THREADS / 64; k++)
    {
        base += k < w ? s[k] : 0u;
        all += s[k];
    }
    *total = all;
    return base + x - v;
}

// Exclusive prefix sum of one digit's tile counts in place, a workgroup per digit, 256 tiles a
// step; totals[digit] = the digit's count.  The sum over the digits below is left to the scatter
// (256 totals, one per thread), so the digits need not wait for one another.  Latency-bound: one
// workgroup with a contiguous run of all 256 nblk counts per thread read them a cache line per
// lane: 371 us a pass over 1M records, now 4.8 us; at 262,144 points (2.7 us a pass) the
// octrees take 10.7 -> 9.2 ms and the interaction lists 11.4 -> 9.5 ms.
template <int UNUSED = 0>
__global__ __launch_bounds__(THREADS) void k_rs_scan(uint32_t* __restrict__ c, int nblk,
                                                    uint32_t* __restrict__ totals)
{
    __shared__ uint32_t s[THREADS / 64];
    uint32_t* const row = c + int64_t(blockIdx.x) * nblk;
    uint32_t run = 0;
    for (int i0 = 0; i0 < nblk; i0 += THREADS)
    {
        const int i = i0 + int(threadIdx.x);
        const uint32_t v = i < nblk ? row[i] : 0u;
        uint32_t total;
        const uint32_t x = block_scan(v, s, &total);
        if (i < nblk)
            row[i] = run + x;
        run += total;
    }
    if (threadIdx.x == 0)
        totals[blockIdx.x] = run;
}

template <class Rec, class Dig>
__global__ __launch_bounds__(THREADS) void k_rs_scatter(const Rec* __restrict__ in,
                                                       Rec* __restrict__ out, int64_t n, Dig dig,
                                                       const uint32_t* __restrict__ offs,
                                                       const uint32_t* __restrict__ totals,
                                                       int nblk)
{
    __shared__ uint32_t cnt[THREADS / 64][256];
    __shared__ uint32_t gofs[256];
    __shared__ uint32_t s_scan[THREADS / 64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    for (int i = threadIdx.x; i < (THREADS / 64) * 256; i += THREADS)
        (&cnt[0][0])[i] = 0;
    uint32_t all;
    gofs[threadIdx.x] = block_scan(totals[threadIdx.x], s_scan, &all) +
                        offs[int64_t(threadIdx.x) * nblk + blockIdx.x];
    __syncthreads();
    const int64_t seg = int64_t(blockIdx.x) * TILE + int64_t(w) * WAVE_SEG;
    const uint64_t below_me = (uint64_t(1) << lane) - 1;
    Rec rec[ITEMS];
    uint32_t dg[ITEMS], rk[ITEMS];
#pragma unroll
    for (int r = 0; r < ITEMS; r++)
    {
        const int64_t i = seg + int64_t(r) * 64 + lane;
        const bool valid = i < n;
        uint32_t d = 0;
        if (valid)
        {
            rec[r] = in[i];
            d = dig(rec[r]);
        }
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; b++)
        {
            const bool set = (d >> b) & 1u;
            const uint64_t m = __ballot(set);
            peers &= set ? m : ~m;
        }
        dg[r] = d;
        rk[r] = 0;
        if (valid)
        {
            const uint32_t below = uint32_t(__popcll(peers & below_me));
            const uint32_t base = cnt[w][d];
            rk[r] = base + below;
            if (below == 0)
                cnt[w][d] = base + uint32_t(__popcll(peers));
        }
    }
    __syncthreads();
    {
        const int d = threadIdx.x;
        uint32_t s = 0;
        for (int v = 0; v < THREADS / 64; v++)
        {
            const uint32_t t = cnt[v][d];
            cnt[v][d] = s;
            s += t;
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ITEMS; r++)
    {
        const int64_t i = seg + int64_t(r) * 64 + lane;
        const int64_t pos = int64_t(gofs[dg[r]]) + cnt[w][dg[r]] + rk[r];
        if (i < n && pos < n)
            out[pos] = rec[r];
    }
}

// Sort n records of a by passes digits (digit_of_pass(p) gives the functor of pass p, least
// significant first), b as the ping-pong buffer and counts as scratch of counts_needed(n)
// words.  Returns the buffer holding the result (a or b).
inline int64_t counts_needed(int64_t n)
{
    return int64_t(256) * ((n + TILE - 1) / TILE) + 256; // per (digit, tile), then per digit
}

template <class Rec, class DigitOfPass>
Rec* sort(Rec* a, Rec* b, int64_t n, int passes, const DigitOfPass& digit_of_pass,
          uint32_t* counts, hipStream_t st)
{
    if (n <= 1)
        return a;
    const int nblk = int((n + TILE - 1) / TILE);
    uint32_t* const totals = counts + int64_t(256) * nblk;
    for (int p = 0; p < passes; p++)
    {
        const auto dig = digit_of_pass(p);
        k_rs_hist<<<nblk, THREADS, 0, st>>>(a, n, dig, counts, nblk);
        k_rs_scan<><<<256, THREADS, 0, st>>>(counts, nblk, totals);
        k_rs_scatter<<<nblk, THREADS, 0, st>>>(a, b, n, dig, counts, totals, nblk);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess)
            throw std::runtime_error(std::string("radix sort: ") + hipGetErrorString(e));
        std::swap(a, b);
    }
    return a;
}

} // namespace radix
} // namespace ifgf
