// Device-wide exclusive scans: the chained scan of the cell-list build
// (cells.hip) and the three-launch scan of the device lattice generator
// (generate.hip).
#pragma once

#include "sph_internal.h"

namespace sph {

// Inclusive scan over a wave; V is unsigned or unsigned long long.
template <class V>
__device__ inline V wave_incl_scan(V v)
{
    const int lane = __lane_id();
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const V t = __shfl_up(v, d, 64);
        if (lane >= d) v += t;
    }
    return v;
}

// Inclusive scan over a 256-thread block; `total` gets the block sum.
template <class V>
__device__ inline V block_incl_scan(V v, V& total)
{
    __shared__ V wsum[4];
    const V w = wave_incl_scan(v);
    const int wid = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 63) wsum[wid] = w;
    __syncthreads();
    V off = 0;
    for (int i = 0; i < wid; ++i) off += wsum[i];
    total = wsum[0] + wsum[1] + wsum[2] + wsum[3];
    __syncthreads();
    return w + off;
}

// Chained scan, one launch (the single-pass scan with decoupled look-back of
// Merrill and Garland, 2016): every block scans its own part and takes the sum
// of the parts before it from their state words.  A state word holds a value
// and, in its top two bits, whether it is the block's own sum or the sum up
// to and including the block; it is written and read as one 64-bit atomic,
// so it needs no fence (values stay below 2^62).  The words and the ticket
// are cleared before the launch.
static constexpr unsigned long long CHAIN_SUM = 1ull << 62, CHAIN_PREFIX = 2ull << 62;
static constexpr unsigned long long CHAIN_VALUE = CHAIN_SUM - 1;

// The block's place in the chain.  Places are handed out in the order in
// which the blocks start, so every block before one that waits is running or
// done, and the wait ends.  Contains a block barrier.
__device__ inline int chain_ticket(unsigned long long* ticket)
{
    __shared__ int place;
    if (threadIdx.x == 0) place = (int)atomicAdd(ticket, 1ull);
    __syncthreads();
    return place;
}

// Sum of the blocks before place b, whose own sum is `sum`; called by one
// whole wave, the same value in every lane.
__device__ inline unsigned long long chain_prefix(unsigned long long* stat, int b,
                                                  unsigned long long sum)
{
    const int lane = __lane_id();
    if (lane == 0)
        __hip_atomic_store(&stat[b], (b == 0 ? CHAIN_PREFIX : CHAIN_SUM) | sum, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    unsigned long long before = 0;
    for (int p = b - 1; p >= 0; p -= 64) {
        // lane l looks at block p - l (blocks before the first: an empty prefix)
        unsigned long long v;
        do {
            v = p - lane >= 0 ? __hip_atomic_load(&stat[p - lane], __ATOMIC_RELAXED,
                                                  __HIP_MEMORY_SCOPE_AGENT)
                              : CHAIN_PREFIX;
        } while (!__all((v & ~CHAIN_VALUE) != 0ull));
        const unsigned long long whole = __ballot((v & CHAIN_PREFIX) != 0ull);
        const int last = whole ? __ffsll((long long)whole) - 1 : 63;
        unsigned long long t = lane <= last ? v & CHAIN_VALUE : 0ull;
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) t += __shfl_xor(t, o);
        before += t;
        if (whole) break;
    }
    if (lane == 0 && b > 0)
        __hip_atomic_store(&stat[b], CHAIN_PREFIX | (before + sum), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    return before;
}

// Scan in three launches: per-block sums, one block scanning the block sums,
// per-block scans plus offset.
static constexpr int SCAN_ITEMS = 16;
static constexpr int SCAN_TILE = 256 * SCAN_ITEMS;

template <class Src>
__global__ __launch_bounds__(256) void k_scan_reduce(Src src, int n, typename Src::V* part)
{
    using V = typename Src::V;
    const int base = blockIdx.x * SCAN_TILE;
    V s = 0;
    for (int it = 0; it < SCAN_ITEMS; ++it) {
        const int i = base + it * 256 + threadIdx.x;
        if (i < n) s += src(i);
    }
    V total;
    block_incl_scan(s, total);
    if (threadIdx.x == 0) part[blockIdx.x] = total;
}

template <class V>
__global__ __launch_bounds__(256) void k_scan_partials(V* part, int nb)
{
    V carry = 0;
    for (int b = 0; b < nb; b += 256) {
        const int i = b + threadIdx.x;
        const V v = i < nb ? part[i] : (V)0;
        V total;
        const V inc = block_incl_scan(v, total);
        if (i < nb) part[i] = carry + inc - v;
        carry += total;
    }
}

// out[i] = exclusive prefix for i < n, out[n] = total.
template <class Src, class O>
__global__ __launch_bounds__(256) void k_scan_down(Src src, int n, const typename Src::V* part,
                                                   O* out)
{
    using V = typename Src::V;
    const int base = blockIdx.x * SCAN_TILE;
    V carry = part[blockIdx.x];
    for (int it = 0; it < SCAN_ITEMS; ++it) {
        const int i = base + it * 256 + threadIdx.x;
        const V v = i < n ? src(i) : (V)0;
        V total;
        const V inc = block_incl_scan(v, total);
        if (i < n) out[i] = (O)(carry + inc - v);
        if (i == n - 1) out[n] = (O)(carry + inc);
        carry += total;
    }
}

template <class Src, class O>
static void scan(sph_system* s, Src src, int n, O* out, typename Src::V* part)
{
    const int nb = (n + SCAN_TILE - 1) / SCAN_TILE;
    k_scan_reduce<<<nb, 256, 0, s->stream>>>(src, n, part);
    k_scan_partials<<<1, 256, 0, s->stream>>>(part, nb);
    k_scan_down<<<nb, 256, 0, s->stream>>>(src, n, part, out);
}


}  // namespace sph
