// Pair-interaction kernels (shared device code of pair64.hip and pair32.hip):
// the device form of _apply_binary! /
// apply_binary! (src/core.jl:94-129) for the registered operators.
//
// Work decomposition.  A tile is up to T targets of one cell (T = 8..64, a
// template parameter).  One 64-lane wave handles a tile: lane = (target t,
// slice s), t = lane % T, s = lane / T, with S = 64 / T slices.
//
// Candidates.  The candidates of a target are the cells key + key_diff of
// the reference; with di innermost, each of the 3 (2D) or 9 (3D) (dj, dk)
// rows is the contiguous cell range [key + L1*dj + L1*L2*dk - 1, ... + 1],
// clamped to [0, key_max) exactly as the reference's linear bounds test
// (src/core.jl:98), so rows wrap and small grids visit aliased cells as
// often as the reference does.  Since the particles are cell-sorted, each
// row is one contiguous particle range (periodic systems: at most two, with
// an image shift each).  All targets of a tile share the cell, hence the
// ranges: the tile's candidate list is the concatenation of its ranges.
//
// Culling.  Only the candidates within reach of the tile -- squared
// distance to the bounding box of its targets not above the predicate's
// threshold -- can be accepted by any target, about half of the list in 3D.
// The list is streamed in 64-candidate steps; each step appends its kept
// candidates (ballot + lane rank) to a ring of 128 LDS slots, and every 64
// kept candidates form a chunk.  The kept order is the list order, and the
// box and the cull test are the same in every pass, so all passes see the
// same chunks.  The testing pass also records each tile's kept candidates
// (and their ranges, for the image shifts of periodic systems); a pass that
// loads its masks reads that list instead of streaming and culling again,
// one chunk per step, so its ring holds a single chunk (64 slots).
//
// Each chunk is handled in two phases:
//   1. mask: the matrix cores (T >= 32, candidate test below) or lane
//      (t, s) itself test the chunk slots s + S*j (j < T) against target t
//      and set bit j of the lane's T-bit mask for slot s + S*j -- or, after
//      a density pass on the same cell list, the lane loads that pass's mask.
//      Interleaving the slices keeps the accepted counts of the lanes
//      alike (neighbouring slots are neighbouring particles);
//   2. interact: the chunk's accepted pairs are cut into runs spread over
//      all 64 lanes (balanced pairs, below), so the pair arithmetic runs
//      once per accepted pair, not once per candidate.
// At the end the S slices of a target are combined with wave shuffles.
// The masks of target t for a chunk form one 64-bit word (the T-bit mask
// of slice s in bits [s*T, s*T + T)), stored at
// mask_base(tile) + chunk * T + t.
//
// Predicate (src/core.jl:104-105, src/algebra.jl:49-60): accept q != p when
// RN(sqrt((d1*d1 + d2*d2) + d3*d3)) <= h.  sqrt is correctly rounded and
// monotonic, so this equals s <= s_thr with s_thr = max{s : RN(sqrt(s)) <= h}
// (computed on the host).  The FP64 kernels evaluate s without FMA
// (-ffp-contract=off), i.e. bit-exactly as the reference.  With T >= 32 both
// modes filter on the matrix cores and settle the close pairs by that exact
// test.  With T = 16 and 8 the mixed kernels evaluate |q|^2 - 2 p.q + |p|^2 in FP32 on tile-relative
// coordinates (three FMAs per candidate): below s_thr (1 - BAND) the pair is
// accepted, above s_thr (1 + BAND) rejected, and in between the exact FP64
// test decides, so their neighbour sets (and masks) are the reference's
// too.  The box test never drops a candidate that the predicate accepts:
// in FP64 each box distance component is a correctly rounded difference no
// larger than the target's, and the mixed test uses the same guard band.
// The identity exclusion p != q is applied once per chunk to the slots that
// hold p: the tile's own targets are always kept, so each occurrence of the
// tile's cell in the list puts them in consecutive slots.
#pragma once

#include <type_traits>

#include "device_cache.h"
#include "sph_internal.h"

namespace sph {

#define COL(c, f, i) ((c).cols[(long long)(f) * (c).cap + (i)])

// Guard band of the mixed predicate, relative to s_thr.  Tile-relative
// coordinates are below 4 h in magnitude; the FP32 expanded form
// |q|^2 - 2 p.q + |p|^2 is then within ~1e-5 * h^2 of the exact squared
// distance and the direct form within ~1e-6 * h^2; the band is 10x wider.
static constexpr double BAND = 1.0e-4;

// The wave's copy of the counters.
__device__ inline int counter_slot() { return (int)(blockIdx.x % CNT_COPIES) * CNT_STRIDE; }

__device__ inline void count_pairs(const PairCtx& c, unsigned n)
{
    // wave reduction of the per-lane counts, one atomic per wave
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) n += __shfl_xor(n, o);
    if (__lane_id() == 0 && n)
        atomicAdd(c.pair_counter + counter_slot(), (unsigned long long)n);
}

// The wave's distance tests (the same value in every lane).
__device__ inline void count_tests(const PairCtx& c, unsigned long long n)
{
    if (c.test_counter && __lane_id() == 0 && n) atomicAdd(c.test_counter + counter_slot(), n);
}

// Tile queues.  The tile range [0, ntiles) is cut into NQUEUE contiguous
// parts, one per queue head.  Block b belongs to queue b % NQUEUE (the XCD
// it runs on, so neighbouring tiles share that XCD's L2).  The first tiles
// of a queue are dealt out to its blocks without an atomic (block b takes
// the (b / NQUEUE)-th share); the rest are taken qgrab at a time from the
// queue head, and when its queue is empty a wave moves on to the others.
// Only blocks that run at once may be dealt tiles -- a block that starts
// when others leave would begin its share after all the rest -- so the grid
// is what the chip holds (launch_resident; otherwise the force pass of a
// 518k-particle collapse step takes 643 instead of 451 us).
// An atomic on one head takes ~10.5 ns, one after the other: with every
// tile behind an atomic, and every idle wave trying all heads, a pass took
// 86 us however little it had to do (8192 waves on 8 heads; a 2D dam break of
// 6514 particles: 13.6 -> 7.2 ms per 50 steps).  A queue whose tiles are all dealt
// out is not touched, and the wave that first finds a queue empty says so in
// the set's mask, which the others read when their queue runs out: one read
// each instead of up to seven failing atomics (97k-particle 2D dam break with
// T = 16, a little more than one tile per wave: 266 -> 165 us per step; 333k
// with T = 32: 306 -> 246).  (Reading another queue's head
// before trying it made the waves that help slower: the force pass of the
// 5.75M-particle dam break took 3.25 instead of 3.06 ms.)
// With one tile per grab the tiles in flight on an XCD are consecutive and
// share their neighbour cells in the L2 (3D: 9.6 instead of 10.6 ms per
// dam-break step); the short 2D tiles take four per grab, which spares
// atomics.
// Every wave leaves once all queues are past their ends.  The state is
// wave-uniform (readfirstlane), so the tile record, the system id and the
// system's parameters are scalar loads held in SGPRs.
struct TileCursor {
    int k;         // queue in use, counted from the own one
    int cur, end;  // tiles in hand
    int deal;      // tiles each block is dealt
};

__device__ inline int queue_lo(int ntiles, int q) { return (int)((long long)ntiles * q / NQUEUE); }

// Tiles of queue q dealt out to its blocks.
__device__ inline int queue_dealt(const TileCursor& tc, int q)
{
    return (int)((gridDim.x + NQUEUE - 1 - q) / NQUEUE) * tc.deal;
}

__device__ inline void tile_cursor_init(const PairCtx& c, int ntiles, TileCursor& tc)
{
    // few tiles: one each, so that every block gets one before any gets two
    tc.deal = (long long)gridDim.x * c.qgrab <= ntiles ? c.qgrab : 1;
    tc.k = 0;
    const int q = (int)(blockIdx.x % NQUEUE);
    const int hi = queue_lo(ntiles, q + 1);
    tc.cur = min(hi, queue_lo(ntiles, q) + (int)(blockIdx.x / NQUEUE) * tc.deal);
    tc.end = min(hi, tc.cur + tc.deal);
}

__device__ inline int next_tile(const PairCtx& c, int ntiles, TileCursor& tc)
{
    if (tc.cur < tc.end) return tc.cur++;
    int* mask = &c.queue[NQUEUE * QSTRIDE];
    unsigned empty = 0;
    for (; tc.k < NQUEUE; ++tc.k) {
        const int q = (int)((blockIdx.x + tc.k) % NQUEUE);
        const int dealt = queue_dealt(tc, q);
        const int lo = queue_lo(ntiles, q) + dealt, hi = queue_lo(ntiles, q + 1);
        if (lo >= hi || ((empty >> q) & 1u)) continue;
        int start = 0;
        if (__lane_id() == 0) start = atomicAdd(&c.queue[q * QSTRIDE], c.qgrab);
        start = __builtin_amdgcn_readfirstlane(start);
        if (start < hi - lo) {
            tc.cur = lo + start;
            tc.end = min(hi, lo + start + c.qgrab);
            return tc.cur++;
        }
        int seen = 0;
        if (__lane_id() == 0) {
            if (start < hi - lo + c.qgrab) atomicOr(mask, 1 << q);  // the first to find it empty
            seen = __hip_atomic_load(mask, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        empty = (unsigned)__builtin_amdgcn_readfirstlane(seen);
    }
    return ntiles;
}

__device__ inline long long mask_base(const int4& td)
{
    return (long long)(unsigned)td.z | ((long long)td.w << 32);
}

// m * 2 + (e <= thr): the predicate shifted into a mask, as one compare
// into VCC and one add with carry (the compiler would spend a select, a
// shift and an OR per bit).  NaN compares false, as e <= thr does.
__device__ inline unsigned shift_in_le(unsigned m, float e, float thr)
{
    unsigned r;
    asm("v_cmp_ge_f32_e32 vcc, %2, %3\n\tv_addc_co_u32_e32 %0, vcc, %1, %1, vcc"
        : "=v"(r)
        : "v"(m), "v"(thr), "v"(e)
        : "vcc");
    return r;
}

__device__ inline unsigned shift_in_le(unsigned m, double e, double thr)
{
    unsigned r;
    asm("v_cmp_ge_f64_e32 vcc, %2, %3\n\tv_addc_co_u32_e32 %0, vcc, %1, %1, vcc"
        : "=v"(r)
        : "v"(m), "v"(thr), "v"(e)
        : "vcc");
    return r;
}

// Per-lane mask of T slots.
template <int T>
using MaskT = typename std::conditional<(T > 32), unsigned long long, unsigned>::type;

template <int T>
__device__ inline int lowest_bit(MaskT<T> m)
{
    if constexpr (T > 32) return __ffsll((long long)m) - 1;
    else return __ffs(m) - 1;
}

// ------------------------------------------------- matrix-core candidate test --
// The test of a chunk's 64 slots against the tile's targets, for T = 64 and
// 32, as a product on the matrix cores: with the target p and the candidate
// q relative to the centre of the targets' box,
//     D = |q|^2 - 2 p.q + (|p|^2 - h^2)
// is a sum of 16 products of 16-bit floats once every coordinate, |q|^2 and
// |p|^2 - h^2 are split into a high and a low half (11 + 11 bits): four
// products per axis, two for |q|^2, two for |p|^2 - h^2.  That is one
// v_mfma_f32_32x32x16_f16 per 32 x 32 block (32 cycles), and the sign of D is
// the answer: one v_alignbit shifts it into the lane's mask.  Per chunk and
// lane that is ~150 vector instructions where three FMAs and two compares
// with carry per test took 448, and no LDS read per test.
//
// D is only a filter.  Coordinates are scaled by a power of two to
// 512 <= h < 1024, so no half overflows or loses bits to underflow.  Its error:
// two halves of 11 bits, both cut, keep 2^-21 of a value; the sum of 16 products
// in FP32 loses at most 16 * 2^-23 of its largest partial sum.  Relative to the
// centre of a box no wider than a cell, a pair near the threshold has
// |q|^2 + 2|p||q| <= 6.8 h^2 with cells of h and <= 9.7 h^2 with the cells of up
// to 4/3 h of a periodic box three cells wide, so the error is below 2.1e-5 h^2
// and below 3.0e-5 h^2 (the products 3e-6 and 5e-6, |q|^2 and the FP32 roundings
// of its terms 4e-6, the rest the sum).  That is the worst case of every rounding
// at once: an emulation over 2.4e7 pairs, half of them from the corners outwards,
// gave 3.8e-6.
// A pair with |D| below TEST_BAND h^2 (above both) is settled by the exact
// FP64 predicate, as in the FP32 test; found by a minimum over the lane's 16
// values per block, and looked for bit by bit only in blocks that hold one
// (about one in twenty).  So the masks are the reference's sets, bit for bit
// what they were.
//
// Layout: acc[i] of lane l holds row 8 (i / 4) + 4 (l / 32) + i % 4 (the
// candidate, operand A) and column l % 32 (the target, operand B); an operand
// lane l holds elements 8 (l / 32) ... + 7 of row l % 32.  Each lane splits
// one slot (and, once per tile, one target) into eight packed registers, the
// first four for l < 32; v_permlane32_swap of register i with i + 4 gives
// both 32-row operands.  Lane l takes slot test_slot(l), so that the bits
// come out in the order of the masks.
//
// Density pass of the 5.75M-particle dam break: 3.79 -> 3.34 ms (mixed);
// of a 1.5M-particle one in FP64: 2.86 -> 2.20 ms.  T = 16 and 8 would leave
// half or more of the columns empty and keep the vector test.
static constexpr double TEST_BAND = 4.0e-5;

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float acc16_t __attribute__((ext_vector_type(16)));
typedef __fp16 half2_t __attribute__((ext_vector_type(2)));

// (a, b) as packed 16-bit floats, rounded towards zero, and what that left.
__device__ inline unsigned split_pair(float a, float b, unsigned& rest)
{
    const half2_t h = __builtin_amdgcn_cvt_pkrtz(a, b);
    const half2_t r = __builtin_amdgcn_cvt_pkrtz(a - (float)h[0], b - (float)h[1]);
    rest = __builtin_bit_cast(unsigned, r);
    return __builtin_bit_cast(unsigned, h);
}

__device__ inline half8_t as_half8(const unsigned* r)
{
    struct R {
        unsigned v[4];
    } t = {{r[0], r[1], r[2], r[3]}};
    return __builtin_bit_cast(half8_t, t);
}

static constexpr unsigned HALF2_256 = 0x5c005c00u;  // (256, 256)

// Slot of the chunk whose candidate lane l holds.
template <int T>
__device__ inline int test_slot(int l)
{
    const int hf = (l >> 2) & 1, b = (l >> 5) * 16 + ((l >> 3) & 3) * 4 + (l & 3);
    return T == 64 ? hf * 32 + b : hf + 2 * b;
}

template <int T>
struct TestTile {
    half8_t p[T / 32];  // targets, 32 rows each
    float band;
};

// x, y, z: the lane's target (lane % T), relative to the centre and scaled;
// hs: h scaled.
template <int T>
__device__ inline void test_targets(TestTile<T>& tt, int lane, float x, float y, float z, float hs)
{
    const float w = (fmaf(z, z, fmaf(y, y, x * x)) - hs * hs) * (1.0f / 256.0f);
    unsigned r[8], zw, zwl;
    r[0] = split_pair(-2.0f * x, -2.0f * y, r[1]);
    zw = split_pair(-2.0f * z, w, zwl);
    r[2] = r[0];
    r[3] = r[1];
    r[4] = (zw & 0xffffu) | (HALF2_256 & 0xffff0000u);  // (z, 256)
    r[5] = r[4];
    r[6] = (zwl & 0xffffu) | (zwl << 16);               // (z low, z low)
    r[7] = (zw >> 16) | (zwl & 0xffff0000u);            // (w, w low)
    if constexpr (T == 64) {
        unsigned a[4], b[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const auto s = __builtin_amdgcn_permlane32_swap(r[i], r[i + 4], false, false);
            a[i] = s[0];
            b[i] = s[1];
        }
        tt.p[0] = as_half8(a);
        tt.p[1] = as_half8(b);
    } else {
        unsigned a[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) a[i] = lane < 32 ? r[i] : r[i + 4];
        tt.p[0] = as_half8(a);
    }
    tt.band = (float)TEST_BAND * hs * hs;
}

// x, y, z: the candidate in slot test_slot(lane), relative to the centre and
// scaled; pad: the slot is past the end of the list.  m: the lane's mask of
// accepted slots (of target lane % T; bit j of slice s is slot s + (64/T) j),
// unsure: those the exact test has to settle.
template <int T>
__device__ inline void test_chunk(const TestTile<T>& tt, float x, float y, float z, bool pad,
                                  MaskT<T>& m, MaskT<T>& unsure)
{
    x = pad ? 0.0f : x;
    y = pad ? 0.0f : y;
    z = pad ? 0.0f : z;
    const float q2 = pad ? 60000.0f : fmaf(z, z, fmaf(y, y, x * x)) * (1.0f / 256.0f);
    unsigned r[8];
    r[0] = split_pair(x, y, r[2]);
    r[1] = r[0];
    r[3] = r[2];
    r[4] = split_pair(z, q2, r[5]);
    r[6] = (r[4] & 0xffffu) | (r[5] << 16);  // (z, z low)
    r[7] = HALF2_256;
    half8_t q[2];
    {
        unsigned a[4], b[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const auto s = __builtin_amdgcn_permlane32_swap(r[i], r[i + 4], false, false);
            a[i] = s[0];
            b[i] = s[1];
        }
        q[0] = as_half8(a);
        q[1] = as_half8(b);
    }
    unsigned mm[T / 32], uu[T / 32];
#pragma unroll
    for (int k = 0; k < T / 32; ++k) mm[k] = uu[k] = 0;
    bool any = false;
#pragma unroll
    for (int cb = 1; cb >= 0; --cb)
#pragma unroll
        for (int k = 0; k < T / 32; ++k) {
            acc16_t d = {};
            d = __builtin_amdgcn_mfma_f32_32x32x16_f16(q[cb], tt.p[k], d, 0, 0, 0);
            float near = fabsf(d[0]);
#pragma unroll
            for (int i = 15; i >= 0; --i)
                mm[k] = __builtin_amdgcn_alignbit(mm[k], __float_as_uint(d[i]), 31);
#pragma unroll
            for (int i = 1; i < 15; i += 2) near = fminf(fminf(fabsf(d[i]), fabsf(d[i + 1])), near);
            near = fminf(fabsf(d[15]), near);
            // one block's 16 results at a time: without this the compiler
            // keeps the four blocks' 64 live and spills (+70 registers)
            asm volatile("" : "+v"(mm[k]), "+v"(near));
            uu[k] <<= 16;
            if (__any(near < tt.band)) {
                any = true;
                unsigned u = 0;
#pragma unroll
                for (int i = 15; i >= 0; --i) u = u * 2 + (fabsf(d[i]) < tt.band ? 1u : 0u);
                uu[k] |= u;
            }
        }
    if constexpr (T == 64) {
        const auto s = __builtin_amdgcn_permlane32_swap(mm[0], mm[1], false, false);
        m = (MaskT<T>)s[0] | ((MaskT<T>)s[1] << 32);
        unsure = 0;
        if (any) {
            const auto v = __builtin_amdgcn_permlane32_swap(uu[0], uu[1], false, false);
            unsure = (MaskT<T>)v[0] | ((MaskT<T>)v[1] << 32);
        }
    } else {
        m = mm[0];
        unsure = uu[0];
    }
    m &= ~unsure;
}

// Whether a tile's box is wider than the filter's error bound covers.  Positions
// are bounded by their cell on every axis but one: the z of a flat periodic
// system is free, and in a batch with a 2D system that is not flat it counts.
// The pairs of such a tile are all settled by the exact test.
template <int ROWS, bool FLAT, bool PERIODIC, class V>
__device__ inline bool filter_too_wide(V z0, V z1, double h)
{
    if constexpr (ROWS == 3 && PERIODIC && !FLAT) return (double)(z1 - z0) > h;
    else return false;
}

// The bits of slice s's slots below n, the end of the list in this chunk.
template <int T>
__device__ inline MaskT<T> slots_below(int s, int n)
{
    constexpr int S = 64 / T;
    const int k = n > s ? (n - s + S - 1) / S : 0;
    return k >= T ? ~MaskT<T>(0) : (MaskT<T>(1) << k) - 1;
}

// --------------------------------------------------------- wave reductions --
// Inclusive prefix sum of v over the wave's lanes, in six DPP steps: the
// row shifts by 1, 2, 4 and 8 lanes scan each row of 16 lanes, then the
// broadcast of lane 15 carries row 0's total into row 1 and row 2's into
// row 3, and the broadcast of lane 31 carries rows 0-1's total into rows 2
// and 3.  Lanes a step does not write add the 0 given as the old value.
// Every lane of the wave must be active.
__device__ inline int wave_scan(int v)
{
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);   // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);   // row_shr:2
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);   // row_shr:4
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);   // row_shr:8
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31
    return v;
}

// Copy of v from the lane a DPP step reads; lanes the step does not write
// keep their own.
template <int CTRL, int ROW_MASK>
__device__ inline float dpp_own(float v)
{
    const int b = __float_as_int(v);
    return __int_as_float(__builtin_amdgcn_update_dpp(b, b, CTRL, ROW_MASK, 0xf, false));
}

template <int CTRL, int ROW_MASK>
__device__ inline double dpp_own(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = (int)b, hi = (int)(b >> 32);
    const int l = __builtin_amdgcn_update_dpp(lo, lo, CTRL, ROW_MASK, 0xf, false);
    const int h = __builtin_amdgcn_update_dpp(hi, hi, CTRL, ROW_MASK, 0xf, false);
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)h << 32) | (unsigned)l));
}

__device__ inline float lane63(float v)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

__device__ inline double lane63(double v)
{
    const long long b = __double_as_longlong(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)b, 63);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(b >> 32), 63);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// Smallest and largest v over the wave (uniform); the steps of wave_scan.
template <class V>
__device__ inline void wave_bounds(V v, V& lo, V& hi)
{
    V a = v, b = v;
    a = fmin(a, dpp_own<0x111, 0xf>(a)); b = fmax(b, dpp_own<0x111, 0xf>(b));
    a = fmin(a, dpp_own<0x112, 0xf>(a)); b = fmax(b, dpp_own<0x112, 0xf>(b));
    a = fmin(a, dpp_own<0x114, 0xf>(a)); b = fmax(b, dpp_own<0x114, 0xf>(b));
    a = fmin(a, dpp_own<0x118, 0xf>(a)); b = fmax(b, dpp_own<0x118, 0xf>(b));
    a = fmin(a, dpp_own<0x142, 0xa>(a)); b = fmax(b, dpp_own<0x142, 0xa>(b));
    a = fmin(a, dpp_own<0x143, 0xc>(a)); b = fmax(b, dpp_own<0x143, 0xc>(b));
    lo = lane63(a);
    hi = lane63(b);
}

// ------------------------------------------------------------ candidates --
// The candidate ranges of a tile: its cell's stencil rows, concatenated.
// pref[i] candidates precede range i; a chunk's slot l holds candidate
// base + l, whose range i satisfies pref[i] <= base + l < pref[i + 1].
// The kept candidates are staged in a ring of at most 128 slots: q (and rg,
// for periodic systems) of each slot, and the kept position of the first
// target at each occurrence of the tile's cell.
template <int ROWS, bool PER, int NQ = 128>
struct Cands {
    static constexpr int MAXR = 2 * ROWS;
    static constexpr int NSH = PER ? MAXR : 1;
    int j0[MAXR];
    int pref[MAXR + 1];
    double sx[NSH], sy[NSH], sz[NSH];  // image shift (periodic systems)
    int q[NQ];                         // particle index of each ring slot (1: not kept,
                                       // in kernels whose operator does not need it)
    int rg[PER ? 128 : 1];             // range of each ring slot
    int self0[MAXR];
};

// Ranges of the tile's candidate list, one lane per range (empty ones are
// kept in place): the lanes' loads of the row ends overlap, and a prefix sum
// concatenates the rows.  Returns the number of ranges; *total receives the
// candidate count.  (One row after the other, each waiting for its loads,
// took ~55 instructions per row and 2-4 us per tile.)
template <int ROWS, bool PERIODIC, int NQ>
__device__ inline int build_cands(const SysDesc& d, const int* cell_start, int lc,
                                  Cands<ROWS, PERIODIC, NQ>& L, int& total)
{
    constexpr int NR = PERIODIC ? 2 * ROWS : ROWS;
    const int lane = __lane_id();
    int len = 0;
    Seg g{};
    if (lane < NR) {
        Seg segs[2];
        const int k = PERIODIC ? lane & 1 : 0;
        const int ns = row_segments<ROWS, PERIODIC>(d, cell_start, lc, PERIODIC ? lane >> 1 : lane,
                                                    segs);
        // field by field: a selected struct would live in scratch
        g.j0 = k ? segs[1].j0 : segs[0].j0;
        g.j1 = k ? segs[1].j1 : segs[0].j1;
        g.sx = k ? segs[1].sx : segs[0].sx;
        g.sy = segs[0].sy;
        g.sz = segs[0].sz;
        if (k < ns) len = g.j1 - g.j0;
    }
    const int incl = wave_scan(len);
    total = __builtin_amdgcn_readlane(incl, 63);
    if (lane < NR) {
        L.j0[lane] = g.j0;
        L.pref[lane] = incl - len;
        if constexpr (PERIODIC) {
            L.sx[lane] = g.sx;
            L.sy[lane] = g.sy;
            L.sz[lane] = g.sz;
        }
    }
    if (lane == 0) L.pref[NR] = total;
    return NR;
}

// Slot of chunk `base` that holds candidate g (g < total): its range and
// particle index.  Ranges are scanned from `cur`, the range of slot 0.
template <int ROWS, bool PER, int NQ>
__device__ inline int slot_range(const Cands<ROWS, PER, NQ>& L, int cur, int g)
{
    int i = cur;
    while (L.pref[i + 1] <= g) ++i;
    return i;
}

// Range of the next chunk's slot 0.
template <int ROWS, bool PER, int NQ>
__device__ inline int advance_range(const Cands<ROWS, PER, NQ>& L, int nr, int cur, int next_base)
{
    while (cur < nr && L.pref[cur + 1] <= next_base) ++cur;
    return cur;
}

template <int ROWS, int NQ>
__device__ inline Seg range_shift(const Cands<ROWS, true, NQ>& L, int i)
{
    Seg g;
    g.j0 = g.j1 = 0;
    g.sx = L.sx[i];
    g.sy = L.sy[i];
    g.sz = L.sz[i];
    return g;
}

// Lanes below this one with their bit set in m.
__device__ inline int lane_rank(unsigned long long m)
{
    return (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32),
                                          __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
}

// Append the lanes' kept candidates to the ring (list order).  fill: kept so
// far; nself: occurrences of the first target so far.  Returns the lane's
// kept position (its ring slot is pos & 127), -1 if its candidate is not
// kept.
template <int ROWS, bool PER, int NQ>
__device__ inline int compact(Cands<ROWS, PER, NQ>& L, int& fill, int& nself, bool keep, int q,
                              int rg, int first)
{
    const unsigned long long km = __ballot(keep);
    const unsigned long long sm = __ballot(keep && q == first);
    const int pos = fill + lane_rank(km);
    if (keep) {
        const int r = pos & 127;
        if constexpr (NQ > 1) L.q[r] = q;
        if constexpr (PER) L.rg[r] = rg;
        if (q == first) L.self0[nself + lane_rank(sm)] = pos;
    }
    fill += __popcll(km);
    nself += __popcll(sm);
    return keep ? pos : -1;
}

// Clear the bits of the chunk's slots (kept positions head ... head + 63)
// that hold the target itself (the reference skips p === q,
// src/core.jl:105): target t sits t slots after the first target at every
// occurrence of the tile's cell.
template <int ROWS, bool PER, int T, int NQ>
__device__ inline void drop_self(const Cands<ROWS, PER, NQ>& L, int nself, int head, int t, int s,
                                 MaskT<T>& m)
{
    constexpr int S = 64 / T;
    for (int k = 0; k < nself; ++k) {
        const int l = L.self0[k] + t - head;
        if (l >= 0 && l < 64 && l % S == s) m &= ~(MaskT<T>(1) << (l / S));
    }
}

// Bounding box of a tile's targets: absolute in the FP64 kernels, relative to
// the tile's first target in the mixed ones.
template <class V>
struct Box {
    V x0, x1, y0, y1, z0, z1;
};

// The box of the lanes' targets (lanes without one hold the first): a few
// DPP steps per tile, where a kernel of its own that read the positions again
// and stored 48 bytes per tile took 50 us per 5.75M-particle build.
template <bool FLAT, class V>
__device__ inline Box<V> tile_box(V x, V y, V z)
{
    Box<V> b;
    wave_bounds(x, b.x0, b.x1);
    wave_bounds(y, b.y0, b.y1);
    b.z0 = b.z1 = V(0);
    if (!FLAT) wave_bounds(z, b.z0, b.z1);
    return b;
}

// Squared distance of (x, y, z) to the box (0 inside), evaluated in the
// predicate's operation order.
template <bool FLAT>
__device__ inline double box_dist2(const Box<double>& b, double x, double y, double z)
{
    const double dx = fmax(fmax(b.x0 - x, x - b.x1), 0.0);
    const double dy = fmax(fmax(b.y0 - y, y - b.y1), 0.0);
    double ss = dx * dx + dy * dy;
    if (!FLAT) {
        const double dz = fmax(fmax(b.z0 - z, z - b.z1), 0.0);
        ss = ss + dz * dz;
    }
    return ss;
}

template <bool FLAT>
__device__ inline float box_dist2(const Box<float>& b, float x, float y, float z)
{
    const float dx = fmaxf(fmaxf(b.x0 - x, x - b.x1), 0.0f);
    const float dy = fmaxf(fmaxf(b.y0 - y, y - b.y1), 0.0f);
    const float dz = FLAT ? 0.0f : fmaxf(fmaxf(b.z0 - z, z - b.z1), 0.0f);
    return fmaf(dz, dz, fmaf(dy, dy, dx * dx));
}

// ------------------------------------------------------ balanced pairs --
// The accepted pairs of a chunk are spread over all 64 lanes instead of
// being walked by the lane that owns the target: the per-lane counts of a
// chunk differ a lot (targets near the chunk's candidates accept many, far
// ones none), and an owner-walked loop runs as long as the busiest lane.
// Per chunk:
//   - the owner lane of target t (slice 0, lane t) publishes the target's
//     64-bit word of accepted slots in LDS;
//   - the pairs are cut into runs of at most B pairs, one target per run,
//     with B a quota from the mean up for which the runs fit in 64 lanes
//     (or, when every target is one run, each owner lane walks its own);
//     lane l takes run l;
//   - the run split is wave-uniform work (DPP scans, ballots, a table
//     lookup), and a lane finds its run from a packed mark and a prefix
//     maximum (split_runs);
//   - a lane reads its target's data from the owner lane (shuffles), skips
//     to its run with a popcount descent and walks the run;
//   - its partial sums go to LDS, and the owner folds the runs of its target
//     in run order, so the result does not depend on timing.
// The words are exact (the mixed test settles its guard band before), so
// the runs -- and the summation order -- are the same whether a pass tests
// the candidates or loads the density pass's words.
template <class Part>
struct Bal {
    unsigned long long w[64];  // accepted slots of each target
    int mark[64];              // run starts: (target + 1, its pop) packed, else 0
    Part part[64];             // each lane's partial sums of the chunk
};

// Bit b of a target's word is slot (b % T) * (64 / T) + b / T of the chunk.
template <int T>
__device__ inline int slot_of_bit(int b)
{
    return (b % T) * (64 / T) + b / T;
}

// w without its n lowest set bits (0 <= n < popcount(w)): the n-th set bit
// is found in the 32-bit half that holds it, halving the field each step.
__device__ inline unsigned long long drop_low_bits(unsigned long long w, int n)
{
    if (n <= 0) return w;
    const unsigned lo = (unsigned)w;
    const int clo = __popc(lo);
    const bool up = n >= clo;
    unsigned x = up ? (unsigned)(w >> 32) : lo;
    n = up ? n - clo : n;
    int pos = up ? 32 : 0;
    int c = __popc(x & 0xffffu);
    if (n >= c) { n -= c; x >>= 16; pos += 16; }
    c = __popc(x & 0xffu);
    if (n >= c) { n -= c; x >>= 8; pos += 8; }
    c = __popc(x & 0xfu);
    if (n >= c) { n -= c; x >>= 4; pos += 4; }
    c = __popc(x & 0x3u);
    if (n >= c) { n -= c; x >>= 2; pos += 2; }
    if (n >= (int)(x & 1u)) pos += 1;
    return w & (~0ull << pos);
}

// Largest v over the wave, 0 <= v < 128, bit by bit from the top: one
// compare per bit, the result is uniform.
__device__ inline int wave_max7(int v)
{
    int r = 0;
#pragma unroll
    for (int b = 6; b >= 0; --b) {
        const int c = r | (1 << b);
        if (__ballot(v >= c) != 0ull) r = c;
    }
    return r;
}

// Copy of v as held by lane src.
template <class V>
__device__ inline V shfl_value(const V& v, int src)
{
    static_assert(sizeof(V) % 4 == 0, "shuffled per 32-bit word");
    V r;
    const int* a = reinterpret_cast<const int*>(&v);
    int* b = reinterpret_cast<int*>(&r);
#pragma unroll
    for (unsigned i = 0; i < sizeof(V) / 4; ++i) b[i] = __shfl(a[i], src);
    return r;
}

// Sum of v over the wave (uniform).
__device__ inline int wave_total(int v) { return __builtin_amdgcn_readlane(wave_scan(v), 63); }

// Inclusive prefix maximum of v >= 0 over the wave's lanes: the steps of
// wave_scan with max for the sum.
__device__ inline int wave_max_scan(int v)
{
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true));   // row_shr:1
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true));   // row_shr:2
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true));   // row_shr:4
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true));   // row_shr:8
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false));  // row_bcast:15
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false));  // row_bcast:31
    return v;
}

// ceil(pop / B) for 0 <= pop <= 64 and a uniform 1 <= B <= 65, branch-free:
// floor((pop + B - 1/2) / B), a value at least 1 / (2B) away from every
// integer, computed as pop * (1/B) + (B - 1/2) / B with one FMA.  The two
// factors are rounded to FP32 at compile time and read from a table with a
// scalar load (B is uniform); the FMA's error stays below 3e-5 / B, so the
// truncation gives the exact quotient.
struct RunDiv {
    float r, c;
};

#define SPH_RUN_DIV(b) {1.0f / (float)(b), ((float)(b) - 0.5f) / (float)(b)}
#define SPH_RUN_DIV8(b)                                                                        \
    SPH_RUN_DIV(b), SPH_RUN_DIV(b + 1), SPH_RUN_DIV(b + 2), SPH_RUN_DIV(b + 3),                \
        SPH_RUN_DIV(b + 4), SPH_RUN_DIV(b + 5), SPH_RUN_DIV(b + 6), SPH_RUN_DIV(b + 7)
static __constant__ RunDiv kRunDiv[72] = {{0.0f, 0.0f},     SPH_RUN_DIV(1),     SPH_RUN_DIV(2),
                                          SPH_RUN_DIV(3),   SPH_RUN_DIV(4),     SPH_RUN_DIV(5),
                                          SPH_RUN_DIV(6),   SPH_RUN_DIV(7),     SPH_RUN_DIV8(8),
                                          SPH_RUN_DIV8(16), SPH_RUN_DIV8(24),   SPH_RUN_DIV8(32),
                                          SPH_RUN_DIV8(40), SPH_RUN_DIV8(48),   SPH_RUN_DIV8(56),
                                          SPH_RUN_DIV8(64)};
#undef SPH_RUN_DIV8
#undef SPH_RUN_DIV

__device__ inline RunDiv run_div(int B) { return kRunDiv[B]; }

__device__ inline int runs_of(int pop, RunDiv d) { return (int)fmaf((float)pop, d.r, d.c); }

// Runs of the chunk.  pop: accepted pairs of the lane's target (owner lanes
// only, 0 elsewhere).  Returns 0 when no target has pairs, else a positive
// value.  When the run length is the largest pop, every target is one run
// and the runs need no moving: own is set and each owner lane walks its own
// target (tt, r0 and cnt are then unused).  That is always so when all 64
// lanes hold a target with pairs, since a shorter run length splits the
// largest and needs 65 runs.  Otherwise sets the lane's run (target tt,
// first rank r0, count cnt) and, for owner lanes, the first run and the
// number of runs of their target.  The wave sums are DPP scans and the
// comparisons with the largest pop are ballots (pop > B on some lane), so
// the split moves no data through LDS until the runs are assigned.
template <class Part>
__device__ inline int split_runs(int lane, int pop, Bal<Part>& bal, bool& own, int& tt, int& r0,
                                 int& cnt, int& first_run, int& nruns)
{
    const unsigned long long with_pairs = __ballot(pop > 0);
    own = false;
    tt = -1;
    r0 = cnt = first_run = nruns = 0;
    if (with_pairs == 0ull) return 0;
    if (with_pairs == ~0ull) {
        own = true;
        return 1;
    }
    const int tot = wave_total(pop);
    // The run length B: the mean (rounded up) or one more if the runs then
    // fit in 64 lanes; else at most two bisection steps between that and
    // ceil(tot / (64 - nz)) (nz: lanes with pairs), which always fits since
    // ceil(pop / B) <= pop / B + 1.  The number of runs does not grow with
    // B; at B >= max(pop) every target is one run.  A full search for the
    // smallest B costs more tests than it saves pairs on sparse chunks.
    int B = (tot + 63) >> 6;  // <= 64: pop <= 64 on each lane
    const int B0 = B;
    // the runs at B and at B + 1 in one scan (16-bit halves: each sum <= 4096,
    // so the low half never carries into the high one); its prefixes serve the
    // run assignment below when B ends at one of the two
    const int n0 = runs_of(pop, run_div(B)), n1 = runs_of(pop, run_div(B + 1));
    const int scan01 = wave_scan(n0 | (n1 << 16));
    const int both = __builtin_amdgcn_readlane(scan01, 63);
    if ((both & 0xffff) > 64 && __ballot(pop > B) != 0ull) {
        ++B;
        if ((both >> 16) > 64 && __ballot(pop > B) != 0ull) {
            const int nz = __popcll(with_pairs);  // < 64: not every lane has pairs
            int lo = B + 1, hi = min((tot + (64 - nz) - 1) / (64 - nz), wave_max7(pop));
            for (int it = 0; it < 2 && lo < hi; ++it) {
                const int mid = (lo + hi) >> 1;
                if (wave_total(runs_of(pop, run_div(mid))) > 64)
                    lo = mid + 1;
                else
                    hi = mid;
            }
            B = hi;
        }
    }
    if (__ballot(pop > B) == 0ull) {  // B >= max(pop)
        own = true;
        return tot;
    }
    int incl;
    if (B == B0) {
        nruns = n0;
        incl = scan01 & 0xffff;
    } else if (B == B0 + 1) {
        nruns = n1;
        incl = scan01 >> 16;
    } else {
        nruns = runs_of(pop, run_div(B));
        incl = wave_scan(nruns);
    }
    first_run = incl - nruns;
    const int used = __builtin_amdgcn_readlane(incl, 63);  // <= 64
    // The lane where a target's runs start gets a mark (target + 1, pop);
    // a lane's run belongs to the last mark at or below it.  The mark, with
    // its lane index added, goes through a prefix maximum: the target
    // numbers grow with the start lanes, so the maximum is that last mark.
    bal.mark[lane] = 0;
    __syncthreads();
    if (nruns > 0 && first_run < 64) bal.mark[first_run] = ((lane + 1) << 16) | (pop << 8);
    __syncthreads();
    int mk = bal.mark[lane];
    if (mk != 0) mk |= lane;
    mk = wave_max_scan(mk);
    if (lane < used) {
        tt = (mk >> 16) - 1;
        r0 = (lane - (mk & 0xff)) * B;
        cnt = min(B, ((mk >> 8) & 0xff) - r0);
    }
    return tot;
}

// Slots of the LDS ring of staged candidates.  A testing pass appends the
// kept candidates of each streamed step behind those not yet worked, so it
// needs two chunks' room; the kept-list kernel stages one chunk per step and
// works it before the next, so one chunk's room does (less LDS, more waves).
template <bool KEPT>
constexpr int ring_slots()
{
    return KEPT ? 64 : 128;
}

// Entries of the candidate-index ring: the kept-list kernel of an operator
// that does not read the index keeps none (LDS for one more wave per SIMD).
template <class Op, bool KEPT>
constexpr int cands_q()
{
    return KEPT && !Op::USES_Q ? 1 : 128;
}

// ------------------------------------------------------------- staging --
// A candidate's fields as loaded from the columns (the image shift already
// added to the position).  A kernel streams its candidates 64 at a time:
// each lane loads one into registers, and the kept ones are converted and
// written to the LDS ring in the same step (the other waves on the SIMD
// cover the loads' latency).  Each operator fills (fetch) and writes (put)
// only the fields it uses.
struct Raw {
    double x, y, z, a0, a1, a2, a3, a4;
};

// Slots past the end of the list: far away, rejected by every test.
__device__ inline Raw pad_raw()
{
    Raw r{};
    r.x = r.y = r.z = 1.0e30;
    return r;
}

template <bool P>
__device__ inline void fetch_pos(const PairCtx& c, int q, const Seg& g, Raw& r)
{
    r.x = shifted<P>(COL(c, C_X, q), g.sx);
    r.y = shifted<P>(COL(c, C_Y, q), g.sy);
    r.z = shifted<P>(COL(c, C_Z, q), g.sz);
}

// Fetch candidate g of the list (a pad past its end) into registers; cur is
// the range of the chunk's first slot.  rq, rg: its particle index and range.
template <int ROWS, bool PERIODIC, class Op, int NQ>
__device__ inline void fetch_slot(const PairCtx& c, const Cands<ROWS, PERIODIC, NQ>& L, int total,
                                  int cur, int g, Raw& raw, int& rq, int& rg)
{
    if (g < total) {
        const int i = slot_range(L, cur, g);
        const int q = L.j0[i] + (g - L.pref[i]);
        Seg sh{};
        if constexpr (PERIODIC) sh = range_shift(L, i);
        raw = Op::template fetch<PERIODIC>(c, q, sh);
        rq = q;
        rg = i;
    } else {
        raw = pad_raw();
        rq = 0;
        rg = 0;
    }
}

// Neighbour-set digest of each target: the number of accepted q and the sum
// modulo 2^64 of mix64(refidx q + 1), written to pair_out[2 refidx p] and
// pair_out[2 refidx p + 1].  Integer sums, so the result does not depend on
// the order in which the pairs are met.
__device__ inline unsigned long long mix64(unsigned long long z)
{
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ULL;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebULL;
    return z ^ (z >> 31);
}

__device__ inline void digest_write(const PairCtx& c, int p, unsigned long long h,
                                    unsigned long long n, int T, bool write)
{
    for (int o = T; o < 64; o <<= 1) {
        h += __shfl_xor(h, o);
        n += __shfl_xor(n, o);
    }
    if (!write) return;
    const long long r = c.refidx[p];
    c.pair_out[2 * r] = (long long)n;
    c.pair_out[2 * r + 1] = (long long)h;
}

// ------------------------------------------------------------------- EOS --
// The equation of state of particle p whose density rho the pass has just
// formed: the expressions of SPH_OP_FIND_PRESSURE(_RHO0).  A kernel of its own
// that read rho back took 43 us of a 5.75M-particle step and 4 of a small one's
// 75; here it costs nothing measurable since the matrix-core test freed the
// registers for it (before, the density kernel spilled and this made its pass
// ~80 us longer; now it spills no vector register).
__device__ inline void write_eos(const PairCtx& c, const SysDesc& d, int p, double rho)
{
    if (c.eos == EOS_NONE) return;
    const double rho0 = c.eos == EOS_RHO0_FIELD ? COL(c, C_RHO0, p) : d.ph.rho0;
    const double P = (d.ph.c * d.ph.c) * (rho - rho0);
    COL(c, C_P, p) = P;
    c.prho2_out[p] = P / (rho * rho);
}

// -------------------------------------------------------------- launch --
// Blocks of a kernel that a device holds at once (one-wave blocks, static
// LDS), 0 if it cannot be asked.  (Every device runs the one gfx950 build, so a
// compute unit holds the same number on each.)
inline int resident_blocks(const void* kernel, int device)
{
    int cus = 0, per_cu = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, 64, 0) != hipSuccess) {
        (void)hipGetLastError();
        return 0;
    }
    return cus * per_cu;
}

// Launch a tile kernel with the blocks it can use: no more than there are
// tiles (grid) and no more than run at once on the handle's device.
static constexpr int RESIDENT_DEVICES = 64, RESIDENT_UNKNOWN = 256 * 8;

template <auto Kernel, class... Args>
inline void launch_resident(int grid, hipStream_t st, const PairCtx& c, Args... args)
{
    static DeviceCache<RESIDENT_DEVICES> cache;
    const int fill = cache.get(c.device, RESIDENT_UNKNOWN, [](int device) {
        return resident_blocks(reinterpret_cast<const void*>(Kernel), device);
    });
    Kernel<<<grid < fill ? grid : fill, 64, 0, st>>>(c, args...);
}

}  // namespace sph
