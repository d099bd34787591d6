// Cell-list builder: the device form of create_cell_list! (src/core.jl:51-90)
// for every system of a batch at once.
//
// Five kernels, all on the handle's stream, no host round trip:
//   1. k_keys        per particle: FP64 find_key (src/structs.jl:97-106) and
//                    the inclusive bounding-box test (src/geometry.jl:24-30);
//                    a particle outside goes to its system's removal bucket.
//                    Periodic systems wrap positions into the box instead.
//                    Global key = the system's cell_base + local key.
//                    Per-bucket counts by wave-aggregated atomics (one atomic
//                    per distinct key in a wave; the input is the previous
//                    sorted order, so a wave usually touches one or two cells)
//   2. k_scan_counts exclusive prefix sum of the counts -> cell_start
//   3. k_scatter     bucket every particle
//   4. k_place       order each bucket by descending reference index, the
//                    order add_index! keeps (src/core.jl:26-41) -- deterministic
//                    whatever order the atomics handed out; the bucket of
//                    retired systems keeps its scatter order, never used --
//                    and move every column into the new order
//   5. k_tile_table  per cell ceil(count/T) tiles and the 64-candidate chunks
//                    a target walks, one scan of both, the tile table of the
//                    pair kernels.  Also the removal: each system's removal
//                    bucket holds its removed particles in descending
//                    reference index, and the reference's swap-with-end
//                    renumbering (src/core.jl:72-81) is replayed per system
//
// This is a counting sort on the global cell key (one radix digit) followed
// by an in-bucket rank.
//
// A small system's build is bound by its launches: with 19 kernels (three for
// each of three scans, of 5 + 3 + 12 us whatever their length) it took about
// 100 us, 30 us with these five; the 5.75M-particle dam break's took 560 us,
// 390 us now (no permutation written and read back, the fluid's acceleration
// left out, no pass for the tiles' boxes).
#include "brick.h"
#include "scan_kernels.h"
#include "sph_internal.h"

namespace sph {


// ---------------------------------------------------------------- prepare --
// Per-system reference-index base of the inverse map and the count at the
// start of the build.  One block of 256 threads; systems in rounds of 256, an
// exclusive scan of the counts per round.
__device__ inline void sys_prep(int nsys, int* sc, int* meta)
{
    __shared__ int part[4];
    if (threadIdx.x == 0) meta[META_NTOT] = meta[META_N];
    if (nsys == 1) {  // nothing to scan, no barrier
        if (threadIdx.x == 0) {
            sc[SC_NTOT] = sc[SC_N];
            sc[SC_REFBASE] = 0;
        }
        return;
    }
    int carry = 0;
    for (int s0 = 0; s0 < nsys; s0 += 256) {
        const int s = s0 + (int)threadIdx.x;
        const int n = s < nsys ? sc[SYSCNT * s + SC_N] : 0;
        int incl = n;
        const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int v = __shfl_up(incl, d);
            if (lane >= d) incl += v;
        }
        if (lane == 63) part[w] = incl;
        __syncthreads();
        int off = carry;
        for (int k = 0; k < w; ++k) off += part[k];
        const int round = part[0] + part[1] + part[2] + part[3];
        if (s < nsys) {
            sc[SYSCNT * s + SC_NTOT] = n;
            sc[SYSCNT * s + SC_REFBASE] = off + incl - n;
        }
        carry += round;
        __syncthreads();
    }
}

// ------------------------------------------------------------------ keys --
// Bucket key of particle i of system s: its cell, the system's removal
// bucket (outside the box, or not finite in a periodic system) or the dead
// bucket (retired system).  Periodic systems wrap the position (written
// back).
__device__ inline int key_of(const SysDesc& d, int s, int nsys, int cells_total, double px,
                             double py, double pz, double* x, double* y, double* z, int i)
{
    const Geo& g = d.g;
    if (!d.live) return cells_total + nsys;
    if (g.periodic) {
        // positions live in [bmin, bmin + box) on the periodic axes
        if (!(isfinite(px) && isfinite(py) && isfinite(pz))) return cells_total + s;
        px = px - g.box[0] * floor((px - g.bmin[0]) / g.box[0]);
        py = py - g.box[1] * floor((py - g.bmin[1]) / g.box[1]);
        x[i] = px;
        y[i] = py;
        long long ci = (long long)floor((px - g.bmin[0]) / g.cell[0]);
        long long cj = (long long)floor((py - g.bmin[1]) / g.cell[1]);
        long long ck = 0;
        if (g.L3 > 1) {
            pz = pz - g.box[2] * floor((pz - g.bmin[2]) / g.box[2]);
            z[i] = pz;
            ck = (long long)floor((pz - g.bmin[2]) / g.cell[2]);
        }
        ci = ci < 0 ? 0 : (ci >= g.L1 ? g.L1 - 1 : ci);
        cj = cj < 0 ? 0 : (cj >= g.L2 ? g.L2 - 1 : cj);
        ck = ck < 0 ? 0 : (ck >= g.L3 ? g.L3 - 1 : ck);
        return d.cell_base + (int)(ci + (long long)g.L1 * (cj + (long long)g.L2 * ck));
    }
    const bool inside = g.bmin[0] <= px && px <= g.bmax[0] && g.bmin[1] <= py &&
                        py <= g.bmax[1] && g.bmin[2] <= pz && pz <= g.bmax[2];
    if (!inside) return cells_total + s;
    long long ci = (long long)floor(px / g.h) - g.kp[0];
    long long cj = (long long)floor(py / g.h) - g.kp[1];
    long long ck = (long long)floor(pz / g.h) - g.kp[2];
    // In range by monotonicity of the correctly rounded division; the clamp
    // only guards memory.
    ci = ci < 0 ? 0 : (ci >= g.L1 ? g.L1 - 1 : ci);
    cj = cj < 0 ? 0 : (cj >= g.L2 ? g.L2 - 1 : cj);
    ck = ck < 0 ? 0 : (ck >= g.L3 ? g.L3 - 1 : ck);
    return d.cell_base + (int)(ci + (long long)g.L1 * (cj + (long long)g.L2 * ck));
}

// What a fused step leaves to the key pass of its next build, on particle i
// at position p (KeyStage): the expressions and the order of k_kick_drift,
// k_cd_kick and k_unary, so the bits of the operators.  STAGE_CD_KICK2_MOVE is
// the kick that ends one collapse_dry step and the kick and move that begin
// the next.
__device__ inline void key_stage(int stage, const Phys& ph, double* cols, long long cap, int i,
                                 double* p)
{
    const bool fluid = cols[C_TYPE * cap + i] == 0.0;
    if (stage == STAGE_KICK_DRIFT) {  // v += dt (a + g), x += dt v
        if (!fluid) return;
        const double k = ph.coeff * ph.dt;
        for (int d = 0; d < 3; ++d) {
            const double v = cols[(C_VX + d) * cap + i] + k * (cols[(C_AX + d) * cap + i] + ph.g[d]);
            cols[(C_VX + d) * cap + i] = v;
            p[d] = p[d] + k * v;
            cols[(C_X + d) * cap + i] = p[d];
        }
        return;
    }
    const double k = 0.5 * ph.dt;
    if (stage == STAGE_CD_EOS_MOVE) {
        double rho = cols[C_RHO * cap + i];
        rho = rho + cols[C_DRHO * cap + i] * ph.dt;
        cols[C_RHO * cap + i] = rho;
        cols[C_DRHO * cap + i] = 0.0;
        cols[C_P * cap + i] = (ph.c * ph.c) * (rho - ph.rho0);
    }
    for (int d = 0; d < 3; ++d) {
        if (fluid) {
            double v = cols[(C_VX + d) * cap + i];
            if (stage != STAGE_CD_EOS_MOVE) {
                const double a = cols[(C_AX + d) * cap + i] + ph.g[d];
                v = v + k * a;
                if (stage == STAGE_CD_KICK2_MOVE) v = v + k * a;
                cols[(C_VX + d) * cap + i] = v;
            }
            p[d] = p[d] + k * v;
            cols[(C_X + d) * cap + i] = p[d];
        }
        cols[(C_AX + d) * cap + i] = 0.0;
    }
}

// With a stage, one launch and one read and write of the positions fewer than
// a kernel of its own (5.75M particles, kick and keys: 90 + 57 us apart,
// 111 us together).
template <bool STAGED>
__global__ __launch_bounds__(256) void k_keys(int stage, const SysDesc* __restrict__ sysd, int nsys,
                                              int cells_total, double* cols, long long cap,
                                              const int* __restrict__ sysid, int* meta,
                                              int* __restrict__ key, int* __restrict__ slot,
                                              unsigned* __restrict__ cnt, int* sc,
                                              unsigned long long* stat, int nstat)
{
    const int n = meta[META_N];
    const int i = blockIdx.x * 256 + threadIdx.x;
    // the scans of this build start from cleared state words
    for (int j = i; j < nstat; j += gridDim.x * 256) stat[j] = 0ull;
    if (blockIdx.x == 0) sys_prep(nsys, sc, meta);
    const int s = i < n ? sysid[i] : 0;
    double *x = cols + C_X * cap, *y = cols + C_Y * cap, *z = cols + C_Z * cap;
    // a wave of one system reads its descriptor once, through the scalar
    // cache (the usual case: systems are contiguous)
    const int s0 = __builtin_amdgcn_readfirstlane(s);
    int k = -1;
    double p[3] = {0.0, 0.0, 0.0};
    if (i < n) {
        p[0] = x[i];
        p[1] = y[i];
        p[2] = z[i];
    }
    if (__all(i >= n || s == s0)) {
        if (i < n) {
            if (STAGED) key_stage(stage, sysd[s0].ph, cols, cap, i, p);
            k = key_of(sysd[s0], s0, nsys, cells_total, p[0], p[1], p[2], x, y, z, i);
        }
    } else if (i < n) {
        if (STAGED) key_stage(stage, sysd[s].ph, cols, cap, i, p);
        k = key_of(sysd[s], s, nsys, cells_total, p[0], p[1], p[2], x, y, z, i);
    }
    if (i < n) key[i] = k;
    // One atomic per distinct key among the wave's lanes.
    const int lane = __lane_id();
    unsigned long long active = __ballot(i < n);
    unsigned myslot = 0;
    while (active) {
        const int leader = __ffsll((long long)active) - 1;
        const int lk = __shfl(k, leader);
        const unsigned long long peers = __ballot(k == lk) & active;
        unsigned base = 0;
        if (lane == leader) base = atomicAdd(&cnt[lk], (unsigned)__popcll(peers));
        base = __shfl(base, leader);
        if ((peers >> lane) & 1ull)
            myslot = base + (unsigned)__popcll(peers & ((1ull << lane) - 1ull));
        active &= ~peers;
    }
    if (i < n) slot[i] = (int)myslot;
}

// ------------------------------------------------------------------ scan --
long long scan_partials_needed(long long n) { return (n + SCAN_TILE - 1) / SCAN_TILE + 1; }

// Exclusive prefix sum of the bucket counts into start[0 .. n], in one
// launch (chained blocks, scan_kernels.h).  The counts are zeroed behind the
// read: the next build finds them cleared.
static constexpr int CSCAN_TILE = 256 * 8;

__global__ __launch_bounds__(256) void k_scan_counts(unsigned* cnt, int n, int* start,
                                                     unsigned long long* stat,
                                                     unsigned long long* ticket)
{
    __shared__ unsigned long long prefix;
    const int b = chain_ticket(ticket);
    const int base = b * CSCAN_TILE + (int)threadIdx.x * 8;
    unsigned v[8];
    unsigned sum = 0;
    if (base + 8 <= n) {
        const uint4 lo = *reinterpret_cast<const uint4*>(cnt + base);
        const uint4 hi = *reinterpret_cast<const uint4*>(cnt + base + 4);
        v[0] = lo.x; v[1] = lo.y; v[2] = lo.z; v[3] = lo.w;
        v[4] = hi.x; v[5] = hi.y; v[6] = hi.z; v[7] = hi.w;
        *reinterpret_cast<uint4*>(cnt + base) = make_uint4(0u, 0u, 0u, 0u);
        *reinterpret_cast<uint4*>(cnt + base + 4) = make_uint4(0u, 0u, 0u, 0u);
    } else {
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            v[k] = base + k < n ? cnt[base + k] : 0u;
            if (base + k < n) cnt[base + k] = 0u;
        }
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) sum += v[k];
    unsigned total;
    unsigned run = block_incl_scan(sum, total) - sum;
    if (threadIdx.x < 64) {
        const unsigned long long p = chain_prefix(stat, b, total);
        if (threadIdx.x == 0) prefix = p;
    }
    __syncthreads();
    run += (unsigned)prefix;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        if (base + k <= n) start[base + k] = (int)run;
        run += v[k];
    }
}

// -------------------------------------------------- scatter, rank, gather --
__global__ __launch_bounds__(256) void k_scatter(const int* meta, const int* __restrict__ key,
                                                 const int* __restrict__ slot,
                                                 const int* __restrict__ ref,
                                                 const int* __restrict__ cell_start,
                                                 int* tmp_idx, int* tmp_key, int* tmp_ref)
{
    const int n = meta[META_NTOT];
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const int k = key[i];
    const int pos = cell_start[k] + slot[i];
    tmp_idx[pos] = i;
    tmp_key[pos] = k;
    tmp_ref[pos] = ref[i];
}

// Totals of the build, per system and overall (one block of 256 threads).
__device__ inline void finalize(const SysDesc* __restrict__ sysd, int nsys, int cells_total,
                                int* sc, int* meta, const int* cell_start)
{
    if (threadIdx.x == 0) {
        const int na = cell_start[cells_total];
        meta[META_NREM] = meta[META_NTOT] - na;
        meta[META_N] = na;
        meta[META_NCELLS] = 0;
    }
    for (int s = threadIdx.x; s < nsys; s += 256) {
        const SysDesc& d = sysd[s];
        const int off = cell_start[d.cell_base];
        const int end = cell_start[d.cell_base + d.g.key_max];
        sc[SYSCNT * s + SC_OFF] = off;
        sc[SYSCNT * s + SC_N] = d.live ? end - off : 0;
        sc[SYSCNT * s + SC_NREM] = cell_start[cells_total + s + 1] - cell_start[cells_total + s];
    }
}

// What k_place moves: the columns and where they go.
struct Move {
    const double* src;
    double* dst;
    const int* isrc;
    int* idst;
    long long cap;
    unsigned skip;     // columns (bit C_*) left out
    int skip_a;        // leave out the acceleration of fluid particles
    const int* sc;     // per-system counters (reference-index base)
    int* inv;
    double* prho2;     // P/rho^2 in the new order, or null
};

// Particle j of the old order, with reference index r, to slot k of the new
// one; with removals in this build, inv maps (system reference base +
// reference index) to the slot.
__device__ inline void move_particle(const Move& mv, int j, int key, int r, int k, bool removals)
{
#pragma unroll
    for (int f = 0; f < NCOL; ++f)
        if (f != C_AX && f != C_AY && f != C_AZ && f != C_TYPE && !((mv.skip >> f) & 1u))
            mv.dst[f * mv.cap + k] = mv.src[f * mv.cap + j];
    const double type = mv.src[C_TYPE * mv.cap + j];
    mv.dst[C_TYPE * mv.cap + k] = type;
    if (!mv.skip_a || type != 0.0) {
        mv.dst[C_AX * mv.cap + k] = mv.src[C_AX * mv.cap + j];
        mv.dst[C_AY * mv.cap + k] = mv.src[C_AY * mv.cap + j];
        mv.dst[C_AZ * mv.cap + k] = mv.src[C_AZ * mv.cap + j];
    }
    if (mv.prho2) {
        const double rho = mv.src[C_RHO * mv.cap + j];
        mv.prho2[k] = mv.src[C_P * mv.cap + j] / (rho * rho);
    }
    const int s = mv.isrc[I_SYS * mv.cap + j];
    mv.idst[I_REF * mv.cap + k] = r;
    mv.idst[I_KEY * mv.cap + k] = key;
    mv.idst[I_SYS * mv.cap + k] = s;
    if (removals) mv.inv[mv.sc[SYSCNT * s + SC_REFBASE] + r] = k;
}

// Rank of each particle in its bucket: the number of bucket members with a
// larger reference index (ties -- particles of different retired systems --
// by scatter position), so the ranks are a permutation of the bucket.
//   - the bucket of retired systems (dead_key) keeps its scatter order: its
//     order is never used, and it can hold whole retired systems;
//   - a block whose threads all lie in one bucket of more than RANK_LDS_MIN
//     particles (a removal bucket after many particles left the box) counts
//     against the bucket staged through LDS, 1024 indices at a time;
//   - otherwise the buckets the block's threads lie in (a few cells of tens
//     to hundreds of particles) are staged through LDS when they fit in
//     RANK_SPAN entries, and each thread counts against its bucket there;
//   - else each thread scans its bucket in global memory.
// The thread then moves its particle: it reads near the old slot and writes
// inside its bucket, so both sides of the permutation stay within a few cache
// lines of its neighbours' (the 5.75M-particle dam break: rank and gather
// apart 61 + 232 us, together 274 us).
static constexpr int RANK_LDS_MIN = 512;
static constexpr int RANK_SPAN = 2048;

__device__ inline int rank_in_bucket(int b0, int n, const int* __restrict__ cell_start,
                                     const int* __restrict__ tmp_key,
                                     const int* __restrict__ tmp_ref, int dead_key, int* tile)
{
    const int u = b0 + (int)threadIdx.x;
    const bool in = u < n;
    const int c0 = tmp_key[b0];
    const int c1 = tmp_key[min(n - 1, b0 + 255)];
    const int s0 = cell_start[c0], e0 = cell_start[c0 + 1];
    if (c0 == c1 && c0 != dead_key && e0 - s0 > RANK_LDS_MIN) {
        const int r = in ? tmp_ref[u] : 0;
        int rank = 0;
        for (int base = s0; base < e0; base += 1024) {
            const int m = min(1024, e0 - base);
            __syncthreads();
            for (int j = threadIdx.x; j < m; j += 256) tile[j] = tmp_ref[base + j];
            __syncthreads();
            for (int j = 0; j < m; ++j) {
                const int rv = tile[j];
                rank += rv > r || (rv == r && base + j < u);
            }
        }
        return s0 + rank;
    }
    // the span of the buckets of the block's first and last thread holds
    // every bucket in between (scatter order is bucket order)
    const int span0 = s0, span1 = cell_start[c1 + 1];
    if (c1 != dead_key && span1 - span0 <= RANK_SPAN) {
        for (int j = threadIdx.x; j < span1 - span0; j += 256) tile[j] = tmp_ref[span0 + j];
        __syncthreads();
        if (!in) return 0;
        // a live bucket (a cell or a system's removal bucket) holds one
        // system's particles, whose reference indices are distinct: the
        // rank is the count of larger ones, read four at a time
        const int c = tmp_key[u];
        const int s = cell_start[c], e = cell_start[c + 1];
        const int r = tile[u - span0];
        int rank = 0, v = s - span0;
        const int ve = e - span0;
        for (; v < ve && (v & 3); ++v) rank += tile[v] > r;
        for (; v + 4 <= ve; v += 4) {
            const int4 q = *reinterpret_cast<const int4*>(&tile[v]);
            rank += (q.x > r) + (q.y > r) + (q.z > r) + (q.w > r);
        }
        for (; v < ve; ++v) rank += tile[v] > r;
        return s + rank;
    }
    if (!in) return 0;
    const int c = tmp_key[u];
    if (c == dead_key) return u;
    const int s = cell_start[c], e = cell_start[c + 1];
    const int r = tmp_ref[u];
    int rank = 0;
#pragma unroll 8
    for (int v = s; v < e; ++v) {
        const int rv = tmp_ref[v];
        rank += rv > r || (rv == r && v < u);
    }
    return s + rank;
}

__global__ __launch_bounds__(256) void k_place(const SysDesc* __restrict__ sysd, int nsys,
                                               int cells_total, int* sc, int* meta,
                                               const int* __restrict__ cell_start,
                                               const int* __restrict__ tmp_idx,
                                               const int* __restrict__ tmp_key,
                                               const int* __restrict__ tmp_ref, Move mv)
{
    __shared__ __align__(16) int tile[RANK_SPAN];
    if (blockIdx.x == 0) finalize(sysd, nsys, cells_total, sc, meta, cell_start);
    const int n = meta[META_NTOT];
    const int b0 = blockIdx.x * 256;
    if (b0 >= n) return;  // whole block past the end (uniform)
    const int k = rank_in_bucket(b0, n, cell_start, tmp_key, tmp_ref, cells_total + nsys, tile);
    const int u = b0 + (int)threadIdx.x;
    if (u < n) move_particle(mv, tmp_idx[u], tmp_key[u], tmp_ref[u], k, cell_start[cells_total] != n);
}

// Removal renumbering (src/core.jl:72-81): with the removed reference
// indices r_1 > r_2 > ... > r_m of a system, particles[r_i] =
// particles[N+1-i] in turn.  One thread per system.
__device__ inline void remove_seq(int s, int cells_total, const int* sc, const int* cell_start,
                                  int* ref, int* inv)
{
    const int m = sc[SYSCNT * s + SC_NREM];
    if (m == 0) return;
    const int first = cell_start[cells_total + s];
    const int ntot = sc[SYSCNT * s + SC_NTOT];
    const int rb = sc[SYSCNT * s + SC_REFBASE];
    for (int i = 0; i < m; ++i) {
        const int r = ref[first + i];  // descending
        const int src = ntot - 1 - i;  // reference position N+1-i (1-based)
        const int slot = inv[rb + src];
        inv[rb + r] = slot;
        ref[slot] = r;
    }
}

// 64-candidate chunks one target of cell c walks: the pair kernels
// concatenate the cell's stencil ranges and cut the list into chunks of 64.
template <int ROWS>
__device__ inline int cell_chunks(const SysDesc& d, const int* cell_start, int lc)
{
    int n = 0;
    for (int row = 0; row < ROWS; ++row) {
        Seg seg[2];
        const int ns = row_segments<ROWS>(d, cell_start, lc, row, seg);
        for (int q = 0; q < 2; ++q)
            if (q < ns) n += seg[q].j1 - seg[q].j0;
    }
    return (n + 63) / 64;
}

// Tile table, in brick order: tile k of the cell c at rank r covers targets
// cell_start[c] + k*T ...; its pair masks start at the mask words of the
// tiles before it (chunks * T words each), its kept-candidate list at 64 / T
// times that.  Each thread takes CELLS consecutive ranks; tiles and mask
// words are scanned together, by two waves of each block (chained blocks).
// The first block also clears the tile queues and, at its end, replays the
// removals.
template <int ROWS, int CELLS>
__global__ __launch_bounds__(256) void k_tile_table(
    const SysDesc* __restrict__ sysd, const int* __restrict__ cell_sys, int ncells,
    const int* __restrict__ cell_start, int T, long long mask_cap, long long kept_cap, int4* tiles,
    int* meta, unsigned long long* mask_total, unsigned long long* stat_tiles,
    unsigned long long* stat_words, unsigned long long* ticket, int* queue, int nsys, int removal,
    const int* sc, int* ref, int* inv)
{
    __shared__ unsigned long long prefix[2];
    __shared__ int with_tiles;
    if (threadIdx.x == 0) with_tiles = 0;
    const int b = chain_ticket(ticket);  // (a block barrier)
    if (b == 0 && threadIdx.x < NQUEUE_SETS * QSET / QSTRIDE) queue[threadIdx.x * QSTRIDE] = 0;
    int cell[CELLS], nt[CELLS];
    long long words[CELLS];  // of one tile
    unsigned tsum = 0;
    unsigned long long wsum = 0;
    int ncell = 0;
#pragma unroll
    for (int k = 0; k < CELLS; ++k) {
        const int r = b * 256 * CELLS + (int)threadIdx.x * CELLS + k;
        cell[k] = nt[k] = 0;
        words[k] = 0;
        if (r < ncells) {
            const SysDesc& d = sysd[cell_sys[r]];
            const int lc = brick_cell(d.g.L1, d.g.L2, d.g.L3, r - d.cell_base);
            const int c = d.cell_base + lc;
            const int n = cell_start[c + 1] - cell_start[c];
            cell[k] = c;
            if (n > 0) {
                nt[k] = (n + T - 1) / T;
                words[k] = (long long)cell_chunks<ROWS>(d, cell_start, lc) * T;
                ++ncell;
            }
        }
        tsum += (unsigned)nt[k];
        wsum += (unsigned long long)(nt[k] * words[k]);
    }
    if (ncell) atomicAdd(&with_tiles, ncell);
    unsigned ttot;
    unsigned long long wtot;
    unsigned trun = block_incl_scan(tsum, ttot) - tsum;
    unsigned long long wrun = block_incl_scan(wsum, wtot) - wsum;
    if (threadIdx.x < 128) {  // the first wave chains the tiles, the second the words
        const int w = threadIdx.x >> 6;
        const unsigned long long p = chain_prefix(w ? stat_words : stat_tiles, b,
                                                  w ? wtot : (unsigned long long)ttot);
        if ((threadIdx.x & 63) == 0) prefix[w] = p;
    }
    __syncthreads();
    trun += (unsigned)prefix[0];
    wrun += prefix[1];
    if (threadIdx.x == 0) {
        if (with_tiles) atomicAdd(&meta[META_NCELLS], with_tiles);
        if (b == (int)gridDim.x - 1) {
            const unsigned long long need = prefix[1] + wtot;
            meta[META_NTILES] = (int)((unsigned)prefix[0] + ttot);
            *mask_total = need;
            meta[META_MASK_OK] = (long long)need <= mask_cap ? 1 : 0;
            // 64 kept-candidate entries per chunk of a tile, T mask words
            meta[META_KEPT_OK] = (long long)(need / T * 64) <= kept_cap ? 1 : 0;
        }
    }
#pragma unroll
    for (int k = 0; k < CELLS; ++k) {
        const int cs = nt[k] > 0 ? cell_start[cell[k]] : 0;
        for (int t = 0; t < nt[k]; ++t) {
            tiles[trun++] = make_int4(cell[k], cs + t * T, (int)(unsigned)(wrun & 0xffffffffull),
                                      (int)(wrun >> 32));
            wrun += (unsigned long long)words[k];
        }
    }
    // The replay is a serial chain of reads (15 ms for 100,000 particles that
    // leave at once), so it comes last: no block of the scan waits for it.
    if (b == 0 && removal && meta[META_NREM] != 0)
        for (int s = threadIdx.x; s < nsys; s += 256) remove_seq(s, ncells, sc, cell_start, ref, inv);
}

// State words of the scans and the count of cells with tiles, cleared for a
// tile table built apart from a cell list.
__global__ __launch_bounds__(256) void k_reset_scans(unsigned long long* stat, int nstat, int* meta)
{
    for (int j = blockIdx.x * 256 + threadIdx.x; j < nstat; j += gridDim.x * 256) stat[j] = 0ull;
    if (blockIdx.x == 0 && threadIdx.x == 0) meta[META_NCELLS] = 0;
}

// ------------------------------------------------------------ host side --
static inline unsigned nblocks(long long n, int b) { return (unsigned)((n + b - 1) / b); }

// Cells per thread of the tile table.  A table's blocks pass their sums on one
// after the other, ~12 ns each, so a large grid wants few blocks; a small one's
// table waits on one thread's loads and divisions (nine rows of them in 3D), so
// it wants one cell per thread.  A build of 20,000 particles with 1 / 8 cells per
// thread, us: 2D 90k cells 66 / 72, 137k 72 / 73, 202k 81 / 76, 1M 146 / 96, 16M
// 982 / 409; 3D 97k 69 / 87, 195k 83 / 87, 262k 91 / 90, 512k 120 / 101, 4M
// 348 / 207; 2, 4, 16 or 32 gain at most 12% over the better of the two.
constexpr int TT_FEW = 1, TT_MANY = 8;

static inline int tt_cells(int rows, long long ncells)
{
    return ncells > (rows == 3 ? 1 << 17 : 1 << 18) ? TT_MANY : TT_FEW;
}

// State words of the build's scans, for `cells` buckets: the counts, tiles
// and mask words of each block (with the most blocks), then one ticket per scan.
static inline int stat_blocks(long long cells) { return (int)(cells / (256 * TT_FEW)) + 2; }
long long scan_state_needed(long long cells) { return 3ll * stat_blocks(cells) + 2; }

static void enqueue_tile_table(sph_system* s, int removal)
{
    const int ncells = (int)s->cells_total;
    const int per = tt_cells(s->rows, ncells);
    const bool many = per == TT_MANY;
    const unsigned nb = nblocks(ncells, 256 * per);
    const int sb = stat_blocks(s->cells_cap);
    unsigned long long* stat = s->scan_state;
    auto k = s->rows == 3 ? (many ? k_tile_table<3, TT_MANY> : k_tile_table<3, TT_FEW>)
                          : (many ? k_tile_table<9, TT_MANY> : k_tile_table<9, TT_FEW>);
    k<<<nb, 256, 0, s->stream>>>(s->sysd, s->cell_sys, ncells, s->cell_start, s->tile_T,
                                 s->masks ? s->mask_cap : 0,
                                 s->kept && (s->kept_rg || !s->periodic) ? s->kept_cap : 0,
                                 s->tiles, s->meta, s->mask_total, stat + sb, stat + 2 * sb,
                                 stat + 3 * sb + 1, s->queue, (int)s->sys_host.size(), removal,
                                 s->sys_cnt, s->icols[s->cur] + I_REF * s->cap, s->inv);
    s->queue_used = 0;
}

// The tile table of the current cell list for another tile size.  A batch
// that holds no system (every one retired, or none added yet) has no cells, no
// tiles and maybe no arrays for them.
void enqueue_tiles(sph_system* s)
{
    if (s->cells_total == 0) return;
    const int nstat = (int)scan_state_needed(s->cells_cap);
    k_reset_scans<<<nblocks(nstat, 256), 256, 0, s->stream>>>(s->scan_state, nstat, s->meta);
    enqueue_tile_table(s, 0);
}

// skip_cols: columns (bit C_*) the caller rewrites for every particle before
// reading them (skip_a: the acceleration of every fluid particle); they are
// not moved, and their values in the new order are undefined.  stage: what the
// step before left to this build's key pass (KeyStage).  prho2: also form
// P/rho^2 in the new order.
void enqueue_build(sph_system* s, unsigned skip_cols, int skip_a, int stage, bool prho2)
{
    hipStream_t st = s->stream;
    const long long cap = s->cap;
    const int nsys = (int)s->sys_host.size();
    const int ncells = (int)s->cells_total;
    const int nbuckets = (int)(s->cells_total + nsys + 1);
    const unsigned nb = nblocks(s->n > 0 ? s->n : 1, 256);
    const int sb = stat_blocks(s->cells_cap);
    double* c = s->cols[s->cur];
    int* ic = s->icols[s->cur];
    unsigned long long* stat = s->scan_state;
    auto keys = stage != STAGE_NONE ? k_keys<true> : k_keys<false>;
    keys<<<nb, 256, 0, st>>>(stage, s->sysd, nsys, ncells, c, cap, ic + I_SYS * cap, s->meta,
                             ic + I_KEY * cap, s->slot, s->cnt, s->sys_cnt, stat,
                             (int)scan_state_needed(s->cells_cap));
    k_scan_counts<<<nblocks(nbuckets + 1, CSCAN_TILE), 256, 0, st>>>(s->cnt, nbuckets, s->cell_start,
                                                                     stat, stat + 3 * sb);
    k_scatter<<<nb, 256, 0, st>>>(s->meta, ic + I_KEY * cap, s->slot, ic + I_REF * cap,
                                  s->cell_start, s->tmp_idx, s->tmp_key, s->tmp_ref);
    const Move mv{c, s->cols[s->cur ^ 1], ic, s->icols[s->cur ^ 1], cap, skip_cols, skip_a,
                  s->sys_cnt, s->inv, prho2 ? s->prho2 : nullptr};
    k_place<<<nb, 256, 0, st>>>(s->sysd, nsys, ncells, s->sys_cnt, s->meta, s->cell_start,
                                s->tmp_idx, s->tmp_key, s->tmp_ref, mv);
    s->cur ^= 1;
    enqueue_tile_table(s, 1);
}

}  // namespace sph
