// boids_kernels.hip — gfx950 kernels of the boid step.
//
// Compiled with -ffp-contract=off: every multiply and add that feeds a
// neighbour decision is rounded separately, exactly as the oracle (and, in
// float mode, the reference's x86-64 build) computes it.  Multiply-adds are
// written explicitly (fmaf) only where a result feeds no exact decision.
//
// Per-pair semantics (all modes) follow Boid::isInsideArea
// (src/boid.cpp:27-42) and the phase-A loop of src/boid_simulation.cpp:153-212;
// sqrt/acos are replaced by exact thresholds computed on the host
// (boids_engine.hip: thresholds()), so the kernels compare
//   s < s_thr        <=>  sqrt(s) < r                 (sqrt monotone, correctly rounded)
//   c >= c_thr, c<=1 <=>  acos(c) <= pi*a              (acos monotone; NaN/|c|>1 reject)
#include "boids_device.h"

namespace boids {


// ---------------------------------------------------------------------------
// All-pairs step: one wave per boid i.  The 64 lanes test the candidates
// j = base + lane against a bound just above the largest radius (near2) and
// append those below it to an LDS list, in ascending j -- the reference's
// summation order (src/boid_simulation.cpp:153-212); whenever it holds 64, they
// go through OrderedSums (src/boid_simulation.cpp:216-248 after the last).
// R = float: bit-identical to boidsim.  R = double: the FP64 promotion.  For
// flocks above 4096 boids (double: 3072), which fill the chip with a wave per
// boid; what bounds it is the tests of the candidates, and in crowded flocks the
// ordered sums.  One update of N = 8192, uniform / all in reach of all, with the
// synchronisation: float 82 / 524 us, FP64 141 / 747 (170 / 5816 and 204 / 7284
// with every candidate decided exactly and the terms handed round by lane reads).
// ---------------------------------------------------------------------------
constexpr int kWaveOwners = kBlock / 64;     // owners (waves) per workgroup

template <typename R, typename St>
__global__ __launch_bounds__(kBlock) void k_allpairs_wave(DevParams P, St in, St out, R* forces,
                                                          uint64_t* digest)
{
    __shared__ uint32_t list[kWaveOwners][128];
    __shared__ typename OrderedSums<R>::Terms terms[kWaveOwners];
    const uint32_t n = P.n;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t i = blockIdx.x * kWaveOwners + wave;
    if (i >= n) return;                                  // the whole wave
    uint32_t* near = list[wave];
    R px = in.x[i], py = in.y[i], pz = in.z[i], vx = in.vx[i], vy = in.vy[i], vz = in.vz[i];
    const R vn = norm3(vx, vy, vz);
    const R reach = reach_of(P, px, py, pz), F = Th<R>::image(P), inv_F = Th<R>::inv_image(P);
    OrderedSums<R> S;

    // candidate positions two batches ahead of the one being tested
    auto fetch = [&](uint32_t base, R& x, R& y, R& z) {
        const uint32_t j = min(base + lane, n - 1);
        x = in.x[j]; y = in.y[j]; z = in.z[j];
    };
    R ax = 0, ay = 0, az = 0, bx = 0, by = 0, bz = 0;
    fetch(0, ax, ay, az);
    if (64 < n) fetch(64, bx, by, bz);
    uint32_t held = 0;
    for (uint32_t base = 0; base < n; base += 64) {
        const R cx = ax, cy = ay, cz = az;
        ax = bx; ay = by; az = bz;
        if (base + 128 < n) fetch(base + 128, bx, by, bz);
        const uint32_t j = base + lane;
        const bool hit = (j < n) & (j != i) & (near2(cx - px, cy - py, cz - pz, F, inv_F) < reach);
        const uint64_t mask = __builtin_amdgcn_ballot_w64(hit);
        if (hit)
            near[held + __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                                  __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u))] = j;
        held += (uint32_t)__popcll(mask);
        wave_lds_order();
        const bool last = base + 64 >= n;
        while (held >= 64 || (last && held > 0)) {
            const uint32_t take = min(64u, held), rest = held - take;
            const uint32_t mine = near[lane], next = near[64 + lane];
            S.add(P, in, px, py, pz, vx, vy, vz, vn, lane, take, lane < take ? mine : 0u, terms[wave], digest != nullptr);
            if (lane < rest) near[lane] = next;
            wave_lds_order();
            held = rest;
        }
    }
    if (digest) S.hash_sums();
    const R dv[9] = {S.total(0), S.total(1), S.total(2), S.total(3), S.total(4),
                     S.total(5), S.total(6), S.total(7), S.total(8)};
    if (lane != 0) return;
    finish_ordered(P, S, dv, i, px, py, pz, vx, vy, vz, forces, digest);
    out.x[i] = px; out.y[i] = py; out.z[i] = pz; out.vx[i] = vx; out.vy[i] = vy; out.vz[i] = vz;
}

// The same for small flocks: four waves per boid test the candidates, a quarter
// of the batches each four at a time in flight, and leave each batch's
// ballot in LDS; the first wave expands the ballots (lane b those of batch b,
// hence at most 64 batches) into the list of ids and sums.  One update, one wave
// per boid / this: float N = 256 6.5 / 5.9 us, 1000 10.3 / 6.6, 2048 15.6 / 10.2,
// 4096 25.2 / 20.9; FP64 1024 11.3 / 7.8, 2048 15.9 / 13.4, 3000 22.8 / 21.2, 4096
// 31.5 / 31.9 (in double the chip is full by then: the line lies at 3072).
constexpr uint32_t kSmallFlock = 4096;

template <typename R, typename St>
__global__ __launch_bounds__(kBlock) void k_allpairs_small(DevParams P, St in, St out, R* forces, uint64_t* digest)
{
    __shared__ uint64_t ballots[kSmallFlock / 64];
    __shared__ uint16_t list[kSmallFlock];
    __shared__ typename OrderedSums<R>::Terms terms;
    const uint32_t n = P.n, i = blockIdx.x;              // the grid has one workgroup per boid
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    R px = in.x[i], py = in.y[i], pz = in.z[i], vx = in.vx[i], vy = in.vy[i], vz = in.vz[i];
    const R reach = reach_of(P, px, py, pz), F = Th<R>::image(P), inv_F = Th<R>::inv_image(P);
    const uint32_t batches = (n + 63) / 64;              // <= 64
    for (uint32_t b0 = wave; b0 < batches; b0 += 4 * kWaveOwners) {      // four batches' loads at once
        R x[4], y[4], z[4];
#pragma unroll
        for (uint32_t t = 0; t < 4; ++t) {
            const uint32_t at = min(64 * (b0 + t * kWaveOwners) + lane, n - 1);
            x[t] = in.x[at]; y[t] = in.y[at]; z[t] = in.z[at];
        }
#pragma unroll
        for (uint32_t t = 0; t < 4; ++t) {
            const uint32_t b = b0 + t * kWaveOwners, j = 64 * b + lane;
            const R s = near2(x[t] - px, y[t] - py, z[t] - pz, F, inv_F);
            const uint64_t mask = __builtin_amdgcn_ballot_w64((j < n) & (j != i) & (s < reach));
            if (lane == 0 && b < batches) ballots[b] = mask;
        }
    }
    __syncthreads();
    if (wave != 0) return;
    uint64_t mask = lane < batches ? ballots[lane] : 0;
    const uint32_t mine = (uint32_t)__popcll(mask);
    uint32_t incl = mine;
#pragma unroll
    for (uint32_t d = 1; d < 64; d <<= 1) {
        const uint32_t t = __shfl_up(incl, d, 64);
        if (lane >= d) incl += t;
    }
    const uint32_t held = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
    for (uint32_t at = incl - mine; mask; mask &= mask - 1)
        list[at++] = (uint16_t)(64 * lane + (uint32_t)__builtin_ctzll(mask));
    wave_lds_order();
    const R vn = norm3(vx, vy, vz);
    OrderedSums<R> S;
    for (uint32_t h = 0; h < held; h += 64)
        S.add(P, in, px, py, pz, vx, vy, vz, vn, lane, min(64u, held - h), h + lane < held ? (uint32_t)list[h + lane] : 0u,
              terms, digest != nullptr);
    if (digest) S.hash_sums();
    const R dv[9] = {S.total(0), S.total(1), S.total(2), S.total(3), S.total(4),
                     S.total(5), S.total(6), S.total(7), S.total(8)};
    if (lane != 0) return;
    finish_ordered(P, S, dv, i, px, py, pz, vx, vy, vz, forces, digest);
    out.x[i] = px; out.y[i] = py; out.z[i] = pz; out.vx[i] = vx; out.vy[i] = vy; out.vz[i] = vz;
}

// ---------------------------------------------------------------------------
// Grid build: cell hash + count, exclusive scan, scatter, in-cell rank +
// gather.  Sorted order is (cell, boid id), independent of history.  Keys
// are global over the flock table (flock cell_base + local cell).
// ---------------------------------------------------------------------------

__global__ __launch_bounds__(kBlock) void k_hash_count(Flocks F, StateF64 st, uint32_t* key,
                                                        uint32_t* rank, uint32_t* count)
{
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= F.n) return;
    const FlockDesc& fd = F.fl[flock_of(F, i)];
    const uint32_t c = fd.cell_base + cell_of(fd.P, st.x[i], st.y[i], st.z[i]);
    key[i] = c;
    rank[i] = atomicAdd(&count[c], 1u);
}

constexpr int kScanThreads = 1024;
constexpr int kScanItems = 4;
constexpr int kScanTile = kScanThreads * kScanItems;

// Tile-local exclusive scan of count[] into start[]; tile totals into
// partials[]; count[] is cleared for the next update's counts.
__global__ __launch_bounds__(kScanThreads) void k_scan_tiles(uint32_t* count, uint32_t* start,
                                                              uint32_t m, uint32_t* partials)
{
    __shared__ uint32_t wsum[17];
    const uint32_t base = blockIdx.x * kScanTile + threadIdx.x * kScanItems;
    uint32_t v[kScanItems];
    uint32_t sum = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        const uint32_t idx = base + k;
        v[k] = idx < m ? count[idx] : 0u;
        sum += v[k];
    }
    uint32_t total;
    uint32_t run = block_exclusive_scan(sum, wsum, &total);
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        const uint32_t idx = base + k;
        if (idx < m) { start[idx] = run; count[idx] = 0u; }
        run += v[k];
    }
    if (threadIdx.x == 0) partials[blockIdx.x] = total;
}

// The whole scan in one workgroup, up to TILES tiles: every thread loads its
// four counters of each tile at once, the waves scan theirs, and one wave
// scans the waves' totals of all tiles -- two barriers whatever TILES is.
template <int TILES>
__global__ __launch_bounds__(kScanThreads) void k_scan_small(uint32_t* count, uint32_t* start, uint32_t m)
{
    static_assert(kScanItems == 4 && kScanThreads == 1024, "16-byte loads, 16 waves");
    __shared__ uint32_t wsum[TILES * 16];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    uint4 v[TILES];
    uint32_t in[TILES];
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
        const uint32_t at = (uint32_t)t * kScanTile + threadIdx.x * 4;
        v[t] = make_uint4(0, 0, 0, 0);
        if (at + 4 <= m) v[t] = *(const uint4*)(count + at);
        else if (at < m) {
            v[t].x = count[at];
            if (at + 1 < m) v[t].y = count[at + 1];
            if (at + 2 < m) v[t].z = count[at + 2];
        }
    }
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
        const uint32_t s = v[t].x + v[t].y + v[t].z + v[t].w;
        uint32_t x = s;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t y = __shfl_up(x, d, 64);
            if (lane >= (uint32_t)d) x += y;
        }
        if (lane == 63) wsum[16 * t + wave] = x;
        in[t] = x - s;
    }
    __syncthreads();
    if (wave == 0) {
        constexpr int PER = (TILES * 16 + 63) / 64;
        uint32_t w[PER], sum = 0;
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            const uint32_t at = lane * PER + k;
            w[k] = at < TILES * 16 ? wsum[at] : 0u;
            sum += w[k];
        }
        uint32_t x = sum;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t y = __shfl_up(x, d, 64);
            if (lane >= (uint32_t)d) x += y;
        }
        x -= sum;
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            const uint32_t at = lane * PER + k;
            if (at < TILES * 16) wsum[at] = x;
            x += w[k];
        }
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
        const uint32_t at = (uint32_t)t * kScanTile + threadIdx.x * 4;
        const uint32_t r = in[t] + wsum[16 * t + wave];
        const uint4 o = make_uint4(r, r + v[t].x, r + v[t].x + v[t].y, r + v[t].x + v[t].y + v[t].z);
        if (at + 4 <= m) {
            *(uint4*)(start + at) = o;
            *(uint4*)(count + at) = make_uint4(0, 0, 0, 0);
        } else if (at < m) {
            start[at] = o.x; count[at] = 0u;
            if (at + 1 < m) { start[at + 1] = o.y; count[at + 1] = 0u; }
            if (at + 2 < m) { start[at + 2] = o.z; count[at + 2] = 0u; }
        }
    }
}

__global__ __launch_bounds__(kScanThreads) void k_scan_partials(uint32_t* partials, uint32_t nt)
{
    __shared__ uint32_t wsum[17];
    uint32_t carry = 0;
    for (uint32_t b = 0; b < nt; b += kScanThreads) {
        const uint32_t idx = b + threadIdx.x;
        const uint32_t v = idx < nt ? partials[idx] : 0u;
        uint32_t total;
        const uint32_t e = block_exclusive_scan(v, wsum, &total);
        if (idx < nt) partials[idx] = e + carry;
        carry += total;
    }
}

// Adds to every tile the totals of the tiles before it: partials[] holds the
// totals themselves (SUM; each workgroup then adds up the ones before its own)
// or their exclusive scan.
template <bool SUM>
__global__ __launch_bounds__(kScanThreads) void k_scan_add(uint32_t* start, uint32_t m,
                                                            const uint32_t* partials)
{
    __shared__ uint32_t wsum[17];
    uint32_t add = 0;
    if (SUM) {
        uint32_t mine = 0;
        for (uint32_t t = threadIdx.x; t < blockIdx.x; t += kScanThreads) mine += partials[t];
        block_exclusive_scan(mine, wsum, &add);
    } else {
        add = partials[blockIdx.x];
    }
    const uint32_t base = blockIdx.x * kScanTile + threadIdx.x * kScanItems;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        const uint32_t idx = base + k;
        if (idx < m) start[idx] += add;
    }
}

// Chunk table of the neighbour kernels, entries (local row, first slot, end
// slot, flock).  Every (y,z) row of cells of every flock (sx G x columns)
// is cut into groups of `span` consecutive columns, and every group into
// runs of `chunk` consecutive sorted boids, cut short where a run would cover
// more than `cspan` columns (sparse stretches), so a chunk lies in one
// row, holds at most `chunk` boids and its tile tables stay small.  A short
// cut moves the run's first column on by at least cspan, so a group has at
// most (span - 1) / cspan of them: the table holds at most n / chunk +
// groups * (1 + (span - 1) / cspan) entries.  One wave per row: the
// row's column starts are read into LDS (coalesced) and one lane walks them.
// Pass 1 counts the row's chunks; pass 2 writes them after those of the rows
// before it (rows in order: neighbouring rows' chunks stay adjacent in the
// table).
// The passes are the first workgroups of the two kernels that sort the boids
// (k_scatter_ranked, k_sort_runs), which need nothing of them: a launch of its
// own costs about 4.5 us whatever it does.  (Their workgroups all carry the rows'
// LDS, 16 bytes a column of the longest row; with 800 columns still no slower.)  While the rows are few (kRowsSum),
// pass 2 adds up the counts of the rows before its own; beyond that a scan
// between the two kernels leaves the offsets in `off`.
// One update, own launches / shared: FP64 N = 16384 159 / 152 us, mixed N = 50021
// 83 / 76, mixed N = 2^20 506 / 491, mixed N = 2^22 4525 / 4490 (6241 rows), 64
// flocks of 16384 735 / 726 (9216 rows).  At kRowsSum the sums read 134 MB of
// cached counts, about what the scan's launches cost.
//
// The bound is the table's capacity (`cap`); pass 2 writes no entry at or
// beyond it, and should the count ever exceed it, *nchunks is clamped to
// the capacity and the full count is left in *overflow (non-zero marks the
// table as cut short; the host reports it as an error).
constexpr int kRowWaves = kBlock / 64;
constexpr uint32_t kRowsSum = 16384;

template <bool WRITE>
__device__ __forceinline__ void rows_pass(const Flocks& F, const Rows& R, const uint32_t* __restrict__ start)
{
    extern __shared__ uint32_t rs[];            // kRowWaves x stride (>= the longest row's columns + 1)
    __shared__ uint32_t wsum[kRowWaves];
    const uint32_t w = threadIdx.x >> 6, lane = threadIdx.x & 63u;
    const uint32_t r0 = blockIdx.x * kRowWaves, r = r0 + w;
    uint32_t before = 0;                        // chunks of the rows before r
    if (WRITE && !R.off) {
        for (uint32_t q = threadIdx.x; q < r0 / 4; q += kBlock) {     // (kRowWaves = 4: whole quads)
            const uint4 c = ((const uint4*)R.count)[q];
            before += c.x + c.y + c.z + c.w;
        }
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) before += __shfl_xor(before, d, 64);
        if (lane == 0) wsum[w] = before;
        __syncthreads();
        before = wsum[0] + wsum[1] + wsum[2] + wsum[3];
        for (uint32_t q = r0; q < min(r, F.rows); ++q) before += R.count[q];
    } else if (WRITE && r < F.rows) {
        before = R.off[r];
    }
    if (r >= F.rows) return;                    // whole waves only: no barrier follows
    const uint32_t f = F.row_flock ? F.row_flock[r] : 0u;
    const FlockDesc& fd = F.fl[f];
    const uint32_t G = (uint32_t)fd.P.sx * (uint32_t)fd.P.G, span = fd.span;   // x columns of the row
    const uint32_t rl = r - fd.row_base;
    const uint32_t c0 = fd.cell_base + rl * G;
    uint32_t* cs = rs + w * R.stride;
    for (uint32_t x = lane; x <= G; x += 64) cs[x] = start[c0 + x];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if (lane != 0) return;
    uint32_t k = before;
    for (uint32_t x0 = 0; x0 < G; x0 += span) {
        const uint32_t x1 = min(G, x0 + span);
        const uint32_t hi = cs[x1];
        uint32_t t0 = cs[x0], xa = x0, next = 0, lim = 0;
        while (t0 < hi) {
            if (next <= t0) {                       // cell of boid t0; crowded cells keep it from chunk to
                                                    // chunk (N = 16384 in 64 blobs, an update: 139.5 -> 135 us)
                while ((next = cs[xa + 1]) <= t0) ++xa;
                lim = xa + R.cspan < x1 ? cs[xa + R.cspan] : hi;
            }
            const uint32_t t1 = min(lim, t0 + R.chunk);
            if (WRITE && k < R.cap) R.table[k] = make_uint4(rl, t0, t1, f);
            ++k;
            t0 = t1;
        }
    }
    if (!WRITE) {
        R.count[r] = k;
    } else if (r + 1 == F.rows) {
        *R.nchunks = min(k, R.cap);
        if (k > R.cap) *R.overflow = k;
    }
}

// The first R.blocks workgroups count the rows' chunks.
__global__ __launch_bounds__(kBlock) void k_scatter_ranked(Flocks F, Rows R, const uint32_t* __restrict__ key,
                                                           const uint32_t* __restrict__ rank,
                                                           const uint32_t* __restrict__ start,
                                                           const uint32_t* __restrict__ id, uint32_t* perm,
                                                           uint32_t* permid)
{
    if (blockIdx.x < R.blocks) { rows_pass<false>(F, R, start); return; }
    const uint32_t s = (blockIdx.x - R.blocks) * kBlock + threadIdx.x;
    if (s >= F.n) return;
    const uint32_t t = start[key[s]] + rank[s];
    perm[t] = s;
    permid[t] = id[s];
}

// In-cell order, step 1: every run of 64 consecutive slots (one wave) is
// sorted by (cell, id) in registers, in place: a bitonic network across the
// wave's lanes over (cell part within the run, id) -- the slots are grouped
// by cell already, so this sorts each cell's part inside the run.  A cell
// spanning runs leaves one ascending part per run, which k_gather merges.
// Keys are 32-bit (6-bit part index, 26-bit id) when every id is below 2^26,
// else 64-bit.  A run already in order (the common case: boids arriving from
// one old cell are ranked in lane order) is left alone.  The first R.blocks
// workgroups write the rows' chunks.
template <typename K>
__device__ __forceinline__ K shfl_xor_key(K v, uint32_t m)
{
    if constexpr (sizeof(K) == 4) {
        return (K)__shfl_xor((uint32_t)v, m, 64);
    } else {
        const uint32_t lo = __shfl_xor((uint32_t)v, m, 64), hi = __shfl_xor((uint32_t)(v >> 32), m, 64);
        return ((K)hi << 32) | lo;
    }
}

template <typename K>
__global__ __launch_bounds__(kBlock) void k_sort_runs(Flocks F, Rows R, const uint32_t* __restrict__ key,
                                                      const uint32_t* __restrict__ start, uint32_t* perm,
                                                      uint32_t* permid)
{
    if (blockIdx.x < R.blocks) { rows_pass<true>(F, R, start); return; }
    const uint32_t t = (blockIdx.x - R.blocks) * kBlock + threadIdx.x;
    const uint32_t lane = threadIdx.x & 63u;
    const bool in = t < F.n;
    uint32_t p = 0u, id = 0u, c = 0xFFFFFFFFu;
    if (in) {
        p = perm[t];
        id = permid[t];
        c = key[p];
    }
    const uint32_t cp = __shfl_up(c, 1, 64), ip = __shfl_up(id, 1, 64);
    const bool fresh = lane == 0 || cp != c;         // first slot of a cell's part
    if (__builtin_amdgcn_ballot_w64(in && !fresh && ip > id) == 0) return;   // wave-uniform
    const uint64_t starts = __builtin_amdgcn_ballot_w64(fresh);
    const uint32_t part = __builtin_amdgcn_mbcnt_hi((uint32_t)(starts >> 32),
                                                    __builtin_amdgcn_mbcnt_lo((uint32_t)starts, 0u)) +
                          (fresh ? 1u : 0u) - 1u;     // parts begun at or before this lane, minus one
    constexpr uint32_t kShift = sizeof(K) == 4 ? 26u : 32u;
    K k = in ? (((K)part << kShift) | (K)id) : ~(K)0;   // past the end: sorts last, never written
    for (uint32_t size = 2; size <= 64; size <<= 1) {
        for (uint32_t stride = size >> 1; stride > 0; stride >>= 1) {
            const K pk = shfl_xor_key(k, stride);
            const uint32_t pp = __shfl_xor(p, stride, 64);
            // ascending blocks of `size` where lane & size == 0: the lower
            // lane of a pair keeps the smaller key there, the larger elsewhere
            const bool keep_min = ((lane & stride) == 0) == ((lane & size) == 0);
            if (keep_min ? pk < k : pk > k) { k = pk; p = pp; }
        }
    }
    if (in) {
        perm[t] = p;
        permid[t] = (uint32_t)(k & (((K)1 << kShift) - 1));
    }
}

// In-cell order, step 2: final slot = cell start + rank of the boid id among
// its cell's ids, so the order inside a cell is ascending id whatever the
// atomics did.  The rank is the slot's position in its own sorted part plus
// a binary search in each other part of the cell (k_sort_runs): O(1) for a
// cell inside one run, O(occupancy / 64 * log 64) for a dense one, instead
// of a pass over the whole cell per boid (a scan of short parts instead of
// the search measured slower: its loop is as long as the part).
__global__ __launch_bounds__(kBlock) void k_gather(Flocks F, const uint32_t* perm,
                                                   const uint32_t* permid, const uint32_t* key,
                                                   const uint32_t* start, StateF64 src, StateF64 dst,
                                                   uint32_t* key_sorted, Lattice lat, int with_lat,
                                                   double2* rec)
{
    const uint32_t t = blockIdx.x * kBlock + threadIdx.x;
    if (t >= F.n) return;
    const uint32_t s = perm[t];
    const uint32_t me = permid[t];
    const uint32_t c = key[s];
    const uint32_t lo = start[c], hi = start[c + 1];
    const uint32_t run = t >> 6;
    uint32_t rank = t - max(lo, run << 6);
    for (uint32_t v = lo >> 6; (v << 6) < hi; ++v) {
        if (v == run) continue;
        const uint32_t a = max(lo, v << 6), b = min(hi, (v + 1) << 6);
        rank += count_below(permid + a, b - a, me);
    }
    const uint32_t f = lo + rank;
    const double x = src.x[s], y = src.y[s], z = src.z[s];
    const double vx = src.vx[s], vy = src.vy[s], vz = src.vz[s];
    dst.x[f] = x; dst.y[f] = y; dst.z[f] = z;
    dst.vx[f] = vx; dst.vy[f] = vy; dst.vz[f] = vz;
    dst.id[f] = me;
    key_sorted[f] = c;
    if (with_lat) {
        const DevParams& P = F.fl[flock_of(F, f)].P;   // slots stay inside their flock
        const double scale = P.lat_scale;
        const bool nan_state = x != x || y != y || z != z || vx != vx || vy != vy || vz != vz;
        const uint32_t nanv = nan_state ? 0x80000000u : 0u;   // NaN state mark
        lat.p[f] = make_uint4(to_lattice(x, scale), to_lattice(y, scale), to_lattice(z, scale),
                              pack_sub(x, y, z, scale) | nanv);
        const double iq = P.inv_vq;
        lat.v[f] = make_float4((float)rint(vx * iq), (float)rint(vy * iq), (float)rint(vz * iq), 0.f);
    }
    if (rec) {                                 // three planes of n records: (x, y), (z, vx), (vy, vz)
        rec[f] = make_double2(x, y);
        rec[(size_t)F.n + f] = make_double2(z, vx);
        rec[2 * (size_t)F.n + f] = make_double2(vy, vz);
    }
}

// State in id order, three values per boid (T = the type the caller asked for).
template <typename T>
__global__ __launch_bounds__(kBlock) void k_unsort_f64(uint32_t n, StateF64 src, T* pos3, T* vel3)
{
    const uint32_t s = blockIdx.x * kBlock + threadIdx.x;
    if (s >= n) return;
    const size_t i = src.id[s];
    pos3[3 * i] = (T)src.x[s]; pos3[3 * i + 1] = (T)src.y[s]; pos3[3 * i + 2] = (T)src.z[s];
    vel3[3 * i] = (T)src.vx[s]; vel3[3 * i + 1] = (T)src.vy[s]; vel3[3 * i + 2] = (T)src.vz[s];
}

// A state that is in id order already, one value per thread: consecutive
// threads write consecutive words, also where out lies in host memory.
template <typename T, typename St>
__global__ __launch_bounds__(kBlock) void k_pack(uint32_t n, St st, T* pos3, T* vel3)
{
    const uint32_t k = blockIdx.x * kBlock + threadIdx.x;
    const uint32_t i = k / 3, c = k - 3 * i;
    if (i >= n) return;
    pos3[k] = (T)(c == 0 ? st.x : c == 1 ? st.y : st.z)[i];
    vel3[k] = (T)(c == 0 ? st.vx : c == 1 ? st.vy : st.vz)[i];
}

// Uploaded state: pos and vel hold boid i's three values at stride * i.
template <typename T>
__global__ __launch_bounds__(kBlock) void k_unpack_f64(uint32_t n, const T* __restrict__ pos,
                                                       const T* __restrict__ vel, uint32_t stride, StateF64 st)
{
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const T *p = pos + (size_t)stride * i, *v = vel + (size_t)stride * i;
    st.x[i] = p[0]; st.y[i] = p[1]; st.z[i] = p[2];
    st.vx[i] = v[0]; st.vy[i] = v[1]; st.vz[i] = v[2];
    st.id[i] = i;
}

__global__ __launch_bounds__(kBlock) void k_unpack_f32(uint32_t n, const float* __restrict__ xyzv6, StateF32 st)
{
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const float* p = xyzv6 + 6 * (size_t)i;
    st.x[i] = p[0]; st.y[i] = p[1]; st.z[i] = p[2];
    st.vx[i] = p[3]; st.vy[i] = p[4]; st.vz[i] = p[5];
}

// Launchers
// ---------------------------------------------------------------------------
static inline uint32_t blocks_for(uint32_t n) { return (n + kBlock - 1) / kBlock; }

template <typename R, typename St>
static hipError_t launch_allpairs(const DevParams& P, St in, St out, R* forces, uint64_t* digest, hipStream_t stream)
{
    if (P.n == 0) return hipSuccess;
    if (P.n <= (sizeof(R) == 4 ? kSmallFlock : 3072))      // k_allpairs_small has the figures
        hipLaunchKernelGGL((k_allpairs_small<R, St>), dim3(P.n), dim3(kBlock), 0, stream, P, in, out, forces, digest);
    else
        hipLaunchKernelGGL((k_allpairs_wave<R, St>), dim3((P.n + kWaveOwners - 1) / kWaveOwners), dim3(kBlock), 0,
                           stream, P, in, out, forces, digest);
    return hipGetLastError();
}

hipError_t launch_allpairs_f32ref(const DevParams& P, StateF32 in, StateF32 out, float* forces,
                                  uint64_t* digest, hipStream_t stream)
{
    return launch_allpairs(P, in, out, forces, digest, stream);
}

hipError_t launch_allpairs_f64(const DevParams& P, StateF64 in, StateF64 out, double* forces,
                               uint64_t* digest, hipStream_t stream)
{
    return launch_allpairs(P, in, out, forces, digest, stream);
}

hipError_t launch_hash_count(Flocks F, StateF64 st, uint32_t* key, uint32_t* rank, uint32_t* count,
                             hipStream_t stream)
{
    if (F.n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_hash_count, dim3(blocks_for(F.n)), dim3(kBlock), 0, stream, F, st, key, rank, count);
    return hipGetLastError();
}

// By size: one workgroup up to 8 tiles (13825 counters: 4.8 us, three launches
// took 13; a workgroup's loads of 128 KB cost about a launch, so more tiles go
// to more workgroups); beyond that two launches, the second adding up the totals of the tiles before each tile
// itself, while these are few enough to read in a turn or two; else three.
// count and start are 16-byte aligned.
hipError_t launch_scan(uint32_t* count, uint32_t* start, uint32_t m, uint32_t* partials,
                       hipStream_t stream)
{
    const uint32_t nt = (m + kScanTile - 1) / kScanTile;
    const dim3 one(1), tiles(nt), threads(kScanThreads);
    if (nt <= 1) {
        hipLaunchKernelGGL(k_scan_small<1>, one, threads, 0, stream, count, start, m);
    } else if (nt <= 4) {
        hipLaunchKernelGGL(k_scan_small<4>, one, threads, 0, stream, count, start, m);
    } else if (nt <= 8) {
        hipLaunchKernelGGL(k_scan_small<8>, one, threads, 0, stream, count, start, m);
    } else {
        hipLaunchKernelGGL(k_scan_tiles, tiles, threads, 0, stream, count, start, m, partials);
        if (nt <= 2 * kScanThreads) {
            hipLaunchKernelGGL(k_scan_add<true>, tiles, threads, 0, stream, start, m, (const uint32_t*)partials);
        } else {
            hipLaunchKernelGGL(k_scan_partials, one, threads, 0, stream, partials, nt);
            hipLaunchKernelGGL(k_scan_add<false>, tiles, threads, 0, stream, start, m, (const uint32_t*)partials);
        }
    }
    return hipGetLastError();
}

hipError_t launch_scatter_ranked(Flocks F, Rows R, int max_cols, uint32_t* row_off, uint32_t* partials,
                                 const uint32_t* key, const uint32_t* rank, const uint32_t* start, const uint32_t* id,
                                 uint32_t* perm, uint32_t* permid, hipStream_t stream)
{
    if (F.count == 0 || R.chunk == 0 || F.rows == 0 || R.cspan < 1 || R.cspan > kChunkSpanMax || max_cols < 1 ||
        max_cols > kSubXMax * kMaxCells)
        return hipErrorInvalidValue;
    R.blocks = (F.rows + kRowWaves - 1) / kRowWaves;
    R.stride = (uint32_t)max_cols + 1;
    const dim3 grid(R.blocks + blocks_for(F.n));
    const size_t dyn = sizeof(uint32_t) * kRowWaves * R.stride;
    hipLaunchKernelGGL(k_scatter_ranked, grid, dim3(kBlock), dyn, stream, F, R, key, rank, start, id, perm, permid);
    hipError_t err = hipGetLastError();
    if (err != hipSuccess) return err;
    R.off = nullptr;
    if (F.rows > kRowsSum) {
        if ((err = launch_scan(R.count, row_off, F.rows, partials, stream)) != hipSuccess) return err;
        R.off = row_off;
    }
    if (F.n <= (1u << 26))
        hipLaunchKernelGGL(k_sort_runs<uint32_t>, grid, dim3(kBlock), dyn, stream, F, R, key, start, perm, permid);
    else
        hipLaunchKernelGGL(k_sort_runs<uint64_t>, grid, dim3(kBlock), dyn, stream, F, R, key, start, perm, permid);
    return hipGetLastError();
}

hipError_t launch_gather(Flocks F, const uint32_t* perm, const uint32_t* permid, const uint32_t* key,
                         const uint32_t* start, StateF64 src, StateF64 dst, uint32_t* key_sorted, Lattice* lat,
                         double2* rec, hipStream_t stream)
{
    if (F.n == 0) return hipSuccess;
    Lattice l = lat ? *lat : Lattice{nullptr, nullptr};
    hipLaunchKernelGGL(k_gather, dim3(blocks_for(F.n)), dim3(kBlock), 0, stream, F, perm, permid,
                       key, start, src, dst, key_sorted, l, lat ? 1 : 0, rec);
    return hipGetLastError();
}

// Plain streaming copy (16 B per lane per iteration): the reference point
// for HBM byte counters (a copy of B bytes moves exactly B in and B out).
__global__ __launch_bounds__(kBlock) void k_copy(const uint4* __restrict__ src, uint4* __restrict__ dst,
                                                 uint64_t n16)
{
    for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < n16; i += (uint64_t)gridDim.x * kBlock)
        dst[i] = src[i];
}

hipError_t launch_copy(const void* src, void* dst, uint64_t bytes, hipStream_t stream)
{
    const uint64_t n16 = bytes / 16;
    if (n16 == 0) return hipSuccess;
    const uint64_t want = (n16 + kBlock - 1) / kBlock;
    const uint32_t grid = (uint32_t)(want < 65536 ? want : 65536);
    hipLaunchKernelGGL(k_copy, dim3(grid), dim3(kBlock), 0, stream, (const uint4*)src, (uint4*)dst, n16);
    return hipGetLastError();
}

hipError_t launch_unsort_f64(uint32_t n, StateF64 src, double* pos3, double* vel3, hipStream_t stream)
{
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_unsort_f64<double>, dim3(blocks_for(n)), dim3(kBlock), 0, stream, n, src, pos3, vel3);
    return hipGetLastError();
}

hipError_t launch_unsort_f64(uint32_t n, StateF64 src, float* pos3, float* vel3, hipStream_t stream)
{
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_unsort_f64<float>, dim3(blocks_for(n)), dim3(kBlock), 0, stream, n, src, pos3, vel3);
    return hipGetLastError();
}

hipError_t launch_pack_f32(uint32_t n, StateF32 st, float* pos3, float* vel3, hipStream_t stream)
{
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL((k_pack<float, StateF32>), dim3(blocks_for(3 * n)), dim3(kBlock), 0, stream, n, st, pos3, vel3);
    return hipGetLastError();
}

hipError_t launch_pack_f32(uint32_t n, StateF32 st, double* pos3, double* vel3, hipStream_t stream)
{
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL((k_pack<double, StateF32>), dim3(blocks_for(3 * n)), dim3(kBlock), 0, stream, n, st, pos3, vel3);
    return hipGetLastError();
}

hipError_t launch_pack_f64(uint32_t n, StateF64 st, float* pos3, float* vel3, hipStream_t stream)
{
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL((k_pack<float, StateF64>), dim3(blocks_for(3 * n)), dim3(kBlock), 0, stream, n, st, pos3, vel3);
    return hipGetLastError();
}

hipError_t launch_pack_f64(uint32_t n, StateF64 st, double* pos3, double* vel3, hipStream_t stream)
{
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL((k_pack<double, StateF64>), dim3(blocks_for(3 * n)), dim3(kBlock), 0, stream, n, st, pos3, vel3);
    return hipGetLastError();
}

hipError_t launch_unpack(uint32_t n, const double* pos3, const double* vel3, StateF64 st, hipStream_t stream)
{
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_unpack_f64<double>, dim3(blocks_for(n)), dim3(kBlock), 0, stream, n, pos3, vel3, 3u, st);
    return hipGetLastError();
}

hipError_t launch_unpack(uint32_t n, const float* xyzv6, StateF64 st, hipStream_t stream)
{
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_unpack_f64<float>, dim3(blocks_for(n)), dim3(kBlock), 0, stream, n, xyzv6, xyzv6 + 3, 6u, st);
    return hipGetLastError();
}

hipError_t launch_unpack(uint32_t n, const float* xyzv6, StateF32 st, hipStream_t stream)
{
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_unpack_f32, dim3(blocks_for(n)), dim3(kBlock), 0, stream, n, xyzv6, st);
    return hipGetLastError();
}

}  // namespace boids
