// boids_f32grid.hip — reference-faithful float grid step (BS_MODE_GRID_F32REF):
// what boidsim_grid computes (src/boid_simulation_grid.cpp:165-293), bit for
// bit.  The reference's grid engine equals its all-pairs engine exactly
// because each boid's candidates are visited in ascending index order
// (:186 copies the primary cell's list; phase A of :153-212 sums in float in
// visit order).  Here the cell list is a counting sort of the float state by
// cell; one wave per owner collects the boids of its 27 cells within the
// largest radius, sorts them by id and adds their terms in ascending id, so
// every float sum adds the same terms in the same order as the reference (an
// owner with more boids in reach than the wave's list holds takes them in
// several windows of ascending ids).  The state stays in id order (as
// boidsim keeps it).
//
// Compiled with -ffp-contract=off: every multiply and add is rounded on its
// own, as the reference's x86-64 build computes it.
#include "boids_device.h"

#include <type_traits>

namespace boids {

// The cells are P.sx to a cell edge on every axis (edge >= the largest
// radius), so a boid's neighbours lie within P.sx cells of its own.
__device__ __forceinline__ uint32_t cell_f32(const DevParams& P, float x, float y, float z)
{
    const uint32_t G = (uint32_t)(P.sx * P.G);
    const double k = (double)P.sx * P.inv_edge;
    return axis_cell((double)x, k, (int)G) + G * (axis_cell((double)y, k, (int)G) + G * axis_cell((double)z, k, (int)G));
}

// Whether a boid lies in the field (its cell then bounds its position): if
// any does not, the step leaves no cell of the 27 out.
__device__ __forceinline__ bool in_field(const DevParams& P, float x, float y, float z)
{
    const double F = P.F * (1.0 + 1e-7);           // (the field edge itself may round up)
    return (double)x >= 0.0 && (double)x <= F && (double)y >= 0.0 && (double)y <= F && (double)z >= 0.0 && (double)z <= F;
}

// Cell key of every boid (id order) and its arrival rank in the cell, for a
// state from outside (k_f32_grid_wave leaves them for the state it writes).
__global__ __launch_bounds__(kBlock) void k_f32_hash(DevParams P, StateF32 st, uint32_t* key, uint32_t* rank,
                                                     uint32_t* count, uint32_t* outside)
{
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= P.n) return;
    const uint32_t c = cell_f32(P, st.x[i], st.y[i], st.z[i]);
    if (!in_field(P, st.x[i], st.y[i], st.z[i])) *outside = 1u;
    key[i] = c;
    rank[i] = atomicAdd(&count[c], 1u);
}

// The candidates' records, grouped by cell in arrival order (the step sorts
// what it keeps by id, so no order inside a cell is needed): position, id in .w.
__global__ __launch_bounds__(kBlock) void k_f32_cells(uint32_t n, StateF32 st, const uint32_t* __restrict__ key,
                                                      const uint32_t* __restrict__ rank,
                                                      const uint32_t* __restrict__ start, float4* rec)
{
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    rec[start[key[i]] + rank[i]] = make_float4(st.x[i], st.y[i], st.z[i], __builtin_bit_cast(float, i));
}

// Smaller (keep = 0) or larger (keep = ~0) of v and lane l ^ S's v, without
// LDS: cross-lane operand modifiers for 1, 2, 4 and 8 (4 = 7 ^ 3), row and half
// swaps for 16 and 32 (which leave a lane its own and its partner's value in
// some order); the median with 0 or ~0 selects.
__device__ __forceinline__ uint32_t med3_u32(uint32_t a, uint32_t b, uint32_t c)
{
    return min(max(min(a, b), c), max(a, b));
}
template <uint32_t S>
__device__ __forceinline__ uint32_t keep_of(uint32_t v, uint32_t keep)
{
    auto dpp = [](uint32_t x, auto ctrl) {
        return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, decltype(ctrl)::value, 0xF, 0xF, true);
    };
    if constexpr (S == 1) return med3_u32(v, dpp(v, std::integral_constant<int, 0xB1>{}), keep);        // quad_perm [1,0,3,2]
    else if constexpr (S == 2) return med3_u32(v, dpp(v, std::integral_constant<int, 0x4E>{}), keep);   // quad_perm [2,3,0,1]
    else if constexpr (S == 4)
        return med3_u32(v, dpp(dpp(v, std::integral_constant<int, 0x141>{}), std::integral_constant<int, 0x1B>{}), keep);
    else if constexpr (S == 8) return med3_u32(v, dpp(v, std::integral_constant<int, 0x128>{}), keep);  // row_ror 8
    else if constexpr (S == 16) {
        const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
        return med3_u32(r[0], r[1], keep);
    } else {
        const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
        return med3_u32(r[0], r[1], keep);
    }
}

// Bitonic sort, ascending, of 64 R keys: element 64 r + lane in k[r].  Steps
// across lanes go by keep_of (through LDS permutes a step waited ~100 cycles
// and took twice the instructions), steps across registers are local.
template <uint32_t R, uint32_t SIZE, uint32_t S>
__device__ __forceinline__ void sort_step(uint32_t (&k)[R], uint32_t lane)
{
    if constexpr (S >= 64) {
        constexpr uint32_t D = S / 64;
#pragma unroll
        for (uint32_t r = 0; r < R; ++r) {
            if (r & D) continue;                                   // handled with its partner
            const bool asc = ((64 * r) & SIZE) == 0;
            const uint32_t lo = min(k[r], k[r + D]), hi = max(k[r], k[r + D]);
            k[r] = asc ? lo : hi;
            k[r + D] = asc ? hi : lo;
        }
    } else {
        // ascending parts: the lane with bit S keeps the larger key; where SIZE
        // is a lane bit, the parts with it set descend
        const uint32_t s = (lane & S) ? ~0u : 0u, d = SIZE < 64 && (lane & SIZE) ? ~0u : 0u;
#pragma unroll
        for (uint32_t r = 0; r < R; ++r) k[r] = keep_of<S>(k[r], SIZE >= 64 && ((64 * r) & SIZE) ? ~s : s ^ d);
    }
    if constexpr (S > 1) sort_step<R, SIZE, S / 2>(k, lane);
    else if constexpr (SIZE < 64 * R) sort_step<R, SIZE * 2, SIZE>(k, lane);
}

// One one-wave workgroup per owner (id order).  (1) The lanes test the
// candidates, 64 at a time, against a bound just above the largest radius and
// append the ids of those within it to an LDS list.  The candidates are the
// boids of the cells that the sphere around the owner touches: lane r holds
// row r of the window (a run of slots, in two parts where it wraps around the
// field), cut to the sphere's extent in that row.  (2) The list is sorted
// (sort_step in registers up to 256 ids, a bitonic network in LDS beyond).
// (3) 64 sorted boids at a time go through OrderedSums.
//
// What bounds it: the waves' own instruction and latency chains (16384 owners
// are 16 waves per SIMD in all).  At N = 16384, uniform / 64 blobs, VALU issue is
// 75 / 53 %, lanes 56 / 64 %, and on average 3.7 / 2.5 waves are resident: in
// blobs the owners of long lists finish last.  One update of the whole engine at N = 16384,
// uniform / 64 blobs: 74.5 / 111.5 us with 27 whole cells an owner, a sort
// through LDS permutes, a launch for each of five build steps; 58 / 94 with two
// build launches and sort_step; 54 / 86 with half cells cut to the sphere and
// the scan in one workgroup; 51 / 85 with the minimum image in one rounding and
// the median selects; 49 / 81 at 6 waves per SIMD (5: 49 / 82, 7: 52 / 85; the
// compiler's own choice is 4).
constexpr uint32_t kF32HitCap = 1024;        // boids per owner sorted in LDS
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(6)))
void k_f32_grid_wave(DevParams P, StateF32 in, StateF32 out, const float4* __restrict__ rec, uint32_t* key,
                     uint32_t* rank, const uint32_t* __restrict__ start, uint32_t* count, uint32_t* outside,
                     float* forces, uint64_t* digest)
{
    __shared__ __align__(16) uint32_t hb[kF32HitCap];
    __shared__ OrderedSums<float>::Terms terms;
    const uint32_t lane = threadIdx.x;
    const uint32_t i = blockIdx.x;                     // the grid has one workgroup per boid
    const float px = in.x[i], py = in.y[i], pz = in.z[i];
    const float vx = in.vx[i], vy = in.vy[i], vz = in.vz[i];
    const float vn = norm3(vx, vy, vz);
    const int sub = P.sx, G = sub * P.G;
    const double kc = (double)sub * P.inv_edge;        // the cell as cell_f32 has it
    const int cx = (int)axis_cell((double)px, kc, G), cy = (int)axis_cell((double)py, kc, G),
              cz = (int)axis_cell((double)pz, kc, G);
    // some boid is not where its cell is (set while this launch runs if one it
    // writes is not; either value will do then), or the field has no filter
    const bool all = __builtin_amdgcn_readfirstlane((int)__hip_atomic_load(outside, __ATOMIC_RELAXED,
                                                                           __HIP_MEMORY_SCOPE_AGENT)) != 0 ||
                     P.reach_cells < 0.f;

    // Lane r: row r of the window, cells cx + x0 .. cx + x1 of it (unwrapped).
    // Ordinarily the (2 sub + 1)^2 rows within sub cells, each cut to the
    // sphere; with a boid outside the field the 27 whole cells around the
    // owner's, uncut.
    const float inv_h = (float)kc;                     // cells per unit
    const int side = all ? 3 * sub : 2 * sub + 1;
    const int lo_y = all ? (cy / sub - 1) * sub - cy : -sub, lo_z = all ? (cz / sub - 1) * sub - cz : -sub;
    const int q = (int)lane;
    const int dy = lo_y + q % side, dz = lo_z + q / side;
    int x0 = all ? (cx / sub - 1) * sub - cx : -sub, x1 = x0 + side - 1;
    bool touched = q < side * side;
    if (!all) {
        // distance from the owner to the row's square of cells, in cells, and the
        // sphere's half-width there (margins of 1e-3 cells cover the rounding)
        const float R = P.reach_cells + 1e-3f;
        const float fy = py * inv_h - (float)cy, fz = pz * inv_h - (float)cz, fx = px * inv_h - (float)cx;
        const float gy = fmaxf(fmaxf((float)dy - fy, fy - (float)(dy + 1)), 0.f);
        const float gz = fmaxf(fmaxf((float)dz - fz, fz - (float)(dz + 1)), 0.f);
        const float w2 = R * R - gy * gy - gz * gz;
        touched = touched && w2 > 0.f;
        const float w = __builtin_amdgcn_sqrtf(fmaxf(w2, 0.f)) + 1e-3f;
        x0 = max(x0, (int)floorf(fx - w));
        x1 = min(x1, (int)floorf(fx + w));
        touched = touched && x0 <= x1;
    }
    uint32_t a0 = 0, n0 = 0, a1 = 0, n1 = 0;           // the run's first part, and the part that wraps
    if (touched) {
        int y = cy + dy, z = cz + dz;
        y += y < 0 ? G : (y >= G ? -G : 0);
        z += z < 0 ? G : (z >= G ? -G : 0);
        const uint32_t row = (uint32_t)G * ((uint32_t)y + (uint32_t)G * (uint32_t)z);
        const int u0 = cx + x0, u1 = cx + x1;
        const int m0 = max(u0, 0), m1 = min(u1, G - 1);
        if (m0 <= m1) { a0 = start[row + (uint32_t)m0]; n0 = start[row + (uint32_t)m1 + 1] - a0; }
        if (u0 < 0) {
            const int e = min(u1, -1) + G;
            a1 = start[row + (uint32_t)(u0 + G)];
            n1 = start[row + (uint32_t)e + 1] - a1;
        } else if (u1 >= G) {
            const int b = max(u0, G) - G;
            a1 = start[row + (uint32_t)b];
            n1 = start[row + (uint32_t)(u1 - G) + 1] - a1;
        }
    }
    uint32_t incl = n0 + n1;
#pragma unroll
    for (uint32_t d = 1; d < 64; d <<= 1) {
        const uint32_t t = __shfl_up(incl, d, 64);
        if (lane >= d) incl += t;
    }
    const uint32_t excl = incl - n0 - n1;              // non-decreasing over the lanes
    const uint32_t M = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
    const bool wraps = __builtin_amdgcn_ballot_w64(n1 != 0) != 0;
    const uint32_t b0 = a0 - excl, b1 = a1 - excl - n0, e0 = excl + n0;

    // (1) the boids within reach whose ids lie in [lo, lo + width): appended to
    // the list as far as it holds them, their number returned.  A superset of
    // the boids within the largest radius will do ((3) decides exactly): the
    // minimum image is taken with one rounding (near2).  Each
    // batch's records are fetched while the previous batch is tested.
    const float Ff = P.image_f, inv_F = P.inv_image_f, reach = reach_of(P, px, py, pz);
    auto record_of = [&](uint32_t m0) {
        const uint32_t m = min(m0 + lane, M - 1);
        // the last row k with excl[k] <= m (binary lifting over the lanes; rows
        // are at most 36)
        uint32_t k = 0;
#pragma unroll
        for (uint32_t st = 32; st > 0; st >>= 1) {
            const uint32_t pr = min(k + st, 63u);
            k = (uint32_t)__shfl((int)excl, (int)pr, 64) <= m ? pr : k;
        }
        uint32_t slot = m + (uint32_t)__shfl((int)b0, (int)k, 64);
        if (wraps) {                                   // (uniform: the permutes read all lanes)
            const uint32_t end = (uint32_t)__shfl((int)e0, (int)k, 64), other = (uint32_t)__shfl((int)b1, (int)k, 64);
            slot = m >= end ? m + other : slot;
        }
        return rec[slot];
    };
    auto collect = [&](uint32_t lo, uint32_t width) __attribute__((always_inline)) {
        uint32_t H = 0;
        float4 qn = M ? record_of(0) : make_float4(0.f, 0.f, 0.f, 0.f);
        for (uint32_t m0 = 0; m0 < M; m0 += 64) {
            const float4 q = qn;
            if (m0 + 64 < M) qn = record_of(m0 + 64);
            const uint32_t j = __builtin_bit_cast(uint32_t, q.w);
            const float s = near2(px - q.x, py - q.y, pz - q.z, Ff, inv_F);
            const bool hit = (m0 + lane < M) & (j != i) & (j - lo < width) & (s < reach);
            const uint64_t mask = __builtin_amdgcn_ballot_w64(hit);
            const uint32_t pos = H + __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                                               __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
            if (hit && pos < kF32HitCap) hb[pos] = j;
            H += (uint32_t)__popcll(mask);
        }
        return H;
    };

    OrderedSums<float> S;
    auto sorted = [&](auto regs, uint32_t H) __attribute__((always_inline)) {
        constexpr uint32_t R = decltype(regs)::value;
        uint32_t k[R];
#pragma unroll
        for (uint32_t r = 0; r < R; ++r) k[r] = 64 * r + lane < H ? hb[64 * r + lane] : ~0u;
        sort_step<R, 2, 1>(k, lane);
#pragma unroll
        for (uint32_t r = 0; r < R; ++r) hb[64 * r + lane] = k[r];
    };

    for (IdWindows ids(P.n, kF32HitCap); ids.more();) {
        const uint32_t H = collect(ids.lo, ids.width);
        if (!ids.take(H)) continue;
        wave_lds_order();
        if (H <= 64) {
            sorted(std::integral_constant<uint32_t, 1>{}, H);
        } else if (H <= 128) {
            sorted(std::integral_constant<uint32_t, 2>{}, H);
        } else if (H <= 256) {
            sorted(std::integral_constant<uint32_t, 4>{}, H);
        } else {
            // (2) bitonic sort of the ids in LDS, padded to a power of two
            uint32_t P2 = 1;
            while (P2 < H) P2 <<= 1;
            for (uint32_t t = H + lane; t < P2; t += 64) hb[t] = ~0u;
            wave_lds_order();
            for (uint32_t size = 2; size <= P2; size <<= 1) {
                for (uint32_t stride = size >> 1; stride > 0; stride >>= 1) {
                    for (uint32_t t = lane; t < P2 / 2; t += 64) {
                        const uint32_t a = 2 * t - (t & (stride - 1)), b = a + stride;
                        const uint32_t ka = hb[a], kb = hb[b];
                        if ((ka > kb) == ((a & size) == 0)) { hb[a] = kb; hb[b] = ka; }
                    }
                    wave_lds_order();
                }
            }
        }
        wave_lds_order();
        for (uint32_t h0 = 0; h0 < H; h0 += 64)        // (3)
            S.add(P, in, px, py, pz, vx, vy, vz, vn, lane, min(64u, H - h0), h0 + lane < H ? hb[h0 + lane] : 0u, terms,
                  digest != nullptr);
    }

    if (digest) S.hash_sums();
    const float dv[9] = {S.total(0), S.total(1), S.total(2), S.total(3), S.total(4),
                         S.total(5), S.total(6), S.total(7), S.total(8)};
    if (lane != 0) return;
    float ox = px, oy = py, oz = pz, ovx = vx, ovy = vy, ovz = vz;
    finish_ordered(P, S, dv, i, ox, oy, oz, ovx, ovy, ovz, forces, digest);
    out.x[i] = ox; out.y[i] = oy; out.z[i] = oz; out.vx[i] = ovx; out.vy[i] = ovy; out.vz[i] = ovz;
    // the written state's cell and arrival rank, for the next update
    const uint32_t nextc = cell_f32(P, ox, oy, oz);
    if (!in_field(P, ox, oy, oz)) *outside = 1u;
    key[i] = nextc;
    rank[i] = atomicAdd(&count[nextc], 1u);
}

static inline uint32_t blocks_of(uint32_t n, uint32_t b) { return (n + b - 1) / b; }

hipError_t launch_f32_hash(const DevParams& P, StateF32 st, uint32_t* key, uint32_t* rank, uint32_t* count,
                           uint32_t* outside, hipStream_t stream)
{
    if (P.n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_f32_hash, dim3(blocks_of(P.n, kBlock)), dim3(kBlock), 0, stream, P, st, key, rank, count,
                       outside);
    return hipGetLastError();
}

hipError_t launch_f32_grid_sort(const DevParams& P, StateF32 st, const uint32_t* key, const uint32_t* rank,
                                uint32_t* count, uint32_t* start, uint32_t* partials, float4* rec, hipStream_t stream)
{
    if (P.n == 0) return hipSuccess;
    const uint32_t Gs = (uint32_t)(P.sx * P.G), ncell = Gs * Gs * Gs;
    hipError_t e = launch_scan(count, start, ncell + 1, partials, stream);    // clears count for the next state
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_f32_cells, dim3(blocks_of(P.n, kBlock)), dim3(kBlock), 0, stream, P.n, st, key, rank,
                       (const uint32_t*)start, rec);
    return hipGetLastError();
}

hipError_t launch_f32_grid_step(const DevParams& P, StateF32 in, StateF32 out, const float4* rec, uint32_t* key,
                                uint32_t* rank, const uint32_t* start, uint32_t* count, uint32_t* outside,
                                float* forces, uint64_t* digest, hipStream_t stream)
{
    if (P.n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_f32_grid_wave, dim3(P.n), dim3(64), 0, stream, P, in, out, rec, key, rank, start, count,
                       outside, forces, digest);
    return hipGetLastError();
}

}  // namespace boids
