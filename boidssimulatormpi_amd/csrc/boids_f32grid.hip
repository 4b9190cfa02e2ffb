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

// The three rule decisions of src/boid.cpp:27-42 for owner p (velocity v,
// |v| = vn) and candidate position t (raw, before the minimum image), with
// the exact float thresholds (s < s_thr <=> sqrtf(s) < r; c >= c_thr &&
// c <= 1 <=> acosf(c) <= pi a).  q receives the shifted candidate position.
struct PairF32 {
    float qx, qy, qz, ex, ey, ez, s;
    bool in_c, in_s, in_a;
};

__device__ __forceinline__ PairF32 decide_f32(const DevParams& P, float px, float py, float pz, float vx, float vy,
                                              float vz, float vn, float tx, float ty, float tz)
{
    PairF32 r;
    r.qx = min_image(tx, px, P.F, P.half);
    r.qy = min_image(ty, py, P.F, P.half);
    r.qz = min_image(tz, pz, P.F, P.half);
    r.ex = px - r.qx; r.ey = py - r.qy; r.ez = pz - r.qz;
    r.s = r.ex * r.ex + r.ey * r.ey + r.ez * r.ez;
    r.in_c = r.s < P.s_thr_f[COH];
    r.in_s = r.s < P.s_thr_f[SEP];
    r.in_a = r.s < P.s_thr_f[ALI];
    if ((r.in_c && P.cone[COH]) || (r.in_s && P.cone[SEP]) || (r.in_a && P.cone[ALI])) {
        const float gx = r.qx - px, gy = r.qy - py, gz = r.qz - pz;
        const float dot = vx * gx + vy * gy + vz * gz;
        const float c = dot / (vn * sqrtf(r.s));
        if (P.cone[COH]) r.in_c = r.in_c && c >= P.c_thr_f[COH] && c <= 1.0f;
        if (P.cone[SEP]) r.in_s = r.in_s && c >= P.c_thr_f[SEP] && c <= 1.0f;
        if (P.cone[ALI]) r.in_a = r.in_a && c >= P.c_thr_f[ALI] && c <= 1.0f;
    }
    return r;
}

__device__ __forceinline__ uint32_t cell_f32(const DevParams& P, float x, float y, float z)
{
    const uint32_t G = (uint32_t)P.G;
    return axis_cell((double)x, P.inv_edge, P.G) +
           G * (axis_cell((double)y, P.inv_edge, P.G) + G * axis_cell((double)z, P.inv_edge, P.G));
}

// Cell key of every boid (id order) and its arrival rank in the cell, for a
// state from outside (k_f32_grid_wave leaves them for the state it writes).
__global__ __launch_bounds__(kBlock) void k_f32_hash(DevParams P, StateF32 st, uint32_t* key, uint32_t* rank,
                                                     uint32_t* count)
{
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= P.n) return;
    const uint32_t c = cell_f32(P, st.x[i], st.y[i], st.z[i]);
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

// Orders this wave's LDS writes before its later LDS reads (a wave's LDS
// operations execute in order; this keeps the compiler from moving them).
__device__ __forceinline__ void wave_lds_order()
{
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

template <typename T>
__device__ __forceinline__ T lane_of(T v, uint32_t l)
{
    return __builtin_bit_cast(T, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), (int)l));
}

// v of lane l ^ S, without LDS: cross-lane operand modifiers for 1, 2, 4 and 8
// (4 = 7 ^ 3), row and half swaps for 16 and 32.
template <uint32_t S>
__device__ __forceinline__ uint32_t xor_lane(uint32_t v, uint32_t lane)
{
    auto dpp = [](uint32_t x, auto ctrl) {
        return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, decltype(ctrl)::value, 0xF, 0xF, true);
    };
    if constexpr (S == 1) return dpp(v, std::integral_constant<int, 0xB1>{});          // quad_perm [1,0,3,2]
    else if constexpr (S == 2) return dpp(v, std::integral_constant<int, 0x4E>{});     // quad_perm [2,3,0,1]
    else if constexpr (S == 4)
        return dpp(dpp(v, std::integral_constant<int, 0x141>{}), std::integral_constant<int, 0x1B>{});
    else if constexpr (S == 8) return dpp(v, std::integral_constant<int, 0x128>{});    // row_ror 8
    else if constexpr (S == 16) {
        const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
        return (lane & 16u) ? r[0] : r[1];
    } else {
        const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
        return (lane & 32u) ? r[0] : r[1];
    }
}

// Bitonic sort, ascending, of 64 R keys: element 64 r + lane in k[r].  Steps
// across lanes take their partner by xor_lane (the same network through LDS
// permutes waited ~100 cycles a step), steps across registers are local.
template <uint32_t R, uint32_t SIZE, uint32_t S>
__device__ __forceinline__ void sort_step(uint32_t (&k)[R], uint32_t lane)
{
#pragma unroll
    for (uint32_t r = 0; r < R; ++r) {
        if constexpr (S >= 64) {
            constexpr uint32_t D = S / 64;
            if (r & D) continue;                                   // handled with its partner
            const bool asc = ((64 * r) & SIZE) == 0;
            const uint32_t lo = min(k[r], k[r + D]), hi = max(k[r], k[r + D]);
            k[r] = asc ? lo : hi;
            k[r + D] = asc ? hi : lo;
        } else {
            const uint32_t p = xor_lane<S>(k[r], lane);
            const bool asc = SIZE >= 64 ? ((64 * r) & SIZE) == 0 : (lane & SIZE) == 0;
            k[r] = ((lane & S) == 0) == asc ? min(k[r], p) : max(k[r], p);
        }
    }
    if constexpr (S > 1) sort_step<R, SIZE, S / 2>(k, lane);
    else if constexpr (SIZE < 64 * R) sort_step<R, SIZE * 2, SIZE>(k, lane);
}

// 64-bit sum over the wave (butterfly), in every lane.
__device__ __forceinline__ uint64_t wave_sum_u64(uint64_t v)
{
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t lo = (uint32_t)__shfl_xor((int)(uint32_t)v, d, 64);
        const uint32_t hi = (uint32_t)__shfl_xor((int)(uint32_t)(v >> 32), d, 64);
        v += ((uint64_t)hi << 32) | lo;
    }
    return v;
}

// One one-wave workgroup per owner (id order).  (1) The lanes test the
// candidates of the 27 cells, 64 at a time over the cells' runs of slots (the
// three cells of a row are one run, two at the field's x faces), against the
// largest radius and append the ids of those within it to an LDS list.  (2) The
// list is sorted (sort_step in registers up to 256 ids, a bitonic network in
// LDS beyond).  (3) For 64 sorted boids at a time the lanes read their states
// by id, take the rule decisions and write the pairs' nine float terms to an
// LDS table, 0 where a rule does not hold; lane c < 9 then adds column c of the
// table in ascending id, so each float sum adds the reference's terms in the
// reference's order (a running sum that starts at +0 is never -0, so adding +0
// leaves it unchanged bit for bit).  The table's columns are kTermStride words
// apart, so the nine lanes' 16-byte reads take different banks.
//
// What bounds it: the waves' own instruction and latency chains (16384 owners
// are 16 waves per SIMD in all).  N = 16384, one update of the whole engine:
// WAVE_FIGURES
constexpr uint32_t kF32HitCap = 1024;        // boids per owner sorted in LDS
constexpr uint32_t kTermStride = 68;
__global__ __launch_bounds__(64) void k_f32_grid_wave(DevParams P, StateF32 in, StateF32 out,
                                                      const float4* __restrict__ rec, uint32_t* key, uint32_t* rank,
                                                      const uint32_t* __restrict__ start, uint32_t* count,
                                                      float* forces, uint64_t* digest)
{
    __shared__ uint32_t hb[kF32HitCap];
    __shared__ uint2 wrapped[9];
    __shared__ __align__(16) float terms[9][kTermStride];   // term c of the block's pair l: terms[c][l]
    const uint32_t lane = threadIdx.x;
    const uint32_t i = blockIdx.x;                     // the grid has one workgroup per boid
    const float px = in.x[i], py = in.y[i], pz = in.z[i];
    const float vx = in.vx[i], vy = in.vy[i], vz = in.vz[i];
    const float vn = norm3(vx, vy, vz);
    const int G = P.G;
    const uint32_t c = key[i];
    const int cx = (int)(c % (uint32_t)G), cy = (int)((c / (uint32_t)G) % (uint32_t)G),
              cz = (int)(c / ((uint32_t)G * (uint32_t)G));

    // Lane r < 9: row r's run of the cells cx-1 .. cx+1, or at a face the part
    // of it that does not wrap; lane 9 + r: the wrapped cell at a face (empty
    // elsewhere).  Then the exclusive prefix of the run lengths.
    const bool face = cx == 0 || cx == G - 1;
    uint32_t ra = 0, rn = 0;
    if (lane < (face ? 18u : 9u)) {
        const int r = lane < 9 ? (int)lane : (int)lane - 9;
        int y = cy + r % 3 - 1, z = cz + r / 3 - 1;
        y += y < 0 ? G : (y >= G ? -G : 0);
        z += z < 0 ? G : (z >= G ? -G : 0);
        const uint32_t row = (uint32_t)G * ((uint32_t)y + (uint32_t)G * (uint32_t)z);
        const int x0 = lane < 9 ? max(cx - 1, 0) : (cx == 0 ? G - 1 : 0);
        const int x1 = lane < 9 ? min(cx + 1, G - 1) : x0;
        ra = start[row + (uint32_t)x0];
        rn = start[row + (uint32_t)x1 + 1] - ra;
    }
    uint32_t incl = rn;
#pragma unroll
    for (uint32_t d = 1; d < 32; d <<= 1) {
        const uint32_t t = __shfl_up(incl, d, 64);
        if (lane >= d) incl += t;
    }
    const uint32_t M = (uint32_t)__builtin_amdgcn_readlane((int)incl, 17);
    // candidate m lies in the last run k with first[k] <= m, at slot m + base[k]:
    // both held in scalar registers (the wrapped runs' in LDS), the base as its
    // step from run to run
    const uint32_t excl = incl - rn, base = ra - excl;
    const uint32_t base0 = (uint32_t)__builtin_amdgcn_readlane((int)base, 0);
    const uint32_t step = base - __shfl_up(base, 1, 64);
    uint32_t first[9], up[9];
#pragma unroll
    for (int k = 1; k < 9; ++k) {
        first[k] = (uint32_t)__builtin_amdgcn_readlane((int)excl, k);
        up[k] = (uint32_t)__builtin_amdgcn_readlane((int)step, k);
    }
    if (lane >= 9 && lane < 18) wrapped[lane - 9] = make_uint2(excl, step);
    wave_lds_order();

    // (1) the boids within the largest radius whose ids lie in [lo, lo + width):
    // appended to the list as far as it holds them, their number returned.
    // Each batch's records are fetched while the previous batch is tested.
    auto record_of = [&](uint32_t m0) {
        const uint32_t m = min(m0 + lane, M - 1);
        uint32_t slot = m + base0;
#pragma unroll
        for (int k = 1; k < 9; ++k) slot += m >= first[k] ? up[k] : 0u;
        if (face) {
            for (int k = 0; k < 9; ++k) slot += m >= wrapped[k].x ? wrapped[k].y : 0u;
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
            const float ex = px - min_image(q.x, px, P.F, P.half);
            const float ey = py - min_image(q.y, py, P.F, P.half);
            const float ez = pz - min_image(q.z, pz, P.F, P.half);
            const bool hit = (m0 + lane < M) & (j != i) & (j - lo < width) & (ex * ex + ey * ey + ez * ez < P.s_max_f);
            const uint64_t mask = __builtin_amdgcn_ballot_w64(hit);
            const uint32_t pos = H + __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                                               __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
            if (hit && pos < kF32HitCap) hb[pos] = j;
            H += (uint32_t)__popcll(mask);
        }
        return H;
    };

    // (3), one block: the terms of the sorted boids h0 .. h0 + 63 of H (lane
    // l holds the id of boid h0 + l in j); lane c < 9 sums column c
    float sum = 0.f;
    int nc = 0, ns = 0, na = 0;
    uint64_t hc = 0, hs = 0, ha = 0;                    // this lane's pairs' id hashes
    auto block = [&](uint32_t h0, uint32_t H, uint32_t j) __attribute__((always_inline)) {
        float t[9] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        bool fc = false, fs = false, fa = false;
        if (h0 + lane < H) {
            const PairF32 r = decide_f32(P, px, py, pz, vx, vy, vz, vn, in.x[j], in.y[j], in.z[j]);
            fc = r.in_c; fs = r.in_s; fa = r.in_a;
            if (fc) { t[0] = r.qx; t[1] = r.qy; t[2] = r.qz; }
            if (fs) {
                const float d = sqrtf(r.s);
                t[3] = r.ex / d; t[4] = r.ey / d; t[5] = r.ez / d;
            }
            if (fa) { t[6] = in.vx[j]; t[7] = in.vy[j]; t[8] = in.vz[j]; }
            if (digest) {
                const uint64_t hh = mix64(j);
                hc += fc ? hh : 0; hs += fs ? hh : 0; ha += fa ? hh : 0;
            }
        }
        nc += __popcll(__builtin_amdgcn_ballot_w64(fc));
        ns += __popcll(__builtin_amdgcn_ballot_w64(fs));
        na += __popcll(__builtin_amdgcn_ballot_w64(fa));
#pragma unroll
        for (int k = 0; k < 9; ++k) terms[k][lane] = t[k];
        wave_lds_order();
        if (lane < 9) {
            const float4* col = (const float4*)terms[lane];
            const uint32_t cnt = (min(64u, H - h0) + 15) / 16;      // the terms beyond H are 0
            for (uint32_t l = 0; l < cnt; ++l) {                    // ascending id: the reference's order
                const float4 a = col[4 * l], b = col[4 * l + 1], d = col[4 * l + 2], e = col[4 * l + 3];
                sum += a.x; sum += a.y; sum += a.z; sum += a.w;
                sum += b.x; sum += b.y; sum += b.z; sum += b.w;
                sum += d.x; sum += d.y; sum += d.z; sum += d.w;
                sum += e.x; sum += e.y; sum += e.z; sum += e.w;
            }
        }
        wave_lds_order();
    };
    auto sorted = [&](auto regs, uint32_t H) __attribute__((always_inline)) {
        constexpr uint32_t R = decltype(regs)::value;
        uint32_t k[R];
#pragma unroll
        for (uint32_t r = 0; r < R; ++r) k[r] = 64 * r + lane < H ? hb[64 * r + lane] : ~0u;
        sort_step<R, 2, 1>(k, lane);
#pragma unroll
        for (uint32_t r = 0; r < R; ++r) hb[64 * r + lane] = k[r];
    };

    // Windows of ascending ids: all of them at once unless more are in reach
    // than the list holds; then narrower ones (one id never overflows it).
    for (uint32_t lo = 0, width = P.n; lo < P.n;) {
        const uint32_t H = collect(lo, width);
        if (H > kF32HitCap) {
            const uint32_t w = (uint32_t)((uint64_t)width * (kF32HitCap * 3 / 4) / H);
            width = max(1u, min(w, width / 2));
            continue;
        }
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
        for (uint32_t h0 = 0; h0 < H; h0 += 64) block(h0, H, h0 + lane < H ? hb[h0 + lane] : 0u);
        lo += min(width, P.n - lo);
    }

    float scx = lane_of(sum, 0), scy = lane_of(sum, 1), scz = lane_of(sum, 2);
    const float ssx = lane_of(sum, 3), ssy = lane_of(sum, 4), ssz = lane_of(sum, 5);
    float sax = lane_of(sum, 6), say = lane_of(sum, 7), saz = lane_of(sum, 8);
    if (digest) { hc = wave_sum_u64(hc); hs = wave_sum_u64(hs); ha = wave_sum_u64(ha); }
    if (lane != 0) return;
    float ox = px, oy = py, oz = pz, ovx = vx, ovy = vy, ovz = vz;
    if (nc != 0) { const float k = (float)nc; scx = scx / k - px; scy = scy / k - py; scz = scz / k - pz; }
    if (na != 0) { const float k = (float)na; sax = sax / k - vx; say = say / k - vy; saz = saz / k - vz; }
    const float wc = P.w_f[COH], ws = P.w_f[SEP], wa = P.w_f[ALI];
    const float dx = (scx * wc + ssx * ws) + sax * wa;
    const float dy = (scy * wc + ssy * ws) + say * wa;
    const float dz = (scz * wc + ssz * ws) + saz * wa;
    if (forces) {
        float* f = forces + 9 * (size_t)i;
        f[0] = scx; f[1] = scy; f[2] = scz; f[3] = ssx; f[4] = ssy; f[5] = ssz; f[6] = sax; f[7] = say; f[8] = saz;
    }
    if (digest) {
        uint64_t* d = digest + 4 * (size_t)i;
        d[0] = (uint64_t)nc | ((uint64_t)ns << 21) | ((uint64_t)na << 42);
        d[1] = hc; d[2] = hs; d[3] = ha;
    }
    integrate<float>(P, ox, oy, oz, ovx, ovy, ovz, dx, dy, dz);
    out.x[i] = ox; out.y[i] = oy; out.z[i] = oz; out.vx[i] = ovx; out.vy[i] = ovy; out.vz[i] = ovz;
    // the written state's cell and arrival rank, for the next update
    const uint32_t nextc = cell_f32(P, ox, oy, oz);
    key[i] = nextc;
    rank[i] = atomicAdd(&count[nextc], 1u);
}

static inline uint32_t blocks_of(uint32_t n, uint32_t b) { return (n + b - 1) / b; }

hipError_t launch_f32_hash(const DevParams& P, StateF32 st, uint32_t* key, uint32_t* rank, uint32_t* count,
                           hipStream_t stream)
{
    if (P.n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_f32_hash, dim3(blocks_of(P.n, kBlock)), dim3(kBlock), 0, stream, P, st, key, rank, count);
    return hipGetLastError();
}

hipError_t launch_f32_grid_sort(const DevParams& P, StateF32 st, const uint32_t* key, const uint32_t* rank,
                                uint32_t* count, uint32_t* start, uint32_t* partials, float4* rec, hipStream_t stream)
{
    if (P.n == 0) return hipSuccess;
    const uint32_t ncell = (uint32_t)P.G * (uint32_t)P.G * (uint32_t)P.G;
    hipError_t e = launch_scan(count, start, ncell + 1, partials, stream);    // clears count for the next state
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_f32_cells, dim3(blocks_of(P.n, kBlock)), dim3(kBlock), 0, stream, P.n, st, key, rank,
                       (const uint32_t*)start, rec);
    return hipGetLastError();
}

hipError_t launch_f32_grid_step(const DevParams& P, StateF32 in, StateF32 out, const float4* rec, uint32_t* key,
                                uint32_t* rank, const uint32_t* start, uint32_t* count, float* forces,
                                uint64_t* digest, hipStream_t stream)
{
    if (P.n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_f32_grid_wave, dim3(P.n), dim3(64), 0, stream, P, in, out, rec, key, rank, start, count,
                       forces, digest);
    return hipGetLastError();
}

}  // namespace boids
