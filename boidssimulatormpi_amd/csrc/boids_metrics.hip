// boids_metrics.hip — flock metrics on the GPU (polarisation, mean
// nearest-neighbour distance, cluster count), for long-run statistical
// comparison of engine modes.  Distances use the periodic metric of the
// reference's analysis tools (tools/calc_distance.pyx:6-14: per axis
// min(|dx|, F - |dx|)).
//
// Input: n positions / velocities in id order (double, AoS x,y,z).  A private
// uniform grid (edge >= eps, >= 3 cells per axis when possible, about one
// boid per cell at most) is built with the engine's scan; the searches run
// over the cell-ordered copy, four lanes per boid (k_m_near), so a wave's 16
// boids sit in neighbouring cells and read the same candidates.
#include "boids_internal.h"

#include <math.h>

namespace boids {

struct MGrid {
    int G;                    // cells per axis (>= 1)
    double F, edge, inv_edge;
    uint32_t n;
};

__device__ __forceinline__ uint32_t m_axis(double x, const MGrid& g)
{
    double c = floor(x * g.inv_edge);
    if (!(c >= 0.0)) c = 0.0;
    if (c > (double)(g.G - 1)) c = (double)(g.G - 1);
    return (uint32_t)c;
}

__device__ __forceinline__ double m_dist2(const double* a, double bx, double by, double bz, double F)
{
    double s = 0.0;
    const double b[3] = {bx, by, bz};
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        double d = fabs(a[k] - b[k]);
        if (F - d < d) d = F - d;
        s += d * d;
    }
    return s;
}

__global__ __launch_bounds__(kBlock) void k_m_hash(MGrid g, const double* pos3, uint32_t* key, uint32_t* rank,
                                                   uint32_t* count)
{
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= g.n) return;
    const double* p = pos3 + 3 * (size_t)i;
    const uint32_t G = (uint32_t)g.G;
    const uint32_t c = m_axis(p[0], g) + G * (m_axis(p[1], g) + G * m_axis(p[2], g));
    key[i] = c;
    rank[i] = atomicAdd(&count[c], 1u);
}

// Cell-ordered copy of the positions (slot = cell start + arrival rank; the
// searches do not depend on the order inside a cell), and every boid its own
// component of size 0.
__global__ __launch_bounds__(kBlock) void k_m_order(MGrid g, const double* pos3, const uint32_t* key,
                                                    const uint32_t* rank, const uint32_t* start, double4* cpos,
                                                    uint32_t* parent, uint32_t* size)
{
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= g.n) return;
    const double* p = pos3 + 3 * (size_t)i;
    cpos[start[key[i]] + rank[i]] = make_double4(p[0], p[1], p[2], __longlong_as_double((long long)i));   // w: the id bits
    parent[i] = i;
    size[i] = 0u;
}

__device__ __forceinline__ uint32_t m_id(const double4& q) { return (uint32_t)__double_as_longlong(q.w); }

__global__ __launch_bounds__(kBlock) void k_m_fill(uint32_t* a, uint32_t n, uint32_t v)
{
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) a[i] = v;
}

__device__ __forceinline__ uint32_t m_find(uint32_t* parent, uint32_t x)
{
    while (true) {
        const uint32_t p = parent[x];
        if (p == x) return x;
        const uint32_t gp = parent[p];
        if (gp != p) parent[x] = gp;                              // path halving: pointers only move rootward
        x = p;
    }
}

__device__ __forceinline__ void m_union(uint32_t* parent, uint32_t a, uint32_t b)
{
    while (true) {
        a = m_find(parent, a);
        b = m_find(parent, b);
        if (a == b) return;
        if (a > b) { const uint32_t t = a; a = b; b = t; }
        const uint32_t old = atomicCAS(&parent[b], b, a);         // hook the larger root under the smaller
        if (old == b) return;
        b = old;
    }
}

// Nearest-neighbour distance of every boid and the links closer than eps
// (edge >= eps, so ring 1 holds them).  Nearest neighbours by growing rings:
// after ring r every point farther than r*edge from the boid's cell has been
// excluded, so the search stops once the best distance is <= r*edge; at about
// a boid per cell few searches go beyond ring 1.
//
// kNearLanes lanes share a boid, each searching its part of the 9 rows of ring
// 1 (away from the field's x faces a row's three cells are one run of slots):
// the searches are chains of dependent loads, and one lane per boid left two
// waves per SIMD at 131072 boids.  A lane collects its links and makes the
// unions after its rows.  Measured at 131072 boids in 64 blobs, eps 0.02: one
// lane per boid in id order with eight cells per boid 1735 us + 198 us (links);
// one lane in cell order, a boid per cell, 318 us + 350 us; this form 124 us
// (about 70 us of it the searches, bound by the latency of the cell starts and
// records, the rest the unions' dependent chains and atomics).
constexpr uint32_t kNearLanes = 4;
constexpr uint32_t kNearLinks = 6;            // links a lane collects; more are made at once
__global__ __launch_bounds__(kBlock) void k_m_near(MGrid g, const uint32_t* __restrict__ start,
                                                   const double4* __restrict__ cpos, double eps2, uint32_t* parent,
                                                   double* nn)
{
    __shared__ uint32_t links[kNearLinks][kBlock];
    const uint32_t tid = threadIdx.x, sub = tid & (kNearLanes - 1);
    const uint32_t s = blockIdx.x * (kBlock / kNearLanes) + tid / kNearLanes;
    if (s >= g.n) return;                                         // all lanes of a boid together
    const double4 me = cpos[s];
    const double p[3] = {me.x, me.y, me.z};
    const uint32_t i = m_id(me);
    const int G = g.G;
    const int cx = (int)m_axis(me.x, g), cy = (int)m_axis(me.y, g), cz = (int)m_axis(me.z, g);
    double best = INFINITY;
    uint32_t nl = 0;
    auto test = [&](const double4& q) {
        const double d = m_dist2(p, q.x, q.y, q.z, g.F);
        const uint32_t j = m_id(q);
        if (j != i && d < best) best = d;
        if (j > i && d < eps2) {
            if (nl < kNearLinks) links[nl++][tid] = j;
            else m_union(parent, i, j);
        }
    };
    if (G >= 3) {
        constexpr int kRows = (9 + kNearLanes - 1) / kNearLanes;
        uint32_t lo[kRows], hi[kRows], row[kRows];
        const bool inner = cx >= 1 && cx <= G - 2;
#pragma unroll
        for (int k = 0; k < kRows; ++k) {
            const int q = (int)sub + (int)kNearLanes * k;
            lo[k] = hi[k] = row[k] = 0;
            if (q < 9) {
                int y = cy + q % 3 - 1, z = cz + q / 3 - 1;
                y += y < 0 ? G : (y >= G ? -G : 0);
                z += z < 0 ? G : (z >= G ? -G : 0);
                row[k] = (uint32_t)G * ((uint32_t)y + (uint32_t)G * (uint32_t)z);
                lo[k] = start[row[k] + (uint32_t)(inner ? cx - 1 : 0)];
                hi[k] = start[row[k] + (uint32_t)(inner ? cx + 2 : G)];
            }
        }
#pragma unroll
        for (int k = 0; k < kRows; ++k) {
            if (inner || G == 3) {
                for (uint32_t t = lo[k]; t < hi[k]; ++t) test(cpos[t]);
            } else if ((int)sub + (int)kNearLanes * k < 9) {      // at an x face: cells 0, 1, G-1 or 0, G-2, G-1
                const int c0 = cx == 0 ? 0 : G - 2;
                for (uint32_t t = start[row[k] + (uint32_t)c0]; t < start[row[k] + (uint32_t)c0 + 2]; ++t) test(cpos[t]);
                const int c1 = cx == 0 ? G - 1 : 0;
                for (uint32_t t = start[row[k] + (uint32_t)c1]; t < start[row[k] + (uint32_t)c1 + 1]; ++t) test(cpos[t]);
            }
        }
    } else {                                                      // one or two cells per axis: all of them
        const uint32_t cells = (uint32_t)(G * G * G);
        for (uint32_t t = start[0] + sub; t < start[cells]; t += kNearLanes) test(cpos[t]);
    }
    for (uint32_t k = 0; k < nl; ++k) m_union(parent, i, links[k][tid]);
    // rings 1 (just searched), 2, ...: the lanes share a ring's rows
    const int rmax = (G + 1) / 2;
    for (int r = 1;; ++r) {
#pragma unroll
        for (uint32_t d = 1; d < kNearLanes; d <<= 1) best = fmin(best, __shfl_xor(best, d, 64));
        const double reach = r * g.edge;
        if (2 * r + 1 >= G || r >= rmax || best <= reach * reach) break;   // every cell visited, or near enough
        const int o = r + 1, span = 2 * o + 1;
        const bool all = span >= G;                               // the rest of the field: search it all
        const int lo = all ? 0 : -o, len = all ? G : span;
        for (int q = (int)sub; q < len * len; q += (int)kNearLanes) {
            const int dy = lo + q % len, dz = lo + q / len;
            int y = cy + dy, z = cz + dz;
            y += y < 0 ? G : (y >= G ? -G : 0);
            z += z < 0 ? G : (z >= G ? -G : 0);
            const uint32_t rw = (uint32_t)G * ((uint32_t)y + (uint32_t)G * (uint32_t)z);
            auto run = [&](int x0, int x1) {                      // cells x0..x1 of the row, unwrapped, x1 - x0 < G
                for (int part = 0; part < 2; ++part) {
                    int a, z1;
                    wrapped_run(x0, x1, G, part, &a, &z1);
                    if (a > z1) continue;
                    const uint32_t e = start[rw + (uint32_t)z1 + 1];
                    for (uint32_t t = start[rw + (uint32_t)a]; t < e; ++t) {
                        const double4 c = cpos[t];
                        const double d = m_dist2(p, c.x, c.y, c.z, g.F);
                        if (m_id(c) != i && d < best) best = d;
                    }
                }
            };
            if (all) run(0, G - 1);
            else if (max(abs(dy), abs(dz)) == o) run(cx - o, cx + o);
            else { run(cx - o, cx - o); run(cx + o, cx + o); }
        }
    }
    if (sub == 0) nn[i] = sqrt(best);
}

// Component sizes (one atomic per distinct root of a wave: neighbouring slots
// mostly share theirs) and, per block of ids, the sums of the unit velocities
// and the nearest-neighbour distances.
__global__ __launch_bounds__(kBlock) void k_m_sizes(uint32_t n, uint32_t* parent, uint32_t* size,
                                                    const double4* __restrict__ cpos, const double* __restrict__ vel3,
                                                    const double* __restrict__ nn, double4* sums)
{
    __shared__ double sh[4][kBlock / 64];
    const uint32_t t = blockIdx.x * kBlock + threadIdx.x;
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    double v[4] = {0, 0, 0, 0};
    bool left = false;
    uint32_t root = 0;
    if (t < n) {
        root = m_find(parent, m_id(cpos[t]));
        left = true;
        const double* u = vel3 + 3 * (size_t)t;
        const double m = sqrt(u[0] * u[0] + u[1] * u[1] + u[2] * u[2]);
        if (m > 0) { v[0] = u[0] / m; v[1] = u[1] / m; v[2] = u[2] / m; }
        v[3] = nn[t];
    }
    for (;;) {                                                    // ends: every turn serves the first lane left
        const uint64_t todo = __builtin_amdgcn_ballot_w64(left);
        if (todo == 0) break;
        const uint32_t first = (uint32_t)__builtin_ctzll(todo);
        const uint32_t r = (uint32_t)__builtin_amdgcn_readlane((int)root, (int)first);
        const uint64_t same = __builtin_amdgcn_ballot_w64(left && root == r);
        if (lane == first) atomicAdd(&size[r], (uint32_t)__popcll(same));
        if (root == r) left = false;
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) v[k] += __shfl_down(v[k], d, 64);
        if (lane == 0) sh[k][wave] = v[k];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double4 b = make_double4(0, 0, 0, 0);
        for (int w = 0; w < kBlock / 64; ++w) { b.x += sh[0][w]; b.y += sh[1][w]; b.z += sh[2][w]; b.w += sh[3][w]; }
        sums[blockIdx.x] = b;
    }
}

// Per block of ids: the roots of components with at least min_size members
// and the largest size (atomics on two words took 37 us at 131072 boids).
__global__ __launch_bounds__(kBlock) void k_m_roots(uint32_t n, const uint32_t* __restrict__ parent,
                                                    const uint32_t* __restrict__ size, uint32_t min_size,
                                                    uint2* tally)
{
    __shared__ uint32_t sh[2][kBlock / 64];
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    const uint32_t sz = i < n && parent[i] == i ? size[i] : 0u;
    const uint64_t in = __builtin_amdgcn_ballot_w64(sz >= min_size && sz > 0);
    uint32_t top = sz;
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) top = max(top, (uint32_t)__shfl_down((int)top, d, 64));
    if ((threadIdx.x & 63u) == 0) { sh[0][threadIdx.x >> 6] = (uint32_t)__popcll(in); sh[1][threadIdx.x >> 6] = top; }
    __syncthreads();
    if (threadIdx.x != 0) return;
    uint32_t c = 0, m = 0;
    for (int w = 0; w < kBlock / 64; ++w) { c += sh[0][w]; m = max(m, sh[1][w]); }
    tally[blockIdx.x] = make_uint2(c, m);
}

// One workgroup: the blocks' sums and tallies into the results, in a fixed
// order (deterministic).
__global__ __launch_bounds__(kBlock) void k_m_results(uint32_t n, uint32_t blocks, const double4* __restrict__ sums,
                                                      const uint2* __restrict__ tally, double* out4)
{
    __shared__ double4 sh[kBlock];
    __shared__ uint2 st[kBlock];
    double4 a = make_double4(0, 0, 0, 0);
    uint2 r = make_uint2(0, 0);
    for (uint32_t b = threadIdx.x; b < blocks; b += kBlock) {
        const double4 q = sums[b];
        const uint2 t = tally[b];
        a.x += q.x; a.y += q.y; a.z += q.z; a.w += q.w;
        r.x += t.x;
        r.y = max(r.y, t.y);
    }
    sh[threadIdx.x] = a;
    st[threadIdx.x] = r;
    __syncthreads();
    for (int w = kBlock / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) {
            const double4 q = sh[threadIdx.x + w];
            const uint2 t = st[threadIdx.x + w];
            sh[threadIdx.x].x += q.x; sh[threadIdx.x].y += q.y; sh[threadIdx.x].z += q.z; sh[threadIdx.x].w += q.w;
            st[threadIdx.x].x += t.x;
            st[threadIdx.x].y = max(st[threadIdx.x].y, t.y);
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const double4 q = sh[0];
        out4[0] = sqrt(q.x * q.x + q.y * q.y + q.z * q.z) / (double)n;
        out4[1] = n > 1 ? q.w / (double)n : INFINITY;
        out4[2] = (double)st[0].x;
        out4[3] = (double)st[0].y;
    }
}

static inline uint32_t mblocks(uint32_t n) { return (n + kBlock - 1) / kBlock; }

// Workspace layout: one function carves the regions, both for sizing
// (base == nullptr) and for the launch, so the two cannot disagree.
struct MetricsWs {
    double4* cpos;      // n    cell-ordered positions (id bits in w)
    double* nn;         // n
    double4* sums;      // blocks of n
    uint32_t *key, *rank, *parent, *size;   // n each
    uint2* tally;       // blocks of n
    uint32_t *count, *start;                // cells each
    uint32_t* partials; // scan tiles
    double* out;        // 4
    size_t bytes;       // total, from the (unaligned) base
};

static_assert(sizeof(double4) == 32, "double4 is 32 bytes");

static MetricsWs metrics_layout(char* base, uint32_t n, int G)
{
    const size_t cells = (size_t)G * G * G + 1;
    const size_t ntiles = (cells + 4095) / 4096;
    MetricsWs m;
    uintptr_t p = ((uintptr_t)base + 255) & ~(uintptr_t)255;
    auto take = [&](size_t bytes) {
        const uintptr_t at = p;
        p = (p + bytes + 255) & ~(uintptr_t)255;
        return at;
    };
    m.cpos = (double4*)take(sizeof(double4) * (size_t)n);
    m.nn = (double*)take(sizeof(double) * (size_t)n);
    m.sums = (double4*)take(sizeof(double4) * (size_t)mblocks(n));
    m.key = (uint32_t*)take(4 * (size_t)n);
    m.rank = (uint32_t*)take(4 * (size_t)n);
    m.parent = (uint32_t*)take(4 * (size_t)n);
    m.size = (uint32_t*)take(4 * (size_t)n);
    m.tally = (uint2*)take(sizeof(uint2) * (size_t)mblocks(n));
    m.count = (uint32_t*)take(4 * cells);
    m.start = (uint32_t*)take(4 * cells);
    m.partials = (uint32_t*)take(4 * ntiles);
    m.out = (double*)take(sizeof(double) * 4);
    m.bytes = (size_t)(p - (uintptr_t)base);
    return m;
}

size_t metrics_workspace_bytes(uint32_t n, int G)
{
    return metrics_layout(nullptr, n, G).bytes + 256;   // + worst-case alignment of a real base
}

size_t metrics_priced_bytes(uint32_t n, int G)
{
    const size_t cells = (size_t)G * G * G + 1, tiles = (cells + 4095) / 4096;
    auto region = [](size_t bytes) { return (bytes + 255) & ~(size_t)255; };
    return region(32 * (size_t)n) + region(8 * (size_t)n) + 6 * region(4 * (size_t)n) + 2 * region(4 * cells) +
           region(4 * tiles) + region(32) + 256;
}

hipError_t launch_metrics(uint32_t n, double F, int G, double eps, uint32_t min_size, const double* pos3,
                          const double* vel3, void* ws, size_t ws_bytes, double** out4_dev, hipStream_t stream)
{
    const MetricsWs m = metrics_layout((char*)ws, n, G);
    if ((char*)(m.out + 4) > (char*)ws + ws_bytes) return hipErrorInvalidValue;   // layout must fit
    *out4_dev = m.out;
    if (n == 0) return hipSuccess;
    MGrid g;
    g.G = G; g.F = F; g.edge = F / G; g.inv_edge = G / F; g.n = n;
    const uint32_t cells = (uint32_t)((size_t)G * G * G + 1);
    const dim3 grid(mblocks(n)), block(kBlock);
    hipLaunchKernelGGL(k_m_fill, dim3(mblocks(cells)), block, 0, stream, m.count, cells, 0u);
    hipLaunchKernelGGL(k_m_hash, grid, block, 0, stream, g, pos3, m.key, m.rank, m.count);
    hipError_t st = launch_scan(m.count, m.start, cells, m.partials, stream);
    if (st != hipSuccess) return st;
    hipLaunchKernelGGL(k_m_order, grid, block, 0, stream, g, pos3, (const uint32_t*)m.key, (const uint32_t*)m.rank,
                       (const uint32_t*)m.start, m.cpos, m.parent, m.size);
    constexpr uint32_t kBoids = kBlock / kNearLanes;               // per workgroup
    hipLaunchKernelGGL(k_m_near, dim3((n + kBoids - 1) / kBoids), block, 0, stream, g, (const uint32_t*)m.start,
                       (const double4*)m.cpos, eps * eps, m.parent, m.nn);
    hipLaunchKernelGGL(k_m_sizes, grid, block, 0, stream, n, m.parent, m.size, (const double4*)m.cpos, vel3,
                       (const double*)m.nn, m.sums);
    hipLaunchKernelGGL(k_m_roots, grid, block, 0, stream, n, (const uint32_t*)m.parent, (const uint32_t*)m.size,
                       min_size, m.tally);
    hipLaunchKernelGGL(k_m_results, dim3(1), block, 0, stream, n, mblocks(n), (const double4*)m.sums,
                       (const uint2*)m.tally, m.out);
    return hipGetLastError();
}

}  // namespace boids
