// gpv_kernels.hip -- gfx950 kernels of the two-level hybrid voxelizer.
//
// Stage map (reference function -> kernels here):
//   index AABB, src/Object.cpp:2272-2318 ........... k_tri_setup
//   Level1 SAT sweep + bins, src/Object.cpp:2256-2342,
//     cuda/CUDAClassifyTessellation.cu:320-401 ...... k_sat_expand
//   Level1 ray parity, src/Object.cpp:716-779 ....... k_ray_expand, k_l1_fill
//   compaction + prefix, src/Object.cpp:3270-3279 ... k_pack_bytes, scan, k_ts_count (boundary_index)
//   bins by boundary voxel (the CSR of :2137-2219) .. k_ts_count, k_ts_scan, k_ts_bucket, k_ts_place
//   Level2 SAT, src/Object.cpp:2344-2424 ............ k_l2_sat
//   Level2 ray parity, src/Object.cpp:1111-1207 ..... k_ts_* (column entries), k_l2_parity
//   counts, src/Object.cpp:3353-3378 ................ k_count_states
//   .raw layout, src/Object.cpp:2934-3075 ........... k_export_*
//
// All launches are 64-wide-wave shaped.  No float atomics: occupancy is set
// with integer OR / ballot only, so results are deterministic.
#include "gpv_device.hpp"
#include "gpv_internal.hpp"
#include "gpv_parcol.hpp"
#include "gpv_satrow.hpp"

namespace gpv {

// ---------------------------------------------------------------------------
// small helpers
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint64_t shfl64(uint64_t v, int src)
{
    const uint32_t lo = __shfl((unsigned)(v & 0xffffffffu), src);
    const uint32_t hi = __shfl((unsigned)(v >> 32), src);
    return ((uint64_t)hi << 32) | lo;
}

// Moves across lanes without LDS (DPP and the row swaps): a cross-lane read
// through LDS waits about a hundred cycles, and the scans and the transpose
// below are chains of six.
template <int kCtrl, int kRows, int kBanks>
__device__ __forceinline__ uint32_t dpp(uint32_t v, uint32_t old)
{
    return (uint32_t)__builtin_amdgcn_update_dpp((int)old, (int)v, kCtrl, kRows, kBanks, false);
}
template <int kCtrl, int kRows>
__device__ __forceinline__ uint32_t dpp_or_0(uint32_t v)
{
    return dpp<kCtrl, kRows, 0xf>(v, 0u);
}
template <int kCtrl, int kRows>
__device__ __forceinline__ uint64_t dpp_or_0(uint64_t v)
{
    return (uint64_t)dpp_or_0<kCtrl, kRows>((uint32_t)v) |
           ((uint64_t)dpp_or_0<kCtrl, kRows>((uint32_t)(v >> 32)) << 32);
}

// inclusive sum over the lanes of a full wave
template <typename T>
__device__ __forceinline__ T wave_incl_scan(T x)
{
    x += dpp_or_0<0x111, 0xf>(x);   // row_shr:1, 2, 4, 8: within rows of 16
    x += dpp_or_0<0x112, 0xf>(x);
    x += dpp_or_0<0x114, 0xf>(x);
    x += dpp_or_0<0x118, 0xf>(x);
    x += dpp_or_0<0x142, 0xa>(x);   // row_bcast:15 into rows 1 and 3
    x += dpp_or_0<0x143, 0xc>(x);   // row_bcast:31 into rows 2 and 3
    return x;
}

// inclusive XOR over the lanes of a full wave
__device__ __forceinline__ uint64_t wave_incl_xor(uint64_t x)
{
    x ^= dpp_or_0<0x111, 0xf>(x);
    x ^= dpp_or_0<0x112, 0xf>(x);
    x ^= dpp_or_0<0x114, 0xf>(x);
    x ^= dpp_or_0<0x118, 0xf>(x);
    x ^= dpp_or_0<0x142, 0xa>(x);
    x ^= dpp_or_0<0x143, 0xc>(x);
    return x;
}

// the value of lane ^ S
template <int S>
__device__ __forceinline__ uint32_t lane_xor(uint32_t v)
{
    if constexpr (S == 1) return dpp<0xb1, 0xf, 0xf>(v, v);         // quad_perm 1,0,3,2
    else if constexpr (S == 2) return dpp<0x4e, 0xf, 0xf>(v, v);    // quad_perm 2,3,0,1
    else if constexpr (S == 4) {                                    // row_shl:4 / row_shr:4 by banks of four
        const uint32_t up = dpp<0x104, 0xf, 0x5>(v, v);
        return dpp<0x114, 0xf, 0xa>(v, up);
    } else if constexpr (S == 8) return dpp<0x128, 0xf, 0xf>(v, v);  // row_ror:8
    else {
        static_assert(S == 16 || S == 32, "lane distance");
        const auto r = S == 16 ? __builtin_amdgcn_permlane16_swap(v, v, false, false)
                               : __builtin_amdgcn_permlane32_swap(v, v, false, false);
        return (__lane_id() & S) ? r[0] : r[1];
    }
}

__device__ __forceinline__ uint64_t wave_sum_u64(uint64_t x)
{
    const uint64_t s = wave_incl_scan<uint64_t>(x);
    return shfl64(s, 63);
}

// Waits until this wave's atomics have been performed.  Between a block's atomics
// and the one that says it is through this is enough where the last block reads
// with atomic loads; a device-scope fence would write the L2 back in every block
// (torus knot 256/8 850 -> 1030 us).
__device__ __forceinline__ void wait_atomics()
{
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// Block-wide sum folded into *dst with one atomic per block (blockDim <= 1024,
// every thread of the block must call it).  Same-address atomics serialise in
// L2, so kernels reduce per block before touching a shared counter.
__device__ __forceinline__ void block_add_u64(uint64_t x, unsigned long long* dst)
{
    __shared__ uint64_t s_part[16];
    x = wave_sum_u64(x);
    const int wid = threadIdx.x >> 6;
    __syncthreads();
    if (__lane_id() == 0) s_part[wid] = x;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint64_t t = 0;
        for (int i = 0; i < (int)((blockDim.x + 63) >> 6); ++i) t += s_part[i];
        if (t) atomicAdd(dst, (unsigned long long)t);
    }
}

// largest t in [0, n) with off[t] <= x, given off[0] <= x < off[n]
__device__ __forceinline__ int64_t find_segment(const uint64_t* __restrict__ off, int64_t n, uint64_t x)
{
    int64_t lo = 0, hi = n;
    while (hi - lo > 1) {
        const int64_t mid = (lo + hi) >> 1;
        if (off[mid] <= x) lo = mid; else hi = mid;
    }
    return lo;
}

// ---------------------------------------------------------------------------
// multi-mesh lookups.  Every kernel that depends on the grid is a template on
// kM: kM = false is the single-mesh form (grid passed by value, no offsets),
// kM = true finds the mesh of its work item in the batch descriptors.
// ---------------------------------------------------------------------------
template <bool kM>
__device__ __forceinline__ const GridDev& grid_of(const GridDev& g0, const Meshes& M, int m)
{
    if constexpr (kM) return M.grids[m];
    else return g0;
}

// mesh owning batch-wide Level1 word w: largest m with off[m].word0 <= w
__device__ __forceinline__ int mesh_of_word(const MeshOff* __restrict__ off, int nm, uint64_t w)
{
    int lo = 0, hi = nm;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (off[mid].word0 <= w) lo = mid; else hi = mid;
    }
    return lo;
}

__device__ __forceinline__ int uniform_i(int v) { return __builtin_amdgcn_readfirstlane(v); }

// Largest m in [0, nm) with key(off[m]) <= x for a wave-uniform x (given
// key(off[0]) <= x), by the whole wave: 64 meshes per round of independent
// loads, so two rounds of latency up to 4096 meshes instead of log2(nm).
template <typename E, typename K>
__device__ __forceinline__ int wave_mesh_search(const E* __restrict__ off, int nm, uint64_t x, K key)
{
    const int lane = __lane_id();
    int lo = 0, hi = nm;   // key(off[lo]) <= x; the answer lies in [lo, hi)
    while (hi - lo > 1) {
        const int step = (hi - lo + 63) / 64;
        const int idx = lo + lane * step;
        const bool le = idx < hi && (uint64_t)key(off[idx]) <= x;
        const uint64_t m = __ballot(le);
        const int L = 63 - __clzll((long long)m);
        const int nlo = lo + L * step;
        hi = nlo + step < hi ? nlo + step : hi;
        lo = nlo;
    }
    return uniform_i(lo);
}

// ---------------------------------------------------------------------------
// fills (used instead of memset so that the same code can sit in a graph)
// ---------------------------------------------------------------------------
__global__ void k_fill_u32(uint32_t* p, uint32_t v, int64_t n)
{
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        p[i] = v;
}
__global__ void k_fill_u64(uint64_t* p, uint64_t v, int64_t n)
{
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        p[i] = v;
}

static int grid_for(int64_t n, int block, int cap = 65536)
{
    int64_t g = (n + block - 1) / block;
    if (g < 1) g = 1;
    if (g > cap) g = cap;
    return (int)g;
}

// entry i of a mesh's center tables (table_layout's order)
__device__ __forceinline__ void table_entry(const GridDev& g, int64_t i)
{
    float* out = const_cast<float*>(g.c1x) + i;
    const int n[3] = {g.nx, g.ny, g.nz};
    const float mn[3] = {g.bminx, g.bminy, g.bminz}, g1[3] = {g.g1x, g.g1y, g.g1z}, g2[3] = {g.g2x, g.g2y, g.g2z};
    const int n2 = g.n2 > 0 ? g.n2 : 0;
    bool found = false;
#pragma unroll
    for (int w = 0; w < 4; ++w)
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const int64_t size = (int64_t)n[a] * (w < 2 ? 1 : n2);
            if (!found && i < size) {
                *out = center_at(w, (int)i, mn[a], g1[a], g2[a], n2, g.l2cuda != 0);
                found = true;
            }
            i -= size;
        }
}

// Everything a run has to find cleared, and one mesh's center tables, in one launch:
// a small call is bound by its launches (4.7 us of host time each, 12 us for a
// copy of tables made on the host).  Bound by the writes of large grids: 490 MB in 47 us.
__global__ __launch_bounds__(256) void k_clear(ClearList L, GridDev g, int64_t ntab)
{
    const int64_t stride = (int64_t)gridDim.x * blockDim.x, first = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (int64_t i = first; i < ntab; i += stride) table_entry(g, i);
    for (int64_t i = first; i < L.end[kClearMax - 1]; i += stride) {
        int r = 0;
#pragma unroll
        for (int k = 0; k + 1 < kClearMax; ++k) r += i >= L.end[k] ? 1 : 0;
        uint64_t* p = L.p[0];
        int64_t b = 0;
#pragma unroll
        for (int k = 1; k < kClearMax; ++k)
            if (r == k) {
                p = L.p[k];
                b = L.end[k - 1];
            }
        p[i - b] = 0;
    }
}

// a batch's center tables, a row of blocks per mesh (on the host they took 0.3 ms of
// a call on 48 mixed meshes or 128 small ones, with nothing for the GPU to do)
__global__ __launch_bounds__(256) void k_tables(Meshes M)
{
    for (int m = (int)blockIdx.y; m < M.nm; m += (int)gridDim.y) {
        const GridDev& g = M.grids[m];
        const int64_t n = table_floats(g);
        for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
            table_entry(g, i);
    }
}

void launch_clear(ClearList L, const GridDev* tables, hipStream_t s)
{
    for (int k = 1; k < kClearMax; ++k) L.end[k] += L.end[k - 1];   // sizes -> ends
    const int64_t ntab = tables ? table_floats(*tables) : 0;
    const int64_t n = L.end[kClearMax - 1] > ntab ? L.end[kClearMax - 1] : ntab;
    if (n <= 0) return;
    k_clear<<<grid_for(n, 256, 8192), 256, 0, s>>>(L, tables ? *tables : GridDev{}, ntab);
}

void launch_tables(const Meshes& M, hipStream_t s)
{
    k_tables<<<dim3(8, (unsigned)(M.nm < 4096 ? M.nm : 4096)), 256, 0, s>>>(M);
}

void launch_fill_u32(uint32_t* p, uint32_t v, int64_t n, hipStream_t s)
{
    if (n <= 0) return;
    k_fill_u32<<<grid_for(n, 256, 8192), 256, 0, s>>>(p, v, n);
}
void launch_fill_u64(uint64_t* p, uint64_t v, int64_t n, hipStream_t s)
{
    if (n <= 0) return;
    k_fill_u64<<<grid_for(n, 256, 8192), 256, 0, s>>>(p, v, n);
}

// ---------------------------------------------------------------------------
// triangle setup: index AABB (src/Object.cpp:2272-2318) and the conservative
// ray-column range used by the all-triangle parity fill
// ---------------------------------------------------------------------------
__device__ __forceinline__ int vertex_index(float v, float mn, float mx, int n)
{
    const float num = v - mn;
    const float den = mx - mn;
    const float r = num / den;
    float s = r * (float)n;
    // identity on [-1, n+1]; only pins down vertices outside the bbox,
    // where the float->int conversion would otherwise be undefined
    s = fminf(fmaxf(s, -1.0f), (float)n + 1.0f);
    int i = (int)s;
    if (i == n && v == mx) i--;
    return i;
}

// first i in [0, n) with tab[i] >= x (n if none)
__device__ __forceinline__ int lower_index(const float* __restrict__ tab, int n, double x)
{
    int a = 0, b = n;
    while (a < b) {
        const int m = (a + b) >> 1;
        if ((double)tab[m] < x) a = m + 1; else b = m;
    }
    return a;
}

// Bound on the columns whose +z ray the float MT test can accept.  With
// U = 2^-24 and |T| bounded over the grid, the computed u, v differ from the
// exact barycentric coordinates of the ray point (w.r.t. the float edges) by
// at most du, dv (rounding of det, of the u/v numerators and of the two
// products by 1/det).  Accepted columns lie in the triangle grown to
// {a >= -du, b >= -dv, a + b <= 1 + 2U + du + dv}; its xy bbox, widened by
// a factor kSafety on du and dv, is returned.
constexpr double kSafety = 4.0;

__device__ bool ray_column_bounds(const float* tv, const MtTri& m, const GridDev& g, double& xlo,
                                  double& xhi, double& ylo, double& yhi)
{
    const double U = 5.9604644775390625e-08;
    const double ad = fabs((double)m.det);
    const double tmx = fmax(fabs((double)g.bminx - tv[0]), fabs((double)g.bmaxx - tv[0]));
    const double tmy = fmax(fabs((double)g.bminy - tv[1]), fabs((double)g.bmaxy - tv[1]));
    const double e1x = m.e1x, e1y = m.e1y, e2x = m.e2x, e2y = m.e2y;
    const double edet = U * (fabs(e1x * e2y) + fabs(e1y * e2x) + ad);
    const double eun = U * (3.0 * (fabs(e2y) * tmx + fabs(e2x) * tmy) + 2.0 * ad);
    const double evn = U * (3.0 * (fabs(e1y) * tmx + fabs(e1x) * tmy) + 2.0 * ad);
    const double den = ad - edet;
    if (den <= 0.5 * ad) {
        xlo = g.bminx; xhi = g.bmaxx; ylo = g.bminy; yhi = g.bmaxy;
        return true;
    }
    const double du = kSafety * ((eun + edet * (1 + 2 * U)) / den + 3 * U);
    const double dv = kSafety * ((evn + edet * (1 + 2 * U)) / den + 3 * U);
    const double ds = du + dv + kSafety * 2 * U;
    const double ca0 = -du, ca1 = 1 + ds + dv, ca2 = -du;
    const double cb0 = -dv, cb1 = -dv, cb2 = 1 + ds + du;
    const double x0 = tv[0] + ca0 * e1x + cb0 * e2x, x1 = tv[0] + ca1 * e1x + cb1 * e2x,
                 x2 = tv[0] + ca2 * e1x + cb2 * e2x;
    const double y0 = tv[1] + ca0 * e1y + cb0 * e2y, y1 = tv[1] + ca1 * e1y + cb1 * e2y,
                 y2 = tv[1] + ca2 * e1y + cb2 * e2y;
    xlo = fmin(x0, fmin(x1, x2)); xhi = fmax(x0, fmax(x1, x2));
    ylo = fmin(y0, fmin(y1, y2)); yhi = fmax(y0, fmax(y1, y2));
    const double sx = 1e-12 * (fabs(xlo) + fabs(xhi) + 1.0), sy = 1e-12 * (fabs(ylo) + fabs(yhi) + 1.0);
    xlo -= sx; xhi += sx; ylo -= sy; yhi += sy;
    return true;
}

// mesh of every triangle of the concatenated soup
__global__ void k_mesh_ids(const MeshOff* __restrict__ off, int nm, int64_t T, uint32_t* __restrict__ tri_mesh)
{
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < T; t += (int64_t)gridDim.x * blockDim.x) {
        int lo = 0, hi = nm;
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if ((int64_t)off[mid].tri0 <= t) lo = mid; else hi = mid;
        }
        tri_mesh[t] = (uint32_t)lo;
    }
}

void launch_mesh_ids(const MeshOff* off, int nm, int64_t T, uint32_t* tri_mesh, hipStream_t s)
{
    if (T <= 0) return;
    k_mesh_ids<<<grid_for(T, 256, 8192), 256, 0, s>>>(off, nm, T, tri_mesh);
}

// Single-mesh form: grid-stride over all triangles, one block reduction into
// the mesh's test counter.  Multi-mesh form: one triangle per thread; blocks
// inside one mesh (tri_mesh is non-decreasing) reduce into that mesh's
// counter, the few straddling blocks add per lane.

// kPart: 1 the SAT half (index AABB, items, test counts), 3 the ray
// half (column bound, items) as well.
template <bool kM, int kPart>
__global__ __launch_bounds__(256) void k_tri_setup(const float* __restrict__ tris, int64_t T, GridDev g0, Meshes M,
                                                   int4* __restrict__ box0, int4* __restrict__ box1,
                                                   uint32_t* __restrict__ sat_items,
                                                   int4* __restrict__ ray_rng,
                                                   uint32_t* __restrict__ ray_items,
                                                   uint64_t* __restrict__ sat_sums, uint64_t* __restrict__ ray_sums,
                                                   unsigned long long* __restrict__ bad_input)
{
    __shared__ uint64_t s_sum[2][4];
    uint64_t tests = 0;
    const int64_t first = (int64_t)blockIdx.x * blockDim.x;
    for (int64_t tb = first; tb < T; tb += (int64_t)gridDim.x * blockDim.x) {
        const int64_t t = tb + threadIdx.x;
        uint32_t nsat = 0, nray = 0;
        if (t < T) {
            const int mesh = kM ? (int)M.tri_mesh[t] : 0;
            const GridDev& g = grid_of<kM>(g0, M, mesh);
            float tv[9];
#pragma unroll
            for (int c = 0; c < 9; ++c) tv[c] = tris[t * 9 + c];
            MtTri m;
            const bool vis = mt_setup(tv, m);
            // the input domain: finite coordinates within +-2^40, where every
            // intermediate of the SAT and of the split +z ray test is finite
            bool bad = false;
#pragma unroll
            for (int c = 0; c < 9; ++c) bad = bad || !(fabsf(tv[c]) <= 0x1p40f);
            if (bad) atomicOr(bad_input, 1ull);
            int lo[3], dd[3];
            const int n[3] = {g.nx, g.ny, g.nz};
            const float mn[3] = {g.bminx, g.bminy, g.bminz};
            const float mx[3] = {g.bmaxx, g.bmaxy, g.bmaxz};
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                const int i0 = vertex_index(tv[a], mn[a], mx[a], n[a]);
                const int i1 = vertex_index(tv[3 + a], mn[a], mx[a], n[a]);
                const int i2 = vertex_index(tv[6 + a], mn[a], mx[a], n[a]);
                int l = min(i0, min(i1, i2));
                int h = max(i0, max(i1, i2));
                l = max(l, 0);
                h = min(h, n[a] - 1);
                lo[a] = l;
                dd[a] = h >= l ? h - l + 1 : 0;
            }
            box0[t] = make_int4(lo[0], lo[1], lo[2], vis ? 1 : 0);
            box1[t] = make_int4(dd[0], dd[1], dd[2], 0);
            const bool any = dd[0] > 0 && dd[1] > 0 && dd[2] > 0;
            nsat = any ? (uint32_t)(dd[0] * dd[1]) : 0u;
            sat_items[t] = nsat;
            tests += any ? (uint64_t)dd[0] * dd[1] * dd[2] : 0;
            if constexpr ((kPart & 2) != 0) {
                // at least one item, so that runs of k_ray_expand with equal items hold equal
                // work where most triangles have no column (48 mixed meshes 1414 us without)
                uint32_t rit = 1;
                int4 rr = make_int4(0, 0, 0, 0);
                if (vis) {
                    double xlo, xhi, ylo, yhi;
                    ray_column_bounds(tv, m, g, xlo, xhi, ylo, yhi);
                    const int ia = lower_index(g.r1x, g.nx, xlo);
                    int ib = lower_index(g.r1x, g.nx, xhi);
                    while (ib < g.nx && (double)g.r1x[ib] <= xhi) ++ib;
                    const int ja = lower_index(g.r1y, g.ny, ylo);
                    int jb = lower_index(g.r1y, g.ny, yhi);
                    while (jb < g.ny && (double)g.r1y[jb] <= yhi) ++jb;
                    if (ib > ia && jb > ja) {
                        rr = make_int4(ia, ja, ib - ia, jb - ja);
                        rit = (uint32_t)((ib - ia) * (jb - ja));
                    }
                }
                ray_rng[t] = rr;
                ray_items[t] = rit;
                nray = rit;
            }
        }
        // the items of these 256 triangles, for the scan
        const int wid = threadIdx.x >> 6;
        const uint64_t a = wave_sum_u64(nsat), b = kPart == 3 ? wave_sum_u64(nray) : 0;
        if (__lane_id() == 0) {
            s_sum[0][wid] = a;
            s_sum[1][wid] = b;
        }
        __syncthreads();
        if (threadIdx.x < 2 && ((kPart >> threadIdx.x) & 1) != 0) {
            const uint64_t* v = s_sum[threadIdx.x];
            (threadIdx.x ? ray_sums : sat_sums)[tb / 256] = (v[0] + v[1]) + (v[2] + v[3]);
        }
        __syncthreads();
    }
    if constexpr (!kM) {
        block_add_u64(tests, &M.ctr[0].tests_l1);
    } else {
        const int64_t last = (first + (int64_t)blockDim.x < T ? first + (int64_t)blockDim.x : T) - 1;
        const uint32_t ma = M.tri_mesh[first], mb = M.tri_mesh[last];
        if (ma == mb) {
            block_add_u64(tests, &M.ctr[ma].tests_l1);
        } else if (tests) {
            atomicAdd(&M.ctr[M.tri_mesh[first + threadIdx.x]].tests_l1, (unsigned long long)tests);
        }
    }
}

template <int kPart>
static void tri_setup_part(const float* tris, int64_t T, const GridDev& g0, const Meshes& M, int4* box0, int4* box1,
                           uint32_t* sat_items, int4* ray_rng, uint32_t* ray_items, uint64_t* sat_sums,
                           uint64_t* ray_sums, unsigned long long* bad_input, hipStream_t s)
{
    if (M.nm > 1)
        k_tri_setup<true, kPart><<<grid_for(T, 256, 1 << 30), 256, 0, s>>>(tris, T, g0, M, box0, box1, sat_items,
                                                                            ray_rng, ray_items, sat_sums, ray_sums,
                                                                            bad_input);
    else
        k_tri_setup<false, kPart><<<grid_for(T, 256, 1024), 256, 0, s>>>(tris, T, g0, M, box0, box1, sat_items,
                                                                          ray_rng, ray_items, sat_sums, ray_sums,
                                                                          bad_input);
}

void launch_tri_setup(const float* tris, int64_t T, const GridDev& g0, const Meshes& M, int4* box0, int4* box1,
                      uint32_t* sat_items, int4* ray_rng, uint32_t* ray_items, uint64_t* sat_sums, uint64_t* ray_sums,
                      int part, unsigned long long* bad_input, hipStream_t s)
{
    if (T <= 0) return;
    if (part == 1)
        tri_setup_part<1>(tris, T, g0, M, box0, box1, sat_items, ray_rng, ray_items, sat_sums, ray_sums, bad_input, s);
    else
        tri_setup_part<3>(tris, T, g0, M, box0, box1, sat_items, ray_rng, ray_items, sat_sums, ray_sums, bad_input, s);
}

// ---------------------------------------------------------------------------
// exclusive scan (reduce -> scan block sums -> apply), 4096 items per block
// ---------------------------------------------------------------------------
constexpr int SCAN_NT = 1024;
constexpr int SCAN_IPT = 4;
constexpr int SCAN_TILE = SCAN_NT * SCAN_IPT;

// the counters of a run and one total into the page-locked read-back, which saves two
// copies; the host waits for the stream before it looks
__device__ __forceinline__ void publish(uint64_t* to, uint64_t v)
{
    __hip_atomic_store(to, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
__device__ __forceinline__ void publish_counts(const Counters* ctr, uint64_t total, uint64_t* pub)
{
    publish(pub + 0, ctr->pairs);
    publish(pub + 1, ctr->colents);
    publish(pub + 2, ctr->bad_input);
    publish(pub + kHOff / 8, total);
}

template <typename TO>
__device__ TO block_excl_scan(TO x, TO* s_wave, TO* s_total)
{
    const int lane = __lane_id(), wid = threadIdx.x >> 6;
    const TO inc = wave_incl_scan<TO>(x);
    if (lane == 63) s_wave[wid] = inc;
    __syncthreads();
    if (wid == 0) {
        const TO w = lane < SCAN_NT / 64 ? s_wave[lane] : (TO)0;
        const TO wi = wave_incl_scan<TO>(w);
        if (lane < SCAN_NT / 64) s_wave[lane] = wi - w;
        if (lane == SCAN_NT / 64 - 1) *s_total = wi;
    }
    __syncthreads();
    const TO r = s_wave[wid] + inc - x;
    return r;
}

template <typename TI, typename TO>
__global__ __launch_bounds__(SCAN_NT) void k_scan_reduce(const TI* __restrict__ in, int64_t n,
                                                         TO* __restrict__ sums,
                                                         unsigned int* __restrict__ max_out)
{
    __shared__ TO s_wave[SCAN_NT / 64];
    __shared__ TO s_total;
    const int64_t base = (int64_t)blockIdx.x * SCAN_TILE + (int64_t)threadIdx.x * SCAN_IPT;
    TO acc = 0;
    TI mx = 0;
#pragma unroll
    for (int k = 0; k < SCAN_IPT; ++k) {
        if (base + k < n) {
            const TI v = in[base + k];
            acc += (TO)v;
            mx = v > mx ? v : mx;
        }
    }
    (void)block_excl_scan<TO>(acc, s_wave, &s_total);
    if (threadIdx.x == 0) sums[blockIdx.x] = s_total;
    if (max_out) {
        unsigned m = (unsigned)mx;
        for (unsigned d = 32; d >= 1; d >>= 1) {
            const unsigned o = __shfl_xor(m, d);
            m = o > m ? o : m;
        }
        if (__lane_id() == 0 && m) atomicMax(max_out, m);
    }
}

template <typename TI, typename TO>
__global__ __launch_bounds__(SCAN_NT) void k_scan_apply(const TI* __restrict__ in, int64_t n,
                                                        const TO* __restrict__ block_prefix,
                                                        TO* __restrict__ out)
{
    __shared__ TO s_wave[SCAN_NT / 64];
    __shared__ TO s_total;
    const int64_t base = (int64_t)blockIdx.x * SCAN_TILE + (int64_t)threadIdx.x * SCAN_IPT;
    TO v[SCAN_IPT];
    TO acc = 0;
#pragma unroll
    for (int k = 0; k < SCAN_IPT; ++k) {
        v[k] = (base + k < n) ? (TO)in[base + k] : (TO)0;
        acc += v[k];
    }
    TO run = block_excl_scan<TO>(acc, s_wave, &s_total) + block_prefix[blockIdx.x];
#pragma unroll
    for (int k = 0; k < SCAN_IPT; ++k) {
        if (base + k < n) out[base + k] = run;
        run += v[k];
        if (base + k == n - 1) out[n] = run;
    }
}

// One scan of n values whose sums over consecutive groups of SCAN_TILE / per are
// known: a block's prefix is the sum of the sums before it.
template <typename TI, typename TO>
struct ScanJob {
    const TI* in;
    const TO* sums;
    TO* out;
    int64_t n;
    int per;   // sums per tile
};

// pub: where the host reads the run's counters and the total, if it does; the
// counters were final before this launch, the total is the last block's
template <typename TI, typename TO>
__device__ __forceinline__ void scan_apply_direct(const ScanJob<TI, TO>& J, const Counters* ctr, uint64_t* pub)
{
    __shared__ TO s_wave[SCAN_NT / 64];
    __shared__ TO s_total;
    if ((int64_t)blockIdx.x * SCAN_TILE >= J.n) return;
    // this block's prefix: the sum of the sums of the blocks before it
    TO pre = 0;
    for (int k = threadIdx.x; k < (int)blockIdx.x * J.per; k += SCAN_NT) pre += J.sums[k];
    (void)block_excl_scan<TO>(pre, s_wave, &s_total);   // leaves the block-wide sum in s_total
    const TO block_prefix = s_total;
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * SCAN_TILE + (int64_t)threadIdx.x * SCAN_IPT;
    TO v[SCAN_IPT];
    TO acc = 0;
#pragma unroll
    for (int k = 0; k < SCAN_IPT; ++k) {
        v[k] = (base + k < J.n) ? (TO)J.in[base + k] : (TO)0;
        acc += v[k];
    }
    TO run = block_excl_scan<TO>(acc, s_wave, &s_total) + block_prefix;
#pragma unroll
    for (int k = 0; k < SCAN_IPT; ++k) {
        if (base + k < J.n) J.out[base + k] = run;
        run += v[k];
        if (base + k == J.n - 1) {
            J.out[J.n] = run;
            if (pub) publish_counts(ctr, (uint64_t)run, pub);
        }
    }
}

template <typename TI, typename TO>
__global__ __launch_bounds__(SCAN_NT) void k_scan_apply_direct(ScanJob<TI, TO> J, const Counters* ctr, uint64_t* pub)
{
    scan_apply_direct(J, ctr, pub);
}

// two scans of the set-up's items in one launch
__global__ __launch_bounds__(SCAN_NT) void k_scan_items(ScanJob<uint32_t, uint64_t> a, ScanJob<uint32_t, uint64_t> b)
{
    scan_apply_direct(blockIdx.y ? b : a, static_cast<const Counters*>(nullptr), static_cast<uint64_t*>(nullptr));
}

// scan_rec(n) uses sums[nb+1], then (nb > 1) rest[nb+1] and scan_rec(nb)'s own
size_t scan_tmp_elems(int64_t n)
{
    if (n <= 0) return 2;
    const int64_t nb = (n + SCAN_TILE - 1) / SCAN_TILE;
    if (nb == 1) return 2;
    return (size_t)(nb + 1) * 2 + scan_tmp_elems(nb);
}

template <typename TI, typename TO>
static void scan_rec(const TI* in, TO* out, int64_t n, TO* tmp, unsigned int* max_out, hipStream_t s)
{
    if (n <= 0) {
        if constexpr (sizeof(TO) == 8) launch_fill_u64(reinterpret_cast<uint64_t*>(out), 0, 1, s);
        else launch_fill_u32(reinterpret_cast<uint32_t*>(out), 0, 1, s);
        return;
    }
    const int64_t nb = (n + SCAN_TILE - 1) / SCAN_TILE;
    TO* sums = tmp;            // nb + 1
    TO* rest = tmp + nb + 1;
    k_scan_reduce<TI, TO><<<(unsigned)nb, SCAN_NT, 0, s>>>(in, n, sums, max_out);
    if (nb <= SCAN_TILE) {
        k_scan_apply_direct<TI, TO><<<(unsigned)nb, SCAN_NT, 0, s>>>(ScanJob<TI, TO>{in, sums, out, n, 1}, nullptr, nullptr);
        return;
    }
    // scan the block sums in place (exclusive) into rest, then apply
    scan_rec<TO, TO>(sums, rest, nb, rest + nb + 1, nullptr, s);
    k_scan_apply<TI, TO><<<(unsigned)nb, SCAN_NT, 0, s>>>(in, n, rest, out);
}

void launch_scan_u32_u64(const uint32_t* in, uint64_t* out, int64_t n, uint64_t* tmp, hipStream_t s)
{
    scan_rec<uint32_t, uint64_t>(in, out, n, tmp, nullptr, s);
}

void launch_scan_u32_u32(const uint32_t* in, uint32_t* out, int64_t n, uint32_t* tmp,
                         unsigned int* max_out, hipStream_t s)
{
    scan_rec<uint32_t, uint32_t>(in, out, n, tmp, max_out, s);
}

// ---------------------------------------------------------------------------
// item expansion: the flattened (triangle, column) space of the Level1 stages
// ---------------------------------------------------------------------------
// 64-ary search by one wave: largest t in [lo, hi) with off[t] <= x, given
// off[lo] <= x and (hi == n or off[hi] > x).  ~log64 rounds of dependent
// loads instead of log2.
__device__ __forceinline__ int64_t wave_find_segment(const uint64_t* __restrict__ off, int64_t lo, int64_t hi,
                                                     uint64_t x)
{
    const int lane = __lane_id();
    while (hi - lo > 1) {
        const int64_t step = (hi - lo + 63) / 64;
        const int64_t idx = lo + (int64_t)lane * step;
        const bool le = idx < hi && off[idx] <= x;
        const uint64_t m = __ballot(le);
        const int L = 63 - __clzll((long long)m);
        const int64_t nlo = lo + (int64_t)L * step;
        hi = nlo + step < hi ? nlo + step : hi;
        lo = nlo;
    }
    return lo;
}

constexpr int PACK_WORDS = 1024;   // words of a k_pack_bytes block

__global__ void k_publish_counts(const Counters* ctr, const uint32_t* total, uint64_t* pub)
{
    publish_counts(ctr, *total, pub);
}

// triangles up to which the block sums of the set-up serve the scans (a block
// adds up all sums before its own); more take the scan's own reduction
constexpr int64_t kSumsMax = int64_t(1) << 24;

void launch_scan_items(const uint32_t* in, uint64_t* out, const uint64_t* sums, const uint32_t* in2, uint64_t* out2,
                       const uint64_t* sums2, int64_t T, uint64_t* tmp, hipStream_t s)
{
    if (T <= 0 || T > kSumsMax) {
        launch_scan_u32_u64(in, out, T, tmp, s);
        if (in2) launch_scan_u32_u64(in2, out2, T, tmp, s);
        return;
    }
    const ScanJob<uint32_t, uint64_t> a{in, sums, out, T, SCAN_TILE / 256}, b{in2, sums2, out2, T, SCAN_TILE / 256};
    k_scan_items<<<dim3((unsigned)((T + SCAN_TILE - 1) / SCAN_TILE), in2 ? 2u : 1u), SCAN_NT, 0, s>>>(a, b);
}

// word counts -> word prefix, from the sums that launch_pack_bytes left
void launch_scan_words(const uint32_t* in, uint32_t* out, int64_t W, const uint32_t* sums, const Counters* ctr,
                       uint64_t* pub, uint32_t* tmp, hipStream_t s)
{
    if (W <= kSumsMax) {
        k_scan_apply_direct<uint32_t, uint32_t><<<(unsigned)((W + SCAN_TILE - 1) / SCAN_TILE), SCAN_NT, 0, s>>>(
            ScanJob<uint32_t, uint32_t>{in, sums, out, W, SCAN_TILE / PACK_WORDS}, ctr, pub);
        return;
    }
    launch_scan_u32_u32(in, out, W, tmp, nullptr, s);
    if (pub) k_publish_counts<<<1, 1, 0, s>>>(ctr, out + W, pub);
}

// which item range [so, so + P) of the wave's lanes holds item l0 + lane (ranges
// in lane order); lanes past the last item get some lane's
__device__ __forceinline__ int wave_item_owner(uint8_t* win, uint32_t so, uint32_t P, uint32_t l0)
{
    const int lane = __lane_id();
    // every range that meets [l0, l0 + 64) marks its first position there (the
    // one running into the window marks 0; starts are distinct), and an item
    // takes the mark at the highest marked position up to its own
    win[lane] = 0xff;
    __builtin_amdgcn_wave_barrier();
    if (P && so < l0 + 64u && so + P > l0) win[so > l0 ? so - l0 : 0u] = (uint8_t)lane;
    __builtin_amdgcn_wave_barrier();
    const uint32_t wj = win[lane];
    const uint64_t marks = __ballot(wj != 0xffu) & ((2ull << lane) - 1ull);
    const int top = marks ? 63 - __clzll((long long)marks) : 0;
    const int j = __shfl((int)wj, top) & 63;
    __builtin_amdgcn_wave_barrier();
    return j;
}

// Append buffer of a block in LDS.  n is the same in every thread: a block
// counts what its waves append before they write, so that it needs no atomic
// but the one global reservation per flush (those of one counter are taken at
// 3.7 ns each, whoever makes them: 64-lane blocks with buffers of their own
// spent 120 of 290 us on them on the torus knot).
template <uint32_t CAP>
struct BlockAppend {
    uint64_t* key;
    uint32_t* val;
    uint64_t* gbase;
    uint32_t n;
};

template <uint32_t CAP>
__device__ __forceinline__ void block_flush(BlockAppend<CAP>& L, const Append64& G)
{
    if (L.n == 0) return;
    if (threadIdx.x == 0) *L.gbase = atomicAdd(G.count, (unsigned long long)L.n);
    __syncthreads();
    const uint64_t gb = *L.gbase;
    for (uint32_t i = threadIdx.x; i < L.n; i += blockDim.x)
        if (gb + i < G.cap) {
            G.key[gb + i] = L.key[i];
            G.val[gb + i] = L.val[i];
        }
    __syncthreads();
    L.n = 0;
}

// the block appends `all` entries, this wave `total` of them after the first
// `before`, this lane cnt of those after the first `excl`: put(store) hands
// each to store(key, val).  Reached after a barrier that followed the last writes.
template <uint32_t CAP, typename P>
__device__ __forceinline__ void block_put(BlockAppend<CAP>& L, const Append64& G, uint32_t all, uint32_t before,
                                          uint32_t total, uint32_t excl, P&& put)
{
    if (L.n + all > CAP) block_flush(L, G);
    if (all > CAP) {   // straight to global memory
        unsigned long long gb = 0;
        if (__lane_id() == 0 && total) gb = atomicAdd(G.count, (unsigned long long)total);
        uint64_t idx = shfl64(gb, 0) + excl;
        put([&](uint64_t key, uint32_t val) {
            if (idx < G.cap) {
                G.key[idx] = key;
                G.val[idx] = val;
            }
            ++idx;
        });
        return;
    }
    uint32_t idx = L.n + before + excl;
    put([&](uint64_t key, uint32_t val) {
        L.key[idx] = key;
        L.val[idx] = val;
        ++idx;
    });
    L.n += all;
}

// Level1 SAT: one item = (triangle, xy column of its index AABB), one lane per
// item.  The layers that pass are an interval up to rounding (sat_column): a
// lane takes its certain layers as a mask and runs the float SAT on the few it
// cannot decide (7 of 10000 columns of a torus knot, 8 of 100 where triangles
// span a whole grid).  Hits set the voxel's boundary byte and append the
// (voxel, triangle) bin pair -- key = batch-wide bit index, value = triangle;
// the highest one becomes the (column, triangle, zmax) entry used by the
// Level2 parity candidates.
//
// A wave owns a run of items and walks it 64 at a time over a window of 64
// triangles, whose item offsets one load brings in; columns of more than 64
// layers take several rounds.  One barrier a round counts what the block appends.
// What bounds it: VALU issue for a third of the time (760 instructions per 64
// items, half of them the triangle's coefficients, which too few columns would
// share on fine meshes), the latency of the gathers and the barrier for the rest: 117
// VGPRs and 37 KB of LDS a block allow four waves a SIMD, of which 2.4 to 3.1 are there.  Against a block of lanes
// that walked each column's layers with the float SAT inside a plane slab:
// torus knot 256 (2.9 M columns) 150 -> 95 us, torus 512 (1.9 M) 115 -> 65,
// drilled plate 512 (13.6 M, triangles up to the grid's size) 1870 -> 490,
// 48 mixed meshes 1900 -> 1080, 128 small ones 480 -> 350.
constexpr uint32_t kSatBlocks = 1024, kSatRounds = 12;
template <bool kM>
__global__ __launch_bounds__(256) void k_sat_expand(const float* __restrict__ tris, int64_t T,
                                                    const int4* __restrict__ box0,
                                                    const int4* __restrict__ box1,
                                                    const uint64_t* __restrict__ off, GridDev g0, Meshes M,
                                                    uint8_t* __restrict__ bbytes, Append64 pairs,
                                                    Append64 cols)
{
    constexpr uint32_t PB = 2048, CB = 1024;
    __shared__ uint64_t s_pk[PB];
    __shared__ uint64_t s_ck[CB];
    __shared__ uint32_t s_pv[PB];
    __shared__ uint32_t s_cv[CB];
    __shared__ uint64_t s_gb[2];
    __shared__ uint4 s_tot[2][4];
    __shared__ uint8_t s_win[4][64];
    const int lane = __lane_id(), wid = threadIdx.x >> 6;
    const uint64_t total = off[T];
    // The blocks that fit on the chip at once, more (up to all) where each still gets
    // kSatRounds rounds of items: a block costs two atomics and a search (level1
    // 512: 1024 blocks 66 us, 4096 103 us), and uneven columns ask for many (drilled plate
    // 512: 749 us with 1024, 489 us with 4096)
    const uint64_t full = total / (256u * kSatRounds), most = gridDim.x;
    const uint32_t nb = (uint32_t)(full < kSatBlocks ? (most < kSatBlocks ? most : kSatBlocks) : full < most ? full : most) & ~7u;
    if (blockIdx.x >= nb) return;
    const uint64_t per = ((total + 4ull * nb - 1) / (4ull * nb) + 63) / 64 * 64;
    // workgroups are dealt to the 8 XCDs round-robin and each XCD has its own
    // L2: the blocks of one XCD take one contiguous run of ranges (nb is a
    // multiple of 8), so that the bytes of neighbouring voxels mostly stay in one L2
    const uint64_t bb = (uint64_t)((blockIdx.x % 8u) * (nb / 8u) + blockIdx.x / 8u) * 4u * per;
    if (bb >= total) return;
    uint64_t base = bb + (uint64_t)wid * per;
    const uint64_t b1 = base + per < total ? base + per : total;
    BlockAppend<PB> lp{s_pk, s_pv, &s_gb[0], 0};
    BlockAppend<CB> lc{s_ck, s_cv, &s_gb[1], 0};
    int64_t t0 = base < b1 ? wave_find_segment(off, 0, T, base) : 0;
    bool pending = false;   // layers left of the items at hand (uniform)
    float tv[9] = {};
    int p = 0, q = 0, z0 = 0, zmax = -1, zb = 0;
    uint32_t t = 0;
    bool vis = false;
    SatColumn sc{0, 0, 0, 0};
    for (uint32_t round = 0;; round ^= 1u) {
        if (!pending && base < b1) {
            uint64_t so, eo;
            uint32_t n;
            for (;;) {
                const int64_t tl = t0 + lane < T ? t0 + lane : T;
                so = off[tl];
                eo = off[tl + 1 < T ? tl + 1 : T];
                const uint64_t wend = shfl64(eo, 63);
                const uint64_t left = (wend < b1 ? wend : b1) - base;
                n = left < 64 ? (uint32_t)left : 64u;
                if (n) break;
                t0 = wave_find_segment(off, t0 + 64, T, base);   // 64 triangles without items
            }
            const uint64_t from = so > base ? so : base;
            const uint32_t P = eo > from ? (uint32_t)(eo - from < 64 ? eo - from : 64) : 0u;
            const uint32_t rel = from - base < 64 ? (uint32_t)(from - base) : 64u;
            const int j = wave_item_owner(s_win[wid], rel, P, 0);
            const uint32_t l = (uint32_t)base + (uint32_t)lane - (uint32_t)__shfl((int)(uint32_t)so, j);
            t = (uint32_t)(t0 + j);
            // the triangles that end here are done
            t0 += __popcll(__ballot(eo <= base + n));
            base += n;
            zb = 0;
            zmax = -1;
            sc = SatColumn{0, 0, 0, 0};
            if ((uint32_t)lane < n) {
                const GridDev& g = grid_of<kM>(g0, M, kM ? (int)M.tri_mesh[t] : 0);
                const int4 q0 = box0[t];
                const int4 q1 = box1[t];
#pragma unroll
                for (int c = 0; c < 9; ++c) tv[c] = tris[(uint64_t)t * 9 + c];
                const uint32_t jq = l / (uint32_t)q1.x;
                const int xi = (int)(l - jq * (uint32_t)q1.x), yi = (int)jq;
                p = q0.x + xi;
                q = q0.y + yi;
                z0 = q0.z;
                vis = q0.w != 0;
                const SatScale s1{g.s1x, g.s1y, g.s1z, g.d1x, g.d1y, g.d1z};
                sc = sat_column(tv, g.c1x[q0.x], g.c1y[q0.y], g.c1z[q0.z], s1, xi, yi, q1.z);
                zb = sc.am;
            }
        }
        const int mesh = kM ? (int)M.tri_mesh[t] : 0;
        const GridDev& g = grid_of<kM>(g0, M, mesh);
        uint64_t hit = 0;
        if (zb < sc.bm) {
            const int m = sc.bm - zb, ia = sc.ai - zb, ib = sc.bi - zb;
            uint64_t und = m < 64 ? (1ull << m) - 1ull : ~0ull;
            hit = ib <= 0 ? 0ull : ib < 64 ? (1ull << ib) - 1ull : ~0ull;
            hit &= ia <= 0 ? ~0ull : ia < 64 ? ~0ull << ia : 0ull;
            und &= ~hit;
            while (und) {
                const int z = __ffsll((unsigned long long)und) - 1;
                und &= und - 1ull;
                if (tri_box_overlap<true, true>(g.c1x[p], g.c1y[q], g.c1z[z0 + zb + z], g.h1x, g.h1y, g.h1z, tv))
                    hit |= 1ull << z;
            }
            if (hit) zmax = z0 + zb + 63 - __clzll((long long)hit);
        }
        const int zf = z0 + zb;   // the layer of bit 0
        zb += 64;
        pending = __any(zb < sc.bm);
        const bool emit = !pending && zmax >= 0 && vis && g.n2 > 0;   // only the Level2 parity reads them
        // what the block's waves append this round
        const uint32_t cnt = (uint32_t)__popcll(hit);
        const uint32_t incl = wave_incl_scan<uint32_t>(cnt);
        const uint64_t em = __ballot(emit);
        if (lane == 63) s_tot[round][wid] = make_uint4(incl, (uint32_t)__popcll(em), pending || base < b1 ? 1u : 0u, 0u);
        __syncthreads();
        uint32_t pall = 0, call = 0, pbef = 0, cbef = 0, more = 0;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const uint4 v = s_tot[round][w];
            pbef += w < wid ? v.x : 0u;
            cbef += w < wid ? v.y : 0u;
            pall += v.x;
            call += v.y;
            more |= v.z;
        }
        block_put(lp, pairs, pall, pbef, (uint32_t)__builtin_amdgcn_readlane((int)incl, 63), incl - cnt, [&](auto&& store) {
            if (!hit) return;
            const uint64_t plane = (uint64_t)g.ny * g.nxw;
            const uint64_t bit0 =
                ((kM ? M.off[mesh].word0 : 0) + (uint64_t)zf * plane + (uint64_t)q * g.nxw) * 64 + (uint64_t)p;
            for (uint64_t h = hit; h; h &= h - 1ull) {
                const uint64_t bit = bit0 + (uint64_t)(__ffsll((unsigned long long)h) - 1) * plane * 64;
                bbytes[bit] = 1;   // every writer stores the same byte value
                store(bit, t);
            }
        });
        block_put(lc, cols, call, cbef, (uint32_t)__popcll(em), (uint32_t)__popcll(em & lanes_below_mask()),
                  [&](auto&& store) {
                      const uint32_t col0 = kM ? M.off[mesh].col0 : 0;
                      if (emit)
                          store(((uint64_t)(col0 + (uint32_t)q * g.nx + p) << 32) | (uint64_t)t, (uint32_t)zmax);
                  });
        if (emit) zmax = -1;
        if (!more) break;
    }
    __syncthreads();
    block_flush(lp, pairs);
    block_flush(lc, cols);
}

void launch_sat_expand(const float* tris, int64_t T, const int4* box0, const int4* box1, const uint64_t* off,
                       const GridDev& g0, const Meshes& M, uint8_t* b, Append64 pairs, Append64 cols, int blocks,
                       hipStream_t s)
{
    if (T <= 0) return;
    // a wave to eight triangles, but 2048 (a box of 12 can hold 10^6 columns): empty blocks cost their launch
    const int64_t want = T / 32 > 512 ? T / 32 : 512;
    const unsigned nb = (unsigned)(((want < blocks ? want : blocks) + 7) / 8 * 8);
    if (M.nm > 1)
        k_sat_expand<true><<<nb, 256, 0, s>>>(tris, T, box0, box1, off, g0, M, b, pairs, cols);
    else
        k_sat_expand<false><<<nb, 256, 0, s>>>(tris, T, box0, box1, off, g0, M, b, pairs, cols);
}

// boundary flags (one byte per padded voxel, 0 or 1, written without atomics by
// the Level1 SAT) -> the boundary bitplane, its popcount per word and per block of
// PACK_WORDS.  Bound by the flags' read: a lane takes 16 of them in one load and
// stores their 16 bits, four lanes make a word.  One flag per lane and a ballot, and the
// popcounts in a pass of their own, took 66 + 5 us on 62 MB of flags (torus 512)
// and 299 + 11 on 490 MB; now 12 and 62.
__global__ __launch_bounds__(1024) void k_pack_bytes(const uint4* __restrict__ by, int64_t W, uint16_t* __restrict__ bits,
                                                     uint32_t* __restrict__ cnt, uint32_t* __restrict__ sums)
{
    __shared__ uint32_t s_sum[16];
    constexpr int U = PACK_WORDS * 4 / 1024;
    const int64_t n = W * 4, i0 = (int64_t)blockIdx.x * (PACK_WORDS * 4) + threadIdx.x;
    uint4 v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = i0 + u * 1024 < n ? by[i0 + u * 1024] : make_uint4(0, 0, 0, 0);
    uint32_t all = 0;
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int64_t i = i0 + u * 1024;
        // bits 0, 8, 16, 24 of a flag word -> its top four
        const uint32_t b = ((v[u].x * 0x10204080u) >> 28) | (((v[u].y * 0x10204080u) >> 28) << 4) |
                           (((v[u].z * 0x10204080u) >> 28) << 8) | (((v[u].w * 0x10204080u) >> 28) << 12);
        uint32_t c = (uint32_t)__popc(b);
        all += c;
        c += lane_xor<1>(c);
        c += lane_xor<2>(c);
        if (i < n) {
            bits[i] = (uint16_t)b;
            if ((i & 3) == 0) cnt[i >> 2] = c;
        }
    }
    all = wave_incl_scan<uint32_t>(all);
    if (__lane_id() == 63) s_sum[threadIdx.x >> 6] = all;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t t = 0;
        for (int k = 0; k < 16; ++k) t += s_sum[k];
        sums[blockIdx.x] = t;
    }
}

size_t pack_sums(int64_t W) { return (size_t)((W + PACK_WORDS - 1) / PACK_WORDS); }

void launch_pack_bytes(const uint8_t* by, int64_t W, uint64_t* bits, uint32_t* cnt, uint32_t* sums, hipStream_t s)
{
    if (W <= 0) return;
    k_pack_bytes<<<(unsigned)pack_sums(W), 1024, 0, s>>>(reinterpret_cast<const uint4*>(by), W,
                                                         reinterpret_cast<uint16_t*>(bits), cnt, sums);
}

// Level1 ray parity, first half: one item = (triangle, column inside its
// conservative bound), one lane per item.  Where the reference's ray test accepts
// the column (det, u, v), the layers that pass are those below one crossing up to
// rounding (par_l1_layers): a lane XORs one bit into the inside plane at
// the layer under the crossing, and where the bounds leave layers undecided runs the
// float t test on them and XORs a bit at each change.  k_l1_fill makes the parity of
// the toggles above a layer.
//
// A wave owns a run of items and walks it 64 at a time over a window of 64
// triangles; waves share nothing.  The crossings of a flat face fall into the same words:
// lanes next to each other with the same word make one atomic.  What bounds it: the latency of a
// round's dependent loads (offsets, triangle, origins), hence all waves the chip
// holds.  Against blocks that appended a hit list through LDS: torus knot 256
// 36.8 -> 21 us, 48 mixed meshes 471 -> 253, 128 small ones 174 -> 90.
template <bool kM>
__global__ __launch_bounds__(256) void k_ray_expand(const float* __restrict__ tris, int64_t T,
                                                    const int4* __restrict__ rng, const uint64_t* __restrict__ off,
                                                    GridDev g0, Meshes M, unsigned long long* __restrict__ ins)
{
    __shared__ uint8_t s_win[4][64];
    const int lane = __lane_id(), wid = threadIdx.x >> 6;
    const uint64_t total = off[T];
    const uint32_t nb = gridDim.x;   // a multiple of 8
    const uint64_t per = ((total + 4ull * nb - 1) / (4ull * nb) + 63) / 64 * 64;
    // the blocks of one XCD take one contiguous run of ranges
    uint64_t base = ((uint64_t)((blockIdx.x % 8u) * (nb / 8u) + blockIdx.x / 8u) * 4u + (uint64_t)wid) * per;
    if (base >= total) return;
    const uint64_t b1 = base + per < total ? base + per : total;
    int64_t t0 = wave_find_segment(off, 0, T, base);
    while (base < b1) {
        uint64_t so, eo;
        uint32_t n;
        for (;;) {
            const int64_t tl = t0 + lane < T ? t0 + lane : T;
            so = off[tl];
            eo = off[tl + 1 < T ? tl + 1 : T];
            const uint64_t wend = shfl64(eo, 63);
            const uint64_t left = (wend < b1 ? wend : b1) - base;
            n = left < 64 ? (uint32_t)left : 64u;
            if (n) break;
            t0 = wave_find_segment(off, t0 + 64, T, base);   // 64 triangles without items
        }
        const uint64_t from = so > base ? so : base;
        const uint32_t P = eo > from ? (uint32_t)(eo - from < 64 ? eo - from : 64) : 0u;
        const uint32_t rel = from - base < 64 ? (uint32_t)(from - base) : 64u;
        const int o = wave_item_owner(s_win[wid], rel, P, 0);
        const uint32_t l = (uint32_t)base + (uint32_t)lane - (uint32_t)__shfl((int)(uint32_t)so, o);
        const uint32_t t = (uint32_t)(t0 + o);
        // the triangles that end here are done
        t0 += __popcll(__ballot(eo <= base + n));
        base += n;
        uint32_t at = ~0u;   // the word that gets the lane's toggle (planes hold less than 2^26 words)
        uint64_t bit = 0;
        if ((uint32_t)lane < n) {
            const int mesh = kM ? (int)M.tri_mesh[t] : 0;
            const GridDev& g = grid_of<kM>(g0, M, mesh);
            const int4 r = rng[t];
            float tv[9];
#pragma unroll
            for (int c = 0; c < 9; ++c) tv[c] = tris[(uint64_t)t * 9 + c];
            const uint32_t rz = r.z > 0 ? (uint32_t)r.z : 1u, jq = l / rz;
            const int i = r.x + (int)(l - jq * rz), j = r.y + (int)jq;
            MtTri m;
            float tx, ty;
            if (r.z > 0 && mt_setup(tv, m) && mt_column(m, tv[0], tv[1], g.r1x[i], g.r1y[j], tx, ty)) {
                // u and v as mt_column has them
                const float px = 0.0f * m.e2z - m.e2y, py = m.e2x - 0.0f * m.e2z;
                const float u = (tx * px + ty * py) * m.inv_det, v = (tx * m.e1y - ty * m.e1x) * m.inv_det;
                int la, lb;
                par_l1_layers(g.r1z, g.nz, g.bminz, (float)g.nz / (g.bmaxz - g.bminz), tv[2], m.e1z, m.e2z, u, v,
                              par_ez(m.e1x, m.e1y, m.e1z, m.e2x, m.e2y, m.e2z, m.inv_det), la, lb);
                const uint32_t plane = (uint32_t)g.ny * (uint32_t)g.nxw;
                const uint32_t w0 = (uint32_t)(kM ? M.off[mesh].word0 : 0) + (uint32_t)j * (uint32_t)g.nxw + (uint32_t)i / 64u;
                bit = 1ull << (i & 63);
                bool in = la > 0;
                for (int k = la; k < lb; ++k) {
                    const bool hit = mt_t_hit(m.e1x, m.e1y, m.e1z, m.e2x, m.e2y, m.e2z, m.inv_det, tx, ty, tv[2], g.r1z[k]);
                    if (hit != in && k > 0) atomicXor(&ins[w0 + (uint32_t)(k - 1) * plane], (unsigned long long)bit);
                    in = hit;
                }
                if (in) at = w0 + (uint32_t)(lb - 1) * plane;
            }
        }
        // one atomic for each run of lanes with the same word
        const uint64_t x = wave_incl_xor(at != ~0u ? bit : 0ull);
        const uint32_t prev = (uint32_t)__shfl((int)at, lane ? lane - 1 : 0), next = (uint32_t)__shfl((int)at, lane < 63 ? lane + 1 : 63);
        const uint64_t heads = __ballot(lane == 0 || at != prev) & ((2ull << lane) - 1ull);
        const int first = 63 - __clzll((long long)heads);
        const uint64_t before = shfl64(x, first ? first - 1 : 0);
        if (at != ~0u && (lane == 63 || at != next)) atomicXor(&ins[at], (unsigned long long)(x ^ (first ? before : 0ull)));
    }
}

void launch_ray_expand(const float* tris, int64_t T, const int4* ray_rng, const uint64_t* off, const GridDev& g0,
                       const Meshes& M, uint64_t* ins, int blocks, hipStream_t s)
{
    if (T <= 0) return;
    unsigned long long* w = reinterpret_cast<unsigned long long*>(ins);
    // as many blocks as the Level1 SAT's launch: a wave to eight triangles
    const int64_t want = T / 32 > 512 ? T / 32 : 512;
    const int64_t cap = blocks < 2048 ? blocks : 2048;
    const unsigned nb = (unsigned)(((want < cap ? want : cap) + 7) / 8 * 8);
    if (M.nm > 1)
        k_ray_expand<true><<<nb, 256, 0, s>>>(tris, T, ray_rng, off, g0, M, w);
    else
        k_ray_expand<false><<<nb, 256, 0, s>>>(tris, T, ray_rng, off, g0, M, w);
}

// Level1 ray parity, second half: the toggles of a (row word, layer) XORed over the
// layers from the top down, in place.  A block takes L1F_W words of a mesh's layer
// (a cache line) in 64 segments of layers: a pass for each segment's XOR, a second (from
// the cache) to write.  Bound by the plane's read and write; the segments
// keep enough loads in flight where a layer has few words.  Takes the place of the hits'
// count, scan, scatter and a t test per layer and hit: 48 mixed meshes 440 -> 20 us,
// torus 512 95 -> 5.5.
constexpr int L1F_U = 8;
template <bool kM>
__global__ __launch_bounds__(1024) void k_l1_fill(GridDev g0, Meshes M, uint64_t* __restrict__ ins)
{
    __shared__ uint64_t s_x[16][L1F_W];
    const int lane = __lane_id(), wid = uniform_i(threadIdx.x >> 6);
    const int mesh = kM ? wave_mesh_search(M.off, M.nm, (uint64_t)blockIdx.x, [](const MeshOff& o) { return (uint64_t)o.ptask0; }) : 0;
    const GridDev& g = grid_of<kM>(g0, M, mesh);
    if (g.l1st) return;   // the stencil fill writes this mesh's inside bits
    const int64_t plane = (int64_t)g.ny * g.nxw;
    const int64_t w = (int64_t)(blockIdx.x - (kM ? M.off[mesh].ptask0 : 0u)) * L1F_W + (lane & (L1F_W - 1));
    uint64_t* p = ins + (kM ? M.off[mesh].word0 : 0) + w;
    const int len = (g.nz + 63) / 64;
    const int z0 = w < plane ? (wid * 4 + lane / L1F_W) * len : g.nz, z1 = z0 + len < g.nz ? z0 + len : g.nz;
    uint64_t own = 0;
    for (int z = z0; z < z1; z += L1F_U) {
        uint64_t v[L1F_U];
#pragma unroll
        for (int k = 0; k < L1F_U; ++k) v[k] = z + k < z1 ? p[(z + k) * plane] : 0ull;
#pragma unroll
        for (int k = 0; k < L1F_U; ++k) own ^= v[k];
    }
    // the segments from the lane's own up to the wave's last, then the later waves'
    const uint64_t a = shfl64(own, (lane + 16) & 63);
    uint64_t acc = own ^ (lane < 48 ? a : 0ull);
    const uint64_t b = shfl64(acc, (lane + 32) & 63);
    acc ^= lane < 32 ? b : 0ull;
    if (lane < L1F_W) s_x[wid][lane] = acc;
    __syncthreads();
    acc ^= own;
    for (int k = wid + 1; k < 16; ++k) acc ^= s_x[k][lane & (L1F_W - 1)];
    for (int z = z1; z > z0; z -= L1F_U) {
        uint64_t v[L1F_U];
#pragma unroll
        for (int k = 0; k < L1F_U; ++k) v[k] = z - 1 - k >= z0 ? p[(z - 1 - k) * plane] : 0ull;
#pragma unroll
        for (int k = 0; k < L1F_U; ++k) {
            acc ^= v[k];
            if (z - 1 - k >= z0) p[(z - 1 - k) * plane] = acc;
        }
    }
}

void launch_l1_fill(const GridDev& g0, const Meshes& M, int64_t blocks, uint64_t* ins, hipStream_t s)
{
    if (blocks <= 0) return;
    if (M.nm > 1)
        k_l1_fill<true><<<(unsigned)blocks, 1024, 0, s>>>(g0, M, ins);
    else
        k_l1_fill<false><<<(unsigned)blocks, 1024, 0, s>>>(g0, M, ins);
}

// ---------------------------------------------------------------------------
// counting sorts by the high 32 bits of a key
// ---------------------------------------------------------------------------
// column entries -> CSR by column of (triangle, zmax); the Level2 parity, which
// reads each once, makes the triangle's Moller-Trumbore record itself
struct ColItem {
    uint32_t x, t, zmax;
};

struct ColSrc {
    using Item = ColItem;
    const uint64_t* key;
    const uint32_t* zmax;
    __device__ uint32_t sort_key(uint64_t i) const { return (uint32_t)(key[i] >> 32); }
    __device__ uint32_t count_key(uint64_t i) const { return sort_key(i); }
    __device__ void keep_key(uint64_t, uint32_t) const {}
    __device__ ColItem item(uint64_t i) const
    {
        const uint64_t k = key[i];
        return ColItem{(uint32_t)(k >> 32), (uint32_t)(k & 0xffffffffu), zmax[i]};
    }
};

// place(pos, it, ok): stores only when ok
struct ColPlace {
    using Item = ColItem;
    uint2* ent;
    __device__ void operator()(uint32_t pos, const ColItem& it, bool ok) const
    {
        if (ok) ent[pos] = make_uint2(it.t, it.zmax);
    }
};

// ---------------------------------------------------------------------------
// a batch's device soups gathered into the batch's soup in one launch (one
// grid row per mesh, each row's blocks striding over the mesh's floats)
// ---------------------------------------------------------------------------
// kHost: the sources are page-locked host memory, read with system-scope
// loads so that no line a cache kept from an earlier call is returned (the
// caller may have rewritten the buffer since)
template <bool kHost>
__global__ __launch_bounds__(256) void k_gather_soups(const SoupPiece* __restrict__ pc, int m0,
                                                      float* __restrict__ dst)
{
    const SoupPiece p = pc[m0 + blockIdx.y];
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < p.n; i += stride) {
        if constexpr (kHost)
            dst[p.at + i] = __hip_atomic_load(p.src + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        else
            dst[p.at + i] = p.src[i];
    }
}

void launch_gather_soups(const SoupPiece* pc, int nm, float* dst, int blocks, bool host, hipStream_t s)
{
    for (int m0 = 0; m0 < nm; m0 += 65535) {
        const int rows = nm - m0 < 65535 ? nm - m0 : 65535;
        if (host)
            k_gather_soups<true><<<dim3((unsigned)blocks, (unsigned)rows), 256, 0, s>>>(pc, m0, dst);
        else
            k_gather_soups<false><<<dim3((unsigned)blocks, (unsigned)rows), 256, 0, s>>>(pc, m0, dst);
    }
}

// ---------------------------------------------------------------------------
// Level1 inside/outside by the GL-stencil-equivalent fill (opt-in,
// gpv_params::l1_stencil; ClassifyInOut2x, src/Object.cpp:1446-1601).  Per
// slice s the reference draws the mesh orthographically over the bbox into a
// 2nx x 2ny stencil, clipped to z <= zs, counts the fragments per sample,
// and calls a voxel inside when more than 2 of its 4 samples hold an odd
// count.  Which samples a triangle covers is the GL driver's choice; the
// rule here is fixed: vertices snapped to 1/256 sample in window
// coordinates, sample (px, py) at (256 px + 128, 256 py + 128), edge
// functions of the counter-clockwise snapped triangle positive, or zero on a
// top or left edge (shared edges count once), no sample for a zero snapped
// area; a covered sample counts in slice s when the height of the triangle's
// plane (float vertices, double arithmetic) over the sample's world point is
// at most the slice's ray-origin z.  A covered sample toggles bit (s0, py,
// px) of a [nz][2ny][2nx] bit set at its first slice s0; the running XOR
// along s is then the stencil's parity, and the 2 x 2 vote writes the
// Level1 inside bits.  Counts are exact (GL's 8-bit stencil saturates).
// The kernels read only the soup and the grid, so the pipeline runs them
// beside the Level1 SAT.
// ---------------------------------------------------------------------------
struct StTri {
    long long X[3], Y[3];             // snapped window coordinates, counter-clockwise
    int pxlo, pxhi, pylo, pyhi;       // samples whose centers lie in the snapped bbox
    double v0x, v0y, v0z, nx, ny, nz; // first vertex and plane normal
};

__device__ __forceinline__ long long st_snap(float x, float lo, float hi, int samples)
{
    double w = ((double)x - (double)lo) / ((double)hi - (double)lo) * (double)samples;
    // vertices far outside the bbox: bounded so that edge functions stay in 64 bits
    w = w < -4194304.0 ? -4194304.0 : (w > 4194304.0 ? 4194304.0 : w);
    return (long long)rint(w * 256.0);
}

__device__ __forceinline__ long long st_floor256(long long a) { return a >= 0 ? a / 256 : -((255 - a) / 256); }

// false when the triangle covers no sample in any slice
__device__ bool st_prepare(const float* __restrict__ tv, const GridDev& g, StTri& s)
{
    const int W = 2 * g.nx, H = 2 * g.ny;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        s.X[i] = st_snap(tv[3 * i], g.bminx, g.bmaxx, W);
        s.Y[i] = st_snap(tv[3 * i + 1], g.bminy, g.bmaxy, H);
    }
    const long long A = (s.X[1] - s.X[0]) * (s.Y[2] - s.Y[0]) - (s.Y[1] - s.Y[0]) * (s.X[2] - s.X[0]);
    if (A == 0) return false;
    if (A < 0) {
        long long t = s.X[1]; s.X[1] = s.X[2]; s.X[2] = t;
        t = s.Y[1]; s.Y[1] = s.Y[2]; s.Y[2] = t;
    }
    s.v0x = (double)tv[0]; s.v0y = (double)tv[1]; s.v0z = (double)tv[2];
    const double e1x = (double)tv[3] - s.v0x, e1y = (double)tv[4] - s.v0y, e1z = (double)tv[5] - s.v0z;
    const double e2x = (double)tv[6] - s.v0x, e2y = (double)tv[7] - s.v0y, e2z = (double)tv[8] - s.v0z;
    s.nx = e1y * e2z - e1z * e2y;
    s.ny = e1z * e2x - e1x * e2z;
    s.nz = e1x * e2y - e1y * e2x;
    if (s.nz == 0.0) return false;
    long long mnx = s.X[0], mxx = s.X[0], mny = s.Y[0], mxy = s.Y[0];
#pragma unroll
    for (int i = 1; i < 3; ++i) {
        mnx = s.X[i] < mnx ? s.X[i] : mnx;
        mxx = s.X[i] > mxx ? s.X[i] : mxx;
        mny = s.Y[i] < mny ? s.Y[i] : mny;
        mxy = s.Y[i] > mxy ? s.Y[i] : mxy;
    }
    const long long xlo = st_floor256(mnx - 128 + 255), xhi = st_floor256(mxx - 128);
    const long long ylo = st_floor256(mny - 128 + 255), yhi = st_floor256(mxy - 128);
    s.pxlo = (int)(xlo < 0 ? 0 : xlo);
    s.pylo = (int)(ylo < 0 ? 0 : ylo);
    s.pxhi = (int)(xhi > W - 1 ? W - 1 : xhi);
    s.pyhi = (int)(yhi > H - 1 ? H - 1 : yhi);
    return s.pxlo <= s.pxhi && s.pylo <= s.pyhi;
}

__device__ __forceinline__ bool st_covers(const StTri& s, int px, int py)
{
    const long long sx = 256ll * px + 128, sy = 256ll * py + 128;
#pragma unroll
    for (int e = 0; e < 3; ++e) {
        const int a = e, b = e == 2 ? 0 : e + 1;
        const long long dx = s.X[b] - s.X[a], dy = s.Y[b] - s.Y[a];
        const long long E = dx * (sy - s.Y[a]) - dy * (sx - s.X[a]);
        if (E < 0 || (E == 0 && !(dy < 0 || (dy == 0 && dx < 0)))) return false;
    }
    return true;
}

// first slice whose clip plane keeps the triangle's point over the sample
// (z_T <= zs); nz when none does
__device__ __forceinline__ int st_slice(const StTri& s, const GridDev& g, int px, int py)
{
    const double l = (double)g.bminx, r = (double)g.bmaxx, b = (double)g.bminy, t = (double)g.bmaxy;
    const double x = l + ((double)px + 0.5) * ((r - l) / (double)(2 * g.nx));
    const double y = b + ((double)py + 0.5) * ((t - b) / (double)(2 * g.ny));
    const double zt = s.v0z - (s.nx * (x - s.v0x) + s.ny * (y - s.v0y)) / s.nz;
    int lo = 0, hi = g.nz;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if ((double)g.r1z[mid] < zt) lo = mid + 1; else hi = mid;
    }
    return lo;
}

__global__ __launch_bounds__(256) void k_st_count(const float* __restrict__ tris, int64_t T, GridDev g,
                                                  uint32_t* __restrict__ cnt)
{
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < T; t += (int64_t)gridDim.x * blockDim.x) {
        StTri s;
        cnt[t] = st_prepare(tris + 9 * t, g, s)
                     ? (uint32_t)(s.pxhi - s.pxlo + 1) * (uint32_t)(s.pyhi - s.pylo + 1)
                     : 0u;
    }
}

// the (triangle, sample) items, ST_RUN consecutive ones per thread: one
// search for the run's first triangle, then forward
constexpr int ST_RUN = 8;
__global__ __launch_bounds__(256) void k_st_toggle(const float* __restrict__ tris, int64_t T, GridDev g,
                                                   const uint64_t* __restrict__ off, int wpr,
                                                   unsigned long long* __restrict__ tog)
{
    const uint64_t N = off[T];
    const int H = 2 * g.ny;
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x * ST_RUN;
    for (uint64_t i0 = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) * ST_RUN; i0 < N; i0 += stride) {
        const uint64_t i1 = i0 + ST_RUN < N ? i0 + ST_RUN : N;
        int64_t t = find_segment(off, T, i0);
        StTri s;
        st_prepare(tris + 9 * t, g, s);
        int64_t at = -1;   // the word of the last toggles and their bits
        unsigned long long bits = 0;
        for (uint64_t i = i0; i < i1; ++i) {
            if (off[t + 1] <= i) {
                do ++t; while (off[t + 1] <= i);
                st_prepare(tris + 9 * t, g, s);
            }
            const uint32_t li = (uint32_t)(i - off[t]);
            const uint32_t bw = (uint32_t)(s.pxhi - s.pxlo + 1);
            const int py = s.pylo + (int)(li / bw), px = s.pxlo + (int)(li % bw);
            if (!st_covers(s, px, py)) continue;
            const int k = st_slice(s, g, px, py);
            if (k >= g.nz) continue;
            const int64_t w = ((int64_t)k * H + py) * wpr + (px >> 6);
            if (w != at) {
                if (bits) atomicXor(&tog[at], bits);
                at = w;
                bits = 0;
            }
            bits ^= 1ull << (px & 63);
        }
        if (bits) atomicXor(&tog[at], bits);
    }
}

// One wave per Level1 row word (row j, 64 voxels) walks the slices: the
// running XOR of the toggles of sample rows 2j and 2j + 1 is the stencil's
// parity at each slice, and a voxel is inside when more than 2 of its
// samples (2x + {0,1}, 2j + {0,1}) are odd.  The slices' toggle words are
// loaded ST_ZU at a time ahead of their use.
constexpr int ST_ZU = 8;
__global__ __launch_bounds__(256) void k_st_vote(const unsigned long long* __restrict__ tog, GridDev g, int wpr,
                                                 uint64_t* __restrict__ ins)
{
    const int64_t w = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int nxw = g.nxw, ny = g.ny, nx = g.nx, nz = g.nz, H = 2 * g.ny;
    if (w >= (int64_t)ny * nxw) return;
    const int lane = __lane_id();
    const int xw = (int)(w % nxw), j = (int)(w / nxw);
    const int x = xw * 64 + lane;
    const int sx = 2 * x, sh = sx & 63;
    // lanes past the row read a word of the row (their votes are masked)
    const int wi = x < nx ? sx >> 6 : 0;
    const int64_t plane = (int64_t)H * wpr;
    const unsigned long long* r0 = tog + (int64_t)(2 * j) * wpr + wi;
    unsigned long long a = 0, b = 0;
    for (int k0 = 0; k0 < nz; k0 += ST_ZU) {
        unsigned long long ta[ST_ZU], tb[ST_ZU];
#pragma unroll
        for (int u = 0; u < ST_ZU; ++u) {
            const int k = k0 + u < nz ? k0 + u : nz - 1;
            ta[u] = r0[k * plane];
            tb[u] = r0[k * plane + wpr];
        }
#pragma unroll
        for (int u = 0; u < ST_ZU; ++u) {
            if (k0 + u >= nz) break;
            a ^= ta[u];
            b ^= tb[u];
            const int odd = (int)((a >> sh) & 1ull) + (int)((a >> (sh + 1)) & 1ull) + (int)((b >> sh) & 1ull) +
                            (int)((b >> (sh + 1)) & 1ull);
            const uint64_t m = __ballot(x < nx && odd > 2);
            if (lane == 0) ins[((int64_t)(k0 + u) * ny + j) * nxw + xw] = m;
        }
    }
}

size_t l1_stencil_words(const GridDev& g)
{
    return (size_t)g.nz * (size_t)(2 * g.ny) * (size_t)((2 * g.nx + 63) / 64);
}

void launch_l1_stencil(const float* tris, int64_t T, const GridDev& g, uint32_t* cnt, uint64_t* off,
                       uint64_t* scan_tmp, uint64_t* tog, uint64_t* ins, hipStream_t s)
{
    const int wpr = (2 * g.nx + 63) / 64;
    unsigned long long* tg = reinterpret_cast<unsigned long long*>(tog);
    launch_fill_u64(tog, 0, (int64_t)l1_stencil_words(g), s);
    if (T > 0) {
        k_st_count<<<grid_for(T, 256, 16384), 256, 0, s>>>(tris, T, g, cnt);
        launch_scan_u32_u64(cnt, off, T, scan_tmp, s);
        k_st_toggle<<<4096, 256, 0, s>>>(tris, T, g, off, wpr, tg);
    }
    const int64_t rows = (int64_t)g.ny * g.nxw;   // one wave each
    k_st_vote<<<(unsigned)((rows * 64 + 255) / 256), 256, 0, s>>>(tg, g, wpr, ins);
}

// ---------------------------------------------------------------------------
// boundary compaction (src/Object.cpp:3270-3279): popcount per word ->
// exclusive scan -> ascending linear indices of the boundary voxels
// ---------------------------------------------------------------------------
// b0 (first boundary rank), l2w0 (first Level2 word) and l2n0 (first Level2
// normal) of every mesh, from the batch-wide word prefix.
__global__ __launch_bounds__(64) void k_mesh_bounds(const uint32_t* __restrict__ wprefix, Meshes M, const Counters* ctr,
                                                    uint64_t* pub)
{
    // one wave: 64 meshes per round, exclusive scans of the Level2 word and
    // normal counts carried across rounds
    const int lane = __lane_id();
    uint64_t l2 = 0, l2n = 0;
    for (int base = 0; base <= M.nm; base += 64) {
        const int m = base + lane;
        uint32_t b0 = 0;
        uint64_t w = 0, nrm = 0;
        if (m <= M.nm) {
            b0 = wprefix[M.off[m].word0];
            if (m < M.nm) {
                const uint64_t nb = wprefix[M.off[m + 1].word0] - b0;
                const GridDev& g = M.grids[m];
                w = nb * (uint64_t)g.w2;
                nrm = g.normals ? nb * (uint64_t)g.n2 * g.n2 * g.n2 : 0;
            }
        }
        const uint64_t wi = wave_incl_scan<uint64_t>(w), ni = wave_incl_scan<uint64_t>(nrm);
        if (m <= M.nm) {
            const MeshRank o{l2 + wi - w, l2n + ni - nrm, b0, 0u};
            M.rank[m] = o;
            uint64_t q[sizeof(MeshRank) / 8];
            __builtin_memcpy(q, &o, sizeof o);
            for (int k = 0; k < (int)(sizeof(MeshRank) / 8); ++k)
                publish(pub + kHOff / 8 + (size_t)m * (sizeof(MeshRank) / 8) + k, q[k]);
        }
        l2 += shfl64(wi, 63);
        l2n += shfl64(ni, 63);
    }
    if (lane == 0) {
        publish(pub + 0, ctr->pairs);
        publish(pub + 1, ctr->colents);
        publish(pub + 2, ctr->bad_input);
    }
}

void launch_mesh_bounds(const uint32_t* wprefix, const Meshes& M, const Counters* ctr, uint64_t* pub, hipStream_t s)
{
    static_assert(sizeof(MeshRank) % 8 == 0, "published by words");
    k_mesh_bounds<<<1, 64, 0, s>>>(wprefix, M, ctr, pub);
}

// The first Level2 SAT group of every mesh of a batch, from the boundary ranks.  One wave:
// a few us, less than the copy of a table made on the host (128 small meshes 1446 -> 1441 us of
// device time).
__global__ __launch_bounds__(64) void k_mesh_groups(Meshes M, int most)
{
    const int lane = __lane_id();
    uint32_t before = 0;
    for (int base = 0; base <= M.nm; base += 64) {
        const int m = base + lane;
        uint32_t n = 0;
        if (m < M.nm) n = (uint32_t)l2_groups(M.grids[m].n2, (int64_t)M.rank[m + 1].b0 - (int64_t)M.rank[m].b0, most);
        const uint32_t incl = wave_incl_scan<uint32_t>(n);
        if (m <= M.nm) M.rank[m].sg0 = before + incl - n;
        before += (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
    }
}

void launch_mesh_groups(const Meshes& M, int most, hipStream_t s) { k_mesh_groups<<<1, 64, 0, s>>>(M, most); }

// ascending linear indices (within the mesh) of the boundary voxels, in a
// batch the mesh of each, and the columns that hold any; block `blk` of `blocks`
template <bool kM>
__device__ __forceinline__ void boundary_index(const uint64_t* __restrict__ bnd, const uint32_t* __restrict__ wprefix,
                                               const GridDev& g0, const Meshes& M, int64_t W, int32_t* __restrict__ bidx,
                                               unsigned long long* __restrict__ occ, uint32_t blk, uint32_t blocks)
{
    for (int64_t w = (int64_t)blk * blockDim.x + threadIdx.x; w < W; w += (int64_t)blocks * blockDim.x) {
        uint64_t bits = bnd[w];
        if (!bits) continue;
        uint32_t pos = wprefix[w];
        const int mesh = kM ? mesh_of_word(M.off, M.nm, (uint64_t)w) : 0;
        const GridDev& g = grid_of<kM>(g0, M, mesh);
        const int64_t wl = w - (int64_t)(kM ? M.off[mesh].word0 : 0);
        const int xw = (int)(wl % g.nxw);
        const int64_t row = wl / g.nxw;
        if (occ)   // an atomic for every word: looking first whether it adds anything costs 45 us at 512 layers
            atomicOr(occ + (kM ? M.off[mesh].cw0 : 0u) + ((uint32_t)row % (uint32_t)g.ny) * (uint32_t)g.nxw + (uint32_t)xw,
                     (unsigned long long)bits);
        while (bits) {
            const int bit = __ffsll((unsigned long long)bits) - 1;
            bits &= bits - 1;
            if constexpr (kM) M.bmesh[pos] = (uint32_t)mesh;
            bidx[pos++] = (int32_t)(row * g.nx + xw * 64 + bit);
        }
    }
}

__device__ __forceinline__ uint32_t rank_of(const uint64_t* __restrict__ bnd,
                                            const uint32_t* __restrict__ wprefix, uint64_t bitidx)
{
    const uint64_t w = bitidx >> 6;
    const int bit = (int)(bitidx & 63);
    const uint64_t below = bit ? (~0ull >> (64 - bit)) : 0ull;
    return wprefix[w] + (uint32_t)__popcll(bnd[w] & below);
}

// ---------------------------------------------------------------------------
// Counting sort of n items by a key in [0, nkeys) in two levels: tiles of
// 2^shift consecutive keys.  Pass 1 (count) and pass 2 (bucket) walk the same
// contiguous item range per block and histogram the tile ids in LDS, so the
// global counters see one atomic per (block, tile) instead of one per item;
// pass 3 (one block per tile) counts its keys in LDS, writes their CSR
// offsets and places every item at its final position.  The order inside one
// key is unspecified (as with any atomic placement).  Each thread keeps TS_U
// items in flight: their loads are issued together (indices clamped to a
// valid item, the LDS atomics and stores predicated), since the per-item
// chains of dependent loads, not bandwidth, bound these passes.
// ---------------------------------------------------------------------------
constexpr int TS_NT = 256;
constexpr int TS_U = 8;   // a block's 2048 items in one round (torus knot 256/8, three passes: 119 -> 110 us with 4 -> 8)

// A bin pair sorts by the rank of its voxel among the boundary voxels; its item
// is (rank, triangle).
struct PairSrc {
    using Item = uint2;
    // per pair, its voxel's bit in the Level1 grid; the count pass writes the
    // voxel's boundary rank over it (ranked: a repeated compaction, whose
    // pairs hold ranks already), so the bucket pass reads the rank directly
    uint64_t* bits;
    bool ranked;
    const uint32_t* tri;
    const uint64_t* bnd;
    const uint32_t* wprefix;
    __device__ uint32_t count_key(uint64_t i) const
    {
        return ranked ? (uint32_t)bits[i] : rank_of(bnd, wprefix, bits[i]);
    }
    __device__ void keep_key(uint64_t i, uint32_t k) const
    {
        if (!ranked) bits[i] = k;
    }
    __device__ uint32_t sort_key(uint64_t i) const { return (uint32_t)bits[i]; }
    __device__ uint2 item(uint64_t i) const { return make_uint2((uint32_t)bits[i], tri[i]); }
};

struct PairPlace {
    using Item = uint2;
    uint32_t* list;
    __device__ void operator()(uint32_t pos, const uint2& it, bool ok) const
    {
        if (ok) list[pos] = it.y;
    }
};

// One sort of a launch: its scratch (total[ntiles], fill[ntiles], done[1], zeros at the
// start, then off[ntiles + 1]) and the blocks that share its items; none: no sort.
template <typename Src>
struct TsSort {
    Src src;
    uint64_t n;
    uint32_t nkeys;
    int shift, ntiles, blocks;
    uint32_t* cnt;
    typename Src::Item* bucket;
    __device__ uint32_t* total() const { return cnt; }
    __device__ uint32_t* fill() const { return cnt + ntiles; }
    __device__ uint32_t* done() const { return cnt + 2 * ntiles; }
    __device__ uint32_t* off() const { return cnt + 2 * ntiles + 1; }
};

__device__ __forceinline__ void ts_range(uint64_t n, int blocks, uint64_t& lo, uint64_t& hi)
{
    const uint64_t per = (n + blocks - 1) / blocks;
    lo = (uint64_t)blockIdx.x * per;
    hi = lo + per < n ? lo + per : n;
}

// LDS histogram of the tile ids of items [lo, hi) of this block
// kCount: the count pass, which takes each item's key from count_key and
// hands it to keep_key (a source may keep it for the later passes); the
// bucket pass reads sort_key
template <bool kCount, typename Src>
__device__ __forceinline__ void ts_histogram(const Src& src, uint64_t lo, uint64_t hi, int shift, uint32_t* s_h)
{
    for (uint64_t i0 = lo + threadIdx.x; i0 < hi; i0 += (uint64_t)TS_U * TS_NT) {
        uint32_t k[TS_U];
#pragma unroll
        for (int u = 0; u < TS_U; ++u) {
            const uint64_t i = i0 + (uint64_t)u * TS_NT;
            k[u] = kCount ? src.count_key(i < hi ? i : i0) : src.sort_key(i < hi ? i : i0);
        }
#pragma unroll
        for (int u = 0; u < TS_U; ++u) {
            const uint64_t i = i0 + (uint64_t)u * TS_NT;
            if (i < hi) {
                atomicAdd(&s_h[k[u] >> shift], 1u);
                if constexpr (kCount) src.keep_key(i, k[u]);
            }
        }
    }
}

// Tile totals -> tile offsets by one block of NT threads; s_h holds
// ts_scan_words(ntiles) words.  Atomic loads: blocks of the same launch added the totals.
template <int NT>
__device__ __forceinline__ void ts_scan(const uint32_t* __restrict__ total, uint32_t* __restrict__ off, int ntiles,
                                        uint32_t* s_h, uint32_t* s_wave)
{
    constexpr int U = 8;
    const int pad = ts_pad(ntiles);
    auto at = [pad](int t) { return t + (t >> pad); };
    for (int t0 = threadIdx.x; t0 < ntiles; t0 += U * NT) {
        uint32_t v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int t = t0 + u * NT;
            v[u] = __hip_atomic_load(&total[t < ntiles ? t : t0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (t0 + u * NT < ntiles) s_h[at(t0 + u * NT)] = v[u];
    }
    __syncthreads();
    const int C = (ntiles + NT - 1) / NT, c0 = (int)threadIdx.x * C, c1 = c0 + C < ntiles ? c0 + C : ntiles;
    uint32_t sum = 0;
    for (int t = c0; t < c1; ++t) sum += s_h[at(t)];
    const int lane = __lane_id(), wid = threadIdx.x >> 6;
    const uint32_t inc = wave_incl_scan<uint32_t>(sum);
    if (lane == 63) s_wave[wid] = inc;
    __syncthreads();
    uint32_t run = inc - sum;
    for (int w = 0; w < wid; ++w) run += s_wave[w];
    for (int t = c0; t < c1; ++t) {
        const uint32_t v = s_h[at(t)];
        s_h[at(t)] = run;
        run += v;
    }
    if (threadIdx.x == NT - 1) off[ntiles] = run;
    __syncthreads();
    for (int t = threadIdx.x; t < ntiles; t += NT) off[t] = s_h[at(t)];
}

// a block per sort
template <typename A, typename B>
__global__ __launch_bounds__(1024) void k_ts_scan(TsSort<A> a, TsSort<B> b)
{
    extern __shared__ uint32_t s_h[];   // [ts_scan_words(ntiles)]
    __shared__ uint32_t s_wave[16];
    if (blockIdx.x == 0 && a.blocks) ts_scan<1024>(a.total(), a.off(), a.ntiles, s_h, s_wave);
    if (blockIdx.x == 1 && b.blocks) ts_scan<1024>(b.total(), b.off(), b.ntiles, s_h, s_wave);
}

// last: the last block of a sort to get through makes the tiles' offsets, and
// s_h holds ts_scan_words(ntiles)
template <typename Src>
__device__ __forceinline__ void ts_count(const TsSort<Src>& S, bool last, uint32_t* s_h, uint32_t* s_wave, uint32_t* s_last)
{
    if ((int)blockIdx.x >= S.blocks) return;
    for (int t = threadIdx.x; t < S.ntiles; t += TS_NT) s_h[t] = 0;
    __syncthreads();
    uint64_t lo, hi;
    ts_range(S.n, S.blocks, lo, hi);
    ts_histogram<true>(S.src, lo, hi, S.shift, s_h);
    __syncthreads();
    for (int t = threadIdx.x; t < S.ntiles; t += TS_NT)
        if (s_h[t]) atomicAdd(&S.total()[t], s_h[t]);
    if (!last) return;
    wait_atomics();
    __syncthreads();
    if (threadIdx.x == 0) *s_last = atomicAdd(S.done(), 1u) == (uint32_t)S.blocks - 1u ? 1u : 0u;
    __syncthreads();
    if (*s_last) ts_scan<TS_NT>(S.total(), S.off(), S.ntiles, s_h, s_wave);
}

// Row 0 of the grid counts the bin pairs, row 1 the column entries, row 2 makes the
// boundary index list: they depend on the boundary plane and the appends alone, and
// one launch costs what each of three does.
template <bool kM>
__global__ __launch_bounds__(TS_NT) void k_ts_count(TsSort<PairSrc> a, TsSort<ColSrc> b, bool last, GridDev g0, Meshes M,
                                                    const uint64_t* __restrict__ bnd, const uint32_t* __restrict__ wprefix,
                                                    int64_t W, int32_t* __restrict__ bidx,
                                                    unsigned long long* __restrict__ occ)
{
    extern __shared__ uint32_t s_h[];   // [ntiles]
    __shared__ uint32_t s_wave[TS_NT / 64];
    __shared__ uint32_t s_last;
    if (blockIdx.y == 0) ts_count(a, last, s_h, s_wave, &s_last);
    else if (blockIdx.y == 1) ts_count(b, last, s_h, s_wave, &s_last);
    else boundary_index<kM>(bnd, wprefix, g0, M, W, bidx, occ, blockIdx.x, gridDim.x);
}

// items (.x = key) to their tile's bucket range; the item is built
// here, where the block reads its inputs in their original order
template <typename Src>
__device__ __forceinline__ void ts_bucket(const TsSort<Src>& S, uint32_t* s_h)   // counts, then this block's next slot per tile
{
    if ((int)blockIdx.x >= S.blocks) return;
    for (int t = threadIdx.x; t < S.ntiles; t += TS_NT) s_h[t] = 0;
    __syncthreads();
    uint64_t lo, hi;
    ts_range(S.n, S.blocks, lo, hi);
    ts_histogram<false>(S.src, lo, hi, S.shift, s_h);
    __syncthreads();
    const uint32_t* off = S.off();
    uint32_t* fill = S.fill();
    for (int t = threadIdx.x; t < S.ntiles; t += TS_NT)
        if (s_h[t]) s_h[t] = off[t] + atomicAdd(&fill[t], s_h[t]);
    __syncthreads();
    for (uint64_t i0 = lo + threadIdx.x; i0 < hi; i0 += (uint64_t)TS_U * TS_NT) {
        typename Src::Item it[TS_U];
#pragma unroll
        for (int u = 0; u < TS_U; ++u) {
            const uint64_t i = i0 + (uint64_t)u * TS_NT;
            it[u] = S.src.item(i < hi ? i : i0);
        }
#pragma unroll
        for (int u = 0; u < TS_U; ++u)
            if (i0 + (uint64_t)u * TS_NT < hi) S.bucket[atomicAdd(&s_h[it[u].x >> S.shift], 1u)] = it[u];
    }
}

__global__ __launch_bounds__(TS_NT) void k_ts_bucket(TsSort<PairSrc> a, TsSort<ColSrc> b)
{
    extern __shared__ uint32_t s_h[];   // [ntiles]
    if (blockIdx.y == 0) ts_bucket(a, s_h);
    else ts_bucket(b, s_h);
}

template <typename Src, typename Place>
__device__ __forceinline__ void ts_place(const TsSort<Src>& S, uint32_t* __restrict__ off, unsigned int* __restrict__ max_out,
                                         const Place& place, uint32_t* s_c /* [2^shift] key counts, then next slots */,
                                         uint32_t* s_wave, uint32_t* s_maxp)
{
    if (!S.blocks || (int)blockIdx.x >= S.ntiles) return;
    uint32_t& s_max = *s_maxp;
    const typename Place::Item* __restrict__ bucket = S.bucket;
    const uint32_t* __restrict__ tile_off = S.off();
    const int shift = S.shift;
    const uint32_t nkeys = S.nkeys;
    const uint32_t T = 1u << shift;
    const uint32_t k0 = (uint32_t)blockIdx.x << shift;
    const uint32_t b0 = tile_off[blockIdx.x], b1 = tile_off[blockIdx.x + 1];
    for (uint32_t j = threadIdx.x; j < T; j += TS_NT) s_c[j] = 0;
    if (threadIdx.x == 0) s_max = 0;
    __syncthreads();
    for (uint32_t i0 = b0 + threadIdx.x; i0 < b1; i0 += TS_U * TS_NT) {
        uint32_t k[TS_U];
#pragma unroll
        for (int u = 0; u < TS_U; ++u) {
            const uint32_t i = i0 + (uint32_t)u * TS_NT;
            k[u] = bucket[i < b1 ? i : i0].x;
        }
#pragma unroll
        for (int u = 0; u < TS_U; ++u)
            if (i0 + (uint32_t)u * TS_NT < b1) atomicAdd(&s_c[k[u] - k0], 1u);
    }
    __syncthreads();
    // exclusive scan of the T counts: thread r owns counts [r*C, (r+1)*C)
    const uint32_t C = T / TS_NT;
    uint32_t sum = 0, mx = 0;
    for (uint32_t c = 0; c < C; ++c) {
        const uint32_t v = s_c[threadIdx.x * C + c];
        sum += v;
        mx = v > mx ? v : mx;
    }
    const int lane = __lane_id(), wid = threadIdx.x >> 6;
    const uint32_t inc = wave_incl_scan<uint32_t>(sum);
    if (lane == 63) s_wave[wid] = inc;
    for (unsigned d = 32; d >= 1; d >>= 1) {
        const uint32_t o = __shfl_xor(mx, d);
        mx = o > mx ? o : mx;
    }
    if (lane == 0 && mx) atomicMax(&s_max, mx);
    __syncthreads();
    uint32_t run = b0 + inc - sum;
    for (int w = 0; w < wid; ++w) run += s_wave[w];
    for (uint32_t c = 0; c < C; ++c) {
        const uint32_t j = threadIdx.x * C + c;
        const uint32_t v = s_c[j];
        s_c[j] = run;
        if (k0 + j < nkeys) off[k0 + j] = run;
        run += v;
    }
    if (k0 + T >= nkeys && threadIdx.x == TS_NT - 1) off[nkeys] = b1;
    if (threadIdx.x == 0 && max_out && s_max) atomicMax(max_out, s_max);
    __syncthreads();
    for (uint32_t i0 = b0 + threadIdx.x; i0 < b1; i0 += TS_U * TS_NT) {
        typename Place::Item it[TS_U];
        uint32_t pos[TS_U];
#pragma unroll
        for (int u = 0; u < TS_U; ++u) {
            const uint32_t i = i0 + (uint32_t)u * TS_NT;
            it[u] = bucket[i < b1 ? i : i0];
        }
#pragma unroll
        for (int u = 0; u < TS_U; ++u)
            pos[u] = i0 + (uint32_t)u * TS_NT < b1 ? atomicAdd(&s_c[it[u].x - k0], 1u) : 0u;
#pragma unroll
        for (int u = 0; u < TS_U; ++u) place(pos[u], it[u], i0 + (uint32_t)u * TS_NT < b1);
    }
}

__global__ __launch_bounds__(TS_NT) void k_ts_place(TsSort<PairSrc> a, uint32_t* boff, unsigned int* max_out, PairPlace pa,
                                                    TsSort<ColSrc> b, uint32_t* coff, ColPlace pb)
{
    extern __shared__ uint32_t s_c[];
    __shared__ uint32_t s_wave[TS_NT / 64];
    __shared__ uint32_t s_max;
    if (blockIdx.y == 0) ts_place(a, boff, max_out, pa, s_c, s_wave, &s_max);
    else ts_place(b, coff, nullptr, pb, s_c, s_wave, &s_max);
}

static_assert(1u << ts_shift(0) == TS_NT, "ts_place: every thread owns at least one key of a tile");

// tiles of any sort with at most nkeys keys
static size_t ts_tiles_most(uint64_t nkeys) { return nkeys <= (1u << 21) ? ts_tiles(nkeys) : nkeys <= (1u << 26) ? 8192 : 16384; }

size_t ts_words(uint64_t nkeys) { return (3 * ts_tiles_most(nkeys) + 3) / 2 * 2; }

template <typename Src>
static TsSort<Src> ts_sort(Src src, uint64_t n, uint32_t nkeys, uint32_t* cnt, void* bucket, int items_per_block)
{
    const uint64_t ipb = (uint64_t)items_per_block;
    const int blocks = nkeys ? (int)std::min<uint64_t>(2048, std::max<uint64_t>(1, (n + ipb - 1) / ipb)) : 0;
    return TsSort<Src>{src, n, nkeys, ts_shift(nkeys), (int)ts_tiles(nkeys), blocks, cnt, static_cast<typename Src::Item*>(bucket)};
}

void launch_bins(const BinPairs& P, const BinCols& C, const uint64_t* bnd, const uint32_t* wprefix, const GridDev& g0,
                 const Meshes& M, int64_t W, int32_t* bidx, uint64_t* occ, int items_per_block, hipStream_t s)
{
    unsigned long long* oc = reinterpret_cast<unsigned long long*>(occ);
    const auto a = ts_sort(PairSrc{P.bits, P.ranked, P.tri, bnd, wprefix}, P.n, P.B, P.cnt, P.bucket, items_per_block);
    const auto b = ts_sort(ColSrc{C.key, C.zmax}, C.n, C.ncol, C.cnt, C.bucket, items_per_block);
    const int blocks = std::max(a.blocks, b.blocks), tiles = std::max(a.ntiles, b.ntiles);
    // Tile offsets by the count's last block where that is less than the launch it
    // saves (5 us): the blocks' counter takes 3.7 ns each, and 256 threads a
    // tile each a round
    const bool last = blocks <= 256 && tiles <= 2048;
    const size_t scan = ts_scan_lds(a.ntiles, b.ntiles) * 4;
    const size_t lds = last ? scan : (size_t)tiles * 4;
    const dim3 grid((unsigned)std::max(blocks, grid_for(W, TS_NT, 2048)), 3);
    if (M.nm > 1)
        k_ts_count<true><<<grid, TS_NT, lds, s>>>(a, b, last, g0, M, bnd, wprefix, W, bidx, oc);
    else
        k_ts_count<false><<<grid, TS_NT, lds, s>>>(a, b, last, g0, M, bnd, wprefix, W, bidx, oc);
    if (!P.B) launch_fill_u32(P.off, 0, 1, s);   // no keys, hence no items
    if (!blocks) return;
    if (!last) k_ts_scan<<<2, 1024, scan, s>>>(a, b);
    k_ts_bucket<<<dim3((unsigned)blocks, 2), TS_NT, (size_t)tiles * 4, s>>>(a, b);
    k_ts_place<<<dim3((unsigned)tiles, 2), TS_NT, (size_t)4 << std::max(a.shift, b.shift), s>>>(a, P.off, P.max_out, PairPlace{P.list}, b,
                                                                                          C.off, ColPlace{C.ent});
}

// Per-mesh bin totals (pairs) and largest bin of a batch: the blocks of a
// mesh (row of the grid) stride over its bins with one atomic each, the
// totals are differences of bin offsets (a block per 256 bins of the batch and
// two atomics a block: 156 us for 48 mixed meshes, 42 for 128 small ones).
__global__ __launch_bounds__(256) void k_mesh_bins(const uint32_t* __restrict__ boff, Meshes M)
{
    __shared__ uint32_t s_max[4];
    for (int m = (int)blockIdx.y; m < M.nm; m += (int)gridDim.y) {
        const uint32_t b0 = M.rank[m].b0, b1 = M.rank[m + 1].b0;
        uint32_t mx = 0;
        for (uint32_t b = b0 + blockIdx.x * 256u + threadIdx.x; b < b1; b += gridDim.x * 256u) {
            const uint32_t c = boff[b + 1] - boff[b];
            mx = c > mx ? c : mx;
        }
        for (unsigned d = 32; d >= 1; d >>= 1) {
            const uint32_t o = __shfl_xor(mx, d);
            mx = o > mx ? o : mx;
        }
        if (__lane_id() == 0) s_max[threadIdx.x >> 6] = mx;
        __syncthreads();
        if (threadIdx.x == 0) {
            for (int i = 0; i < 4; ++i) mx = s_max[i] > mx ? s_max[i] : mx;
            if (mx) atomicMax(&M.ctr[m].max_per_voxel, mx);
            if (blockIdx.x == 0) M.ctr[m].pairs = (unsigned long long)(boff[b1] - boff[b0]);
        }
        __syncthreads();
    }
}

void launch_mesh_bins(const uint32_t* boff, int64_t B, const Meshes& M, hipStream_t s)
{
    if (B <= 0) return;
    const int per = grid_for(B / M.nm, 2048, 64);
    k_mesh_bins<<<dim3((unsigned)per, (unsigned)(M.nm < 65535 ? M.nm : 65535)), 256, 0, s>>>(boff, M);
}

// ---------------------------------------------------------------------------
// Level2 SAT (src/Object.cpp:2344-2424).  One wave per group of consecutive
// boundary voxels of a mesh (l2_group_voxels).  Up to 32 bin entries at a time
// are staged, two lanes each: what the rows of the entry share
// (gpv_satrow.hpp) goes to LDS.  The lanes then take the (entry, row of
// sub-voxels) items, drop the columns that the (x, y) predicates fail (kPieces: and put
// what is left of each row in a ring, in pieces of 2, 4 or 8 columns, which keep the
// lanes of a round about equally long) and walk the others, which gives per column the
// layers the SAT accepts for certain and those it has to be run on: the
// first go straight into the wave's accumulator, the others (0.05 per entry
// on the torus knot, 9 on a lattice-snapped mesh at 512/16) queue for the
// reference's float SAT in 64-lane batches.
//
// What bounds it: VALU issue (0.58-0.65 of the measured rate at 4.5 waves per
// SIMD; 85 registers and 7 KB of LDS allow five).  Running the float SAT on
// every box a plane slab kept took 3.0e8 more instructions on the torus knot:
// 0.556 -> 0.277 ms alone at 256/8; lattice-snapped mesh at 512/16, 5.25 ->
// 3.6 ms.  Two staging lanes per entry and 32 entries per staging, because the
// 40 floats an entry's rows share would otherwise fill LDS (64 entries: three
// waves per SIMD), and recomputing them in every row costs 330 instructions a
// round (torus knot 0.36 ms).
// ---------------------------------------------------------------------------
// ring of queued (triangle, sub-voxel) entries per wave: a round pushes at
// most 64 entries onto fewer than 64 already queued, so it holds 128
constexpr int L2_QCAP = 128;
constexpr int L2_STAGE = 32;   // entries staged at once
// ring of row pieces per wave: a round pushes at most 192 onto fewer than 64
constexpr uint32_t L2_SEGS = 256;

// value of a float register in lane `l` (l uniform across the wave)
__device__ __forceinline__ float lane_f(float v, int l)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// Lane l holds row l of a 64x64 bit matrix (bit j = entry (l, j)); returns
// column l (bit j = entry (j, l)).  Six block swaps of halving size.
template <int K>
__device__ __forceinline__ uint64_t transpose_step(uint64_t v)
{
    constexpr int s = 32 >> K;
    constexpr uint64_t masks[6] = {0x00000000FFFFFFFFull, 0x0000FFFF0000FFFFull, 0x00FF00FF00FF00FFull,
                                   0x0F0F0F0F0F0F0F0Full, 0x3333333333333333ull, 0x5555555555555555ull};
    constexpr uint64_t m = masks[K];
    const uint64_t x = (uint64_t)lane_xor<s>((uint32_t)v) | ((uint64_t)lane_xor<s>((uint32_t)(v >> 32)) << 32);
    // the upper lane of each pair keeps the ~m half
    const uint64_t lo = (v & m) | ((x & m) << s);
    const uint64_t hi = (v & ~m) | ((x & ~m) >> s);
    return (__lane_id() & s) ? hi : lo;
}

__device__ __forceinline__ uint64_t wave_transpose64(uint64_t v)
{
    v = transpose_step<0>(v);
    v = transpose_step<1>(v);
    v = transpose_step<2>(v);
    v = transpose_step<3>(v);
    v = transpose_step<4>(v);
    return transpose_step<5>(v);
}

// the sub-center positions of a group's voxels, far from the origin (gpv_satrow.hpp)
template <bool kFar>
struct L2Pos {};
template <>
struct L2Pos<true> {
    float pos[kL2GroupMax][3][16];
};

// LDS of one wave of the Level2 SAT
template <bool kPieces, bool kFar>
struct L2Lds : L2Pos<kFar> {
    union {
        float4 e[L2_STAGE][kSatEntry4];                  // staged entries
        unsigned long long words[kL2GroupBytes / 8];     // output words, once the bins are done
    };
    // per sub-column (v * n2^2 + q * n2 + p) its layer bits, in bytes up to
    // n2 = 8 and in 16 bits above
    uint32_t acc[kL2GroupBytes / 4];
    uint32_t q[L2_QCAP];          // ring of queued SAT entries
    uint32_t dec[L2_STAGE];       // staged entry: first column, row and layer, last layer, columns, voxel, loose
    uint32_t vb[kL2GroupMax + 1]; // group voxel v: first bin entry
    int ci[kL2GroupMax][3];       // its sub-center 0 in the tables
    uint8_t win[64];              // per round: staged entry starting at each item position
    uint16_t seg[kPieces ? L2_SEGS : 1];   // ring of row pieces: entry | row << 5 | column << 9 | columns - 1 << 13
};

// where the layer bits of sub-column `col` lie: word index and first bit
__device__ __forceinline__ uint32_t l2_col_word(uint32_t col, int n2, uint32_t& bit)
{
    const int sh = n2 > 8 ? 1 : 2;
    bit = (col & ((1u << sh) - 1u)) << (5 - sh);
    return col >> sh;
}

// Full float SAT for queued entries (one per lane); entry = p | q<<4 | r<<8 |
// v<<12 | j<<16 where v is the voxel in the group and j the bin entry from base.
template <bool kPieces, bool kFar>
__device__ __forceinline__ void l2_sat_run(uint32_t ent, bool valid, L2Lds<kPieces, kFar>& L, const GridDev& g,
                                           const float* __restrict__ tris, const uint32_t* __restrict__ list,
                                           uint32_t base)
{
    if (!valid) return;
    const int n2 = g.n2;
    const int p = ent & 15, q = (ent >> 4) & 15, r = (ent >> 8) & 15, v = (ent >> 12) & 15;
    uint32_t bit;
    const uint32_t w = l2_col_word((uint32_t)((v * n2 + q) * n2 + p), n2, bit);
    if ((L.acc[w] >> (bit + r)) & 1u) return;
    const uint64_t t = list[base + (ent >> 16)];
    float tv[9];
#pragma unroll
    for (int c = 0; c < 9; ++c) tv[c] = tris[t * 9 + c];
    if (tri_box_overlap(g.c2x[L.ci[v][0] + p], g.c2y[L.ci[v][1] + q], g.c2z[L.ci[v][2] + r], g.h2x, g.h2y, g.h2z, tv))
        atomicOr(&L.acc[w], 1u << (bit + r));
}

// The boxes of a voxel that pass the SAT's predicate of one box axis, c their
// n centers: the float test's two halves fl(lo - c) > h and fl(hi - c) < -h (lo, hi
// the triangle's extent) are monotone along c, so they are those from first to
// last, searched from k on.
__device__ __forceinline__ int l2_axis_first(const float* __restrict__ c, int n, float lo, float h, int k)
{
    k = k < 0 ? 0 : k < n ? k : n;
    while (k < n && lo - c[k] > h) ++k;
    while (k > 0 && !(lo - c[k - 1] > h)) --k;
    return k;
}

__device__ __forceinline__ int l2_axis_last(const float* __restrict__ c, int n, float hi, float h, int k)
{
    k = k < -1 ? -1 : k < n ? k : n - 1;
    while (k + 1 < n && !(hi - c[k + 1] < -h)) ++k;
    while (k >= 0 && hi - c[k] < -h) --k;
    return k;
}

template <bool kM, int W, bool kPieces, bool kFar>
__global__ __launch_bounds__(64 * W) void k_l2_sat(const float* __restrict__ tris, const int32_t* __restrict__ bidx,
                                                   int64_t B, int64_t ngroups, int gmost,
                                                   const uint32_t* __restrict__ boff,
                                                   const uint32_t* __restrict__ list,
                                                   GridDev g0, Meshes M, uint64_t* __restrict__ sat2)
{
    __shared__ L2Lds<kPieces, kFar> s_l[W];
    const int wv = threadIdx.x >> 6;
    const int lane = __lane_id();
    L2Lds<kPieces, kFar>& L = s_l[wv];
    const int64_t grp = (int64_t)blockIdx.x * W + wv;
    if (grp >= ngroups) return;
    int mesh = 0;
    if constexpr (kM)
        mesh = wave_mesh_search(M.rank, M.nm, (uint64_t)grp, [](const MeshRank& o) { return (uint64_t)o.sg0; });
    const GridDev& g = grid_of<kM>(g0, M, mesh);
    const int n2 = g.n2, w2 = g.w2, nsc = n2 * n2;
    if (kM && n2 == 0) return;
    const int64_t mb0 = kM ? (int64_t)M.rank[mesh].b0 : 0, mb1 = kM ? (int64_t)M.rank[mesh + 1].b0 : B;
    const int G = l2_group_voxels(n2, gmost);
    const int64_t vb0 = mb0 + (grp - (kM ? (int64_t)M.rank[mesh].sg0 : 0)) * G;
    if (vb0 >= mb1) return;
    const int nv = (int)(mb1 - vb0 < G ? mb1 - vb0 : G);
    uint64_t* out = sat2 + (kM ? M.rank[mesh].l2w0 : 0) + (uint64_t)(vb0 - mb0) * w2;
    for (int i = lane; i < (nv * nsc * (n2 > 8 ? 2 : 1) + 3) / 4; i += 64) L.acc[i] = 0u;
    if (lane <= nv) L.vb[lane] = boff[vb0 + lane];
    if (lane < nv) {
        const int vox = bidx[vb0 + lane];
        const int nxy = g.nx * g.ny;
        const int k1 = vox / nxy;
        const int ij = vox - k1 * nxy;
        const int j1 = ij / g.nx;
        const int i1 = ij - j1 * g.nx;
        L.ci[lane][0] = i1 * n2;
        L.ci[lane][1] = j1 * n2;
        L.ci[lane][2] = k1 * n2;
    }
    __builtin_amdgcn_wave_barrier();
    const SatScale sc{g.s2x, g.s2y, g.s2z, g.d2x, g.d2y, g.d2z};
    const SatScale se = kFar ? sat_scale_far(sc) : sc;   // of the entries
    const int half = n2 > 8 ? 8 : 4;
    if constexpr (kFar) {
        for (int i = lane; i < nv * 48; i += 64) {
            const int v = i / 48, a = (i - v * 48) >> 4, p = i & 15;
            const float* c = (a == 0 ? g.c2x : a == 1 ? g.c2y : g.c2z) + L.ci[v][a];
            const float s = a == 0 ? sc.sx : a == 1 ? sc.sy : sc.sz;
            L.pos[v][a][p] = p < n2 ? (c[p] - c[0]) * s + (a == 2 ? 1.0f : 0.0f) : __builtin_inff();
        }
    }
    uint32_t qh = 0, qt = 0;   // ring head/tail (uniform)
    const uint32_t e0 = (uint32_t)uniform_i((int)L.vb[0]), e1 = (uint32_t)uniform_i((int)L.vb[nv]);
    uint32_t qbase = e0;       // the bin entry that queued entries count from
    for (uint32_t base = e0; base < e1; base += L2_STAGE) {
        if (base - qbase > 0xffffu - L2_STAGE) {   // their 16 bits would not do
            const bool valid = (uint32_t)lane < qt - qh;
            l2_sat_run(valid ? L.q[(qh + lane) % L2_QCAP] : 0u, valid, L, g, tris, list, qbase);
            qh = qt;
            qbase = base;
            __builtin_amdgcn_wave_barrier();
        }
        // staging: lanes j and j + 32 make bin entry base + j
        const int js = lane & (L2_STAGE - 1), h = lane >> 5;
        const uint32_t i = base + (uint32_t)js;
        uint32_t P = 0;   // rows of the entry (lanes below 32)
        int v = 0, a0 = 0, a1 = -1, az = 0;
        bool loose = false;
        if (i < e1) {
            const uint64_t t = list[i];
            float tv[9];
#pragma unroll
            for (int c = 0; c < 9; ++c) tv[c] = tris[t * 9 + c];
            int hi = nv;   // the voxel whose entries hold i: vb[v] <= i < vb[v + 1]
            while (hi - v > 1) {
                const int mid = (v + hi) >> 1;
                if (L.vb[mid] <= i) v = mid;
                else hi = mid;
            }
            const float *cx = g.c2x + L.ci[v][0], *cy = g.c2y + L.ci[v][1], *cz = g.c2z + L.ci[v][2];
            loose = sat_entry_part(h, tv, cx[0], cy[0], cz[0], se, L.e[js]);
            // box axes: x and the first layer by the lower lane, y and the last by the upper
            const float lo = h ? fminf(fminf(tv[1], tv[4]), tv[7]) : fminf(fminf(tv[0], tv[3]), tv[6]);
            const float top = h ? fmaxf(fmaxf(tv[1], tv[4]), tv[7]) : fmaxf(fmaxf(tv[0], tv[3]), tv[6]);
            const float* c = h ? cy : cx;
            const float hh = h ? g.h2y : g.h2x, s = h ? sc.sy : sc.sx, c0 = h ? cy[0] : cx[0];
            const float dev = h ? sc.dy : sc.dx;
            const float z = h ? fmaxf(fmaxf(tv[2], tv[5]), tv[8]) : fminf(fminf(tv[2], tv[5]), tv[8]);
            bool clear = true;
            a0 = sat_axis_end((lo - c0) * s, n2, dev, clear);
            a1 = sat_axis_end((top - c0) * s, n2, dev, clear);
            az = sat_axis_end((z - cz[0]) * sc.sz, n2, sc.dz, clear);
            if (!clear) {
                a0 = l2_axis_first(c, n2, lo, hh, a0);
                a1 = l2_axis_last(c, n2, top, hh, a1);
                az = h ? l2_axis_last(cz, n2, z, g.h2z, az) : l2_axis_first(cz, n2, z, g.h2z, az);
            }
            a0 = a0 > 0 ? a0 : 0;
            a1 = a1 < n2 ? a1 : n2 - 1;
            az = h ? (az < n2 ? az : n2 - 1) : (az > 0 ? az : 0);
        }
        {
            // the upper lane's run of rows, last layer and looseness
            const int qa = (int)lane_xor<32>((uint32_t)a0), qb = (int)lane_xor<32>((uint32_t)a1),
                      rb = (int)lane_xor<32>((uint32_t)az);
            const uint64_t bad = __ballot(loose);
            if (h == 0 && a1 >= a0 && qb >= qa && rb >= az) {
                L.dec[js] = (uint32_t)a0 | ((uint32_t)qa << 4) | ((uint32_t)az << 8) | ((uint32_t)rb << 12) |
                            ((uint32_t)(a1 - a0) << 16) | ((uint32_t)v << 20) |
                            (((bad >> js) | (bad >> (js + 32))) & 1ull ? 0x80000000u : 0u);
                P = (uint32_t)(qb - qa + 1);
            }
        }
        const uint32_t incl = wave_incl_scan<uint32_t>(P);
        const uint32_t so = incl - P;   // this lane's entry: items [so, so + P)
        const uint32_t S = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
        __builtin_amdgcn_wave_barrier();
        // the chunk's (entry, row) items, 64 per round, less the columns that the (x, y)
        // predicates fail.  kPieces: what is left of each row goes to the ring in pieces
        // of 2, 4 or 8 columns, and 64 of those make a round
        uint32_t rh = 0, rt = 0;   // ring head/tail (uniform)
        for (uint32_t l0 = 0;;) {
            int j, q, p, left;   // entry, row, first column, columns
            if (rt - rh < 64 && l0 < S) {
                // each item's entry: every entry with items in [l0, l0 + 64) marks
                // its first position there (the one running into the window marks
                // 0; starts are distinct), and item l takes the mark at the highest
                // marked position <= l
                L.win[lane] = 0xff;
                __builtin_amdgcn_wave_barrier();
                if (P && so < l0 + 64u && so + P > l0) L.win[so > l0 ? so - l0 : 0u] = (uint8_t)lane;
                __builtin_amdgcn_wave_barrier();
                const uint32_t wj = L.win[lane];
                const uint64_t marks = __ballot(wj != 0xffu) & ((2ull << lane) - 1ull);
                const int top = marks ? 63 - __clzll((long long)marks) : 0;
                j = __shfl((int)wj, top) & (L2_STAGE - 1);
                const uint32_t so_j = (uint32_t)__shfl((int)so, j);
                __builtin_amdgcn_wave_barrier();
                const uint32_t l = l0 + (uint32_t)lane;
                l0 += 64;
                // lanes past the last item repeat one with no columns to do
                const uint32_t d = L.dec[j];
                q = (int)(((d >> 4) & 15) + (l - so_j));
                p = d & 15;
                left = (int)((d >> 16) & 15) + 1;   // columns of the row
                if constexpr (kFar) {
                    const int vj = (int)((d >> 20) & 15u);
                    sat_row_range_far(L.e[j], L.pos[vj][1][q & 15], L.pos[vj][0], half, d >> 31 != 0, p, left);
                } else sat_row_range(L.e[j], q, d >> 31 != 0, p, left);
                left = l < S && left > 0 ? left : 0;
                if constexpr (kPieces) {
                    // pieces of each size, in fields of their own (at most 512, 256, 128 in all)
                    const uint32_t pk = (uint32_t)((left + 1) >> 1) | ((uint32_t)((left + 3) >> 2) << 11) |
                                        ((uint32_t)((left + 7) >> 3) << 21);
                    const uint32_t inc = wave_incl_scan<uint32_t>(pk);
                    const uint32_t tot = (uint32_t)__builtin_amdgcn_readlane((int)inc, 63);
                    const uint32_t n2s = tot & 0x7ffu, n4s = (tot >> 11) & 0x3ffu, n8s = tot >> 21;
                    // the cheapest: a piece costs about 120 instructions, a column 62
                    uint32_t sh = 3, fs = 21, best = 616u * n8s;
                    if (n4s <= L2_SEGS - 64 && 368u * n4s <= best) sh = 2, fs = 11, best = 368u * n4s;
                    if (n2s <= L2_SEGS - 64 && 244u * n2s <= best) sh = 1, fs = 0;
                    const uint32_t mask = sh == 1 ? 0x7ffu : 0x3ffu;
                    const uint32_t own = (pk >> fs) & mask, at = rt + (((inc - pk) >> fs) & mask);
                    for (uint32_t k = 0; __ballot(k < own); ++k)
                        if (k < own) {
                            const uint32_t done = k << sh, cnt = min((uint32_t)left - done, 1u << sh);
                            L.seg[(at + k) % L2_SEGS] = (uint16_t)((uint32_t)j | ((uint32_t)q << 5) | (((uint32_t)p + done) << 9) | ((cnt - 1u) << 13));
                        }
                    rt += (tot >> fs) & mask;
                    __builtin_amdgcn_wave_barrier();
                    continue;
                }
            } else {
                if constexpr (!kPieces) break;
                const uint32_t np = rt - rh < 64 ? rt - rh : 64u;
                if (!np) break;
                // lanes past the last piece repeat one with no columns to do
                const uint32_t pc = L.seg[(rh + ((uint32_t)lane < np ? (uint32_t)lane : 0u)) % L2_SEGS];
                rh += np;
                j = (int)(pc & 31u);
                q = (int)((pc >> 5) & 15u);
                p = (int)((pc >> 9) & 15u);
                left = (uint32_t)lane < np ? (int)(pc >> 13) + 1 : 0;
            }
            asm("" : "+v"(left));   // a plain number to the loop: a compare a column, not the select above
            const uint32_t d = L.dec[j];
            const int ra = (d >> 8) & 15, rb = (d >> 12) & 15, v = (int)((d >> 20) & 15u);
            const bool loose = d >> 31 != 0;
            SatRow row;
            if constexpr (kFar) row = sat_row_xy(L.e[j], L.pos[v][1][q & 15], -1e9f, 1e9f, L.pos[v][0][p & 15]);
            else row = sat_row_at(L.e[j], q, ra, rb, p);
            if (__ballot(loose)) sat_row_loose(row, loose, kFar ? -1 : ra, kFar ? 1 << 30 : rb);
            const uint32_t layers = (2u << rb) - (1u << ra);
            uint32_t col = (uint32_t)((v * n2 + q) * n2 + p);
            const uint32_t ent = (uint32_t)p | ((uint32_t)q << 4) | ((uint32_t)v << 12) | ((base - qbase + (uint32_t)j) << 16);
            for (int k = 0;; ++k, ++col) {
                const bool on = k < left;
                if (!__ballot(on)) break;
                uint32_t unk = 0;
                if (on) {
                    uint32_t in, may;
                    if constexpr (kFar) {
                        // (the last column takes no step)
                        const float step = k + 1 < left ? L.pos[v][0][p + k + 1] - L.pos[v][0][p + k] : 0.0f;
                        sat_row_column_far(row, L.pos[v][2], half, layers, step, in, may);
                    } else sat_row_column(row, in, may);
                    unk = may & ~in;
                    if (in) {
                        uint32_t bit;
                        const uint32_t w = l2_col_word(col, n2, bit);
                        atomicOr(&L.acc[w], in << bit);
                    }
                }
                // the undecided boxes, one layer per lane per pass
                for (uint64_t m; (m = __ballot(unk != 0)) != 0;) {
                    if (unk) {
                        const uint32_t r = (uint32_t)__ffs(unk) - 1u;
                        L.q[(qt + (uint32_t)__popcll(m & lanes_below_mask())) % L2_QCAP] = (ent + (uint32_t)k) | (r << 8);
                        unk &= unk - 1;
                    }
                    qt += (uint32_t)__popcll(m);
                    __builtin_amdgcn_wave_barrier();
                    if (qt - qh >= 64) {   // a full wave of work
                        l2_sat_run(L.q[(qh + lane) % L2_QCAP], true, L, g, tris, list, qbase);
                        qh += 64;
                        __builtin_amdgcn_wave_barrier();
                    }
                }
            }
        }
    }
    if (qt != qh) {
        const bool valid = (uint32_t)lane < qt - qh;
        l2_sat_run(valid ? L.q[(qh + lane) % L2_QCAP] : 0u, valid, L, g, tris, list, qbase);
    }
    __builtin_amdgcn_wave_barrier();
    // layer bits per sub-column -> words of sub-voxels: bit s of word m is
    // sub-voxel 64 m + s = layer * n2^2 + sub-column
    const uint8_t* a8 = reinterpret_cast<const uint8_t*>(L.acc);
    const uint16_t* a16 = reinterpret_cast<const uint16_t*>(L.acc);
    if (n2 == 8) {
        // bit 8v + r of lane c: layer r of sub-column c of voxel v; transposed,
        // lane 8v + r holds word r of voxel v
        for (int v0 = 0; v0 < nv; v0 += 8) {
            uint64_t b = 0;
            for (int v = 0; v < 8 && v0 + v < nv; ++v) b |= (uint64_t)a8[(v0 + v) * 64 + lane] << (8 * v);
            b = wave_transpose64(b);
            if (v0 * 8 + lane < nv * 8) out[v0 * 8 + lane] = b;
        }
        return;
    }
    if (n2 == 16) {
        // bit 16k + r of lane c: layer r of sub-column 64k + c; transposed, lane
        // 16k + r holds word 4r + k
        for (int v = 0; v < nv; ++v) {
            uint64_t b = 0;
            for (int k = 0; k < 4; ++k) b |= (uint64_t)a16[v * 256 + k * 64 + lane] << (16 * k);
            out[v * 64 + 4 * (lane & 15) + (lane >> 4)] = wave_transpose64(b);
        }
        return;
    }
    const float inv = GPV_RCP((float)nsc);
    for (int m = 0; m < w2; ++m) {
        const int s = 64 * m + lane;
        const int r = (int)(((float)s + 0.5f) * inv);   // exact: s + 1/2 is at least 1/512 of n2^2 from a multiple
        const int sub = s - r * nsc;
        for (int v = 0; v < nv; ++v) {
            const uint32_t bits = n2 > 8 ? (uint32_t)a16[v * nsc + sub] : (uint32_t)a8[v * nsc + sub];
            const uint64_t wd = __ballot(r < n2 && ((bits >> r) & 1u));
            if (lane == 0) L.words[v * w2 + m] = wd;
        }
    }
    __builtin_amdgcn_wave_barrier();
    for (int i = lane; i < nv * w2; i += 64) out[i] = L.words[i];
}

template <int W, bool kPieces, bool kFar = false>
static void launch_l2_sat_w(const float* tris, const int32_t* bidx, int64_t B, int64_t ngroups, int gmost,
                            const uint32_t* boff, const uint32_t* list, const GridDev& g0, const Meshes& M,
                            uint64_t* sat2, hipStream_t s)
{
    const unsigned blocks = (unsigned)((ngroups + W - 1) / W);
    if (M.nm > 1)
        k_l2_sat<true, W, kPieces, kFar><<<blocks, 64 * W, 0, s>>>(tris, bidx, B, ngroups, gmost, boff, list, g0, M, sat2);
    else
        k_l2_sat<false, W, kPieces, kFar><<<blocks, 64 * W, 0, s>>>(tris, bidx, B, ngroups, gmost, boff, list, g0, M, sat2);
}

template <bool kPieces>
static void launch_l2_sat_p(const float* tris, const int32_t* bidx, int64_t B, int64_t ngroups, int gmost,
                            const uint32_t* boff, const uint32_t* list, int waves, const GridDev& g0, const Meshes& M,
                            uint64_t* sat2, hipStream_t s)
{
    if (waves <= 1) launch_l2_sat_w<1, kPieces>(tris, bidx, B, ngroups, gmost, boff, list, g0, M, sat2, s);
    else if (waves == 2) launch_l2_sat_w<2, kPieces>(tris, bidx, B, ngroups, gmost, boff, list, g0, M, sat2, s);
    else launch_l2_sat_w<4, kPieces>(tris, bidx, B, ngroups, gmost, boff, list, g0, M, sat2, s);
}

void launch_l2_sat(const float* tris, const int32_t* bidx, int64_t B, int64_t ngroups, int gmost, const uint32_t* boff,
                   const uint32_t* list, int n2max, bool far, int waves, const GridDev& g0, const Meshes& M,
                   uint64_t* sat2, hipStream_t s)
{
    if (B <= 0 || ngroups <= 0) return;
    // one wave a block is the default of `waves` as well
    if (far) {
        if (n2max > 8) launch_l2_sat_w<1, true, true>(tris, bidx, B, ngroups, gmost, boff, list, g0, M, sat2, s);
        else launch_l2_sat_w<1, false, true>(tris, bidx, B, ngroups, gmost, boff, list, g0, M, sat2, s);
        return;
    }
    // Rows in pieces above n2 = 8, where a round of whole rows waits for one of up to 16
    // columns (lattice-snapped mesh at 512/16: 2.54 -> 2.24 ms alone).  Shorter rows do not
    // pay for the ring: torus knot 256/8 the same, 128 small meshes at 64/4 2.25 -> 2.29 ms in all
    if (n2max > 8) launch_l2_sat_p<true>(tris, bidx, B, ngroups, gmost, boff, list, waves, g0, M, sat2, s);
    else launch_l2_sat_p<false>(tris, bidx, B, ngroups, gmost, boff, list, waves, g0, M, sat2, s);
}

// ---------------------------------------------------------------------------
// Level2 ray parity (src/Object.cpp:1111-1207), by xy columns.  A boundary
// voxel (i1, j1, k1) takes the triangles of the bins at z' >= k1 in its column,
// which are the column's (triangle, zmax) entries with zmax >= k1, and each of
// its sub-voxels counts those whose +z ray test passes.  One wave takes one
// column (or two or four adjacent ones, l2_parity_columns): for every (entry, sub-column) pair
// that the float det/u/v test accepts it finds the number of layers whose
// t > 1e-6 holds -- the layers below the crossing, bounded by gpv_parcol.hpp,
// with the float test deciding the few within rounding of it -- and toggles one
// bit there.  The toggles at or above a layer are then its parity.
//
// Pairs, not voxels: an entry's accepted sub-columns are found once for the
// column (by rows of its xy range, then by the columns each row can accept),
// where a wave per voxel repeated every entry above each voxel: torus knot
// 256/8 0.232 -> 0.129 ms alone (1.82e8 -> 0.72e8 instructions), lattice-snapped
// mesh 512/16 3.90 -> 2.24 ms, 128 small meshes 0.60 -> 0.39 ms.
//
// From 8,192 columns on those without a boundary voxel are known from the bins' launch, a
// bit each: their waves leave at once (a scan of 512 layers by every one of 262,144
// columns took 0.89 ms of an almost empty grid at 512/16, now 0.06).
//
// A column of several windows looks up each window's voxels in the 64-layer words that hold
// them (28,000 columns of 16,000 layers at n2 = 4 28.3 -> 6.5 ms with every word scanned once).
// A wave per voxel is still the faster way in a few hundred columns of thousands of layers at
// n2 = 16 (by a quarter).
//
// What bounds it: the chain of dependent LDS and global reads of each wave
// (VALU issue 0.39-0.47), hence one wave per block (an empty column's wave
// leaves at once; two waves a block took 0.15 ms on the torus knot), 80
// registers for six waves per SIMD (three waves: 0.18 ms, eight: no gain), scans
// and transposes without LDS, and 32 staged entries.  Four columns per wave at
// n2 = 8 took 0.31 ms.
// ---------------------------------------------------------------------------
constexpr int L2P_STAGE = 32;    // entries staged at once
constexpr int L2P_SHARE = 4;     // waves that share a column where there are few
constexpr int L2P_SLOTS = 128;   // boundary voxels of a window, all columns of the wave

// LDS of the V waves that take a column (or a few) together in the Level2 parity
template <int KB, int V>
struct L2PLds {
    // staged entries of each: e1, e2x | e2y, e2z, inv, v1x | v1y, dz, mu, delta | l0, cap, column, v1z
    float4 e[V][L2P_STAGE][4];
    // per (column, slot, sub-column) its toggles, in bytes up to n2 = 8 and in
    // 16 bits above; a column's row past its slots holds the parity of the windows above
    uint32_t acc[KB / 4];
    uint32_t slotb[L2P_SLOTS];   // boundary voxel of each slot
    float ox[16], oy[16];        // origins of the columns (c * n2 + p) and of the row
    uint8_t win[V][64];
};

// parity waves of a mesh with ncol columns
int64_t l2_parity_waves(int n2, int64_t ncol, bool many)
{
    return n2 <= 0 ? 0 : ncol / l2_parity_columns(n2, many);
}

// between the phases of a column
template <int V>
__device__ __forceinline__ void l2_parity_barrier()
{
    if constexpr (V > 1) __syncthreads();
    else __builtin_amdgcn_wave_barrier();
}

// C adjacent columns (i1 .., j1) of a mesh by one wave: 1, 2 (at n2 <= 8) or 4 (at n2 <= 4);
// or, V > 1, by the V waves of a block, this one `wv`, which share the entries.
template <int C, int KB, int V, bool kFar>
__device__ __forceinline__ void l2_parity_columns_wave(L2PLds<KB, V>& L, int wv, uint32_t wave, const L2Heavy& H, uint64_t* cb, int nw,
                                                       const GridDev& g, int i1, int j1,
                                                       uint64_t word0, uint32_t col0, uint32_t b0, uint32_t cw0,
                                                       const uint64_t* __restrict__ occ,
                                                       const uint64_t* __restrict__ bnd,
                                                       const uint32_t* __restrict__ wprefix,
                                                       const uint32_t* __restrict__ coff,
                                                       const uint2* __restrict__ ent, const float* __restrict__ tris,
                                                       uint64_t* __restrict__ out)
{
    const int lane = __lane_id(), tid = wv * 64 + lane;
    constexpr int NT = V * 64;
    float4(*const E)[4] = L.e[wv];
    uint8_t* const win = L.win[wv];
    const int n2 = g.n2, w2 = g.w2, nsc = n2 * n2, nz = g.nz;
    const int bit0 = i1 & 63;
    const uint32_t cword = (uint32_t)j1 * (uint32_t)g.nxw + (uint32_t)(i1 >> 6);
    if (occ && !((occ[cw0 + cword] >> bit0) & ((1u << C) - 1u))) return;   // no boundary voxel in these columns
    const int fb = C == 1 && n2 > 8 ? 2 : 1;
    uint32_t* pre = reinterpret_cast<uint32_t*>(cb + C * nw);
    const uint32_t gcol = col0 + (uint32_t)(j1 * g.nx + i1);
    uint32_t ce[C + 1];   // the columns' first entries
#pragma unroll
    for (int c = 0; c <= C; ++c) ce[c] = coff[gcol + (uint32_t)c];
    if (V == 1 && H.list && ce[C] - ce[0] > H.above * C) {   // left to the second launch
        if (lane == 0) {
            const uint32_t at = atomicAdd(H.count, 1u);
            if ((int64_t)at < H.most) H.list[at] = wave;
        }
        return;
    }
    if (tid < C * n2) L.ox[tid] = g.r2x[i1 * n2 + tid];
    if (tid < n2) L.oy[tid] = g.r2y[j1 * n2 + tid];
    // slots of a column per window; one more row carries what lies above it
    const int Wn = min(KB / (C * nsc * fb) - 1, L2P_SLOTS / C);
    // the columns' boundary voxels: a bit per layer, their number below each
    // word of bits, and the boundary index of each slot of the window [lo, hi)
    const uint64_t word = word0 + (uint64_t)cword;
    const uint64_t plane = (uint64_t)g.ny * g.nxw;
    uint32_t S[C], lo[C], hi[C];
    auto scan = [&](bool first) {
#pragma unroll
        for (int c = 0; c < C; ++c) S[c] = first ? 0u : S[c];   // the columns' totals, once made
        for (int kw = 0; kw * 64 < nz; ++kw) {
            if (!first) {   // past 64 layers with nothing in the window
                bool any = false;
#pragma unroll
                for (int c = 0; c < C; ++c) {
                    const uint32_t p = pre[c * nw + kw];
                    any = any || (p < hi[c] && p + (uint32_t)__popcll(cb[c * nw + kw]) > lo[c]);
                }
                if (!any) continue;
            }
            const int k = kw * 64 + lane;
            uint64_t bits = 0;
            uint32_t base = 0;
            if (k < nz) {
                const uint64_t w = word + (uint64_t)k * plane;
                bits = bnd[w];
                base = wprefix[w] - b0;
            }
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const uint64_t m = __ballot((bits >> (bit0 + c)) & 1ull);
                const uint32_t rank = (first ? S[c] : pre[c * nw + kw]) + (uint32_t)__popcll(m & lanes_below_mask());
                if (first && tid == 0) {
                    cb[c * nw + kw] = m;
                    pre[c * nw + kw] = S[c];
                }
                if (wv == 0 && ((m >> lane) & 1ull) && rank >= lo[c] && rank < hi[c])
                    L.slotb[c * Wn + (int)(rank - lo[c])] = base + (uint32_t)__popcll(bits & ((1ull << (bit0 + c)) - 1ull));
                if (first) S[c] += (uint32_t)__popcll(m);
            }
        }
    };
#pragma unroll
    for (int c = 0; c < C; ++c) {
        lo[c] = 0u;
        hi[c] = (uint32_t)Wn;
    }
    scan(true);
    uint32_t most = 0;
#pragma unroll
    for (int c = 0; c < C; ++c) most = max(most, S[c]);
    if (most == 0) return;
    const SatScale sc{g.s2x, g.s2y, g.s2z, g.d2x, g.d2y, g.d2z};
    const float gx = 2.0f * g.h2x, gy = 2.0f * g.h2y, inv_n2 = GPV_RCP((float)n2);
    const float* rz = g.r2z;
    const bool scaled = sc.dx >= 0.0f && sc.dy >= 0.0f && sc.dz >= 0.0f;
    uint8_t* a8 = reinterpret_cast<uint8_t*>(L.acc);
    uint16_t* a16 = reinterpret_cast<uint16_t*>(L.acc);
    // windows of slots from the top down (one, but for columns of many boundary voxels)
    for (uint32_t w0 = 0; w0 < most; w0 += (uint32_t)Wn) {
#pragma unroll
        for (int c = 0; c < C; ++c) {
            hi[c] = S[c] > w0 ? S[c] - w0 : 0u;
            lo[c] = hi[c] > (uint32_t)Wn ? hi[c] - (uint32_t)Wn : 0u;
        }
        if (most > (uint32_t)Wn) {
            if (w0 == 0) l2_parity_barrier<V>();   // cb and pre
            scan(false);
        }
        // clear the slots; the row past them keeps the parity of all windows above
        if (w0 == 0) {
            for (int i = tid; i < (C * (Wn + 1) * nsc * fb + 3) / 4; i += NT) L.acc[i] = 0u;
        } else {
            for (int i = tid; i < C * Wn * nsc; i += NT) {
                const int c = C == 1 ? 0 : i / (Wn * nsc);
                const int at = i + c * nsc;
                if (fb == 2) a16[at] = 0;
                else a8[at] = 0;
            }
        }
        l2_parity_barrier<V>();
        for (uint32_t base = ce[0] + (uint32_t)wv * L2P_STAGE; base < ce[C]; base += V * L2P_STAGE) {
            const uint32_t i = base + (uint32_t)lane;
            uint32_t P = 0;   // rows of this lane's entry
            int q0 = 0;
            if (lane < L2P_STAGE && i < ce[C]) {
                const uint2 en = ent[i];
                float tv[9];
#pragma unroll
                for (int k = 0; k < 9; ++k) tv[k] = tris[(uint64_t)en.x * 9 + k];
                MtTri m;
                mt_setup(tv, m);   // entries exist only for triangles whose det passes
                int c = 0;
#pragma unroll
                for (int k = 1; k < C; ++k) c += (int)(i >= ce[k]);
                const int zmax = (int)en.y;
                ParEntry r;
                r.e1x = m.e1x; r.e1y = m.e1y; r.e1z = m.e1z; r.e2x = m.e2x;
                r.e2y = m.e2y; r.e2z = m.e2z; r.inv = m.inv_det; r.v1x = tv[0];
                r.v1y = tv[1];
                r.l0 = zmax * n2;
                const float ox0 = L.ox[c * n2], oy0 = L.oy[0];
                par_entry(r, tv[2], par_oz(g.bminz, 2.0f * g.h1z, 2.0f * g.h2z, zmax), ox0, oy0, gx, gy, n2, sc);
                // candidate for the voxels up to zmax (all with the CUDA kernels' whole-column lists)
                const int cap = (g.l2cuda ? nz : zmax + 1) * n2;
                float ez = 0.0f;
                if constexpr (kFar) {
                    ez = scaled ? par_ez(m.e1x, m.e1y, m.e1z, m.e2x, m.e2y, m.e2z, m.inv_det) : 3.0e38f;
                    r.delta = par_delta_far(r, ox0, oy0, gx, gy, n2, sc);
                    r.mu = par_mu_far(ez, sc, nz * n2);
                }
                bool meets = true;
                if (most > (uint32_t)Wn) {
                    // some toggle may fall into this window's slots
                    uint32_t clo = lo[0], chi = hi[0];
#pragma unroll
                    for (int k = 1; k < C; ++k) {
                        clo = c == k ? lo[k] : clo;
                        chi = c == k ? hi[k] : chi;
                    }
                    int lmin, lmax;
                    par_z_range(r, sc.sz, cap, lmin, lmax);
                    auto upto = [&](int n) -> uint32_t {   // boundary voxels at or below layer n - 1
                        if (n <= 0) return 0u;
                        const int k = (int)(((float)(n - 1) + 0.5f) * inv_n2);
                        return pre[c * nw + (k >> 6)] + (uint32_t)__popcll(cb[c * nw + (k >> 6)] & ((2ull << (k & 63)) - 1ull));
                    };
                    meets = upto(lmin) <= chi && upto(lmax) > clo;
                }
                const int nq = !meets ? 0 : kFar ? par_rows_far(r, L.oy, sc.sy, n2, q0) : par_rows(r, oy0, sc.sy, n2, sc.dy, q0);
                P = nq > 0 ? (uint32_t)nq : 0u;
                E[lane][0] = make_float4(m.e1x, m.e1y, m.e1z, m.e2x);
                E[lane][1] = make_float4(m.e2y, m.e2z, m.inv_det, tv[0]);
                E[lane][2] = make_float4(tv[1], r.dz, kFar ? ez : r.mu, r.delta);   // (the pairs make mu of ez)
                E[lane][3] = make_float4(__int_as_float(r.l0), __int_as_float(cap), __int_as_float(c), tv[2]);
            }
            const uint32_t incl = wave_incl_scan<uint32_t>(P);
            const uint32_t so = incl - P;
            const uint32_t rows = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
            __builtin_amdgcn_wave_barrier();
            // the (entry, row) items: the columns each row can accept
            for (uint32_t l0 = 0; l0 < rows; l0 += 64) {
                const int j = wave_item_owner(win, so, P, l0) & (L2P_STAGE - 1);
                const int q = __shfl(q0, j) + (int)(l0 + (uint32_t)lane - (uint32_t)__shfl((int)so, j));
                int p0 = 0, np = 0;
                if (l0 + (uint32_t)lane < rows) {
                    const float4 a = E[j][0], b = E[j][1], d = E[j][2];
                    const int c = C == 1 ? 0 : __float_as_int(E[j][3].z);
                    ParEntry r;
                    r.e1x = a.x; r.e1y = a.y; r.e2x = a.w;
                    r.e2y = b.x; r.inv = b.z; r.v1x = b.w;
                    r.v1y = d.x; r.delta = d.w;
                    np = kFar ? par_cols_far(r, L.ox + c * n2, L.oy[q], gx, n2, p0)
                              : par_cols(r, L.ox[c * n2], L.oy[0], gx, gy, n2, q, p0);
                    np = np > 0 ? np : 0;
                }
                const uint32_t pincl = wave_incl_scan<uint32_t>((uint32_t)np);
                const uint32_t pso = pincl - (uint32_t)np;
                const uint32_t pairs = (uint32_t)__builtin_amdgcn_readlane((int)pincl, 63);
                const int pq = p0 | (q << 8) | (j << 16);
                // the (entry, sub-column) pairs
                for (uint32_t m0 = 0; m0 < pairs; m0 += 64) {
                    const int o = wave_item_owner(win, pso, (uint32_t)np, m0);
                    const int v = __shfl(pq, o);
                    const uint32_t at = m0 + (uint32_t)lane - (uint32_t)__shfl((int)pso, o);
                    if (m0 + (uint32_t)lane < pairs) {
                        const int pp = (v & 255) + (int)at, qq = (v >> 8) & 255, jj = v >> 16;
                        const float4 a = E[jj][0], b = E[jj][1], d = E[jj][2], f = E[jj][3];
                        const int c = C == 1 ? 0 : __float_as_int(f.z);
                        // the float det/u/v test (mt_column)
                        const float tx = L.ox[c * n2 + pp] - b.w, ty = L.oy[qq] - d.x;
                        const float u = (tx * -b.x + ty * a.w) * b.z;
                        const float vv = (tx * a.y - ty * a.x) * b.z;
                        int la = 0, lb = 0;
                        const bool accepted = !((u < 0.f) | (u > 1.f) | (vv < 0.f) | (u + vv > 1.f));
                        if (accepted) {
                            ParEntry r;
                            r.e1z = a.z; r.e2z = b.y; r.dz = d.y; r.mu = d.z;
                            r.l0 = __float_as_int(f.x);
                            if (kFar) r.mu = par_mu_far(d.z, sc, nz * n2);
                            par_layers(r, u, vv, sc.sz, __float_as_int(f.y), la, lb);
                            if (kFar && lb - la > 1) {
                                const float zc = (u * a.z + vv * b.y) - 1.0e-6f;
                                par_narrow(rz, n2, inv_n2, f.w, zc - 2.0f * d.z, zc + 2.0f * d.z, la, lb);
                            }
                        }
                        uint32_t clo = lo[0], chi = hi[0];
#pragma unroll
                        for (int k = 1; k < C; ++k) {
                            clo = c == k ? lo[k] : clo;
                            chi = c == k ? hi[k] : chi;
                        }
                        const uint32_t sub = (uint32_t)(c * (Wn + 1) * nsc + qq * n2 + pp);
                        // layers below la pass, none from lb on passes, the float test says
                        // which of those between do: a toggle wherever that changes
                        bool pass = accepted;   // whether the layer before passes
                        for (int l = la; pass || l < lb;) {
                            int n = lb;         // the next change
                            for (; l < lb; ++l) {
                                const int k = (int)(((float)l + 0.5f) * inv_n2);
                                if (!((cb[c * nw + (k >> 6)] >> (k & 63)) & 1ull)) {
                                    l = (k + 1) * n2 - 1;   // no boundary voxel here
                                    continue;
                                }
                                if (mt_t_hit(a.x, a.y, a.z, a.w, b.x, b.y, b.z, tx, ty, f.w, rz[l]) != pass) {
                                    n = l++;
                                    break;
                                }
                            }
                            // (past lb with the last state `false`: nothing to toggle)
                            if (n == lb && !pass) break;
                            pass = !pass;
                            if (n > 0) {
                                // `n` layers pass: a toggle at layer n - 1 of its voxel, or at the
                                // top of the next boundary voxel below
                                const int k = (int)(((float)(n - 1) + 0.5f) * inv_n2);
                                const uint64_t bw = cb[c * nw + (k >> 6)];
                                const uint32_t upto =
                                    pre[c * nw + (k >> 6)] + (uint32_t)__popcll(bw & ((2ull << (k & 63)) - 1ull));
                                if (upto > clo && upto <= chi) {
                                    const int bit = ((bw >> (k & 63)) & 1ull) ? n - 1 - k * n2 : n2 - 1;
                                    uint32_t sh;
                                    const uint32_t wi = l2_col_word((upto - 1u - clo) * (uint32_t)nsc + sub, n2, sh);
                                    atomicXor(&L.acc[wi], 1u << (sh + bit));
                                }
                            }
                        }
                    }
                }
            }
        }
        l2_parity_barrier<V>();
        // toggles -> parities, from each column's top slot down
        const uint32_t layers = (1u << n2) - 1u;
        for (int it = tid; it < C * nsc; it += NT) {
            const int c = C == 1 ? 0 : it / nsc;
            const int sub = it - c * nsc;
            uint32_t n = hi[0] - lo[0];
#pragma unroll
            for (int k = 1; k < C; ++k) n = c == k ? hi[k] - lo[k] : n;
            const int r0 = c * (Wn + 1) * nsc + sub, top = r0 + Wn * nsc;
            uint32_t above = fb == 2 ? (uint32_t)a16[top] : (uint32_t)a8[top];
            for (int s = (int)n - 1; s >= 0; --s) {
                const int at = r0 + s * nsc;
                uint32_t x = fb == 2 ? (uint32_t)a16[at] : (uint32_t)a8[at];
                x ^= x >> 1;
                x ^= x >> 2;
                x ^= x >> 4;
                x ^= x >> 8;   // bit r: toggles at r and above
                const uint32_t y = x ^ (above ? layers : 0u);
                if (fb == 2) a16[at] = (uint16_t)y;
                else a8[at] = (uint8_t)y;
                above ^= x & 1u;
            }
            if (fb == 2) a16[top] = (uint16_t)above;
            else a8[top] = (uint8_t)above;
        }
        l2_parity_barrier<V>();
        // the slots' words
        if (C <= 2 && n2 == 8) {
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const int n = (int)(hi[c] - lo[c]);
                for (int v0 = wv * 8; v0 < n; v0 += 8 * V) {
                    // bit 8v + r of lane t: layer r of sub-column t of slot v0 + v
                    uint64_t x = 0;
                    for (int v = 0; v < 8 && v0 + v < n; ++v)
                        x |= (uint64_t)a8[(c * (Wn + 1) + v0 + v) * 64 + lane] << (8 * v);
                    x = wave_transpose64(x);
                    const int v = v0 + (lane >> 3);
                    if (v < n) out[(uint64_t)L.slotb[c * Wn + v] * 8 + (uint64_t)(lane & 7)] = x;
                }
            }
        } else if (C == 1 && n2 == 16) {
            const int n = (int)(hi[0] - lo[0]);
            for (int v = wv; v < n; v += V) {
                // bit 16k + r of lane c: layer r of sub-column 64k + c
                uint64_t x = 0;
                for (int k = 0; k < 4; ++k) x |= (uint64_t)a16[v * 256 + k * 64 + lane] << (16 * k);
                out[(uint64_t)L.slotb[v] * 64 + (uint64_t)(4 * (lane & 15) + (lane >> 4))] = wave_transpose64(x);
            }
        } else {
            const float inv = GPV_RCP((float)nsc);
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const int n = (int)(hi[c] - lo[c]);
                // lane t of a run of 64 keeps word t of the column's (slot, word) list
                for (int t0 = wv * 64; t0 < n * w2; t0 += NT) {
                    uint64_t mine = 0;
                    int v = t0 / w2, m = t0 - v * w2;
                    const int te = min(64, n * w2 - t0);
                    for (int t = 0; t < te; ++t) {
                        const int s = 64 * m + lane;
                        const int r = (int)(((float)s + 0.5f) * inv);   // exact: s + 1/2 is at least 1/512 of n2^2 from a multiple
                        const int at = (c * (Wn + 1) + v) * nsc + (s - r * nsc);
                        const uint32_t x = fb == 2 ? (uint32_t)a16[at] : (uint32_t)a8[at];
                        const uint64_t wd = __ballot(r < n2 && ((x >> r) & 1u));
                        if (lane == t) mine = wd;
                        if (++m == w2) {
                            m = 0;
                            ++v;
                        }
                    }
                    if (lane < te) {
                        const int v1 = (t0 + lane) / w2;
                        out[(uint64_t)L.slotb[c * Wn + v1] * (uint64_t)w2 + (uint64_t)(t0 + lane - v1 * w2)] = mine;
                    }
                }
            }
        }
        l2_parity_barrier<V>();
    }
}

// W waves a block: each with columns of its own (V = 1), or all with the same (V = W), those
// of H's list if there is one
template <bool kM, int KB, int W, int V, bool kFar>
__global__ __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(V > 1 || kFar ? 5 : W == 1 ? 6 : 3))) void k_l2_parity(const uint64_t* __restrict__ bnd,
                                                      const uint32_t* __restrict__ wprefix,
                                                      const uint64_t* __restrict__ occ, int64_t nwaves, bool many, int nw,
                                                      const uint32_t* __restrict__ coff,
                                                      const uint2* __restrict__ ent, const float* __restrict__ tris,
                                                      GridDev g0, Meshes M, L2Heavy H, uint64_t* __restrict__ par2)
{
    static_assert(V == 1 || V == W, "waves of a column");
    __shared__ L2PLds<KB, V> s_l[W / V];
    extern __shared__ uint64_t s_cb[];   // per group of waves: 4 * nw words of column bits, then 4 * nw counts
    const int wid = uniform_i((int)threadIdx.x >> 6), grp = V > 1 ? 0 : wid, wv = V > 1 ? wid : 0;
    // runs of 16 blocks (adjacent columns, which share boundary words) to one XCD
    uint32_t blk = blockIdx.x;
    if ((gridDim.x & 127u) == 0) blk = ((blk >> 7) << 7) + ((blk & 7u) << 4) + ((blk >> 3) & 15u);
    uint64_t* cb = s_cb + (size_t)grp * 6 * nw;
    const int64_t first = (int64_t)blk * (W / V) + grp;
    const bool listed = V > 1 && H.list;
    const int64_t n = listed ? min((int64_t)*H.count, H.most) : nwaves;
    for (int64_t at = first; at < n; at += listed ? (int64_t)gridDim.x : n) {   // one turn but for a list
        const int64_t wave = listed ? (int64_t)H.list[at] : at;
        int mesh = 0;
        if constexpr (kM)   // the mesh whose waves hold this one
            mesh = wave_mesh_search(M.off, M.nm, (uint64_t)wave, [](const MeshOff& o) { return (uint64_t)o.pw0; });
        const GridDev& g = grid_of<kM>(g0, M, mesh);
        if (kM && g.n2 == 0) continue;
        const int C = l2_parity_columns(g.n2, many);
        const int col = (int)(wave - (kM ? (int64_t)M.off[mesh].pw0 : 0)) * C;
        const int j1 = col / g.nx, i1 = col - j1 * g.nx;
        const uint64_t word0 = kM ? M.off[mesh].word0 : 0;
        const uint32_t col0 = kM ? M.off[mesh].col0 : 0, b0 = kM ? M.rank[mesh].b0 : 0;
        const uint32_t cw0 = kM ? M.off[mesh].cw0 : 0;
        uint64_t* out = par2 + (kM ? M.rank[mesh].l2w0 : 0);
        if (C == 2)
            l2_parity_columns_wave<2, KB, V, kFar>(s_l[grp], wv, (uint32_t)wave, H, cb, nw, g, i1, j1, word0, col0, b0, cw0, occ, bnd, wprefix, coff, ent, tris, out);
        else if (C == 4)
            l2_parity_columns_wave<4, KB, V, kFar>(s_l[grp], wv, (uint32_t)wave, H, cb, nw, g, i1, j1, word0, col0, b0, cw0, occ, bnd, wprefix, coff, ent, tris, out);
        else
            l2_parity_columns_wave<1, KB, V, kFar>(s_l[grp], wv, (uint32_t)wave, H, cb, nw, g, i1, j1, word0, col0, b0, cw0, occ, bnd, wprefix, coff, ent, tris, out);
    }
}

template <int KB, int W, int V = 1, bool kFar = false>
static void launch_l2_parity_w(const uint64_t* bnd, const uint32_t* wprefix, const uint64_t* occ, int64_t nwaves, bool many, int nzmax,
                               const uint32_t* coff, const uint2* ent, const float* tris, const GridDev& g0, const Meshes& M,
                               const L2Heavy& H, uint64_t* par2, hipStream_t s)
{
    constexpr int G = W / V;   // groups of waves a block
    // a list is mostly short or empty: no more blocks than the chip holds at once
    const int64_t n = V > 1 && H.list ? (H.most < 1536 ? H.most : 1536) : nwaves;
    unsigned blocks = (unsigned)((n + G - 1) / G);
    if (blocks >= 1024) blocks = (blocks + 127u) & ~127u;   // whole rounds of the XCD mapping
    const int nw = (nzmax + 63) / 64;
    const size_t lds = (size_t)G * 6 * nw * sizeof(uint64_t);
    if (M.nm > 1)
        k_l2_parity<true, KB, W, V, kFar><<<blocks, 64 * W, lds, s>>>(bnd, wprefix, occ, nwaves, many, nw, coff, ent, tris, g0, M, H, par2);
    else
        k_l2_parity<false, KB, W, V, kFar><<<blocks, 64 * W, lds, s>>>(bnd, wprefix, occ, nwaves, many, nw, coff, ent, tris, g0, M, H, par2);
}

template <int KB>
static void launch_l2_parity_k(const uint64_t* bnd, const uint32_t* wprefix, const uint64_t* occ, int64_t nwaves, bool many, int nzmax,
                               const uint32_t* coff, const uint2* ent, const float* tris, int waves, const GridDev& g0, const Meshes& M,
                               const L2Heavy& H, bool far, uint64_t* par2, hipStream_t s)
{
    if (far) launch_l2_parity_w<KB, 1, 1, true>(bnd, wprefix, occ, nwaves, many, nzmax, coff, ent, tris, g0, M, H, par2, s);
    else if (waves <= 1) launch_l2_parity_w<KB, 1>(bnd, wprefix, occ, nwaves, many, nzmax, coff, ent, tris, g0, M, H, par2, s);
    else if (waves == 2) launch_l2_parity_w<KB, 2>(bnd, wprefix, occ, nwaves, many, nzmax, coff, ent, tris, g0, M, H, par2, s);
    else launch_l2_parity_w<KB, 4>(bnd, wprefix, occ, nwaves, many, nzmax, coff, ent, tris, g0, M, H, par2, s);
}

void launch_l2_parity(const uint64_t* bnd, const uint32_t* wprefix, const uint64_t* occ, int64_t B, int64_t nwaves, bool many, int n2max, int nzmax,
                      const uint32_t* coff, const uint2* ent, const float* tris, int waves, const GridDev& g0, const Meshes& M,
                      const L2Heavy& H, bool far, uint64_t* par2, hipStream_t s)
{
    if (nwaves <= 0) return;
    // Up to 1,024 columns the chip holds four waves for each, with room for 128 boundary
    // voxels a window (31 at n2 = 16): a wave to a column left most of it idle, and every
    // window of a tall column stages all of its entries (rods of 12 x 12 columns: 512 layers at
    // n2 = 16 816 -> 338 us in all, 2,048 at 8 742 -> 720; 200,000 triangles at 8/16 772 -> 589; eight
    // waves the same or slower)
    auto share = [&](const L2Heavy& list) {
        if (far) launch_l2_parity_w<16384, L2P_SHARE, L2P_SHARE, true>(bnd, wprefix, occ, nwaves, many, nzmax, coff, ent, tris, g0, M, list, par2, s);
        else launch_l2_parity_w<16384, L2P_SHARE, L2P_SHARE>(bnd, wprefix, occ, nwaves, many, nzmax, coff, ent, tris, g0, M, list, par2, s);
    };
    // So they do where a column takes more than eight windows of a wave's own on average (rods of 1,200
    // columns and 4,096 layers at n2 = 16 3.75 -> 1.82 ms, 1,100 and 8,192 at 8 3.38 -> 1.99; 7,488
    // and 8,192 at 8, seven windows, 3.00 -> 3.35)
    const int64_t slot = (int64_t)n2max * n2max * (n2max > 8 ? 2 : 1);   // bytes of a boundary voxel
    if (nwaves <= 1024 || B * slot > 8 * (n2max <= 8 ? 2048 : 4096) * nwaves) {
        share(L2Heavy{});
        return;
    }
    // More columns: a wave takes its own, with room for 31 voxels at n2 = 8 and 7 at 16 (four
    // waves to each: lattice-snapped mesh at 512/16 1.8 -> 4.3 ms), but for those of many entries,
    // which would outlast all others: 2,000 overlapping triangles in a tenth of a 256/8 grid
    // 1.63 -> 0.54 ms, of a 512/16 one 8.1 -> 3.0
    if (n2max <= 8)
        launch_l2_parity_k<2048>(bnd, wprefix, occ, nwaves, many, nzmax, coff, ent, tris, waves, g0, M, H, far, par2, s);
    else
        launch_l2_parity_k<4096>(bnd, wprefix, occ, nwaves, many, nzmax, coff, ent, tris, waves, g0, M, H, far, par2, s);
    if (H.list) share(H);
}

// ---------------------------------------------------------------------------
// normals.  Face normal: side1 = v1 - v0, side2 = v2 - v0, their cross
// product, VectorNormalize (src/Object.cpp:3233-3240; the load-time
// faceNormal of :521-526 is the same float expression on the same points).
// VectorNormalize (includes/FloatVector.h:332-341) divides by the float
// magnitude of the left-to-right sum of squares when it is nonzero; sqrtf and
// the division are correctly rounded here.  The reference sums in bin order,
// which its CPU sweep makes ascending in triangle id, so bins are sorted
// before any sum.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void normalize3(float& x, float& y, float& z)
{
    const float m = sqrtf(x * x + y * y + z * z);
    if (m != 0.0f) {
        x = x / m;
        y = y / m;
        z = z / m;
    }
}

__global__ void k_face_normals(const float* __restrict__ tris, int64_t T, float* __restrict__ fn)
{
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < T; t += (int64_t)gridDim.x * blockDim.x) {
        const float* tv = tris + 9 * t;
        const float a0 = tv[3] - tv[0], a1 = tv[4] - tv[1], a2 = tv[5] - tv[2];
        const float b0 = tv[6] - tv[0], b1 = tv[7] - tv[1], b2 = tv[8] - tv[2];
        float x = a1 * b2 - b1 * a2;
        float y = a2 * b0 - b2 * a0;
        float z = a0 * b1 - b0 * a1;
        normalize3(x, y, z);
        fn[3 * t + 0] = x;
        fn[3 * t + 1] = y;
        fn[3 * t + 2] = z;
    }
}

void launch_face_normals(const float* tris, int64_t T, float* fn, hipStream_t s)
{
    if (T <= 0) return;
    k_face_normals<<<grid_for(T, 256, 16384), 256, 0, s>>>(tris, T, fn);
}

// true when boundary voxel b's mesh asks for normals (wave-uniform)
template <bool kM>
__device__ __forceinline__ bool wants_normals(const Meshes& M, int64_t b)
{
    if constexpr (kM) return M.grids[uniform_i((int)M.bmesh[b])].normals != 0;
    else return true;
}

// One wave per boundary voxel: the bin's triangle ids (distinct) ranked by
// counting smaller ids, written in ascending order to slist.
template <bool kM>
__global__ __launch_bounds__(256) void k_sort_bins(const uint32_t* __restrict__ list,
                                                   const uint32_t* __restrict__ boff, int64_t B, Meshes M,
                                                   uint32_t* __restrict__ slist)
{
    const int64_t b = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    if (b >= B || !wants_normals<kM>(M, b)) return;
    const int lane = __lane_id();
    const uint32_t e0 = boff[b], n = boff[b + 1] - e0;
    for (uint32_t bi = 0; bi < n; bi += 64) {
        const uint32_t ti = bi + lane < n ? list[e0 + bi + lane] : 0xffffffffu;
        uint32_t rank = 0;
        for (uint32_t bj = 0; bj < n; bj += 64) {
            const uint32_t tj = bj + lane < n ? list[e0 + bj + lane] : 0xffffffffu;
            const uint32_t m = n - bj < 64 ? n - bj : 64;
            for (uint32_t k = 0; k < m; ++k)
                rank += (uint32_t)((uint32_t)__builtin_amdgcn_readlane((int)tj, (int)k) < ti);
        }
        if (bi + lane < n) slist[e0 + rank] = ti;
    }
}

void launch_sort_bins(const uint32_t* list, const uint32_t* boff, int64_t B, const GridDev& g0, const Meshes& M,
                      uint32_t* slist, hipStream_t s)
{
    (void)g0;
    if (B <= 0) return;
    const unsigned blocks = (unsigned)((B * 64 + 255) / 256);
    if (M.nm > 1) k_sort_bins<true><<<blocks, 256, 0, s>>>(list, boff, B, M, slist);
    else k_sort_bins<false><<<blocks, 256, 0, s>>>(list, boff, B, M, slist);
}

// Level1 normal of a boundary voxel (src/Object.cpp:3219-3253): the face
// normals of its sorted bin summed in order, divided by the count, normalized.
template <bool kM>
__global__ __launch_bounds__(256) void k_l1_normals(const uint32_t* __restrict__ slist,
                                                    const uint32_t* __restrict__ boff, int64_t B,
                                                    const float* __restrict__ fn, Meshes M,
                                                    float* __restrict__ l1n)
{
    const int64_t b = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    if (b >= B || !wants_normals<kM>(M, b)) return;
    const int lane = __lane_id();
    const uint32_t e0 = boff[b], n = boff[b + 1] - e0;
    float sx = 0.0f, sy = 0.0f, sz = 0.0f;
    for (uint32_t bi = 0; bi < n; bi += 64) {
        float fx = 0.0f, fy = 0.0f, fz = 0.0f;
        if (bi + lane < n) {
            const uint64_t t = slist[e0 + bi + lane];
            fx = fn[3 * t];
            fy = fn[3 * t + 1];
            fz = fn[3 * t + 2];
        }
        const uint32_t m = n - bi < 64 ? n - bi : 64;
        for (uint32_t k = 0; k < m; ++k) {
            sx = sx + lane_f(fx, (int)k);
            sy = sy + lane_f(fy, (int)k);
            sz = sz + lane_f(fz, (int)k);
        }
    }
    const float cnt = (float)n;
    float x = sx / cnt, y = sy / cnt, z = sz / cnt;
    normalize3(x, y, z);
    if (lane == 0) {
        l1n[3 * b + 0] = x;
        l1n[3 * b + 1] = y;
        l1n[3 * b + 2] = z;
    }
}

void launch_l1_normals(const uint32_t* slist, const uint32_t* boff, int64_t B, const float* fn, const GridDev& g0,
                       const Meshes& M, float* l1n, hipStream_t s)
{
    (void)g0;
    if (B <= 0) return;
    const unsigned blocks = (unsigned)((B * 64 + 255) / 256);
    if (M.nm > 1) k_l1_normals<true><<<blocks, 256, 0, s>>>(slist, boff, B, fn, M, l1n);
    else k_l1_normals<false><<<blocks, 256, 0, s>>>(slist, boff, B, fn, M, l1n);
}

// Level2 normals (AddPointToVoxel src/Object.cpp:2705-2720 under the loop nest
// of :2372-2400, averaged at :2404-2421): per Level2 voxel, the face normals
// of the bin triangles whose SAT hits it, in bin order, over their count,
// normalized; (0, 0, 0) where none hits.  One wave per boundary voxel, each
// lane owning L2N_G Level2 voxels per pass; the box-axis predicates are
// evaluated once per (triangle, sub-index) by ballot, as in k_l2_sat.
constexpr int L2N_G = 8;

template <bool kM>
__global__ __launch_bounds__(256) void k_l2_normals(const float* __restrict__ tris,
                                                    const int32_t* __restrict__ bidx, int64_t B,
                                                    const uint32_t* __restrict__ boff,
                                                    const uint32_t* __restrict__ slist,
                                                    const float* __restrict__ fn, GridDev g0, Meshes M,
                                                    float* __restrict__ l2n)
{
    const int64_t b = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    if (b >= B) return;
    const int mesh = kM ? uniform_i((int)M.bmesh[b]) : 0;
    const GridDev& g = grid_of<kM>(g0, M, mesh);
    const int n2 = g.n2, gnx = g.nx, gny = g.ny;
    if (n2 == 0 || (kM && !g.normals)) return;
    const float h2x = g.h2x, h2y = g.h2y, h2z = g.h2z;
    const int S = n2 * n2 * n2;
    float* out = l2n + 3 * (kM ? M.rank[mesh].l2n0 + (uint64_t)(b - M.rank[mesh].b0) * S : (uint64_t)b * S);
    const int v = bidx[b];
    const int nxy = gnx * gny;
    const int k1 = v / nxy;
    const int ij = v - k1 * nxy;
    const int j1 = ij / gnx;
    const int i1 = ij - j1 * gnx;
    const float* c2x = g.c2x + (int64_t)i1 * n2;
    const float* c2y = g.c2y + (int64_t)j1 * n2;
    const float* c2z = g.c2z + (int64_t)k1 * n2;
    const int lane = __lane_id();
    const float cxl = lane < n2 ? c2x[lane] : 0.0f;
    const float cyl = lane < n2 ? c2y[lane] : 0.0f;
    const float czl = lane < n2 ? c2z[lane] : 0.0f;
    const uint32_t e0 = boff[b], n = boff[b + 1] - e0;
    for (int s0 = 0; s0 < S; s0 += 64 * L2N_G) {
        float ax[L2N_G], ay[L2N_G], az[L2N_G], ac[L2N_G];
        float ccx[L2N_G], ccy[L2N_G], ccz[L2N_G];
        int sp[L2N_G], sq[L2N_G], sr[L2N_G];
        // centers of this lane's Level2 voxels, gathered while every lane is active
#pragma unroll
        for (int k = 0; k < L2N_G; ++k) {
            const int sv = s0 + k * 64 + lane;
            ax[k] = ay[k] = az[k] = ac[k] = 0.0f;
            sp[k] = sv % n2;
            sq[k] = (sv / n2) % n2;
            sr[k] = (sv / (n2 * n2)) % n2;
            ccx[k] = __shfl(cxl, sp[k]);
            ccy[k] = __shfl(cyl, sq[k]);
            ccz[k] = __shfl(czl, sr[k]);
        }
        for (uint32_t e = 0; e < n; ++e) {
            const uint64_t t = slist[e0 + e];
            float tv[9];
#pragma unroll
            for (int c = 0; c < 9; ++c) tv[c] = tris[t * 9 + c];
            const uint64_t mx = __ballot(lane < n2 && sat_axis_ok(tv[0], tv[3], tv[6], cxl, h2x));
            const uint64_t my = __ballot(lane < n2 && sat_axis_ok(tv[1], tv[4], tv[7], cyl, h2y));
            const uint64_t mz = __ballot(lane < n2 && sat_axis_ok(tv[2], tv[5], tv[8], czl, h2z));
            if (!mx || !my || !mz) continue;
            const float fx = fn[3 * t], fy = fn[3 * t + 1], fz = fn[3 * t + 2];
#pragma unroll
            for (int k = 0; k < L2N_G; ++k) {
                const int sv = s0 + k * 64 + lane;
                if (sv >= S || !((mx >> sp[k]) & (my >> sq[k]) & (mz >> sr[k]) & 1ull)) continue;
                if (tri_box_overlap<false>(ccx[k], ccy[k], ccz[k], h2x, h2y, h2z, tv)) {
                    ax[k] = ax[k] + fx;
                    ay[k] = ay[k] + fy;
                    az[k] = az[k] + fz;
                    ac[k] = ac[k] + 1.0f;
                }
            }
        }
#pragma unroll
        for (int k = 0; k < L2N_G; ++k) {
            const int sv = s0 + k * 64 + lane;
            if (sv >= S) continue;
            float x = 0.0f, y = 0.0f, z = 0.0f;
            if (ac[k] > 0.0f) {
                x = ax[k] / ac[k];
                y = ay[k] / ac[k];
                z = az[k] / ac[k];
                normalize3(x, y, z);
            }
            out[3 * (int64_t)sv + 0] = x;
            out[3 * (int64_t)sv + 1] = y;
            out[3 * (int64_t)sv + 2] = z;
        }
    }
}

void launch_l2_normals(const float* tris, const int32_t* bidx, int64_t B, const uint32_t* boff,
                       const uint32_t* slist, const float* fn, const GridDev& g0, const Meshes& M, float* l2n,
                       hipStream_t s)
{
    if (B <= 0) return;
    const unsigned blocks = (unsigned)((B * 64 + 255) / 256);
    if (M.nm > 1) k_l2_normals<true><<<blocks, 256, 0, s>>>(tris, bidx, B, boff, slist, fn, g0, M, l2n);
    else k_l2_normals<false><<<blocks, 256, 0, s>>>(tris, bidx, B, boff, slist, fn, g0, M, l2n);
}

// .raw normal byte: outputDType(n * normScale + normBias), normScale =
// 256.0/3.0 and normBias = 127.0 as floats (src/Object.cpp:2940-2942, 3032-3034)
__device__ __forceinline__ uint8_t normal_byte(float v)
{
    const float y = v * 85.33333587646484375f;
    return (uint8_t)(int)(y + 127.0f);
}

// Level1Normal.raw: 3 bytes per Level1 voxel, [z][y][x]; only boundary voxels
// carry a normal, the rest are 0 -> 127
__global__ void k_export_l1_normals(const uint64_t* __restrict__ bnd, const uint32_t* __restrict__ wprefix,
                                    uint32_t base, const float* __restrict__ l1n, GridDev g, int64_t n1,
                                    uint8_t* __restrict__ out)
{
    for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < n1; v += (int64_t)gridDim.x * blockDim.x) {
        const int x = (int)(v % g.nx);
        const int64_t row = v / g.nx;
        const int64_t w = row * g.nxw + (x >> 6);
        float nx = 0.0f, ny = 0.0f, nz = 0.0f;
        if ((bnd[w] >> (x & 63)) & 1ull) {
            const uint64_t r = rank_of(bnd, wprefix, (uint64_t)w * 64 + (uint64_t)(x & 63)) - base;
            nx = l1n[3 * r];
            ny = l1n[3 * r + 1];
            nz = l1n[3 * r + 2];
        }
        out[3 * v + 0] = normal_byte(nx);
        out[3 * v + 1] = normal_byte(ny);
        out[3 * v + 2] = normal_byte(nz);
    }
}

void launch_export_l1_normals(const uint64_t* bnd, const uint32_t* wprefix, uint32_t base, const float* l1n,
                              const GridDev& g, uint8_t* out, hipStream_t s)
{
    const int64_t n1 = (int64_t)g.nx * g.ny * g.nz;
    if (n1 <= 0) return;
    k_export_l1_normals<<<grid_for(n1, 256, 65536), 256, 0, s>>>(bnd, wprefix, base, l1n, g, n1, out);
}

__global__ void k_export_l2_normals(const float* __restrict__ l2n, int64_t n, uint8_t* __restrict__ out)
{
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        out[i] = normal_byte(l2n[i]);
}

void launch_export_l2_normals(const float* l2n, int64_t n, uint8_t* out, hipStream_t s)
{
    if (n <= 0) return;
    k_export_l2_normals<<<grid_for(n, 256, 65536), 256, 0, s>>>(l2n, n, out);
}

// ---------------------------------------------------------------------------
// counts (src/Object.cpp:3353-3378)
// ---------------------------------------------------------------------------
// Single-mesh form: a grid-stride pass over both planes.  Multi-mesh form:
// blockIdx.y is the mesh, blockIdx.x strides over that mesh's words.
template <bool kM>
__global__ void k_count_states(const uint64_t* __restrict__ bnd, const uint64_t* __restrict__ ins, int64_t W,
                               const uint64_t* __restrict__ sat2, const uint64_t* __restrict__ par2,
                               int64_t W2, Meshes M, unsigned long long* __restrict__ done, uint64_t* __restrict__ pub)
{
    __shared__ uint32_t s_last;
    const int mesh = kM ? (int)blockIdx.y : 0;
    const uint64_t w_lo = kM ? M.off[mesh].word0 : 0, w_hi = kM ? M.off[mesh + 1].word0 : (uint64_t)W;
    const uint64_t l_lo = kM ? M.rank[mesh].l2w0 : 0, l_hi = kM ? M.rank[mesh + 1].l2w0 : (uint64_t)W2;
    uint64_t a = 0, b = 0, c = 0;
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = w_lo + (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < w_hi; i += stride)
        a += (uint64_t)__popcll(ins[i] & ~bnd[i]);
    // the Level2 planes four words per lane at a time, their loads issued
    // together (the blocks are few: they add into one counter each)
    constexpr int U = 4;
    uint64_t i = l_lo + (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i + (U - 1) * stride < l_hi; i += U * stride) {
        uint64_t p[U], q[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            p[u] = par2[i + u * stride];
            q[u] = sat2[i + u * stride];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            b += (uint64_t)__popcll(p[u] & ~q[u]);
            c += (uint64_t)__popcll(q[u]);
        }
    }
    for (; i < l_hi; i += stride) {
        b += (uint64_t)__popcll(par2[i] & ~sat2[i]);
        c += (uint64_t)__popcll(sat2[i]);
    }
    block_add_u64(a, &M.ctr[mesh].l1_inside);
    block_add_u64(b, &M.ctr[mesh].l2_inside);
    block_add_u64(c, &M.ctr[mesh].l2_boundary);
    if constexpr (kM) return;
    // the last block publishes the counters (a batch has thousands of blocks, at 3.7 ns
    // each on one counter: k_publish_meshes)
    if (threadIdx.x == 0) {
        wait_atomics();
        s_last = atomicAdd(done, 1ull) == (unsigned long long)gridDim.x * gridDim.y - 1ull ? 1u : 0u;
    }
    __syncthreads();
    if (!s_last) return;
    const uint64_t* ctr = reinterpret_cast<const uint64_t*>(M.ctr);
    for (int k = threadIdx.x; k < (int)(sizeof(MeshCtr) / 8); k += blockDim.x)
        publish(pub + k, __hip_atomic_load(ctr + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}

__global__ __launch_bounds__(256) void k_publish_meshes(const uint64_t* __restrict__ ctr, int n, uint64_t* __restrict__ pub)
{
    for (int k = (int)(blockIdx.x * blockDim.x + threadIdx.x); k < n; k += (int)(gridDim.x * blockDim.x)) publish(pub + k, ctr[k]);
}

void launch_count_states(const uint64_t* bnd, const uint64_t* ins, int64_t W, const uint64_t* sat2,
                         const uint64_t* par2, int64_t W2, const Meshes& M, unsigned long long* done, uint64_t* pub,
                         hipStream_t s)
{
    static_assert(sizeof(MeshCtr) % 8 == 0, "published by words");
    const int64_t n = W > W2 ? W : W2;
    if (M.nm > 1) {
        const int64_t per = (n + M.nm - 1) / M.nm;
        const dim3 grid((unsigned)grid_for(per, 256, 64), (unsigned)M.nm);
        k_count_states<true><<<grid, 256, 0, s>>>(bnd, ins, W, sat2, par2, W2, M, done, pub);
        const int words = M.nm * (int)(sizeof(MeshCtr) / 8);
        k_publish_meshes<<<grid_for(words, 256, 64), 256, 0, s>>>(reinterpret_cast<const uint64_t*>(M.ctr), words, pub);
    } else {
        k_count_states<false><<<grid_for(n, 256, 512), 256, 0, s>>>(bnd, ins, W, sat2, par2, W2, M, done, pub);
    }
}

// ---------------------------------------------------------------------------
// device memory -> page-locked host memory, a row of blocks per piece: 16 bytes a
// lane where the source allows it, bytes otherwise (and for the rest)
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_copy_out(CopyOut L)
{
    const char* src = L.src[0];
    char* dst = L.dst[0];
    int64_t n = L.n[0];
#pragma unroll
    for (int k = 1; k < kCopyMax; ++k)
        if ((int)blockIdx.y == k) {
            src = L.src[k];
            dst = L.dst[k];
            n = L.n[k];
        }
    const int64_t i0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, stride = (int64_t)gridDim.x * blockDim.x;
    const int64_t wide = (reinterpret_cast<uintptr_t>(src) | reinterpret_cast<uintptr_t>(dst)) & 15 ? 0 : n / 16;
    for (int64_t i = i0; i < wide; i += stride) reinterpret_cast<uint4*>(dst)[i] = reinterpret_cast<const uint4*>(src)[i];
    for (int64_t i = wide * 16 + i0; i < n; i += stride) dst[i] = src[i];
}

void launch_copy_out(const CopyOut& L, int pieces, hipStream_t s)
{
    int64_t most = 0;
    for (int k = 0; k < pieces; ++k) most = L.n[k] > most ? L.n[k] : most;
    if (pieces <= 0 || most <= 0) return;
    k_copy_out<<<dim3((unsigned)grid_for((most + 15) / 16, 256, 256), (unsigned)pieces), 256, 0, s>>>(L);
}

// ---------------------------------------------------------------------------
// egress: one byte per voxel holding state * unit (unit 1: the 0/1/2 states;
// unit 127: the .raw bytes uint8(state * 127.0f), src/Object.cpp:3024-3063)
// and the int32 exclusive boundary prefix per Level1 voxel
// ---------------------------------------------------------------------------
__global__ void k_export_l1(const uint64_t* __restrict__ bnd, const uint64_t* __restrict__ ins, GridDev g,
                            int64_t n1, uint8_t unit, uint8_t* __restrict__ out)
{
    for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < n1; v += (int64_t)gridDim.x * blockDim.x) {
        const int x = (int)(v % g.nx);
        const int64_t row = v / g.nx;
        const int64_t w = row * g.nxw + (x >> 6);
        const uint64_t bit = 1ull << (x & 63);
        out[v] = (bnd[w] & bit) ? (uint8_t)(2 * unit) : ((ins[w] & bit) ? unit : (uint8_t)0);
    }
}

void launch_export_l1(const uint64_t* bnd, const uint64_t* ins, const GridDev& g, uint8_t unit, uint8_t* out,
                      hipStream_t s)
{
    const int64_t n1 = (int64_t)g.nx * g.ny * g.nz;
    if (n1 <= 0) return;
    k_export_l1<<<grid_for(n1, 256, 65536), 256, 0, s>>>(bnd, ins, g, n1, unit, out);
}

__global__ void k_export_prefix(const uint64_t* __restrict__ bnd, const uint32_t* __restrict__ wprefix,
                                uint32_t base, GridDev g, int64_t n1, int32_t* __restrict__ out)
{
    for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < n1; v += (int64_t)gridDim.x * blockDim.x) {
        const int x = (int)(v % g.nx);
        const int64_t row = v / g.nx;
        const uint64_t bitidx = (uint64_t)(row * g.nxw + (x >> 6)) * 64 + (uint64_t)(x & 63);
        out[v] = (int32_t)(rank_of(bnd, wprefix, bitidx) - base);
    }
}

void launch_export_prefix(const uint64_t* bnd, const uint32_t* wprefix, uint32_t base, const GridDev& g,
                          int32_t* out, hipStream_t s)
{
    const int64_t n1 = (int64_t)g.nx * g.ny * g.nz;
    if (n1 <= 0) return;
    k_export_prefix<<<grid_for(n1, 256, 65536), 256, 0, s>>>(bnd, wprefix, base, g, n1, out);
}

__global__ void k_export_l2(const uint64_t* __restrict__ sat2, const uint64_t* __restrict__ par2, int64_t B,
                            int n23, int w2, uint8_t unit, uint8_t* __restrict__ out)
{
    const int64_t n = B * n23;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t b = i / n23;
        const int s = (int)(i - b * n23);
        const int64_t w = b * w2 + (s >> 6);
        const uint64_t bit = 1ull << (s & 63);
        out[i] = (sat2[w] & bit) ? (uint8_t)(2 * unit) : ((par2[w] & bit) ? unit : (uint8_t)0);
    }
}

void launch_export_l2(const uint64_t* sat2, const uint64_t* par2, int64_t B, const GridDev& g, uint8_t unit,
                      uint8_t* out, hipStream_t s)
{
    const int n23 = g.n2 * g.n2 * g.n2;
    if (B <= 0 || n23 <= 0) return;
    k_export_l2<<<grid_for(B * n23, 256, 65536), 256, 0, s>>>(sat2, par2, B, n23, g.w2, unit, out);
}

}  // namespace gpv
