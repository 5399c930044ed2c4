// gpv_internal.hpp -- shared host/device declarations of libgpv (not public).
#pragma once

#include "gpv.h"

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace gpv {

// Grid constants and per-axis center tables of one mesh.
// Bit layout of every Level1 bitplane: word w = (z*ny + y)*nxw + x/64,
// bit x%64 (rows padded to whole 64-bit words), so words are in the
// reference's linear order z*ny*nx + y*nx + x and a boundary rank is a
// popcount prefix.  Level2: w2 = ceil(n2^3/64) words per boundary voxel,
// bit s = (r*n2 + q)*n2 + p inside the block ([b][r][q][p] order).
struct GridDev {
    int nx, ny, nz, nxw;
    int n2, w2;
    int normals;           // this mesh asks for Level1/Level2 normals
    int l2cuda;            // Level2 in the reference's CUDA arithmetic (gpv_params::cuda_level2)
    int l1st;              // Level1 inside/outside by the GL-stencil-equivalent fill (gpv_params::l1_stencil)
    float bminx, bminy, bminz, bmaxx, bmaxy, bmaxz;
    float g1x, g1y, g1z, g2x, g2y, g2z;   // voxel sizes of both levels
    float h1x, h1y, h1z;   // Level1 half extents
    float h2x, h2y, h2z;   // Level2 half extents
    float s1x, s1y, s1z, d1x, d1y, d1z;   // Level1 SAT columns: scale and table deviation per axis (SatScale)
    float s2x, s2y, s2z, d2x, d2y, d2z;   // Level2 SAT rows: scale and table deviation per axis (SatScale)
    const float* c1x; const float* c1y; const float* c1z;   // [n]    Level1 SAT centers
    const float* r1x; const float* r1y; const float* r1z;   // [n]    Level1 ray origins
    const float* c2x; const float* c2y; const float* c2z;   // [n*n2] Level2 SAT centers
    const float* r2x; const float* r2y; const float* r2z;   // [n*n2] Level2 ray origins
};

// Floats of a mesh's center tables: [SAT centers x, y, z | ray origins x, y, z] of
// Level1 (n each), then of Level2 (n * n2 each).
__host__ __device__ inline int64_t table_floats(const GridDev& g)
{
    return 2 * ((int64_t)g.nx + g.ny + g.nz) * (1 + (g.n2 > 0 ? g.n2 : 0));
}

// Entry k of a center table along one axis (which: 0 Level1 SAT, 1 Level1 ray, 2
// Level2 SAT, 3 Level2 ray), with the reference's float and double expressions
// (src/Object.cpp:2329-2331, 743-745, 2369-2391, 1134-1160).  Additions and products
// only (halving is exact) and no contraction, so host and device agree to the bit.
__host__ __device__ inline float center_at(int which, int k, float bmin, float g1, float g2, int n2, bool cuda_l2)
{
    const float ext1 = (float)((double)g1 / 2.0);
    if (which == 0) return (float)((k + 0.5) * (double)ext1 * 2 + (double)bmin);
    if (which == 1) return (float)((double)bmin + (k + 0.5) * (double)g1);
    const int i = k / n2, p = k - i * n2;
    const float mid = (float)((i + 0.5) * (double)g1 + (double)bmin);
    if (cuda_l2) {
        const float ext2 = (float)((double)g2 / 2.0);
        const float two_p1 = (float)(2 * p + 1);
        const float prod = two_p1 * ext2;
        const float sum = prod + mid;
        return sum - ext1;
    }
    if (which == 2) return (float)((p + 0.5) * (double)g2 + (double)mid - (double)ext1);
    const float minp = (float)i * g1 + bmin;
    return (float)((double)minp + (p + 0.5) * (double)g2);
}

// From an eighth of a sub-voxel of table deviation on (SatScale), Level2 positions are taken
// from the tables themselves (gpv_satrow.hpp, gpv_parcol.hpp), so that a grid's distance from the
// origin no longer costs float tests: 60,000 triangles at 128/16, deviations 0.09, 0.29, 0.86, 2.9
// and 29: by the tables 548, 593, 625, 703 and 1168 us in all, by equal steps 488, 700, 1461, 7359 and
// more than 12,000; at 128/8, 0.14: 336 and 327.
constexpr float kFarDev = 0x1p-3f;

inline bool level2_far(const GridDev& g)
{
    const float d = g.d2x > g.d2y ? g.d2x : g.d2y;
    return g.n2 > 0 && (d > g.d2z ? d : g.d2z) > kFarDev;
}

// Where one mesh of a batch lives in the batch-wide arrays.  A batch
// concatenates the meshes' soups (tri0), Level1 bitplanes (word0) and xy
// columns (col0); entry nm is the sentinel holding the totals.  Set when the run is
// created and never written again: kernels on both streams read it.
struct MeshOff {
    uint64_t word0;
    uint32_t col0;
    uint32_t tri0;
    uint32_t ptask0;   // first Level1 fill block (L1F_W words of a layer)
    uint32_t pw0;      // first Level2 parity wave
    uint32_t cw0;      // first word of the columns' occupancy (a bit per column, rows padded to words)
    uint32_t pad;
};

// The same for what follows from the boundary scan, a table of its own because the
// main stream writes it while the Level1 parity runs on the other one.
struct MeshRank {
    uint64_t l2w0;
    uint64_t l2n0;   // first Level2 normal (one per Level2 voxel of meshes with normals)
    uint32_t b0;
    uint32_t sg0;    // first Level2 SAT group (k_mesh_groups)
};

// Per-mesh results accumulated on the device.
struct MeshCtr {
    unsigned long long tests_l1;      // sum of clipped index-AABB volumes
    unsigned long long l1_inside;
    unsigned long long l2_inside;
    unsigned long long l2_boundary;
    unsigned long long pairs;         // Level1 (voxel, triangle) bin entries
    unsigned int max_per_voxel;
    unsigned int pad;
};

// A batch as kernels see it.  With nm == 1 kernels run their single-mesh
// instantiation: the grid comes from the by-value GridDev, every offset is
// 0 and only ctr is used.
struct Meshes {
    const GridDev* grids;       // [nm]
    const MeshOff* off;         // [nm + 1]
    MeshRank* rank;             // [nm + 1]
    const uint32_t* tri_mesh;   // [T]  mesh of each triangle (non-decreasing)
    uint32_t* bmesh;            // [B]  mesh of each boundary voxel (non-decreasing)
    MeshCtr* ctr;               // [nm]
    int nm;
};

// Append-buffer descriptor: a device counter and a capacity.  Writers past
// the capacity are dropped; the host sees count > cap and regrows.
struct Append64 {
    unsigned long long* count;
    uint64_t* key;
    uint32_t* val;     // optional payload (nullptr if none)
    uint64_t cap;
};

// Device-side counters of one pipeline run (batch-wide).
struct Counters {
    unsigned long long pairs;       // Level1 SAT (voxel, triangle) pairs
    unsigned long long colents;     // (column, triangle, zmax) entries
    unsigned long long bad_input;   // nonzero: a vertex coordinate is not finite or beyond +-2^40
    unsigned long long done;        // blocks of the state counts that are through
};
// page-locked read-back, written by kernels: Counters | B (one mesh) or MeshRank[nm + 1] | MeshCtr[nm]
constexpr size_t kHOff = 64;

// Launch shapes of a new context, and what the autotuner tries of each field: the
// default and values around it, so that it finds its way back from any start.  Group
// thresholds count bin entries a voxel; 0 and 2^20 are never and always.
constexpr gpv_tune kTuneDefault{16, 56, 2048, 1, 1, 1, 128};
struct TuneField {
    int gpv_tune::*field;
    int n, values[6];
};
constexpr TuneField kTuneSweep[] = {
    {&gpv_tune::expand_blocks_per_cu, 4, {4, 8, 16, 32}},
    {&gpv_tune::l2_group_below, 6, {0, 14, 28, 56, 112, 1 << 20}},
    {&gpv_tune::sort_items_per_block, 4, {1024, 2048, 4096, 8192}},
    {&gpv_tune::l2_overlap, 2, {0, 1}},
    {&gpv_tune::l2_sat_waves, 3, {1, 2, 4}},
    {&gpv_tune::l2_parity_waves, 3, {1, 2, 4}},
};

// sets the calling thread's gpv_last_error text and returns code
int set_error(int code, const char* msg);
// restarts the context pool's peak of bytes in use from the bytes in use now
void pool_reset_peak(gpv_ctx* c);

// ---- launch wrappers (gpv_kernels.hip) ------------------------------------
// Launchers that take the batch view M and a grid g0 run the single-mesh
// instantiation (grid g0) when M.nm == 1, the multi-mesh one otherwise.
// up to kClearMax regions, their sizes in words of 8 bytes in `end`
constexpr int kClearMax = 5;
struct ClearList {
    uint64_t* p[kClearMax];
    int64_t end[kClearMax];
};
// clears them and, unless nullptr, makes one mesh's center tables
void launch_clear(ClearList L, const GridDev* tables, hipStream_t s);
// the center tables of a batch
void launch_tables(const Meshes& M, hipStream_t s);
void launch_fill_u32(uint32_t* p, uint32_t v, int64_t n, hipStream_t s);
void launch_fill_u64(uint64_t* p, uint64_t v, int64_t n, hipStream_t s);

void launch_mesh_ids(const MeshOff* off, int nm, int64_t T, uint32_t* tri_mesh, hipStream_t s);
// part 1 (and 3) also raise *bad_input for a coordinate outside the domain;
// *_sums[k]: the items of triangles [256 k, 256 k + 256)
void launch_tri_setup(const float* tris, int64_t T, const GridDev& g0, const Meshes& M, int4* box0, int4* box1,
                      uint32_t* sat_items, int4* ray_rng, uint32_t* ray_items, uint64_t* sat_sums,
                      uint64_t* ray_sums, int part,
                      unsigned long long* bad_input, hipStream_t s);

// exclusive scan of n u32 into out[0..n] (out[n] = total); tmp sized by
// scan_tmp_elems(n).  If max_out != nullptr the max input is atomically
// folded into it.
size_t scan_tmp_elems(int64_t n);
void launch_scan_u32_u64(const uint32_t* in, uint64_t* out, int64_t n, uint64_t* tmp, hipStream_t s);
void launch_scan_u32_u32(const uint32_t* in, uint32_t* out, int64_t n, uint32_t* tmp, unsigned int* max_out,
                         hipStream_t s);
// item offsets of T triangles from launch_tri_setup's counts and sums; a
// second set (in2, or nullptr) in the same launch
void launch_scan_items(const uint32_t* in, uint64_t* out, const uint64_t* sums, const uint32_t* in2, uint64_t* out2,
                       const uint64_t* sums2, int64_t T, uint64_t* tmp, hipStream_t s);
// word prefix from launch_pack_bytes's counts and sums (pack_sums(W) of them); pub
// (or nullptr): the counters and the total go to the page-locked read-back
size_t pack_sums(int64_t W);
void launch_scan_words(const uint32_t* in, uint32_t* out, int64_t W, const uint32_t* sums, const Counters* ctr,
                       uint64_t* pub, uint32_t* tmp, hipStream_t s);

void launch_sat_expand(const float* tris, int64_t T, const int4* box0, const int4* box1, const uint64_t* off,
                       const GridDev& g0, const Meshes& M, uint8_t* bbytes, Append64 pairs, Append64 cols, int blocks,
                       hipStream_t s);
// boundary bytes (W * 64, aligned to 16) -> boundary bitplane (W words) and its popcounts
void launch_pack_bytes(const uint8_t* by, int64_t W, uint64_t* bits, uint32_t* cnt, uint32_t* sums, hipStream_t s);
// XORs the toggles of the accepted ray crossings into the inside plane (cleared by the caller)
void launch_ray_expand(const float* tris, int64_t T, const int4* ray_rng, const uint64_t* off, const GridDev& g0,
                       const Meshes& M, uint64_t* ins, int blocks, hipStream_t s);

// Two-level counting sort: tiles of 2^8 to 2^13 keys, at most 8192 tiles below 2^26
// keys and 16384 at 2^27.  The count and bucket passes hold a counter per
// tile in every block's LDS (32 KiB at 8192 tiles: five blocks per CU, where 16384
// tiles allowed two), the place pass one per key of its tile (at most 32 KiB).
constexpr int ts_shift(uint64_t nkeys)
{
    int lg = 0;
    while ((1ull << lg) < nkeys) ++lg;
    const int sh = lg - 13;
    return sh < 8 ? 8 : sh > 13 ? 13 : sh;
}
constexpr size_t ts_tiles(uint64_t nkeys)
{
    const int shift = ts_shift(nkeys);
    return (size_t)((nkeys + (1u << shift) - 1) >> shift);
}
// The scan over a sort's tiles by one block lies in LDS, tile t at word t + (t >>
// ts_pad): up to 8192 tiles a word in 33 is left out so that the threads' runs start in
// different banks; more fill 64 KiB as they are.
__host__ __device__ constexpr int ts_pad(int ntiles) { return ntiles <= 8192 ? 5 : 31; }
__host__ __device__ constexpr size_t ts_scan_words(int ntiles) { return (size_t)ntiles + (size_t)(ntiles >> ts_pad(ntiles)); }
// LDS words of a launch whose blocks scan one of two sorts' tiles each.  More tiles can
// take fewer words (8193 with 8192), so the larger need counts, not the larger sort.
constexpr size_t ts_scan_lds(int a, int b)
{
    return ts_scan_words(a) > ts_scan_words(b) ? ts_scan_words(a) : ts_scan_words(b);
}
// words of scratch of a sort with at most nkeys keys, zeros at its start
size_t ts_words(uint64_t nkeys);

// bin pairs (key = batch-wide boundary bit index, triangle) -> CSR by boundary rank
// (off[B + 1], list); B <= 2^27.  The pairs' voxel bits are replaced by their
// boundary ranks (ranked: they hold ranks already); max_out (or nullptr): the largest bin
struct BinPairs {
    uint64_t* bits;
    bool ranked;
    const uint32_t* tri;
    uint64_t n;
    uint32_t B;
    uint32_t* cnt;   // [ts_words(B)]
    void* bucket;    // 8 bytes a pair
    uint32_t* off;
    unsigned int* max_out;
    uint32_t* list;
};
// column entries (key = column << 32 | triangle) -> CSR by column of (triangle,
// zmax); ncol <= 2^27, 0: none
struct BinCols {
    const uint64_t* key;
    const uint32_t* zmax;
    uint64_t n;
    uint32_t ncol;
    uint32_t* cnt;   // [ts_words(ncol)]
    void* bucket;    // 12 bytes an entry
    uint32_t* off;
    uint2* ent;
};
// both sorts, the boundary index list and (unless nullptr) the bits of the columns that
// hold boundary voxels, in occ (cleared by the caller)
void launch_bins(const BinPairs& P, const BinCols& C, const uint64_t* bnd, const uint32_t* wprefix, const GridDev& g0,
                 const Meshes& M, int64_t W, int32_t* bidx, uint64_t* occ, int items_per_block, hipStream_t s);

// Level2 SAT voxel groups (k_l2_sat): consecutive boundary voxels of a mesh
// that share a wave, at most `most` and kL2GroupMax of them, their layer bits
// (a byte per sub-column, two above n2 = 8) within kL2GroupBytes of LDS
constexpr int kL2GroupMax = 16;
constexpr int kL2GroupBytes = 1024;
__host__ __device__ inline int l2_group_voxels(int n2, int most)
{
    int c = n2 > 0 ? kL2GroupBytes / (n2 * n2 * (n2 > 8 ? 2 : 1)) : kL2GroupMax;
    if (c > kL2GroupMax) c = kL2GroupMax;
    return c < most ? c : most;
}
// groups of a mesh with nb boundary voxels
__host__ __device__ inline int64_t l2_groups(int n2, int64_t nb, int most)
{
    if (n2 <= 0) return 0;
    const int64_t c = l2_group_voxels(n2, most);
    return (nb + c - 1) / c;
}
// Level1 fill: a block takes L1F_W words of a mesh's layer, all layers
constexpr int L1F_W = 16;
inline int64_t l1_fill_blocks(const GridDev& g) { return ((int64_t)g.ny * g.nxw + L1F_W - 1) / L1F_W; }
// one mesh's soup (n floats, device memory or page-locked host memory mapped
// into the device's address space) and its place in the batch's soup
struct SoupPiece {
    const float* src;
    uint64_t at;
    uint64_t n;
};
void launch_gather_soups(const SoupPiece* pc, int nm, float* dst, int blocks, bool host, hipStream_t s);

// GL-stencil-equivalent Level1 fill of one mesh (soup tris[T], grid g):
// overwrites the mesh's Level1 inside bits ins[nz*ny*nxw].  Scratch: cnt[T],
// off[T+1], scan_tmp[scan_tmp_elems(T)], tog[l1_stencil_words(g)].
size_t l1_stencil_words(const GridDev& g);
void launch_l1_stencil(const float* tris, int64_t T, const GridDev& g, uint32_t* cnt, uint64_t* off,
                       uint64_t* scan_tmp, uint64_t* tog, uint64_t* ins, hipStream_t s);
// toggles -> inside bits, in place, but for the stencil meshes; blocks: l1_fill_blocks of all meshes
void launch_l1_fill(const GridDev& g0, const Meshes& M, int64_t blocks, uint64_t* ins, hipStream_t s);

// b0, l2w0 and l2n0 of every mesh (and the totals in entry nm) from the word prefix
// and the counters, to the page-locked read-back pub as well
void launch_mesh_bounds(const uint32_t* wprefix, const Meshes& M, const Counters* ctr, uint64_t* pub, hipStream_t s);
// sg0 of every mesh (and the total in entry nm) from b0
void launch_mesh_groups(const Meshes& M, int most, hipStream_t s);
// per-mesh bin totals and largest bin (multi-mesh runs)
void launch_mesh_bins(const uint32_t* boff, int64_t B, const Meshes& M, hipStream_t s);

// ngroups waves of at most gmost voxels each (l2_group_voxels); waves: per block (1, 2, 4)
void launch_l2_sat(const float* tris, const int32_t* bidx, int64_t B, int64_t ngroups, int gmost, const uint32_t* boff,
                   const uint32_t* list, int n2max, bool far, int waves, const GridDev& g0, const Meshes& M,
                   uint64_t* sat2, hipStream_t s);
// Level2 parity: a wave takes l2_parity_columns adjacent columns of a mesh
// (grids are multiples of four in x): four at n2 <= 4, two up to 8, in runs of at least
// kL2ParityMany columns, where the shared prologue and fuller rounds pay (128 small meshes
// at 64/4 0.39 ms with four; 48 mixed ones 6.09 -> 5.90 ms in all with two at n2 = 8),
// one in smaller runs, where the longest wave counts (icosphere 64/4: 24
// us with four)
constexpr int64_t kL2ParityMany = 1 << 16;
__host__ __device__ inline int l2_parity_columns(int n2, bool many) { return !many || n2 > 8 ? 1 : n2 <= 4 ? 4 : 2; }
// its waves for a mesh with ncol columns (none when Level2 is off)
int64_t l2_parity_waves(int n2, int64_t ncol, bool many);
// Waves whose columns hold more than `above` entries each leave them to a second launch,
// where several waves share them: a count (zero at the start) and room for `most` of them
struct L2Heavy {
    uint32_t* count;
    uint32_t* list;   // nullptr: no second launch
    uint32_t above;
    int64_t most;
};
// More than 128 (256: 4.4 ms in place of 2.9 where 2,000 triangles overlap in a tenth of a
// 512/16 grid) and than four times what the run's columns hold on average: columns that are
// all alike are better taken by a wave each (400,000 triangles at 64/4 268 -> 302 us in all with
// 128 alone).  Below 16,384 waves no column outlasts the others by enough to pay for the
// launch (most = 0).
inline L2Heavy l2_heavy(uint64_t ncols, int64_t ncol, int64_t nwaves)
{
    const uint64_t mean = ncols / (uint64_t)(ncol > 0 ? ncol : 1);
    const uint64_t above = 4 * mean > 128 ? 4 * mean : 128;
    return L2Heavy{nullptr, nullptr, (uint32_t)above, nwaves < 16384 ? 0 : (int64_t)(ncols / (above + 1))};
}
// B boundary voxels; n2max, nzmax: the largest Level2 resolution and layer count of the run; occ: the
// columns that hold boundary voxels (or nullptr)
void launch_l2_parity(const uint64_t* bnd, const uint32_t* wprefix, const uint64_t* occ, int64_t B, int64_t nwaves, bool many,
                      int n2max, int nzmax, const uint32_t* coff, const uint2* ent, const float* tris, int waves,
                      const GridDev& g0, const Meshes& M, const L2Heavy& H, bool far, uint64_t* par2, hipStream_t s);

// normals (src/Object.cpp:3219-3253 Level1, 2372-2421 + 2705-2720 Level2)
void launch_face_normals(const float* tris, int64_t T, float* fn, hipStream_t s);
void launch_sort_bins(const uint32_t* list, const uint32_t* boff, int64_t B, const GridDev& g0, const Meshes& M,
                      uint32_t* slist, hipStream_t s);
void launch_l1_normals(const uint32_t* slist, const uint32_t* boff, int64_t B, const float* fn, const GridDev& g0,
                       const Meshes& M, float* l1n, hipStream_t s);
void launch_l2_normals(const float* tris, const int32_t* bidx, int64_t B, const uint32_t* boff,
                       const uint32_t* slist, const float* fn, const GridDev& g0, const Meshes& M, float* l2n,
                       hipStream_t s);
void launch_export_l1_normals(const uint64_t* bnd, const uint32_t* wprefix, uint32_t base, const float* l1n,
                              const GridDev& g, uint8_t* out, hipStream_t s);
void launch_export_l2_normals(const float* l2n, int64_t n, uint8_t* out, hipStream_t s);

// counts the states (done: a zero counter) and publishes the meshes' counters to pub
void launch_count_states(const uint64_t* bnd, const uint64_t* ins, int64_t W, const uint64_t* sat2,
                         const uint64_t* par2, int64_t W2, const Meshes& M, unsigned long long* done, uint64_t* pub,
                         hipStream_t s);

// up to kCopyMax pieces of device memory and their places in page-locked host memory
constexpr int kCopyMax = 4;
struct CopyOut {
    const char* src[kCopyMax];
    char* dst[kCopyMax];
    int64_t n[kCopyMax];
};
void launch_copy_out(const CopyOut& L, int pieces, hipStream_t s);

// egress of one mesh (pointers already offset to that mesh's words)
void launch_export_l1(const uint64_t* bnd, const uint64_t* ins, const GridDev& g, uint8_t unit, uint8_t* out,
                      hipStream_t s);
void launch_export_prefix(const uint64_t* bnd, const uint32_t* wprefix, uint32_t base, const GridDev& g,
                          int32_t* out, hipStream_t s);
void launch_export_l2(const uint64_t* sat2, const uint64_t* par2, int64_t B, const GridDev& g, uint8_t unit,
                      uint8_t* out, hipStream_t s);

}  // namespace gpv
