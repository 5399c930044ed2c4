// gpv_parcol.hpp -- the ray parities by crossings instead of voxel by voxel.
//
// For the +z ray of a sub-column (x, y) the Moller-Trumbore test of one column
// entry (triangle) accepts or rejects by det/u/v, which do not depend on the
// origin's z, and then passes where t >= eps (src/TriRayIntersection.cpp:
// 78-131).  In exact arithmetic t falls with the origin's height, so the
// sub-layers that pass are those below one crossing height; the parity of
// every voxel of the column follows from the crossings.  The float test is
// within rounding of that: functions here bound which sub-columns it can
// accept and below and above which layers it is certain to pass or fail; the
// kernel runs the reference's float expressions on the rest.
//
// U = 2^-24.  e1, e2 are the record's float edges, inv = fl(1/det),
// N_a = |e1_b e2_c| + |e1_c e2_b|, T = o - v1.
//
// Acceptance.  u = fl((Tx px + Ty py) inv) and v likewise lie within
//   delta = 64 U (1 + |inv| ((|e1y| + |e2y|) tmx + (|e1x| + |e2x|) tmy + N_z))
// of the barycentric coordinates a, b of the ray's point with respect to the
// float edges (3 U per numerator, |inv| N_z 3 U and 2 U for the reciprocal, one
// product; tm bounds |T| over the column), and the formulas below within half of
// that of a, b.  So an accepted sub-column satisfies a, b >= -delta,
// a + b <= 1 + 2 delta; delta also carries the deviation of the origin tables from
// equal steps (SatScale).
//
// Crossing.  The float s = e2 . (T x e1) is within 6.1 U B of the exact one, B =
// sum |T_a| N_a, and t >= eps means s >= eps |det| up to 2 U and the det's own 2.1 U N_z; |T_a| <=
// 2 (|e1_a| + |e2_a|) for an accepted ray at its crossing where 64 U N_z <=
// |det|.  The crossing height taken here, v1z + u e1z + v e2z - eps, is off by at
// most 3 U |inv| (|Tx| N_x + |Ty| N_y + N_z (|e1z| + |e2z|)) and rounding.  So the
// float test agrees with the crossing at every height farther from it than
//   Ez = 64 U |inv| sum (|e1_a| + |e2_a|) N_a + 16 U (|e1z| + |e2z|) + (2^-12 + 4 U N_z |inv|) eps
// (|det| >= 1e-6 by the det test); worse conditioned records get Ez infinite.
#pragma once

#include "gpv_satrow.hpp"

namespace gpv {

// Ez of a record (z units)
__host__ __device__ __forceinline__ float par_ez(float e1x, float e1y, float e1z, float e2x, float e2y, float e2z,
                                                 float inv)
{
    constexpr float U = 0x1p-24f;
    const float nx = fabsf(e1y * e2z) + fabsf(e1z * e2y), ny = fabsf(e1z * e2x) + fabsf(e1x * e2z),
                nz = fabsf(e1x * e2y) + fabsf(e1y * e2x);
    const float ai = fabsf(inv);
    const float sx = fabsf(e1x) + fabsf(e2x), sy = fabsf(e1y) + fabsf(e2y), sz = fabsf(e1z) + fabsf(e2z);
    const float b = sx * nx + sy * ny + sz * nz;
    const bool ok = 64.0f * U * nz * ai <= 1.0f && b * ai < 1e30f;
    return ok ? 64.0f * U * (ai * b) + (16.0f * U * sz + 1.0e-6f * (0x1p-12f + 4.0f * U * nz * ai)) : 3.0e38f;
}

// A record with its bounds in one column.
struct ParEntry {
    float e1x, e1y, e1z, e2x, e2y, e2z, inv, v1x, v1y;
    float dz;      // v1z - eps less the origin height of layer l0
    float mu;      // margin of the crossing, in layers
    float delta;
    int l0;        // first layer of the record's voxel zmax
};

// delta of a record; (ox0, oy0) the column's first origin, gx, gy its sub-voxels
__host__ __device__ __forceinline__ float par_delta(const ParEntry& r, float ox0, float oy0, float gx, float gy, int n2,
                                                    float devx, float devy)
{
    constexpr float U = 0x1p-24f;
    const float tmx = fabsf(ox0 - r.v1x) + (float)n2 * gx, tmy = fabsf(oy0 - r.v1y) + (float)n2 * gy;
    const float sx = fabsf(r.e1x) + fabsf(r.e2x), sy = fabsf(r.e1y) + fabsf(r.e2y);
    const float nz = fabsf(r.e1x * r.e2y) + fabsf(r.e1y * r.e2x);
    return 64.0f * U + fabsf(r.inv) * (64.0f * U * (sy * tmx + sx * tmy + nz) + (sy * devx * gx + sx * devy * gy));
}

// the parts of an entry that depend on the column: z1 the record's v1z, oz0 the
// origin height of layer l0 (from the grid's bounds, par_oz), (ox0, oy0) the column's first origin, gx, gy its
// sub-voxels
__host__ __device__ __forceinline__ void par_entry(ParEntry& r, float z1, float oz0, float ox0, float oy0, float gx,
                                                   float gy, int n2, const SatScale& g)
{
    r.dz = (z1 - oz0) - 1.0e-6f;
    // across voxels the origin table keeps within 5.5 U cmax of equal steps and
    // oz0 within 4 U cmax of it, together less than 5 dz
    r.mu = fminf(par_ez(r.e1x, r.e1y, r.e1z, r.e2x, r.e2y, r.e2z, r.inv) * g.sz, 3.0e38f) + 5.0f * g.dz;
    r.delta = par_delta(r, ox0, oy0, gx, gy, n2, g.dx, g.dy);
    if (!(g.dx >= 0.0f && g.dy >= 0.0f && g.dz >= 0.0f)) {   // no scale: everything is undecided
        r.mu = 3.0e38f;
        r.delta = 3.0e38f;
    }
}

// origin height of the first layer of voxel k (bmin + k g, half a sub-voxel up)
__host__ __device__ __forceinline__ float par_oz(float bmin, float g1, float g2, int k)
{
    return bmin + ((float)k * g1 + 0.5f * g2);
}

// layers that hold every toggle of an entry's accepted sub-columns: between
// la and lb of par_layers at the ends of the triangle's z range, grown
__host__ __device__ __forceinline__ void par_z_range(const ParEntry& r, float sz, int cap, int& lmin, int& lmax)
{
    const float lo = fminf(fminf(r.e1z, r.e2z), 0.0f), hi = fmaxf(fmaxf(r.e1z, r.e2z), 0.0f);
    const float grow = 4.0f * r.delta * (fabsf(r.e1z) + fabsf(r.e2z));
    const float m = r.mu + 0.01f + 1e-6f * (fabsf(r.dz) + hi - lo) * sz;
    const float a = fmaxf(((lo - grow) + r.dz) * sz + 1.0f - m, -1.0e8f), b = fminf(((hi + grow) + r.dz) * sz + 1.0f + m, 1.0e8f);
    // a NaN leaves the range whole
    lmin = a >= -1.0e8f ? r.l0 + (int)floorf(fminf(a, 1.0e8f)) : 0;
    lmax = b <= 1.0e8f ? r.l0 + (int)floorf(fmaxf(b, -1.0e8f)) : cap;
    lmin = lmin < 0 ? 0 : lmin > cap ? cap : lmin;
    lmax = lmax < 0 ? 0 : lmax > cap ? cap : lmax;
}

// rows [q0, q0 + n) that can hold an accepted sub-column
__host__ __device__ __forceinline__ int par_rows(const ParEntry& r, float oy0, float sy, int n2, float devy, int& q0)
{
    constexpr float U = 0x1p-24f;
    const float y = (r.v1y - oy0) * sy, a = r.e1y * sy, b = r.e2y * sy;
    const float lo = y + fminf(fminf(a, b), 0.0f), hi = y + fmaxf(fmaxf(a, b), 0.0f);
    const float grow = 4.0f * r.delta * (fabsf(a) + fabsf(b)) + 16.0f * U * (fabsf(y) + fabsf(a) + fabsf(b)) + devy + 0.01f;
    // written so that a NaN leaves the row range whole
    const float f = fminf(fmaxf(ceilf(lo - grow), 0.0f), (float)n2), g = fminf(fmaxf(floorf(hi + grow), -1.0f), (float)(n2 - 1));
    q0 = lo - grow >= 0.0f ? (int)f : 0;
    const int q1 = hi + grow < (float)(n2 - 1) ? (int)g : n2 - 1;
    return q1 - q0 + 1;
}

// of a constraint c0 + c1 x >= 0, its bound on x
__host__ __device__ __forceinline__ void par_bound(float c0, float c1, float& lo, float& hi)
{
    const float t = -c0 * GPV_RCP(c1);
    lo = c1 > 0.0f ? fmaxf(lo, t) : lo;
    hi = c1 < 0.0f ? fminf(hi, t) : hi;
}

// columns [p0, p0 + n) of row q that can be accepted
__host__ __device__ __forceinline__ int par_cols(const ParEntry& r, float ox0, float oy0, float gx, float gy, int n2, int q,
                                                 int& p0)
{
    const float tx = ox0 - r.v1x, ty = (oy0 - r.v1y) + (float)q * gy;
    const float a0 = (r.e2x * ty - r.e2y * tx) * r.inv, a1 = -(r.e2y * r.inv) * gx;
    const float b0 = (r.e1y * tx - r.e1x * ty) * r.inv, b1 = (r.e1y * r.inv) * gx;
    float lo = 0.0f, hi = (float)(n2 - 1);
    par_bound(a0 + r.delta, a1, lo, hi);
    par_bound(b0 + r.delta, b1, lo, hi);
    par_bound((1.0f + 2.0f * r.delta) - (a0 + b0), -(a1 + b1), lo, hi);
    const float f = fminf(ceilf(lo - 0.01f), 32.0f), g = fmaxf(floorf(hi + 0.01f), -1.0f);
    p0 = (int)fmaxf(f, 0.0f);
    return (int)g - p0 + 1;
}

// The layers an accepted sub-column with coordinates u, v passes: all below
// `la`, none from `lb` on, both within [0, cap].
__host__ __device__ __forceinline__ void par_layers(const ParEntry& r, float u, float v, float sz, int cap, int& la, int& lb)
{
    // layer l0 + x is at the crossing's height; l passes for l < that, hence + 1
    const float x = ((u * r.e1z + v * r.e2z) + r.dz) * sz + 1.0f;
    const float a = floorf(fmaxf(x - r.mu, -1.0e8f)), b = floorf(fminf(x + r.mu, 1.0e8f));
    la = r.l0 + (int)fminf(a, 1.0e8f);
    lb = r.l0 + (int)fmaxf(b, -1.0e8f);
    la = la < 0 ? 0 : la > cap ? cap : la;
    lb = lb < 0 ? 0 : lb > cap ? cap : lb;
}

// ---------------------------------------------------------------------------
// Grids far from the origin (as for the SAT, gpv_satrow.hpp: the tables' deviation from
// equal steps is whole sub-voxels).  These take the origins themselves: `delta`
// without the deviation, rows and columns by the tables (within a voxel
// non-decreasing), and of par_layers' [la, lb) the layers that Level1's comparison
// decides (par_l1_layers).
// ---------------------------------------------------------------------------
__host__ __device__ __forceinline__ float par_delta_far(const ParEntry& r, float ox0, float oy0, float gx, float gy, int n2,
                                                        const SatScale& g)
{
    const float wide = fminf(2.0f * fmaxf(g.dx, g.dy) + 1.0f, 1e8f);   // the column is at most n2 and this wide
    const SatScale f = sat_scale_far(g);
    return f.dx >= 0.0f && f.dy >= 0.0f ? par_delta(r, ox0, oy0, gx, gy, n2 + (int)wide, f.dx, f.dy) : 3.0e38f;
}

// margin of the crossing in layers, of `layers` in the grid.  The origins lie within 2 U cmax + U ext
// of bmin + k g1 + (r + 1/2) g2 (8 U cmax in the CUDA kernels' expression), par_oz within U cmax + 2 U ext, and
// g1 within U of n2 g2: with ext = `layers` g2, less than 1.5 dz and 4 U `layers` together.
__host__ __device__ __forceinline__ float par_mu_far(float ez, const SatScale& g, int layers)
{
    const bool ok = g.dx >= 0.0f && g.dy >= 0.0f && g.dz >= 0.0f;
    return ok ? fminf(ez * g.sz, 3.0e38f) + (1.5f * g.dz + 0x1p-21f * (float)layers) : 3.0e38f;
}

// rows [q0, q0 + n) that can hold an accepted sub-column; oy: the column's n2 origins
__host__ __device__ __forceinline__ int par_rows_far(const ParEntry& r, const float* oy, float sy, int n2, int& q0)
{
    constexpr float U = 0x1p-24f;
    const float y = (r.v1y - oy[0]) * sy, a = r.e1y * sy, b = r.e2y * sy;
    const float lo = y + fminf(fminf(a, b), 0.0f), hi = y + fmaxf(fmaxf(a, b), 0.0f);
    const float grow = 4.0f * r.delta * (fabsf(a) + fabsf(b)) + 16.0f * U * (fabsf(y) + fabsf(a) + fabsf(b)) + 0.01f;
    // written so that a NaN leaves the row range whole
    int f = 0, n = n2;
    while (f < n2 && (oy[f] - oy[0]) * sy < lo - grow) ++f;
    while (n > f && (oy[n - 1] - oy[0]) * sy > hi + grow) --n;
    q0 = f;
    return n - f;
}

// columns [p0, p0 + n) of the row at height oyq that can be accepted; ox: the column's n2 origins
__host__ __device__ __forceinline__ int par_cols_far(const ParEntry& r, const float* ox, float oyq, float gx, int n2, int& p0)
{
    const float tx = ox[0] - r.v1x, ty = oyq - r.v1y;
    const float a0 = (r.e2x * ty - r.e2y * tx) * r.inv, a1 = -(r.e2y * r.inv) * gx;
    const float b0 = (r.e1y * tx - r.e1x * ty) * r.inv, b1 = (r.e1y * r.inv) * gx;
    float lo = 0.0f, hi = 1e30f;
    par_bound(a0 + r.delta, a1, lo, hi);
    par_bound(b0 + r.delta, b1, lo, hi);
    par_bound((1.0f + 2.0f * r.delta) - (a0 + b0), -(a1 + b1), lo, hi);
    lo = (lo - 0.01f) * gx;
    hi = (hi + 0.01f) * gx;
    int f = 0, n = n2;
    while (f < n2 && ox[f] - ox[0] < lo) ++f;
    while (n > f && ox[n - 1] - ox[0] > hi) --n;
    p0 = f;
    return n - f;
}

// Of the layers [la, lb) of the origin table rz, those at the lower end that pass for
// certain and those at the upper end that do not, taken off: a layer passes where
// rz - v1z < lo and does not where it is > hi.  Across voxels the table may step back,
// so each voxel's layers are searched by themselves.
__host__ __device__ __forceinline__ void par_narrow(const float* rz, int n2, float inv_n2, float v1z, float lo, float hi,
                                                    int& la, int& lb)
{
    while (la < lb) {
        const int end = ((int)(((float)la + 0.5f) * inv_n2) + 1) * n2, e = end < lb ? end : lb;
        if (rz[e - 1] - v1z < lo) {
            la = e;
            continue;
        }
        int b = e - 1;
        while (la < b) {
            const int m = (la + b) >> 1;
            if (rz[m] - v1z < lo) la = m + 1;
            else b = m;
        }
        break;
    }
    while (lb > la) {
        const int beg = (int)(((float)(lb - 1) + 0.5f) * inv_n2) * n2, s = beg > la ? beg : la;
        if (rz[s] - v1z > hi) {
            lb = s;
            continue;
        }
        int a = s + 1;
        while (a < lb) {
            const int m = (a + lb) >> 1;
            if (rz[m] - v1z > hi) lb = m;
            else a = m + 1;
        }
        break;
    }
}

// Level1: the same crossing against the layers of a grid's column.  Layers [0, la)
// of the ray-origin table r1z (nz, non-decreasing) pass for certain, none from
// lb on.  The layers are compared as the float test's own T.z = fl(o.z - v1.z), so
// only the crossing's height over v1 is rounded: Ez twice over covers that.
// The estimate from the table's ends (zmin, inv_g = layers per z unit) only says where the search begins.
__host__ __device__ __forceinline__ void par_l1_layers(const float* r1z, int nz, float zmin, float inv_g, float v1z,
                                                       float e1z, float e2z, float u, float v, float ez, int& la, int& lb)
{
    const float zc = (u * e1z + v * e2z) - 1.0e-6f;
    const float lo = zc - 2.0f * ez, hi = zc + 2.0f * ez;
    // a NaN starts at 0
    int k = (int)fminf(fmaxf(((lo + v1z) - zmin) * inv_g + 0.5f, 0.0f), (float)nz);
    while (k < nz && r1z[k] - v1z < lo) ++k;
    while (k > 0 && !(r1z[k - 1] - v1z < lo)) --k;
    la = k;
    while (k < nz && !(r1z[k] - v1z > hi)) ++k;
    lb = k;
}

}  // namespace gpv
