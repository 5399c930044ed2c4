// gpv_satrow.hpp -- the Level2 SAT decided for whole rows of sub-voxels, the
// Level1 SAT for whole columns of a triangle's index AABB.
//
// The SAT (src/TriBoxIntersection.cpp:135-210) of one triangle against the
// n2^3 boxes of a boundary voxel is a conjunction of predicates that are
// linear in the box center c: nine edge predicates |f(c) - mid| <= half, each
// in two coordinates of c, the plane predicate |N.(c - t0)| <= R, and the
// three box-axis predicates.  For a fixed row (c.y) and column (c.x) every
// predicate that involves c.z is an interval of c.z, so the boxes that pass
// are one run of layers: the largest lower end to the smallest upper end.
// The reference evaluates the predicates in float; with M a bound on how far
// its value and the one computed here can lie from the exact one, a layer
// inside [lo + M, hi - M] passes the float predicate for certain and one
// outside [lo - M, hi + M] fails it for certain.  Each column so gets two
// masks of layers, `in` (every predicate holds) and `may` (none certainly
// fails); the caller runs the reference's own float SAT on may & ~in, a few
// boxes in a thousand, and no result changes.
//
// Units.  Each axis is scaled by s = fl(1/g2) and measured from the triangle's
// first vertex t0: the voxel's sub-center p lies at p - xi with
// xi = (t0 - c0) s, c0 its sub-center 0, up to dev: the float tables round
// each center, by at most 2.1 U cmax in the reference's double expression (8 U
// cmax in the float one of its CUDA kernels), U = 2^-24, cmax the largest
// |center|; 256 U more pay for keeping positions as index offsets.  Predicates scale by positive constants with the axes; half
// extents become 0.5.
//
// Bounds.  A_a = ext_a + 0.5 bounds |t_i - c| on every box whose box-axis
// predicates hold (only those are asked for); |E_a| <= ext_a.  For an edge E
// in the coordinates (u, w), S = |E_w| A_u + |E_u| A_w and T = A_u A_w:
//   reference: v = fl(t - c), e = fl(v_b - v_a), |e - E| <= U (2A + |E|), the
//     two products, their difference and the radius: 5.2 U S + 12.2 U T;
//   here: E = fl(t_b - t_a) s (2U), positions (3U A and dev), slopes and
//     reciprocals (1 ulp, 3U), the area N (8.5 U T), sums, and at most 16
//     additions along the row (48 U S): 65 U S + 8.5 U T + |E_w| dev_u + |E_u| dev_w.
// M = 128 U S + 32 U T + (dev terms) is used.  Where |E_u| is too small to divide
// by, it is replaced by 16 U |E_w| A_u / A_w, which moves f by at most
// 32 U |E_w| A_u (within the 128).  An edge with E_u = E_w = 0 always passes: its
// float components are exactly zero.  The plane: with G the sums of products
// of edge and A that bound its error,
//   M = 64 U sum A (|N| + G) + sum |N| dev + 2^-19 R
// (reference 9.2 U A|N| + 21 U A G, here 40 U A|N| + 11 U A G; the last term
// pays for keeping |N_z| away from zero).  Where a magnitude leaves the range
// these products need (A above 2^24 sub-voxels, a reciprocal above 1e20, a
// nearly degenerate triangle other than a segment), or g2 is outside [2^-40, 2^40], the entry is
// `loose`: every layer asked for is undecided.
#pragma once

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

namespace gpv {

// s = fl(1/g2) per axis and the deviation of the center tables in sub-voxels
struct SatScale {
    float sx, sy, sz;
    float dx, dy, dz;
};

// one axis of SatScale; `lo`/`hi` the grid's bounds on it, g2 its sub-voxel.
// dev < 0 marks a size outside the range the bounds hold for.
inline void sat_scale_axis(float lo, float hi, float g2, bool cuda_l2, float& s, float& dev)
{
    s = 0.0f;
    dev = -1.0f;
    if (!(g2 >= 0x1p-40f && g2 <= 0x1p40f)) return;
    s = 1.0f / g2;
    const double cmax = fmax(fabs((double)lo), fabs((double)hi));
    dev = (float)((cuda_l2 ? 8.0 : 2.1) * 0x1p-24 * 1.01 * cmax / (double)g2 + 256.0 * 0x1p-24);
}

// What the rows of one (triangle, voxel) pair share: 10 groups of four floats,
// in the voxel's sub-center indices (a layer counts as >= lo from
// trunc(lo + 1) on, hence centers one up).
//   0-2  the edges' predicates in (y, z): slope, center at y = 0, half width of
//        the outer and of the inner interval (in layers)
//   3-5  the same in (x, z)
//   6    the edges' predicates in (x, y), over half: coefficients of x; margin
//   7    coefficients of y; slope of the plane in x
//   8    constants; slope of the plane in y
//   9    plane: center at x = y = 0, half widths
constexpr int kSatEntry4 = 10;

#ifdef __HIP_DEVICE_COMPILE__
#define GPV_RCP(x) __builtin_amdgcn_rcpf(x)
#else
#define GPV_RCP(x) (1.0f / (x))
#endif

// an edge's predicate in (u, z): slope, center (base +- kh, kh the signed half
// of the triangle's width there) and half widths
__host__ __device__ __forceinline__ float4 sat_edge_z(float eu, float ez, bool zero, float area, float base, float rho,
                                                      float c1, float c2, float t, float off, float& rmax)
{
    const float ae = fmaxf(fabsf(eu), rho * fabsf(ez));
    const float r = zero ? 0.0f : GPV_RCP(ae);
    rmax = fmaxf(rmax, r);
    const float rs = copysignf(r, eu);
    const float al = ez * rs, aa = fabsf(al);
    const float kh = area * rs;
    const float half = fabsf(kh) + (aa * 0.5f + (zero ? 1e30f : 0.5f));
    const float m = aa * c1 + (r * t + c2);
    return make_float4(al, (base + kh) - al * off, half + m, half - m);
}

// Part `h` (0 or 1) of the entry of triangle tv in the voxel whose sub-center
// 0 is c0 (kBox: in the index AABB whose first center is c0, where a box may
// miss the triangle's extent by the rounding of the index and of the tables):
// 0 writes groups 0-2 and 9, 1 the others (the plane's slopes included).  Two
// lanes can make one entry on the device; looseness has to be combined from both
// parts.  `plane`: the plane cannot be bounded, which makes the entry loose unless the
// triangle is a segment (sat_segment); returned are the other reasons.
template <bool kBox>
__host__ __device__ __forceinline__ bool sat_entry_terms(int h, const float* tv, float c0x, float c0y, float c0z,
                                                         const SatScale& g, float4* out, bool& plane)
{
    constexpr float U = 0x1p-24f;
    const float t0x = tv[0], t0y = tv[1], t0z = tv[2], t1x = tv[3], t1y = tv[4], t1z = tv[5], t2x = tv[6],
                t2y = tv[7], t2z = tv[8];
    // edges, raw (for the exact zeros) and in sub-voxels
    const float r0x = t1x - t0x, r0y = t1y - t0y, r0z = t1z - t0z;
    const float r1x = t2x - t1x, r1y = t2y - t1y, r1z = t2z - t1z;
    const float r2x = t0x - t2x, r2y = t0y - t2y, r2z = t0z - t2z;
    const float e0x = r0x * g.sx, e0y = r0y * g.sy, e0z = r0z * g.sz;
    const float e1x = r1x * g.sx, e1y = r1y * g.sy, e1z = r1z * g.sz;
    const float e2x = r2x * g.sx, e2y = r2y * g.sy, e2z = r2z * g.sz;
    // extents: the longest edge of each axis spans the other two
    const float Ax = fmaxf(fmaxf(fabsf(e0x), fabsf(e1x)), fabsf(e2x)) * 1.00001f +
                     (kBox ? 0.51f + 2.0f * g.dx : 0.50001f);
    const float Ay = fmaxf(fmaxf(fabsf(e0y), fabsf(e1y)), fabsf(e2y)) * 1.00001f +
                     (kBox ? 0.51f + 2.0f * g.dy : 0.50001f);
    const float Az = fmaxf(fmaxf(fabsf(e0z), fabsf(e1z)), fabsf(e2z)) * 1.00001f +
                     (kBox ? 0.51f + 2.0f * g.dz : 0.50001f);
    const float Nx = e0y * e1z - e0z * e1y, Ny = e0z * e1x - e0x * e1z, Nz = e0x * e1y - e0y * e1x;
    const float rz = GPV_RCP(Az) * (16.0f * U);
    const float zeta = (t0z - c0z) * g.sz + 1.0f, xi = (t0x - c0x) * g.sx, eta = (t0y - c0y) * g.sy;
    float rmax = 0.0f;
    {
        // (y, z) or (x, z)
        const float Au = h ? Ax : Ay, du = h ? g.dx : g.dy;
        const float rho = Au * rz, c1 = 128.0f * U * Au + du, c2 = 128.0f * U * Az + g.dz, t = 32.0f * U * Au * Az;
        const float area = 0.5f * (h ? -Ny : Nx), off = h ? xi : eta;
        const float u0 = h ? r0x : r0y, u1 = h ? r1x : r1y, u2 = h ? r2x : r2y, su = h ? g.sx : g.sy;
        float4* o = out + 3 * h;
        o[0] = sat_edge_z(u0 * su, e0z, fmaxf(fabsf(u0), fabsf(r0z)) == 0.0f, area, zeta, rho, c1, c2, t, off, rmax);
        o[1] = sat_edge_z(u1 * su, e1z, fmaxf(fabsf(u1), fabsf(r1z)) == 0.0f, -area, zeta, rho, c1, c2, t, off, rmax);
        o[2] = sat_edge_z(u2 * su, e2z, fmaxf(fabsf(u2), fabsf(r2z)) == 0.0f, area, zeta, rho, c1, c2, t, off, rmax);
    }
    bool loose = !(fmaxf(fmaxf(Ax, Ay), Az) < 0x1p24f) || !(fminf(fminf(g.dx, g.dy), g.dz) >= 0.0f);
    // the plane
    const float anx = fabsf(Nx), any = fabsf(Ny), anz = fabsf(Nz);
    const float R = 0.5f * (anx + any + anz);
    const float r = GPV_RCP(fmaxf(anz, R * rz));
    const float rs = copysignf(r, Nz);
    const float pa = -Nx * rs, pb = -Ny * rs;
    if (h) {
        // (x, y), over its half width
        const float hn = 0.5f * Nz, ah = fabsf(hn);
        const float q0 = fmaxf(fabsf(r0x), fabsf(r0y)) == 0.0f ? 0.0f : GPV_RCP(ah + 0.5f * (fabsf(e0x) + fabsf(e0y)));
        const float q1 = fmaxf(fabsf(r1x), fabsf(r1y)) == 0.0f ? 0.0f : GPV_RCP(ah + 0.5f * (fabsf(e1x) + fabsf(e1y)));
        const float q2 = fmaxf(fabsf(r2x), fabsf(r2y)) == 0.0f ? 0.0f : GPV_RCP(ah + 0.5f * (fabsf(e2x) + fabsf(e2y)));
        const float q = fmaxf(fmaxf(q0, q1), q2);
        rmax = fmaxf(rmax, q);
        const float m = 256.0f * U * fmaxf(Ax, Ay) + (q * (32.0f * U * Ax * Ay) + 2.0f * fmaxf(g.dx, g.dy));
        out[6] = make_float4(e0y * q0, e1y * q1, e2y * q2, m);
        out[7] = make_float4(-e0x * q0, -e1x * q1, -e2x * q2, pa);
        out[8] = make_float4((hn - (e0y * xi - e0x * eta)) * q0, (-hn - (e1y * xi - e1x * eta)) * q1,
                             (hn - (e2y * xi - e2x * eta)) * q2, pb);
    } else {
        const float Q = (Ax * anx + Ay * any + Az * anz) +
                        2.0f * (Ax * Ay * (fabsf(e0z) + fabsf(e1z)) + Ax * Az * (fabsf(e0y) + fabsf(e1y)) +
                                Ay * Az * (fabsf(e0x) + fabsf(e1x)));
        const float M = 64.0f * U * Q + (g.dx * anx + g.dy * any + g.dz * anz) + 0x1p-19f * R;
        const float hw = R * r, mp = M * r + g.dz;
        out[9] = make_float4(zeta - (pa * xi + pb * eta), hw + mp, hw - mp, 0.0f);
    }
    plane = !(r < 1e12f);
    return loose || !(rmax < 1e20f);
}

// Two vertices the same: the reference's normal is exactly zero (a zero edge, or one the
// negative of the other) and its plane test passes everywhere.  So is the normal here, its
// reciprocal infinite, and each of the plane's terms a NaN, which fmaxf and fminf pass over: the
// plane bounds nothing.
__host__ __device__ __forceinline__ bool sat_segment(const float* tv)
{
    return (tv[0] == tv[3] && tv[1] == tv[4] && tv[2] == tv[5]) || (tv[3] == tv[6] && tv[4] == tv[7] && tv[5] == tv[8]) ||
           (tv[6] == tv[0] && tv[7] == tv[1] && tv[8] == tv[2]);
}

// The same, and whether the part makes the entry loose.
__host__ __device__ __forceinline__ bool sat_entry_part(int h, const float* tv, float c0x, float c0y, float c0z,
                                                        const SatScale& g, float4* out)
{
    bool plane;
    const bool loose = sat_entry_terms<false>(h, tv, c0x, c0y, c0z, g, out, plane);
    return loose || (plane && !sat_segment(tv));
}

// A box axis: with x the triangle's least (greatest) coordinate in centers from the
// voxel's sub-center 0, the float predicate's half fl(x - c) > h (< -h) fails
// for the centers from (up to) floor(x + 1/2) on.  Returns that, within [-2,
// n + 2]; clear = false where x + 1/2 lies so near an integer that the rounding
// of the table (dev), of x and of the test (57 U together) could decide.
__host__ __device__ __forceinline__ int sat_axis_end(float x, int n, float dev, bool& clear)
{
    const float y = fminf(fmaxf(x, -2.0f), (float)n + 2.0f) + 0.5f, f = floorf(y);
    clear = clear && dev >= 0.0f && fabsf((y - f) - 0.5f) < 0.5f - (2.0f * dev + 0x1p-18f);
    return (int)f;
}

// One row of an entry, positioned at a column.
struct SatRow {
    float a0, a1, a2, w0, w1, w2, m0, m1, m2, n0, n1, n2;   // (x, z): slope, center, half widths
    float e0, e1, e2, u0, u1, u2, um;                       // (x, y): step, value, margin
    float pa, pw, pm, pn;                                   // plane: step, center, half widths
    float lom, loi, him, hii;                               // box axis and (y, z)
};

// the columns x where |e x + c| <= lim can hold, a hundredth of a column wide of them
__host__ __device__ __forceinline__ void sat_x_range(float e, float c, float lim, float& lo, float& hi)
{
    const float r = GPV_RCP(e);
    const float a = (-lim - c) * r, b = (lim - c) * r;
    lo = fmaxf(lo, fminf(a, b));
    hi = fminf(hi, fmaxf(a, b));
}

// Row q: of the columns [p, p + left) it drops those at either end that the (x, y)
// predicates certainly fail (unless `keep`).
__host__ __device__ __forceinline__ void sat_row_range(const float4* e, int q, bool keep, int& p, int& left)
{
    const float4 c6 = e[6], c7 = e[7], c8 = e[8];
    const float y = (float)q;
    const float u0 = c7.x * y + c8.x, u1 = c7.y * y + c8.y, u2 = c7.z * y + c8.z;
    const float lim = 1.0f + c6.w;
    float lo = (float)p - 0.5f, hi = (float)(p + left) - 0.5f;
    sat_x_range(c6.x, u0, lim, lo, hi);
    sat_x_range(c6.y, u1, lim, lo, hi);
    sat_x_range(c6.z, u2, lim, lo, hi);
    // columns in [lo - 0.01, hi + 0.01]; both ends lie in (p - 1, p + left) unless the row is empty
    const int p1 = (int)fminf(fmaxf(lo + 0.99f, 0.0f), 16.0f), pe = (int)fminf(fmaxf(hi + 1.01f, 0.0f), 16.0f);
    left = keep ? left : pe - p1;
    p = keep ? p : p1;
}

// The row at height y with layers from `zlo` below `zhi`, positioned at x.
__host__ __device__ __forceinline__ SatRow sat_row_xy(const float4* e, float y, float zlo, float zhi, float x)
{
    SatRow s;
    const float4 c6 = e[6], c7 = e[7], c8 = e[8], pl = e[9];
    const float u0 = c7.x * y + c8.x, u1 = c7.y * y + c8.y, u2 = c7.z * y + c8.z;
    s.lom = s.loi = zlo;
    s.him = s.hii = zhi;
#ifdef __HIP_DEVICE_COMPILE__
#pragma unroll
#endif
    for (int k = 0; k < 3; ++k) {
        const float4 c = e[k];
        const float w = c.x * y + c.y;
        s.lom = fmaxf(s.lom, w - c.z); s.loi = fmaxf(s.loi, w - c.w);
        s.him = fminf(s.him, w + c.z); s.hii = fminf(s.hii, w + c.w);
    }
    const float4 x0 = e[3], x1 = e[4], x2 = e[5];
    s.a0 = x0.x; s.w0 = x0.x * x + x0.y; s.m0 = x0.z; s.n0 = x0.w;
    s.a1 = x1.x; s.w1 = x1.x * x + x1.y; s.m1 = x1.z; s.n1 = x1.w;
    s.a2 = x2.x; s.w2 = x2.x * x + x2.y; s.m2 = x2.z; s.n2 = x2.w;
    s.e0 = c6.x; s.u0 = c6.x * x + u0;
    s.e1 = c6.y; s.u1 = c6.y * x + u1;
    s.e2 = c6.z; s.u2 = c6.z * x + u2;
    s.um = c6.w;
    s.pa = c7.w; s.pw = (c7.w * x + c8.w * y) + pl.x; s.pm = pl.y; s.pn = pl.z;
    return s;
}

// Row q with layers [ra, rb], positioned at column p.
__host__ __device__ __forceinline__ SatRow sat_row_at(const float4* e, int q, int ra, int rb, int p)
{
    return sat_row_xy(e, (float)q, (float)ra, (float)rb + 1.0f, (float)p);
}

// A row of a loose entry (nothing of it is bounded): all layers of its columns undecided,
// none certain.  Every term is set: an entry is loose where its coefficients may be
// infinite or NaN, those of the (x, y) predicates among them.
__host__ __device__ __forceinline__ void sat_row_loose(SatRow& s, bool loose, int ra, int rb)
{
    if (!loose) return;
    s.a0 = s.a1 = s.a2 = s.pa = 0.0f;
    s.w0 = s.w1 = s.w2 = s.pw = 0.0f;
    s.m0 = s.m1 = s.m2 = s.pm = 1e30f;
    s.n0 = s.n1 = s.n2 = s.pn = 0.0f;
    s.lom = s.loi = (float)ra;
    s.him = (float)rb + 1.0f;
    s.hii = 0.0f;
    s.e0 = s.e1 = s.e2 = 0.0f;
    s.u0 = s.u1 = s.u2 = 0.0f;
    s.um = 3e38f;
}

// ---------------------------------------------------------------------------
// Grids far from the origin.  There a float hardly tells one sub-center from the
// next, `dev` is whole sub-voxels, and rows that count positions in equal steps
// leave most boxes undecided.  These take the sub-centers themselves instead: the voxel's
// positions X, Y (from its first center, in sub-voxels) and Z (one up, as the
// entry's layers), 16 each, non-decreasing (within a voxel every step of the tables' expressions
// is monotone), infinite past n2.  What `dev` paid for is gone but for the
// positions' own rounding, 3 U of at most 16 + 2 dev.  A row steps by
// slope * (X[p + 1] - X[p]), two roundings more per addition: at most 4 U S.
// ---------------------------------------------------------------------------
__host__ __device__ __forceinline__ SatScale sat_scale_far(SatScale g)
{
    // (dev < 0 stays what it is: loose)
    g.dx = g.dx >= 0.0f ? 0x1p-24f * (256.0f + 32.0f * g.dx) : g.dx;
    g.dy = g.dy >= 0.0f ? 0x1p-24f * (256.0f + 32.0f * g.dy) : g.dy;
    g.dz = g.dz >= 0.0f ? 0x1p-24f * (256.0f + 32.0f * g.dz) : g.dz;
    return g;
}

// how many of the 2 * half (8 or 16) positions are at most x
__host__ __device__ __forceinline__ int sat_count_le(const float* pos, int half, float x)
{
    int i = 0;
    for (int s = half; s; s >>= 1) i += pos[i + s - 1] <= x ? s : 0;
    return i + (pos[i] <= x ? 1 : 0);
}

// sat_row_range for the row at height y
__host__ __device__ __forceinline__ void sat_row_range_far(const float4* e, float y, const float* X, int half, bool keep,
                                                           int& p, int& left)
{
    const float4 c6 = e[6], c7 = e[7], c8 = e[8];
    const float u0 = c7.x * y + c8.x, u1 = c7.y * y + c8.y, u2 = c7.z * y + c8.z;
    const float lim = 1.0f + c6.w;
    float lo = -1e30f, hi = 1e30f;
    sat_x_range(c6.x, u0, lim, lo, hi);
    sat_x_range(c6.y, u1, lim, lo, hi);
    sat_x_range(c6.z, u2, lim, lo, hi);
    const int a = sat_count_le(X, half, lo - 0.01f), b = sat_count_le(X, half, hi + 0.01f);
    const int p1 = a > p ? a : p, pe = b < p + left ? b : p + left;
    left = keep ? left : pe - p1;
    p = keep ? p : p1;
}

// truncation that takes anything below 0 to 0
__host__ __device__ __forceinline__ uint32_t sat_trunc(float x)
{
#ifdef __HIP_DEVICE_COMPILE__
    uint32_t r;
    asm("v_cvt_u32_f32 %0, %1" : "=v"(r) : "v"(x));
    return r;
#else
    return x > 0.0f ? (uint32_t)x : 0u;
#endif
}

// The current column's layer masks (sat_row_loose first for a loose entry); steps the
// row to the next column.
__host__ __device__ __forceinline__ void sat_row_column(SatRow& s, uint32_t& in, uint32_t& may)
{
    const float lom = fmaxf(fmaxf(s.w0 - s.m0, s.w1 - s.m1), fmaxf(fmaxf(s.w2 - s.m2, s.pw - s.pm), s.lom));
    const float loi = fmaxf(fmaxf(s.w0 - s.n0, s.w1 - s.n1), fmaxf(fmaxf(s.w2 - s.n2, s.pw - s.pn), s.loi));
    const float him = fminf(fminf(s.w0 + s.m0, s.w1 + s.m1), fminf(fminf(s.w2 + s.m2, s.pw + s.pm), s.him));
    const float hii = fminf(fminf(s.w0 + s.n0, s.w1 + s.n1), fminf(fminf(s.w2 + s.n2, s.pw + s.pn), s.hii));
    const float u = fmaxf(fmaxf(fabsf(s.u0), fabsf(s.u1)), fabsf(s.u2)) - 1.0f;
    s.w0 += s.a0; s.w1 += s.a1; s.w2 += s.a2; s.pw += s.pa;
    s.u0 += s.e0; s.u1 += s.e1; s.u2 += s.e2;
    // layers [trunc(lo), trunc(hi)) with hi at most 16
    const uint32_t m = ~(~0u << sat_trunc(him)) & (~0u << sat_trunc(fminf(lom, 16.0f)));
    const uint32_t n = ~(~0u << sat_trunc(hii)) & (~0u << sat_trunc(fminf(loi, 16.0f)));
    may = !(u > s.um) ? m : 0u;
    in = u < -s.um ? n : 0u;
}

// The same far from the origin, for the layers of `rows` (a bit each); the row was set up
// with layers of any height, `step` is X[p + 1] - X[p].
__host__ __device__ __forceinline__ void sat_row_column_far(SatRow& s, const float* Z, int half, uint32_t rows, float step,
                                                            uint32_t& in, uint32_t& may)
{
    const float lom = fmaxf(fmaxf(s.w0 - s.m0, s.w1 - s.m1), fmaxf(fmaxf(s.w2 - s.m2, s.pw - s.pm), s.lom));
    const float loi = fmaxf(fmaxf(s.w0 - s.n0, s.w1 - s.n1), fmaxf(fmaxf(s.w2 - s.n2, s.pw - s.pn), s.loi));
    const float him = fminf(fminf(s.w0 + s.m0, s.w1 + s.m1), fminf(fminf(s.w2 + s.m2, s.pw + s.pm), s.him));
    const float hii = fminf(fminf(s.w0 + s.n0, s.w1 + s.n1), fminf(fminf(s.w2 + s.n2, s.pw + s.pn), s.hii));
    const float u = fmaxf(fmaxf(fabsf(s.u0), fabsf(s.u1)), fabsf(s.u2)) - 1.0f;
    s.w0 += s.a0 * step; s.w1 += s.a1 * step; s.w2 += s.a2 * step; s.pw += s.pa * step;
    s.u0 += s.e0 * step; s.u1 += s.e1 * step; s.u2 += s.e2 * step;
    const int a = sat_count_le(Z, half, lom), b = sat_count_le(Z, half, him);
    int c = a, d = b;
    while (c < d && Z[c] <= loi) ++c;
    while (d > c && Z[d - 1] > hii) --d;
    const uint32_t m = ~(~0u << b) & (~0u << a) & rows;
    const uint32_t n = ~(~0u << d) & (~0u << c) & rows;
    may = !(u > s.um) ? m : 0u;
    in = u < -s.um ? n : 0u;
}

// ---------------------------------------------------------------------------
// The same for one column of a triangle's Level1 index AABB: any number of
// layers, as index intervals, and the box-axis predicates (whose boxes the
// AABB only approximates) among the bounded ones.  Their values: the
// reference's t - c (U A) against ours (3 U A and dev), A at most the extent
// and half a voxel: 16 U (extent + 1) + 2 dev.
// ---------------------------------------------------------------------------
struct SatColumn {
    int am, ai, bi, bm;   // layers [ai, bi) pass; of [am, bm) the others are undecided; the rest fail
};

// (x, y): the column in the AABB, whose first center is c0 and which has
// `layers` layers
__host__ __device__ __forceinline__ SatColumn sat_column(const float* tv, float c0x, float c0y, float c0z,
                                                         const SatScale& g, int xi, int yi, int layers)
{
    constexpr float U = 0x1p-24f;
    float4 e[kSatEntry4];
    bool plane;   // the same for both parts
    bool loose = sat_entry_terms<true>(0, tv, c0x, c0y, c0z, g, e, plane);
    loose = sat_entry_terms<true>(1, tv, c0x, c0y, c0z, g, e, plane) || loose;
    const float x = (float)xi, y = (float)yi, n = (float)layers;
    // box axes: the triangle's extent, half a voxel more on each side
    const float x0 = (fminf(fminf(tv[0], tv[3]), tv[6]) - c0x) * g.sx, x1 = (fmaxf(fmaxf(tv[0], tv[3]), tv[6]) - c0x) * g.sx;
    const float y0 = (fminf(fminf(tv[1], tv[4]), tv[7]) - c0y) * g.sy, y1 = (fmaxf(fmaxf(tv[1], tv[4]), tv[7]) - c0y) * g.sy;
    const float z0 = (fminf(fminf(tv[2], tv[5]), tv[8]) - c0z) * g.sz, z1 = (fmaxf(fmaxf(tv[2], tv[5]), tv[8]) - c0z) * g.sz;
    const float far = fmaxf(fmaxf(x0 - x, x - x1), fmaxf(y0 - y, y - y1)) - 0.5f;
    const float mxy = 16.0f * U * (fmaxf(x1 - x0, y1 - y0) + 1.0f) + 2.0f * fmaxf(g.dx, g.dy);
    const float mz = 16.0f * U * ((z1 - z0) + 1.0f) + 2.0f * g.dz;
    float lom = fmaxf(0.0f, (z0 + 0.5f) - mz), loi = fmaxf(0.0f, (z0 + 0.5f) + mz);
    float him = fminf(n, (z1 + 1.5f) + mz), hii = fminf(n, (z1 + 1.5f) - mz);
#ifdef __HIP_DEVICE_COMPILE__
#pragma unroll
#endif
    for (int k = 0; k < 6; ++k) {
        const float4 c = e[k];
        const float w = c.x * (k < 3 ? y : x) + c.y;
        lom = fmaxf(lom, w - c.z); loi = fmaxf(loi, w - c.w);
        him = fminf(him, w + c.z); hii = fminf(hii, w + c.w);
    }
    const float4 c6 = e[6], c7 = e[7], c8 = e[8], pl = e[9];
    const float pw = (c7.w * x + c8.w * y) + pl.x;
    lom = fmaxf(lom, pw - pl.y); loi = fmaxf(loi, pw - pl.z);
    him = fminf(him, pw + pl.y); hii = fminf(hii, pw + pl.z);
    const float u = fmaxf(fmaxf(fabsf((c6.x * x + c7.x * y) + c8.x), fabsf((c6.y * x + c7.y * y) + c8.y)),
                          fabsf((c6.z * x + c7.z * y) + c8.z)) - 1.0f;
    SatColumn s;
    s.am = (int)fminf(lom, n);
    s.bm = (int)fmaxf(him, 0.0f);
    s.ai = (int)fminf(loi, n);
    s.bi = (int)fmaxf(hii, 0.0f);
    if (!(u < -c6.w) || !(far < -mxy)) s.ai = s.bi = 0;
    if (u > c6.w || far > mxy) s.am = s.bm = 0;
    if ((loose || plane) && (loose || !sat_segment(tv))) {
        s.am = s.ai = s.bi = 0;
        s.bm = layers;
    }
    return s;
}

}  // namespace gpv
