// Host harness for the row form of the Level2 SAT (gpview_amd/csrc/
// gpv_satrow.hpp): tests/test_sat_rows.py compares its masks with the
// reference's SAT.  Test tooling only.
#include <stdint.h>
#include "gpv_satrow.hpp"

static bool axis_ok(float a0, float a1, float a2, float c, float h)
{
    const float d0 = a0 - c, d1 = a1 - c, d2 = a2 - c;
    float mn = d0, mx = d0;
    if (d1 < mn) mn = d1;
    if (d1 > mx) mx = d1;
    if (d2 < mn) mn = d2;
    if (d2 > mx) mx = d2;
    return !((mn > h) | (mx < -h));
}

// Case i: triangle tv[9i..], a voxel's sub-center tables cx/cy/cz[n2*i..],
// grid bounds lo/hi[3i..], sub-voxel g2[3i..], half extents h[3i..].  Per
// column (q * n2 + p): the layer masks `in` and `may`.  Rows are cut to the
// boxes whose box-axis predicates hold, as the kernel does.
extern "C" void satrow_batch(int64_t n, int n2, const float* tv, const float* cx, const float* cy, const float* cz,
                             const float* lo, const float* hi, const float* g2, const float* h, int cuda_l2,
                             uint32_t* in, uint32_t* may)
{
    for (int64_t i = 0; i < n; ++i) {
        const float* t = tv + 9 * i;
        const float *X = cx + n2 * i, *Y = cy + n2 * i, *Z = cz + n2 * i;
        gpv::SatScale g;
        gpv::sat_scale_axis(lo[3 * i], hi[3 * i], g2[3 * i], cuda_l2 != 0, g.sx, g.dx);
        gpv::sat_scale_axis(lo[3 * i + 1], hi[3 * i + 1], g2[3 * i + 1], cuda_l2 != 0, g.sy, g.dy);
        gpv::sat_scale_axis(lo[3 * i + 2], hi[3 * i + 2], g2[3 * i + 2], cuda_l2 != 0, g.sz, g.dz);
        int pa = n2, pb = -1, ra = n2, rb = -1;
        for (int p = 0; p < n2; ++p) {
            if (axis_ok(t[0], t[3], t[6], X[p], h[3 * i])) { pa = p < pa ? p : pa; pb = p; }
            if (axis_ok(t[2], t[5], t[8], Z[p], h[3 * i + 2])) { ra = p < ra ? p : ra; rb = p; }
        }
        float4 e[gpv::kSatEntry4];
        bool loose = gpv::sat_entry_part(0, t, X[0], Y[0], Z[0], g, e);
        loose = gpv::sat_entry_part(1, t, X[0], Y[0], Z[0], g, e) || loose;
        for (int q = 0; q < n2; ++q) {
            uint32_t* oi = in + (int64_t)(i * n2 + q) * n2;
            uint32_t* om = may + (int64_t)(i * n2 + q) * n2;
            for (int p = 0; p < n2; ++p) oi[p] = om[p] = 0;
            if (pb < 0 || rb < 0 || !axis_ok(t[1], t[4], t[7], Y[q], h[3 * i + 1])) continue;
            int p = pa, left = pb - pa + 1;
            gpv::sat_row_range(e, q, loose, p, left);
            gpv::SatRow s = gpv::sat_row_at(e, q, ra, rb, p);
            const uint32_t all = ((2u << rb) - 1u) & ~((1u << ra) - 1u);
            for (int k = 0; k < left; ++k) {
                gpv::sat_row_column(s, oi[p + k], om[p + k]);
                if (loose) {
                    oi[p + k] = 0;
                    om[p + k] = all;
                }
            }
        }
    }
}

// The same with every row walked in pieces of `piece` columns, each begun at its own
// column with sat_row_at and, for a loose entry, sat_row_loose: the kernel's own
// sequence, with no word of the harness's about loose entries.
extern "C" void satrow_pieces(int64_t n, int n2, int piece, const float* tv, const float* cx, const float* cy, const float* cz,
                              const float* lo, const float* hi, const float* g2, const float* h, int cuda_l2,
                              uint32_t* in, uint32_t* may, uint8_t* is_loose)
{
    for (int64_t i = 0; i < n; ++i) {
        const float* t = tv + 9 * i;
        const float *X = cx + n2 * i, *Y = cy + n2 * i, *Z = cz + n2 * i;
        gpv::SatScale g;
        gpv::sat_scale_axis(lo[3 * i], hi[3 * i], g2[3 * i], cuda_l2 != 0, g.sx, g.dx);
        gpv::sat_scale_axis(lo[3 * i + 1], hi[3 * i + 1], g2[3 * i + 1], cuda_l2 != 0, g.sy, g.dy);
        gpv::sat_scale_axis(lo[3 * i + 2], hi[3 * i + 2], g2[3 * i + 2], cuda_l2 != 0, g.sz, g.dz);
        int pa = n2, pb = -1, ra = n2, rb = -1;
        for (int p = 0; p < n2; ++p) {
            if (axis_ok(t[0], t[3], t[6], X[p], h[3 * i])) { pa = p < pa ? p : pa; pb = p; }
            if (axis_ok(t[2], t[5], t[8], Z[p], h[3 * i + 2])) { ra = p < ra ? p : ra; rb = p; }
        }
        float4 e[gpv::kSatEntry4];
        bool loose = gpv::sat_entry_part(0, t, X[0], Y[0], Z[0], g, e);
        loose = gpv::sat_entry_part(1, t, X[0], Y[0], Z[0], g, e) || loose;
        is_loose[i] = loose;
        for (int q = 0; q < n2; ++q) {
            uint32_t* oi = in + (int64_t)(i * n2 + q) * n2;
            uint32_t* om = may + (int64_t)(i * n2 + q) * n2;
            for (int p = 0; p < n2; ++p) oi[p] = om[p] = 0;
            if (pb < 0 || rb < 0 || !axis_ok(t[1], t[4], t[7], Y[q], h[3 * i + 1])) continue;
            int p = pa, left = pb - pa + 1;
            gpv::sat_row_range(e, q, loose, p, left);
            for (; left > 0; p += piece, left -= piece) {
                gpv::SatRow s = gpv::sat_row_at(e, q, ra, rb, p);
                gpv::sat_row_loose(s, loose, ra, rb);
                for (int k = 0; k < (left < piece ? left : piece); ++k) gpv::sat_row_column(s, oi[p + k], om[p + k]);
            }
        }
    }
}

// satrow_pieces with the positions taken from the tables (grids far from the origin).
extern "C" void satrow_far(int64_t n, int n2, int piece, const float* tv, const float* cx, const float* cy, const float* cz,
                           const float* lo, const float* hi, const float* g2, const float* h, int cuda_l2,
                           uint32_t* in, uint32_t* may, uint8_t* is_loose)
{
    const int half = n2 > 8 ? 8 : 4;
    for (int64_t i = 0; i < n; ++i) {
        const float* t = tv + 9 * i;
        const float* C[3] = {cx + n2 * i, cy + n2 * i, cz + n2 * i};
        gpv::SatScale g;
        gpv::sat_scale_axis(lo[3 * i], hi[3 * i], g2[3 * i], cuda_l2 != 0, g.sx, g.dx);
        gpv::sat_scale_axis(lo[3 * i + 1], hi[3 * i + 1], g2[3 * i + 1], cuda_l2 != 0, g.sy, g.dy);
        gpv::sat_scale_axis(lo[3 * i + 2], hi[3 * i + 2], g2[3 * i + 2], cuda_l2 != 0, g.sz, g.dz);
        float pos[3][16];
        const float s[3] = {g.sx, g.sy, g.sz};
        int end[3][2];
        for (int a = 0; a < 3; ++a) {
            end[a][0] = n2;
            end[a][1] = -1;
            for (int p = 0; p < 16; ++p) {
                pos[a][p] = p < n2 ? (C[a][p] - C[a][0]) * s[a] + (a == 2 ? 1.0f : 0.0f) : __builtin_inff();
                if (p < n2 && axis_ok(t[a], t[3 + a], t[6 + a], C[a][p], h[3 * i + a])) {
                    end[a][0] = p < end[a][0] ? p : end[a][0];
                    end[a][1] = p;
                }
            }
        }
        const int pa = end[0][0], pb = end[0][1], ra = end[2][0], rb = end[2][1];
        const gpv::SatScale f = gpv::sat_scale_far(g);
        float4 e[gpv::kSatEntry4];
        bool loose = gpv::sat_entry_part(0, t, C[0][0], C[1][0], C[2][0], f, e);
        loose = gpv::sat_entry_part(1, t, C[0][0], C[1][0], C[2][0], f, e) || loose;
        is_loose[i] = loose;
        for (int q = 0; q < n2; ++q) {
            uint32_t* oi = in + (int64_t)(i * n2 + q) * n2;
            uint32_t* om = may + (int64_t)(i * n2 + q) * n2;
            for (int p = 0; p < n2; ++p) oi[p] = om[p] = 0;
            if (pb < 0 || rb < 0 || q < end[1][0] || q > end[1][1]) continue;
            int p = pa, left = pb - pa + 1;
            gpv::sat_row_range_far(e, pos[1][q], pos[0], half, loose, p, left);
            for (; left > 0; p += piece, left -= piece) {
                gpv::SatRow r = gpv::sat_row_xy(e, pos[1][q], -1e9f, 1e9f, pos[0][p]);
                gpv::sat_row_loose(r, loose, -1, 1 << 30);
                const int m = left < piece ? left : piece;
                for (int k = 0; k < m; ++k)
                    gpv::sat_row_column_far(r, pos[2], half, (2u << rb) - (1u << ra), k + 1 < m ? pos[0][p + k + 1] - pos[0][p + k] : 0.0f,
                                            oi[p + k], om[p + k]);
            }
        }
    }
}

// Level1: case i's index AABB (lo, dd: 3 ints each) on a grid with centers
// cx/cy/cz, bounds lo3/hi3 and voxel g1; per column of it in (q, p) order from
// off[i]: [am, ai, bi, bm).
extern "C" void satcol_batch(int64_t n, const float* tv, const int32_t* lo, const int32_t* dd, const float* cx,
                             const float* cy, const float* cz, const float* lo3, const float* hi3, const float* g1,
                             const int64_t* off, int32_t* out)
{
    gpv::SatScale g;
    gpv::sat_scale_axis(lo3[0], hi3[0], g1[0], false, g.sx, g.dx);
    gpv::sat_scale_axis(lo3[1], hi3[1], g1[1], false, g.sy, g.dy);
    gpv::sat_scale_axis(lo3[2], hi3[2], g1[2], false, g.sz, g.dz);
    for (int64_t i = 0; i < n; ++i) {
        const int32_t *l = lo + 3 * i, *d = dd + 3 * i;
        int32_t* o = out + 4 * off[i];
        for (int q = 0; q < d[1]; ++q)
            for (int p = 0; p < d[0]; ++p, o += 4) {
                const gpv::SatColumn s = gpv::sat_column(tv + 9 * i, cx[l[0]], cy[l[1]], cz[l[2]], g, p, q, d[2]);
                o[0] = s.am; o[1] = s.ai; o[2] = s.bi; o[3] = s.bm;
            }
    }
}

// The box-axis ends of sat_axis_end: n cases, `m` centers each; lo, hi the
// triangle's extent, end = {first, last, clear}.
extern "C" void sataxis_batch(int64_t n, int m, const float* lo, const float* hi, const float* c, const float* bmin,
                              const float* bmax, const float* g2, int cuda, int32_t* end)
{
    for (int64_t i = 0; i < n; ++i) {
        float s, dev;
        gpv::sat_scale_axis(bmin[i], bmax[i], g2[i], cuda != 0, s, dev);
        bool clear = true;
        end[3 * i] = gpv::sat_axis_end((lo[i] - c[m * i]) * s, m, dev, clear);
        end[3 * i + 1] = gpv::sat_axis_end((hi[i] - c[m * i]) * s, m, dev, clear);
        end[3 * i + 2] = clear;
    }
}
