// Host harness for the ray parities' crossing bounds (gpview_amd/csrc/
// gpv_parcol.hpp): tests/test_parity_columns.py compares them with the float
// ray test.  Test tooling only.
#include <stdint.h>
#include "gpv_parcol.hpp"

// Case i: triangle tv[9i..] and a column with origins ox/oy[n2*i..]; oz[nl]
// the layer origins of the grid, l0[i] the first layer of the record's voxel.
// out[6i..]: accepted sub-columns, accepted ones outside the candidate range,
// candidates, (accepted, layer) tests that contradict the certain layers or
// crossings outside the entry's z range,
// undecided layers, det rejected.
extern "C" void parcol_batch(int64_t n, int n2, int nl, const float* tv, const float* ox, const float* oy,
                             const float* oz, const int32_t* l0, const float* lo, const float* hi, const float* g2,
                             const float* h, const float* g1z, int cuda_l2, uint32_t eps_bits, int64_t* out)
{
    float eps;
    __builtin_memcpy(&eps, &eps_bits, 4);
    for (int64_t i = 0; i < n; ++i) {
        const float* t = tv + 9 * i;
        const float *X = ox + (int64_t)n2 * i, *Y = oy + (int64_t)n2 * i;
        int64_t* o = out + 6 * i;
        gpv::SatScale g;
        gpv::sat_scale_axis(lo[3 * i], hi[3 * i], g2[3 * i], cuda_l2 != 0, g.sx, g.dx);
        gpv::sat_scale_axis(lo[3 * i + 1], hi[3 * i + 1], g2[3 * i + 1], cuda_l2 != 0, g.sy, g.dy);
        gpv::sat_scale_axis(lo[3 * i + 2], hi[3 * i + 2], g2[3 * i + 2], cuda_l2 != 0, g.sz, g.dz);
        gpv::ParEntry r;
        r.e1x = t[3] - t[0]; r.e1y = t[4] - t[1]; r.e1z = t[5] - t[2];
        r.e2x = t[6] - t[0]; r.e2y = t[7] - t[1]; r.e2z = t[8] - t[2];
        const float px = 0.0f * r.e2z - r.e2y, py = r.e2x - 0.0f * r.e2z, pz = 0.0f * r.e2y - 0.0f * r.e2x;
        const float det = r.e1x * px + r.e1y * py + r.e1z * pz;
        if ((double)det > -1e-6 && (double)det < 1e-6) {
            o[5] = 1;
            continue;
        }
        r.inv = 1.f / det;
        r.v1x = t[0]; r.v1y = t[1];
        r.l0 = l0[i];
        gpv::par_entry(r, t[2], gpv::par_oz(lo[3 * i + 2], g1z[i], g2[3 * i + 2], l0[i] / n2), X[0], Y[0], 2.0f * h[3 * i], 2.0f * h[3 * i + 1], n2, g);
        int q0, zlo, zhi;
        gpv::par_z_range(r, g.sz, nl, zlo, zhi);
        const int nq = gpv::par_rows(r, Y[0], g.sy, n2, g.dy, q0);
        for (int q = 0; q < n2; ++q) {
            int p0 = 0, np = 0;
            const bool row = q >= q0 && q < q0 + nq;
            if (row) np = gpv::par_cols(r, X[0], Y[0], 2.0f * h[3 * i], 2.0f * h[3 * i + 1], n2, q, p0);
            for (int p = 0; p < n2; ++p) {
                const bool cand = row && p >= p0 && p < p0 + np;
                o[2] += cand;
                const float tx = X[p] - t[0], ty = Y[q] - t[1];
                const float u = (tx * px + ty * py) * r.inv;
                const float qz = tx * r.e1y - ty * r.e1x;
                const float v = qz * r.inv;
                if ((u < 0.f) | (u > 1.f) | (v < 0.f) | (u + v > 1.f)) continue;
                ++o[0];
                if (!cand) {
                    ++o[1];
                    continue;
                }
                int la, lb;
                gpv::par_layers(r, u, v, g.sz, nl, la, lb);
                o[4] += lb - la;
                o[3] += la < zlo || lb > zhi;
                for (int l = 0; l < nl; ++l) {
                    const float tz = oz[l] - t[2];
                    const float qx = ty * r.e1z - tz * r.e1y, qy = tz * r.e1x - tx * r.e1z;
                    const bool hit = (r.e2x * qx + r.e2y * qy + r.e2z * qz) * r.inv >= eps;
                    if (l < la ? !hit : l >= lb ? hit : false) ++o[3];
                }
            }
        }
    }
}

// parcol_batch with the positions taken from the tables (grids far from the origin).
extern "C" void parcol_far(int64_t n, int n2, int nl, const float* tv, const float* ox, const float* oy,
                           const float* oz, const int32_t* l0, const float* lo, const float* hi, const float* g2,
                           const float* h, const float* g1z, int cuda_l2, uint32_t eps_bits, int64_t* out)
{
    float eps;
    __builtin_memcpy(&eps, &eps_bits, 4);
    for (int64_t i = 0; i < n; ++i) {
        const float* t = tv + 9 * i;
        const float *X = ox + (int64_t)n2 * i, *Y = oy + (int64_t)n2 * i;
        int64_t* o = out + 6 * i;
        gpv::SatScale g;
        gpv::sat_scale_axis(lo[3 * i], hi[3 * i], g2[3 * i], cuda_l2 != 0, g.sx, g.dx);
        gpv::sat_scale_axis(lo[3 * i + 1], hi[3 * i + 1], g2[3 * i + 1], cuda_l2 != 0, g.sy, g.dy);
        gpv::sat_scale_axis(lo[3 * i + 2], hi[3 * i + 2], g2[3 * i + 2], cuda_l2 != 0, g.sz, g.dz);
        gpv::ParEntry r;
        r.e1x = t[3] - t[0]; r.e1y = t[4] - t[1]; r.e1z = t[5] - t[2];
        r.e2x = t[6] - t[0]; r.e2y = t[7] - t[1]; r.e2z = t[8] - t[2];
        const float px = 0.0f * r.e2z - r.e2y, py = r.e2x - 0.0f * r.e2z, pz = 0.0f * r.e2y - 0.0f * r.e2x;
        const float det = r.e1x * px + r.e1y * py + r.e1z * pz;
        if ((double)det > -1e-6 && (double)det < 1e-6) {
            o[5] = 1;
            continue;
        }
        r.inv = 1.f / det;
        r.v1x = t[0]; r.v1y = t[1];
        r.l0 = l0[i];
        const float gx = 2.0f * h[3 * i], gy = 2.0f * h[3 * i + 1];
        gpv::par_entry(r, t[2], gpv::par_oz(lo[3 * i + 2], g1z[i], g2[3 * i + 2], l0[i] / n2), X[0], Y[0], gx, gy, n2, g);
        int q0, zlo, zhi;
        r.delta = gpv::par_delta_far(r, X[0], Y[0], gx, gy, n2, g);
        const bool scaled = g.dx >= 0.0f && g.dy >= 0.0f && g.dz >= 0.0f;
        const float ez = scaled ? gpv::par_ez(r.e1x, r.e1y, r.e1z, r.e2x, r.e2y, r.e2z, r.inv) : 3.0e38f;
        r.mu = gpv::par_mu_far(ez, g, nl);
        gpv::par_z_range(r, g.sz, nl, zlo, zhi);
        const int nq = gpv::par_rows_far(r, Y, g.sy, n2, q0);
        for (int q = 0; q < n2; ++q) {
            int p0 = 0, np = 0;
            const bool row = q >= q0 && q < q0 + nq;
            if (row) np = gpv::par_cols_far(r, X, Y[q], gx, n2, p0);
            for (int p = 0; p < n2; ++p) {
                const bool cand = row && p >= p0 && p < p0 + np;
                o[2] += cand;
                const float tx = X[p] - t[0], ty = Y[q] - t[1];
                const float u = (tx * px + ty * py) * r.inv;
                const float qz = tx * r.e1y - ty * r.e1x;
                const float v = qz * r.inv;
                if ((u < 0.f) | (u > 1.f) | (v < 0.f) | (u + v > 1.f)) continue;
                ++o[0];
                if (!cand) {
                    ++o[1];
                    continue;
                }
                int la, lb;
                gpv::par_layers(r, u, v, g.sz, nl, la, lb);
                o[3] += la < zlo || lb > zhi;
                const int wa = la, wb = lb;
                if (lb - la > 1) {
                    const float zc = (u * r.e1z + v * r.e2z) - 1.0e-6f;
                    gpv::par_narrow(oz, n2, 1.0f / (float)n2, t[2], zc - 2.0f * ez, zc + 2.0f * ez, la, lb);
                }
                o[3] += la < wa || lb > wb || lb < la;
                o[4] += lb - la;
                for (int l = 0; l < nl; ++l) {
                    const float tz = oz[l] - t[2];
                    const float qx = ty * r.e1z - tz * r.e1y, qy = tz * r.e1x - tx * r.e1z;
                    const bool hit = (r.e2x * qx + r.e2y * qy + r.e2z * qz) * r.inv >= eps;
                    if (l < la ? !hit : l >= lb ? hit : false) ++o[3];
                }
            }
        }
    }
}

// Level1: case i, triangle tv[9i..] and a column (ox[i], oy[i]) over the layer
// origins oz[nl] of a grid from zmin to zmax.  out[4i..]: accepted, layers that
// contradict the certain ones, undecided layers, layers that pass.
extern "C" void parl1_batch(int64_t n, int nl, const float* tv, const float* ox, const float* oy, const float* oz,
                            float zmin, float zmax, uint32_t eps_bits, int64_t* out)
{
    float eps;
    __builtin_memcpy(&eps, &eps_bits, 4);
    for (int64_t i = 0; i < n; ++i) {
        const float* t = tv + 9 * i;
        int64_t* o = out + 4 * i;
        const float e1x = t[3] - t[0], e1y = t[4] - t[1], e1z = t[5] - t[2];
        const float e2x = t[6] - t[0], e2y = t[7] - t[1], e2z = t[8] - t[2];
        const float px = 0.0f * e2z - e2y, py = e2x - 0.0f * e2z, pz = 0.0f * e2y - 0.0f * e2x;
        const float det = e1x * px + e1y * py + e1z * pz;
        if ((double)det > -1e-6 && (double)det < 1e-6) continue;
        const float inv = 1.f / det;
        const float tx = ox[i] - t[0], ty = oy[i] - t[1];
        const float u = (tx * px + ty * py) * inv, v = (tx * e1y - ty * e1x) * inv;
        if ((u < 0.f) | (u > 1.f) | (v < 0.f) | (u + v > 1.f)) continue;
        o[0] = 1;
        int la, lb;
        gpv::par_l1_layers(oz, nl, zmin, (float)nl / (zmax - zmin), t[2], e1z, e2z, u, v,
                           gpv::par_ez(e1x, e1y, e1z, e2x, e2y, e2z, inv), la, lb);
        o[1] += la < 0 || lb < la || lb > nl;
        o[2] = lb - la;
        for (int l = 0; l < nl; ++l) {
            const float tz = oz[l] - t[2];
            const float qx = ty * e1z - tz * e1y, qy = tz * e1x - tx * e1z, qz = tx * e1y - ty * e1x;
            const bool hit = (e2x * qx + e2y * qy + e2z * qz) * inv >= eps;
            o[1] += l < la ? !hit : l >= lb ? hit : false;
            o[3] += hit;
        }
    }
}
