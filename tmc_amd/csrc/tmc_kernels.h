// tmc_kernels.h -- topologically correct Marching Cubes on the GPU
// (mc/MarchingCubes.cpp: t_mc :150-318, p_slice :322-1303; the CUDA
// counterpart is cuda_tmc/MarchingCubes.cu t_slice :1366).
//
// The active cells come from the DMC sweep (same classification, f >= iso,
// same per-(row, segment) lists, whose flat order is the reference's
// (k, j, i) cell order).  Then:
//   k_tmc_cells      each active cell's word: case, the cut edges it owns,
//                    table triangles; the ambiguous cells listed;
//   k_tmc_amb_count  the listed cells' inner vertices and triangles from the
//                    decider slicing (kept out of the cell walk, where one
//                    ambiguous lane would hold up its wave);
//   scans            over the active cells: each cell's first vertex and
//                    triangle -- the reference's numbering, first sight in
//                    cell order;
//   k_tmc_emit       positions and normals of the cells' edge vertices, and
//                    the table triangles of the non-ambiguous cells;
//   k_tmc_emit_amb   inner vertices and triangles of the listed cells.
// A grid edge is owned by the first cell containing it in (k, j, i) order;
// that cell is active because the edge is cut, so its active index is found
// from the sweep's activity words.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "dmc_extract_kernels.h"
#include "tmc_mc_tables.h"

namespace tmc {

__device__ __constant__ uint64_t c_tmc_tri[256] = TMC_CASE_TRIANGLES_INIT;
__device__ __constant__ uint64_t c_tmc_amb[4] = TMC_AMBIGUOUS_MASK_INIT;

// Edge e: end corners (corner c = i + 2 j + 4 k) packed as v0 | v1 << 4, the
// lower one first (mc/MarchingCubes.cpp:153-159).
__device__ __constant__ uint8_t c_tmc_ev[12] = {0x10, 0x31, 0x32, 0x20, 0x54, 0x75, 0x76, 0x64, 0x40, 0x51, 0x73, 0x62};
// faces seen from outside: corners and edges in oriented order
// (mc/MarchingCubes.h:84-107), one nibble each
__device__ __constant__ uint16_t c_tmc_fv[6] = {0x3120, 0x6475, 0x1504, 0x7362, 0x2064, 0x7531};
__device__ __constant__ uint16_t c_tmc_fe[6] = {0x0123, 0x4765, 0x4908, 0x2A6B, 0x83B7, 0x95A1};
// local coordinates of the edge points per axis: 2 bits per edge, 3 = along
// the edge (mc/MarchingCubes.cpp:896-903)
constexpr unsigned kTmcLCoord[3] = {1324855u, 5299420u, 16733440u};

__device__ __forceinline__ bool tmc_ambiguous(unsigned icase) { return (c_tmc_amb[icase >> 6] >> (icase & 63)) & 1ull; }

// Cut edges of a case: x-edges 0 2 4 6 join corners that differ in bit 0,
// y-edges 3 1 7 5 in bit 1, z-edges 8 9 11 10 in bit 2.
__device__ __forceinline__ unsigned tmc_cut_mask(unsigned icase) {
    const unsigned x = icase ^ (icase >> 1), y = icase ^ (icase >> 2), z = icase ^ (icase >> 4);
    return (x & 0x55u) | (y & 2u) | (y & 1u) << 3 | (y & 0x20u) | (y & 0x10u) << 3 | (z & 3u) << 8 | (z & 8u) << 7 |
           (z & 4u) << 9;
}

// Edges of cell (i, j, k) that it owns (it is their first cell): the three
// that meet the far corner, and those that the grid's lower sides leave
// without an earlier cell.
__device__ __forceinline__ unsigned tmc_owned_mask(int i, int j, int k) {
    const unsigned i0 = i == 0, j0 = j == 0, k0 = k == 0;
    return (1u << 5 | 1u << 6 | 1u << 10) | k0 * (1u << 1 | 1u << 2) | j0 * (1u << 4 | 1u << 9) |
           i0 * (1u << 7 | 1u << 11) | (j0 & k0) | (i0 & k0) << 3 | (i0 & j0) << 8;
}

// An active cell's word: case (bits 0-7), "no triangles" (bit 8, a singular
// face), inner vertices (9-11), owned cut edges (12-23), triangles (24-31).
__device__ __forceinline__ unsigned tmc_own(uint32_t code) { return (code >> 12) & 0xFFFu; }
__device__ __forceinline__ unsigned tmc_new_vertices(uint32_t code) {
    return (unsigned)__popc(code & 0xFFF000u) + ((code >> 9) & 7u);
}
// Their scans: new vertices, triangles.
template <bool TRIS>
struct ScanTmc {
    static constexpr bool kMap = false;
    const uint32_t* p;
    __device__ __forceinline__ static uint32_t of(uint32_t w) { return TRIS ? w >> 24 : tmc_new_vertices(w); }
    __device__ __forceinline__ uint32_t at(int64_t i) const { return of(p[i]); }
    __device__ __forceinline__ void vec16(int64_t base, uint32_t v[kScanIPT]) const {
#pragma unroll
        for (int q = 0; q < kScanIPT / 4; q++) {
            const uint4 t = reinterpret_cast<const uint4*>(p + base)[q];
            v[4 * q] = of(t.x);
            v[4 * q + 1] = of(t.y);
            v[4 * q + 2] = of(t.z);
            v[4 * q + 3] = of(t.w);
        }
    }
};

__device__ __forceinline__ double tmc_decider(double f0, double f1, double f2, double f3) {
    return (f0 * f3 - f1 * f2) / (f0 + f3 - f1 - f2);
}

// p_slice: contours of an ambiguous cell from the face deciders, then its
// triangles (local refs: 0..11 edge vertices, 12..17 inner vertices) and
// inner vertices (local coordinates), handed to `em` in the reference's
// order.  Returns false where a singular face cannot be triangulated: the
// reference then leaves the cell without triangles.
template <class Emit>
__device__ bool tmc_slice(const double F[8], unsigned icase, double i0, Emit& em) {
    double ecoord[12];
#pragma unroll
    for (int e = 0; e < 12; e++) {
        const unsigned a = c_tmc_ev[e] & 0xF, b = c_tmc_ev[e] >> 4;
        ecoord[e] = (((icase >> a) ^ (icase >> b)) & 1u) ? (i0 - F[a]) / (F[b] - F[a]) : 0.0;
    }
    int8_t to[12];
#pragma unroll
    for (int e = 0; e < 12; e++) to[e] = -1;
    bool f_flag[6];
    for (int f = 0; f < 6; f++) {
        f_flag[f] = false;
        const unsigned fv = c_tmc_fv[f], fe = c_tmc_fe[f];
        const double f0 = F[fv & 0xF], f1 = F[(fv >> 4) & 0xF], f2 = F[(fv >> 8) & 0xF], f3 = F[fv >> 12];
        const int e0 = fe & 0xF, e1 = (fe >> 4) & 0xF, e2 = (fe >> 8) & 0xF, e3 = fe >> 12;
        const int fc = (f0 >= i0) | (f1 >= i0) << 1 | (f2 >= i0) << 2 | (f3 >= i0) << 3;
        switch (fc) {
        case 1: to[e0] = e3; break;
        case 2: to[e1] = e0; break;
        case 3: to[e1] = e3; break;
        case 4: to[e3] = e2; break;
        case 5: to[e0] = e2; break;
        case 6:
        case 9: {
            const double val = tmc_decider(f0, f1, f2, f3);
            bool sep;   // the pairing of val > i0
            if (val > i0) sep = true;
            else if (val < i0) sep = false;
            else {
                f_flag[f] = true;
                const unsigned e_flag = 0x218;
                double c0 = ecoord[e0], c1 = ecoord[e1], c2 = ecoord[e2], c3 = ecoord[e3];
                if ((e_flag >> (f * 2)) & 1u) { c0 = 1 - c0; c2 = 1 - c2; }
                if ((e_flag >> (f * 2)) & 2u) { c1 = 1 - c1; c3 = 1 - c3; }
                if (c1 < c3 && c0 > c2) sep = fc != 6;
                else if (c1 > c3 && c0 < c2) sep = fc == 6;
                else return false;
            }
            if (fc == 6) {
                if (sep) { to[e3] = e0; to[e1] = e2; }
                else { to[e1] = e0; to[e3] = e2; }
            } else {
                if (sep) { to[e0] = e1; to[e2] = e3; }
                else { to[e0] = e3; to[e2] = e1; }
            }
        } break;
        case 7: to[e1] = e2; break;
        case 8: to[e2] = e1; break;
        case 10: to[e2] = e0; break;
        case 11: to[e2] = e3; break;
        case 12: to[e3] = e1; break;
        case 13: to[e0] = e1; break;
        case 14: to[e3] = e0; break;
        default: break;
        }
    }
    // closed contours, each started at its smallest edge: edges packed 4
    // bits each in walk order, contour c from bit 4 * cst[c]
    int cnt = 0;
    int csz[4] = {0, 0, 0, 0}, cst[4] = {0, 0, 0, 0};
    uint64_t cedge = 0;
    int used_slots = 0;
    for (int e = 0; e < 12 && cnt < 4; e++) {
        if (to[e] < 0) continue;
        cst[cnt] = used_slots;
        int pos = 0, t = to[e];
        cedge |= (uint64_t)e << (4 * (used_slots + pos));
        // every cut edge has one outgoing and one incoming segment, so the
        // walk closes; the bounds only keep a malformed case in range
        while (t != e && t >= 0 && used_slots + pos < 11) {
            pos++;
            cedge |= (uint64_t)t << (4 * (used_slots + pos));
            const int nx = to[t];
            to[t] = -1;
            t = nx;
        }
        csz[cnt] = pos + 1;
        used_slots += pos + 1;
        cnt++;
    }
    auto ce = [&](int c, int r) { return (int)((cedge >> (4 * (cst[c] + r))) & 0xF); };

    double ui[2] = {0, 0}, vi[2] = {0, 0}, wi[2] = {0, 0};
    unsigned q_sol = 0;
    const double a = (F[0] - F[1]) * (-F[6] + F[7] + F[4] - F[5]) - (F[4] - F[5]) * (-F[2] + F[3] + F[0] - F[1]);
    const double b = (i0 - F[0]) * (-F[6] + F[7] + F[4] - F[5]) + (F[0] - F[1]) * (F[6] - F[4]) -
                     (i0 - F[4]) * (-F[2] + F[3] + F[0] - F[1]) - (F[4] - F[5]) * (F[2] - F[0]);
    const double c = (i0 - F[0]) * (F[6] - F[4]) - (i0 - F[4]) * (F[2] - F[0]);
    double disc = b * b - 4 * a * c;
    if (disc > 0) {
        disc = sqrt(disc);
        ui[0] = (-b - disc) / (2 * a);
        ui[1] = (-b + disc) / (2 * a);
        for (int s = 0; s < 2; s++) {
            const double g1 = F[0] * (1 - ui[s]) + F[1] * ui[s];
            const double g2 = F[2] * (1 - ui[s]) + F[3] * ui[s];
            vi[s] = (i0 - g1) / (g2 - g1);
            if (isnan(vi[s]) || isinf(vi[s])) vi[s] = -1.0;
        }
        for (int s = 0; s < 2; s++) {
            const double g1 = F[0] * (1 - ui[s]) + F[1] * ui[s];
            const double g2 = F[4] * (1 - ui[s]) + F[5] * ui[s];
            wi[s] = (i0 - g1) / (g2 - g1);
            if (isnan(wi[s]) || isinf(wi[s])) wi[s] = -1.0;
        }
        if (f_flag[0]) { if (wi[0] < wi[1]) wi[0] = 0; else wi[1] = 0; }
        if (f_flag[1]) wi[1] = 1;   // both branches of the reference set wi[1]
        if (f_flag[2]) { if (vi[0] < vi[1]) vi[0] = 0; else vi[1] = 0; }
        if (f_flag[3]) { if (vi[0] > vi[1]) vi[0] = 1; else vi[1] = 1; }
        if (f_flag[4]) { if (ui[0] < ui[1]) ui[0] = 0; else ui[1] = 0; }
        if (f_flag[5]) { if (ui[0] > ui[1]) ui[0] = 1; else ui[1] = 1; }
        q_sol |= (0 < ui[0] && ui[0] < 1) ? 1u : 0u;
        q_sol |= (0 < ui[1] && ui[1] < 1) ? 2u : 0u;
        q_sol |= (0 < vi[0] && vi[0] < 1) ? 4u : 0u;
        q_sol |= (0 < vi[1] && vi[1] < 1) ? 8u : 0u;
        q_sol |= (0 < wi[0] && wi[0] < 1) ? 16u : 0u;
        q_sol |= (0 < wi[1] && wi[1] < 1) ? 32u : 0u;
    }
    auto ev = [&](int e, int x) {
        const unsigned fl = (kTmcLCoord[x] >> (2 * e)) & 3u;
        return fl == 3u ? ecoord[e] : (double)fl;
    };
    if (__popc(q_sol) == 6) {
        // tunnel, or one contour with 12 vertices: the inner hexagon
        const double hu[6] = {ui[0], ui[0], ui[1], ui[1], ui[1], ui[0]};
        const double hv[6] = {vi[0], vi[0], vi[0], vi[1], vi[1], vi[1]};
        const double hw[6] = {wi[0], wi[1], wi[1], wi[1], wi[0], wi[0]};
        int not_tunnel = 0xF;
        if (cnt == 3) {
            const double uc_min = (ui[0] < ui[1]) ? ui[0] : ui[1];
            const double uc_max = (ui[0] < ui[1]) ? ui[1] : ui[0];
            for (int t = 0; t < cnt; t++) {
                if (csz[t] != 3) continue;
                double umin = 2, umax = -2;
                const int x0 = ce(t, 0), x1 = ce(t, 1), x2 = ce(t, 2);
                const double u0 = ev(x0, 0), u1 = ev(x1, 0), u2 = ev(x2, 0);
                umin = (u0 < umin) ? u0 : umin;
                umin = (u1 < umin) ? u1 : umin;
                umin = (u2 < umin) ? u2 : umin;
                umax = (u0 > umax) ? u0 : umax;
                umax = (u1 > umax) ? u1 : umax;
                umax = (u2 > umax) ? u1 : umax;   // the reference takes u1 here
                if (uc_min > umax || uc_max < umin) {
                    not_tunnel = t;
                    em.tri(x0, x1, x2);
                }
            }
        }
        for (int s = 0; s < 6; s++) em.inner(s, hu[s], hv[s], hw[s]);
        uint64_t tcon = 0;   // nearest hexagon vertex of each contour edge, 4 bits per edge
        for (int t = 0; t < cnt; t++) {
            if (not_tunnel == t) continue;
            const int sz = csz[t];
            for (int r = 0; r < sz; r++) {
                unsigned index = 0xFu;
                double dist = 1000.;
                const int ci = ce(t, r);
                const double ue = ev(ci, 0), ve = ev(ci, 1), we = ev(ci, 2);
                for (int s = 0; s < 6; s++) {
                    const double du = ue - hu[s], dv = ve - hv[s], dw = we - hw[s];
                    const double val = du * du + dv * dv + dw * dw;
                    if (dist > val) {
                        index = (unsigned)s;
                        dist = val;
                    }
                }
                tcon = (tcon & ~(0xFull << (4 * ci))) | ((uint64_t)index << (4 * ci));
            }
            for (int r = 0; r < sz; r++) {
                const int t1 = ce(t, r), t2 = ce(t, (r + 1) % sz);
                const int c1 = (int)((tcon >> (4 * t1)) & 0xF), c2 = (int)((tcon >> (4 * t2)) & 0xF);
                if (c1 > 5 || c2 > 5) continue;   // no nearest vertex (not reached with finite coordinates)
                int dst = c1 - c2 < 0 ? c2 - c1 : c1 - c2;
                if (dst > 2) dst = 6 - dst;
                if (dst == 0) {
                    em.tri(t1, t2, 12 + c1);
                } else if (dst == 1) {
                    const double l1 = (ev(t1, 0) - hu[c2]) * (ev(t1, 0) - hu[c2]) + (ev(t1, 1) - hv[c2]) * (ev(t1, 1) - hv[c2]) +
                                      (ev(t1, 2) - hw[c2]) * (ev(t1, 2) - hw[c2]);
                    const double l2 = (ev(t2, 0) - hu[c1]) * (ev(t2, 0) - hu[c1]) + (ev(t2, 1) - hv[c1]) * (ev(t2, 1) - hv[c1]) +
                                      (ev(t2, 2) - hw[c1]) * (ev(t2, 2) - hw[c1]);
                    if (l1 < l2) {
                        em.tri(t1, t2, 12 + c2);
                        em.tri(t1, 12 + c2, 12 + c1);
                    } else {
                        em.tri(t1, t2, 12 + c1);
                        em.tri(t2, 12 + c2, 12 + c1);
                    }
                } else if (dst == 2) {
                    const int dmax = c1 > c2 ? c1 : c2, dmin = c1 < c2 ? c1 : c2;
                    const int cm = ((dmax + 2) % 6 == dmin) ? (dmax + 1) % 6 : (dmax + dmin) / 2;
                    em.tri(t1, t2, 12 + cm);
                    em.tri(t1, 12 + cm, 12 + c1);
                    em.tri(t2, 12 + c2, 12 + cm);
                }
            }
        }
        if (cnt == 1) {
            const bool s_ = tmc_decider(F[0], F[1], F[2], F[3]) <= i0;
            const bool of_ = (wi[1] < wi[0]) ? s_ : !s_;
            if (!of_) {
                em.tri(12, 14, 13);
                em.tri(14, 16, 15);
                em.tri(12, 17, 16);
                em.tri(12, 16, 14);
            } else {
                em.tri(12, 13, 14);
                em.tri(14, 15, 16);
                em.tri(12, 16, 17);
                em.tri(12, 14, 16);
            }
        }
        return true;
    }
    const unsigned nr_u = ((q_sol & 0x5u) == 0x5u) + ((q_sol & 0xAu) == 0xAu);
    const unsigned nr_v = ((q_sol & 0x11u) == 0x11u) + ((q_sol & 0x22u) == 0x22u);
    const unsigned nr_w = ((q_sol & 0x18u) == 0x18u) + ((q_sol & 0x24u) == 0x24u);
    const unsigned nr_t = nr_u + nr_v + nr_w;
    if (nr_t == nr_u || nr_t == nr_v || nr_t == nr_w) {
        // no saddle point inside: fans of the contours of 3 to 6 edges
        for (int t = 0; t < cnt; t++) {
            const int c0 = ce(t, 0), c1 = ce(t, 1), c2 = ce(t, 2);
            switch (csz[t]) {
            case 3: em.tri(c0, c1, c2); break;
            case 4:
                em.tri(c0, c1, c2);
                em.tri(c0, c2, ce(t, 3));
                break;
            case 5:
                em.tri(c0, c1, c2);
                em.tri(c0, c2, ce(t, 3));
                em.tri(c0, ce(t, 3), ce(t, 4));
                break;
            case 6:
                em.tri(c0, c1, ce(t, 3));
                em.tri(c1, c2, ce(t, 3));
                em.tri(c0, ce(t, 3), ce(t, 4));
                em.tri(c0, ce(t, 4), ce(t, 5));
                break;
            default: break;
            }
        }
        return true;
    }
    // one inner vertex, joined to the contours of more than three edges
    const unsigned f00 = q_sol & 1u, f01 = (q_sol >> 1) & 1u, f10 = (q_sol >> 2) & 1u, f11 = (q_sol >> 3) & 1u,
                   f20 = (q_sol >> 4) & 1u, f21 = (q_sol >> 5) & 1u;
    const double d00 = f00, d01 = f01, d10 = f10, d11 = f11, d20 = f20, d21 = f21;
    const unsigned fc1 = f00 * f10 + f01 * f11, fc2 = f00 * f20 + f01 * f21, fc3 = f10 * f21 + f11 * f20;
    double uc = 0, vc = 0, wc = 0;
    switch (fc1 + fc2 + fc3) {
    case 2:
        if (fc1 == 0) {
            uc = d00 * ui[0] + d01 * ui[1];
            vc = d10 * vi[0] + d11 * vi[1];
            wc = d10 * wi[1] + d11 * wi[0];
        } else if (fc2 == 0) {
            uc = d00 * ui[0] + d01 * ui[1];
            vc = d00 * vi[0] + d01 * vi[1];
            wc = d00 * wi[1] + d01 * wi[0];
        } else if (fc3 == 0) {
            uc = d10 * ui[0] + d11 * ui[1];
            vc = d10 * vi[0] + d11 * vi[1];
            wc = d10 * wi[0] + d11 * wi[1];
        }
        break;
    case 3:
        uc = (d00 * ui[0] + d01 * ui[1]) / (double)(f00 + f01);
        vc = (d10 * vi[0] + d11 * vi[1]) / (double)(f10 + f11);
        wc = (d20 * wi[0] + d21 * wi[1]) / (double)(f20 + f21);
        break;
    case 4:
        if (f20 + f21 == 1) {
            uc = d20 * ui[0] + d21 * ui[1];
            vc = d21 * vi[0] + d20 * vi[1];
            wc = d20 * wi[0] + d21 * wi[1];
        } else if (f10 + f11 == 1) {
            uc = d10 * ui[0] + d11 * ui[1];
            vc = d10 * vi[0] + d11 * vi[1];
            wc = d11 * wi[0] + d10 * wi[1];
        } else if (f00 + f01 == 1) {
            uc = d00 * ui[0] + d01 * ui[1];
            vc = d00 * vi[0] + d01 * vi[1];
            wc = d00 * wi[0] + d01 * wi[1];
        }
        break;
    default: break;
    }
    bool used = false;
    for (int t = 0; t < cnt; t++) {
        const int sz = csz[t];
        if (sz == 3) {
            em.tri(ce(t, 0), ce(t, 1), ce(t, 2));
        } else {
            used = true;
            for (int r = 0; r < sz; r++) em.tri(ce(t, r), ce(t, (r + 1) % sz), 12);
        }
    }
    if (used) em.inner(0, uc, vc, wc);
    return true;
}

// Counting emitter: triangles and inner vertices of a cell.
struct TmcCount {
    int nt = 0, ninner = 0;
    __device__ void tri(int, int, int) { nt++; }
    __device__ void inner(int s, double, double, double) { ninner = s + 1 > ninner ? s + 1 : ninner; }
};

// Corner values of cell (i, j, k) as doubles.
template <class T>
__device__ __forceinline__ void tmc_corners(const T* __restrict__ field, const Dims& d, int i, int j, int k,
                                            double F[8]) {
    const int64_t sy = d.nx, sz = (int64_t)d.nx * d.ny;
    const T* p = field + (int64_t)k * sz + (int64_t)j * sy + i;
#pragma unroll
    for (int c = 0; c < 8; c++) F[c] = (double)p[(c & 1) + ((c >> 1) & 1) * sy + (c >> 2) * sz];
}

// K_T1: one wave per group of (row, segment)s as in k_cells, cells in the
// flat active order: per active cell its cell index and its word.  Ambiguous
// cells are listed (amb[0] = count, from amb[1]): a wave gathers them in LDS
// and a block adds them to the list at its end (an add per wave and turn made
// the counter's queue half of this kernel: 625 us at 1024^3, now 307).
constexpr int kTmcAmb = 256;             // ambiguous cells a wave holds
constexpr int kTmcCellsBlocks = 4096;    // at most: the blocks' adds to the counter
__global__ void __launch_bounds__(kBlock) k_tmc_cells(VolTable vt, int64_t groups, const uint32_t* __restrict__ lists,
                                                       const uint32_t* __restrict__ segCount,
                                                       const uint32_t* __restrict__ segBase,
                                                       uint32_t* __restrict__ acell, uint32_t* __restrict__ acode,
                                                       uint32_t* __restrict__ amb) {
    __shared__ uint32_t s_amb[kBlock / kWave][kTmcAmb];
    __shared__ uint32_t s_n[kBlock / kWave], s_base;
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int64_t wpb = kBlock / kWave;
    uint32_t* held = s_amb[wave];
    uint32_t nheld = 0;   // wave-uniform
    const VolDesc V = vt.desc[0];   // a copy: the list's stores could otherwise change it
    const Dims d = V.d;
    for (int64_t g = (int64_t)blockIdx.x * wpb + __builtin_amdgcn_readfirstlane(wave); g < groups;
         g += (int64_t)gridDim.x * wpb) {
        const GroupLanes L = load_group(V, g, lane, segCount, segBase);
        for (uint32_t x0 = 0; x0 < L.total; x0 += kWave) {
            const uint32_t x = x0 + lane, a = L.first + x;
            const int s = group_seg(L, x);
            const uint32_t rel = (uint32_t)__shfl((int)L.rel, s, kWave);
            const int j = __shfl(L.j, s, kWave), k = __shfl(L.k, s, kWave);
            bool isamb = false;
            if (x < L.total) {
                const uint32_t e = lists[((g << V.gsh) + s) * kSeg + (x - rel)];
                const int i = (int)(e & 0xFFFFFFu);
                const unsigned icase = e >> 24;
                isamb = tmc_ambiguous(icase);
                const uint32_t nt = isamb ? 0u : (uint32_t)(c_tmc_tri[icase] >> 60);
                acell[a] = ((uint32_t)k * (uint32_t)(d.ny - 1) + (uint32_t)j) * (uint32_t)d.C + (uint32_t)i;
                acode[a] = icase | (tmc_cut_mask(icase) & tmc_owned_mask(i, j, k)) << 12 | nt << 24;
            }
            const uint64_t m = __ballot(isamb);
            if (m) {
                if (isamb)
                    held[nheld + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                                           __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u))] = a;
                nheld += (uint32_t)__popcll(m);
                if (nheld > kTmcAmb - kWave) {   // no room for another turn
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    uint32_t base = 0;
                    if (lane == 0) base = atomicAdd(amb, nheld);
                    base = (uint32_t)__shfl((int)base, 0, kWave);
                    for (uint32_t y = lane; y < nheld; y += kWave) amb[1 + base + y] = held[y];
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    nheld = 0;
                }
            }
        }
    }
    if (lane == 0) s_n[wave] = nheld;
    __syncthreads();
    uint32_t at = 0, all = 0;
#pragma unroll
    for (int w = 0; w < kBlock / kWave; w++) {
        if (w < wave) at += s_n[w];
        all += s_n[w];
    }
    if (all == 0) return;
    if (threadIdx.x == 0) s_base = atomicAdd(amb, all);
    __syncthreads();
    for (uint32_t y = lane; y < nheld; y += kWave) amb[1 + s_base + at + y] = held[y];
}

// K_T2: the listed ambiguous cells' inner vertices and triangles from the
// decider slicing, into the cell's word; bit 8 marks one whose singular face
// could not be triangulated (no triangles), counted in stats[0].
template <class T>
__global__ void __launch_bounds__(kBlock) k_tmc_amb_count(VolTable vt, const uint32_t* __restrict__ amb,
                                                           const uint32_t* __restrict__ acell,
                                                           uint32_t* __restrict__ acode,
                                                           unsigned long long* __restrict__ stats) {
    const uint32_t n = amb[0];
    const VolDesc& V = vt.desc[0];
    for (uint32_t s = blockIdx.x * kBlock + threadIdx.x; s < n; s += gridDim.x * kBlock) {
        const uint32_t a = amb[1 + s];
        int i, j, k;
        uint32_t r;
        cell_ijk(acell[a], V.d, i, j, k, r);
        const uint32_t code = acode[a];
        double F[8];
        tmc_corners(static_cast<const T*>(V.field), V.d, i, j, k, F);
        TmcCount c;
        if (tmc_slice(F, code & 0xFFu, V.iso, c)) {
            acode[a] = code | (uint32_t)c.ninner << 9 | (uint32_t)c.nt << 24;
        } else {
            acode[a] = code | 0x100u;
            atomicAdd(&stats[0], 1ull);
        }
    }
}

// Gradient at corner c of cell (i, j, k): central differences inside the
// grid, one-sided at its border (mc/MarchingCubes.cpp:1450-1512).  The
// neighbours inside the cell come from its corner values F (the same
// doubles); only the three outside it are loaded.
template <class T>
__device__ __forceinline__ void tmc_corner_gradient(const T* __restrict__ field, const Dims& d, const GridGeom& geo,
                                                    const double F[8], int i, int j, int k, int c, double n[3]) {
    const int cx = c & 1, cy = (c >> 1) & 1, cz = c >> 2;
    const int x = i + cx, y = j + cy, z = k + cz;
    const int64_t sy = d.nx, sz = (int64_t)d.nx * d.ny;
    const T* p = field + (int64_t)z * sz + (int64_t)y * sy + x;
    // x == 0 only at cx == 0, x == nx - 1 only at cx == 1 (likewise y, z)
    if (x == 0) n[0] = (F[c | 1] - F[c]) / geo.dx;
    else if (x == d.nx - 1) n[0] = (F[c] - F[c & ~1]) / geo.dx;
    else n[0] = (cx ? (double)p[1] - F[c & ~1] : F[c | 1] - (double)p[-1]) / (2 * geo.dx);
    if (y == 0) n[1] = (F[c | 2] - F[c]) / geo.dy;
    else if (y == d.ny - 1) n[1] = (F[c] - F[c & ~2]) / geo.dy;
    else n[1] = (cy ? (double)p[sy] - F[c & ~2] : F[c | 2] - (double)p[-sy]) / (2 * geo.dy);
    if (z == 0) n[2] = (F[c | 4] - F[c]) / geo.dz;
    else if (z == d.nz - 1) n[2] = (F[c] - F[c & ~4]) / geo.dz;
    else n[2] = (cz ? (double)p[sz] - F[c & ~4] : F[c | 4] - (double)p[-sz]) / (2 * geo.dz);
}

// The vertex ids of a cell's cut edges, from the words and first vertices of
// the cells that own them.  Owners are at most one row, one plane and one cell
// back: three rows are looked up (the position of cell i there; cell i - 1 is
// the one before), and only where a cut edge needs them.  At a lower side of
// the grid the row before falls together with this one.  false: an owner does
// not list the edge (never, as long as all cells see the same corner signs).
struct TmcRef {
    uint32_t code, first;
};
__device__ __forceinline__ bool tmc_edge_ids(const SegLists& L, const Dims& d, int64_t A, int64_t a, int i, int j,
                                             int k, uint32_t code, uint32_t first, const uint32_t* __restrict__ acode,
                                             const uint32_t* __restrict__ vofs, int32_t ev[12]) {
    const unsigned cut = tmc_cut_mask(code & 0xFFu);
    const bool di = i > 0, dj = j > 0, dk = k > 0;
    const int64_t rs = L.rsBase + ((int64_t)k * (d.ny - 1) + j) * L.S + i / kSeg;
    const int64_t up = L.S, upk = (int64_t)(d.ny - 1) * L.S;
    // position of cell i of a row (where it is active; cell i - 1 is before it)
    auto rank = [&](int64_t row) { return active_at(seg_words(L.mask, L.base, row), i); };
    const bool wantK = dk && (cut & 0x00Eu || (cut & 1u && !dj));    // edges 1, 2, 3; 0
    const bool wantJ = dj && (cut & 0x310u || (cut & 1u && !dk));    // edges 4, 8, 9; 0
    const bool wantJK = dj && dk && (cut & 1u);
    uint32_t atK = 0, atJ = 0, atJK = 0;
    if (wantK) atK = rank(rs - upk);
    if (wantJ) atJ = rank(rs - up);
    if (wantJK) atJK = rank(rs - upk - up);
    const TmcRef self{code, first};
    const uint32_t last = (uint32_t)(A - 1);
    auto ref = [&](uint32_t at) {
        const uint32_t x = min(at, last);
        return TmcRef{acode[x], vofs[x]};
    };
    TmcRef Sm = self, K0 = self, Km = self, J0 = self, Jm = self, JK0 = self;
    if (di && cut & 0x988u) Sm = ref((uint32_t)a - 1u);   // edges 7, 11; 3 at k = 0, 8 at j = 0
    if (wantK) K0 = ref(atK);
    if (wantJ) J0 = ref(atJ);
    if (wantJK) JK0 = ref(atJK);
    Km = K0;
    Jm = J0;
    if (di) {
        if (!dk) Km = Sm;
        else if (cut & 0x008u) Km = ref(atK - 1u);
        if (!dj) Jm = Sm;
        else if (cut & 0x100u) Jm = ref(atJ - 1u);
    }
    if (!(dj && dk)) JK0 = dj ? J0 : K0;
    bool ok = true;
    // edge e of this cell is edge oe of its owner
    auto id = [&](int e, const TmcRef& o, int oe) {
        const unsigned own = tmc_own(o.code);
        ok = ok && (!((cut >> e) & 1u) || ((own >> oe) & 1u));
        ev[e] = (int32_t)(o.first + (uint32_t)__popc(own & ((1u << oe) - 1u)));
    };
    id(0, JK0, (dj ? 2 : 0) + (dk ? 4 : 0));
    id(1, K0, dk ? 5 : 1);
    id(2, K0, dk ? 6 : 2);
    id(3, Km, (dk ? 4 : 0) + (di ? 1 : 3));
    id(4, J0, dj ? 6 : 4);
    id(5, self, 5);
    id(6, self, 6);
    id(7, Sm, di ? 5 : 7);
    id(8, Jm, dj ? (di ? 10 : 11) : (di ? 9 : 8));
    id(9, J0, dj ? 10 : 9);
    id(10, self, 10);
    id(11, Sm, di ? 10 : 11);
    return ok;
}

// Writing emitter: triangles with global vertex ids (edge refs through ev,
// inner refs from ibase) and the inner vertices' positions and normals, the
// trilinear blends of the corners' in the reference's operation order.
struct TmcWrite {
    const double (*P)[3];
    const double (*N)[3];
    const int32_t* ev;
    int32_t ibase;
    double* vpos;
    double* vnrm;
    int32_t* tris;
    int64_t t;
    __device__ int32_t id(int r) const { return r < 12 ? ev[r] : ibase + (r - 12); }
    __device__ void tri(int a, int b, int c) {
        int32_t* o = tris + 3 * t;
        o[0] = id(a);
        o[1] = id(b);
        o[2] = id(c);
        t++;
    }
    __device__ static double blend(const double (*q)[3], int x, double u, double v, double w) {
        return (1 - w) * ((1 - v) * (q[0][x] + u * (q[1][x] - q[0][x])) + v * (q[2][x] + u * (q[3][x] - q[2][x]))) +
               w * ((1 - v) * (q[4][x] + u * (q[5][x] - q[4][x])) + v * (q[6][x] + u * (q[7][x] - q[6][x])));
    }
    __device__ void inner(int s, double u, double v, double w) {
        double* p = vpos + 3 * (int64_t)(ibase + s);
        double* n = vnrm + 3 * (int64_t)(ibase + s);
        double q[3];
#pragma unroll
        for (int x = 0; x < 3; x++) p[x] = blend(P, x, u, v, w);
#pragma unroll
        for (int x = 0; x < 3; x++) q[x] = blend(N, x, u, v, w);
        const double f = sqrt(q[0] * q[0] + q[1] * q[1] + q[2] * q[2]);
        n[0] = q[0] / f;
        n[1] = q[1] / f;
        n[2] = q[2] / f;
    }
};

// One component of the gradient at a grid point: central inside the grid,
// one-sided at its border (mc/MarchingCubes.cpp:1450-1512); p at the point,
// x its coordinate of n, s the stride.
template <class T>
__device__ __forceinline__ void tmc_around(const T* __restrict__ p, int x, int n, int64_t s, T& lo, T& hi) {
    lo = p[x > 0 ? -s : 0];
    hi = p[x < n - 1 ? s : 0];
}
template <class T>
__device__ __forceinline__ double tmc_slope(T lo, T hi, int x, int n, double h, double rh2) {
    const double e = (double)hi - (double)lo;
    double g = div_by(e, 2 * h, rh2);
    if (__builtin_expect(x == 0 || x == n - 1, 0)) g = e / h;
    return g;
}

// K_T3: edge vertices of all active cells, table triangles of those that are
// not ambiguous.  A block takes kBlock cells; their new vertices have
// consecutive ids and so have their triangles, so both are listed in LDS and
// given a thread each: consecutive threads write consecutive vertices, and a
// vertex's 14 field values are in flight together.
//
// Bound by memory: at 1024^3 7.9 GB read (the field's lines around the surface,
// of which it needs a few points, by more than one L2) and 2.4 GB written, 4.9
// TB/s.
// (12 loads a vertex instead of 14, rows read as vectors, or stores staged
// through LDS changed nothing.)  One thread
// per cell that walked its twelve edges in turn ran vertices and lookups
// divergently and scattered its writes: 4.35 + 0.20 ms at 1024^3 (a pass that
// packed the owners' words included), now 2.09; 129^3 doubles 26 + 6 us, now 11.
template <class T>
__global__ void __launch_bounds__(kBlock) k_tmc_emit(VolTable vt, const uint32_t* __restrict__ acell,
                                                      const uint32_t* __restrict__ acode,
                                                      const uint32_t* __restrict__ vofs,
                                                      const uint32_t* __restrict__ tofs,
                                                      const unsigned long long* __restrict__ segMask,
                                                      const uint32_t* __restrict__ segBase, int64_t A,
                                                      double* __restrict__ vpos, double* __restrict__ vnrm,
                                                      int32_t* __restrict__ tris,
                                                      unsigned long long* __restrict__ unresolved) {
    __shared__ int32_t s_ev[12][kBlock];
    __shared__ int s_i[kBlock], s_j[kBlock], s_k[kBlock];
    __shared__ uint32_t s_code[kBlock], s_first[kBlock], s_tri[kBlock];
    __shared__ uint16_t s_vert[12 * kBlock];   // cell of the block | edge << 8
    __shared__ uint16_t s_tris[5 * kBlock];    // cell of the block | triangle << 8
    __shared__ uint32_t s_sum[kBlock / kWave];
    const VolDesc& V = vt.desc[0];
    const Dims d = V.d;
    const T* __restrict__ field = static_cast<const T*>(V.field);
    const SegLists L{segMask, segBase, V.S, V.rsBase};
    const int tid = threadIdx.x, wave = tid / kWave;
    const int64_t sy = d.nx, sz = (int64_t)d.nx * d.ny;
    for (int64_t a0 = (int64_t)blockIdx.x * kBlock; a0 < A; a0 += (int64_t)gridDim.x * kBlock) {
        const int64_t a = a0 + tid;
        uint32_t code = 0, nt = 0;
        unsigned own = 0;
        if (a < A) {
            code = acode[a];
            const uint32_t first = vofs[a], tri = tofs[a];
            int i, j, k;
            uint32_t r;
            cell_ijk(acell[a], d, i, j, k, r);
            own = tmc_own(code);
            s_i[tid] = i;
            s_j[tid] = j;
            s_k[tid] = k;
            s_code[tid] = code;
            s_first[tid] = first;
            s_tri[tid] = tri;
            if (!tmc_ambiguous(code & 0xFFu)) {
                nt = code >> 24;
                int32_t ev[12];
                if (!tmc_edge_ids(L, d, A, a, i, j, k, code, first, acode, vofs, ev)) atomicAdd(unresolved, 1ull);
#pragma unroll
                for (int e = 0; e < 12; e++) s_ev[e][tid] = ev[e];
            }
        }
        // places in the two lists: prefix sums over the block, vertices in the
        // low half (at most 12 * 256), triangles in the high one
        const uint32_t mine = (uint32_t)__popc(own) | nt << 16;
        uint32_t upto = mine;
#pragma unroll
        for (int w = 1; w < kWave; w *= 2) {
            const uint32_t t = (uint32_t)__shfl_up((int)upto, w, kWave);
            if ((tid & (kWave - 1)) >= w) upto += t;
        }
        if ((tid & (kWave - 1)) == kWave - 1) s_sum[wave] = upto;
        __syncthreads();
        uint32_t at = upto - mine, all = 0;
#pragma unroll
        for (int w = 0; w < kBlock / kWave; w++) {
            if (w < wave) at += s_sum[w];
            all += s_sum[w];
        }
        {
            uint32_t p = at & 0xFFFFu;
            for (unsigned m = own; m; m &= m - 1u) s_vert[p++] = (uint16_t)(tid | (__ffs(m) - 1) << 8);
            p = at >> 16;
            for (uint32_t t = 0; t < nt; t++) s_tris[p++] = (uint16_t)(tid | t << 8);
        }
        __syncthreads();
        const uint32_t nv = all & 0xFFFFu, ntri = all >> 16;
        for (uint32_t p = tid; p < nv; p += kBlock) {
            const int c = s_vert[p] & 0xFF, e = s_vert[p] >> 8;
            const uint32_t id = s_first[c] + (uint32_t)__popc(tmc_own(s_code[c]) & ((1u << e) - 1u));
            // first point of the edge, axis
            const int ax = e >= 8 ? 2 : e & 1;
            const int x = s_i[c] + (int)(0x622u >> e & 1u), y = s_j[c] + (int)(0xC44u >> e & 1u),
                      z = s_k[c] + (int)(0x0F0u >> e & 1u);
            const int x1 = x + (ax == 0), y1 = y + (ax == 1), z1 = z + (ax == 2);
            const T* p0 = field + (int64_t)z * sz + (int64_t)y * sy + x;
            const T* p1 = p0 + (ax == 0 ? 1 : ax == 1 ? sy : sz);
            T lo0[3], hi0[3], lo1[3], hi1[3];
            const T f0 = *p0, f1 = *p1;
            tmc_around(p0, x, d.nx, (int64_t)1, lo0[0], hi0[0]);
            tmc_around(p0, y, d.ny, sy, lo0[1], hi0[1]);
            tmc_around(p0, z, d.nz, sz, lo0[2], hi0[2]);
            tmc_around(p1, x1, d.nx, (int64_t)1, lo1[0], hi1[0]);
            tmc_around(p1, y1, d.ny, sy, lo1[1], hi1[1]);
            tmc_around(p1, z1, d.nz, sz, lo1[2], hi1[2]);
            const double F0 = (double)f0, l = (V.iso - F0) / ((double)f1 - F0);
            const GridGeom geo = V.geo;
            double q[3];
            q[0] = (1 - l) * tmc_slope(lo0[0], hi0[0], x, d.nx, geo.dx, V.rdx2[0]) +
                   l * tmc_slope(lo1[0], hi1[0], x1, d.nx, geo.dx, V.rdx2[0]);
            q[1] = (1 - l) * tmc_slope(lo0[1], hi0[1], y, d.ny, geo.dy, V.rdx2[1]) +
                   l * tmc_slope(lo1[1], hi1[1], y1, d.ny, geo.dy, V.rdx2[1]);
            q[2] = (1 - l) * tmc_slope(lo0[2], hi0[2], z, d.nz, geo.dz, V.rdx2[2]) +
                   l * tmc_slope(lo1[2], hi1[2], z1, d.nz, geo.dz, V.rdx2[2]);
            const double s = sqrt(q[0] * q[0] + q[1] * q[1] + q[2] * q[2]);
            const double rs = 1.0 / s;
            double* o = vpos + 3 * (int64_t)id;
            o[0] = (1 - l) * (geo.x0 + x * geo.dx) + l * (geo.x0 + x1 * geo.dx);
            o[1] = (1 - l) * (geo.y0 + y * geo.dy) + l * (geo.y0 + y1 * geo.dy);
            o[2] = (1 - l) * (geo.z0 + z * geo.dz) + l * (geo.z0 + z1 * geo.dz);
            double* n = vnrm + 3 * (int64_t)id;
            n[0] = div_by(q[0], s, rs);
            n[1] = div_by(q[1], s, rs);
            n[2] = div_by(q[2], s, rs);
        }
        for (uint32_t p = tid; p < ntri; p += kBlock) {
            const int c = s_tris[p] & 0xFF, t = s_tris[p] >> 8;
            const uint32_t wd = (uint32_t)(c_tmc_tri[s_code[c] & 0xFFu] >> (12 * t));
            int32_t* o = tris + 3 * ((int64_t)s_tri[c] + t);
            o[0] = s_ev[wd >> 8 & 0xFu][c];   // reversed: positive corners outside
            o[1] = s_ev[wd >> 4 & 0xFu][c];
            o[2] = s_ev[wd & 0xFu][c];
        }
        __syncthreads();   // before the next cells
    }
}

// K_T4: the ambiguous cells k_tmc_cells listed (amb[0] = count, cells from
// amb[1]): inner vertices and triangles, sliced with the asymptotic decider.
template <class T>
__global__ void __launch_bounds__(kBlock) k_tmc_emit_amb(VolTable vt, const uint32_t* __restrict__ amb,
                                                          const uint32_t* __restrict__ acell,
                                                          const uint32_t* __restrict__ acode,
                                                          const uint32_t* __restrict__ vofs,
                                                          const uint32_t* __restrict__ tofs,
                                                          const unsigned long long* __restrict__ segMask,
                                                          const uint32_t* __restrict__ segBase, int64_t A,
                                                          double* __restrict__ vpos, double* __restrict__ vnrm,
                                                          int32_t* __restrict__ tris,
                                                          unsigned long long* __restrict__ unresolved) {
    const uint32_t cells = amb[0];
    const VolDesc& V = vt.desc[0];
    const Dims d = V.d;
    const GridGeom geo = V.geo;
    const T* __restrict__ field = static_cast<const T*>(V.field);
    const SegLists L{segMask, segBase, V.S, V.rsBase};
    for (uint32_t s = blockIdx.x * kBlock + threadIdx.x; s < cells; s += gridDim.x * kBlock) {
        const uint32_t a = amb[1 + s], code = acode[a];
        if (code & 0x100u) continue;   // singular face: no triangles
        int i, j, k;
        uint32_t r;
        cell_ijk(acell[a], d, i, j, k, r);
        const uint32_t first = vofs[a];
        int32_t ev[12];
        if (!tmc_edge_ids(L, d, A, a, i, j, k, code, first, acode, vofs, ev)) atomicAdd(unresolved, 1ull);
        double F[8], P[8][3], N[8][3];
        tmc_corners(field, d, i, j, k, F);
        for (int c = 0; c < 8; c++) {
            P[c][0] = geo.x0 + (i + (c & 1)) * geo.dx;
            P[c][1] = geo.y0 + (j + ((c >> 1) & 1)) * geo.dy;
            P[c][2] = geo.z0 + (k + (c >> 2)) * geo.dz;
            tmc_corner_gradient(field, d, geo, F, i, j, k, c, N[c]);
        }
        TmcWrite w{P, N, ev, (int32_t)(first + (uint32_t)__popc(tmc_own(code))), vpos, vnrm, tris, (int64_t)tofs[a]};
        tmc_slice(F, code & 0xFFu, V.iso, w);
    }
}

}  // namespace tmc
