// dmc_quad_kernels.h -- quadrilaterals and their halfedges, straight from the
// cells.
//
// A halfedge of a quadrilateral runs between the vertices of two cells that
// share a cell face, the quadrilateral's grid edge being one of the face's
// four edges.  Two cells share one face only, so the halfedges on a vertex
// pair {a, b} -- the reference's map entry
// (cpp_dmc/DualMarchingCubes.cpp:488-671) -- are those of the face's interior
// cut edges whose contour in the one cell is a and in the other is b: at most
// four, all known from the records of the cells around.  So the first
// halfedge build needs no lookup by vertex pair.
#pragma once
#include "dmc_extract_kernels.h"
#include "dmc_mesh_kernels.h"

namespace tmc {

// The halfedge of a quadrilateral that crosses the face between cells A and B,
// where the quadrilateral's grid edge is edge ea of A and eb of B, as
// halfedge << 1 | starts at A's vertex.  bit: field below iso at the edge's
// first point.
__device__ __forceinline__ uint32_t crossing_key(uint32_t q, int ea, int eb, int bit) {
    const int sa = edge_slot(ea, bit), sb = edge_slot(eb, bit);
    const bool from = ((sa + 1) & 3) == sb;
    return (4u * q + (uint32_t)(from ? sa : sb)) << 1 | (uint32_t)from;
}

template <class T>
__device__ __forceinline__ T by_type(int t, T x, T y, T z) {
    return t == 0 ? x : t == 1 ? y : z;
}

// Edges of a cell that come later in the quadrilaterals' order (owner cell in
// (k, j, i) order, then x, y, z) than edge e, in spread form: the last
// interior edge of a contour carries the largest halfedge leaving its vertex.
constexpr uint32_t later_edges(int e) {
    constexpr int order[12] = {0, 3, 8, 1, 9, 2, 11, 10, 4, 7, 5, 6};
    uint32_t m = 0;
    bool after = false;
    for (int x = 0; x < 12; x++) {
        if (after) m |= 1u << (2 * order[x]);
        if (order[x] == e) after = true;
    }
    return m;
}

// Where k_quads writes the first halfedge build.
struct QuadOut {
    int32_t* quads;
    uint8_t* colors;
    int32_t* twin;
    uint8_t* flag;
    int32_t* hev;
    int32_t* val;    // valence per vertex, out-degrees so far (null: not wanted)
    uint8_t* dead;   // face marks of the simplifications, cleared (with val)
    BndRec* recs;
    uint32_t reccap;
    Sizes* S;
    unsigned long long* vst;   // per-volume counts (a batch without simplification)
};

// Twin and flag of the halfedge `own` (a crossing key) from the other
// members of its group (keys, 0xFFFFFFFF: none) where there are two or more:
// twin_rule over local keys.  va, vb: the vertices of cells A and B.
__device__ __forceinline__ void crowded_edge(uint32_t own, uint32_t k0, uint32_t k1, uint32_t k2, int32_t va,
                                             int32_t vb, const QuadOut& o, int32_t& tw, uint8_t& fl) {
    uint32_t g[4] = {own, k0, k1, k2};
#pragma unroll
    for (int x = 0; x < 3; x++)
#pragma unroll
        for (int y = 0; y < 3 - x; y++) {
            const uint32_t lo = min(g[y], g[y + 1]), hi = max(g[y], g[y + 1]);
            g[y] = lo;
            g[y + 1] = hi;
        }
    auto he = [&](int x) { return (int32_t)(g[x] >> 1); };
    auto org = [&](int x) { return (g[x] & 1u) ? va : vb; };
    const bool four = g[3] != 0xFFFFFFFFu;
    const int32_t h = (int32_t)(own >> 1);
    tw = -1;
    if (four) {
        fl = 1;
        const bool ab = org(0) != org(1);   // pairs (0, 1)(2, 3), else (0, 2)(1, 3)
        const int32_t p0 = he(0), p1 = ab ? he(1) : he(2), p2 = ab ? he(2) : he(1), p3 = he(3);
        tw = h == p0 ? p1 : h == p1 ? p0 : h == p2 ? p3 : p2;
        return;
    }
    fl = 2;
    int a, b, l;
    if (org(0) != org(1)) { a = 0; b = 1; l = 2; }
    else if (org(0) != org(2)) { a = 0; b = 2; l = 1; }
    else { a = 1; b = 2; l = 0; }
    const int32_t pa = a == 0 ? he(0) : he(1), pb = b == 1 ? he(1) : he(2);
    tw = h == pa ? pb : h == pb ? pa : -1;
    if (h == he(0)) {
        BndRec r;
        r.a = a == 0 ? org(0) : org(1);
        r.b = b == 1 ? org(1) : org(2);
        r.lone = l == 0 ? he(0) : l == 1 ? he(1) : he(2);
        r.key = he_key(va, vb);
        r.pad = 0;
        put_record(o.recs, &o.S->nrec, o.reccap, &o.S->ovf, r);
    }
}

// A cell around a quadrilateral's grid edge.
struct Around {
    uint32_t at;      // flat index
    uint32_t cell;    // linear cell index
    uint32_t rs;      // its (row, segment)
    int x;            // its position in the row
    uint32_t same;    // edges of the contour of the grid edge (spread form)
    uint32_t in;      // the interior ones of these
    int32_t v;        // that contour's vertex
};

// Three edges of the face between cells A and B besides the quadrilateral's
// own, in A (low) and in B (high nibble), one byte each.
__device__ __forceinline__ int face_ea(uint32_t f, int n) { return (int)((f >> (8 * n)) & 0xFu); }
__device__ __forceinline__ int face_eb(uint32_t f, int n) { return (int)((f >> (8 * n + 4)) & 0xFu); }

// ---------------------------------------------------------------------------
// K4: quadrilaterals and their halfedges.  Each complete quadrilateral belongs
// to the grid edge e0 (x), e3 (y) or e8 (z) of the cell at its lower corner;
// ascending (cell, direction) is the reference's map order
// (cpp_dmc/DualMarchingCubes.h:215-223, :663-676).  Colour: 3*parity + dir
// (cpp_dmc/DualMarchingCubes.cpp:180-183).
//
// A block takes kBlock active cells, lists their quadrilaterals in LDS (their
// ids are consecutive) and gives each a thread, whatever its direction: the
// cells O (the owner), U, V and UV around the edge, and across each of their
// four faces the quadrilateral of the face's other edge on the same two
// contours, whose owner is A or the next cell of A's row, next row or next
// plane.  The thread writes the quadrilateral, its twins and its flags whole,
// counts a boundary halfedge into the vertex it ends at, and writes he_v of a
// vertex where the edge is the last interior one of its contour.  Two or more
// others on a face are rare (crowded_edge).
//
// Bound by the latency of the gathers around: the activity words that find a
// cell of another row, then its 16-byte record, then its group's base.  So
// waves in flight count most: at 1024^3 1.64 ms at 4 waves per SIMD (as
// compiled, 123 VGPRs), 1.46 at 5, 1.41 at 6 (80 VGPRs, a few spilled), 1.59
// at 7.  It replaced 8-byte scatters of (halfedge, destination) pairs into
// rows by vertex, a scan of the rows and a second kernel that paired them:
// 2.07 + 0.06 + 1.10 ms at 1024^3 (14 GB moved), 1.46 + 0.05 + 0.84 ms for
// 1,024 small volumes, now 1.26.  One thread per cell, its three directions in
// turn, left a third of the lanes busy: 2.63 ms.
// ---------------------------------------------------------------------------
template <bool MANY>
__global__ void __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(6, 6))) k_quads(VolTable vt, const uint4* __restrict__ rec,
                                                   const uint32_t* __restrict__ grpV,
                                                   const uint32_t* __restrict__ grpQ, DevN dA,
                                                   const unsigned long long* __restrict__ segMask,
                                                   const uint32_t* __restrict__ segBase, QuadOut o,
                                                   uint32_t* unresolved) {
    __shared__ uint4 s_rec[kBlock];
    __shared__ int s_i[kBlock], s_vol[MANY ? kBlock : 1];
    __shared__ uint32_t s_rs[kBlock];
    __shared__ uint16_t s_list[3 * kBlock];   // cell of the block | direction << 8 | parity << 10
    __shared__ uint32_t s_q0, s_nq;
    const int64_t A = dA.get();
    HeCount cnt;
    // one volume (MANY false): a copy of its descriptor, which the stores below
    // could otherwise change: 1024^3 1.43 -> 1.39 ms, 512^3 blobs 440 -> 398 us
    const VolDesc V0 = vt.desc[0];
    for (int64_t a0 = (int64_t)blockIdx.x * kBlock; a0 < A; a0 += (int64_t)gridDim.x * kBlock) {
        const int tid = threadIdx.x;
        {
            const int64_t a = a0 + tid;
            uint32_t q0 = 0, par = 0;
            unsigned own = 0;
            if (a < A) {
                const int vol = MANY ? vol_of(vt.aBase, vt.n, a) : 0;
                const VolDesc& V = MANY ? vt.desc[vol] : V0;
                const uint4 w = rec[a];
                const ActRec R{w.x, w.y, w.z, w.w};
                int i, j, k;
                uint32_t r;
                cell_ijk(R.cell, V.d, i, j, k, r);
                s_rec[tid] = w;
                s_i[tid] = i;
                const uint32_t rs = (uint32_t)V.rsBase + r * (uint32_t)V.S + (uint32_t)i / kSeg;
                s_rs[tid] = rs;
                if (MANY) s_vol[tid] = vol;
                par = (uint32_t)((i & 1) | (j & 1) << 1 | (k & 1) << 2);
                // a cell's own edges 0, 3 and 8 are interior where all four
                // cells around them exist
                own = (R.aux & 1u) | (R.aux >> 6 & 1u) << 1 | (R.aux >> 16 & 1u) << 2;
                q0 = grpQ[rs >> V.gsh] + R.qloc();
                if (tid == 0) s_q0 = q0;
                if (a == A - 1 || tid == kBlock - 1) s_nq = q0 + (uint32_t)__popc(own);   // where they end
            }
            __syncthreads();
            uint32_t p = q0 - s_q0;
            for (; own; own &= own - 1u) s_list[p++] = (uint16_t)(tid | (__ffs(own) - 1) << 8 | par << 10);
            __syncthreads();
        }
        const uint32_t qbase = s_q0, nq = s_nq - qbase;
        for (uint32_t p = tid; p < nq; p += kBlock) {
            const uint32_t q = qbase + p, entry = s_list[p];
            const int ci = entry & 0xFF, t = (entry >> 8) & 3;
            const VolDesc& V = MANY ? vt.desc[s_vol[ci]] : V0;
            const int i = s_i[ci];
            const uint4 w = s_rec[ci];
            const uint32_t C = (uint32_t)V.d.C, rows = (uint32_t)(V.d.ny - 1), S = (uint32_t)V.S, SP = S * rows;
            const uint32_t CP = C * rows;
            const int gsh = V.gsh;
            const uint32_t rs0 = s_rs[ci];
            const uint32_t back = ((uint32_t)i % kSeg) == 0u ? 1u : 0u;   // cell i-1 is in the segment before
            const uint32_t a = (uint32_t)(a0 + ci);
            uint32_t bad = 0;
            auto last = [&](uint32_t at) { return (uint32_t)min((int64_t)at, A - 1); };
            auto before = [](uint32_t at) { return at > 0u ? at - 1u : 0u; };
            // the three other cells: x edge (j-1), (k-1), both; y edge (i-1),
            // (k-1), both; z edge (i-1), (j-1), both
            const uint32_t rsV = rs0 - (t == 2 ? S : SP);
            const SegWords wV = seg_words(segMask, segBase, rsV);
            uint32_t atU = before(a), atUV, rsU = rs0 - back, rsUV = rsV - back;
            const uint32_t atV = last(active_at(wV, i));
            if (t == 0) {
                rsU = rs0 - S;
                rsUV = rsV - S;
                const SegWords wU = seg_words(segMask, segBase, rsU), wUV = seg_words(segMask, segBase, rsUV);
                atU = last(active_at(wU, i));
                atUV = last(active_at(wUV, i));
            } else {
                atUV = before(atV);
            }
            const uint4 rU = rec[atU], rV = rec[atV], rUV = rec[atUV];
            auto around = [&](const uint4& x, uint32_t at, uint32_t rs, uint32_t cell, int cx, int e) __attribute__((always_inline)) {
                const ActRec N{x.x, x.y, x.z, x.w};
                Around c;
                c.at = at;
                c.cell = cell;
                c.rs = rs;
                c.x = cx;
                const uint32_t map = N.code >> 8, tc = (map >> (2 * e)) & 3u;
                c.same = contour_spread(map, tc);
                c.in = c.same & N.aux;
                c.v = (int32_t)(grpV[rs >> gsh] + N.vloc() + (uint32_t)__popc(N.used() & ((1u << tc) - 1u)));
                // not that cell: the field changed under the sweep; ids in
                // range, and the build is redone
                if (__builtin_expect(N.cell != cell, 0)) {
                    bad = 1;
                    c.in = c.same = 0;
                    c.v = 0;
                }
                return c;
            };
            const uint32_t dU = t == 0 ? C : 1u, dV = t == 2 ? C : CP;
            const int xU = t == 0 ? i : i - 1;
            const Around O = around(w, a, rs0, w.x, i, by_type(t, 0, 3, 8));
            const Around U = around(rU, atU, rsU, w.x - dU, xU, by_type(t, 2, 1, 9));
            const Around W = around(rV, atV, rsV, w.x - dV, i, by_type(t, 4, 7, 11));
            const Around UW = around(rUV, atUV, rsUV, w.x - dU - dV, xU, by_type(t, 6, 5, 10));
            const int bit = (int)(~w.y & 1u);
            // key of the quadrilateral of edge ea of P (eb of Q), owned by P or
            // the next cell of its row, of the next row or of the next plane
            auto key_of = [&](const Around& P, int ea, int eb) __attribute__((always_inline)) {
                const bool jn = ea == 2 || ea == 11, kn = ea == 4 || ea == 7, in = ea == 1 || ea == 9;
                const uint32_t rs = P.rs + (jn ? S : kn ? SP : in && ((uint32_t)(P.x + 1) % kSeg) == 0u ? 1u : 0u);
                uint32_t at = P.at + (in ? 1u : 0u);
                if (jn || kn) at = active_at(seg_words(segMask, segBase, rs), P.x);
                const uint4 x = rec[last(at)];
                const ActRec N{x.x, x.y, x.z, x.w};
                const int ax = edge_axis(ea);
                uint32_t id = grpQ[rs >> gsh] + N.qloc() + (ax >= 1 ? N.aux & 1u : 0u) + (ax == 2 ? N.aux >> 6 & 1u : 0u);
                if (__builtin_expect(N.cell != P.cell + (jn ? C : kn ? CP : in ? 1u : 0u), 0)) {
                    bad = 1;
                    id = 0;
                }
                return crossing_key(id, ea, eb, (int)(~N.code & 1u));
            };
            // the face's other edges f (in P | in Q << 4, one byte each) on the
            // two contours
            auto matches = [](const Around& P, const Around& Q, uint32_t f) __attribute__((always_inline)) {
                uint32_t m = 0;
#pragma unroll
                for (int n = 0; n < 3; n++) m |= ((P.in >> (2 * face_ea(f, n))) & (Q.same >> (2 * face_eb(f, n))) & 1u) << n;
                return m;
            };
            const uint32_t fOU = by_type(t, 0x64A9B8u, 0xAB5798u, 0xAB5713u);
            const uint32_t fOV = by_type(t, 0x516273u, 0x516240u, 0x64A920u);
            const uint32_t fU = by_type(t, 0x514073u, 0x624073u, 0x6420B8u);
            const uint32_t fV = by_type(t, 0xA920B8u, 0xAB9813u, 0x579813u);
            const uint32_t mOU = matches(O, U, fOU), mOV = matches(O, W, fOV), mU = matches(U, UW, fU),
                           mV = matches(W, UW, fV);
            // twin across a face with at most one match
            auto twin_of = [&](const Around& P, uint32_t f, uint32_t m) __attribute__((always_inline)) {
                if (!m) return -1;
                const uint32_t e = f >> (m & 1u ? 0 : m & 2u ? 8 : 16);
                return (int32_t)(key_of(P, (int)(e & 0xFu), (int)(e >> 4 & 0xFu)) >> 1);
            };
            int32_t tOU = twin_of(O, fOU, mOU), tOV = twin_of(O, fOV, mOV), tU = twin_of(U, fU, mU),
                    tV = twin_of(W, fV, mV);
            uint32_t flOU = 0, flOV = 0, flU = 0, flV = 0;
            auto many = [](uint32_t m) { return (m & (m - 1u)) != 0u; };
            if (__builtin_expect(many(mOU) || many(mOV) || many(mU) || many(mV), 0)) {
#pragma unroll 1
                for (int f = 0; f < 4; f++) {
                    const uint32_t m = f == 0 ? mOU : f == 1 ? mOV : f == 2 ? mU : mV;
                    if (!many(m)) continue;
                    const uint32_t fc = f == 0 ? fOU : f == 1 ? fOV : f == 2 ? fU : fV;
                    Around P{};
                    P.at = f < 2 ? O.at : f == 2 ? U.at : W.at;
                    P.cell = f < 2 ? O.cell : f == 2 ? U.cell : W.cell;
                    P.rs = f < 2 ? O.rs : f == 2 ? U.rs : W.rs;
                    P.x = f == 2 ? U.x : i;
                    const int32_t va = f < 2 ? O.v : f == 2 ? U.v : W.v, vb = f == 0 ? U.v : f == 1 ? W.v : UW.v;
                    const int eO = by_type(t, 0, 3, 8), eU = by_type(t, 2, 1, 9), eW = by_type(t, 4, 7, 11),
                              eUW = by_type(t, 6, 5, 10);
                    uint32_t key[3] = {0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu};
#pragma unroll
                    for (int n = 0; n < 3; n++)
                        if ((m >> n) & 1u) key[n] = key_of(P, face_ea(fc, n), face_eb(fc, n));
                    int32_t tw;
                    uint8_t fl;
                    crowded_edge(crossing_key(q, f < 2 ? eO : f == 2 ? eU : eW, f == 0 ? eU : f == 1 ? eW : eUW, bit),
                                 key[0], key[1], key[2], va, vb, o, tw, fl);
                    cnt.add(fl);
                    vol_count_of(o.vst, MANY ? s_vol[ci] : 0, fl);
                    tOU = f == 0 ? tw : tOU;
                    tOV = f == 1 ? tw : tOV;
                    tU = f == 2 ? tw : tU;
                    tV = f == 3 ? tw : tV;
                    flOU = f == 0 ? fl : flOU;
                    flOV = f == 1 ? fl : flOV;
                    flU = f == 2 ? fl : flU;
                    flV = f == 3 ? fl : flV;
                }
            }
            // corners in order from O's: O, U, UW, W or O, W, UW, U; halfedge n
            // runs from corner n to corner n + 1
            const bool viaU = (t == 1) != (bit != 0);
            const int s0 = t == 1 ? (bit ? 1 : 3) : 0;   // O's corner
            const int32_t c1 = viaU ? U.v : W.v, c3 = viaU ? W.v : U.v;
            const int32_t h0 = viaU ? tOU : tOV, h1 = viaU ? tU : tV, h2 = viaU ? tV : tU, h3 = viaU ? tOV : tOU;
            const uint32_t cf = viaU ? flOU | flU << 8 | flV << 16 | flOV << 24 : flOV | flV << 8 | flU << 16 | flOU << 24;
            // rotate by s0 (0, 1 or 3)
            auto turn = [&](int32_t x0, int32_t x1, int32_t x2, int32_t x3) __attribute__((always_inline)) {
                return make_int4(s0 == 0 ? x0 : s0 == 1 ? x3 : x1, s0 == 0 ? x1 : s0 == 1 ? x0 : x2,
                                 s0 == 0 ? x2 : s0 == 1 ? x1 : x3, s0 == 0 ? x3 : s0 == 1 ? x2 : x0);
            };
            reinterpret_cast<int4*>(o.quads)[q] = turn(O.v, c1, UW.v, c3);
            reinterpret_cast<int4*>(o.twin)[q] = turn(h0, h1, h2, h3);
            reinterpret_cast<uint32_t*>(o.flag)[q] = cf << (8 * s0) | (s0 ? cf >> (32 - 8 * s0) : 0u);
            o.colors[q] = (uint8_t)(3 * (entry >> 10) + (uint32_t)t);
            // valence: a boundary halfedge adds one to the vertex it ends at
            if (o.val) {
                if (h0 < 0) atomicAdd(&o.val[c1], 1);
                if (h1 < 0) atomicAdd(&o.val[UW.v], 1);
                if (h2 < 0) atomicAdd(&o.val[c3], 1);
                if (h3 < 0) atomicAdd(&o.val[O.v], 1);
                o.dead[q] = 0;
            }
            // he_v: the edge is the last interior one of the vertex's contour
            constexpr uint32_t l0 = later_edges(0), l3 = later_edges(3), l8 = later_edges(8), l2 = later_edges(2),
                               l1 = later_edges(1), l9 = later_edges(9), l4 = later_edges(4), l7 = later_edges(7),
                               l11 = later_edges(11), l6 = later_edges(6), l5 = later_edges(5), l10 = later_edges(10);
            const int32_t h = (int32_t)(4u * q);
            if ((O.in & by_type(t, l0, l3, l8)) == 0u) o.hev[O.v] = h + s0;
            if ((U.in & by_type(t, l2, l1, l9)) == 0u) o.hev[U.v] = h + ((s0 + (viaU ? 1 : 3)) & 3);
            if ((W.in & by_type(t, l4, l7, l11)) == 0u) o.hev[W.v] = h + ((s0 + (viaU ? 3 : 1)) & 3);
            if ((UW.in & by_type(t, l6, l5, l10)) == 0u) o.hev[UW.v] = h + ((s0 + 2) & 3);
            if (__builtin_expect(bad, 0)) atomicAdd(unresolved, 1u);
        }
        __syncthreads();   // the lists are taken again
    }
    cnt.flush(o.S->hep);
}

}  // namespace tmc
