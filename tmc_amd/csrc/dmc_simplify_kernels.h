// dmc_simplify_kernels.h -- the 3X3Y and 3333 simplifications on the live mesh.
//
// The mesh keeps the cell stage's numbering while it is simplified: removed
// faces and vertices are only marked, and one compaction at the end renumbers
// the rest (order-preserving, so every rule that depends on the order of faces
// or vertices sees the order it would see after a compaction per stage).  A
// stage changes what lies around its merging faces and nothing else:
//
//   k_stage_mark, k_stage_claim   the candidates and which of them merge; the
//                    last face to remove a vertex claims it (the reference's sequential loop,
//                    cpp_dmc/DualMarchingCubes.cpp:916-1094);
//   k_stage_sort     the regular ones: both merging vertices closed fans of
//                    three faces, all edges around in groups of two, the
//                    merged vertex's four neighbours distinct.  Their effect
//                    is known locally: two pairs of halfedges become twins,
//                    two corners are renamed;
//   k_stage_merge    applies these;
//   k_stage_irregular, k_stage_rewrite, k_stage_pair   the others (boundary,
//                    non-manifold or degenerate neighbourhoods), launched
//                    always and empty where there are none: every face with a
//                    changed corner is rewritten, and the halfedges on a
//                    changed vertex are paired again by vertex pair.
//
// 3333 is built the same way (k_stage_claim3333, k_stage_cut3333, ...).  A pass
// that meets what the in-place form does not express (a vertex merged into a
// removed one, whose result depends on the compacted numbering; a face left
// with a removed corner) sets need_generic and is run again with a compaction
// and a generic halfedge build per stage.
#pragma once
#include "dmc_mesh_kernels.h"

namespace tmc {

// A claim on a vertex: the stage (1..3) above the claiming face, so that later
// stages outrank earlier ones and the array is cleared once per pass.  A
// vertex with a claim is removed.
constexpr int kClaimShift = 29;
constexpr int32_t kClaimFace = (1 << kClaimShift) - 1;
__device__ __forceinline__ bool removed(int32_t claim) { return claim > kClaimFace; }

// Vertex state bits: changed irregularly in stage s (1 << (s - 1)), removed
// irregularly (faces have to be searched for it), he_v taken again at the end.
constexpr uint8_t kVsGone = 8, kVsRetake = 16;

// The live mesh and the working arrays of its simplification.
struct Live {
    int32_t* quads;
    int32_t* twin;
    uint8_t* flag;
    int32_t* hev;
    int32_t* val;      // valence
    uint8_t* dead;     // faces: 0 alive (bit 0 merged, bits 1, 2: dropped by 3333)
    uint8_t* vs;       // vertex states
    int32_t* claim;    // last claim on each vertex
    int32_t* last;     // 3X3Y: last irregular face to move each vertex; 3333: the vertex that takes its place
    double* pos;
    double* nrm;
    uint8_t* p;        // 3X3Y: faces of the pattern; 3333: 2 irregular pattern faces
    uint8_t* em;       // merging faces: which pair of vertices merges (1 / 2); rewritten ones: halfedges to pair
    uint32_t* list;    // merging / pattern faces of the stage, then the rewritten ones
    int4* frame;       // the merging faces' frames, two words of four (MergeFrame)
    uint32_t* irr;     // candidates, then the irregular ones of the list
    int32_t* head;     // changed vertices: their halfedges to pair, a list through ...
    int4* ent;         // ... entry h of halfedge h (next, origin, destination, changed vertex)
    BndRec* recs;
    uint32_t reccap;
    Sizes* S;
    unsigned long long* vst;   // per-volume counts of a batch
    const int64_t* qb;         // first face of each volume
    int nvol;
    int stage;
    __device__ __forceinline__ int32_t tag(int64_t f) const { return (stage << kClaimShift) | (int32_t)f; }
    __device__ __forceinline__ bool claimed_now(int32_t c) const { return (c >> kClaimShift) == stage; }
    __device__ __forceinline__ uint8_t changed() const { return (uint8_t)(1u << (stage - 1)); }
    __device__ __forceinline__ int32_t dest(int32_t h) const { return quads[he_next(h)]; }
};

// Signed counts of flagged halfedges taken off or added, flushed once per
// block (every thread of the block calls flush).
struct HeDelta {
    int n4 = 0, n3 = 0, err = 0;
    __device__ __forceinline__ void add(uint8_t fl, int by) {
        n4 += fl == 1 ? by : 0;
        n3 += fl == 2 ? by : 0;
        err += fl == kFlagErrFirst ? by : 0;
    }
    __device__ __forceinline__ void flush(unsigned long long (*hep)[3]) const {
        __shared__ int sm[3];
        if (threadIdx.x < 3) sm[threadIdx.x] = 0;
        __syncthreads();
        const int a = wave_sum(n4), b = wave_sum(n3), e = wave_sum(err);
        if ((threadIdx.x & (kWave - 1)) == 0) {
            if (a) atomicAdd(&sm[0], a);
            if (b) atomicAdd(&sm[1], b);
            if (e) atomicAdd(&sm[2], e);
        }
        __syncthreads();
        if (threadIdx.x < 3 && sm[threadIdx.x])
            atomicAdd(&hep[blockIdx.x & (kHeParts - 1)][threadIdx.x], (unsigned long long)(long long)sm[threadIdx.x]);
    }
};
__device__ __forceinline__ void vol_delta(const Live& m, int32_t h, uint8_t fl, int by) {
    if (!m.vst || (fl != 1 && fl != 2 && fl != kFlagErrFirst)) return;
    atomicAdd(&m.vst[3 * vol_of(m.qb, m.nvol, h >> 2) + (fl == 1 ? 0 : fl == 2 ? 1 : 2)],
              (unsigned long long)(long long)by);
}

__device__ __forceinline__ void vs_or(uint8_t* vs, int32_t v, uint32_t bits) {
    atomicOr(reinterpret_cast<uint32_t*>(vs) + (v >> 2), bits << (8 * (v & 3)));
}

// The face lists of a stage.  A block walks a contiguous range of faces and
// gathers its entries in LDS, so that the list's counter takes few adds and
// the list keeps neighbouring faces together.
constexpr int kListBuf = 2048;
constexpr int kListIlp = 4;   // faces a thread looks at per turn: their gathers are in flight together
constexpr int kListTurn = kListIlp * kBlock;
struct ListBuf {
    uint32_t* buf;    // LDS, kListBuf entries
    uint32_t* n;      // LDS: entries held, then the base of a flush
    uint32_t* out;
    uint32_t* count;
    // at most kListIlp adds per thread and turn
    __device__ __forceinline__ void add(bool has, uint32_t x) const {
        const uint64_t m = __ballot(has);
        if (!m) return;
        uint32_t base = 0;
        const int leader = __ffsll((unsigned long long)m) - 1;
        if ((int)__lane_id() == leader) base = atomicAdd(&n[0], (uint32_t)__popcll(m));
        base = (uint32_t)__shfl((int)base, leader, kWave);
        if (has) buf[base + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u))] = x;
    }
    // every thread of the block calls these, once per turn / at the end
    __device__ __forceinline__ void end_turn() const {
        __syncthreads();
        const uint32_t held = n[0];
        __syncthreads();   // the next turn adds
        if (held > kListBuf - kListTurn) flush();
    }
    __device__ __forceinline__ void flush() const {
        __syncthreads();
        const uint32_t k = n[0];
        if (threadIdx.x == 0) n[1] = k ? atomicAdd(count, k) : 0u;
        __syncthreads();
        const uint32_t base = n[1];
        for (uint32_t i = threadIdx.x; i < k; i += kBlock) out[base + i] = buf[i];
        __syncthreads();
        if (threadIdx.x == 0) n[0] = 0;
        __syncthreads();
    }
};
// a block's share of n items: whole turns where there are many
__device__ __forceinline__ int64_t block_share(int64_t n) {
    const int64_t each = (n + (int64_t)gridDim.x - 1) / (int64_t)gridDim.x;
    const int64_t unit = each > kListTurn ? kListTurn : kBlock;
    return (each + unit - 1) / unit * unit;
}
// Calls fn(f, in range) for the block's share of n faces, kListIlp faces per
// thread and turn, consecutive threads on consecutive faces; then end().
template <class F, class E>
__device__ __forceinline__ void for_share(int64_t n, F&& fn, E&& end_turn) {
    const int64_t share = block_share(n), begin = (int64_t)blockIdx.x * share, end = min(n, begin + share);
    for (int64_t f0 = begin; f0 < end; f0 += kListTurn) {
        fn(f0 + threadIdx.x, end);
        end_turn();
    }
}

// Kept vertices of valence 0, counted at each stage's start.
__device__ __forceinline__ void count_zero(const Live& m) {
    const int64_t nv = (int64_t)m.S->nv;
    unsigned int z = 0;
    TMC_GRID_STRIDE(v, nv) z += m.val[v] == 0 && !removed(m.claim[v]);
    z = wave_sum(z);
    if ((threadIdx.x & (kWave - 1)) == 0 && z) atomicAdd(&m.S->zero, z);
}

// Candidates of the stage among the live faces, listed in m.irr: 3X3Y the
// pattern (cpp_dmc/DualMarchingCubes.cpp:889-913), also kept per face for its
// neighbours; 3333 the faces of four valence-3 corners (:1190-1301 asks more).
// Bound by the valence gathers: four faces per thread keep sixteen in flight.
template <bool k3333>
__global__ void __launch_bounds__(kBlock) k_stage_mark(Live m) {
    __shared__ uint32_t buf[kListBuf], n[2];
    if (threadIdx.x == 0) n[0] = 0;
    __syncthreads();
    const ListBuf L{buf, n, m.irr, &m.S->ncand[m.stage]};
    for_share((int64_t)m.S->nq, [&](int64_t f0, int64_t end) {
        bool r[kListIlp];
        int4 q[kListIlp];
        uint8_t dead[kListIlp];
#pragma unroll
        for (int u = 0; u < kListIlp; u++) {
            const int64_t f = f0 + u * kBlock;
            const bool in = f < end;
            q[u] = in ? reinterpret_cast<const int4*>(m.quads)[f] : make_int4(0, 0, 0, 0);
            dead[u] = in ? m.dead[f] : 1;
        }
#pragma unroll
        for (int u = 0; u < kListIlp; u++) {
            const int a = m.val[q[u].x], b = m.val[q[u].y], c = m.val[q[u].z], d = m.val[q[u].w];
            r[u] = k3333 ? a == 3 && b == 3 && c == 3 && d == 3
                         : (a == 3 && b >= 5 && c == 3 && d >= 5) || (a >= 5 && b == 3 && c >= 5 && d == 3);
            r[u] = r[u] && !dead[u];
        }
#pragma unroll
        for (int u = 0; u < kListIlp; u++) {
            const int64_t f = f0 + u * kBlock;
            if (f < end) m.p[f] = !k3333 && r[u];
            L.add(r[u], (uint32_t)f);
        }
    }, [&] { L.end_turn(); });
    L.flush();
    // every vertex of the cell stage has a face
    if (m.stage > 1) count_zero(m);
}

// The merging faces among the candidates: each claims the vertex it removes.
__global__ void __launch_bounds__(kBlock) k_stage_claim(Live m, const uint8_t* __restrict__ colors) {
    __shared__ uint32_t buf[kListBuf], n[2];
    if (threadIdx.x == 0) n[0] = 0;
    __syncthreads();
    const ListBuf L{buf, n, m.list, &m.S->nlist[m.stage]};
    const int64_t nv = (int64_t)m.S->nv;
    for_share((int64_t)m.S->ncand[m.stage], [&](int64_t i0, int64_t end) {
        for (int u = 0; u < kListIlp; u++) {
            const int64_t i = i0 + u * kBlock;
            const int64_t f = i < end ? (int64_t)m.irr[i] : 0;
            const int d = i < end ? merge_decision(f, m.quads, m.val, m.p, colors, m.twin, m.flag, nv) : 0;
            if (d) {
                const int4 q = reinterpret_cast<const int4*>(m.quads)[f];
                m.em[f] = (uint8_t)d;
                atomicMax(&m.claim[d == 1 ? q.z : q.w], m.tag(f));
            }
            L.add(d != 0, (uint32_t)f | (uint32_t)(d == 2) << 31);
        }
    }, [&] { L.end_turn(); });
    L.flush();
}

// A merging face in the frame of its merge: t stays (moved), r goes; the
// halfedges of its edges (t, n1), (n1, r), (r, n3), (n3, t) and their twins.
struct MergeFrame {
    int32_t f, t, n1, r, n3;
    int32_t A, C, D, B;   // twins of the edges in that order
};
__device__ __forceinline__ MergeFrame merge_frame(const Live& m, uint32_t e) {
    MergeFrame x;
    x.f = (int32_t)(e & (uint32_t)kClaimFace);
    const int4 q = reinterpret_cast<const int4*>(m.quads)[x.f], w = reinterpret_cast<const int4*>(m.twin)[x.f];
    const bool second = (e >> 31) != 0u;   // the corners 1 and 3 merge
    x.t = second ? q.y : q.x;
    x.n1 = second ? q.z : q.y;
    x.r = second ? q.w : q.z;
    x.n3 = second ? q.x : q.w;
    x.A = second ? w.y : w.x;
    x.C = second ? w.z : w.y;
    x.D = second ? w.w : w.z;
    x.B = second ? w.x : w.w;
    return x;
}
// The frame of list entry i as k_stage_sort left it: read whole instead of
// from two rows of which the list uses one in ten.
__device__ __forceinline__ MergeFrame load_frame(const Live& m, int64_t i, uint32_t e) {
    const int4 v = m.frame[2 * i], h = m.frame[2 * i + 1];
    return MergeFrame{(int32_t)(e & (uint32_t)kClaimFace), v.x, v.y, v.z, v.w, h.x, h.y, h.z, h.w};
}

// What vertex v is called after the stage: itself, or the vertex its last
// claim merges it into; -1 if that one is removed too.
__device__ __forceinline__ int32_t renamed(const Live& m, int32_t v) {
    const int32_t c = m.claim[v];
    if (!m.claimed_now(c)) return v;
    const int32_t g = c & kClaimFace;
    const int32_t t = m.em[g] == 1 ? m.quads[4 * (int64_t)g] : m.quads[4 * (int64_t)g + 1];
    return m.claimed_now(m.claim[t]) ? -1 : t;
}

constexpr uint32_t kListIrregular = 1u << 30;

// Appends the lanes' entries, one add per wave.
__device__ __forceinline__ void append_wave(bool has, uint32_t x, uint32_t* __restrict__ out, uint32_t* count) {
    const uint64_t k = __ballot(has);
    if (!k) return;
    uint32_t base = 0;
    const int leader = __ffsll((unsigned long long)k) - 1;
    if ((int)__lane_id() == leader) base = atomicAdd(count, (uint32_t)__popcll(k));
    base = (uint32_t)__shfl((int)base, leader, kWave);
    if (has) out[base + __builtin_amdgcn_mbcnt_hi((uint32_t)(k >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)k, 0u))] = x;
}

// Is a merge regular?  t: the fan f, A's face, B's face closes and is all of
// t's faces (valence 3 counts them); r: likewise with C and D.  Then the
// halfedges on the merged vertex are A, next(A), B, prev(B), C, prev(C), D,
// next(D), on its edges to n1, x, n3 and y: four groups of two if these four
// are distinct under their new names.
__global__ void __launch_bounds__(kBlock) k_stage_sort(Live m) {
    const int64_t n = (int64_t)m.S->nlist[m.stage];
    TMC_GRID_STRIDE(i, n) {
        const uint32_t e = m.list[i];
        const MergeFrame x = merge_frame(m, e);
        bool ok = false;
        if (reinterpret_cast<const uint32_t*>(m.flag)[x.f] == 0u && (x.A | x.B | x.C | x.D) >= 0) {
            const int32_t gA = x.A >> 2, gB = x.B >> 2, gC = x.C >> 2, gD = x.D >> 2;
            const int32_t nA = he_next(x.A), pB = he_prev(x.B), pC = he_prev(x.C), nD = he_next(x.D);
            const uint32_t* flag4 = reinterpret_cast<const uint32_t*>(m.flag);
            const uint32_t fl = flag4[gA] | flag4[gB] | flag4[gC] | flag4[gD];
            const int32_t oA = m.quads[x.A], oB = m.quads[x.B], oC = m.quads[x.C], oD = m.quads[x.D];
            const int32_t dA = m.quads[nA], dB = m.dest(x.B), dC = m.dest(x.C), dD = m.quads[nD];
            const int32_t tA = m.twin[nA], tD = m.twin[nD];
            const int32_t vx = m.dest(nA), vy = m.dest(nD);
            ok = fl == 0u && gA != gB && gC != gD && oA == x.n1 && dA == x.t && oB == x.t && dB == x.n3 &&
                 oC == x.r && dC == x.n1 && oD == x.n3 && dD == x.r && tA == pB && tD == pC;
            if (ok) {
                const int32_t X = renamed(m, vx), Y = renamed(m, vy);
                ok = !m.claimed_now(m.claim[x.t]) && X >= 0 && Y >= 0 && x.n1 != x.n3 && x.n1 != X && x.n1 != Y &&
                     x.n3 != X && x.n3 != Y && X != Y && X != x.t && Y != x.t;
            }
        }
        if (ok) {
            m.frame[2 * i] = make_int4(x.t, x.n1, x.r, x.n3);
            m.frame[2 * i + 1] = make_int4(x.A, x.C, x.D, x.B);
        } else {
            m.list[i] = e | kListIrregular;
            atomicMax(&m.last[x.t], m.tag(x.f));
        }
        append_wave(!ok, e, m.irr, &m.S->nirr[m.stage]);
    }
}

// The midpoint position and normalised mean normal of vertices a and b, to t
// (cpp_dmc/DualMarchingCubes.cpp:960-1000).
__device__ __forceinline__ void merge_geometry(const Live& m, int64_t t, int64_t a, int64_t b) {
    double np[3], nn[3];
#pragma unroll
    for (int c = 0; c < 3; c++) {
        np[c] = m.pos[3 * a + c] + 0.5 * (m.pos[3 * b + c] - m.pos[3 * a + c]);
        nn[c] = m.nrm[3 * a + c] + 0.5 * (m.nrm[3 * b + c] - m.nrm[3 * a + c]);
    }
    const double s = sqrt(nn[0] * nn[0] + nn[1] * nn[1] + nn[2] * nn[2]);
#pragma unroll
    for (int c = 0; c < 3; c++) {
        m.pos[3 * t + c] = np[c];
        m.nrm[3 * t + c] = nn[c] / s;
    }
}
// the two vertices a merge lies between, in the reference's order
__device__ __forceinline__ void merge_between(const MergeFrame& x, uint32_t e, int32_t& a, int32_t& b) {
    const bool second = (e >> 31) != 0u;
    a = second ? x.n3 : x.n1;
    b = second ? x.n1 : x.n3;
}

// A face that loses a corner at vertex v (which is neither moved nor removed).
__device__ __forceinline__ void lose_corner(const Live& m, int32_t v, int32_t f) {
    atomicSub(&m.val[v], 1);
    if ((m.hev[v] >> 2) == f) vs_or(m.vs, v, kVsRetake);
}

// The regular merges: write rows of the faces around that belong to no other
// merge.
__global__ void __launch_bounds__(kBlock) k_stage_merge(Live m) {
    const int64_t n = (int64_t)m.S->nlist[m.stage];
    TMC_GRID_STRIDE(i, n) {
        const uint32_t e = m.list[i];
        if (e & kListIrregular) continue;
        const MergeFrame x = load_frame(m, i, e);
        int32_t a, b;
        merge_between(x, e, a, b);
        merge_geometry(m, x.t, a, b);
        const int32_t nA = he_next(x.A), nD = he_next(x.D);
        m.twin[x.A] = x.C;
        m.twin[x.C] = x.A;
        m.twin[x.B] = x.D;
        m.twin[x.D] = x.B;
        m.quads[x.C] = x.t;
        m.quads[nD] = x.t;
        m.dead[x.f] = 1;
        m.val[x.t] = 4;
        m.hev[x.t] = max(max(nA, x.B), max(x.C, nD));
        lose_corner(m, x.n1, x.f);
        lose_corner(m, x.n3, x.f);
    }
}

// A vertex changed irregularly: its halfedges are paired again, its valence
// and he_v are counted again from them.
__device__ __forceinline__ void change_vertex(const Live& m, int32_t v) {
    vs_or(m.vs, v, m.changed());
    m.val[v] = 0;
    m.hev[v] = -1;
    m.head[v] = -1;
}

__global__ void __launch_bounds__(kBlock) k_stage_irregular(Live m) {
    const int64_t n = (int64_t)m.S->nirr[m.stage];
    if (n == 0) return;
    HeDelta cnt;
    TMC_GRID_STRIDE(i, n) {
        const uint32_t e = m.irr[i];
        const MergeFrame x = merge_frame(m, e);
        m.dead[x.f] = 1;
        if (m.last[x.t] == m.tag(x.f)) {
            int32_t a, b;
            merge_between(x, e, a, b);
            merge_geometry(m, x.t, a, b);
        }
        const int32_t v[2] = {x.t, x.r};
#pragma unroll
        for (int k = 0; k < 2; k++) {
            if (m.claimed_now(m.claim[v[k]])) vs_or(m.vs, v[k], kVsGone);
            const int32_t u = renamed(m, v[k]);
            if (u < 0) m.S->need_generic = 1u;
            else change_vertex(m, u);
        }
        lose_corner(m, x.n1, x.f);
        lose_corner(m, x.n3, x.f);
        // boundary halfedges of the face that end at n1 or n3
        if (x.A < 0) atomicSub(&m.val[x.n1], 1);
        if (x.D < 0) atomicSub(&m.val[x.n3], 1);
        const uint32_t fl = reinterpret_cast<const uint32_t*>(m.flag)[x.f];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const uint8_t b = (uint8_t)(fl >> (8 * k));
            cnt.add(b, -1);
            vol_delta(m, 4 * x.f + k, b, -1);
        }
    }
    cnt.flush(m.S->hep);
}

// Every live face with a corner that was removed or changed irregularly: the
// corners' new names (3333: a pattern face's corners are replaced), and its
// halfedges on a changed vertex linked into that vertex's list (entry h is
// halfedge h's); such faces are listed in m.list, which the merges are done
// with, their halfedges in m.em.  3-face records with such an end are dropped.
__device__ __forceinline__ uint32_t rewrite_face(const Live& m, int64_t f, const int4& q, const uint8_t (&s)[4],
                                                 bool is3333, HeDelta& cnt) {
    const uint8_t ch = m.changed();
    const bool pattern = is3333 && m.p[f] == 2;
    const int32_t x[4] = {q.x, q.y, q.z, q.w};
    int32_t r[4];
    uint8_t sr[4];
    bool lost = false;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        r[k] = x[k];
        if (pattern) r[k] = m.last[x[k]];
        else if (s[k] & kVsGone) r[k] = is3333 ? -1 : renamed(m, x[k]);
        if (r[k] < 0) {
            lost = true;
            r[k] = x[k];
        }
        sr[k] = r[k] == x[k] ? s[k] : m.vs[r[k]];
    }
    if (lost) m.S->need_generic = 1u;   // a removed corner without a new name
    reinterpret_cast<int4*>(m.quads)[f] = make_int4(r[0], r[1], r[2], r[3]);
    const int4 t4 = reinterpret_cast<const int4*>(m.twin)[f];
    const int32_t tw[4] = {t4.x, t4.y, t4.z, t4.w};
    const uint32_t fl = reinterpret_cast<const uint32_t*>(m.flag)[f];
    uint32_t aff = 0;   // halfedges to pair again
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int b = (k + 1) & 3;
        if (!((sr[k] | sr[b]) & ch)) continue;
        aff |= 1u << k;
        const int32_t h = (int32_t)(4 * f) + k;
        const uint8_t o = (uint8_t)(fl >> (8 * k));
        cnt.add(o, -1);
        vol_delta(m, h, o, -1);
        // a boundary halfedge leaves a vertex that is counted on
        if (tw[k] < 0 && !(s[b] & (ch | kVsGone))) atomicSub(&m.val[x[b]], 1);
        if (sr[k] & ch) {
            atomicAdd(&m.val[r[k]], 1);
            atomicMax(&m.hev[r[k]], h);
        }
        const int32_t w = (sr[k] & sr[b] & ch) ? min(r[k], r[b]) : (sr[k] & ch) ? r[k] : r[b];
        m.ent[h] = make_int4(atomicExch(&m.head[w], h), r[k], r[b], w);
    }
    if (aff) m.em[f] = (uint8_t)aff;
    return aff;
}

__global__ void __launch_bounds__(kBlock) k_stage_rewrite(Live m, int is3333) {
    __shared__ uint32_t buf[kListBuf], n[2];
    if (m.S->nirr[m.stage] == 0u) return;
    if (threadIdx.x == 0) n[0] = 0;
    __syncthreads();
    const ListBuf L{buf, n, m.list, &m.S->nent[m.stage]};
    const uint8_t ch = m.changed();
    HeDelta cnt;
    for_share((int64_t)m.S->nq, [&](int64_t f0, int64_t end) {
        int4 q[kListIlp];
        uint8_t s[kListIlp][4];
        bool hit[kListIlp];
#pragma unroll
        for (int u = 0; u < kListIlp; u++) {
            const int64_t f = f0 + u * kBlock;
            hit[u] = f < end && !m.dead[f];
            q[u] = f < end ? reinterpret_cast<const int4*>(m.quads)[f] : make_int4(0, 0, 0, 0);
        }
#pragma unroll
        for (int u = 0; u < kListIlp; u++) {
            s[u][0] = m.vs[q[u].x];
            s[u][1] = m.vs[q[u].y];
            s[u][2] = m.vs[q[u].z];
            s[u][3] = m.vs[q[u].w];
            const bool pattern = is3333 && hit[u] && m.p[f0 + u * kBlock] == 2;
            hit[u] = hit[u] && (pattern || ((s[u][0] | s[u][1] | s[u][2] | s[u][3]) & (ch | kVsGone)));
        }
#pragma unroll
        for (int u = 0; u < kListIlp; u++) {
            const int64_t f = f0 + u * kBlock;
            const uint32_t aff = hit[u] ? rewrite_face(m, f, q[u], s[u], is3333 != 0, cnt) : 0u;
            L.add(aff != 0u, (uint32_t)f);
        }
    }, [&] { L.end_turn(); });
    L.flush();
    const int64_t nr = min((int64_t)m.S->nrec, (int64_t)m.reccap);
    TMC_GRID_STRIDE(i, nr) {
        const BndRec r = m.recs[i];
        if (r.key == ~0ull) continue;
        const uint8_t s = m.vs[(int32_t)(r.key >> 32)] | m.vs[(int32_t)(r.key & 0xFFFFFFFFull)];
        if ((s & (ch | kVsGone)) || m.dead[r.lone >> 2]) m.recs[i].key = ~0ull;
    }
    cnt.flush(m.S->hep);
}

// The listed faces' linked halfedges, paired by vertex pair
// (cpp_dmc/DualMarchingCubes.cpp:574-669): all halfedges on a pair with a
// changed vertex are in that vertex's list (both changed: the smaller one's).
__global__ void __launch_bounds__(kBlock) k_stage_pair(Live m) {
    const int64_t n = 4 * (int64_t)m.S->nent[m.stage];
    if (n == 0) return;
    HeDelta cnt;
    TMC_GRID_STRIDE(i, n) {
        const uint32_t f = m.list[i >> 2];
        if (!((m.em[f] >> (i & 3)) & 1u)) continue;
        const int32_t h = (int32_t)(4u * f) + (int32_t)(i & 3);
        const int4 own = m.ent[h];
        const int32_t a = own.y, b = own.z;
        int32_t g[5];
#pragma unroll
        for (int k = 0; k < 5; k++) g[k] = 0x7FFFFFFF;
        int c = 0;
        for (int32_t e = m.head[own.w]; e >= 0;) {
            const int4 x = m.ent[e];
            if ((x.y == a && x.z == b) || (x.y == b && x.z == a)) {
                group_insert(g, e);
                c++;
            }
            e = x.x;
        }
        int32_t tw;
        uint8_t fl;
        twin_rule(m.quads, c, g, h, tw, fl);
        m.twin[h] = tw;
        m.flag[h] = fl;
        if (tw < 0) atomicAdd(&m.val[b], 1);
        cnt.add(fl, 1);
        vol_delta(m, h, fl, 1);
        if (c == 3 && g[0] == h) put_record(m.recs, &m.S->nrec, m.reccap, &m.S->ovf, three_record(m.quads, g, h));
    }
    cnt.flush(m.S->hep);
}

// The 3333 patterns among the candidates (cpp_dmc/DualMarchingCubes.cpp:
// 1190-1301): the four corners are claimed, the four faces around dropped.
__global__ void __launch_bounds__(kBlock) k_stage_claim3333(Live m) {
    __shared__ uint32_t buf[kListBuf], n[2];
    if (threadIdx.x == 0) n[0] = 0;
    __syncthreads();
    const ListBuf L{buf, n, m.list, &m.S->nlist[m.stage]};
    const int64_t nv = (int64_t)m.S->nv;
    for_share((int64_t)m.S->ncand[m.stage], [&](int64_t i0, int64_t end) {
        for (int u = 0; u < kListIlp; u++) {
            const int64_t i = i0 + u * kBlock;
            const int64_t f = i < end ? (int64_t)m.irr[i] : 0;
            int32_t vq[4], vo[4], fn[4];
            const bool has = i < end && pattern3333(f, m.quads, m.twin, m.flag, m.val, nv, vq, vo, fn);
            if (has) {
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    atomicMax(&m.claim[vq[k]], m.tag(f));
                    m.dead[fn[k]] = 2;
                }
            }
            L.add(has, (uint32_t)f);
        }
    }, [&] { L.end_turn(); });
    L.flush();
}

// The regular patterns: the corners' fans close over the four dropped faces,
// all edges around in groups of at most two, nothing else dropped beyond.
// The face takes the outer vertices, and its halfedges the place of the
// dropped faces' outer ones.
__global__ void __launch_bounds__(kBlock) k_stage_cut3333(Live m) {
    const int64_t n = (int64_t)m.S->nlist[m.stage];
    TMC_GRID_STRIDE(i, n) {
        const int32_t f = (int32_t)m.list[i];
        const int4 q = reinterpret_cast<const int4*>(m.quads)[f], w = reinterpret_cast<const int4*>(m.twin)[f];
        const int32_t vq[4] = {q.x, q.y, q.z, q.w}, T[4] = {w.x, w.y, w.z, w.w};
        const uint32_t* flag4 = reinterpret_cast<const uint32_t*>(m.flag);
        uint32_t fl = flag4[f];
        int32_t vo[4], X[4];
        bool ok = m.dead[f] == 0;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int32_t t = T[k], t1 = he_next(t), t2 = he_next(t1);
            fl |= flag4[t >> 2];
            ok = ok && m.claim[vq[k]] == m.tag(f) && m.quads[t] == vq[(k + 1) & 3] && m.quads[t1] == vq[k] &&
                 m.twin[t1] == he_prev(T[(k + 3) & 3]);
            vo[k] = m.quads[t2];
            X[k] = m.twin[t2];
            ok = ok && (X[k] < 0 || !m.dead[X[k] >> 2]);
#pragma unroll
            for (int l = 0; l < k; l++) ok = ok && (T[l] >> 2) != (t >> 2);
        }
        ok = ok && fl == 0u;
        if (ok) {
            reinterpret_cast<int4*>(m.quads)[f] = make_int4(vo[0], vo[1], vo[2], vo[3]);
            reinterpret_cast<int4*>(m.twin)[f] = make_int4(X[0], X[1], X[2], X[3]);
#pragma unroll
            for (int k = 0; k < 4; k++) {
                if (X[k] >= 0) m.twin[X[k]] = 4 * f + k;
                vs_or(m.vs, vo[k], kVsRetake);
            }
        } else {
            m.p[f] = 2;
        }
        append_wave(!ok, (uint32_t)f, m.irr, &m.S->nirr[m.stage]);
    }
}

__global__ void __launch_bounds__(kBlock) k_stage_irregular3333(Live m) {
    const int64_t n = (int64_t)m.S->nirr[m.stage];
    if (n == 0) return;
    HeDelta cnt;
    TMC_GRID_STRIDE(i, n) {
        const int32_t f = (int32_t)m.irr[i];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int32_t v = m.quads[4 * (int64_t)f + k], t = m.twin[4 * (int64_t)f + k];
            vs_or(m.vs, v, kVsGone);
            // the last pattern to claim a corner replaces it
            if (m.claim[v] == m.tag(f)) m.last[v] = m.quads[he_next(he_next(t))];
            // a dropped face, once: its corners that stay are changed
            const int32_t g = t >> 2;
            const uint32_t old = atomicOr(reinterpret_cast<uint32_t*>(m.dead) + (g >> 2), 4u << (8 * (g & 3)));
            if ((old >> (8 * (g & 3))) & 4u) continue;
            const uint32_t fl = reinterpret_cast<const uint32_t*>(m.flag)[g];
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const uint8_t b = (uint8_t)(fl >> (8 * c));
                cnt.add(b, -1);
                vol_delta(m, 4 * g + c, b, -1);
                const int32_t u = m.quads[4 * (int64_t)g + c];
                if (!removed(m.claim[u])) change_vertex(m, u);
            }
        }
    }
    cnt.flush(m.S->hep);
}

// ---------------------------------------------------------------------------
// The compaction at the end: kept vertices and live faces in their order.
// ---------------------------------------------------------------------------
// Vertices: positions and normals, he_v (-1 where the faces take it again),
// and the 3-face records under the new numbers.
__global__ void __launch_bounds__(kBlock) k_final_vertices(Live m, const int32_t* __restrict__ vmap,
                                                            const int32_t* __restrict__ qmap,
                                                            double* __restrict__ pos2, double* __restrict__ nrm2,
                                                            int32_t* __restrict__ hev2, BndRec* __restrict__ recs2) {
    const int64_t nv = (int64_t)m.S->nv;
    TMC_GRID_STRIDE(v, nv) {
        const int64_t y = vmap[v];
        if (y < 0) continue;
        double a[3], b[3];
#pragma unroll
        for (int c = 0; c < 3; c++) {
            a[c] = m.pos[3 * v + c];
            b[c] = m.nrm[3 * v + c];
        }
        const int32_t e = (m.vs[v] & kVsRetake) ? -1 : m.hev[v];
        const int32_t g = e < 0 ? -1 : qmap[e >> 2];
#pragma unroll
        for (int c = 0; c < 3; c++) {
            pos2[3 * y + c] = a[c];
            nrm2[3 * y + c] = b[c];
        }
        hev2[y] = g < 0 ? -1 : 4 * g + (e & 3);
    }
    const int64_t nr = min((int64_t)m.S->nrec, (int64_t)m.reccap);
    TMC_GRID_STRIDE(i, nr) {
        BndRec r = m.recs[i];
        if (r.key == ~0ull) continue;
        const int32_t y0 = vmap[(int32_t)(r.key >> 32)], y1 = vmap[(int32_t)(r.key & 0xFFFFFFFFull)];
        const int32_t g = qmap[r.lone >> 2];
        r.a = vmap[r.a];
        r.b = vmap[r.b];
        if (y0 < 0 || y1 < 0 || r.a < 0 || r.b < 0 || g < 0) continue;
        r.key = he_key(y0, y1);
        r.lone = 4 * g + (r.lone & 3);
        put_record(recs2, &m.S->nrec_final, m.reccap, &m.S->ovf, r);
    }
}

// Faces: corners, twins and flags (the markers of groups of more than four
// cleared), and he_v of the vertices that take it again.
__global__ void __launch_bounds__(kBlock) k_final_faces(Live m, const int32_t* __restrict__ vmap,
                                                         const int32_t* __restrict__ qmap,
                                                         int32_t* __restrict__ quads2, int32_t* __restrict__ twin2,
                                                         uint8_t* __restrict__ flag2, int32_t* __restrict__ hev2) {
    const int64_t nq = (int64_t)m.S->nq;
    TMC_GRID_STRIDE(f, nq) {
        const int32_t g = qmap[f];
        if (g < 0) continue;
        const int4 q = reinterpret_cast<const int4*>(m.quads)[f], t = reinterpret_cast<const int4*>(m.twin)[f];
        uint32_t fl = reinterpret_cast<const uint32_t*>(m.flag)[f];
        const uint8_t s[4] = {m.vs[q.x], m.vs[q.y], m.vs[q.z], m.vs[q.w]};
        const int4 r = make_int4(vmap[q.x], vmap[q.y], vmap[q.z], vmap[q.w]);
        auto he = [&](int32_t h) { return h < 0 ? -1 : 4 * qmap[h >> 2] + (h & 3); };
        reinterpret_cast<int4*>(quads2)[g] = r;
        reinterpret_cast<int4*>(twin2)[g] = make_int4(he(t.x), he(t.y), he(t.z), he(t.w));
        if (fl & 0x80808080u) fl &= ~(((fl & 0x80808080u) >> 7) * 0xFFu);
        reinterpret_cast<uint32_t*>(flag2)[g] = fl;
        const int32_t c[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
        for (int k = 0; k < 4; k++)
            if ((s[k] & kVsRetake) && c[k] >= 0) atomicMax(&hev2[c[k]], 4 * g + k);
    }
}

// Last of the halfedges: the 3-face overrides of he_v
// (cpp_dmc/DualMarchingCubes.cpp:603-637) -- of the records on a lone vertex
// the largest key writes -- and, after a simplification, the compacted counts
// become the mesh's.  Three steps over the records: clear the lone vertices'
// keys, take the largest, let its record write.
struct Overrides {
    Sizes* S;
    const BndRec* recs;
    uint32_t reccap;
    const int32_t* quads;
    unsigned long long* ovr;
    int32_t* he_v;
    int compacted;
    __device__ __forceinline__ int64_t count() const {
        return min((int64_t)(compacted ? S->nrec_final : S->nrec), (int64_t)reccap);
    }
    __device__ __forceinline__ void step(int which, int64_t i, int64_t nv) const {
        const BndRec r = recs[i];
        const int32_t v = quads[r.lone];
        if (!vid_ok(v, nv)) return;
        if (which == 0) __hip_atomic_store(&ovr[v], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        else if (which == 1) atomicMax(&ovr[v], r.key + 1ull);
        else if (__hip_atomic_load(&ovr[v], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == r.key + 1ull) he_v[v] = r.lone;
    }
    // (none of these counts is read by a thread that may still run)
    __device__ __forceinline__ void commit() const {
        if (!compacted) return;
        S->nv = S->nn;
        S->nq = S->qn;
        S->recmax = S->nrec > S->recmax ? S->nrec : S->recmax;
        S->nrec = S->nrec_final;
    }
};

// A pass with room for at most kFinishRecords records, the room that a context
// starts with (a smooth surface has none): one block does all three steps.  Its
// own stores and atomics meet in this block's L2; the waits order them.
constexpr int64_t kFinishRecords = 1024;
__global__ void __launch_bounds__(1024) k_finish(Overrides o) {
    const int64_t n = o.count(), nv = (int64_t)(o.compacted ? o.S->nn : o.S->nv);
    for (int which = 0; which < 3 && n > 0; which++) {
        for (int64_t i = threadIdx.x; i < n; i += blockDim.x) o.step(which, i, nv);
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        __builtin_amdgcn_s_waitcnt(0);
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        __syncthreads();
    }
    if (threadIdx.x == 0) o.commit();
}
// More, as noisy fields have: a launch per step.  223 / 1,003 / 1,903 / 7,995 /
// 23,565 records (noise three points thick) in one block 4.5 / 9.4 / 16.5 / 67
// / 274 us, in three launches 13.7 to 14.2.
__global__ void __launch_bounds__(kBlock) k_finish_step(Overrides o, int which) {
    const int64_t n = o.count(), nv = (int64_t)(o.compacted ? o.S->nn : o.S->nv);
    TMC_GRID_STRIDE(i, n) o.step(which, i, nv);
    if (which == 2 && blockIdx.x == 0 && threadIdx.x == 0) o.commit();
}

}  // namespace tmc
