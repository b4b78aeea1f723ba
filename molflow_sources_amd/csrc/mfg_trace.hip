// mfg_trace.hip -- HIP kernels of the MI355X test-particle tracer (gfx950).
//
// k_trace: one persistent launch traces a whole batch of desorptions. Each
// lane owns one particle in registers; dead lanes refill from a global work
// queue with one atomic per wave (ballot + mbcnt), first from the particles
// the previous launch parked. Per event the lanes of a wave walk an 8-wide
// BVH of 128 B nodes with 8-bit quantised FP32 boxes together, from one task
// stack in LDS (the top of the tree is copied to LDS per block); facets are
// tested in FP64. A lane then applies the event of reference
// src/Simulation/Particle.cpp:207-396 (desorption, bounce, absorption,
// transparent pass, teleport, link, leak, volume events). Tallies are u64 /
// FP64 atomics: lanes of a wave that update the same facet counter (or
// desorb from the same facet) add through one set of atomics, the counters
// of a few hot facets are summed per block in LDS, and the global counters
// are kept per lane and flushed once per wave at exit.
//
// Random numbers: Philox4x32-10 keyed by the variant seed, counter
// (particle index, block, 0); a lane draws them in the same order as the
// CPU restatement, so seeded runs are comparable event by event.
#include <hip/hip_runtime.h>

#include <mutex>
#include <type_traits>

#include "mfg_internal.h"

namespace {

constexpr double kPi = 3.14159265358979323846;
constexpr double kInv2p32 = 2.3283064365386962890625e-10;

// ------------------------------------------------------------------ RNG
__device__ __forceinline__ void philox10(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3, uint32_t k0,
                                         uint32_t k1, uint32_t& o0, uint32_t& o1, uint32_t& o2, uint32_t& o3) {
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        uint32_t lo0 = 0xD2511F53u * c0, hi0 = __umulhi(0xD2511F53u, c0);
        uint32_t lo1 = 0xCD9E8D57u * c2, hi1 = __umulhi(0xCD9E8D57u, c2);
        uint32_t n0 = hi1 ^ c1 ^ k0, n2 = hi0 ^ c3 ^ k1;
        c0 = n0; c1 = lo1; c2 = n2; c3 = lo0;
        k0 += 0x9E3779B9u; k1 += 0xBB67AE85u;
    }
    o0 = c0; o1 = c1; o2 = c2; o3 = c3;
}

__device__ __forceinline__ double u2d(uint32_t x) { return ((double)x + 0.5) * kInv2p32; }

struct Rng {
    uint32_t k0, k1, p0, p1, blk, b0, b1, b2, b3, avail;
    __device__ void init(uint64_t seed, uint64_t pid) {
        k0 = (uint32_t)seed; k1 = (uint32_t)(seed >> 32);
        p0 = (uint32_t)pid; p1 = (uint32_t)(pid >> 32);
        blk = 0; avail = 0;
    }
    __device__ __forceinline__ double rnd() {
        if (avail == 0) {
            philox10(p0, p1, blk, 0u, k0, k1, b0, b1, b2, b3);
            ++blk;
            avail = 4;
        }
        uint32_t r = b0;
        b0 = b1; b1 = b2; b2 = b3;
        --avail;
        return u2d(r);
    }
    __device__ double coin(uint32_t event, uint32_t facet) const {
        uint32_t o0, o1, o2, o3;
        philox10(p0, p1, event, 0x80000000u | facet, k0, k1, o0, o1, o2, o3);
        return u2d(o0);
    }
};

// The draws of one wall event: what the particle's block has left and the
// next block, so that the block function runs once per event for the whole
// wave; called at each draw that finds its lane's block empty, it ran at
// nearly every draw of every event for some lane (3 draws a bounce, 4 words
// a block). Rng's own state is unchanged until done().
struct EventDraws {
    Rng& g;
    uint32_t w0, w1, w2, w3, w4, w5, w6, w7, left;
    __device__ __forceinline__ EventDraws(Rng& r) : g(r) {
        philox10(g.p0, g.p1, g.blk, 0u, g.k0, g.k1, w4, w5, w6, w7);
        // the next block's words follow the `avail` words left
        const bool a1 = (g.avail & 1u) != 0, a2 = (g.avail & 2u) != 0, a4 = (g.avail & 4u) != 0;
        w0 = g.avail ? g.b0 : w4;
        w1 = g.avail > 1u ? g.b1 : (a1 ? w4 : w5);
        w2 = g.avail > 2u ? g.b2 : (a2 ? w4 : a1 ? w5 : w6);
        w3 = a4 ? g.b3 : (a2 ? (a1 ? w4 : w5) : a1 ? w6 : w7);
        const uint32_t x4 = a4 ? w4 : (a2 ? (a1 ? w5 : w6) : w7);   // avail 1..4 (0: past the end)
        const uint32_t x5 = a4 ? w5 : (a1 ? w6 : w7), x6 = a4 ? w6 : w7;
        w4 = x4; w5 = x5; w6 = x6;
        left = g.avail + 4u;
    }
    __device__ __forceinline__ double rnd() {
        if (left == 0) {
            // an event of more than 4 draws
            ++g.blk;
            philox10(g.p0, g.p1, g.blk, 0u, g.k0, g.k1, w0, w1, w2, w3);
            left = 4;
        }
        const uint32_t r = w0;
        w0 = w1; w1 = w2; w2 = w3; w3 = w4; w4 = w5; w5 = w6; w6 = w7;
        --left;
        return u2d(r);
    }
    __device__ __forceinline__ void done() {
        g.b0 = w0; g.b1 = w1; g.b2 = w2; g.b3 = w3;
        if (left >= 4u) g.avail = left - 4u;   // the next block untouched: drawn again later
        else { g.avail = left; ++g.blk; }
    }
};

// ------------------------------------------------------------------ math helpers
struct d3 { double x, y, z; };
__device__ __forceinline__ d3 mk(double x, double y, double z) { return {x, y, z}; }
__device__ __forceinline__ d3 add(d3 a, d3 b) { return {a.x + b.x, a.y + b.y, a.z + b.z}; }
__device__ __forceinline__ d3 sub(d3 a, d3 b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ d3 scl(double s, d3 a) { return {s * a.x, s * a.y, s * a.z}; }
__device__ __forceinline__ double dot(d3 a, d3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ double fdot(d3 a, d3 b) { return fma(a.x, b.x, fma(a.y, b.y, a.z * b.z)); }
__device__ __forceinline__ d3 cross(d3 a, d3 b) { return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x}; }
__device__ __forceinline__ double nrm(d3 a) { return sqrt(dot(a, a)); }
__device__ __forceinline__ d3 unitv(d3 a) { double n = nrm(a); return n > 0 ? scl(1.0 / n, a) : a; }
__device__ __forceinline__ d3 ld3(const double* p) { return {p[0], p[1], p[2]}; }

__device__ __forceinline__ void atomic_addd(double* p, double v) { unsafeAtomicAdd(p, v); }
__device__ __forceinline__ void atomic_addu(void* p, unsigned long long v) {
    atomicAdd(reinterpret_cast<unsigned long long*>(p), v);
}

__device__ __forceinline__ uint32_t mbcnt(uint64_t m) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}
__device__ __forceinline__ unsigned long long wave_sum_u(unsigned long long v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// ------------------------------------------------------------------ tables
struct XYRef { const double* x; const double* y; uint32_t n; };

__device__ __forceinline__ double interp_y(double x, XYRef t, bool logx, bool logy, bool extrapolate) {
    uint32_t n = t.n;
    if (n == 0) return 0.0;
    if (n == 1) return t.y[0];
    uint32_t i;
    if (x <= t.x[0]) {
        if (!extrapolate) return t.y[0];
        i = 0;
    } else if (x >= t.x[n - 1]) {
        if (!extrapolate) return t.y[n - 1];
        i = n - 2;
    } else {
        uint32_t lo = 0, hi = n - 1;
        while (hi - lo > 1) { uint32_t mid = (lo + hi) / 2; if (t.x[mid] <= x) lo = mid; else hi = mid; }
        i = lo;
    }
    double x0 = t.x[i], x1 = t.x[i + 1], y0 = t.y[i], y1 = t.y[i + 1];
    if (logx) { x0 = log10(x0); x1 = log10(x1); x = log10(x); }
    if (logy) { y0 = log10(y0); y1 = log10(y1); }
    double y = (x1 == x0) ? y0 : y0 + (x - x0) * (y1 - y0) / (x1 - x0);
    return logy ? pow(10.0, y) : y;
}

// interp_x with a guide table: guide[k] is the last point whose y is at or
// below k/K of the table's last y, so a lookup starts one or two points
// before the answer; the interval found is the binary search's.
__device__ double interp_x_guided(double y, XYRef t, const uint32_t* guide, uint32_t K) {
    uint32_t n = t.n;
    uint32_t i;
    double ylast = t.y[n - 1];
    if (y >= ylast) {
        i = n - 2;
    } else {
        uint32_t k = (uint32_t)fmax(0.0, fmin((double)(K - 1), y / ylast * (double)K));
        i = guide[k];
        while (i > 0 && t.y[i] > y) --i;
        while (i + 1 < n - 1 && t.y[i + 1] <= y) ++i;
    }
    double y0 = t.y[i], y1 = t.y[i + 1], x0 = t.x[i], x1 = t.x[i + 1];
    if (y1 == y0) return x0;
    return x0 + (y - y0) * (x1 - x0) / (y1 - y0);
}

// The same interval and value from the block's LDS copy of a Maxwell CDF:
// (speed, cumulative) points and one byte per guide entry. The guide only
// says where the search starts, so the scale K / last y may be rounded.
struct MaxwellLds {
    double2 p[MFG_MAXWELL_POINTS];
    uint8_t guide[MFG_MAXWELL_GUIDE];
};
static_assert(sizeof(MaxwellLds) == MFG_MAXWELL_LDS, "MFG_MAXWELL_LDS is the size of MaxwellLds");
__device__ __forceinline__ double maxwell_lds(const MaxwellLds* M, double y, double scale) {
    constexpr uint32_t n = MFG_MAXWELL_POINTS;
    uint32_t i = M->guide[(uint32_t)fmin((double)(MFG_MAXWELL_GUIDE - 1), y * scale)];
    double2 a = M->p[i], b = M->p[i + 1];
    while (i > 0 && a.y > y) { --i; b = a; a = M->p[i]; }
    while (i + 1 < n - 1 && b.y <= y) { ++i; a = b; b = M->p[i + 1]; }
    if (b.y == a.y) return a.x;
    return a.x + (y - a.y) * (b.x - a.x) / (b.y - a.y);
}

__device__ __forceinline__ double interp_x(double y, XYRef t) {
    uint32_t n = t.n;
    if (n == 1) return t.x[0];
    uint32_t i;
    if (y < t.y[0]) i = 0;
    else if (y >= t.y[n - 1]) i = n - 2;
    else {
        uint32_t lo = 0, hi = n - 1;
        while (hi - lo > 1) { uint32_t mid = (lo + hi) / 2; if (t.y[mid] <= y) lo = mid; else hi = mid; }
        i = lo;
    }
    double y0 = t.y[i], y1 = t.y[i + 1], x0 = t.x[i], x1 = t.x[i + 1];
    if (y1 == y0) return x0;
    return x0 + (y - y0) * (x1 - x0) / (y1 - y0);
}

// ------------------------------------------------------------------ geometry
__device__ __forceinline__ bool in_poly(const double* __restrict__ p, uint32_t n, double u, double v) {
    bool inside = false;
    double uj = p[2 * (n - 1)], vj = p[2 * (n - 1) + 1];
    for (uint32_t i = 0; i < n; ++i) {
        double ui = p[2 * i], vi = p[2 * i + 1];
        if ((vi > v) != (vj > v)) {
            double x = (uj - ui) * (v - vi) / (vj - vi) + ui;
            if (u < x) inside = !inside;
        }
        uj = ui; vj = vi;
    }
    return inside;
}

// in_poly for more than 4 vertices through the slab index stored after the
// (u,v) list: the same crossing predicate on the edges that straddle v
// (exactly those the loop above toggles on), found by a binary search over
// the sorted vertex heights.
__device__ __forceinline__ uint32_t low_bits(double d) { return (uint32_t)__double_as_longlong(d); }
__device__ bool in_poly_slabs(const double* __restrict__ p, uint32_t n, double u, double v) {
    const double* S = p + 2 * (size_t)n;
    const uint32_t m = low_bits(S[0]);
    const double* w = S + 1;
    if (!(v >= w[0] && v < w[m - 1])) return false;   // no straddling edge (NaN included)
    uint32_t lo = 0, hi = m - 1;                       // w[lo] <= v < w[hi]
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (w[mid] <= v) lo = mid; else hi = mid;
    }
    const uint32_t e0 = low_bits(S[1 + m + lo]), e1 = low_bits(S[2 + m + lo]);
    const double2* E = reinterpret_cast<const double2*>(S + 2 + 2 * (size_t)m);
    bool inside = false;
    for (uint32_t e = e0; e < e1; ++e) {
        const double2 a = E[2 * e], b = E[2 * e + 1];   // (u_i, v_i), (u_j, v_j)
        const double x = (b.x - a.x) * (v - a.y) / (b.y - a.y) + a.x;
        if (u < x) inside = !inside;
    }
    return inside;
}
__device__ __forceinline__ bool in_polygon(const double* __restrict__ p, uint32_t n, double u, double v) {
    return n > 4 ? in_poly_slabs(p, n, u, v) : in_poly(p, n, u, v);
}

// in_poly for a triangle held in registers: the same crossing tests in the
// same order as the loop above with n = 3.
__device__ __forceinline__ bool crossing(double ui, double vi, double uj, double vj, double u, double v) {
    if ((vi > v) != (vj > v)) {
        double x = (uj - ui) * (v - vi) / (vj - vi) + ui;
        return u < x;
    }
    return false;
}
__device__ __forceinline__ bool in_tri(double2 p0, double2 p1, double2 p2, double u, double v) {
    bool inside = false;
    if (crossing(p0.x, p0.y, p2.x, p2.y, u, v)) inside = !inside;
    if (crossing(p1.x, p1.y, p0.x, p0.y, u, v)) inside = !inside;
    if (crossing(p2.x, p2.y, p1.x, p1.y, u, v)) inside = !inside;
    return inside;
}
// in_poly for a quadrilateral held in registers (n = 4, same order)
__device__ __forceinline__ bool in_quad(const double* __restrict__ uv, double u, double v) {
    const double2* q = reinterpret_cast<const double2*>(uv);
    const double2 p0 = q[0], p1 = q[1], p2 = q[2], p3 = q[3];
    bool inside = false;
    if (crossing(p0.x, p0.y, p3.x, p3.y, u, v)) inside = !inside;
    if (crossing(p1.x, p1.y, p0.x, p0.y, u, v)) inside = !inside;
    if (crossing(p2.x, p2.y, p1.x, p1.y, u, v)) inside = !inside;
    if (crossing(p3.x, p3.y, p2.x, p2.y, u, v)) inside = !inside;
    return inside;
}

// A triangle's corner k on one axis: 0, 1 or the third value (code: which
// corner has 0, which has 1).
__device__ __forceinline__ double corner(uint32_t code, uint32_t k, double other) {
    return (code & 3u) == k ? 0.0 : ((code >> 2) & 3u) == k ? 1.0 : other;
}

// Ray/facet test on a leaf record; the same arithmetic, operation for
// operation, as the CPU restatement (explicit fma dot products, contraction
// off elsewhere). The record's 128 B are loaded together before the first
// decision (one round trip); polygons of 4 and more corners are read only
// when the ray meets the facet's rectangle.
__device__ __forceinline__ bool leaf_test(const LeafFacet* __restrict__ L, const LeafUV* __restrict__ LU,
                                          const double* __restrict__ poly, d3 P, d3 D, int32_t skip, double& t, double& u, double& v, int32_t& id, uint32_t& flags) {
    const uint4 hd = reinterpret_cast<const uint4*>(L)[0];
    const double2* q = reinterpret_cast<const double2*>(L);
    const double2 q1 = q[1], q2 = q[2], q3 = q[3], q4 = q[4], q5 = q[5], q6 = q[6], q7 = q[7];
    id = (int32_t)hd.x;
    flags = hd.y & MFG_LEAF_FLAGS;
    const uint32_t code = hd.y >> 24;
    const d3 O = mk(__longlong_as_double((long long)(((unsigned long long)hd.w << 32) | hd.z)), q1.x, q1.y);
    const d3 N = mk(q2.x, q2.y, q3.x), U = mk(q3.y, q4.x, q4.y), V = mk(q5.x, q5.y, q6.x);
    const double iu = q6.y, iv = code ? 1.0 / dot(V, V) : q7.y;
    double denom = fdot(N, D);
    d3 w = sub(O, P);
    t = fdot(N, w) / denom;
    d3 X = mk(fma(t, D.x, P.x), fma(t, D.y, P.y), fma(t, D.z, P.z));
    d3 r = sub(X, O);
    u = fdot(r, U) * iu;
    v = fdot(r, V) * iv;
    // non-short-circuit: every operand (the whole record) is needed here
    bool ok = (denom != 0.0) & (((flags & FF_2SIDED) != 0u) | !(denom > 0.0)) & (t > 0.0) &
              !((u < 0.0) | (u > 1.0) | (v < 0.0) | (v > 1.0)) & (id != skip);
    if (!ok) return false;
    if (code) {
        const uint32_t cv = code >> 4;
        return in_tri(make_double2(corner(code, 0, q7.x), corner(cv, 0, q7.y)),
                      make_double2(corner(code, 1, q7.x), corner(cv, 1, q7.y)),
                      make_double2(corner(code, 2, q7.x), corner(cv, 2, q7.y)), u, v);
    }
    const unsigned long long at = (unsigned long long)__double_as_longlong(q7.x);
    const double* p = poly + 2 * (size_t)(uint32_t)at;
    const uint32_t n = (uint32_t)(at >> 32);
    return n == 4u ? in_quad(LU->uv, u, v) : in_polygon(p, n, u, v);
}

struct Ray32 { float ox, oy, oz, ix, iy, iz; };

__device__ __forceinline__ float safe_inv(double d) {
    float f = (float)d;
    if (fabsf(f) < 1e-30f) f = (f < 0.0f) ? -1e-30f : 1e-30f;
    // correctly rounded: of 6 million rays from 500 to 900 model extents away
    // 105 lost their first hit with v_rcp_f32 (1 ulp) and not with this
    // division, 69 the other way round
    return 1.0f / f;
}

__device__ __forceinline__ Ray32 make_ray32(d3 P, d3 D) {
    return {(float)P.x, (float)P.y, (float)P.z, safe_inv(D.x), safe_inv(D.y), safe_inv(D.z)};
}

// A node's 128 B as eight 16-byte loads issued together (one round trip).
// Words: c0 = origin x,y,z + (ex, ey, ez, leaf mask) bytes; c1 = node_base,
// leaf_base, leaf counts, inner mask (byte 0); c2..c4 = low planes of x, y,
// z and c5..c7 = high planes, two FP16 steps per word (slot 2i low half,
// 2i + 1 high half).
struct NodeRegs {
    uint4 c0, c1, c2, c3, c4, c5, c6, c7;
};

__device__ __forceinline__ NodeRegs load_node(const BvhNode* __restrict__ nd) {
    const uint4* q = reinterpret_cast<const uint4*>(nd);
    NodeRegs n;
    n.c0 = q[0]; n.c1 = q[1]; n.c2 = q[2]; n.c3 = q[3]; n.c4 = q[4]; n.c5 = q[5]; n.c6 = q[6]; n.c7 = q[7];
    return n;
}

// A node from the block's LDS copy of the top of the tree, else from HBM.
__device__ __forceinline__ NodeRegs load_node_at(const BvhNode* __restrict__ nodes, const uint4* lnodes,
                                                 uint32_t n_lds, int32_t node) {
    if ((uint32_t)node < n_lds) {
        const uint4* q = lnodes + (size_t)node * 8;
        NodeRegs n;
        n.c0 = q[0]; n.c1 = q[1]; n.c2 = q[2]; n.c3 = q[3]; n.c4 = q[4]; n.c5 = q[5]; n.c6 = q[6]; n.c7 = q[7];
        return n;
    }
    return load_node(nodes + node);
}

__device__ __forceinline__ uint32_t node_leaves(const NodeRegs& n) { return n.c0.w >> 24; }
__device__ __forceinline__ uint32_t node_inner(const NodeRegs& n) { return n.c1.w & 0xffu; }
// inner child of slot c: the node_base-th node plus the inner slots before c
__device__ __forceinline__ int32_t node_inner_child(const NodeRegs& n, uint32_t c) {
    return (int32_t)n.c1.x + (int32_t)__popc(node_inner(n) & ((1u << c) - 1u));
}
// leaf child of slot c: (first record, facets); its records follow those of
// the leaf slots before c, each holding 1 + its 4-bit count facets
__device__ __forceinline__ uint32_t nibble_sum(uint32_t v) {
    const uint32_t t = (v & 0x0f0f0f0fu) + ((v >> 4) & 0x0f0f0f0fu);
    return (t * 0x01010101u) >> 24;
}
__device__ __forceinline__ void node_leaf_child(const NodeRegs& n, uint32_t c, uint32_t& first, uint32_t& cnt) {
    const uint32_t below = (1u << c) - 1u;
    const uint32_t cw = n.c1.z;
    first = n.c1.y + (uint32_t)__popc(node_leaves(n) & below) + nibble_sum(cw & ((1u << (4u * c)) - 1u));
    cnt = ((cw >> (4u * c)) & 15u) + 1u;
}
// 2^e as a float (|e| < 127)
__device__ __forceinline__ float exp2i(int e) { return __int_as_float((e + 127) << 23); }
// the FP16 step of slot 2i (lo) or 2i + 1 (hi) of a plane word, as a float
// (converted inside the v_fma_mix_f32 that uses it)
__device__ __forceinline__ float step_lo(uint32_t w) { return (float)__builtin_bit_cast(_Float16, (unsigned short)(w & 0xffffu)); }
__device__ __forceinline__ float step_hi(uint32_t w) { return (float)__builtin_bit_cast(_Float16, (unsigned short)(w >> 16)); }
__device__ __forceinline__ uint32_t word_of(const uint4& v, uint32_t i) {
    return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w;
}

// Slab test of the node's children against [0, tmax]: the hit mask.
// A bound q (an integer step) on an axis sits at o + q 2^e, so its ray
// parameter is (o + q 2^e - ray_o) / d = fma(q, 2^e/d, (o - ray_o)/d): two
// per-node constants per axis, then one fma per bound (q held as an FP16
// value, so conversion and fma are one v_fma_mix_f32 with the same single
// rounding). The quantised boxes enclose the FP64 boxes padded by 1e-5 of
// the model extent, far above the FP32 rounding of these steps, so the
// test never drops a box that holds an FP64 hit: a ray through a point of
// the unpadded box spends at least 1e-5 extent / |d| of its parameter
// inside the padded one (within [0, tmax] as well, since tmax is at or
// beyond that hit), against FP32 errors near 1e-7 extent / |d|, so no
// tolerance is added to a <= b. The errors grow with the distance R of the
// ray's origin, to about 3e-7 R / |d| (five roundings), so this holds up to
// R of some 30 extents; farther out a hit near a box's edge can be lost (1 of
// 200,000 at 320 extents).
__device__ __forceinline__ uint32_t node_hits(const NodeRegs& n, const Ray32& r, float tmax) {
    const float ox = __uint_as_float(n.c0.x), oy = __uint_as_float(n.c0.y), oz = __uint_as_float(n.c0.z);
    const uint32_t ew = n.c0.w;
    const float ax = exp2i((int)(int8_t)(ew & 0xffu)) * r.ix, ay = exp2i((int)(int8_t)((ew >> 8) & 0xffu)) * r.iy;
    const float az = exp2i((int)(int8_t)((ew >> 16) & 0xffu)) * r.iz;
    const float bx = (ox - r.ox) * r.ix, by = (oy - r.oy) * r.iy, bz = (oz - r.oz) * r.iz;
    // fma(q, a, b) is monotonic in q, rising when the axis' 1/d is >= 0: the
    // low bound is then the entry plane and the high one the exit plane, and
    // the reverse otherwise (an empty slot, low 255 > high 0, still misses)
    const bool px = r.ix >= 0.0f, py = r.iy >= 0.0f, pz = r.iz >= 0.0f;
    const uint4 nx = px ? n.c2 : n.c5, fx = px ? n.c5 : n.c2;
    const uint4 ny = py ? n.c3 : n.c6, fy = py ? n.c6 : n.c3;
    const uint4 nz = pz ? n.c4 : n.c7, fz = pz ? n.c7 : n.c4;
    uint32_t mask = 0;
#pragma unroll
    for (uint32_t c = 0; c < 8; ++c) {
        const uint32_t i = c >> 1;
        const uint32_t wnx = word_of(nx, i), wfx = word_of(fx, i), wny = word_of(ny, i);
        const uint32_t wfy = word_of(fy, i), wnz = word_of(nz, i), wfz = word_of(fz, i);
        const bool hi = (c & 1u) != 0;
        const float tnx = fmaf(hi ? step_hi(wnx) : step_lo(wnx), ax, bx), tfx = fmaf(hi ? step_hi(wfx) : step_lo(wfx), ax, bx);
        const float tny = fmaf(hi ? step_hi(wny) : step_lo(wny), ay, by), tfy = fmaf(hi ? step_hi(wfy) : step_lo(wfy), ay, by);
        const float tnz = fmaf(hi ? step_hi(wnz) : step_lo(wnz), az, bz), tfz = fmaf(hi ? step_hi(wfz) : step_lo(wfz), az, bz);
        float a = fmaxf(fmaxf(tnx, tny), fmaxf(tnz, 0.0f));
        float b = fminf(fminf(tfx, tfy), fminf(tfz, tmax));
        if (a <= b) mask |= 1u << c;
    }
    return mask & (node_leaves(n) | node_inner(n));
}

__device__ __forceinline__ float widen(double t) {
    if (t > 3.0e38) return 3.0e38f;
    return (float)t * 1.000004f + 1e-30f;
}

struct HitRec { int32_t facet; double t; };

// ---------------------------------------------------------------- DES_ANGLEMAP
// Sampling of a recorded incident-angle map (AnglemapGeneration.cpp:15-410),
// on the table block described in TraceParams::am_src. lower_index is the
// index of the last CDF value <= key (-1 below the first); weigh(a, b, w) =
// a + (b - a) * w.
struct AmSrc {
    int W, L, H;
    double limit, ratio, total;
    const double *line, *cdf, *pc, *pp;
};
__device__ __forceinline__ AmSrc am_view(const double* b) {
    AmSrc A;
    A.W = (int)b[0]; A.L = (int)b[1]; A.H = (int)b[2];
    A.limit = b[3]; A.ratio = b[4]; A.total = b[5];
    const int T = A.L + A.H;
    A.line = b + 6; A.cdf = A.line + T; A.pc = A.cdf + T; A.pp = A.pc + (size_t)T * A.W;
    return A;
}
__device__ __forceinline__ double am_weigh(double a, double b, double w) { return a + (b - a) * w; }
__device__ int am_lower_index(double key, const double* A, int n) {
    int lo = 0, hi = n;   // first element > key
    while (lo < hi) { int mid = (lo + hi) / 2; if (A[mid] <= key) lo = mid + 1; else hi = mid; }
    return lo - 1;
}
__device__ int am_weighed_lower_index(double key, double w, const double* A, const double* B, int n) {
    int lo = 0, hi = n;
    while (lo < hi) { int mid = (lo + hi) / 2; if (am_weigh(A[mid], B[mid], w) <= key) lo = mid + 1; else hi = mid; }
    return lo - 1;
}
__device__ __forceinline__ double am_theta(const AmSrc& A, double ti) {
    if ((size_t)ti < (size_t)A.L) return A.limit * ti / (double)A.L;
    return A.limit + (kPi / 2.0 - A.limit) * (ti - (double)A.L) / (double)A.H;
}
__device__ __forceinline__ double am_phi(const AmSrc& A, double pi_) {
    double w = (double)A.W;
    double c = (pi_ < w) ? pi_ : pi_ - w;
    return -kPi + 2.0 * kPi * c / w;
}
__device__ double am_phi_pdf(const AmSrc& A, double ti, int plo) {
    const int W = A.W, T = A.L + A.H;
    const size_t p = (size_t)(((plo % W) + W) % W);
    if (ti < 0.5) return A.pp[p];
    if (ti > (double)T - 0.5) return A.pp[(size_t)(T - 1) * W + p];
    size_t tl = (size_t)(ti - 0.5);
    double ov = ti - 0.5 - (double)tl;
    return am_weigh(A.pp[tl * W + p], A.pp[(tl + 1) * W + p], ov);
}
__device__ double am_phi_cdf(const AmSrc& A, double ti, int plo) {
    const int W = A.W, L = A.L, T = A.L + A.H;
    auto line = [&](size_t t) { return (plo < W) ? A.pc[t * W + plo] : 1.0 + A.pc[t * W]; };
    if (ti < (double)L) {
        if (ti < 0.5) return line(0);
        if (ti > (double)L - 0.5) return line((size_t)(L - 1));
    } else {
        if (ti < (double)L + 0.5) return line((size_t)L);
        if (ti > (double)T - 0.5) return line((size_t)(T - 1));
    }
    size_t tl = (size_t)(ti - 0.5);
    double ov = ti - 0.5 - (double)tl;
    return am_weigh(line(tl), line(tl + 1), ov);
}
__device__ void am_generate_theta(const AmSrc& A, double r, double& theta, int& tlo, double& ov) {
    const int L = A.L, H = A.H;
    const double* cdf = A.cdf;
    auto quad = [&](int t, double c) {
        double step = am_theta(A, (double)t + 1.5) - am_theta(A, (double)t + 0.5);
        double b = A.line[t] / A.total / step;
        double a = 0.5 * (A.line[t + 1] - A.line[t]) / A.total / (step * step);
        double dy = r - c;
        double dx = (-b + sqrt(b * b + 4 * a * dy)) / (2 * a);
        return dx / step;
    };
    if (r < A.ratio) {
        tlo = am_lower_index(r, cdf, L);
        if (tlo == -1) {
            ov = 0.5 * r / cdf[0];
            theta = am_theta(A, ov);
        } else if (tlo == L - 1) {
            ov = 0.5 * (r - cdf[tlo]) / (A.ratio - cdf[tlo]);
            theta = am_theta(A, (double)tlo + 0.5 + ov);
        } else {
            if (A.line[tlo] == A.line[tlo + 1]) ov = (r - cdf[tlo]) / (cdf[tlo + 1] - cdf[tlo]);
            else ov = quad(tlo, cdf[tlo]);
            theta = am_theta(A, (double)tlo + 0.5 + ov);
        }
    } else {
        tlo = L + am_lower_index(r, cdf + L, H);
        if (tlo == L - 1) {
            ov = 0.5 * (r - A.ratio) / (cdf[L] - A.ratio);
            theta = am_theta(A, (double)L + ov);
        } else if (tlo == L + H - 1) {
            ov = 0.5 * (r - cdf[tlo]) / (1.0 - cdf[tlo]);
            theta = am_theta(A, (double)tlo + 0.5 + ov);
        } else {
            if (A.line[tlo] == A.line[tlo + 1]) ov = (r - cdf[tlo]) / (cdf[tlo + 1] - cdf[tlo]);
            else ov = quad(tlo, cdf[tlo]);
            theta = am_theta(A, (double)tlo + 0.5 + ov);
        }
    }
}
__device__ double am_generate_phi(const AmSrc& A, int tlo, double ov, double r) {
    const int W = A.W, L = A.L, T = A.L + A.H;
    if (W == 1) return -kPi + 2.0 * kPi * r;
    int plo;
    double w;
    const double* C = A.pc;
    auto edge = [&](int t) {
        r += C[(size_t)t * W];
        plo = am_lower_index(r, C + (size_t)t * W, W);
        w = ov;
    };
    auto between = [&](int t) {
        double div = A.line[t] * (1.0 - ov) + A.line[t + 1] * ov;
        w = div > 0.0 ? (ov * A.line[t + 1]) / div : ov;
        r += am_weigh(C[(size_t)t * W], C[(size_t)(t + 1) * W], w);
        plo = am_weighed_lower_index(r, w, C + (size_t)t * W, C + (size_t)(t + 1) * W, W);
    };
    if (tlo < L) {
        if (tlo == -1) edge(0);
        else if (tlo == L - 1) edge(tlo);
        else between(tlo);
    } else {
        if (tlo == L - 1) edge(L);
        else if (tlo == T - 1) edge(tlo);
        else between(tlo);
    }
    const double ti = (double)tlo + 0.5 + w;
    double pov;
    if (plo == -1) {
        pov = 0.5 * r / am_phi_cdf(A, ti, 0);
        return am_phi(A, pov);
    }
    double p0 = am_phi_pdf(A, ti, plo), p1 = am_phi_pdf(A, ti, plo + 1);
    if (p0 == p1) {
        double c0 = am_phi_cdf(A, ti, plo);
        pov = (r - c0) / (am_phi_cdf(A, ti, plo + 1) - c0);
    } else {
        double step = 2.0 * kPi / (double)W;
        double c = am_phi_cdf(A, ti, plo);
        double b = p0 / step;
        double a = 0.5 * (p1 - p0) / (step * step);
        double dy = r - c;
        double D = b * b + 4 * a * dy;
        if (D < 0) pov = (r - c) / (am_phi_cdf(A, ti, ((plo + 1) % W + W) % W) - c);
        else pov = ((-b + sqrt(b * b + 4 * a * dy)) / (2 * a)) / step;
    }
    return am_phi(A, (double)plo + 0.5 + pov);
}

__device__ __forceinline__ double td_opacity(const TraceParams& P, const DVariant* var, int32_t f, double time) {
    const DPhys& ph = P.phys[f];
    const DTable tb = P.params[var->param_base + ph.opacity_param];
    return interp_y(time, XYRef{P.tab_x + tb.off, P.tab_y + tb.off, tb.n}, tb.log_x, tb.log_y, false);
}

// Traversal stack of one lane (the second walk of a transparent model): the
// first `lds_cap` entries in LDS (laid out [entry][lane]), deeper entries
// (rare) in a per-lane global area.
struct LaneStack {
    uint32_t* lds;
    uint32_t lds_cap, cap;
    int32_t* spill;
    __device__ __forceinline__ void push(uint32_t& sp, int32_t v) const {
        if (sp < lds_cap) {
            lds[sp * 64u] = (uint32_t)v;
            ++sp;
        } else if (sp < cap) {
            spill[sp - lds_cap] = v;
            ++sp;
        }
    }
    __device__ __forceinline__ int32_t pop(uint32_t& sp) const {
        --sp;
        return sp < lds_cap ? (int32_t)lds[sp * 64u] : spill[sp - lds_cap];
    }
};

// The same value, unknown to the optimiser: what is computed from it belongs
// to this place of the loop instead of being kept in registers all through
// it (LDS addresses of a lane's slots cost an instruction or two).
__device__ __forceinline__ uint32_t here(uint32_t v) {
    asm volatile("" : "+v"(v));
    return v;
}

// Orders this wave's LDS accesses before and after it (the hardware runs
// them in order; this keeps the compiler from moving them or from splitting
// the control flow around it).
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Inclusive sum over the lanes below and including this one (all 64 active).
__device__ __forceinline__ uint32_t wave_scan(uint32_t v) {
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false);   // row_shr:1
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false);   // row_bcast:15
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false);   // row_bcast:31
    return v;
}

// CH children of a node against a ray (the test of node_hits for the slots
// from c on), from the node's header and those slots' plane steps.
template <int CH>
struct ChildRegs {
    typedef typename std::conditional<CH == 1, uint16_t, uint32_t>::type Steps;   // CH FP16 steps
    uint4 c0, c1;
    Steps lx, ly, lz, hx, hy, hz;
};
template <int CH, typename Q>
__device__ __forceinline__ ChildRegs<CH> load_child(const Q* nd, uint32_t part) {
    const uint4* q = reinterpret_cast<const uint4*>(nd);
    const auto* h = reinterpret_cast<const typename ChildRegs<CH>::Steps*>(nd) + 16 / CH + part;
    constexpr int A = 8 / CH;   // one axis
    return {q[0], q[1], h[0], h[A], h[2 * A], h[3 * A], h[4 * A], h[5 * A]};
}
__device__ __forceinline__ float half_bits(uint32_t v) { return (float)__builtin_bit_cast(_Float16, (unsigned short)v); }
// bit k: child k of the CH is entered before tmax (a slot without a child is
// masked by the caller)
template <int CH>
__device__ __forceinline__ uint32_t child_hits(const ChildRegs<CH>& n, const Ray32& r, float tmax) {
    const uint32_t ew = n.c0.w;
    const float ax = exp2i((int)(int8_t)(ew & 0xffu)) * r.ix, ay = exp2i((int)(int8_t)((ew >> 8) & 0xffu)) * r.iy;
    const float az = exp2i((int)(int8_t)((ew >> 16) & 0xffu)) * r.iz;
    const float bx = (__uint_as_float(n.c0.x) - r.ox) * r.ix, by = (__uint_as_float(n.c0.y) - r.oy) * r.iy;
    const float bz = (__uint_as_float(n.c0.z) - r.oz) * r.iz;
    const bool px = r.ix >= 0.0f, py = r.iy >= 0.0f, pz = r.iz >= 0.0f;
    const uint32_t nx = px ? n.lx : n.hx, fx = px ? n.hx : n.lx, ny = py ? n.ly : n.hy, fy = py ? n.hy : n.ly;
    const uint32_t nz = pz ? n.lz : n.hz, fz = pz ? n.hz : n.lz;
    uint32_t m = 0;
#pragma unroll
    for (int k = 0; k < CH; ++k) {
        const int sh = 16 * k;
        const float a = fmaxf(fmaxf(fmaf(half_bits(nx >> sh), ax, bx), fmaf(half_bits(ny >> sh), ay, by)),
                              fmaxf(fmaf(half_bits(nz >> sh), az, bz), 0.0f));
        const float b = fminf(fminf(fmaf(half_bits(fx >> sh), ax, bx), fmaf(half_bits(fy >> sh), ay, by)),
                              fminf(fmaf(half_bits(fz >> sh), az, bz), tmax));
        if (a <= b) m |= 1u << k;
    }
    return m;
}

// A node step of a wave with at most 8 CH tasks on its stack: 8 / CH lanes a
// node, CH children a lane. False, with nothing done, if the facets of the
// leaves met might not fit the list.
template <int CH>
__device__ __forceinline__ bool few_nodes(const TraceParams& P, WaveLds& W, const uint4* lnodes, uint32_t lane,
                                          uint32_t& top, uint32_t& waiting) {
    constexpr uint32_t G = 8u / CH;
    const uint32_t bits = P.task_bits, low = (1u << bits) - 1u;
    const uint32_t part = lane % G, group = lane / G;
    const bool on = group < top;
    uint32_t tag = 0, hit = 0, im = 0, lm = 0;
    uint4 hd{};
    if (on) {
        const uint32_t w = W.nodes[top - 1u - group], ray = w >> bits, node = w & low;
        tag = w & ~low;
        ChildRegs<CH> nd;
        if (node < P.lds_nodes) nd = load_child<CH>(lnodes + (size_t)node * 8, part);
        else nd = load_child<CH>(P.nodes + node, part);
        const float4 a = W.ra[ray], b = W.rb[ray];
        im = nd.c1.w & 0xffu;
        lm = nd.c0.w >> 24;
        hit = child_hits<CH>(nd, Ray32{a.x, a.y, a.z, b.x, b.y, b.z}, a.w) << (CH * part);
        hd = nd.c1;
    }
    uint64_t leaves[CH];
    uint32_t n_leaves = 0;
#pragma unroll
    for (int k = 0; k < CH; ++k) {
        leaves[k] = __ballot((hit & lm) >> (CH * part + k) & 1u);
        n_leaves += (uint32_t)__popcll(leaves[k]);
    }
    if (CH > 1 && waiting + n_leaves * P.child_lanes > MFG_WALK_LEAVES) return false;
    wave_sync();
    top = 0;
#pragma unroll
    for (int k = 0; k < CH; ++k) {
        const uint32_t c = CH * part + k, below = (1u << c) - 1u;
        const bool inner = ((hit & im) >> c) & 1u;
        const uint64_t m = __ballot(inner);
        if (inner) W.nodes[top + mbcnt(m)] = tag | (hd.x + (uint32_t)__popc(im & below));
        top += (uint32_t)__popcll(m);
        if (leaves[k]) {
            const bool leaf = ((hit & lm) >> c) & 1u;
            const uint32_t first = hd.y + (uint32_t)__popc(lm & below) + nibble_sum(hd.z & ((1u << (4u * c)) - 1u));
            const uint32_t cnt = leaf ? ((hd.z >> (4u * c)) & 15u) + 1u : 0u;
            uint64_t ml = leaves[k];
            for (uint32_t i = 0; ml; ml = __ballot(cnt > ++i)) {
                if (cnt > i) W.leaves[waiting + mbcnt(ml)] = tag | (first + i);
                waiting += (uint32_t)__popcll(ml);
            }
        }
    }
    wave_sync();
    return true;
}

// What the opacity coin of a ray needs from the lane that owns it.
struct CoinState {
    uint32_t k0, k1, p0, p1, event;
    double time;
    const DVariant* var;
};

// Nearest hard hit of the wave's up to 64 rays, walked together: ray r sits
// in slot r of W (walk_load), and the wave shares one stack of (ray, node)
// tasks and one list of (ray, facet record) tasks. A node step gives each
// lane one of the topmost tasks, whichever ray it belongs to; the inner
// children hit go back on the stack and the facets of the leaf children hit
// into the list, at offsets from one scan over the lanes. A facet step
// gives each lane one record. A facet step runs once 64 records wait or no
// node does, so both kinds of step run with nearly all lanes at work as
// long as the wave has work, and a ray whose walk is long is helped by the
// lanes whose rays are done: with one ray per lane instead (each lane its
// own stack, leaves tested by wave vote) 14 % of the lanes were active on
// the beam pipe, for 28 node and 21 facet iterations per wave where the 64
// rays' 11 nodes and 5 facets each fill about 18. Beam pipe (1e5 facets, 6e5
// desorptions a launch): 121.5 -> 91.3 ms per launch, its drain 166 -> 82 ms;
// 2e4 low-flux particles (all tail) 456 -> 158 ms; the 1e6-particle tube 7.7
// -> 5.7 ms.
//
// The nearest hit is the minimum over the same facet tests, with ties going
// to the lower facet id, so it does not depend on the order or the lanes
// the tests run on.
//
// With at most 8 (16) tasks on the stack (a wave with few rays: a run's
// tail, or a small run) a node step gives each of them 8 (4) lanes, one for
// each child (two): the serial chain of 8 box tests and the loops that push
// the children shrink to one or two tests and stores a lane.
//
// A wave with at most kSeedRays rays starts them at the children of their
// roots (Root::first): the step that tests a root's 8 boxes for one ray has 8
// of 64 lanes at work, and the next one has lanes for all 8 children anyway.
// 16 variants 137.9 -> 131.2 ms, 5k-facet pipe 25.6 -> 25.0, 1000 tube
// particles 0.80 -> 0.77; with up to 8 rays (a full node step) 134.6, 25.7
// and 0.79, with 16 138 and low flux 73.8 -> 81.4.
//
// Bounds. A node step commits the tasks of its first lanes only, as many as
// leave the stack below its capacity less a reserve and the list within
// its capacity; the other tasks stay where they are. Lane 0 (the topmost
// task) may use the reserve, so once the stack is up to it the walk is depth
// first, which adds at most width - 1 entries a level: the reserve holds
// that for the deepest tree the host accepts. The list has room for lane
// 0's facets (8 leaves of 16) whenever a node step runs (below 64 waiting).
constexpr uint32_t kSeedRays = 2;
template <bool TRANSP>
__device__ void walk(const TraceParams& P, WaveLds& W, PassLds* pass, const uint4* lnodes, uint32_t lane, bool live, Root root,
                     const CoinState& cs) {
    const uint32_t bits = P.task_bits, low = (1u << bits) - 1u;
    uint32_t top, waiting = 0;   // wave-uniform
    {
        const bool on = live && root.node >= 0;
        uint64_t m = __ballot(on);
        top = (uint32_t)__popcll(m);
        if (top <= kSeedRays) {
            for (top = 0; m; m &= m - 1ull) {
                const uint32_t ray = (uint32_t)__builtin_ctzll(m);
                const uint32_t s = (uint32_t)__builtin_amdgcn_readlane((int)root.first, (int)ray);
                if (lane < (s & 15u)) W.nodes[top + lane] = (ray << bits) | ((s >> 4) + lane);
                top += s & 15u;
            }
        } else if (on) {
            W.nodes[mbcnt(m)] = (lane << bits) | (uint32_t)root.node;
        }
    }
    wave_sync();
    while (top + waiting != 0) {
        if (top != 0 && top <= 16u && waiting < 64u && P.child_lanes) {
            if (top <= 8u ? few_nodes<1>(P, W, lnodes, lane, top, waiting) : few_nodes<2>(P, W, lnodes, lane, top, waiting)) continue;
        }
        if (waiting < 64u && top != 0) {
            const bool on = lane < top;
            uint32_t tag = 0, inner = 0, im = 0, lm = 0, cw = 0, own = 0;
            int32_t node_base = 0;
            NodeRegs nd{};
            if (on) {
                const uint32_t w = W.nodes[top - 1u - lane], ray = w >> bits;
                tag = w & ~low;
                nd = load_node_at(P.nodes, lnodes, P.lds_nodes, (int32_t)(w & low));
                const float4 a = W.ra[ray], b = W.rb[ray];
                const Ray32 r{a.x, a.y, a.z, b.x, b.y, b.z};
                const uint32_t m = node_hits(nd, r, a.w);   // children entering before the nearest hit
                inner = node_inner(nd);
                im = m & inner;
                lm = m & node_leaves(nd);
                cw = nd.c1.z;
                node_base = (int32_t)nd.c1.x;
                // facets of the hit leaves: one more than each one's 4-bit count
                uint32_t e = (lm | (lm << 12)) & 0x000f000fu;
                e = (e | (e << 6)) & 0x03030303u;
                e = (e | (e << 3)) & 0x11111111u;
                own = (uint32_t)__popc(im) | (((uint32_t)__popc(lm) + nibble_sum(cw & (e * 15u))) << 16);
            }
            const uint32_t upto = wave_scan(own);
            // lanes that commit: a prefix
            const uint32_t after = top - 1u - lane + (upto & 0xffffu);
            const bool fits = on && after <= (lane == 0 ? MFG_WALK_NODES : MFG_WALK_NODES - MFG_WALK_RESERVE) &&
                              waiting + (upto >> 16) <= MFG_WALK_LEAVES;
            const uint64_t miss = __ballot(!fits);
            const uint32_t n = miss ? (uint32_t)__builtin_ctzll(miss) : 64u;
            const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)upto, (int)n - 1);
            wave_sync();
            if (lane < n) {
                uint32_t at = top - n + (total & 0xffffu) - (upto & 0xffffu);   // lane 0's children on top
                while (im) {
                    const uint32_t c = (uint32_t)__builtin_ctz(im);
                    im &= im - 1u;
                    W.nodes[at++] = tag | (uint32_t)(node_base + (int32_t)__popc(inner & ((1u << c) - 1u)));
                }
                at = waiting + ((upto - own) >> 16);
                while (lm) {
                    const uint32_t c = (uint32_t)__builtin_ctz(lm);
                    lm &= lm - 1u;
                    uint32_t first, cnt;
                    node_leaf_child(nd, c, first, cnt);
                    for (uint32_t k = 0; k < cnt; ++k) W.leaves[at++] = tag | (first + k);
                }
            }
            top = (uint32_t)__builtin_amdgcn_readfirstlane((int)(top - n + (total & 0xffffu)));
            waiting = (uint32_t)__builtin_amdgcn_readfirstlane((int)(waiting + (total >> 16)));
            wave_sync();
        } else {
            const uint32_t n = waiting < 64u ? waiting : 64u;
            waiting -= n;
            uint32_t ray = 0, rec = 0;
            double t = 0.0, u, v;
            int32_t f = -1;
            uint32_t fl = FF_OPAQUE;
            bool hit = false;
            if (lane < n) {
                const uint32_t w = W.leaves[waiting + lane];
                ray = w >> bits;
                rec = w & low;
                const double2 a = W.p01[ray], b = W.p2d0[ray], c = W.d12[ray];
                hit = leaf_test(P.leaves + rec, P.leaf_uv + rec, P.poly, mk(a.x, a.y, b.x), mk(b.y, c.x, c.y),
                                __float_as_int(W.rb[ray].w), t, u, v, f, fl);
            }
            if constexpr (TRANSP) {
                const bool coin = hit && !(fl & FF_OPAQUE);
                if (__ballot(coin)) {
                    // the ray's stream, event and clock, from the lane that owns it
                    Rng g;
                    g.k0 = __shfl(cs.k0, ray, 64); g.k1 = __shfl(cs.k1, ray, 64);
                    g.p0 = __shfl(cs.p0, ray, 64); g.p1 = __shfl(cs.p1, ray, 64);
                    const uint32_t ev = __shfl(cs.event, ray, 64);
                    const double tm = __shfl(cs.time, ray, 64);
                    const DVariant* var = (const DVariant*)__shfl((unsigned long long)cs.var, ray, 64);
                    if (coin) {
                        double op = (fl & FF_TD_OPACITY) ? td_opacity(P, var, f, tm) : (double)P.phys[f].opacity;
                        if (op < 1.0) hit = (op > 0.0) && g.coin(ev, (uint32_t)(f - (int32_t)var->facet_base)) < op;
                        if (!hit) {
                            const uint32_t k = atomicAdd(&pass->n[ray], 1u);
                            if (k < MFG_PASSES) pass->rec[ray][k] = rec;
                        }
                    }
                }
            }
            if (__ballot(hit)) {
                // lanes of one ray settle their nearest t by an LDS minimum
                // (t > 0: its bits order like the number), then the facet
                const unsigned long long tb = hit ? (unsigned long long)__double_as_longlong(t) : ~0ull;
                unsigned long long old = 0, cur = 0;
                if (hit) old = atomicMin(&W.t[ray], tb);
                wave_sync();
                if (hit) cur = W.t[ray];
                const bool best = hit && cur == tb;
                if (best && old > tb) W.facet[ray] = 0x7fffffff;   // first at this distance
                wave_sync();
                if (best) {
                    atomicMin(&W.facet[ray], f);
                    W.ra[ray].w = widen(t);
                }
            }
            wave_sync();
        }
    }
}

// Ray slot of this lane for walk().
__device__ __forceinline__ void walk_load(WaveLds& W, uint32_t lane, d3 p, d3 d, int32_t skip, double tmax) {
    const Ray32 r = make_ray32(p, d);
    W.ra[lane] = make_float4(r.ox, r.oy, r.oz, widen(tmax));
    W.rb[lane] = make_float4(r.ix, r.iy, r.iz, __int_as_float(skip));
    W.p01[lane] = make_double2(p.x, p.y);
    W.p2d0[lane] = make_double2(p.z, d.x);
    W.d12[lane] = make_double2(d.y, d.z);
    W.t[lane] = (unsigned long long)__double_as_longlong(tmax);
    W.facet[lane] = -1;
}

// (u,v) of a hit at distance t on a facet: the operations of leaf_test.
__device__ __forceinline__ void hit_uv(const DFacet* __restrict__ F, d3 P, d3 D, double t, double& u, double& v) {
    d3 X = mk(fma(t, D.x, P.x), fma(t, D.y, P.y), fma(t, D.z, P.z));
    d3 r = sub(X, ld3(F->O));
    u = fdot(r, ld3(F->U)) * F->invU2;
    v = fdot(r, ld3(F->V)) * F->invV2;
}

// A wall event's facet in registers (DHit without its rarely used words).
struct HitRegs {
    d3 N, nU, nV;
    double sticking, sqrt_temp;
    uint32_t flags;
    int32_t hot;
};
__device__ __forceinline__ HitRegs load_hit(const DHit* __restrict__ h) {
    const double2* q = reinterpret_cast<const double2*>(h);
    const double2 q0 = q[0], q1 = q[1], q2 = q[2], q3 = q[3], q4 = q[4];
    const uint4 q5 = reinterpret_cast<const uint4*>(h)[5];
    return {mk(q0.x, q0.y, q1.x), mk(q1.y, q2.x, q2.y), mk(q3.x, q3.y, q4.x), q4.y,
            __longlong_as_double((long long)(((unsigned long long)q5.y << 32) | q5.x)), q5.z, (int32_t)q5.w};
}

#define MFG_IN __device__ __forceinline__

// ------------------------------------------------------------------ tracer
// ONE: the launch has a single variant, whose constants come with the kernel
// arguments (scalar loads, no round trip on the event's path); otherwise
// every lane follows its own variant's record.
// Without a feature that reads them, a particle has no clock, path length,
// decay time, hit position or bounce count (CLOCKED false: they would be
// live across every walk), and its weight is 1 without low flux. With one
// line read per event and these constants at hand, the event of a lone
// particle took 10,000 instead of 21,000 cycles (most of it serial loads),
// that of a full wave on the beam pipe 54,000 instead of 86,000; beam-pipe
// launch 91.3 -> 72.5 ms, textured tube 18.2 -> 14.5 ms, low flux 165 -> 120.
template <uint32_t FEAT, bool ONE>
struct Tracer {
    static constexpr bool CLOCKED = (FEAT & FEAT_ALL & ~(uint32_t)FEAT_LOWFLUX) != 0;
    static constexpr bool WEIGHTED = (FEAT & FEAT_LOWFLUX) != 0;
    const TraceParams& P;
    WaveLds& W;                       // this wave's walk area
    PassLds* pass;                    // this wave's transparent passes
    int32_t* spill;                   // this lane's stack entries beyond the LDS part (second walk)
    // particle state (reference Particle.h:95-122)
    d3 pos, dir;
    double time, vel, ori, gen_time, dist, decay_t, scatter_path, hu, hv;
    int32_t structure, last_hit, tele_from;
    uint32_t nb_bounces, nb_events;
    Rng rng;
    const DVariant* var;
    // lane accumulators (flushed once per wave); unweighted particles need
    // neither weight sum, and without a clock every path ends on a facet, so
    // the two path sums are one
    uint32_t acc_hits, acc_des, acc_absorbed;
    double acc_hit_equiv, acc_abs_equiv, acc_dist_total, acc_dist_full;
    uint32_t acc_decay;
    uint32_t tr_n;
    uint32_t* adj_cnt;
    uint32_t seg_n;                   // adjoint: target scores since the last survived sticky collision
    int32_t* seg_t;
    double* seg_x;
    double* hot;                      // LDS counters of the hot facets' first P.hot_slots slots (8 words each)
    double* profs;                    // LDS slices of the profiles kept there
    const uint4* lnodes;              // LDS copy of the first P.lds_nodes BVH nodes
    const MaxwellLds* maxwell;        // LDS copy of the Maxwell CDF (P.maxwell_scale > 0)
    // pending slot-0 facet counter update of this lane (the event's other
    // slots are added at once)
    int32_t pend_f, pend_hot;
    uint32_t pend_hits;
    double pend_he, pend_abs, pend_s1v, pend_svo, pend_s1pv;

    MFG_IN Tracer(const TraceParams& p, WaveLds& w, PassLds* pl, int32_t* sp) : P(p), W(w), pass(pl), spill(sp) {
        acc_hits = acc_des = acc_absorbed = 0;
        acc_hit_equiv = acc_abs_equiv = acc_dist_total = acc_dist_full = 0.0;
        acc_decay = 0;
        tr_n = 0;
        adj_cnt = nullptr;
        seg_n = 0;
        seg_t = nullptr;
        seg_x = nullptr;
        var = ONE ? p.variants : nullptr;
        hot = profs = nullptr;
        lnodes = nullptr;
        maxwell = nullptr;
        ori = 1.0;
        time = gen_time = dist = hu = hv = 0.0;
        decay_t = scatter_path = 1e100;
        tele_from = -1;
        nb_bounces = nb_events = 0;
        clear_pending();
    }

    MFG_IN const DVariant& vc() const {
        if constexpr (ONE) return P.one;
        else return *var;
    }
    MFG_IN uint64_t pid() const { return ((uint64_t)rng.p1 << 32) | rng.p0; }
    MFG_IN double w() const {         // the particle's weight
        if constexpr (WEIGHTED) return ori;
        else return 1.0;
    }
    MFG_IN void add_hit() {
        ++acc_hits;
        if constexpr (WEIGHTED) acc_hit_equiv += ori;
    }

    MFG_IN int32_t local(int32_t f) const { return f - (int32_t)vc().facet_base; }

    MFG_IN void trace(int32_t f, int32_t kind) {
        if constexpr ((FEAT & FEAT_TRACE) != 0) {
            if (pid() < P.trace_n && tr_n < P.trace_k) {
                size_t at = (size_t)pid() * P.trace_k + tr_n;
                P.trace_facet[at] = f < 0 ? f : local(f);
                P.trace_kind[at] = kind;
                ++tr_n;
            }
        }
        (void)f; (void)kind;
    }
    MFG_IN int moment(double t) const {
        if constexpr ((FEAT & FEAT_MOMENTS) != 0) {
            uint32_t n = vc().n_moments;
            if (n == 0) return -1;
            const double* S = P.mom_start + vc().mom_base;
            uint32_t lo = 0, hi = n;  // first start >= t
            while (lo < hi) { uint32_t mid = (lo + hi) / 2; if (S[mid] < t) lo = mid + 1; else hi = mid; }
            uint32_t lb = lo;
            if (lb != 0) --lb;
            if (S[lb] <= t && t < P.mom_end[vc().mom_base + lb]) return (int)lb + 1;
        }
        (void)t;
        return -1;
    }
    MFG_IN double param_at(int32_t id, double t, double c) const {
        if constexpr ((FEAT & FEAT_TDPARAM) != 0) {
            if (id >= 0) {
                const DTable tb = P.params[vc().param_base + id];
                return interp_y(t, XYRef{P.tab_x + tb.off, P.tab_y + tb.off, tb.n}, tb.log_x, tb.log_y, false);
            }
        }
        (void)id; (void)t;
        return c;
    }
    MFG_IN double sticking(const HitRegs& H, int32_t f) const {
        if constexpr ((FEAT & FEAT_ADJOINT) != 0) {
            const int32_t g = P.hits[f].adj_group;
            if (g >= 0) return P.adj_sticking[g];
        }
        if constexpr ((FEAT & FEAT_TDPARAM) != 0) {
            if (H.flags & FF_TD_STICKING) return param_at(P.phys[f].sticking_param, time, H.sticking);
        }
        return H.sticking;
    }
    MFG_IN double temperature(const DPhys& ph) const { return param_at(ph.temperature_param, time, ph.temperature); }

    MFG_IN mfg_facet_counters* fc(int32_t f, int slot) const {
        return P.fc + vc().fc_base + (size_t)slot * vc().n_facets + (uint32_t)local(f);
    }

    // IncreaseFacetCounter (Particle.cpp:1193-1230). Slot 0 goes to the
    // lane's pending record (summed across the wave before the atomics);
    // moment slots and force terms go straight to memory.
    MFG_IN void counter(const HitRegs& H, int32_t f, int m, uint32_t hit, uint32_t des, uint32_t abs_, double s1v, double svo,
                            d3 imp, d3 imp2, d3 impm) {
        double he = (double)hit * w();
        double s1pv = (hit || des) ? (he + (double)des) / vel : 0.0;
        bool force = false;
        if constexpr ((FEAT & FEAT_FORCE) != 0) force = vc().enable_force != 0;
        if (!force && des == 0) {
            if constexpr (CLOCKED) { if (pend_f >= 0 && pend_f != f) flush_pending_direct(); }
            pend_f = f;
            pend_hot = H.hot;
            pend_hits += hit;
            pend_he += he;
            pend_abs += (double)abs_ * w();
            pend_s1v += w() * s1v;
            pend_svo += w() * svo;
            pend_s1pv += s1pv;
        }
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            int slot = k == 0 ? 0 : m;
            if (k == 1 && m <= 0) break;
            if (k == 0 && !force && des == 0) continue;
            if constexpr ((FEAT & FEAT_MOMENTS) != 0) {
                // a hot facet's moment slots, like its slot 0, in LDS
                if (k == 1 && !force && des == 0 && H.hot >= 0 && (uint32_t)m < P.hot_slots) {
                    add_hot(H.hot, m, hit, weighted() ? he : 0.0, (double)abs_ * w(), w() * s1v, w() * svo, s1pv);
                    continue;
                }
            }
            mfg_facet_counters* c = fc(f, slot);
            if (hit) { atomic_addu(&c->nb_mc_hit, hit); if (weighted()) atomic_addd(&c->nb_hit_equiv, he); }
            if (des) atomic_addu(&c->nb_desorbed, des);
            if (abs_) atomic_addd(&c->nb_abs_equiv, (double)abs_ * w());
            if (s1v != 0.0) atomic_addd(&c->sum_1_per_ort_velocity, w() * s1v);
            if (svo != 0.0) atomic_addd(&c->sum_v_ort, w() * svo);
            if (hit || des) atomic_addd(&c->sum_1_per_velocity, s1pv);
            if constexpr ((FEAT & FEAT_FORCE) != 0) {
                if (force) {
                    double* fo = P.force + vc().force_base + ((size_t)slot * vc().n_facets + (uint32_t)local(f)) * 9;
                    atomic_addd(fo + 0, ori * imp.x); atomic_addd(fo + 1, ori * imp.y); atomic_addd(fo + 2, ori * imp.z);
                    atomic_addd(fo + 3, ori * imp2.x); atomic_addd(fo + 4, ori * imp2.y); atomic_addd(fo + 5, ori * imp2.z);
                    atomic_addd(fo + 6, ori * impm.x); atomic_addd(fo + 7, ori * impm.y); atomic_addd(fo + 8, ori * impm.z);
                }
            }
        }
        if constexpr ((FEAT & FEAT_ADJOINT) != 0) {
            const int32_t at = P.hits[f].adj_target;
            if (hit && at >= 0) adjoint_score(at, P.hits[f].adj_group, he, false);
        }
        (void)imp; (void)imp2; (void)impm;
    }
    // Counter record of a hot facet in LDS (field order of mfg_facet_counters).
    MFG_IN void add_hot(int32_t idx, int slot, uint32_t hits, double he, double ab, double s1v, double svo, double s1pv) {
        double* h = hot + 8 * ((uint32_t)idx * P.hot_slots + (uint32_t)slot);
        if (hits) atomicAdd(reinterpret_cast<unsigned long long*>(h), (unsigned long long)hits);
        if (he != 0.0) atomic_addd(h + 1, he);
        if (ab != 0.0) atomic_addd(h + 3, ab);
        if (s1v != 0.0) atomic_addd(h + 4, s1v);
        if (svo != 0.0) atomic_addd(h + 5, svo);
        if (s1pv != 0.0) atomic_addd(h + 6, s1pv);
    }
    // Without low-flux weighting every particle weighs 1, so nb_hit_equiv
    // equals nb_mc_hit: it is not added here (one atomic less per hit) and
    // the host fills it in when it reads the counters.
    MFG_IN bool weighted() const {
        if constexpr (WEIGHTED) return vc().low_flux != 0;
        return false;
    }
    // Atomics of this lane's pending slot-0 record, then clear it.
    MFG_IN void flush_pending_direct() {
        if (pend_f < 0) return;
        const bool w = weighted();
        if (pend_hot >= 0) {
            add_hot(pend_hot, 0, pend_hits, w ? pend_he : 0.0, pend_abs, pend_s1v, pend_svo, pend_s1pv);
            clear_pending();
            return;
        }
        mfg_facet_counters* cc = P.fc + vc().fc_base + (uint32_t)local(pend_f);
        if (pend_hits) {
            atomic_addu(&cc->nb_mc_hit, pend_hits);
            if (w) atomic_addd(&cc->nb_hit_equiv, pend_he);
        }
        if (pend_abs != 0.0) atomic_addd(&cc->nb_abs_equiv, pend_abs);
        if (pend_s1v != 0.0) atomic_addd(&cc->sum_1_per_ort_velocity, pend_s1v);
        if (pend_svo != 0.0) atomic_addd(&cc->sum_v_ort, pend_svo);
        if (pend_s1pv != 0.0) atomic_addd(&cc->sum_1_per_velocity, pend_s1pv);
        clear_pending();
    }
    MFG_IN void clear_pending() {
        pend_f = pend_hot = -1; pend_hits = 0;
        pend_he = pend_abs = pend_s1v = pend_svo = pend_s1pv = 0.0;
    }
    // Path score of a hit-equivalent x on a target:
    // d x / d s_g = x * (-n_g / (1 - s_g)) (+ x / s_t for the absorbed part).
    MFG_IN void adjoint_score(int t, int group, double x, bool absorbed_part) {
        if constexpr ((FEAT & FEAT_ADJOINT) != 0) {
            atomic_addd(P.adj_j0 + t, x);
            uint32_t G = P.adj_groups;
            for (uint32_t g = 0; g < G; ++g) {
                double s = P.adj_sticking[g];
                double d = -x * (double)adj_cnt[g] / (1.0 - s);
                if (absorbed_part && group == (int)g) d += x / s;
                if (d != 0.0) atomic_addd(P.adj_jac + (size_t)t * G + g, d);
            }
            // kept for the cutoff term until the particle survives a sticky collision
            if (seg_n < MFG_ADJ_SEG) { seg_t[seg_n] = t; seg_x[seg_n] = x; }
            ++seg_n;
        }
        (void)t; (void)group; (void)x; (void)absorbed_part;
    }
    // The low-flux cutoff's term of dE[J]/ds_g (not a derivative of any
    // single path): the particle ends at collision K, W_{K-1} (1 - s_K) <=
    // c < W_{K-1}; a rise ds of s_g ends it at K-1 instead with probability
    // f(0) n_g ds / (1 - s_g) (n_g: its collisions with group g up to K-1,
    // f(0): density of ln(W_{K-1}/c) at 0), losing the scores recorded since
    // it survived K-1. In the renewal limit ln(W_{K-1}/c) is uniform on
    // (0, -ln(1 - s_K)] given K, so the term is
    //   dJ_t/ds_g += -sum x_t n_g / ((1 - s_g)(-ln(1 - s_K))).
    MFG_IN void cutoff_boundary(int group, double sK) {
        if constexpr ((FEAT & FEAT_ADJOINT) != 0) {
            if (seg_n > MFG_ADJ_SEG) atomicOr(P.adj_seg_overflow, 1ull);
            const double dK = -log1p(-sK);
            const uint32_t n_seg = seg_n < MFG_ADJ_SEG ? seg_n : MFG_ADJ_SEG;
            if (!(dK > 0.0) || n_seg == 0) return;
            const uint32_t G = P.adj_groups;
            for (uint32_t i = 0; i < n_seg; ++i) {
                const int t = seg_t[i];
                const double x = seg_x[i];
                for (uint32_t g = 0; g < G; ++g) {
                    const double n = (double)adj_cnt[g] - (group == (int)g ? 1.0 : 0.0);
                    if (n > 0.0) atomic_addd(P.adj_jac + (size_t)t * G + g, -x * n / ((1.0 - P.adj_sticking[g]) * dK));
                }
            }
        }
        (void)group; (void)sK;
    }
    MFG_IN void counter_force(const HitRegs& H, int32_t f, int m, uint32_t hit, uint32_t des, uint32_t abs_, double s1v,
                                  double svo, double sign) {
        d3 z = mk(0, 0, 0), v2 = z, mom = z, vv = z;
        if constexpr ((FEAT & FEAT_FORCE) != 0) {
            if (vc().enable_force) {
                vv = scl(sign * vel, dir);
                v2 = mk(vv.x * vv.x, vv.y * vv.y, vv.z * vv.z);
                mom = cross(sub(pos, ld3(vc().torque)), vv);
            }
        }
        (void)sign;
        counter(H, f, m, hit, des, abs_, s1v, svo, vv, v2, mom);
    }
    MFG_IN bool cell(const DPhys& ph, uint32_t& add) const {
        int tu = (int)(hu * ph.tex_wp), tv = (int)(hv * ph.tex_hp);
        tu = tu > ph.tex_w - 1 ? ph.tex_w - 1 : tu;
        tv = tv > ph.tex_h - 1 ? ph.tex_h - 1 : tv;
        if (tu < 0 || tv < 0) return false;
        add = (uint32_t)tu + (uint32_t)tv * (uint32_t)ph.tex_w;
        return true;
    }
    MFG_IN double ort(const HitRegs& H) const { return fabs(dot(dir, H.N)); }
    // RecordHitOnTexture (Particle.cpp:977-1004)
    // The steady-state cell of an event's records is added to in this lane's
    // slot of W (staged: W.t names the cell, ~0 none yet) and goes to memory
    // with the wave's others after the event.
    MFG_IN void texture(const HitRegs& H, int32_t f, int m, bool count, double vf, double of, bool staged = true) {
        const DPhys& ph = P.phys[f];
        uint32_t add;
        if (!cell(ph, add)) return;
        double ov = vc().c_factor * vel * ort(H);
        const uint64_t at = vc().tex_base + (uint64_t)ph.tex_off + add;
        const double n = count ? w() : 0.0, sv = w() * of * ov * P.tex_inc[at], s1 = w() * vf / ov;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            int slot = k == 0 ? 0 : m;
            if (k == 1 && m <= 0) break;
            if (k == 0 && staged) {
                const uint32_t lane = here(__lane_id());
                double* S = W.cell + 3u * lane;
                if (W.t[lane] == ~0ull) {
                    W.t[lane] = at;
                    S[0] = n; S[1] = sv; S[2] = s1;
                    continue;
                }
                if (W.t[lane] == at) {
                    S[0] += n; S[1] += sv; S[2] += s1;
                    continue;
                }
            }
            mfg_texture_cell* c = P.tex + at + (size_t)slot * vc().n_tex;
            if (count) atomic_addd(&c->count_equiv, n);
            atomic_addd(&c->sum_1_per_ort_velocity, s1);
            atomic_addd(&c->sum_v_ort_per_area, sv);
        }
    }
    // RecordDirectionVector (Particle.cpp:1006-1023)
    MFG_IN void direction(int32_t f, int m) {
        const DPhys& ph = P.phys[f];
        if (ph.dir_off < 0) return;
        uint32_t add;
        if (!cell(ph, add)) return;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            int slot = k == 0 ? 0 : m;
            if (k == 1 && m <= 0) break;
            mfg_direction_cell* c = P.dir + vc().dir_base + (size_t)slot * vc().n_dir + (size_t)ph.dir_off + add;
            atomic_addd(&c->dir[0], ori * dir.x * vel);
            atomic_addd(&c->dir[1], ori * dir.y * vel);
            atomic_addd(&c->dir[2], ori * dir.z * vel);
            atomic_addu(&c->count, 1ull);
        }
    }
    // Adds to slice p of a facet's profile: in LDS for the profiles and slots
    // kept there (TraceParams::prof_slots), else in memory.
    MFG_IN void slice(const DPhys& ph, int slot, size_t p, bool count, double s1, double sv, bool sums) {
        if (ph.prof_hot >= 0 && (uint32_t)slot < P.prof_slots) {
            double* s = profs + 3u * (((uint32_t)ph.prof_hot * P.prof_slots + (uint32_t)slot) * MFG_PROFILE_SIZE + (uint32_t)p);
            if (count) atomic_addd(s, w());
            if (sums) { atomic_addd(s + 1, sv); atomic_addd(s + 2, s1); }
            return;
        }
        mfg_profile_slice* s = P.prof + vc().prof_base + (size_t)slot * vc().n_prof + (size_t)ph.prof_off + p;
        if (count) atomic_addd(&s->count_equiv, w());
        if (sums) { atomic_addd(&s->sum_v_ort, sv); atomic_addd(&s->sum_1_per_ort_velocity, s1); }
    }
    // ProfileFacet (Particle.cpp:1025-1085)
    MFG_IN void profile(const HitRegs& H, int32_t f, int m, bool count, double vf, double of) {
        if (!(H.flags & FF_PROFILE)) return;
        const DPhys& ph = P.phys[f];
        int pt = ph.profile_type;
        double a = ort(H);
        if (count && pt == MFG_PROFILE_ANGULAR) {
            double th = acos(fmin(1.0, a));
            long p = (long)(th / (kPi / 2) * (double)MFG_PROFILE_SIZE);
            p = p < 0 ? 0 : (p > MFG_PROFILE_SIZE - 1 ? MFG_PROFILE_SIZE - 1 : p);
            for (int k = 0; k < 2; ++k) {
                int slot = k == 0 ? 0 : m;
                if (k == 1 && m <= 0) break;
                slice(ph, slot, (size_t)p, true, 0.0, 0.0, false);
            }
        } else if (pt == MFG_PROFILE_U || pt == MFG_PROFILE_V) {
            double c = pt == MFG_PROFILE_U ? hu : hv;
            if (!(c >= 0.0)) return;
            double x = c * (double)MFG_PROFILE_SIZE;
            if (!(x < (double)MFG_PROFILE_SIZE)) return;
            size_t p = (size_t)x;
            double ov = vel * a;
            for (int k = 0; k < 2; ++k) {
                int slot = k == 0 ? 0 : m;
                if (k == 1 && m <= 0) break;
                slice(ph, slot, p, count, w() * vf / ov, w() * of * vc().c_factor * ov, true);
            }
        } else if (count && (pt == MFG_PROFILE_VELOCITY || pt == MFG_PROFILE_ORT_VELOCITY || pt == MFG_PROFILE_TAN_VELOCITY)) {
            double d = pt == MFG_PROFILE_VELOCITY ? 1.0 : (pt == MFG_PROFILE_ORT_VELOCITY ? a : sqrt(fmax(0.0, 1 - a * a)));
            double x = d * vel / ph.max_speed * (double)MFG_PROFILE_SIZE;
            if (!(x >= 0.0) || !(x < (double)MFG_PROFILE_SIZE)) return;
            size_t p = (size_t)x;
            for (int k = 0; k < 2; ++k) {
                int slot = k == 0 ? 0 : m;
                if (k == 1 && m <= 0) break;
                slice(ph, slot, (size_t)p, true, 0.0, 0.0, false);
            }
        }
    }
    MFG_IN void polar(const HitRegs& H, double& th, double& phv) const {
        double lu = dot(dir, H.nU), lv = dot(dir, H.nV), ln = dot(dir, H.N);
        th = acos(fmax(-1.0, fmin(1.0, ln)));
        phv = atan2(lv, lu);
    }
    // RecordAngleMap (Particle.cpp:1104-1136). The angles only select a bin,
    // so they are evaluated in FP32.
    MFG_IN void angle_map(const HitRegs& H, int32_t f) {
        if (!(H.flags & FF_ANGLEMAP)) return;
        const DPhys& ph = P.phys[f];
        if (ph.am_off < 0) return;
        double lu = dot(dir, H.nU), lv = dot(dir, H.nV), ln = dot(dir, H.N);
        double th = (double)acosf((float)fmax(-1.0, fmin(1.0, ln)));
        double phv = (double)atan2f((float)lv, (float)lu);
        if (th > kPi / 2.0) th = fabs(kPi - th);
        long ti;
        if (th < ph.am_theta_limit) {
            if (ph.am_lo == 0) return;
            ti = (long)(th / ph.am_theta_limit * (double)ph.am_lo);
        } else {
            if (ph.am_hi == 0) return;
            ti = (long)ph.am_lo + (long)((th - ph.am_theta_limit) / (kPi / 2.0 - ph.am_theta_limit) * (double)ph.am_hi);
        }
        long nt = (long)(ph.am_lo + ph.am_hi);
        ti = ti < 0 ? 0 : (ti > nt - 1 ? nt - 1 : ti);
        long pi_ = (long)((phv + 3.1415926) / (2.0 * kPi) * (double)ph.am_phi);
        pi_ = pi_ < 0 ? 0 : (pi_ > (long)ph.am_phi - 1 ? (long)ph.am_phi - 1 : pi_);
        atomic_addu(P.am + vc().am_base + (size_t)ph.am_off + (size_t)ti * ph.am_phi + pi_, 1ull);
    }
    // LogHit (Particle.cpp:1087-1102)
    MFG_IN void log_hit(const HitRegs& H, int32_t f) {
        if constexpr ((FEAT & FEAT_LOG) != 0) {
            if (vc().log_facet == f) {
                unsigned long long at = atomicAdd(P.log_count, 1ull);
                if (at < vc().log_limit) {
                    mfg_log_entry e;
                    e.u = hu; e.v = hv;
                    polar(H, e.hit_theta, e.hit_phi);
                    e.ori_ratio = ori; e.particle_decay_moment = decay_t; e.time = time; e.velocity = vel;
                    P.log[at] = e;
                }
            }
        }
        (void)H; (void)f;
    }
    MFG_IN void hist_add(double* g, uint32_t nb, uint32_t nd, uint32_t nt, uint32_t bbin, double dbin, double tbin) {
        uint32_t off = 0;
        if (nb) { uint32_t b = nb_bounces / bbin; atomic_addd(g + off + (b < nb - 1 ? b : nb - 1), ori); off += nb; }
        if (nd) {
            double x = dist / dbin;
            uint32_t b = x < (double)(nd - 1) ? (uint32_t)x : nd - 1;
            atomic_addd(g + off + b, ori); off += nd;
        }
        if (nt) {
            double x = (time - gen_time) / tbin;
            uint32_t b = x < (double)(nt - 1) ? (uint32_t)x : nt - 1;
            atomic_addd(g + off + b, ori);
        }
    }
    // RecordHistograms (Particle.cpp:926-975), called on absorption
    MFG_IN void histograms(int32_t f, int m) {
        if constexpr ((FEAT & FEAT_HIST) != 0) {
            const DPhys& ph = P.phys[f];
            for (int k = 0; k < 2; ++k) {
                int slot = k == 0 ? 0 : m;
                if (k == 1 && m <= 0) break;
                if (vc().n_gh)
                    hist_add(P.gh + vc().gh_base + (size_t)slot * vc().n_gh, vc().gh_nb_bounce, vc().gh_nb_dist,
                             vc().gh_nb_time, vc().gh_bounce_bin, vc().gh_dist_bin, vc().gh_time_bin);
                if (ph.fh_off >= 0)
                    hist_add(P.fh + vc().fh_base + (size_t)slot * vc().n_fh + ph.fh_off, ph.fh_nb_bounce, ph.fh_nb_dist,
                             ph.fh_nb_time, ph.fh_bounce_bin, ph.fh_dist_bin, ph.fh_time_bin);
            }
        }
        (void)f; (void)m;
    }
    MFG_IN d3 polar_to_cart(const HitRegs& H, double cos_t, double sin_t, double phv, bool reverse) const {
        double s, c;
        sincos(phv, &s, &c);
        double n = reverse ? -cos_t : cos_t;
        return add(add(scl(sin_t * c, H.nU), scl(sin_t * s, H.nV)), scl(n, H.N));
    }
    // TreatMovingFacet (Physics.cpp:22-39)
    MFG_IN void moving(d3& d, double& v) const {
        if constexpr ((FEAT & FEAT_MOVING) != 0) {
            d3 a = mk(0, 0, 0);
            if (vc().motion_type == 1) a = ld3(vc().motion2);
            else if (vc().motion_type == 2) a = cross(ld3(vc().motion2), scl(0.01, sub(pos, ld3(vc().motion1))));
            d3 nv = add(scl(v, d), a);
            v = nrm(nv);
            d = unitv(nv);
        }
        (void)d; (void)v;
    }
    template <typename G>
    MFG_IN double maxwell_speed(G& g, double sq) {
        const double r = g.rnd();
        if (P.maxwell_scale > 0.0) return maxwell_lds(maxwell, r, P.maxwell_scale) * sq;
        XYRef t{P.tab_x + vc().maxwell_base, P.tab_y + vc().maxwell_base, MFG_MAXWELL_POINTS};
        return interp_x_guided(r, t, P.guides + vc().maxwell_guide, MFG_MAXWELL_GUIDE) * sq;
    }
    MFG_IN d3 emit(const HitRegs& H, const DPhys& ph, int type, double n_exp, bool reverse) {
        if (type == MFG_DES_UNIFORM) {
            double c = rng.rnd(); double phv = rng.rnd() * 2.0 * kPi;
            return polar_to_cart(H, c, sqrt(1 - c * c), phv, reverse);
        }
        if (type == MFG_DES_COSINE_N) {
            double c = pow(rng.rnd(), 1.0 / (n_exp + 1.0)); double phv = rng.rnd() * 2.0 * kPi;
            return polar_to_cart(H, c, sqrt(1 - c * c), phv, reverse);
        }
        if constexpr ((FEAT & FEAT_AMSRC) != 0) {
            if (type == MFG_DES_ANGLEMAP) {   // Particle.cpp:599-621: the map holds incident angles
                const AmSrc A = am_view(P.am_src + ph.am_src_off);
                double th, ov;
                int tlo;
                am_generate_theta(A, rng.rnd(), th, tlo, ov);
                double phv = am_generate_phi(A, tlo, ov, rng.rnd());
                double t2 = kPi - th;
                return polar_to_cart(H, cos(t2), sin(t2), phv, false);
            }
        }
        double a = rng.rnd(); double phv = rng.rnd() * 2.0 * kPi;
        return polar_to_cart(H, sqrt(a), sqrt(1 - a), phv, reverse);
    }

    // StartFromSource (Particle.cpp:407-685) without the source-facet
    // counter, which the caller adds (summed across the wave).
    MFG_IN int32_t start(uint64_t local_pid) {
        rng.init(var->seed, local_pid);
        nb_events = 0;
        tr_n = 0;
        if constexpr ((FEAT & FEAT_ADJOINT) != 0) {
            for (uint32_t g = 0; g < P.adj_groups; ++g) adj_cnt[g] = 0;
            seg_n = 0;
        }
        double r = rng.rnd() * vc().total_des;
        const double* cum = P.src_cum + vc().src_base;
        uint32_t n = vc().src_n;
        uint32_t lo = 0, hi = n;  // first cum > r
        while (lo < hi) { uint32_t mid = (lo + hi) / 2; if (cum[mid] <= r) lo = mid + 1; else hi = mid; }
        uint32_t k = lo < n ? lo : n - 1;
        int32_t src = P.src_facet[vc().src_base + k];
        const DFacet* F = P.facets + src;
        const DPhys& ph = P.phys[src];
        const HitRegs H = load_hit(P.hits + src);
        bool reverse = false;
        if (H.flags & FF_2SIDED) reverse = rng.rnd() > 0.5;
        long map_w = -1, map_h = -1;
        if constexpr ((FEAT & FEAT_OGMAP) != 0) {
            if (ph.flags & FF_OGMAP) {
                double base = k ? cum[k - 1] : 0.0;
                double rem = (r - base) / vc().latest * (1.38E-23 * ph.temperature);
                const double* oc = P.og_cdf + ph.og_off;
                uint32_t nc = ph.og_w * ph.og_h, a = 0, b = nc;
                while (a < b) { uint32_t mid = (a + b) / 2; if (oc[mid] <= rem) a = mid + 1; else b = mid; }
                uint32_t cellv = a < nc ? a : nc - 1;
                map_h = (long)(cellv / ph.og_w);
                map_w = (long)cellv - map_h * (long)ph.og_w;
            }
        }
        last_hit = src;
        double rt = rng.rnd();
        if constexpr (CLOCKED) time = rt * vc().latest;
        if constexpr ((FEAT & FEAT_TDPARAM) != 0) {
            if (ph.id_index >= 0) {
                const DTable tb = P.ids[vc().id_base + ph.id_index];
                XYRef t{P.tab_x + tb.off, P.tab_y + tb.off, tb.n};
                time = interp_x(rt * t.y[t.n - 1], t);
            }
        }
        gen_time = time;
        if (vc().use_maxwell) vel = maxwell_speed(rng, H.sqrt_temp);
        else vel = 145.469 * sqrt(ph.temperature / vc().gas_mass);
        ori = 1.0;
        decay_t = 1e100;
        scatter_path = 1e100;
        if constexpr ((FEAT & FEAT_VOLUME) != 0) {
            if (vc().enable_decay) decay_t = time + (1.44269 * vc().half_life) * -log(rng.rnd());
            if (vc().scatter_enabled) scatter_path = vc().scatter_mfp * -log(rng.rnd());
        }
        nb_bounces = 0;
        dist = 0.0;
        bool found = false;
        const double* poly = P.poly + 2 * (size_t)F->poly_off;
        uint32_t pn = F->poly_n;
        d3 O = ld3(F->O), U = ld3(F->U), V = ld3(F->V);
        for (int tr = 0; tr < 1000 && !found; ++tr) {
            double u, v;
            if ((FEAT & FEAT_OGMAP) != 0 && map_w >= 0) {
                double a = rng.rnd(), b = rng.rnd();
                double wp = ph.og_wp, hp = ph.og_hp;
                u = (map_w < (long)ph.og_w - 1) ? ((double)map_w + a) / wp : ((double)map_w + a * (wp - ((double)ph.og_w - 1.0))) / wp;
                v = (map_h < (long)ph.og_h - 1) ? ((double)map_h + b) / hp : ((double)map_h + b * (hp - ((double)ph.og_h - 1.0))) / hp;
            } else {
                u = rng.rnd();
                v = rng.rnd();
            }
            if (in_polygon(poly, pn, u, v)) {
                pos = add(add(O, scl(u, U)), scl(v, V));
                hu = u; hv = v;
                found = true;
            }
        }
        if (!found) {
            if ((FEAT & FEAT_OGMAP) != 0 && map_w >= 0) {
                hu = ((double)map_w + 0.5) / ph.og_wp;
                hv = ((double)map_h + 0.5) / ph.og_hp;
                pos = add(add(O, scl(hu, U)), scl(hv, V));
            } else {
                hu = 0.5; hv = 0.5;
                pos = ld3(ph.centre);
            }
        }
        dir = emit(H, ph, ph.desorb_type, ph.des_exp, reverse);
        structure = ph.super_idx;
        tele_from = -1;
        if constexpr ((FEAT & FEAT_MOVING) != 0) {
            if ((ph.flags & FF_MOVING) && vc().motion_type) moving(dir, vel);
        }
        return src;
    }

    // Records of a desorption other than the facet counter of slot 0.
    MFG_IN void desorption_records(int32_t src, int m, double ov) {
        const HitRegs H = load_hit(P.hits + src);
        if (m > 0 || ((FEAT & FEAT_FORCE) != 0 && vc().enable_force)) {
            // moment slot (and force terms) per lane
            d3 z = mk(0, 0, 0), v2 = z, mom = z, vv = z;
            if constexpr ((FEAT & FEAT_FORCE) != 0) {
                if (vc().enable_force) {
                    vv = scl(vel, dir);
                    v2 = mk(vv.x * vv.x, vv.y * vv.y, vv.z * vv.z);
                    mom = cross(sub(pos, ld3(vc().torque)), vv);
                    double* fo = P.force + vc().force_base + (size_t)(uint32_t)local(src) * 9;
                    atomic_addd(fo + 0, vv.x); atomic_addd(fo + 1, vv.y); atomic_addd(fo + 2, vv.z);
                    atomic_addd(fo + 3, v2.x); atomic_addd(fo + 4, v2.y); atomic_addd(fo + 5, v2.z);
                    atomic_addd(fo + 6, mom.x); atomic_addd(fo + 7, mom.y); atomic_addd(fo + 8, mom.z);
                }
            }
            if (m > 0 && H.hot >= 0 && (uint32_t)m < P.hot_slots) {
                double* h = hot + 8 * ((uint32_t)H.hot * P.hot_slots + (uint32_t)m);
                atomicAdd(reinterpret_cast<unsigned long long*>(h + 2), 1ull);
                atomic_addd(h + 4, 2.0 / ov);
                atomic_addd(h + 5, vc().c_factor * ov);
                atomic_addd(h + 6, 1.0 / vel);
            } else if (m > 0) {
                mfg_facet_counters* c = fc(src, m);
                atomic_addu(&c->nb_desorbed, 1ull);
                atomic_addd(&c->sum_1_per_ort_velocity, 2.0 / ov);
                atomic_addd(&c->sum_v_ort, vc().c_factor * ov);
                atomic_addd(&c->sum_1_per_velocity, 1.0 / vel);
            }
            if (m > 0) {
                if constexpr ((FEAT & FEAT_FORCE) != 0) {
                    if (vc().enable_force) {
                        double* fo = P.force + vc().force_base + ((size_t)m * vc().n_facets + (uint32_t)local(src)) * 9;
                        atomic_addd(fo + 0, vv.x); atomic_addd(fo + 1, vv.y); atomic_addd(fo + 2, vv.z);
                        atomic_addd(fo + 3, v2.x); atomic_addd(fo + 4, v2.y); atomic_addd(fo + 5, v2.z);
                        atomic_addd(fo + 6, mom.x); atomic_addd(fo + 7, mom.y); atomic_addd(fo + 8, mom.z);
                    }
                }
            }
        }
        profile(H, src, m, false, 2.0, 1.0);
        log_hit(H, src);
        if ((H.flags & FF_COUNT_DES) && (H.flags & FF_TEXTURE)) texture(H, src, m, true, 2.0, 1.0, false);
        trace(src, 0);
    }

    // RegisterTransparentPass (Particle.cpp:1232-1257)
    MFG_IN void transparent_pass(int32_t f, double tp) {
        const HitRegs H = load_hit(P.hits + f);
        double df = ort(H);
        int m = moment(time + tp / 100.0 / vel);
        d3 z = mk(0, 0, 0);
        counter(H, f, m, 1, 0, 0, 2.0 / (vel * df), 2.0 * vc().c_factor * vel * df, z, z, z);
        if ((H.flags & FF_COUNT_TRANS) && (H.flags & FF_TEXTURE)) texture(H, f, m, true, 2.0, 2.0);
        if (H.flags & FF_COUNT_DIR) direction(f, m);
        log_hit(H, f);
        profile(H, f, m, true, 2.0, 2.0);
        angle_map(H, f);
        trace(f, 3);
    }
    // RecordAbsorb (Particle.cpp:888-924)
    MFG_IN void record_absorb(const HitRegs& H, int32_t f) {
        add_hit();
        if constexpr (WEIGHTED) acc_abs_equiv += ori;
        else ++acc_absorbed;
        int m = moment(time);
        histograms(f, m);
        double ov = vel * ort(H);
        bool scored = false;
        if constexpr ((FEAT & FEAT_ADJOINT) != 0) {
            const int32_t at = P.hits[f].adj_target;
            if (at >= 0) {
                // the absorbed part carries its own d/ds_t term
                for (int k = 0; k < 2; ++k) {
                    int slot = k == 0 ? 0 : m;
                    if (k == 1 && m <= 0) break;
                    mfg_facet_counters* c = fc(f, slot);
                    atomic_addu(&c->nb_mc_hit, 1ull);
                    atomic_addd(&c->nb_hit_equiv, ori);
                    atomic_addd(&c->nb_abs_equiv, ori);
                    atomic_addd(&c->sum_1_per_ort_velocity, ori * 2.0 / ov);
                    atomic_addd(&c->sum_v_ort, ori * vc().c_factor * ov);
                    atomic_addd(&c->sum_1_per_velocity, ori / vel);
                }
                adjoint_score(at, P.hits[f].adj_group, ori, true);
                scored = true;
            }
        }
        if (!scored) counter_force(H, f, m, 1, 0, 1, 2.0 / ov, vc().c_factor * ov, 1.0);
        log_hit(H, f);
        profile(H, f, m, true, 2.0, 1.0);
        angle_map(H, f);
        if ((H.flags & FF_COUNT_ABS) && (H.flags & FF_TEXTURE)) texture(H, f, m, true, 2.0, 1.0);
        if (H.flags & FF_COUNT_DIR) direction(f, m);
    }
    // UpdateVelocity (Particle.cpp:1138-1163)
    MFG_IN void update_velocity(EventDraws& g, const HitRegs& H, int32_t f) {
        double sq = H.sqrt_temp;
        if constexpr ((FEAT & FEAT_TDPARAM) != 0) { if (H.flags & FF_TD_TEMP) sq = sqrt(temperature(P.phys[f])); }
        if (H.flags & FF_FULL_ACC) {
            vel = vc().use_maxwell ? maxwell_speed(g, sq) : 145.469 * sq / vc().gas_mass;
        } else {
            double o2 = vel * vel, n2;
            if (vc().use_maxwell) { double vv = maxwell_speed(g, sq); n2 = vv * vv; }
            else n2 = 29369.939 * (temperature(P.phys[f]) / vc().gas_mass);
            vel = sqrt(o2 + (n2 - o2) * P.hits[f].accomodation);
        }
    }
    // PerformBounce (Particle.cpp:691-838)
    MFG_IN void bounce(EventDraws& g, const HitRegs& H, int32_t f) {
        add_hit();
        if constexpr ((FEAT & FEAT_TELEPORT) != 0) {
            if (H.flags & FF_LINK) {
                int m = moment(time);
                d3 z = mk(0, 0, 0);
                counter(H, f, m, 1, 0, 0, 0.0, 0.0, z, z, z);
                structure = P.phys[f].super_dest - 1;
                if constexpr ((FEAT & FEAT_MOVING) != 0) { if (H.flags & FF_MOVING) moving(dir, vel); }
                log_hit(H, f);
                profile(H, f, m, true, 2.0, 2.0);
                angle_map(H, f);
                if ((H.flags & FF_COUNT_TRANS) && (H.flags & FF_TEXTURE)) texture(H, f, m, true, 2.0, 2.0);
                if (H.flags & FF_COUNT_DIR) direction(f, m);
                trace(f, 5);
                return;
            }
        }
        double dn = dot(dir, H.N);
        bool revert = (H.flags & FF_2SIDED) && dn > 0.0;
        double ov_in = vel * fabs(dn);
        int m = moment(time);
        counter_force(H, f, m, 1, 0, 0, 1.0 / ov_in, vc().c_factor * ov_in, 1.0);
        if constexpr (CLOCKED) ++nb_bounces;
        if ((H.flags & FF_COUNT_REFL) && (H.flags & FF_TEXTURE)) texture(H, f, m, true, 1.0, 1.0);
        if (H.flags & FF_COUNT_DIR) direction(f, m);
        log_hit(H, f);
        profile(H, f, m, true, 1.0, 1.0);
        angle_map(H, f);
        update_velocity(g, H, f);
        int m_out = m;
        if constexpr ((FEAT & FEAT_SOJOURN) != 0) {
            if (H.flags & FF_SOJOURN) {
                const DPhys& ph = P.phys[f];
                double A = exp(-ph.sojourn_e / (8.31 * temperature(ph)));
                time += -log(g.rnd()) / (A * ph.sojourn_freq);
                m_out = moment(time);
            }
        }
        if (H.flags & FF_DIFFUSE) {
            double a = g.rnd(); double phv = g.rnd() * 2.0 * kPi;
            dir = polar_to_cart(H, sqrt(a), sqrt(1 - a), phv, revert);
        } else {
            const DHit& C = P.hits[f];
            double rt = g.rnd();
            if (rt < C.diffuse) {
                double a = g.rnd(); double phv = g.rnd() * 2.0 * kPi;
                dir = polar_to_cart(H, sqrt(a), sqrt(1 - a), phv, revert);
            } else if (rt < C.diffuse + C.specular) {
                dir = sub(dir, scl(2.0 * dot(dir, H.N), H.N));
            } else {
                double c = pow(g.rnd(), 1.0 / (P.phys[f].cos_exp + 1.0)); double phv = g.rnd() * 2.0 * kPi;
                dir = polar_to_cart(H, c, sqrt(1 - c * c), phv, revert);
            }
        }
        if constexpr ((FEAT & FEAT_MOVING) != 0) {
            if ((H.flags & FF_MOVING) && vc().motion_type) moving(dir, vel);
        }
        double ov_out = vel * ort(H);
        counter_force(H, f, m_out, 0, 0, 0, 1.0 / ov_out, vc().c_factor * ov_out, -1.0);
        if ((H.flags & FF_COUNT_REFL) && (H.flags & FF_TEXTURE)) texture(H, f, m_out, false, 1.0, 1.0);
        profile(H, f, m_out, false, 1.0, 1.0);
        last_hit = f;
        trace(f, 1);
    }
    // PerformTeleport (Particle.cpp:76-183). "Back to origin" (teleport_dest
    // = -1) goes to the destination of the particle's previous teleport:
    // the reference records teleportedFrom = destIndex (:122). A destination
    // in every structure (super_idx -1) keeps the particle's structure; the
    // reference would index its structure list with -1 there (:121, :245).
    MFG_IN void teleport(const HitRegs& H, int32_t f) {
        const DPhys& ph = P.phys[f];
        trace(f, 4);
        int32_t dest = ph.teleport_dest == -1 ? tele_from : ph.teleport_dest - 1;
        if (dest < 0 || dest >= (int32_t)vc().n_facets) { last_hit = f; return; }
        int32_t dg = dest + (int32_t)vc().facet_base;
        const DFacet* D = P.facets + dg;
        const DPhys& dph = P.phys[dg];
        if (dph.super_idx >= 0) structure = dph.super_idx;
        tele_from = dest;
        int m = moment(time);
        if ((H.flags & FF_COUNT_TRANS) && (H.flags & FF_TEXTURE)) texture(H, f, m, true, 2.0, 2.0);
        if (H.flags & FF_COUNT_DIR) direction(f, m);
        profile(H, f, m, true, 2.0, 2.0);
        log_hit(H, f);
        angle_map(H, f);
        double lu = dot(dir, H.nU), lv = dot(dir, H.nV), ln = dot(dir, H.N);
        dir = add(add(scl(lu, ld3(dph.nU)), scl(lv, ld3(dph.nV))), scl(ln, ld3(D->N)));
        double u = hu, v = hv;
        d3 O = ld3(D->O), U = ld3(D->U), V = ld3(D->V);
        pos = add(add(O, scl(u, U)), scl(v, V));
        const double* poly = P.poly + 2 * (size_t)D->poly_off;
        if (!in_polygon(poly, D->poly_n, u, v)) {
            for (int tr = 0; tr < 1000; ++tr) {
                u = rng.rnd(); v = rng.rnd();
                if (in_polygon(poly, D->poly_n, u, v)) { pos = add(add(O, scl(u, U)), scl(v, V)); break; }
            }
        }
        last_hit = dg;
        double ov = vel * ort(H);
        d3 z = mk(0, 0, 0);
        counter(H, f, m, 1, 0, 0, 2.0 / ov, 2.0 * vc().c_factor * ov, z, z, z);
    }
    // PerformScatter (Particle.cpp:840-886, Physics.cpp:41-63)
    MFG_IN bool scatter() {
        add_hit();
        ++nb_bounces;
        double rho = vc().scatter_rho, mr = vc().scatter_mr;
        double b = rho * sqrt(rng.rnd());
        double a = sqrt(rho * rho - b * b);
        double ctg = 1.0 / (2.0 * a * b) * (rho * rho * mr + b * b - a * a);
        double th = atan(1.0 / ctg);
        double az = 2.0 * kPi * rng.rnd();
        d3 rv = dir.x != 0.0 ? mk(0, 0, 1) : (dir.y != 0.0 ? mk(1, 0, 1) : mk(1, 0, 0));
        d3 un = unitv(cross(dir, rv)), vn = unitv(cross(dir, un));
        double st = sin(th), ct = cos(th), sa, ca;
        sincos(az, &sa, &ca);
        dir = add(add(scl(st * ca, un), scl(st * sa, vn)), scl(ct, dir));
        double q = mr * rho / b * st;
        vel = sqrt(vel * vel / (1.0 + q * q));
        scatter_path = dist + vc().scatter_mfp * -log(rng.rnd());
        trace(-1, 8);
        return !(vc().scatter_cutoff && vel < vc().scatter_cut);
    }

    // Add this lane's global counters to its variant and clear them.
    // ---- particles kept between launches
    MFG_IN void save(CarryRec& r, uint64_t events_left, uint32_t vi) const {
        r.pos[0] = pos.x; r.pos[1] = pos.y; r.pos[2] = pos.z;
        r.dir[0] = dir.x; r.dir[1] = dir.y; r.dir[2] = dir.z;
        r.time = time; r.vel = vel; r.ori = w(); r.gen_time = gen_time; r.dist = dist;
        r.decay_t = decay_t; r.scatter_path = scatter_path; r.hu = hu; r.hv = hv;
        r.pid = pid(); r.events_left = events_left;
        r.k0 = rng.k0; r.k1 = rng.k1; r.blk = rng.blk;
        r.b0 = rng.b0; r.b1 = rng.b1; r.b2 = rng.b2; r.b3 = rng.b3; r.avail = rng.avail;
        r.structure = structure; r.last_hit = last_hit; r.tele_from = tele_from;
        r.nb_bounces = nb_bounces; r.nb_events = nb_events; r.variant = vi; r.tr_n = tr_n;
    }
    MFG_IN uint64_t restore(const CarryRec& r) {
        pos = mk(r.pos[0], r.pos[1], r.pos[2]);
        dir = mk(r.dir[0], r.dir[1], r.dir[2]);
        vel = r.vel;
        if constexpr (WEIGHTED) ori = r.ori;
        if constexpr (CLOCKED) {
            time = r.time; gen_time = r.gen_time; dist = r.dist;
            decay_t = r.decay_t; scatter_path = r.scatter_path; hu = r.hu; hv = r.hv;
            tele_from = r.tele_from; nb_bounces = r.nb_bounces; nb_events = r.nb_events; tr_n = r.tr_n;
        }
        rng.k0 = r.k0; rng.k1 = r.k1; rng.p0 = (uint32_t)r.pid; rng.p1 = (uint32_t)(r.pid >> 32);
        rng.blk = r.blk; rng.b0 = r.b0; rng.b1 = r.b1; rng.b2 = r.b2; rng.b3 = r.b3; rng.avail = r.avail;
        structure = r.structure; last_hit = r.last_hit;
        return r.events_left;
    }

    MFG_IN double hit_equiv() const { return WEIGHTED ? acc_hit_equiv : (double)acc_hits; }
    MFG_IN double abs_equiv() const { return WEIGHTED ? acc_abs_equiv : (double)acc_absorbed; }
    MFG_IN double dist_full() const { return CLOCKED ? acc_dist_full : acc_dist_total; }
    MFG_IN void flush_lane() {
        if (var == nullptr) return;
        DGlobal* gl = P.glob + vc().glob_index;
        if (acc_hits) atomic_addu(&gl->nb_mc_hit, acc_hits);
        if (acc_des) atomic_addu(&gl->nb_desorbed, acc_des);
        if (hit_equiv() != 0.0) atomic_addd(&gl->nb_hit_equiv, hit_equiv());
        if (abs_equiv() != 0.0) atomic_addd(&gl->nb_abs_equiv, abs_equiv());
        if (acc_dist_total != 0.0) atomic_addd(&gl->dist_total, acc_dist_total);
        if (dist_full() != 0.0) atomic_addd(&gl->dist_full, dist_full());
        if (acc_decay) atomic_addu(&gl->nb_decayed, acc_decay);
        acc_hits = acc_des = acc_absorbed = acc_decay = 0;
        acc_hit_equiv = acc_abs_equiv = acc_dist_total = acc_dist_full = 0.0;
    }

    MFG_IN Root find_root() const {
        if constexpr (ONE) { if (P.one_root.node != -2) return P.one_root; }
        return P.roots[vc().root_base + (uint32_t)structure];
    }
    // One event of an alive particle (one SimulationMCStep iteration): its
    // ray goes into the wave's walk, which all lanes run together (also
    // those without a particle), then finish() treats what it met.
    MFG_IN HitRec trace_ray(uint32_t lane, bool alive) {
        Root root{-1, 0u};
        if (alive) {
            if constexpr (CLOCKED) ++nb_events;
            root = find_root();
            walk_load(W, lane, pos, dir, last_hit, 1e300);
            if constexpr ((FEAT & FEAT_TRANSPARENT) != 0) pass->n[lane] = 0;
        }
        const CoinState cs{rng.k0, rng.k1, rng.p0, rng.p1, nb_events, time, var};
        walk<(FEAT & FEAT_TRANSPARENT) != 0>(P, W, pass, lnodes, here(lane), alive, root, cs);
        lane = here(lane);
        // the ray is read back from its slot: not held in registers meanwhile
        const double2 a = W.p01[lane], b = W.p2d0[lane], c = W.d12[lane];
        pos = mk(a.x, a.y, b.x);
        dir = mk(b.y, c.x, c.y);
        const HitRec h{W.facet[lane], __longlong_as_double((long long)W.t[lane])};
        W.t[lane] = ~0ull;   // now the texture cell of the event
        return h;
    }
    // Returns false when the particle ends.
    MFG_IN bool finish(uint32_t lane, HitRec h) {
        constexpr bool TR = (FEAT & FEAT_TRANSPARENT) != 0;
        if (h.facet < 0) {  // leak
            atomic_addu(&P.glob[vc().glob_index].nb_leak, 1ull);   // rare: no register kept for it
            unsigned long long at = atomicAdd(P.leak_count, 1ull);
            if (at < P.leak_cap) {
                double* L = P.leaks + at * 6;
                L[0] = pos.x; L[1] = pos.y; L[2] = pos.z; L[3] = dir.x; L[4] = dir.y; L[5] = dir.z;
            }
            trace(-1, 6);
            return false;
        }
        double travel = h.t;
        int ev = 0;
        if constexpr ((FEAT & FEAT_VOLUME) != 0) {
            if (!vc().calc_const_flow) { double dl = vel * 100.0 * (vc().latest - time); if (dl < travel) { travel = dl; ev = 1; } }
            if (vc().enable_decay) { double dd = vel * 100.0 * (decay_t - time); if (dd < travel) { travel = dd; ev = 2; } }
            if (vc().scatter_enabled) { double ds = scatter_path - dist; if (ds < travel) { travel = ds; ev = 3; } }
        }
        if constexpr (TR) {
            if (vc().flags & FEAT_TRANSPARENT) {
                // every transparent pass closer than `travel`: the ones the
                // walk met and noted (in record order, the walk's own order
                // depending on the wave), or all of them from a second walk
                // of this lane if there were more than it notes
                const double save_u = hu, save_v = hv;
                const uint32_t n_pass = pass->n[lane];
                if (n_pass != 0 && n_pass <= MFG_PASSES) {
                    uint32_t q[MFG_PASSES];
#pragma unroll
                    for (uint32_t k = 0; k < MFG_PASSES; ++k) q[k] = k < n_pass ? pass->rec[lane][k] : ~0u;
#pragma unroll
                    for (uint32_t i = 1; i < MFG_PASSES; ++i)
#pragma unroll
                        for (uint32_t k = 0; k + i < MFG_PASSES; ++k)
                            if (q[k] > q[k + 1]) { const uint32_t x = q[k]; q[k] = q[k + 1]; q[k + 1] = x; }
                    for (uint32_t k = 0; k < n_pass; ++k) {
                        const uint32_t rec = k == 0 ? q[0] : k == 1 ? q[1] : k == 2 ? q[2] : q[3];
                        double t, u, v;
                        int32_t f;
                        uint32_t fl;
                        (void)leaf_test(P.leaves + rec, P.leaf_uv + rec, P.poly, pos, dir, last_hit, t, u, v, f, fl);
                        if (!(t < travel)) continue;
                        hu = u; hv = v;
                        transparent_pass(f, t);
                    }
                } else if (n_pass != 0) {
                    const int32_t root = find_root().node;
                    const LaneStack S{W.nodes + lane, MFG_LANE_STACK, P.stack_total, spill};
                    Ray32 r = make_ray32(pos, dir);
                    float tbf = widen(travel);
                    uint32_t sp = 0;
                    int32_t node = root;
                    for (;;) {
                        const NodeRegs nd = load_node_at(P.nodes, lnodes, P.lds_nodes, node);
                        uint32_t msk = node_hits(nd, r, tbf);
                        while (msk) {
                            uint32_t c = (uint32_t)__builtin_ctz(msk);
                            msk &= msk - 1u;
                            if (node_inner(nd) & (1u << c)) {
                                S.push(sp, node_inner_child(nd, c));
                                continue;
                            }
                            uint32_t first, cnt;
                            node_leaf_child(nd, c, first, cnt);
                            for (uint32_t kk = 0; kk < cnt; ++kk) {
                                double t, u, v;
                                int32_t f;
                                uint32_t fl;
                                bool hit = leaf_test(P.leaves + first + kk, P.leaf_uv + first + kk, P.poly, pos, dir, last_hit,
                                                     t, u, v, f, fl);
                                if (!hit || (fl & FF_OPAQUE)) continue;
                                if (!(t < travel)) continue;
                                double op = (fl & FF_TD_OPACITY) ? td_opacity(P, var, f, time) : (double)P.phys[f].opacity;
                                bool hard = op >= 1.0 || (op > 0.0 && rng.coin(nb_events, (uint32_t)local(f)) < op);
                                if (hard) continue;
                                hu = u; hv = v;
                                transparent_pass(f, t);
                            }
                        }
                        if (sp == 0) break;
                        node = S.pop(sp);
                    }
                }
                hu = save_u; hv = save_v;
            }
        }
        const int32_t f = h.facet;
        const HitRegs H = load_hit(P.hits + f);
        // the hit's facet coordinates, for the recordings that use them
        if (ev == 0 && (CLOCKED || (H.flags & (FF_TEXTURE | FF_PROFILE)))) hit_uv(P.facets + f, pos, dir, h.t, hu, hv);
        pos = add(pos, scl(travel, dir));
        if constexpr (CLOCKED) time += travel / 100.0 / vel;
        if (ev == 0) {
            acc_dist_total += travel;
            if constexpr (CLOCKED) { acc_dist_full += travel; dist += travel; }
            if constexpr ((FEAT & FEAT_TELEPORT) != 0) {
                if (H.flags & FF_TELEPORT) { teleport(H, f); return true; }
            }
            // absorption, or the weight's absorbed part (low flux), then the
            // bounce of what is left
            const double s = sticking(H, f);
            EventDraws g(rng);
            bool rec, go, lowflux = false;
            double w0 = 1.0;
            if constexpr (WEIGHTED) { lowflux = vc().low_flux != 0; w0 = ori; }
            if (!lowflux) {
                rec = s == 1.0 || (s > 0.0 && g.rnd() < s);
                go = !rec;
            } else {
                rec = s > 0.0;
                go = true;
                if constexpr (WEIGHTED) { if (rec) ori *= s; }
            }
            if (rec) record_absorb(H, f);
            if constexpr (WEIGHTED) {
                if (lowflux) {
                    ori = w0 * (1.0 - s);
                    if constexpr ((FEAT & FEAT_ADJOINT) != 0) { const int32_t g = P.hits[f].adj_group; if (rec && g >= 0) adj_cnt[g] += 1; }
                    go = ori > vc().low_flux_cutoff;
                    if constexpr ((FEAT & FEAT_ADJOINT) != 0) {
                        if (rec && go) seg_n = 0;
                        if (rec && !go) cutoff_boundary(P.hits[f].adj_group, s);
                    }
                }
            }
            if (go) bounce(g, H, f);
            else trace(f, 2);
            g.done();
            return go;
        }
        if (ev == 1 || ev == 2) {
            acc_dist_total += travel;
            ++acc_decay;
            trace(-1, 7);
            return false;
        }
        acc_dist_total += travel; acc_dist_full += travel; dist += travel;
        bool ok = scatter();
        last_hit = -1;
        if (!ok) { ++acc_decay; return false; }
        return true;
    }
};

__device__ __forceinline__ uint32_t find_variant(const uint64_t* prefix, uint32_t n, uint64_t g) {
    uint32_t lo = 0, hi = n;  // largest v with prefix[v] <= g
    while (hi - lo > 1) { uint32_t mid = (lo + hi) / 2; if (prefix[mid] <= g) lo = mid; else hi = mid; }
    return lo;
}

constexpr int kFewRecords = 8;   // fewer records than this go out lane by lane (nothing to merge, one LDS round trip less)

template <uint32_t FEAT, bool ONE>
__device__ __forceinline__ void trace_body(const TraceParams& P) {
    extern __shared__ __align__(16) unsigned char lds_base[];
    const uint32_t lane = __lane_id();
    WaveLds& W = reinterpret_cast<WaveLds*>(lds_base)[threadIdx.x >> 6];
    const size_t gl = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    int32_t* spill = P.stack_spill ? P.stack_spill + gl * (P.stack_total - MFG_LANE_STACK) : nullptr;
    // after the waves' walk areas: their pass areas (transparent models), the
    // hot-facet counters, the profile slices, the Maxwell table, and the copy
    // of the top of the tree (128 B a node), whose 16 B loads set the
    // alignment that every part keeps
    static_assert(sizeof(WaveLds) % 16 == 0 && sizeof(PassLds) % 16 == 0 && sizeof(MaxwellLds) % 16 == 0 &&
                  3 * MFG_PROFILE_SIZE * sizeof(double) % 16 == 0 && sizeof(mfg_facet_counters) % 16 == 0,
                  "parts of a block's LDS are multiples of 16 B");
    unsigned char* lds_next = lds_base + (blockDim.x >> 6) * sizeof(WaveLds);
    PassLds* pass = nullptr;
    if constexpr ((FEAT & FEAT_TRANSPARENT) != 0) {
        pass = reinterpret_cast<PassLds*>(lds_next) + (threadIdx.x >> 6);
        lds_next += (blockDim.x >> 6) * sizeof(PassLds);
    }
    Tracer<FEAT, ONE> T(P, W, pass, spill);
    double* hot = reinterpret_cast<double*>(lds_next);
    const uint32_t hot_words = 8u * P.n_hot * P.hot_slots;
    for (uint32_t i = threadIdx.x; i < hot_words; i += blockDim.x) hot[i] = 0.0;
    double* profs = hot + hot_words;
    const uint32_t prof_words = 3u * MFG_PROFILE_SIZE * P.n_prof_hot * P.prof_slots;
    for (uint32_t i = threadIdx.x; i < prof_words; i += blockDim.x) profs[i] = 0.0;
    MaxwellLds* maxwell = reinterpret_cast<MaxwellLds*>(profs + prof_words);
    if (P.maxwell_scale > 0.0) {
        const DVariant& v = ONE ? P.one : P.variants[0];
        for (uint32_t i = threadIdx.x; i < MFG_MAXWELL_POINTS; i += blockDim.x)
            maxwell->p[i] = make_double2(P.tab_x[v.maxwell_base + i], P.tab_y[v.maxwell_base + i]);
        for (uint32_t i = threadIdx.x; i < MFG_MAXWELL_GUIDE; i += blockDim.x)
            maxwell->guide[i] = (uint8_t)P.guides[v.maxwell_guide + i];
    }
    uint4* lnodes = reinterpret_cast<uint4*>(maxwell + (P.maxwell_scale > 0.0 ? 1 : 0));
    {
        const uint4* g = reinterpret_cast<const uint4*>(P.nodes);
        for (uint32_t i = threadIdx.x; i < 8u * P.lds_nodes; i += blockDim.x) lnodes[i] = g[i];
    }
    __syncthreads();
    T.hot = hot;
    T.profs = profs;
    T.maxwell = maxwell;
    T.lnodes = lnodes;
    if constexpr ((FEAT & FEAT_ADJOINT) != 0) {
        T.adj_cnt = P.adj_counts + (size_t)(blockIdx.x * blockDim.x + threadIdx.x) * P.adj_groups;
        T.seg_t = P.adj_seg_t + (size_t)(blockIdx.x * blockDim.x + threadIdx.x) * MFG_ADJ_SEG;
        T.seg_x = P.adj_seg_x + (size_t)(blockIdx.x * blockDim.x + threadIdx.x) * MFG_ADJ_SEG;
    }
    // few work items are spread over all waves: lanes beyond the quota stay
    // without a particle and help with the others' walks
    bool alive = false, done = lane >= P.lane_quota;
    uint32_t vi = 0;
    uint64_t events_left = 0;
    // work items: first the particles the previous launch left in flight,
    // then this launch's desorptions
    uint64_t n_in = 0;
    const CarryRec* carry_in = nullptr;
    CarryRec* carry_out = nullptr;
    unsigned long long* n_out = nullptr;
    if (P.carry) {
        uint32_t half = (uint32_t)P.carry_ctl[2] & 1u;
        n_in = P.carry_ctl[half];
        carry_in = P.carry + (size_t)half * P.carry_cap;
        carry_out = P.carry + (size_t)(half ^ 1u) * P.carry_cap;
        n_out = P.carry_ctl + (half ^ 1u);
    }
    const uint64_t items = n_in + P.total;
    const uint64_t t_start = wall_clock64();
    // kept in a register: read from the arguments at every event it cost a
    // lone particle 2 % (5k-facet pipe 27.5 ms, 27.0 so)
    const uint32_t refill_at = (uint32_t)__builtin_amdgcn_readfirstlane((int)(P.lane_quota < P.refill_at ? P.lane_quota : P.refill_at));
    uint32_t iter = 0;   // the loop is wave-uniform, and so is this count
    // the stop flag lives in host memory: a read crosses the bus, so it is
    // polled every 64 iterations, not at every refill
    int stop = __builtin_amdgcn_readfirstlane(*P.stop_flag);
    for (;;) {
        // the wall clock and the stop flag (read every 64 iterations) are
        // one value for the wave: expired and stop are uniform
        bool expired = false;
        if ((++iter & 63u) == 0u) {
            expired = __builtin_amdgcn_readfirstlane((int)((uint64_t)(wall_clock64() - t_start) > P.time_limit)) != 0;
            stop = __builtin_amdgcn_readfirstlane(*P.stop_flag);
        }
        if (expired && lane == 0) atomicMax(P.expired, 1ull);
        bool need = !alive && !done;
        uint64_t mask = expired ? 0ull : __ballot(need);
        // a refill costs the wave about the same for one lane as for many,
        // and a lane without a ray is no loss to the walk: wait for several
        if ((uint32_t)__popcll(mask) < refill_at && __ballot(alive)) mask = 0ull;
        bool dry = false;   // some lane of this wave found the queue exhausted
        if (mask) {
            uint32_t cnt = (uint32_t)__popcll(mask);
            uint32_t leader = (uint32_t)__ffsll((unsigned long long)mask) - 1;
            unsigned long long base = 0;
            if (iter == 1) {
                // the first items are dealt out by wave index: thousands of
                // waves taking them from the queue's one word would wait for
                // each other
                base = (unsigned long long)(gl >> 6) * P.lane_quota;
            } else {
                if (lane == leader) base = P.dealt + atomicAdd(P.next_particle, (unsigned long long)cnt);
                base = __shfl(base, leader, 64);
            }
            // after a stop request no new particle starts; resumed ones still
            // run (to the end, or back into the carry buffer)
            const uint64_t limit = stop ? n_in : items;
            bool started = false;
            int32_t src = -1;
            if (need) {
                uint64_t g = base + mbcnt(mask);
                if (g < n_in) {
                    const CarryRec& r = carry_in[g];
                    if constexpr (!ONE) {
                        vi = r.variant;
                        if (T.var != P.variants + vi) T.flush_lane();
                        T.var = P.variants + vi;
                    }
                    events_left = T.restore(r);
                    alive = true;
                } else if (g < limit) {
                    uint64_t d = g - n_in;
                    if constexpr (!ONE) {
                        vi = find_variant(P.var_prefix, P.n_variants, d);
                        if (T.var != P.variants + vi) T.flush_lane();
                        T.var = P.variants + vi;
                    }
                    ++T.acc_des;
                    uint64_t lp = (ONE ? d : d - P.var_prefix[vi]) + T.var->pid_base;
                    src = T.start(lp);
                    started = true;
                    alive = true;
                    events_left = P.max_events ? P.max_events : ~0ull;
                } else {
                    done = true;
                }
            }
            dry = __ballot(done && need) != 0;
            // desorption counters: lanes sharing the leader's source facet
            // add through one set of atomics
            uint64_t smask = __ballot(started);
            if (smask) {
                double ov = 0.0, w1 = 0.0, w2 = 0.0, w3 = 0.0;
                int m = -1;
                if (started) {
                    ov = T.vel * fabs(dot(T.dir, ld3(P.hits[src].N)));
                    w1 = 2.0 / ov; w2 = T.vc().c_factor * ov; w3 = 1.0 / T.vel;
                    m = T.moment(T.time);
                }
                uint32_t sl = (uint32_t)__ffsll((unsigned long long)smask) - 1;
                int32_t key = __shfl(src, sl, 64);
                bool grp = started && src == key;
                uint64_t gmask = __ballot(grp);
                double s1 = wave_sum(grp ? w1 : 0.0), s2 = wave_sum(grp ? w2 : 0.0), s3 = wave_sum(grp ? w3 : 0.0);
                if (grp && lane == sl) {
                    const int32_t hi = P.hits[src].hot_idx;
                    if (hi >= 0) {
                        double* h = hot + 8 * ((uint32_t)hi * P.hot_slots);
                        atomicAdd(reinterpret_cast<unsigned long long*>(h + 2), (unsigned long long)__popcll(gmask));
                        atomic_addd(h + 4, s1);
                        atomic_addd(h + 5, s2);
                        atomic_addd(h + 6, s3);
                    } else {
                        mfg_facet_counters* c = T.fc(src, 0);
                        atomic_addu(&c->nb_desorbed, (unsigned long long)__popcll(gmask));
                        atomic_addd(&c->sum_1_per_ort_velocity, s1);
                        atomic_addd(&c->sum_v_ort, s2);
                        atomic_addd(&c->sum_1_per_velocity, s3);
                    }
                }
                if (started && !grp) {
                    mfg_facet_counters* c = T.fc(src, 0);
                    atomic_addu(&c->nb_desorbed, 1ull);
                    atomic_addd(&c->sum_1_per_ort_velocity, w1);
                    atomic_addd(&c->sum_v_ort, w2);
                    atomic_addd(&c->sum_1_per_velocity, w3);
                }
                if (started) T.desorption_records(src, m, ov);
            }
        }
        if ((P.carry_keep && dry) || expired) {
            // the queue is empty (or the time limit is reached): park this
            // wave's particles for the next launch instead of running their
            // tails here; without carry, expiry ends them where they are
            uint64_t am = P.carry_keep ? __ballot(alive) : 0ull;
            if (am) {
                uint32_t al = (uint32_t)__ffsll((unsigned long long)am) - 1;
                unsigned long long ob = 0;
                if (lane == al) ob = atomicAdd(n_out, (unsigned long long)__popcll(am));
                ob = __shfl(ob, al, 64);
                if (alive) T.save(carry_out[ob + mbcnt(am)], events_left, vi);
            }
            break;
        }
        if (!__ballot(!done)) break;
        const HitRec met = T.trace_ray(here(lane), alive);
        if (alive) {
            alive = T.finish(here(lane), met);
            if (alive && --events_left == 0) alive = false;
        }
        // slot-0 facet counters of this iteration: lanes that updated the
        // same facet as the first pending lane add through one set of atomics
        uint64_t pm = __ballot(T.pend_f >= 0);
        if (pm) {
            uint32_t ld = (uint32_t)__ffsll((unsigned long long)pm) - 1;
            int32_t key = __shfl(T.pend_f, ld, 64);
            bool grp = T.pend_f == key;
            uint64_t gm = __ballot(grp);
            if (__popcll(gm) > 1) {
                double he = 0.0;
                if constexpr ((FEAT & FEAT_LOWFLUX) != 0) he = wave_sum(grp ? T.pend_he : 0.0);
                double ab = wave_sum(grp ? T.pend_abs : 0.0);
                double s1 = wave_sum(grp ? T.pend_s1v : 0.0), sv = wave_sum(grp ? T.pend_svo : 0.0);
                double sp = wave_sum(grp ? T.pend_s1pv : 0.0);
                unsigned long long hc = wave_sum_u(grp ? (unsigned long long)T.pend_hits : 0ull);
                if (lane == ld) {
                    T.pend_hits = (uint32_t)hc; T.pend_he = he; T.pend_abs = ab;
                    T.pend_s1v = s1; T.pend_svo = sv; T.pend_s1pv = sp;
                } else if (grp) {
                    T.clear_pending();
                }
            }
            // the records of the other facets: adjacent lanes add adjacent words
            // (3.. of a record), which leave the CU as one request. Device-
            // scope atomics are served at 2.35e10 requests a second however
            // many words one holds (1e5 records: 7.8e9 records a second with
            // a request for each of 3 words, 2.3e10 with 3 or 4 words in one).
            const bool cold = T.pend_f >= 0 && T.pend_hot < 0;
            const uint64_t cm = __ballot(cold);
            if (T.pend_f >= 0 && (!cold || __popcll(cm) < kFewRecords)) T.flush_pending_direct();
            if (__popcll(cm) >= kFewRecords) {
                constexpr uint32_t NW = decltype(T)::WEIGHTED ? 5 : 4;
                const uint32_t ln = here(lane);
                unsigned long long at = ~0ull;
                if (cold) {
                    at = T.vc().fc_base + (uint32_t)T.local(T.pend_f);
                    double* a = W.sums + NW * ln;
                    a[0] = T.pend_abs; a[1] = T.pend_s1v; a[2] = T.pend_svo; a[3] = T.pend_s1pv;
                    if constexpr (NW == 5) a[4] = T.weighted() ? T.pend_he : 0.0;   // in `reserved`: the read adds it
                    if (T.pend_hits) atomic_addu(&P.fc[at].nb_mc_hit, T.pend_hits);
                    T.clear_pending();
                }
                W.record[ln] = at;
                wave_sync();
#pragma unroll
                for (uint32_t q = 0; q < NW; ++q) {
                    const uint32_t j = q * 64u + ln, r = j / NW;
                    const unsigned long long rec = W.record[r];
                    const double v = W.sums[j];
                    if (rec != ~0ull && v != 0.0) atomic_addd(reinterpret_cast<double*>(P.fc + rec) + 3u + j % NW, v);
                }
                wave_sync();
            }
        }
        // the texture cells of this iteration, three words each, likewise
        const uint32_t ln = here(lane);
        if (__ballot(W.t[ln] != ~0ull)) {
            wave_sync();
#pragma unroll
            for (uint32_t q = 0; q < 3; ++q) {
                const uint32_t j = q * 64u + ln, r = j / 3u;
                const unsigned long long at = W.t[r];
                if (at == ~0ull) continue;
                const double v = W.cell[j];
                if (v != 0.0) atomic_addd(reinterpret_cast<double*>(P.tex + at) + j % 3u, v);
            }
            wave_sync();
        }
    }
    // flush lane accumulators: one set of atomics per wave for a single
    // variant, per lane otherwise
    if constexpr (ONE) {
        double he = wave_sum(T.hit_equiv()), ae = wave_sum(T.abs_equiv());
        double d1 = wave_sum(T.acc_dist_total), d2 = wave_sum(T.dist_full());
        unsigned long long hits = wave_sum_u(T.acc_hits), des = wave_sum_u(T.acc_des);
        unsigned long long dc = wave_sum_u(T.acc_decay);
        if (lane == 0) {
            DGlobal* gl = P.glob + P.one.glob_index;
            if (hits) atomic_addu(&gl->nb_mc_hit, hits);
            if (des) atomic_addu(&gl->nb_desorbed, des);
            if (he != 0.0) atomic_addd(&gl->nb_hit_equiv, he);
            if (ae != 0.0) atomic_addd(&gl->nb_abs_equiv, ae);
            if (d1 != 0.0) atomic_addd(&gl->dist_total, d1);
            if (d2 != 0.0) atomic_addd(&gl->dist_full, d2);
            if (dc) atomic_addu(&gl->nb_decayed, dc);
        }
    } else {
        T.flush_lane();
    }
    // every wave of the block has left the loop: add the block's hot-facet
    // sums to the global records
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < hot_words; i += blockDim.x) {
        const uint32_t k = (i >> 3) / P.hot_slots, slot = (i >> 3) % P.hot_slots, fld = i & 7u;
        if (fld == 7u) continue;
        double* g = reinterpret_cast<double*>(P.fc + P.hot_fc[k] + (size_t)slot * P.one.n_facets) + fld;
        if (fld == 0u || fld == 2u) {
            unsigned long long v = *reinterpret_cast<unsigned long long*>(hot + i);
            if (v) atomic_addu(reinterpret_cast<unsigned long long*>(g), v);
        } else if (hot[i] != 0.0) {
            atomic_addd(g, hot[i]);
        }
    }
    // and its profile slices
    for (uint32_t i = threadIdx.x; i < prof_words; i += blockDim.x) {
        if (profs[i] == 0.0) continue;
        const uint32_t per = 3u * MFG_PROFILE_SIZE, k = i / per, slot = k % P.prof_slots;
        double* g = reinterpret_cast<double*>(P.prof + P.hot_prof[k / P.prof_slots] + (size_t)slot * P.one.n_prof);
        atomic_addd(g + i % per, profs[i]);
    }
}

// One instantiation per occupancy bound: WAVES waves per SIMD caps the
// VGPR budget (cold per-particle state spills to scratch at the higher
// bounds); the host autotuner picks the fastest for a model.
template <uint32_t FEAT, int WAVES, bool ONE>
__global__ void __launch_bounds__(256, WAVES) k_trace(TraceParams P) {
    trace_body<FEAT, ONE>(P);
}

// One block per CU of 256 lanes per wave slot (768 lanes at 3 waves per
// SIMD, 1024 at 4): all waves of a CU share one LDS copy of the top of the
// tree, which can then hold several times the nodes of a 256-lane block's
// copy (single-variant launches: the others keep no copy).
template <uint32_t FEAT, int WAVES>
__global__ void __launch_bounds__(256 * WAVES, WAVES) k_trace_cu(TraceParams P) {
    trace_body<FEAT, true>(P);
}

// Parked particles that a launch did not claim: the launch deals out items
// [0, dealt), its queue hands out the `claimed` next ones, and the first
// n_in of all items are the resumed particles, so
// [min(dealt + claimed, n_in), n_in) were never taken. That happens only
// when the launch time limit stops the claims (a dry queue means every item was
// claimed). These records are appended to the output half after the ones
// the waves parked themselves.
__device__ __forceinline__ void carry_counts(const unsigned long long* ctl, const unsigned long long* claimed, uint64_t dealt,
                                             uint64_t& half, uint64_t& first, uint64_t& n, uint64_t& n_out) {
    half = ctl[2] & 1ull;
    const uint64_t n_in = ctl[half];
    first = dealt + *claimed < n_in ? dealt + *claimed : n_in;
    n = n_in - first;
    n_out = ctl[half ^ 1ull];
}
__global__ void k_carry_rescue(const unsigned long long* ctl, const unsigned long long* claimed, uint64_t dealt,
                               CarryRec* carry, uint64_t cap) {
    uint64_t half, first, n, n_out;
    carry_counts(ctl, claimed, dealt, half, first, n, n_out);
    const CarryRec* in = carry + half * cap;
    CarryRec* out = carry + (half ^ 1ull) * cap;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        if (n_out + i < cap) out[n_out + i] = in[first + i];
}
// After a launch (and the rescue): the half it resumed from is consumed,
// and the half that received its leftovers becomes the next launch's
// input. overflow is set if the rescued records did not fit.
__global__ void k_carry_flip(unsigned long long* ctl, const unsigned long long* claimed, uint64_t dealt, uint64_t cap,
                             unsigned long long* overflow) {
    if (threadIdx.x == 0) {
        uint64_t half, first, n, n_out;
        carry_counts(ctl, claimed, dealt, half, first, n, n_out);
        uint64_t total = n_out + n;
        if (total > cap) { *overflow = 1ull; total = cap; }
        ctl[half ^ 1ull] = total;
        ctl[half] = 0ull;
        ctl[2] = half ^ 1ull;
    }
}

// Fixed ray batches: a wave takes p.rays_per_wave rays at a time.
__global__ void __launch_bounds__(256) k_intersect(IsectParams p) {
    extern __shared__ __align__(16) unsigned char lds_base[];
    const uint32_t lane = __lane_id();
    WaveLds& W = reinterpret_cast<WaveLds*>(lds_base)[threadIdx.x >> 6];
    TraceParams tp{};
    tp.poly = p.poly; tp.nodes = p.nodes; tp.leaves = p.leaves; tp.leaf_uv = p.leaf_uv; tp.task_bits = p.task_bits;
    tp.child_lanes = p.child_lanes;
    const uint64_t wave = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const uint64_t i = wave * p.rays_per_wave + lane;
    const bool live = lane < p.rays_per_wave && i < p.n;
    d3 P = mk(0, 0, 0), D = mk(0, 0, 1);
    if (live) {
        P = ld3(p.origins + 3 * i);
        D = ld3(p.dirs + 3 * i);
        int32_t skip = p.last_hit ? p.last_hit[i] : -1;
        if (skip >= 0) skip += (int32_t)p.facet_base;
        walk_load(W, lane, P, D, skip, 1e300);
    }
    walk<false>(tp, W, nullptr, nullptr, lane, live, p.root, CoinState{});
    if (!live) return;
    const int32_t f = W.facet[lane];
    const double t = __longlong_as_double((long long)W.t[lane]);
    double u = 0.0, v = 0.0;
    if (f >= 0) hit_uv(p.facets + f, P, D, t, u, v);
    p.out_facet[i] = f >= 0 ? f - (int32_t)p.facet_base : -1;
    p.out_t[i] = f >= 0 ? t : 0.0;
    p.out_u[i] = u;
    p.out_v[i] = v;
}

// Clears several arrays of 8-byte words in one launch.
__global__ void __launch_bounds__(256) k_zero(ZeroList z) {
    const uint64_t first = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x, stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint32_t k = 0; k < z.n; ++k)
        for (uint64_t i = first; i < z.words[k]; i += stride) z.p[k][i] = 0;
}

__global__ void k_backward(const double* jac, const double* up, double* grad, uint32_t nt, uint32_t ng, double scale) {
    uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= ng) return;
    double s = 0.0;
    for (uint32_t t = 0; t < nt; ++t) s += up[t] * jac[(size_t)t * ng + g];
    grad[g] = s * scale;
}

// Instantiated feature sets: a model runs on the smallest one covering its
// features (fewer live registers, higher occupancy).
constexpr uint32_t kLean = 0;
constexpr uint32_t kLowFlux = FEAT_LOWFLUX;
constexpr uint32_t kLowFluxAdj = FEAT_LOWFLUX | FEAT_ADJOINT;
constexpr uint32_t kFull = FEAT_ALL;
constexpr uint32_t kFullAdj = FEAT_ALL | FEAT_ADJOINT;

}  // namespace

size_t mfg_wave_lds(uint32_t model_features) {
    return sizeof(WaveLds) + ((mfg_trace_kernel_features(model_features) & FEAT_TRANSPARENT) ? sizeof(PassLds) : 0);
}

uint32_t mfg_trace_kernel_features(uint32_t model_features) {
    const uint32_t rest = model_features & FEAT_ALL & ~FEAT_LOWFLUX;
    if (model_features & FEAT_ADJOINT) return rest ? kFullAdj : kLowFluxAdj;
    if (rest) return kFull;
    return (model_features & FEAT_LOWFLUX) ? kLowFlux : kLean;
}

namespace {
typedef void (*TraceKernel)(TraceParams);
// [feature set][waves per SIMD - 1]; null where not instantiated
// The one-block-per-CU kernels (lean and low-flux feature sets, 3 or 4
// waves per SIMD: 768 or 1024 lanes; low flux with the adjoint at 3).
TraceKernel kernel_cu(uint32_t features, int waves) {
    if (waves == 3) {
        if (features == kLean) return k_trace_cu<kLean, 3>;
        if (features == kLowFlux) return k_trace_cu<kLowFlux, 3>;
        if (features == kLowFluxAdj) return k_trace_cu<kLowFluxAdj, 3>;
    } else if (waves == 4) {
        if (features == kLean) return k_trace_cu<kLean, 4>;
        if (features == kLowFlux) return k_trace_cu<kLowFlux, 4>;
    }
    return nullptr;
}

template <bool ONE>
TraceKernel kernel_of(uint32_t features, int waves) {
    constexpr int N = 4;   // occupancy bounds 1..4 waves per SIMD (a fifth's walk areas do not fit the LDS)
    static TraceKernel lean[N] = {nullptr, k_trace<kLean, 2, ONE>, k_trace<kLean, 3, ONE>, k_trace<kLean, 4, ONE>};
    static TraceKernel full[N] = {k_trace<kFull, 1, ONE>, k_trace<kFull, 2, ONE>, k_trace<kFull, 3, ONE>, nullptr};
    static TraceKernel lowflux[N] = {nullptr, k_trace<kLowFlux, 2, ONE>, k_trace<kLowFlux, 3, ONE>, k_trace<kLowFlux, 4, ONE>};
    TraceKernel* t = features == kLean ? lean : features == kFull ? full : features == kLowFlux ? lowflux : nullptr;
    if constexpr (ONE) {
        // the adjoint takes one model
        static TraceKernel adj[N] = {k_trace<kFullAdj, 1, true>, k_trace<kFullAdj, 2, true>, nullptr, nullptr};
        static TraceKernel lowflux_adj[N] = {nullptr, k_trace<kLowFluxAdj, 2, true>, k_trace<kLowFluxAdj, 3, true>,
                                             k_trace<kLowFluxAdj, 4, true>};
        if (!t) t = features == kLowFluxAdj ? lowflux_adj : adj;
    }
    if (!t) return nullptr;
    if (waves < 1) waves = 1;
    if (waves > N) waves = N;
    for (int w = waves; w >= 1; --w) if (t[w - 1]) return t[w - 1];
    for (int w = waves; w <= N; ++w) if (t[w - 1]) return t[w - 1];
    return nullptr;
}
TraceKernel kernel_for(uint32_t features, bool single, int waves, int block) {
    if (block > 256) return single ? kernel_cu(features, block / 256) : nullptr;
    return single ? kernel_of<true>(features, waves) : kernel_of<false>(features, waves);
}
}  // namespace

int mfg_trace_variants(uint32_t features, int* waves_out, int cap) {
    uint32_t f = mfg_trace_kernel_features(features);
    int lo = 1, hi = 2;
    if (f == kLean || f == kLowFlux || f == kLowFluxAdj) { lo = 2; hi = 4; }
    else if (f == kFull) hi = 3;
    int n = 0;
    for (int w = lo; w <= hi && n < cap; ++w) waves_out[n++] = w;
    return n;
}

int mfg_trace_has_cu_block(uint32_t features, bool single, int block) {
    return single && block % 256 == 0 && kernel_cu(mfg_trace_kernel_features(features), block / 256) != nullptr;
}

int mfg_trace_occupancy(uint32_t features, bool single, int waves, int block, size_t lds) {
    int n = 0;
    const uint32_t f = mfg_trace_kernel_features(features);
    TraceKernel k = kernel_for(f, single, waves, block);
    if (!k) return 0;
    hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k, block, lds);
    return e == hipSuccess ? n : 1;
}

int mfg_launch_trace(const TraceParams& p, uint32_t features, bool single, int waves, int grid, int block, void* stream) {
    size_t lds = (size_t)(block / 64) * mfg_wave_lds(features) + ((size_t)p.n_hot * p.hot_slots * 8 + (size_t)p.n_prof_hot * p.prof_slots * 3 * MFG_PROFILE_SIZE) * sizeof(double) +
                 (p.maxwell_scale > 0.0 ? sizeof(MaxwellLds) : 0) + (size_t)p.lds_nodes * sizeof(BvhNode);
    const uint32_t f = mfg_trace_kernel_features(features);
    TraceKernel k = kernel_for(f, single, waves, block);
    if (!k) return -1;
    hipLaunchKernelGGL(k, dim3(grid), dim3(block), lds, (hipStream_t)stream, p);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int mfg_launch_carry_flip(unsigned long long* ctl, const unsigned long long* claimed, uint64_t dealt, CarryRec* carry, uint64_t cap,
                          unsigned long long* overflow, void* stream) {
    uint64_t blocks = (cap + 255) / 256;
    if (blocks > 1024) blocks = 1024;
    if (blocks == 0) blocks = 1;
    hipLaunchKernelGGL(k_carry_rescue, dim3((uint32_t)blocks), dim3(256), 0, (hipStream_t)stream, ctl, claimed, dealt,
                       carry, cap);
    if (hipGetLastError() != hipSuccess) return -1;
    hipLaunchKernelGGL(k_carry_flip, dim3(1), dim3(64), 0, (hipStream_t)stream, ctl, claimed, dealt, cap, overflow);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int mfg_launch_intersect(const IsectParams& p, void* stream) {
    const int block = 256;
    const uint64_t waves = (p.n + p.rays_per_wave - 1) / p.rays_per_wave;
    const uint64_t grid = (waves + block / 64 - 1) / (block / 64);
    if (grid == 0) return 0;
    hipLaunchKernelGGL(k_intersect, dim3((uint32_t)grid), dim3(block), (block / 64) * sizeof(WaveLds), (hipStream_t)stream, p);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int mfg_launch_zero(const ZeroList& z, void* stream) {
    uint64_t most = 0;
    for (uint32_t k = 0; k < z.n; ++k) most = most > z.words[k] ? most : z.words[k];
    if (most == 0) return 0;
    uint64_t grid = (most + 255) / 256;
    if (grid > 4096) grid = 4096;
    hipLaunchKernelGGL(k_zero, dim3((uint32_t)grid), dim3(256), 0, (hipStream_t)stream, z);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

// Device staging of the allocation-free fixed-ray-batch entry
// (mfg_intersect_batch_static): origins, directions, skip ids and the four
// outputs of up to MFG_STATIC_MAX_RAYS rays, at the fixed offsets of
// StaticRays. Every GPU the library runs on holds its own copy until the
// process ends; host code reaches it only through the address that
// mfg_scratch_address returns for the current device.
static __device__ __align__(256) unsigned char scratch[sizeof(StaticRays)];

namespace {
std::mutex g_scratch_mutex;
void* g_scratch_ptr[MFG_MAX_DEVICES] = {};
}  // namespace

int mfg_scratch_address(int device, StaticRays** out) {
    if (!out || device < 0 || device >= MFG_MAX_DEVICES) return -1;
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[device]) {
        int cur = -1;
        if (hipGetDevice(&cur) != hipSuccess || cur != device) return -1;   // the device must be current
        void* p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return -1;
        g_scratch_ptr[device] = p;
    }
    *out = static_cast<StaticRays*>(g_scratch_ptr[device]);
    return 0;
}

int mfg_launch_backward(const double* jac, const double* up, double* grad, uint32_t nt, uint32_t ng, double scale,
                        void* stream) {
    hipLaunchKernelGGL(k_backward, dim3((ng + 63) / 64), dim3(64), 0, (hipStream_t)stream, jac, up, grad, nt, ng, scale);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}
