// vg_mac.hip -- near-field treecode at grid points (accurate mode; this
// build's own method, no reference counterpart).
//
// The reference treecode opens only the cell that contains the query
// (vortonSim.cpp:1819-1856) and is accurate to a few tens of percent.  This
// mode keeps the same NestedGrid cluster pyramid but:
//   * opens every cell within +-near_k cells of the query's brick on every
//     layer (the near box), applying the remaining children as clusters;
//   * corrects each applied cluster with its first moment about the centroid
//     (order 1): u -= s/|d|^3 [a - 3/|d|^2 (D d) x d], D[b][e] = sum Omega_b
//     (y - c)_e, a = antisymmetric part of D;
//   * sums the leaf near box directly over its vortons (cell-sorted lists).
//
// GPU mapping: one wave = one 4x4x4 brick of grid points.  Near boxes are
// per brick, so every loop bound and branch is uniform across the wave.  The
// clusters of a layer are enumerated from the parent layer's near box: each
// lane reads one parent's mask of non-empty children (written by the tree
// build), and the children outside this layer's near box are queued in LDS.
// Every 64 queued clusters are staged in LDS.  A lane holds a row of four
// points and the four lanes of a row take every fourth cluster each
// (BrickRows), so an LDS read and a cluster's y and z terms serve four
// points; the lanes' shares are summed when the layer ends.  Batches whose
// clusters all have one size skip the per-cluster size test, and clusters
// that lie beyond the core radius by construction skip the core test.
//
// With one point per lane the five 16-byte LDS reads of a cluster took the
// LDS return path 40 of the CU's cycles per 64 interactions, more than their
// arithmetic: 3.0 ms for the 1M-vorton walk (129^3 points, near_k 3) and 3.5
// ms for 256 effects of 33^3 (near_k 2).  With four they take 10 and the walk
// is bound by VALU issue: 1.17e9 VALU instructions a launch, 4 cycles of a
// SIMD each, are 1.91 ms at 2.4 GHz, the LDS path 0.8: 1.89 and 2.5 ms.
// Capping the 101 registers at 96 or 80 for more waves was slower (2.9 ms
// against 2.7 for the whole frame): the four points' interleaved chains hide
// latency better than more waves do.  Grids of 1 to 3 points on two axes, whose
// layers hold a few clusters each, were up to a tenth faster with one point per
// lane (3x3x513, near_k 1: 37.8 against 42.7 us).
#include "vg_internal.h"

namespace vg {
vg_status tree_checked_view(const vg_tree *t, TreeView *v);

namespace {

struct MacParams {
    int k;
    float spread;
    float circ;
    uint32_t nb[3];
    uint32_t nbricks;
    int expand_from;  // layers >= expand_from go through brick-centred local expansions
};

__device__ __forceinline__ uint32_t uni(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }

// Cumulative decimation of layer l relative to the leaf layer, per axis.
__device__ __forceinline__ uint32_t layer_scale(const TreeView &tv, int l, int a) {
    uint32_t s = 1;
    for (int j = 1; j <= l; ++j) s *= tv.dec[j][a];
    return s;
}

// Children a parent may queue per round, and entries of the far-cluster queue.
constexpr uint32_t kTake = 8, kQueue = 64 + 64 * kTake;

// Per-wave LDS staging area: 64 fetched clusters (or vortons) at a time.
struct WaveStage {
    float4 P[64], W[64], M0[64], M1[64], M2[64];
    // leaf row tables (offsets in [0, 64), starts in [64, 128)), or the
    // cluster queue of the layers above
    uint32_t rows[kQueue];
};

// Lane-strided walk over the cells of a bx x by x bz box: lane `lane` visits
// cells t = lane, lane + 64, ... as (x, y, z) = (t % bx, t / bx % by,
// t / (bx by)), stepped without divisions (64 = qz bx by + ry bx + rx, one
// carry per axis).  t < bx by bz exactly when z < bz.
struct BoxIter {
    int x, y, z, bx, by, rx, ry, qz;
};

__device__ __forceinline__ BoxIter box_begin(int bx, int by, uint32_t lane) {
    BoxIter it;
    const int bxy = bx * by;
    it.bx = bx;
    it.by = by;
    it.z = (int)lane / bxy;
    const int r = (int)lane - it.z * bxy;
    it.y = r / bx;
    it.x = r - it.y * bx;
    it.qz = 64 / bxy;
    const int r64 = 64 - it.qz * bxy;
    it.ry = r64 / bx;
    it.rx = r64 - it.ry * bx;
    return it;
}

__device__ __forceinline__ void box_next(BoxIter &it) {
    it.x += it.rx;
    int c = it.x >= it.bx ? 1 : 0;
    it.x -= c ? it.bx : 0;
    it.y += it.ry + c;
    c = it.y >= it.by ? 1 : 0;
    it.y -= c ? it.by : 0;
    it.z += it.qz + c;
}

// Offset of a cell of a layer (the tree's grids hold fewer than 2^32 points).
__device__ __forceinline__ uint32_t cell_offset(const vg_grid_desc &g, int x, int y, int z) {
    return (uint32_t)x + g.np[0] * ((uint32_t)y + g.np[1] * (uint32_t)z);
}

// Kernel factors for one cluster size; contributions are accumulated
// unscaled and multiplied by s = (2/3) r^3 when the size changes or the
// layer ends (every cluster of a tree normally has the vorton size).
struct SizeFactors {
    float size = -1.0f, r2 = 0.f, s = 0.f, ir3 = 0.f;
};

__device__ __forceinline__ SizeFactors size_factors(float size, float spread) {
    SizeFactors f;
    f.size = size;
    const float radius = size * 0.5f * spread;
    f.r2 = radius * radius;
    f.s = (2.0f / 3.0f) * f.r2 * radius;
    f.ir3 = __builtin_amdgcn_rcpf(f.r2 * radius);
    return f;
}

// A lane's share of a brick: the four points x0..x0+3 of one (y, z) row.
// The four lanes of a quad own the same row and take every fourth item
// (cluster or vorton) each, so an item's LDS reads and its y and z terms
// serve four points of a lane.
struct Row4 {
    float x[4], y, z;
};
struct Part4 {
    float x[4], y[4], z[4];
};

__device__ __forceinline__ void part_clear(Part4 &p) {
#pragma unroll
    for (int i = 0; i < 4; ++i) p.x[i] = p.y[i] = p.z[i] = 0.f;
}

// DPP exchange inside a quad: lane ^ 1 (0xB1) or lane ^ 2 (0x4E).
template <int CTRL>
__device__ __forceinline__ float quad_swap(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, true));
}

// The quad's four shares of four points summed so that lane l keeps point
// l & 3: each step sends the half of the points it gives up.
__device__ __forceinline__ float quad_own(const float v[4], uint32_t lane) {
    const bool hi2 = (lane & 2u) != 0u, hi1 = (lane & 1u) != 0u;
    const float a = (hi2 ? v[2] : v[0]) + quad_swap<0x4E>(hi2 ? v[0] : v[2]);
    const float b = (hi2 ? v[3] : v[1]) + quad_swap<0x4E>(hi2 ? v[1] : v[3]);
    return (hi1 ? b : a) + quad_swap<0xB1>(hi1 ? a : b);
}

// Adds the quad's shares times scale to the lane's own point and clears them.
__device__ __forceinline__ void part_flush(Part4 &p, float scale, float3 &own, uint32_t lane) {
    own.x += quad_own(p.x, lane) * scale;
    own.y += quad_own(p.y, lane) * scale;
    own.z += quad_own(p.z, lane) * scale;
    part_clear(p);
}

// Monopole (+ first-moment) contribution of one cluster to a row's four
// points, unscaled by s (SCALED: times f.s).  m0..m2 carry the first
// moment's rows times 3 (.xyz, staged so by the walk) and its antisymmetric
// part (.w, unscaled).
// FAR: the caller knows the cluster lies outside the core radius (the law
// inside the core never applies); d2 carries 1e-24 so that a cluster of
// zero vorticity (whose centroid defaults to the origin) adds 0 even at a
// query point on the origin (1e-24 is below half an ulp of any squared
// distance above 1e-16, so elsewhere it can only settle a rounding tie).
//
// One point takes 18 VALU operations and an rsq with first moments (9 and
// an rsq without); the y and z parts of the distance, of D d and of the
// cross products are formed once for the four points.
template <int POLICY, int ORDER, bool FAR, bool SCALED>
__device__ __forceinline__ void cluster_row(Part4 &part, const Row4 &q, float4 p, float4 w,
                                            float4 m0, float4 m1, float4 m2,
                                            const SizeFactors &f) {
    const float dy = q.y - p.y, dz = q.z - p.z;
    const float dyz = FAR ? fmaf(dz, dz, fmaf(dy, dy, 1e-24f)) : fmaf(dz, dz, dy * dy);
    // D d without its x term
    const float t0 = fmaf(m0.z, dz, m0.y * dy), t1 = fmaf(m1.z, dz, m1.y * dy),
                t2 = fmaf(m2.z, dz, m2.y * dy);
    // w x d without its x terms
    const float cx = fmaf(w.y, dz, -(w.z * dy)), cy = w.x * dz, cz = w.x * dy;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float dx = q.x[i] - p.x;
        const float d2 = fmaf(dx, dx, dyz);
        float law, rs2;
        if (POLICY == VG_RSQRT_REFERENCE) {
            rs2 = __builtin_amdgcn_rcpf(d2);
            law = finvsqrtf(d2) * rs2;
        } else {
            const float rs = __builtin_amdgcn_rsqf(d2);
            rs2 = rs * rs;
            law = rs2 * rs;
        }
        const bool inside = !FAR && d2 < f.r2;
        float lm = inside ? f.ir3 : law;
        if (SCALED) lm *= f.s;
        if (ORDER >= 1) {
            // (w x d) lm - (a - 3 rs2 (t x d)) ld with t = D d folds into
            // ((w + c3 t3) x d) lm - a ld with t3 = 3 D d, c3 = rs2 outside
            // the core, 0 inside (where ld = 0): one cross product
            const float c3 = inside ? 0.0f : rs2;
            const float vx = fmaf(c3, fmaf(m0.x, dx, t0), w.x);
            const float vy = fmaf(c3, fmaf(m1.x, dx, t1), w.y);
            const float vz = fmaf(c3, fmaf(m2.x, dx, t2), w.z);
            if (FAR) {
                // lm = ld: ((v x d) - a) lm, three fused operations a row
                part.x[i] = fmaf(fmaf(vy, dz, -fmaf(vz, dy, m0.w)), lm, part.x[i]);
                part.y[i] = fmaf(fmaf(vz, dx, -fmaf(vx, dz, m1.w)), lm, part.y[i]);
                part.z[i] = fmaf(fmaf(vx, dy, -fmaf(vy, dx, m2.w)), lm, part.z[i]);
            } else {
                const float ld = inside ? 0.0f : lm;
                part.x[i] += (vy * dz - vz * dy) * lm - m0.w * ld;
                part.y[i] += (vz * dx - vx * dz) * lm - m1.w * ld;
                part.z[i] += (vx * dy - vy * dx) * lm - m2.w * ld;
            }
        } else {
            part.x[i] = fmaf(cx, lm, part.x[i]);
            part.y[i] = fmaf(fmaf(w.z, dx, -cy), lm, part.y[i]);
            part.z[i] = fmaf(fmaf(-w.y, dx, cz), lm, part.z[i]);
        }
        // the rarely taken forms finish one point before the next: four
        // interleaved ones would set the kernel's register count
        if (ORDER >= 1 && !FAR) __builtin_amdgcn_sched_barrier(0);
    }
}

// Local (Taylor) expansion about the brick centre of one cluster's field:
// monopole to second order, first moment to first order.  With d = c_b - c,
// K = d/|d|^3, u = s [Om x K(d) - sum_b e_b x (D_b . grad) K(d)]:
//   c0     = u(c_b)
//   c1[i][j] = du_i/dx_j                                 (9)
//   c2[i][p] = d2u_i/dx_j dx_k, p = 00 11 22 01 02 12   (18)
// Each lane expands its own cluster; the brick sums the lanes.
struct Expansion {
    float c0[3], c1[3][3], c2[3][6];
};

__device__ __forceinline__ void expansion_zero(Expansion &E) {
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        E.c0[i] = 0.f;
#pragma unroll
        for (int j = 0; j < 3; ++j) E.c1[i][j] = 0.f;
#pragma unroll
        for (int p = 0; p < 6; ++p) E.c2[i][p] = 0.f;
    }
}

__device__ __forceinline__ float3 cross3(float3 a, float3 b) {
    return make_float3(a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x);
}

template <int ORDER>
__device__ __forceinline__ void expansion_add(Expansion &E, float3 cb, float4 p, float4 w, float4 m0,
                                              float4 m1, float4 m2, float spread) {
    const float3 d = make_float3(cb.x - p.x, cb.y - p.y, cb.z - p.z);
    const float r2 = d.x * d.x + d.y * d.y + d.z * d.z;
    const float ir = __builtin_amdgcn_rsqf(r2);
    const float ir2 = ir * ir, ir3 = ir2 * ir, ir5 = ir3 * ir2, ir7 = ir5 * ir2;
    const float radius = p.w * 0.5f * spread;
    const float s = (2.0f / 3.0f) * radius * radius * radius;
    const float3 om = make_float3(s * w.x, s * w.y, s * w.z);
    const float dv[3] = {d.x, d.y, d.z};
    // Om x e_j and Om x d
    const float3 oe[3] = {make_float3(0.f, om.z, -om.y), make_float3(-om.z, 0.f, om.x),
                          make_float3(om.y, -om.x, 0.f)};
    const float3 od = cross3(om, d);
    E.c0[0] += od.x * ir3;
    E.c0[1] += od.y * ir3;
    E.c0[2] += od.z * ir3;
    // J[:, j] = e_j ir3 - 3 d d_j ir5
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const float f = -3.0f * ir5 * dv[j];
        E.c1[0][j] += oe[j].x * ir3 + od.x * f;
        E.c1[1][j] += oe[j].y * ir3 + od.y * f;
        E.c1[2][j] += oe[j].z * ir3 + od.z * f;
    }
    // c2[:, jk] = Om x T_jk. with T_jkb = d_j d_k K_b = 15 ir7 d_j d_k d_b
    // - 3 ir5 (delta_jb d_k + delta_kb d_j + delta_jk d_b), fully symmetric:
    // its 10 distinct components once, then one cross product per jk
    {
        const float a = -3.0f * ir5, g = 15.0f * ir7;
        const float gx = g * d.x, gy = g * d.y;
        const float xx = gx * d.x, yy = gy * d.y, zz = g * d.z * d.z, xy = gx * d.y;
        const float xxa = xx + a, yya = yy + a, zza = zz + a;
        const float txxx = d.x * (xxa + 2.0f * a), tyyy = d.y * (yya + 2.0f * a),
                    tzzz = d.z * (zza + 2.0f * a);
        const float txxy = d.y * xxa, txxz = d.z * xxa, tyyx = d.x * yya, tyyz = d.z * yya,
                    tzzx = d.x * zza, tzzy = d.y * zza, txyz = xy * d.z;
        const float3 T[6] = {make_float3(txxx, txxy, txxz), make_float3(tyyx, tyyy, tyyz),
                             make_float3(tzzx, tzzy, tzzz), make_float3(txxy, tyyx, txyz),
                             make_float3(txxz, txyz, tzzx), make_float3(txyz, tyyz, tzzy)};
#pragma unroll
        for (int q = 0; q < 6; ++q) {
            E.c2[0][q] = fmaf(om.y, T[q].z, fmaf(-om.z, T[q].y, E.c2[0][q]));
            E.c2[1][q] = fmaf(om.z, T[q].x, fmaf(-om.x, T[q].z, E.c2[1][q]));
            E.c2[2][q] = fmaf(om.x, T[q].y, fmaf(-om.y, T[q].x, E.c2[2][q]));
        }
    }
    if (ORDER >= 1) {
        // D rows (scaled), antisymmetric part a, t_b = D_b . d
        const float3 D0 = make_float3(s * m0.x, s * m0.y, s * m0.z);
        const float3 D1 = make_float3(s * m1.x, s * m1.y, s * m1.z);
        const float3 D2 = make_float3(s * m2.x, s * m2.y, s * m2.z);
        const float3 av = make_float3(s * m0.w, s * m1.w, s * m2.w);
        const float3 t = make_float3(D0.x * d.x + D0.y * d.y + D0.z * d.z,
                                     D1.x * d.x + D1.y * d.y + D1.z * d.z,
                                     D2.x * d.x + D2.y * d.y + D2.z * d.z);
        const float3 td = cross3(t, d);
        // c0 += -a ir3 + 3 ir5 (t x d)
        E.c0[0] += -av.x * ir3 + 3.0f * ir5 * td.x;
        E.c0[1] += -av.y * ir3 + 3.0f * ir5 * td.y;
        E.c0[2] += -av.z * ir3 + 3.0f * ir5 * td.z;
        // c1[:, j] += 3 ir5 [t x e_j + d_j a + col_j x d] - 15 ir7 d_j (t x d)
        const float3 col[3] = {make_float3(D0.x, D1.x, D2.x), make_float3(D0.y, D1.y, D2.y),
                               make_float3(D0.z, D1.z, D2.z)};
        const float3 te[3] = {make_float3(0.f, t.z, -t.y), make_float3(-t.z, 0.f, t.x),
                              make_float3(t.y, -t.x, 0.f)};
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const float3 cd = cross3(col[j], d);
            const float a3 = 3.0f * ir5, b15 = 15.0f * ir7 * dv[j];
            E.c1[0][j] += a3 * (te[j].x + dv[j] * av.x + cd.x) - b15 * td.x;
            E.c1[1][j] += a3 * (te[j].y + dv[j] * av.y + cd.y) - b15 * td.y;
            E.c1[2][j] += a3 * (te[j].z + dv[j] * av.z + cd.z) - b15 * td.z;
        }
    }
}

// Sum of the lanes' expansions (xor butterfly: every lane ends with the same
// bits) evaluated at offset x from the brick centre.
__device__ __forceinline__ float3 expansion_eval(Expansion &E, float3 x) {
    float *v = &E.c0[0];
#pragma unroll
    for (int i = 0; i < 30; ++i) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) v[i] += __shfl_xor(v[i], off, 64);
    }
    const float xv[3] = {x.x, x.y, x.z};
    float u[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        u[i] = E.c0[i] + E.c1[i][0] * xv[0] + E.c1[i][1] * xv[1] + E.c1[i][2] * xv[2] +
               0.5f * (E.c2[i][0] * xv[0] * xv[0] + E.c2[i][1] * xv[1] * xv[1] +
                       E.c2[i][2] * xv[2] * xv[2]) +
               E.c2[i][3] * xv[0] * xv[1] + E.c2[i][4] * xv[0] * xv[2] +
               E.c2[i][5] * xv[1] * xv[2];
    }
    return make_float3(u[0], u[1], u[2]);
}

// Inclusive sum over the wave: DPP shifts within rows of 16 lanes, then the
// last lane of each row (pair of rows) broadcast to the next.
template <int CTRL, int ROWS>
__device__ __forceinline__ uint32_t dpp_add(uint32_t v) {
    return v + (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xf, false);
}
__device__ __forceinline__ uint32_t wave_scan(uint32_t v) {
    v = dpp_add<0x111, 0xf>(v);  // row_shr:1
    v = dpp_add<0x112, 0xf>(v);  // row_shr:2
    v = dpp_add<0x114, 0xf>(v);  // row_shr:4
    v = dpp_add<0x118, 0xf>(v);  // row_shr:8
    v = dpp_add<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
    v = dpp_add<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3
    return v;
}

// Enumerates the non-empty cells of layer l that are children of the cells
// lo..hi of layer l + 1 and lie outside the near box n0..n1, through the LDS
// queue Q (kQueue entries).  Each lane takes one parent and reads its mask of
// non-empty children (so empty and near cells are never loaded); a wave scan
// of the counts gives each lane the slots of its children, up to kTake of
// them per round (one scan per round instead of one ballot per child).
// consume(first, count) then takes every full batch of 64 cell offsets from
// Q[first], the last batch of the layer as it is.
template <class Consume>
__device__ __forceinline__ void far_children(const TreeView &tv, int l, const int lo[3],
                                             const int hi[3], const int n0[3], const int n1[3],
                                             uint32_t *Q, uint32_t lane, Consume &&consume) {
    uint32_t qn = 0;  // entries waiting, fewer than 64 between rounds
    const vg_grid_desc &gl = tv.layer[l], &gp = tv.layer[l + 1];
    const uint32_t *__restrict__ Cm = tv.C[l + 1];
    const int dx = (int)tv.dec[l + 1][0], dy = (int)tv.dec[l + 1][1];
    const int dz = (int)tv.dec[l + 1][2];
    const bool halves = dx == 2 && dy == 2 && dz == 2;
    const uint32_t sy = gl.np[0], sz = gl.np[0] * gl.np[1];
    const int px = hi[0] - lo[0] + 1, py = hi[1] - lo[1] + 1, pz = hi[2] - lo[2] + 1;
    const int ptotal = px * py * pz;
    BoxIter it = box_begin(px, py, lane);
    uint32_t m = 0u, cbase = 0u;
    int base = 0;
    for (;;) {
        bool last = false;
        while (__ballot(m != 0u) == 0ull) {  // the next 64 parents
            if (base >= ptotal) {
                last = true;
                break;
            }
            if (it.z < pz) {
                const int ax = lo[0] + it.x, ay = lo[1] + it.y, az = lo[2] + it.z;
                m = Cm[cell_offset(gp, ax, ay, az)];
                const int cx = ax * dx, cy = ay * dy, cz = az * dz;
                cbase = cell_offset(gl, cx, cy, cz);
                if (halves) {
                    // bits of the children on the low and high side of each axis
                    // that lie inside the near box
                    const uint32_t nx = (cx >= n0[0] && cx <= n1[0] ? 0x55u : 0u) |
                                        (cx + 1 >= n0[0] && cx + 1 <= n1[0] ? 0xaau : 0u);
                    const uint32_t ny = (cy >= n0[1] && cy <= n1[1] ? 0x33u : 0u) |
                                        (cy + 1 >= n0[1] && cy + 1 <= n1[1] ? 0xccu : 0u);
                    const uint32_t nz = (cz >= n0[2] && cz <= n1[2] ? 0x0fu : 0u) |
                                        (cz + 1 >= n0[2] && cz + 1 <= n1[2] ? 0xf0u : 0u);
                    m &= ~(nx & ny & nz);
                } else {
                    // children of this parent inside the near box, per axis (a
                    // decimation is at most 3)
                    uint32_t nx = 0u, ny = 0u, nz = 0u;
#pragma unroll
                    for (int i = 0; i < 3; ++i) {
                        if (i < dx && cx + i >= n0[0] && cx + i <= n1[0]) nx |= 1u << i;
                        if (i < dy && cy + i >= n0[1] && cy + i <= n1[1]) ny |= 1u << i;
                        if (i < dz && cz + i >= n0[2] && cz + i <= n1[2]) nz |= 1u << i;
                    }
                    if (nx && ny && nz) {
                        uint32_t nm = 0u;
#pragma unroll
                        for (int k = 0; k < 3; ++k)
#pragma unroll
                            for (int j = 0; j < 3; ++j)
                                if (((nz >> k) & (ny >> j) & 1u) != 0u)
                                    nm |= nx << (dx * (j + dy * k));
                        m &= ~nm;
                    }
                }
            }
            base += 64;
            box_next(it);
        }
        if (!last) {
            const uint32_t c = min((uint32_t)__popc(m), kTake);
            const uint32_t incl = wave_scan(c);
            uint32_t at = qn + incl - c;
#pragma unroll
            for (uint32_t i = 0; i < kTake; ++i) {
                if (i < c) {
                    const uint32_t bit = (uint32_t)__builtin_ctz(m);
                    m &= m - 1u;
                    uint32_t off;
                    if (halves) {
                        off = cbase + (bit & 1u) + ((bit & 2u) ? sy : 0u) + ((bit & 4u) ? sz : 0u);
                    } else {
                        const uint32_t jk = bit / (uint32_t)dx, k = jk / (uint32_t)dy;
                        off = cbase + (bit - jk * (uint32_t)dx) + (jk - k * (uint32_t)dy) * sy +
                              k * sz;
                    }
                    Q[at++] = off;
                }
            }
            qn += (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
        }
        uint32_t first = 0;
        if (qn >= (last ? 1u : 64u)) {
            __builtin_amdgcn_wave_barrier();
            do {
                const uint32_t cnt = min(64u, qn - first);
                consume(first, cnt);
                first += cnt;
            } while (first + (last ? 1u : 64u) <= qn);
        }
        if (last) break;
        if (first) {
            const uint32_t rest = qn - first;
            const uint32_t moved = lane < rest ? Q[first + lane] : 0u;
            __builtin_amdgcn_wave_barrier();
            if (lane < rest) Q[lane] = moved;
            __builtin_amdgcn_wave_barrier();
            qn = rest;
        }
    }
}

// The points of one brick as the lanes of its wave hold them.  A row is the
// four points of a brick along its row axis `ax`; the row axis is the first
// one whose four points all exist (a brick at the grid's upper faces has
// fewer on some axes), and the other two axes follow it cyclically, which
// keeps the sense of the cross products.  A row's lanes (4, 16 or 64 of
// them, as few rows allow) take the items of a batch in turn.
struct BrickRows {
    uint32_t ax, ay, az;  // grid axes of the rotated x, y, z
    uint32_t slots;       // lanes per row
    uint32_t slot;        // this lane's
    Row4 q;               // this lane's row, rotated axes
    uint32_t pt[3];       // the lane's own point, grid axes
    bool owner;           // the lane writes its own point
};

__device__ __forceinline__ BrickRows brick_rows(const vg_grid_desc &g, const uint32_t bb[3],
                                                uint32_t lane) {
    uint32_t nv[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) nv[a] = min(4u, g.np[a] - 4 * bb[a]);
    BrickRows r;
    r.ax = nv[0] == 4u ? 0u : nv[1] == 4u ? 1u : nv[2] == 4u ? 2u : 0u;
    r.ay = r.ax == 2u ? 0u : r.ax + 1u;
    r.az = r.ay == 2u ? 0u : r.ay + 1u;
    auto pick = [](const uint32_t v[3], uint32_t a) { return a == 0u ? v[0] : a == 1u ? v[1] : v[2]; };
    const uint32_t nx = pick(nv, r.ax), ny = pick(nv, r.ay), nz = pick(nv, r.az);
    const uint32_t rows = ny * nz;
    r.slots = rows == 1u ? 64u : rows <= 4u ? 16u : 4u;
    r.slot = lane & (r.slots - 1u);
    uint32_t row = rows == 1u ? 0u : rows <= 4u ? lane >> 4 : lane >> 2;
    const bool live = row < rows;
    if (!live) row = rows - 1u;
    const uint32_t jz = row / ny, jy = row - jz * ny;
    const uint32_t jx = r.slot & 3u;
    r.owner = live && r.slot < 4u && jx < nx;
    const uint32_t b0[3] = {4 * bb[0], 4 * bb[1], 4 * bb[2]};
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) {
        const uint32_t ix = min(i, nx - 1u);
        uint32_t p[3];
#pragma unroll
        for (uint32_t a = 0; a < 3; ++a) p[a] = b0[a] + (a == r.ax ? ix : a == r.ay ? jy : jz);
        const float3 c = grid_query_point(g, p[0], p[1], p[2]);
        const float cv[3] = {c.x, c.y, c.z};
        r.q.x[i] = r.ax == 0u ? cv[0] : r.ax == 1u ? cv[1] : cv[2];
        r.q.y = r.ay == 0u ? cv[0] : r.ay == 1u ? cv[1] : cv[2];
        r.q.z = r.az == 0u ? cv[0] : r.az == 1u ? cv[1] : cv[2];
        if (i == min(jx, nx - 1u)) {
#pragma unroll
            for (int a = 0; a < 3; ++a) r.pt[a] = p[a];
        }
    }
    return r;
}

// (x, y, z) with x moved to the row axis: component ax first.
__device__ __forceinline__ float4 rotate(float4 v, uint32_t ax) {
    if (ax == 0u) return v;
    return ax == 1u ? make_float4(v.y, v.z, v.x, v.w) : make_float4(v.z, v.x, v.y, v.w);
}
// ... and back.
__device__ __forceinline__ float3 rotate_back(float3 v, uint32_t ax) {
    if (ax == 0u) return v;
    return ax == 1u ? make_float3(v.z, v.x, v.y) : make_float3(v.y, v.z, v.x);
}

// Sum over a row's lanes beyond the quad (16 or 64 lanes per row).
__device__ __forceinline__ float3 row_sum(float3 v, uint32_t slots) {
    for (uint32_t m = 4u; m < slots; m <<= 1) {
        v.x += __shfl_xor(v.x, (int)m, 64);
        v.y += __shfl_xor(v.y, (int)m, 64);
        v.z += __shfl_xor(v.z, (int)m, 64);
    }
    return v;
}

// One wave evaluates one brick of grid points; S is the wave's LDS slot.
template <int POLICY, int ORDER, int COUNT>
__device__ __forceinline__ void mac_brick(const TreeView &tv, const vg_grid_desc &g,
                                          const MacParams &mp, uint32_t brick, WaveStage &S,
                                          float *__restrict__ out,
                                          unsigned long long *__restrict__ counts) {
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t bb[3] = {brick % mp.nb[0], (brick / mp.nb[0]) % mp.nb[1],
                            brick / (mp.nb[0] * mp.nb[1])};
    int cl0[3], cl1[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const int nc = (int)g.np[a] - 1;
        const int first = (int)(4 * bb[a]);
        int last = first + 3;
        if (last > (int)g.np[a] - 1) last = (int)g.np[a] - 1;
        cl0[a] = first < nc - 1 ? first : nc - 1;
        cl1[a] = last < nc - 1 ? last : nc - 1;
    }
    const BrickRows br = brick_rows(g, bb, lane);
    const Row4 &q = br.q;
    const uint32_t slot = br.slot, slots = br.slots;
    float3 sum = make_float3(0.f, 0.f, 0.f), comp = sum;
    unsigned long long n_clusters = 0, n_pairs = 0, n_expand = 0;
    const bool expanding = mp.expand_from >= 1 && mp.expand_from <= (int)tv.depth - 2;
    const float spread = mp.spread;
    const int depth = (int)tv.depth;
    SizeFactors f;
    int lo[3] = {0, 0, 0}, hi[3] = {0, 0, 0};
    for (int l = depth - 2; l >= 0; --l) {
        const vg_grid_desc &gl = tv.layer[l];
        int c0[3], c1[3], n0[3], n1[3];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const int dec = (int)tv.dec[l + 1][a];
            const int sc = (int)layer_scale(tv, l, a);
            c0[a] = lo[a] * dec;
            c1[a] = hi[a] * dec + dec - 1;
            const int ncl = (int)gl.np[a] - 1;
            int blo = cl0[a] / sc - mp.k, bhi = cl1[a] / sc + mp.k;
            blo = blo < 0 ? 0 : blo;
            bhi = bhi > ncl - 1 ? ncl - 1 : bhi;
            n0[a] = blo > c0[a] ? blo : c0[a];
            n1[a] = bhi < c1[a] ? bhi : c1[a];
        }
        const float4 *__restrict__ P = tv.P[l];
        const float4 *__restrict__ W = tv.W[l];
        const float4 *__restrict__ M = tv.M[l];
        // A cluster of this layer outside the near box lies at least k of
        // its cells from every point of the brick (its centroid is inside
        // its cell; the 0.99 absorbs the grid points' inward nudge): core
        // radii below that never apply.
        float far2;
        {
            const float h = fminf(gl.cell[0], fminf(gl.cell[1], gl.cell[2]));
            const float dmin = 0.99f * (float)mp.k * h;
            far2 = dmin * dmin;
        }
        const int bx = c1[0] - c0[0] + 1, by = c1[1] - c0[1] + 1, bz = c1[2] - c0[2] + 1;
        const int total = bx * by * bz;
        if (expanding && l >= mp.expand_from) {
            // these layers were applied by k_mac_expand, which left the raw
            // (unscaled by circ) expansion value in out
            if (COUNT) {
                BoxIter it = box_begin(bx, by, lane);
                for (int base = 0; base < total; base += 64, box_next(it)) {
                    bool use = false;
                    if (it.z < bz) {
                        const int cx = c0[0] + it.x, cy = c0[1] + it.y, cz = c0[2] + it.z;
                        const bool near = cx >= n0[0] && cx <= n1[0] && cy >= n0[1] &&
                                          cy <= n1[1] && cz >= n0[2] && cz <= n1[2];
                        if (!near) use = P[cell_offset(gl, cx, cy, cz)].w != 0.0f;
                    }
                    n_expand += __popcll(__ballot(use));
                }
            } else if (l == mp.expand_from && br.owner) {
                const size_t o = point_offset(g, br.pt[0], br.pt[1], br.pt[2]);
                const float4 u =
                    rotate(make_float4(out[3 * o], out[3 * o + 1], out[3 * o + 2], 0.f), br.ax);
                kahan_add(sum, comp, make_float3(u.x, u.y, u.z));
            }
#pragma unroll
            for (int a = 0; a < 3; ++a) { lo[a] = n0[a]; hi[a] = n1[a]; }
            continue;
        }
        Part4 part;
        part_clear(part);
        float3 own = make_float3(0.f, 0.f, 0.f);
        if (COUNT) {
            BoxIter it = box_begin(bx, by, lane);
            for (int base = 0; base < total; base += 64, box_next(it)) {
                bool use = false;
                if (it.z < bz) {
                    const int cx = c0[0] + it.x, cy = c0[1] + it.y, cz = c0[2] + it.z;
                    const bool near = cx >= n0[0] && cx <= n1[0] && cy >= n0[1] &&
                                      cy <= n1[1] && cz >= n0[2] && cz <= n1[2];
                    if (!near) use = P[cell_offset(gl, cx, cy, cz)].w != 0.0f;
                }
                n_clusters += __popcll(__ballot(use));
            }
        } else {
            // Far clusters of the layer come through the LDS queue, 64 at a
            // time (fewer than 64 wait between rounds).
            uint32_t *Q = S.rows;
            auto consume = [&](uint32_t first, uint32_t cnt) {
                // lanes past the count stage the first cluster's position
                // with zero vorticity: they add nothing
                const bool use = lane < cnt;
                const uint32_t off = Q[first + (use ? lane : 0u)];
                const float4 p = P[off];
                float4 w = make_float4(0.f, 0.f, 0.f, 0.f), m0 = w, m1 = w, m2 = w;
                if (use) {
                    w = W[off];
                    if (ORDER) {
                        m0 = M[3 * (size_t)off];
                        m1 = M[3 * (size_t)off + 1];
                        m2 = M[3 * (size_t)off + 2];
                    }
                }
                S.P[lane] = rotate(p, br.ax);
                S.W[lane] = rotate(w, br.ax);
                if (ORDER) {
                    if (br.ax != 0u) {
                        const float4 r0 = rotate(m0, br.ax), r1 = rotate(m1, br.ax),
                                     r2 = rotate(m2, br.ax);
                        m0 = br.ax == 1u ? r1 : r2;
                        m1 = br.ax == 1u ? r2 : r0;
                        m2 = br.ax == 1u ? r0 : r1;
                    }
                    // rows times 3 (cluster_row's convention), once per cluster
                    S.M0[lane] = make_float4(3.0f * m0.x, 3.0f * m0.y, 3.0f * m0.z, m0.w);
                    S.M1[lane] = make_float4(3.0f * m1.x, 3.0f * m1.y, 3.0f * m1.z, m1.w);
                    S.M2[lane] = make_float4(3.0f * m2.x, 3.0f * m2.y, 3.0f * m2.z, m2.w);
                }
                // the batch's clusters have one size (the usual case: one
                // vorton size per tree)?
                const float size = __int_as_float((int)uni((uint32_t)__float_as_int(p.w)));
                const bool one_size = __ballot(p.w != size) == 0ull;
                if (!one_size || size != f.size) {
                    part_flush(part, f.s, own, lane);
                    f = size_factors(size, spread);
                }
                __builtin_amdgcn_wave_barrier();
                const uint32_t steps = (cnt + slots - 1u) / slots;  // one cluster per slot a step
                if (one_size && f.r2 < far2) {
                    for (uint32_t k = 0, j = slot; k < steps; ++k, j += slots)
                        cluster_row<POLICY, ORDER, true, false>(part, q, S.P[j], S.W[j], S.M0[j],
                                                                S.M1[j], S.M2[j], f);
                } else {
                    // one size keeps part in units of s; several sizes scale
                    // each cluster by its own
                    SizeFactors fj = f;
                    fj.s = 1.0f;
                    for (uint32_t k = 0, j = slot; k < steps; ++k, j += slots) {
                        const float4 cp = S.P[j];
                        if (!one_size) fj = size_factors(cp.w, spread);
                        cluster_row<POLICY, ORDER, false, true>(part, q, cp, S.W[j], S.M0[j],
                                                                S.M1[j], S.M2[j], fj);
                    }
                    if (!one_size) part_flush(part, 1.0f, own, lane);
                }
                __builtin_amdgcn_wave_barrier();
            };
            far_children(tv, l, lo, hi, n0, n1, Q, lane, consume);
            __builtin_amdgcn_wave_barrier();
            part_flush(part, f.s, own, lane);
        }
        kahan_add(sum, comp, own);
#pragma unroll
        for (int a = 0; a < 3; ++a) { lo[a] = n0[a]; hi[a] = n1[a]; }
    }
    // Leaf near box (or every vorton when the tree has one layer), fetched by
    // rows: the vortons of cells x0..x1 of one (y, z) row are contiguous in
    // the cell-sorted arrays.
    const vg_grid_desc &g0 = tv.layer[0];
    if (depth == 1) {
        lo[0] = lo[1] = lo[2] = 0;
        hi[0] = (int)g0.np[0] - 2;
        hi[1] = (int)g0.np[1] - 2;
        hi[2] = (int)g0.np[2] - 2;
    }
    {
        Part4 part;
        part_clear(part);
        float3 own = make_float3(0.f, 0.f, 0.f);
        const int ry = hi[1] - lo[1] + 1, rz = hi[2] - lo[2] + 1;
        const int nrows = ry * rz;
        for (int rbase = 0; rbase < nrows; rbase += 64) {
            const int r = rbase + (int)lane;
            uint32_t rs = 0, rc = 0;
            if (r < nrows) {
                const int cy = lo[1] + r % ry, cz = lo[2] + r / ry;
                const size_t k0 = point_offset(g0, lo[0], cy, cz);
                const size_t k1 = point_offset(g0, hi[0], cy, cz);
                rs = tv.cell_start[k0];
                rc = tv.cell_start[k1] + tv.cell_count[k1] - rs;
            }
            // inclusive scan of the row counts across the wave
            const uint32_t incl = wave_scan(rc);
            const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
            if (COUNT) {
                n_pairs += total;
                continue;
            }
            S.rows[lane] = incl - rc;
            S.rows[64 + lane] = rs;
            __builtin_amdgcn_wave_barrier();
            for (uint32_t vbase = 0; vbase < total; vbase += 64) {
                // lanes past the count stage the first vorton's position with
                // zero vorticity: they add nothing
                const uint32_t cnt = total - vbase < 64u ? total - vbase : 64u;
                const bool use = lane < cnt;
                const uint32_t t = use ? vbase + lane : vbase;
                // last row whose offset is <= t
                int lo_i = 0, hi_i = 63;
                while (lo_i < hi_i) {
                    const int mid = (lo_i + hi_i + 1) >> 1;
                    if (S.rows[mid] <= t) lo_i = mid;
                    else hi_i = mid - 1;
                }
                const uint32_t idx = S.rows[64 + lo_i] + (t - S.rows[lo_i]);
                const float4 p = tv.sorted_p[idx];
                float4 w = make_float4(0.f, 0.f, 0.f, 0.f);
                if (use) w = tv.sorted_w[idx];
                const float size = __int_as_float((int)uni((uint32_t)__float_as_int(p.w)));
                const bool one_size = __ballot(p.w != size) == 0ull;
                if (!one_size || size != f.size) {
                    part_flush(part, f.s, own, lane);
                    f = size_factors(size, spread);
                }
                __builtin_amdgcn_wave_barrier();
                S.P[lane] = rotate(p, br.ax);
                S.W[lane] = rotate(w, br.ax);
                __builtin_amdgcn_wave_barrier();
                const uint32_t steps = (cnt + slots - 1u) / slots;
                if (one_size) {
                    for (uint32_t k = 0, j = slot; k < steps; ++k, j += slots) {
                        const float4 vp = S.P[j];
                        cluster_row<POLICY, 0, false, false>(part, q, vp, S.W[j], vp, vp, vp, f);
                    }
                } else {
                    for (uint32_t k = 0, j = slot; k < steps; ++k, j += slots) {
                        const float4 vp = S.P[j];
                        cluster_row<POLICY, 0, false, true>(part, q, vp, S.W[j], vp, vp, vp,
                                                            size_factors(vp.w, spread));
                    }
                    part_flush(part, 1.0f, own, lane);
                }
                __builtin_amdgcn_wave_barrier();
            }
        }
        part_flush(part, f.s, own, lane);
        kahan_add(sum, comp, own);
    }
    if (COUNT) {
        // the ballot must run on every lane: inside the lane-0 branch only
        // lane 0 would vote
        const unsigned long long nv = (unsigned long long)__popcll(__ballot(br.owner));
        if (lane == 0) {
            atomicAdd(&counts[0], n_clusters * nv);
            atomicAdd(&counts[1], n_pairs * nv);
            atomicAdd(&counts[2], n_expand);
        }
        return;
    }
    sum = rotate_back(row_sum(sum, slots), br.ax);
    if (br.owner) {
        const size_t o = point_offset(g, br.pt[0], br.pt[1], br.pt[2]);
        out[3 * o] = sum.x * mp.circ;
        out[3 * o + 1] = sum.y * mp.circ;
        out[3 * o + 2] = sum.z * mp.circ;
    }
}

// Layers >= expand_from of the near-field walk for one brick: every lane
// expands its fetched clusters about the brick centre, the wave sums the
// expansions and each point writes their raw value (not yet scaled by circ)
// to out, where the per-point walk picks it up.  Kept apart from mac_brick
// so the per-point walk keeps its small register footprint.
template <int ORDER>
__device__ __forceinline__ void expand_brick(const TreeView &tv, const vg_grid_desc &g,
                                             const MacParams &mp, uint32_t brick,
                                             uint32_t *__restrict__ Q, float *__restrict__ out) {
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t bb[3] = {brick % mp.nb[0], (brick / mp.nb[0]) % mp.nb[1],
                            brick / (mp.nb[0] * mp.nb[1])};
    const uint32_t lp[3] = {lane & 3u, (lane >> 2) & 3u, lane >> 4};
    uint32_t pt[3];
    bool valid = true;
    int cl0[3], cl1[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const uint32_t p = 4 * bb[a] + lp[a];
        valid = valid && p < g.np[a];
        pt[a] = p < g.np[a] ? p : g.np[a] - 1;
        const int nc = (int)g.np[a] - 1;
        const int first = (int)(4 * bb[a]);
        int last = first + 3;
        if (last > (int)g.np[a] - 1) last = (int)g.np[a] - 1;
        cl0[a] = first < nc - 1 ? first : nc - 1;
        cl1[a] = last < nc - 1 ? last : nc - 1;
    }
    const float3 q = grid_query_point(g, pt[0], pt[1], pt[2]);
    float3 cb;
    {
        const float nudge = 1.0f - 2.0f * FLT_EPSILON;
        cb.x = g.min[0] + ((float)(4 * bb[0]) + 1.5f) * (g.cell[0] * nudge);
        cb.y = g.min[1] + ((float)(4 * bb[1]) + 1.5f) * (g.cell[1] * nudge);
        cb.z = g.min[2] + ((float)(4 * bb[2]) + 1.5f) * (g.cell[2] * nudge);
    }
    Expansion E;
    expansion_zero(E);
    // Accepted clusters (layer << 28 | offset) queue up in Q and are expanded
    // 64 at a time, one per lane, so that no lane idles on an empty or near
    // candidate cell while the others expand.
    uint32_t qn = 0;  // wave-uniform queue length, < 128
    auto expand_one = [&](uint32_t e) {
        const int l = (int)(e >> 28);
        const uint32_t off = e & 0x0fffffffu;
        const float4 p = tv.P[l][off];
        const float4 w = tv.W[l][off];
        float4 m0 = p, m1 = p, m2 = p;
        if (ORDER) {
            m0 = tv.M[l][3 * (size_t)off];
            m1 = tv.M[l][3 * (size_t)off + 1];
            m2 = tv.M[l][3 * (size_t)off + 2];
        }
        expansion_add<ORDER>(E, cb, p, w, m0, m1, m2, mp.spread);
    };
    int lo[3] = {0, 0, 0}, hi[3] = {0, 0, 0};
    for (int l = (int)tv.depth - 2; l >= mp.expand_from; --l) {
        const vg_grid_desc &gl = tv.layer[l];
        int c0[3], c1[3], n0[3], n1[3];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const int dec = (int)tv.dec[l + 1][a];
            const int sc = (int)layer_scale(tv, l, a);
            c0[a] = lo[a] * dec;
            c1[a] = hi[a] * dec + dec - 1;
            const int ncl = (int)gl.np[a] - 1;
            int blo = cl0[a] / sc - mp.k, bhi = cl1[a] / sc + mp.k;
            blo = blo < 0 ? 0 : blo;
            bhi = bhi > ncl - 1 ? ncl - 1 : bhi;
            n0[a] = blo > c0[a] ? blo : c0[a];
            n1[a] = bhi < c1[a] ? bhi : c1[a];
        }
        const int bx = c1[0] - c0[0] + 1, by = c1[1] - c0[1] + 1, bz = c1[2] - c0[2] + 1;
        const int total = bx * by * bz;
        BoxIter it = box_begin(bx, by, lane);
        for (int base = 0; base < total; base += 64, box_next(it)) {
            bool take = false;
            uint32_t off = 0;
            if (it.z < bz) {
                const int cx = c0[0] + it.x, cy = c0[1] + it.y, cz = c0[2] + it.z;
                const bool near = cx >= n0[0] && cx <= n1[0] && cy >= n0[1] && cy <= n1[1] &&
                                  cz >= n0[2] && cz <= n1[2];
                if (!near) {
                    off = cell_offset(gl, cx, cy, cz);
                    take = tv.P[l][off].w != 0.0f;
                }
            }
            const unsigned long long m = __ballot(take);
            if (take) {
                const uint32_t below = (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
                Q[qn + below] = ((uint32_t)l << 28) | off;
            }
            qn += (uint32_t)__popcll(m);
            if (qn >= 64) {
                __builtin_amdgcn_wave_barrier();
                expand_one(Q[lane]);
                const uint32_t rest = qn - 64;
                const uint32_t moved = lane < rest ? Q[64 + lane] : 0u;
                __builtin_amdgcn_wave_barrier();
                if (lane < rest) Q[lane] = moved;
                __builtin_amdgcn_wave_barrier();
                qn = rest;
            }
        }
#pragma unroll
        for (int a = 0; a < 3; ++a) { lo[a] = n0[a]; hi[a] = n1[a]; }
    }
    __builtin_amdgcn_wave_barrier();
    if (lane < qn) expand_one(Q[lane]);
    const float3 u = expansion_eval(E, make_float3(q.x - cb.x, q.y - cb.y, q.z - cb.z));
    if (valid) {
        const size_t o = point_offset(g, pt[0], pt[1], pt[2]);
        out[3 * o] = u.x;
        out[3 * o + 1] = u.y;
        out[3 * o + 2] = u.z;
    }
}

template <int ORDER>
__global__ __launch_bounds__(256) void k_mac_expand(const TreeView tv, vg_grid_desc g, MacParams mp,
                                                    float *__restrict__ out) {
    __shared__ uint32_t queue[4][128];
    const uint32_t wave = uni(threadIdx.x >> 6);
    const uint32_t brick = uni(blockIdx.x * 4 + wave);
    if (brick >= mp.nbricks) return;
    expand_brick<ORDER>(tv, g, mp, brick, queue[wave], out);
}

// Brick counts of a tree's own leaf layer.
__device__ __forceinline__ void tree_bricks(const vg_grid_desc &g, MacParams &p) {
    for (int a = 0; a < 3; ++a) p.nb[a] = (g.np[a] + 3) / 4;
    p.nbricks = p.nb[0] * p.nb[1] * p.nb[2];
}

template <int ORDER, int WPB>
__global__ __launch_bounds__(64 * WPB) void k_mac_expand_batch(const TreeView *__restrict__ views,
                                                               const float2 *__restrict__ mollify,
                                                               MacParams mp,
                                                               float *__restrict__ out,
                                                               size_t out_stride) {
    __shared__ uint32_t queue[WPB][128];
    const uint32_t wave = uni(threadIdx.x >> 6);
    const uint32_t brick = uni(blockIdx.x * WPB + wave);
    const uint32_t tree = blockIdx.y;
    const TreeView &tv = views[tree];
    MacParams p = mp;
    if (p.nbricks == 0) tree_bricks(tv.layer[0], p);  // trees of their own shapes
    if (brick >= p.nbricks) return;
    p.spread = mollify[tree].x;
    expand_brick<ORDER>(tv, tv.layer[0], p, brick, queue[wave], out + tree * out_stride);
}

template <int POLICY, int ORDER, int COUNT>
__global__ __launch_bounds__(256) void k_mac_grid(const TreeView tv, vg_grid_desc g, MacParams mp,
                                                  float *__restrict__ out,
                                                  unsigned long long *__restrict__ counts) {
    __shared__ WaveStage stage[4];
    const uint32_t wave = uni(threadIdx.x >> 6);
    const uint32_t brick = uni(blockIdx.x * 4 + wave);
    if (brick >= mp.nbricks) return;
    mac_brick<POLICY, ORDER, COUNT>(tv, g, mp, brick, stage[wave], out, counts);
}

// Many trees of one shape at once: blockIdx.y selects the tree (its view,
// mollification and output slab), WPB waves per block cover WPB bricks.
template <int POLICY, int ORDER, int WPB>
__global__ __launch_bounds__(64 * WPB) void k_mac_grid_batch(const TreeView *__restrict__ views,
                                                             const float2 *__restrict__ mollify,
                                                             MacParams mp, float *__restrict__ out,
                                                             size_t out_stride) {
    __shared__ WaveStage stage[WPB];
    const uint32_t wave = uni(threadIdx.x >> 6);
    const uint32_t brick = uni(blockIdx.x * WPB + wave);
    const uint32_t tree = blockIdx.y;
    const TreeView &tv = views[tree];
    MacParams p = mp;
    if (p.nbricks == 0) tree_bricks(tv.layer[0], p);  // trees of their own shapes
    if (brick >= p.nbricks) return;
    const float2 sc = mollify[tree];
    p.spread = sc.x;
    p.circ = sc.y;
    mac_brick<POLICY, ORDER, 0>(tv, tv.layer[0], p, brick, stage[wave], out + tree * out_stride,
                                nullptr);
}

// Work-queue forms for trees of different shapes: a grid of resident
// workgroups that take (tree, brick) items from a device counter until none
// is left, so every wave reaches the exit and uneven trees balance across
// the chip.  Items are numbered tree by tree in queue order (the
// largest trees first): brick_start[q] is the first item of the q-th tree
// (tree id order[q]), brick_start[trees] the total; each tree's bricks come
// from its own leaf layer.
// The walk's waves take one item at a time: its bricks are long and uneven,
// so a wave that finishes early goes on at once.
__device__ __forceinline__ uint32_t take_item(uint32_t *__restrict__ counter) {
    uint32_t item = 0;
    if ((threadIdx.x & 63) == 0) item = atomicAdd(counter, 1u);
    return uni((uint32_t)__shfl((int)item, 0, 64));
}

// The expansion's workgroups take WPB consecutive items at a time: its bricks
// are short and even, and adjacent bricks share their clusters in the CU's
// caches, as with a plain launch of WPB bricks per workgroup.  grab_items
// returns the first item, the same in every wave; every wave of the
// workgroup calls it (it holds two barriers).
template <int WPB>
__device__ __forceinline__ uint32_t grab_items(uint32_t *__restrict__ counter) {
    __shared__ uint32_t first;
    if (threadIdx.x == 0) first = atomicAdd(counter, (uint32_t)WPB);
    __syncthreads();
    const uint32_t f = uni(first);
    __syncthreads();  // read by every wave before the next grab overwrites it
    return f;
}

// Tree and brick of work item `item` (< brick_start[trees]).
__device__ __forceinline__ void item_brick(const uint32_t *__restrict__ order,
                                           const uint32_t *__restrict__ brick_start,
                                           uint32_t trees, uint32_t item, uint32_t &tree,
                                           uint32_t &brick) {
    uint32_t lo = 0, hi = trees;  // brick_start[lo] <= item < brick_start[hi]
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (brick_start[mid] <= item) lo = mid;
        else hi = mid;
    }
    tree = uni(order[lo]);
    brick = item - brick_start[lo];
}

template <int ORDER, int WPB>
__global__ __launch_bounds__(64 * WPB) void k_mac_expand_queue(
    const TreeView *__restrict__ views, const float2 *__restrict__ mollify, MacParams mp,
    float *__restrict__ out, size_t out_stride, const uint32_t *__restrict__ order,
    const uint32_t *__restrict__ brick_start, uint32_t trees, uint32_t *__restrict__ counter) {
    __shared__ uint32_t queue[WPB][128];
    const uint32_t wave = uni(threadIdx.x >> 6);
    const uint32_t total = brick_start[trees];
    for (;;) {
        const uint32_t first = grab_items<WPB>(counter);
        if (first >= total) break;  // the same in every wave of the workgroup
        const uint32_t item = first + wave;
        if (item < total) {
            uint32_t tree, brick;
            item_brick(order, brick_start, trees, item, tree, brick);
            const TreeView &tv = views[tree];
            MacParams p = mp;
            p.spread = mollify[tree].x;
            tree_bricks(tv.layer[0], p);
            expand_brick<ORDER>(tv, tv.layer[0], p, brick, queue[wave], out + tree * out_stride);
        }
    }
}

template <int POLICY, int ORDER, int WPB>
__global__ __launch_bounds__(64 * WPB) void k_mac_grid_queue(
    const TreeView *__restrict__ views, const float2 *__restrict__ mollify, MacParams mp,
    float *__restrict__ out, size_t out_stride, const uint32_t *__restrict__ order,
    const uint32_t *__restrict__ brick_start, uint32_t trees, uint32_t *__restrict__ counter) {
    __shared__ WaveStage stage[WPB];
    const uint32_t wave = uni(threadIdx.x >> 6);
    const uint32_t total = brick_start[trees];
    for (;;) {
        const uint32_t item = take_item(counter);
        if (item >= total) break;
        uint32_t tree, brick;
        item_brick(order, brick_start, trees, item, tree, brick);
        const TreeView &tv = views[tree];
        const float2 sc = mollify[tree];
        MacParams p = mp;
        p.spread = sc.x;
        p.circ = sc.y;
        tree_bricks(tv.layer[0], p);
        mac_brick<POLICY, ORDER, 0>(tv, tv.layer[0], p, brick, stage[wave],
                                    out + tree * out_stride, nullptr);
        __builtin_amdgcn_wave_barrier();
    }
}

__global__ void k_clear_counters(uint32_t *__restrict__ c) {
    if (threadIdx.x < 2) c[threadIdx.x] = 0u;
}

// Workgroups of `block` threads of kernel k that fit on the whole chip at once.
template <typename K>
vg_status resident_blocks(K k, int block, uint32_t *out) {
    int dev = 0, cus = 0, per_cu = 0;
    VG_HIP(hipGetDevice(&dev));
    VG_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    VG_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k, block, 0));
    *out = (uint32_t)((per_cu > 0 ? per_cu : 1) * (cus > 0 ? cus : 1));
    return VG_OK;
}

template <int COUNT>
vg_status run_mac(const vg_tree *t, const vg_grid_desc *g, int near_k, int order, int expand_from,
                  float spread, float circ, int policy, float *out, unsigned long long *counts,
                  hipStream_t s) {
    TreeView tv;
    VG_TRY(tree_checked_view(t, &tv));
    VG_REQUIRE(g, "grid is null");
    VG_REQUIRE(near_k >= 0 && near_k <= 16, "near_k must be in [0, 16]");
    VG_REQUIRE(order == 0 || order == 1, "order must be 0 (monopole) or 1 (dipole)");
    VG_REQUIRE(policy == VG_RSQRT_REFERENCE || policy == VG_RSQRT_ACCURATE, "bad rsqrt policy");
    for (int a = 0; a < 3; ++a)
        VG_REQUIRE(g->np[a] == tv.layer[0].np[a],
                   "grid must have the tree's leaf geometry (the grid template)");
    VG_REQUIRE(!has_orphan_cells(tv),
               "the tree's grid leaves cells without a parent cluster (a cell count that is odd "
               "and above 3 on some layer); define the grid with power-of-two cells");
    MacParams mp;
    mp.k = near_k;
    mp.spread = spread;
    mp.circ = circ;
    for (int a = 0; a < 3; ++a) mp.nb[a] = (g->np[a] + 3) / 4;
    mp.nbricks = mp.nb[0] * mp.nb[1] * mp.nb[2];
    mp.expand_from = expand_from;
    const dim3 grid(ceil_div(mp.nbricks, 4));
    const char *name = COUNT ? "vg_tree_mac_count" : "vg_tree_velocity_grid_mac";
    using K = void (*)(const TreeView, vg_grid_desc, MacParams, float *, unsigned long long *);
    K k;
    if (policy == VG_RSQRT_REFERENCE)
        k = order ? k_mac_grid<VG_RSQRT_REFERENCE, 1, COUNT> : k_mac_grid<VG_RSQRT_REFERENCE, 0, COUNT>;
    else
        k = order ? k_mac_grid<VG_RSQRT_ACCURATE, 1, COUNT> : k_mac_grid<VG_RSQRT_ACCURATE, 0, COUNT>;
    if (!COUNT && expand_from >= 1 && expand_from <= (int)tv.depth - 2) {
        // the expansion queue packs (layer << 28 | offset)
        VG_REQUIRE(tv.depth <= 17 && capacity(tv.layer[expand_from]) < (1u << 28),
                   "grid too large for local expansions");
        VG_TRY(launch("vg_tree_mac_expand", order ? k_mac_expand<1> : k_mac_expand<0>, grid,
                      dim3(256), 0, s, tv, *g, mp, out));
    }
    return launch(name, k, grid, dim3(256), 0, s, tv, *g, mp, out, counts);
}

}  // namespace

vg_status mac_velocity_grid(const vg_tree *t, const vg_grid_desc *g, int near_k, int order,
                            float spread, float circ, int policy, float *out, hipStream_t s) {
    return run_mac<0>(t, g, near_k, order, -1, spread, circ, policy, out, nullptr, s);
}

// Batched walk over `trees` trees of one shape (views and per-tree
// (spread, circ) in device memory); out holds trees slabs of out_stride
// floats.  waves_per_block in {1, 2, 4}.
vg_status mac_velocity_grid_batch(const TreeView *views, const float2 *mollify, uint32_t trees,
                                  const uint32_t np[3], int near_k, int order, int expand_from,
                                  int policy, int waves_per_block, float *out, size_t out_stride,
                                  hipStream_t s, const BatchQueue *queue, bool own_shapes) {
    VG_REQUIRE(near_k >= 0 && near_k <= 16, "near_k must be in [0, 16]");
    VG_REQUIRE(order == 0 || order == 1, "order must be 0 or 1");
    VG_REQUIRE(policy == VG_RSQRT_REFERENCE || policy == VG_RSQRT_ACCURATE, "bad rsqrt policy");
    VG_REQUIRE(waves_per_block == 1 || waves_per_block == 2 || waves_per_block == 4,
               "waves_per_block must be 1, 2 or 4");
    MacParams mp;
    mp.k = near_k;
    mp.spread = 1.0f;
    mp.circ = 1.0f;
    for (int a = 0; a < 3; ++a) mp.nb[a] = (np[a] + 3) / 4;
    mp.nbricks = mp.nb[0] * mp.nb[1] * mp.nb[2];
    mp.expand_from = expand_from;
    // the plain launch covers np's bricks; with own_shapes each tree's
    // workgroups past its own brick count leave at once
    const uint32_t launch_bricks = mp.nbricks;
    if (own_shapes) mp.nbricks = 0;
    using K = void (*)(const TreeView *, const float2 *, MacParams, float *, size_t);
    K tab[2][2][3] = {
        {{k_mac_grid_batch<0, 0, 1>, k_mac_grid_batch<0, 0, 2>, k_mac_grid_batch<0, 0, 4>},
         {k_mac_grid_batch<0, 1, 1>, k_mac_grid_batch<0, 1, 2>, k_mac_grid_batch<0, 1, 4>}},
        {{k_mac_grid_batch<1, 0, 1>, k_mac_grid_batch<1, 0, 2>, k_mac_grid_batch<1, 0, 4>},
         {k_mac_grid_batch<1, 1, 1>, k_mac_grid_batch<1, 1, 2>, k_mac_grid_batch<1, 1, 4>}}};
    const int wi = waves_per_block == 1 ? 0 : waves_per_block == 2 ? 1 : 2;
    if (queue) {
        // trees of different shapes, each within np: work-queue kernels
        using KQ = void (*)(const TreeView *, const float2 *, MacParams, float *, size_t,
                            const uint32_t *, const uint32_t *, uint32_t, uint32_t *);
        VG_TRY(launch("vg_batch_queue_clear", k_clear_counters, dim3(1), dim3(64), 0, s,
                      queue->counters));
        if (expand_from >= 1) {
            VG_REQUIRE((size_t)np[0] * np[1] * np[2] < (1u << 28),
                       "grid too large for local expansions");
            KQ te[2][3] = {{k_mac_expand_queue<0, 1>, k_mac_expand_queue<0, 2>,
                            k_mac_expand_queue<0, 4>},
                           {k_mac_expand_queue<1, 1>, k_mac_expand_queue<1, 2>,
                            k_mac_expand_queue<1, 4>}};
            uint32_t nb = 0;
            VG_TRY(resident_blocks(te[order][wi], 64 * waves_per_block, &nb));
            VG_TRY(launch("vg_batch_expand", te[order][wi], dim3(nb), dim3(64 * waves_per_block),
                          0, s, views, mollify, mp, out, out_stride, queue->order,
                          queue->brick_start, trees, queue->counters + 1));
        }
        KQ tq[2][2][3] = {
            {{k_mac_grid_queue<0, 0, 1>, k_mac_grid_queue<0, 0, 2>, k_mac_grid_queue<0, 0, 4>},
             {k_mac_grid_queue<0, 1, 1>, k_mac_grid_queue<0, 1, 2>, k_mac_grid_queue<0, 1, 4>}},
            {{k_mac_grid_queue<1, 0, 1>, k_mac_grid_queue<1, 0, 2>, k_mac_grid_queue<1, 0, 4>},
             {k_mac_grid_queue<1, 1, 1>, k_mac_grid_queue<1, 1, 2>, k_mac_grid_queue<1, 1, 4>}}};
        uint32_t nb = 0;
        VG_TRY(resident_blocks(tq[policy][order][wi], 64 * waves_per_block, &nb));
        return launch("vg_batch_velocity_grid", tq[policy][order][wi], dim3(nb),
                      dim3(64 * waves_per_block), 0, s, views, mollify, mp, out, out_stride,
                      queue->order, queue->brick_start, trees, queue->counters);
    }
    if (expand_from >= 1) {
        // trees of the batch share one shape; the walk checks the depth.
        // The expansion queue packs (layer << 28 | offset).
        VG_REQUIRE((size_t)np[0] * np[1] * np[2] < (1u << 28),
                   "grid too large for local expansions");
        using KE = void (*)(const TreeView *, const float2 *, MacParams, float *, size_t);
        KE te[2][3] = {{k_mac_expand_batch<0, 1>, k_mac_expand_batch<0, 2>, k_mac_expand_batch<0, 4>},
                       {k_mac_expand_batch<1, 1>, k_mac_expand_batch<1, 2>, k_mac_expand_batch<1, 4>}};
        VG_TRY(launch("vg_batch_expand", te[order][wi],
                      dim3(ceil_div(launch_bricks, waves_per_block), trees),
                      dim3(64 * waves_per_block), 0, s, views, mollify, mp, out, out_stride));
    }
    return launch("vg_batch_velocity_grid", tab[policy][order][wi],
                  dim3(ceil_div(launch_bricks, waves_per_block), trees), dim3(64 * waves_per_block),
                  0, s, views, mollify, mp, out, out_stride);
}
}  // namespace vg

using namespace vg;

VG_API vg_status vg_tree_velocity_grid_mac(const vg_tree *t, const vg_grid_desc *g, int near_k,
                                           int order, int expand_from, float spread, float circ,
                                           int rsqrt_policy, float *out, vg_stream s) {
    VG_REQUIRE(out, "out is null");
    return run_mac<0>(t, g, near_k, order, expand_from, spread, circ, rsqrt_policy, out, nullptr,
                      (hipStream_t)s);
}

VG_API vg_status vg_tree_mac_work(const vg_tree *t, const vg_grid_desc *g, int near_k,
                                  int expand_from, uint64_t *clusters, uint64_t *pairs,
                                  uint64_t *expansions, vg_stream stream) {
    VG_REQUIRE(clusters && pairs, "null output");
    hipStream_t s = (hipStream_t)stream;
    unsigned long long *d = nullptr;
    VG_TRY(salloc((void **)&d, 3 * sizeof(unsigned long long), s));
    vg_status st = zero_fill(d, 3 * sizeof(unsigned long long), s);
    if (st == VG_OK) st = run_mac<1>(t, g, near_k, 0, expand_from, 1.0f, 1.0f, 0, nullptr, d, s);
    unsigned long long h[3] = {0, 0, 0};
    if (st == VG_OK) {
        hipError_t e = hipMemcpyAsync(h, d, sizeof h, hipMemcpyDeviceToHost, s);
        if (e == hipSuccess) e = hipStreamSynchronize(s);
        if (e != hipSuccess) st = device_error(e, "mac work copy", __FILE__, __LINE__);
    }
    sfree(d, s);
    *clusters = h[0];
    *pairs = h[1];
    if (expansions) *expansions = h[2];
    return st;
}
