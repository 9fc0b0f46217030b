// vg_pse.hip -- viscous diffusion of vorticity by particle strength exchange
// (VortonSim::DiffuseAndDissipateVorticityPSE, vortonSim.cpp:3616-3922), on
// the partition of PartitionVortons (:3578-3607, particle.cpp:398-435),
// which is the influence tree's leaf cell lists.
//
// The reference's result depends on the order of its in-place exchanges.
// This follows its threaded build (USE_TBB, :3855-3860): every even z slice
// of cells, then every odd one; inside a slice, cells in (y, x) order,
// inside a cell vortons in index order.  Each live vorton h exchanges with
// the later vortons of its cell and then with those of 7 forward cells
// (+x, +y, +x+y, +z, +x+z, +y+z, +x+y+z; :3711-3728):
//   f = clamp(2 nu dt exp(-d^2 / (4 size_h)^2), -0.5, 0.5)
//   e = f (Omega_h - Omega_t),  Omega_h -= e,  Omega_t += e
// and then dissipates, Omega_h -= nu dt Omega_h.
//
// Schedule.  Cell (x, y) of a slice writes the vortons of cells
// {x, x+1} x {y, y+1} of that slice and the next, so two cells conflict only
// when |dx| <= 1 and |dy| <= 1.  Stepping T = x + 2y visits conflicting
// cells in the reference's (y, x) order (T grows by 1 for (+1, 0) and by
// 1..3 for (-1..+1, +1)) and never puts two of them in one step, so the
// cells of a step run in parallel and the result equals the serial
// traversal bit for bit.  Slices of one parity touch disjoint vortons
// (z, z+1), so each gets a workgroup; a barrier separates steps and a
// launch separates the phases.  A step lasts as long as its busiest wave, so
// k_pse_schedule first deals the non-empty cells of every step to the
// waves, largest first, each to the least loaded wave.
//
// A cell's exchanges are a serial chain, and the chains are what the call
// waits for: 47k systolic steps (pse_cell_chain) in 540 cells on the slowest
// slices of the two phases at 1M vortons (129^3), 16.5 ms when a step moved
// all of Omega and its index down the lanes and stored through memory, 3.4
// ms now.  So a step carries as little as it can:
//   * the exchange fraction f of a pair depends on positions and sizes only:
//     k_pse_fractions computes all of them over the whole chip beforehand, in
//     the order the steps read them, with the step's other decisions (which
//     lane exchanges, which adopts its own vorton) folded into f;
//   * f is shared by the three components of Omega, which are otherwise
//     independent: each has its own workgroup per slice (blockIdx.y);
//   * a cell's partners wait in LDS, so a step is one lane shift and one
//     exchange of one float.
// The vorton state lives in the tree's cell-sorted order (positions and
// sizes from the tree, angular velocities gathered from the caller and
// scattered back), so a cell's vortons are contiguous.  exp is vg_pse_exp,
// the same function as the oracle's.
//
// The form is chosen for the whole call: one cell of more than kChainPartners
// partners, a wavefront step of more cells than k_pse_schedule deals (flat
// grids from 513x257 cells) or 8 GB of fractions or more give it k_pse_phase,
// whose steps move all of Omega, with the fractions precomputed by rows
// (k_pse_row_fractions) or, where those fill 8 GB too, formed in the chain:
// 1M vortons with 8 cells of 320 take 20.3 ms (24.7 when one wave formed each
// cell's fractions, 28.2 with them in the chain), 8M in 700x300x8 cells 749
// (1148 in the chain).
#include <cstdlib>
#include <type_traits>

#include "vg_internal.h"

namespace vg {
vg_status tree_checked_view(const vg_tree *t, TreeView *v);

namespace {

constexpr int kPseThreads = 512;     // k_pse_phase
constexpr int kChainThreads = 1024;  // k_pse_phase_chain (512: 4.5 against 4.0 ms, with the stretching)
constexpr int kPseWaves = kPseThreads / 64, kChainWaves = kChainThreads / 64;
// Vortons of a cell and its 7 forward cells that the chain's LDS buffers hold
// (16 waves share 160 KB); 1M vortons at 129^3 have at most 442.
constexpr uint32_t kChainPartners = 2400;
// LDS floats of a wave's partner buffer besides the partners: up to 63 + 3
// before them and up to 70 after (pse_cell_chain's out and in).
constexpr uint32_t kBufFront = 68, kBufBack = 80;
constexpr size_t kLdsBytes = 160 * 1024;  // of a CU

// Cody-Waite reduction with the 16-bit split of ln 2, degree-7 Taylor
// polynomial, 2^k from the exponent bits; 0 below -87.
__device__ __forceinline__ float pse_exp(float x) {
#pragma clang fp contract(off)
    if (x != x) return x;
    if (x < -87.0f) return 0.0f;
    const float k = __builtin_rintf(x * 1.44269504f);
    const float r = (x - k * 0.693145751953125f) - k * 1.42860677e-06f;
    const float p =
        1.0f + r * (1.0f + r * (0.5f + r * (0.166666672f + r * (0.0416666679f +
        r * (0.00833333377f + r * (0.00138888892f + r * 0.000198412701f))))));
    return p * __int_as_float(((int)k + 127) << 23);
}

// Exchange fraction of the pair (here h, partner t): depends on positions
// and the here-vorton's size only.
__device__ __forceinline__ float pse_fraction(const float4 ph, float r2, const float4 pt,
                                              float nu_dt2) {
#pragma clang fp contract(off)
    const float sx = ph.x - pt.x, sy = ph.y - pt.y, sz = ph.z - pt.z;
    const float d2 = sx * sx + sy * sy + sz * sz;
    const float f = nu_dt2 * pse_exp(-d2 / r2);
    return f < -0.5f ? -0.5f : (f > 0.5f ? 0.5f : f);
}

__device__ __forceinline__ void exchange_f(float4 &wh, float4 &w, float f) {
#pragma clang fp contract(off)
    const float ex = (wh.x - w.x) * f, ey = (wh.y - w.y) * f, ez = (wh.z - w.z) * f;
    wh.x -= ex;
    wh.y -= ey;
    wh.z -= ez;
    w.x += ex;
    w.y += ey;
    w.z += ez;
}

__device__ __forceinline__ void exchange(const float4 ph, float r2, float4 &wh, const float4 pt,
                                         float4 *__restrict__ wt, float nu_dt2) {
    float4 w = *wt;
    exchange_f(wh, w, pse_fraction(ph, r2, pt, nu_dt2));
    *wt = w;
}

struct PseArgs {
    uint32_t nx, ny, nz;
    const uint32_t *start, *count;  // per leaf point (cell = its min corner)
    const float4 *p;                // sorted (x, y, z, size)
    float4 *w;                      // sorted (Omega, alive)
    float nu_dt2, dissipation;
    // k_pse_phase's exchange fractions of the systolic cells, precomputed (or
    // null): the cell with leaf point c holds frac[frac_off[c] + i n + j] for
    // here-vorton i < k and partner j < n (0 where j <= i).
    const float *frac;
    const uint32_t *frac_off;
};

__device__ __forceinline__ void pse_cell(const PseArgs &a, uint32_t x, uint32_t y, uint32_t z) {
#pragma clang fp contract(off)
    const uint32_t nx = a.nx, nxy = a.nx * a.ny;
    const uint32_t c = x + nx * y + nxy * z;
    const uint32_t fwd[7] = {1, nx, 1 + nx, nxy, 1 + nxy, nx + nxy, 1 + nx + nxy};
    const uint32_t b = a.start[c], e = b + a.count[c];
    for (uint32_t i = b; i < e; ++i) {
        float4 wh = a.w[i];
        if (wh.w == 0.f) continue;  // dead: neither initiates nor dissipates
        const float4 ph = a.p[i];
        const float range = 4.0f * ph.w;
        const float r2 = range * range;
        for (uint32_t j = i + 1; j < e; ++j) exchange(ph, r2, wh, a.p[j], a.w + j, a.nu_dt2);
#pragma unroll
        for (int k = 0; k < 7; ++k) {
            const uint32_t cn = c + fwd[k];
            const uint32_t bn = a.start[cn], en = bn + a.count[cn];
            for (uint32_t j = bn; j < en; ++j) exchange(ph, r2, wh, a.p[j], a.w + j, a.nu_dt2);
        }
        wh.x -= wh.x * a.dissipation;
        wh.y -= wh.y * a.dissipation;
        wh.z -= wh.z * a.dissipation;
        a.w[i] = wh;
    }
}

// Wave-wide form of pse_cell: the cell's partner list (its own vortons, then
// those of the 7 forward cells, in order) is held in registers, partner j in
// lane j % 64, slot j / 64.  For each live here-vorton the lanes compute the
// exchange fractions of all its partners at once (positions only), then the
// wave walks the partners in order: the running Omega_h is wave-uniform and
// each step reads one partner through readlane and selects its new value
// into the owning lane, with the same operations, in the same order, as
// pse_cell.  Cells with more than kSlots * 64 partners fall back to
// pse_cell on lane 0.
constexpr int kSlots = 9;

__device__ __forceinline__ float lane_get(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}
// The value v (wave-uniform) into lane `lane` of old.
__device__ __forceinline__ float lane_set(float v, float old, int lane) {
    return (int)(threadIdx.x & 63) == lane ? v : old;
}

// Systolic form for cells with several vortons.  Pair (i, j) needs Omega_h
// after pairs (i, j' < j) and Omega_t after pairs (i' < i, j); lane l holds
// here-vorton i = B + l while the partners stream down the lanes, one lane
// per step: partner j enters lane 0 at step j - B and meets lane l at step
// j - B + l, after lanes 0 .. l-1 have exchanged with it.  At j == i the
// incoming value is the here-vorton itself, already updated by the earlier
// here-vortons, and the lane adopts it.  Every variable sees the same
// operations in the same order as in pse_cell, with the serial chain
// shortened from k * n exchanges to k + n steps.  Here-vortons go in chunks
// of 64 lanes. Partners are read from memory in windows of 64 and leave the
// last lane back into memory, with a fence before the next chunk reads them.
constexpr uint32_t kSystolicMin = 4;

__device__ __forceinline__ uint32_t partner_index(const uint32_t base[8], const uint32_t pre[9],
                                                  uint32_t j) {
    uint32_t g = base[0] + j;
#pragma unroll
    for (int q = 1; q < 8; ++q) g = j >= pre[q] ? base[q] + (j - pre[q]) : g;
    return g;
}

// Lane l takes v from lane l - 1 and lane 0 takes `in`: the whole-wave DPP
// shift (wave_shr:1; lane 0 has no source lane and keeps the old value,
// here `in`), a register move instead of an LDS permute on the serial chain.
__device__ __forceinline__ float wave_shr(float v, float in) {
    return __int_as_float(
        __builtin_amdgcn_update_dpp(__float_as_int(in), __float_as_int(v), 0x138, 0xf, 0xf, false));
}

__device__ __forceinline__ float4 wave_shr4(float4 v, float4 in) {
    return make_float4(wave_shr(v.x, in.x), wave_shr(v.y, in.y), wave_shr(v.z, in.z),
                       wave_shr(v.w, in.w));
}

__device__ __forceinline__ float4 lane4(float4 v, int l) {
    return make_float4(lane_get(v.x, l), lane_get(v.y, l), lane_get(v.z, l), lane_get(v.w, l));
}

__device__ __forceinline__ void pse_cell_systolic(const PseArgs &a, const uint32_t base[8],
                                                  const uint32_t pre[9], uint32_t k, uint32_t n) {
#pragma clang fp contract(off)
    const int lane = (int)(threadIdx.x & 63);
    for (uint32_t B = 0; B < k; B += 64) {
        const uint32_t L = k - B < 64u ? k - B : 64u;
        const uint32_t i = B + (uint32_t)lane;
        float4 wh = make_float4(0.f, 0.f, 0.f, 0.f), ph = wh, sp = wh, sw = wh, bp = wh, bw = wh;
        float r2 = 0.f;
        bool live = false;
        const uint32_t steps = (n - B) + L - 1;
        for (uint32_t t = 0; t < steps; ++t) {
            if ((t & 63u) == 0) {  // the next 64 partners to enter, one per lane
                const uint32_t jj = B + t + (uint32_t)lane;
                if (jj < n) {
                    const uint32_t g = partner_index(base, pre, jj);
                    bp = a.p[g];
                    bw = a.w[g];
                }
            }
            sp = wave_shr4(sp, lane4(bp, (int)(t & 63u)));
            sw = wave_shr4(sw, lane4(bw, (int)(t & 63u)));
            const int jl = (int)t - lane;  // partner j - B at this lane
            const uint32_t j = B + (uint32_t)jl;
            if ((uint32_t)lane < L && jl >= 0 && j < n) {
                if (j == i) {
                    wh = sw;
                    ph = sp;
                    live = sw.w != 0.f;
                    const float range = 4.0f * ph.w;
                    r2 = range * range;
                } else if (j > i && live) {
                    exchange(ph, r2, wh, sp, &sw, a.nu_dt2);
                }
                if (j == n - 1) {  // the lane's last partner: done
                    if (live) {
                        wh.x -= wh.x * a.dissipation;
                        wh.y -= wh.y * a.dissipation;
                        wh.z -= wh.z * a.dissipation;
                    }
                    a.w[partner_index(base, pre, i)] = wh;
                }
                // a partner that is not a here-vorton of this chunk leaves
                // the last lane with its value for the next chunk
                if ((uint32_t)lane == L - 1 && j >= B + L) a.w[partner_index(base, pre, j)] = sw;
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
    }
}

// Lane l takes lane l + 1 (wrapping): the whole-wave DPP rotation
// (wave_rol:1), so the window's next partner is always in lane 0.
__device__ __forceinline__ float wave_rol(float v) {
    return __int_as_float(
        __builtin_amdgcn_update_dpp(__float_as_int(v), __float_as_int(v), 0x134, 0xf, 0xf, false));
}
__device__ __forceinline__ float4 wave_rol4(float4 v) {
    return make_float4(wave_rol(v.x), wave_rol(v.y), wave_rol(v.z), wave_rol(v.w));
}
__device__ __forceinline__ uint32_t wave_rol_u(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x134, 0xf, 0xf, false);
}
__device__ __forceinline__ uint32_t wave_shr_u(uint32_t v, uint32_t in) {
    return (uint32_t)__builtin_amdgcn_update_dpp((int)in, (int)v, 0x138, 0xf, 0xf, false);
}

// The systolic cell with its fractions read from a.frac: only Omega (and
// its vorton's index, for the write-back of partners leaving the last lane)
// streams down the lanes.  The window of 64 loaded partners rotates by one
// lane per step, so lane 0 always holds the next partner to enter; each
// lane's fractions are loaded kFracAhead steps before use (a lane walks its
// row of the fraction block left to right).
constexpr int kFracAhead = 8;

__device__ __forceinline__ void pse_cell_systolic_frac(const PseArgs &a, uint32_t c,
                                                       const uint32_t base[8],
                                                       const uint32_t pre[9], uint32_t k,
                                                       uint32_t n) {
#pragma clang fp contract(off)
    const int lane = (int)(threadIdx.x & 63);
    const float *__restrict__ fc = a.frac + a.frac_off[c];
    for (uint32_t B = 0; B < k; B += 64) {
        const uint32_t L = k - B < 64u ? k - B : 64u;
        const uint32_t i = B + (uint32_t)lane;
        const uint32_t gi = base[0] + i;  // here-vortons are the cell's own
        float4 wh = make_float4(0.f, 0.f, 0.f, 0.f), sw = wh, bw = wh;
        uint32_t sg = 0, bg = 0;
        bool live = false;
        const uint32_t steps = (n - B) + L - 1;
        // fraction of this lane at step t (0 unless it exchanges then)
        auto fetch = [&](uint32_t t) -> float {
            const int jl = (int)t - lane;
            const uint32_t j = B + (uint32_t)jl;
            return ((uint32_t)lane < L && jl > lane && j < n) ? fc[(size_t)i * n + j] : 0.f;
        };
        float cur[kFracAhead], nxt[kFracAhead];
#pragma unroll
        for (int d = 0; d < kFracAhead; ++d) cur[d] = fetch((uint32_t)d);
        for (uint32_t t0 = 0; t0 < steps; t0 += kFracAhead) {
#pragma unroll
            for (int d = 0; d < kFracAhead; ++d) nxt[d] = fetch(t0 + kFracAhead + (uint32_t)d);
#pragma unroll
            for (int d = 0; d < kFracAhead; ++d) {
                const uint32_t t = t0 + (uint32_t)d;
                if (t >= steps) break;
                if ((t & 63u) == 0) {  // the next 64 partners to enter, one per lane
                    const uint32_t jj = B + t + (uint32_t)lane;
                    if (jj < n) {
                        bg = partner_index(base, pre, jj);
                        bw = a.w[bg];
                    }
                }
                sw = wave_shr4(sw, bw);  // lane 0 takes the window's lane 0
                sg = wave_shr_u(sg, bg);
                bw = wave_rol4(bw);
                bg = wave_rol_u(bg);
                const int jl = (int)t - lane;  // partner j - B at this lane
                const uint32_t j = B + (uint32_t)jl;
                if ((uint32_t)lane < L && jl >= 0 && j < n) {
                    if (jl == lane) {  // j == i: the here-vorton itself
                        wh = sw;
                        live = sw.w != 0.f;
                    } else if (jl > lane && live) {
                        exchange_f(wh, sw, cur[d]);
                    }
                    if (j == n - 1) {  // the lane's last partner: done
                        if (live) {
                            wh.x -= wh.x * a.dissipation;
                            wh.y -= wh.y * a.dissipation;
                            wh.z -= wh.z * a.dissipation;
                        }
                        a.w[gi] = wh;
                    }
                    // a partner that is not a here-vorton of this chunk leaves
                    // the last lane with its value for the next chunk
                    if ((uint32_t)lane == L - 1 && j >= B + L) a.w[sg] = sw;
                }
            }
#pragma unroll
            for (int d = 0; d < kFracAhead; ++d) cur[d] = nxt[d];
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
    }
}

__device__ __forceinline__ void pse_cell_wave(const PseArgs &a, uint32_t x, uint32_t y, uint32_t z) {
#pragma clang fp contract(off)
    const int lane = (int)(threadIdx.x & 63);
    const uint32_t nx = a.nx, nxy = a.nx * a.ny;
    const uint32_t c = x + nx * y + nxy * z;
    const uint32_t offs[8] = {0, 1, nx, 1 + nx, nxy, 1 + nxy, nx + nxy, 1 + nx + nxy};
    uint32_t base[8], pre[9];
    pre[0] = 0;
#pragma unroll
    for (int r = 0; r < 8; ++r) {
        base[r] = a.start[c + offs[r]];
        pre[r + 1] = pre[r] + a.count[c + offs[r]];
    }
    const uint32_t k = pre[1], n = pre[8];
    if (k == 0) return;
    if (k >= kSystolicMin) {
        if (a.frac)
            pse_cell_systolic_frac(a, c, base, pre, k, n);
        else
            pse_cell_systolic(a, base, pre, k, n);
        return;
    }
    if (n > 64u * kSlots) {
        if (lane == 0) pse_cell(a, x, y, z);
        return;
    }
    float4 P[kSlots], W[kSlots];
    int G[kSlots];
#pragma unroll
    for (int s = 0; s < kSlots; ++s) {
        const uint32_t j = (uint32_t)lane + 64u * s;
        G[s] = -1;
        P[s] = W[s] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (j < n) {
            uint32_t g = base[0] + j;
#pragma unroll
            for (int q = 1; q < 8; ++q) g = j >= pre[q] ? base[q] + (j - pre[q]) : g;
            G[s] = (int)g;
            P[s] = a.p[g];
            W[s] = a.w[g];
        }
    }
    for (uint32_t i = 0; i < k; ++i) {
        const int si = (int)(i >> 6), li = (int)(i & 63);
        float4 wh = make_float4(0.f, 0.f, 0.f, 0.f), ph = wh;
#pragma unroll
        for (int s = 0; s < kSlots; ++s)
            if (s == si) {
                wh = make_float4(lane_get(W[s].x, li), lane_get(W[s].y, li), lane_get(W[s].z, li),
                                 lane_get(W[s].w, li));
                ph = make_float4(lane_get(P[s].x, li), lane_get(P[s].y, li), lane_get(P[s].z, li),
                                 lane_get(P[s].w, li));
            }
        if (wh.w == 0.f) continue;  // dead: neither initiates nor dissipates
        const float range = 4.0f * ph.w;
        const float r2 = range * range;
        float f[kSlots];
#pragma unroll
        for (int s = 0; s < kSlots; ++s) {
            const float sx = ph.x - P[s].x, sy = ph.y - P[s].y, sz = ph.z - P[s].z;
            const float d2 = sx * sx + sy * sy + sz * sz;
            float fs = a.nu_dt2 * pse_exp(-d2 / r2);
            f[s] = fs < -0.5f ? -0.5f : (fs > 0.5f ? 0.5f : fs);
        }
#pragma unroll
        for (int s = 0; s < kSlots; ++s) {
            const uint32_t j0 = 64u * s;
            const uint32_t lo = i + 1 > j0 ? i + 1 - j0 : 0;
            const uint32_t hi = n > j0 ? (n - j0 < 64u ? n - j0 : 64u) : 0;
            for (uint32_t L = lo; L < hi; ++L) {
                const int l = (int)L;
                const float fj = lane_get(f[s], l);
                const float tx = lane_get(W[s].x, l), ty = lane_get(W[s].y, l),
                            tz = lane_get(W[s].z, l);
                const float ex = (wh.x - tx) * fj, ey = (wh.y - ty) * fj, ez = (wh.z - tz) * fj;
                wh.x -= ex;
                wh.y -= ey;
                wh.z -= ez;
                W[s].x = lane_set(tx + ex, W[s].x, l);
                W[s].y = lane_set(ty + ey, W[s].y, l);
                W[s].z = lane_set(tz + ez, W[s].z, l);
            }
        }
        wh.x -= wh.x * a.dissipation;
        wh.y -= wh.y * a.dissipation;
        wh.z -= wh.z * a.dissipation;
#pragma unroll
        for (int s = 0; s < kSlots; ++s)
            if (s == si) {
                W[s].x = lane_set(wh.x, W[s].x, li);
                W[s].y = lane_set(wh.y, W[s].y, li);
                W[s].z = lane_set(wh.z, W[s].z, li);
            }
    }
#pragma unroll
    for (int s = 0; s < kSlots; ++s)
        if (G[s] >= 0) a.w[G[s]] = W[s];
}

__global__ void k_pse_zero64(unsigned long long *v) { v[threadIdx.x] = 0ull; }

// A cell's own vortons and those of its 7 forward cells, in partner order.
struct CellPartners {
    uint32_t base[8], pre[9];
};
__device__ __forceinline__ CellPartners cell_partners(const PseArgs &a, uint32_t c) {
    const uint32_t nx = a.nx, nxy = a.nx * a.ny;
    const uint32_t offs[8] = {0, 1, nx, 1 + nx, nxy, 1 + nxy, nx + nxy, 1 + nx + nxy};
    CellPartners p;
    p.pre[0] = 0;
#pragma unroll
    for (int r = 0; r < 8; ++r) {
        p.base[r] = a.start[c + offs[r]];
        p.pre[r + 1] = p.pre[r] + a.count[c + offs[r]];
    }
    return p;
}

// The vortons of slices z and z + 1: contiguous in the cell-sorted order.
struct SlicePair {
    uint32_t first, count;
};
__device__ __forceinline__ SlicePair slice_pair(const PseArgs &a, uint32_t z, uint32_t n) {
    const uint32_t nxy = a.nx * a.ny;
    const uint32_t first = a.start[z * nxy];
    return SlicePair{first, (z + 2 < a.nz ? a.start[(z + 2) * nxy] : n) - first};
}

// Systolic steps of the chunk of L here-vortons starting at B of a cell with
// n partners, in groups of four (a lane reads four fractions at a time).
__device__ __forceinline__ uint32_t chunk_groups(uint32_t n, uint32_t B, uint32_t L) {
    return ((n - B) + L - 1 + 3) / 4;
}

// Floats of a cell's fractions by rows (PseArgs::frac): those of the systolic
// cells only.
__device__ __forceinline__ unsigned long long row_fractions(uint32_t k, uint32_t n) {
    return k >= kSystolicMin ? (unsigned long long)k * n : 0ull;
}

// Fractions (floats) of each leaf point's cell in the chain's order, their
// 64-bit sum, the largest partner count, the largest number of vortons in two
// adjacent slices, and the sum by rows (totals[0..3]).  A grid-stride loop: with one workgroup per 256 points the
// two atomics of each took 157 us at 129^3.
__global__ __launch_bounds__(256) void k_pse_frac_size(PseArgs a, uint32_t cells, uint32_t n_all,
                                                       uint32_t *__restrict__ size,
                                                       unsigned long long *__restrict__ totals) {
    __shared__ unsigned long long part[256];
    __shared__ unsigned long long part_rows[256];
    __shared__ uint32_t most[256];
    unsigned long long sum = 0, rows = 0;
    uint32_t widest = 0;
    for (uint32_t c = blockIdx.x * blockDim.x + threadIdx.x; c < cells;
         c += gridDim.x * blockDim.x) {
        const uint32_t k = a.count[c];
        unsigned long long f = 0;
        if (k) {
            const uint32_t n = cell_partners(a, c).pre[8];
            for (uint32_t B = 0; B < k; B += 64) {
                const uint32_t L = k - B < 64u ? k - B : 64u;
                f += 4ull * L * chunk_groups(n, B, L);
            }
            widest = max(widest, n);
            rows += row_fractions(k, n);
        }
        size[c] = f < 0x80000000ull ? (uint32_t)f : 0x80000000u;
        sum += f;
    }
    part[threadIdx.x] = sum;
    part_rows[threadIdx.x] = rows;
    most[threadIdx.x] = widest;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) {
            part[threadIdx.x] += part[threadIdx.x + w];
            part_rows[threadIdx.x] += part_rows[threadIdx.x + w];
            most[threadIdx.x] = max(most[threadIdx.x], most[threadIdx.x + w]);
        }
        __syncthreads();
    }
    if (threadIdx.x == 0 && part[0]) {
        atomicAdd(&totals[0], part[0]);
        atomicAdd(&totals[3], part_rows[0]);
        atomicMax(&totals[1], (unsigned long long)most[0]);
    }
    if (blockIdx.x == 0) {
        uint32_t pair = 0;
        for (uint32_t z = threadIdx.x; z + 1 < a.nz; z += blockDim.x)
            pair = max(pair, slice_pair(a, z, n_all).count);
        atomicMax(&totals[2], (unsigned long long)pair);
    }
}

// The fractions' sizes by rows, and which cells have more than one wave
// computes (wide[0] of them from wide[1] on, in no order).
constexpr uint32_t kRowsPerWave = 1u << 16;
__global__ __launch_bounds__(256) void k_pse_row_size(PseArgs a, uint32_t cells,
                                                      uint32_t *__restrict__ size,
                                                      uint32_t *__restrict__ wide) {
    const uint32_t c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= cells) return;
    const uint32_t k = a.count[c];
    const uint32_t f =
        k >= kSystolicMin ? (uint32_t)row_fractions(k, cell_partners(a, c).pre[8]) : 0u;
    size[c] = f;
    if (f > kRowsPerWave) wide[1 + atomicAdd(&wide[0], 1u)] = c;
}

// A cell's fractions by rows, every `stride`th from `first` on: the same
// operations as the in-chain exchange, so the same bits.
__device__ __forceinline__ void row_fractions_of(const PseArgs &a, uint32_t c,
                                                 const CellPartners &cp, uint32_t first,
                                                 uint32_t stride, float *__restrict__ frac) {
#pragma clang fp contract(off)
    const uint32_t n = cp.pre[8], total = cp.pre[1] * n;  // (below 2^31: the sum of them is)
    float *__restrict__ fc = frac + a.frac_off[c];
    for (uint32_t q = first; q < total; q += stride) {
        const uint32_t i = q / n, j = q - i * n;
        float f = 0.f;
        if (j > i) {
            const float4 ph = a.p[cp.base[0] + i];
            const float range = 4.0f * ph.w;
            f = pse_fraction(ph, range * range, a.p[partner_index(cp.base, cp.pre, j)], a.nu_dt2);
        }
        fc[q] = f;
    }
}

// One wave per leaf point's cell, and kWideParts workgroups for the cells past
// that: with one wave for those, too, a cell of 6,000 vortons took 222 ms a
// call instead of 103.
constexpr uint32_t kWideParts = 64;
__global__ __launch_bounds__(256) void k_pse_row_fractions(PseArgs a, uint32_t cells,
                                                           float *__restrict__ frac) {
    const uint32_t c = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (c >= cells) return;
    const uint32_t k = a.count[c];
    if (k < kSystolicMin) return;
    const CellPartners cp = cell_partners(a, c);
    if (row_fractions(k, cp.pre[8]) <= kRowsPerWave)
        row_fractions_of(a, c, cp, threadIdx.x & 63, 64, frac);
}
__global__ __launch_bounds__(256) void k_pse_row_fractions_wide(PseArgs a,
                                                                const uint32_t *__restrict__ wide,
                                                                float *__restrict__ frac) {
    for (uint32_t w = blockIdx.x / kWideParts; w < wide[0]; w += gridDim.x / kWideParts) {
        const uint32_t c = wide[1 + w];
        row_fractions_of(a, c, cell_partners(a, c), blockIdx.x % kWideParts * 256 + threadIdx.x,
                         kWideParts * 256, frac);
    }
}

// What a lane does at a step of the chain: exchange with the fraction (|f|
// <= 0.5, or NaN), adopt the incoming value as its here-vorton (kAdopt: an
// exchange at f = 1 from Omega_h = -0 gives Omega_h = Omega_t exactly), or
// nothing (kSkip).
constexpr float kAdopt = 1.0f, kSkip = -1.0f;

// The fractions of every cell in the order of the chain's steps, one wave
// per leaf point's cell: chunk by chunk, four steps of lane 0, of lane 1, ...
// The same operations as the in-chain exchange, so the same bits.
__global__ __launch_bounds__(256) void k_pse_fractions(PseArgs a, uint32_t cells,
                                                       const float *__restrict__ alive,
                                                       const uint32_t *__restrict__ frac_off,
                                                       float *__restrict__ frac) {
#pragma clang fp contract(off)
    const uint32_t c = blockIdx.x * 4 + (threadIdx.x >> 6);
    const uint32_t lane = threadIdx.x & 63;
    if (c >= cells) return;
    const uint32_t k = a.count[c];
    if (k == 0) return;
    const CellPartners cp = cell_partners(a, c);
    const uint32_t n = cp.pre[8];
    float *__restrict__ fc = frac + frac_off[c];
    for (uint32_t B = 0; B < k; B += 64) {
        const uint32_t L = k - B < 64u ? k - B : 64u;
        const uint32_t total = 4 * L * chunk_groups(n, B, L);
        for (uint32_t q = lane; q < total; q += 64) {
            const uint32_t g = q / (4 * L), r = q - g * (4 * L);
            const uint32_t l = r >> 2, t = 4 * g + (r & 3u);
            const uint32_t i = B + l, j = B + t - l;
            float f = kSkip;
            if (t >= l && j < n) {
                if (j == i) {
                    f = kAdopt;
                } else if (j > i && alive[cp.base[0] + i] != 0.f) {
                    const float4 ph = a.p[cp.base[0] + i];
                    const float range = 4.0f * ph.w;
                    f = pse_fraction(ph, range * range, a.p[partner_index(cp.base, cp.pre, j)],
                                     a.nu_dt2);
                }
            }
            fc[q] = f;
        }
        fc += total;
    }
}

// Groups of four steps whose fractions a lane holds ahead of their use
// (4, 6 and 8 groups: 3.88, 3.90 and 4.00 ms for the vorticity update, this
// call and the stretching, at 1M vortons).
constexpr int kRing = 4;

// A cell as the chain takes it: its partners and its fractions.
struct ChainCell {
    CellPartners cp;
    const float4 *F;
};
// What it is made of, one load for the wave: lanes 0-7 hold the cell's and
// its forward cells' starts, lanes 8-15 their counts, the others the offset
// of its fractions.  (Loaded one by one, each value waited for the one
// before it and for the fractions in flight.)
__device__ __forceinline__ uint32_t chain_cell_load(const PseArgs &a, uint32_t c,
                                                    const uint32_t *__restrict__ frac_off,
                                                    uint32_t lane) {
    const uint32_t at = c + (lane & 1u) + ((lane & 2u) ? a.nx : 0u) +
                        ((lane & 4u) ? a.nx * a.ny : 0u);
    const uint32_t *src = lane < 8u ? a.start + at : lane < 16u ? a.count + at : frac_off + c;
    return *src;
}
__device__ __forceinline__ ChainCell chain_cell(uint32_t v, const float *__restrict__ frac) {
    ChainCell cell;
    cell.cp.pre[0] = 0;
#pragma unroll
    for (int r = 0; r < 8; ++r) {
        cell.cp.base[r] = (uint32_t)__builtin_amdgcn_readlane((int)v, r);
        cell.cp.pre[r + 1] = cell.cp.pre[r] + (uint32_t)__builtin_amdgcn_readlane((int)v, 8 + r);
    }
    cell.F = reinterpret_cast<const float4 *>(
        frac + (uint32_t)__builtin_amdgcn_readlane((int)v, 16));
    return cell;
}

// What a lane holds of a chunk before its first step: whether its
// here-vorton is alive, and the fractions of the first kRing groups.
struct ChainLead {
    float live;
    float4 q[kRing];
};
__device__ __forceinline__ void lead_load(ChainLead &lead, const ChainCell &cell, const float4 *F,
                                          uint32_t B, const float *__restrict__ alive,
                                          uint32_t lane) {
    const uint32_t k = cell.cp.pre[1], L = k - B < 64u ? k - B : 64u;
    const uint32_t last = chunk_groups(cell.cp.pre[8], B, L) - 1, ll = lane < L ? lane : L - 1;
    lead.live = alive[cell.cp.base[0] + B + ll];
#pragma unroll
    for (uint32_t r = 0; r < kRing; ++r) lead.q[r] = F[min(r, last) * L + ll];
}

__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// One component of Omega of one cell, by one wave: the systolic form (see
// pse_cell_systolic) with the fractions precomputed.  The partners' values
// wait in LDS (buf[0, n), filled by the caller); partner j of a chunk
// starting at B enters lane 0 at step j - B, moves up one lane per step, and
// leaves lane L - 1 back into buf, where the next chunk, or the write-back at
// the end, finds it.  lead is the first chunk's; w is where the vortons'
// values live, by index in the cell-sorted order.
// The loops run at least once and load on every path, so that the compiler
// can count the loads in flight and wait for the one it needs: with loads
// behind a branch every group waited for the newest of them (5.4 against 3.1
// ms for the two phases at 1M vortons).
__device__ __forceinline__ void pse_cell_chain(const PseArgs &a, const ChainCell &cell,
                                               ChainLead &lead,
                                               const float *__restrict__ alive, float *w,
                                               float *buf) {
#pragma clang fp contract(off)
    const uint32_t lane = threadIdx.x & 63;
    const CellPartners &cp = cell.cp;
    const uint32_t k = cp.pre[1], n = cp.pre[8];
    const float4 *F = cell.F;
    float4 (&q)[kRing] = lead.q;
    uint32_t B = 0;
    do {
        const uint32_t L = k - B < 64u ? k - B : 64u;
        const uint32_t groups = chunk_groups(n, B, L);
        // lanes past the last follow it (they receive what leaves it)
        const uint32_t ll = lane < L ? lane : L - 1;
        const bool leaves = lane == L - 1;
        float wh = -0.f, sw = 0.f;
        float4 in = *reinterpret_cast<const float4 *>(buf + B);
        float *out = buf + B - (L - 1);  // of the value leaving at step 0
        // DEAD: the chunk has dead here-vortons, and what passes them keeps its
        // bits, the sign of a zero among them.  Where all are alive a skipped
        // value is read no more, and one select instead of two does (3.97
        // against 3.88 ms a vorticity update at 1M vortons).
        auto steps = [&](auto DEAD) {
            uint32_t g0 = 0;
            do {
#pragma unroll
                for (uint32_t r = 0; r < kRing; ++r) {
                    const uint32_t g = g0 + r;
                    if (g < groups) {
                        const float f[4] = {q[r].x, q[r].y, q[r].z, q[r].w};
                        const float v[4] = {in.x, in.y, in.z, in.w};
                        in = *reinterpret_cast<const float4 *>(buf + B + 4 * (g + 1));
                        float o[4];
#pragma unroll
                        for (int d = 0; d < 4; ++d) {
                            sw = wave_shr(sw, v[d]);  // lane 0 takes the next partner
                            const float e = (wh - sw) * f[d];
                            const bool go = f[d] != kSkip;
                            if (DEAD) {
                                wh = go ? wh - e : wh;
                                sw = go ? sw + e : sw;
                            } else {
                                const float ex = go ? e : 0.f;
                                wh -= ex;
                                sw += ex;
                            }
                            o[d] = sw;
                        }
                        // values below B belong to steps before the first partner
                        // has passed; their places in buf are no longer read
                        if (4 * g + 3 >= L - 1 && leaves) {
#pragma unroll
                            for (int d = 0; d < 4; ++d) out[4 * g + d] = o[d];
                        }
                    }
                    q[r] = F[min(g + kRing, groups - 1) * L + ll];
                }
                g0 += kRing;
            } while (g0 < groups);
        };
        if (__ballot(lead.live == 0.f))
            steps(std::true_type());
        else
            steps(std::false_type());
        F += groups * L;
        if (lead.live != 0.f) wh -= wh * a.dissipation;
        if (lane < L) w[cp.base[0] + B + lane] = wh;
        B += 64;
        if (B < k) lead_load(lead, cell, F, B, alive, lane);
    } while (B < k);
    wave_lds_fence();
    for (uint32_t j = k + lane; j < n; j += 64) w[partner_index(cp.base, cp.pre, j)] = buf[j];
}

// Cells of wavefront step t of a slice: x + 2y = t, y from
// max(0, ceil((t - cx + 1) / 2)) to min(cy - 1, t / 2).
__device__ __forceinline__ void step_rows(int t, int cx, int cy, int &ylo, int &yhi) {
    ylo = t - (cx - 1) > 0 ? (t - (cx - 1) + 1) / 2 : 0;
    yhi = t / 2 < cy - 1 ? t / 2 : cy - 1;
}

// Work of a cell in steps of pse_cell_wave: the partner stream of each chunk
// of 64 here-vortons in the systolic form, k n in the small-cell form; 0 for
// an empty cell (nothing to do), at least 1 otherwise.  The chain form
// (CHAIN) is systolic throughout and pays about 24 steps' time per cell for
// its loads and stores.
template <bool CHAIN>
__device__ __forceinline__ uint32_t cell_cost(const PseArgs &a, uint32_t c) {
    const uint32_t k = a.count[c];
    if (k == 0) return 0u;
    const uint32_t n = cell_partners(a, c).pre[8];
    uint64_t cost = CHAIN ? 24 : 0;
    if (!CHAIN && k < kSystolicMin) {
        cost = (uint64_t)k * n;
    } else {
        for (uint32_t b = 0; b < k; b += 64) cost += (n - b) + (k - b < 64u ? k - b : 64u) - 1;
    }
    // a non-empty cell must never look empty: at least 1, saturated
    return cost == 0 ? 1u : (cost > 0xffffffffull ? 0xffffffffu : (uint32_t)cost);
}

// Cells of one wavefront step share no vortons, so any assignment of them to
// the waves gives the same result; the step lasts as long as the busiest
// wave.  One wave per (step t, slice z) assigns the step's non-empty cells,
// largest first, each to the wave with the least work so far (greedy LPT),
// and writes them grouped by wave: perm[sched * M + i] for i in
// [wstart[(WAVES + 1) sched + w], wstart[(WAVES + 1) sched + w + 1]), sched =
// z steps + t.  Up to kSchedSlots * 64 cells per step.
constexpr int kSchedSlots = 4;

template <int WAVES, bool CHAIN>
__global__ __launch_bounds__(64) void k_pse_schedule(PseArgs a, uint32_t steps, uint32_t M,
                                                     uint32_t *__restrict__ perm,
                                                     uint32_t *__restrict__ wstart) {
    const int t = (int)blockIdx.x;
    const uint32_t z = blockIdx.y;
    const int lane = (int)threadIdx.x;
    const int cx = (int)a.nx - 1, cy = (int)a.ny - 1;
    int ylo, yhi;
    step_rows(t, cx, cy, ylo, yhi);
    const uint32_t nx = a.nx, nxy = a.nx * a.ny;
    uint32_t rem[kSchedSlots];  // cost still to assign (0 once assigned or empty)
    int slot_w[kSchedSlots], slot_pos[kSchedSlots];
#pragma unroll
    for (int q = 0; q < kSchedSlots; ++q) {
        const int y = ylo + lane + 64 * q;
        rem[q] = y <= yhi ? cell_cost<CHAIN>(a, (uint32_t)(t - 2 * y) + nx * (uint32_t)y + nxy * z) : 0u;
        slot_w[q] = -1;
        slot_pos[q] = 0;
    }
    uint32_t load[WAVES], cnt[WAVES];
#pragma unroll
    for (int w = 0; w < WAVES; ++w) load[w] = cnt[w] = 0u;
    for (;;) {
        uint32_t best = rem[0];
#pragma unroll
        for (int q = 1; q < kSchedSlots; ++q) best = rem[q] > best ? rem[q] : best;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            const uint32_t o = (uint32_t)__shfl_xor((int)best, off, 64);
            best = o > best ? o : best;
        }
        best = __builtin_amdgcn_readfirstlane(best);
        if (best == 0u) break;
        // the first (slot, lane) holding it, and the least loaded wave
        int sel_q = 0, sel_lane = 0;
#pragma unroll
        for (int q = kSchedSlots - 1; q >= 0; --q) {
            const unsigned long long m = __ballot(rem[q] == best);
            if (m) {
                sel_q = q;
                sel_lane = (int)__builtin_ctzll(m);
            }
        }
        int w = 0;
#pragma unroll
        for (int v = 1; v < WAVES; ++v) w = load[v] < load[w] ? v : w;
        uint32_t pos = 0;
#pragma unroll
        for (int v = 0; v < WAVES; ++v) {
            if (v == w) {
                pos = cnt[v];
                cnt[v] += 1u;
                load[v] += best;
            }
        }
#pragma unroll
        for (int q = 0; q < kSchedSlots; ++q) {
            if (q == sel_q && lane == sel_lane) {
                slot_w[q] = w;
                slot_pos[q] = (int)pos;
                rem[q] = 0u;
            }
        }
    }
    uint32_t ws[WAVES + 1];
    ws[0] = 0;
#pragma unroll
    for (int v = 0; v < WAVES; ++v) ws[v + 1] = ws[v] + cnt[v];
    const size_t sched = (size_t)z * steps + (size_t)t;
    if (lane <= WAVES) {
        uint32_t v = 0;
#pragma unroll
        for (int u = 0; u <= WAVES; ++u) v = lane == u ? ws[u] : v;
        wstart[(WAVES + 1) * sched + (size_t)lane] = v;
    }
#pragma unroll
    for (int q = 0; q < kSchedSlots; ++q) {
        if (slot_w[q] >= 0) {
            uint32_t base = 0;
#pragma unroll
            for (int u = 0; u < WAVES; ++u) base = slot_w[q] == u ? ws[u] : base;
            perm[sched * M + base + (uint32_t)slot_pos[q]] = (uint32_t)(ylo + lane + 64 * q);
        }
    }
}

// The schedule as one list per slice and wave: cells (step << 16 | y) in step
// order, list[z steps M + lstart[(kChainWaves + 1) z + w] ...].
__global__ __launch_bounds__(kChainThreads) void k_pse_lists(uint32_t steps, uint32_t M,
                                                             const uint32_t *__restrict__ perm,
                                                             const uint32_t *__restrict__ wstart,
                                                             uint32_t *__restrict__ list,
                                                             uint32_t *__restrict__ lstart) {
    __shared__ uint32_t total[kChainWaves];
    const uint32_t z = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    auto cells = [&](uint32_t t, uint32_t &b, uint32_t &e) {
        const size_t at = (kChainWaves + 1) * ((size_t)z * steps + t) + wave;
        b = wstart[at];
        e = wstart[at + 1];
    };
    uint32_t sum = 0, b, e;
    for (uint32_t t = lane; t < steps; t += 64) {
        cells(t, b, e);
        sum += e - b;
    }
    for (int off = 32; off > 0; off >>= 1) sum += (uint32_t)__shfl_xor((int)sum, off, 64);
    if (lane == 0) total[wave] = sum;
    __syncthreads();
    uint32_t at = 0;
    for (uint32_t v = 0; v < wave; ++v) at += total[v];
    if (lane == 0) {
        lstart[(kChainWaves + 1) * z + wave] = at;
        if (wave + 1 == kChainWaves) lstart[(kChainWaves + 1) * z + kChainWaves] = at + sum;
    }
    const size_t region = (size_t)z * steps * M;
    for (uint32_t t0 = 0; t0 < steps; t0 += 64) {
        const uint32_t t = t0 + lane;
        b = e = 0;
        if (t < steps) cells(t, b, e);
        uint32_t incl = e - b;
        for (int off = 1; off < 64; off <<= 1) {
            const uint32_t o = (uint32_t)__shfl_up((int)incl, off, 64);
            if ((int)lane >= off) incl += o;
        }
        uint32_t p = at + incl - (e - b);
        for (uint32_t i = b; i < e; ++i)
            list[region + p++] = (t << 16) | perm[((size_t)z * steps + t) * M + i];
        at += (uint32_t)__shfl((int)incl, 63, 64);
    }
}

// One component (blockIdx.y) of one slice z = phase + 2 blockIdx.x: every wave
// goes through its list of cells, with a workgroup barrier between wavefront
// steps.  What a cell needs besides Omega does not change during the call,
// so the next cell's partners and first fractions are fetched while the
// current one runs.
// RESIDENT: the component of both slices' vortons stays in LDS for the whole
// phase (`buf_floats` per wave, then the values), so a step waits for no
// global load or store: 3.88 against 4.10 ms for the vorticity update at 1M
// vortons.
// Otherwise (slices too full for the LDS) they stay in w3.
template <bool RESIDENT>
__global__ __launch_bounds__(kChainThreads) void k_pse_phase_chain(
    PseArgs a, uint32_t phase, uint32_t steps, uint32_t M, const uint32_t *__restrict__ list,
    const uint32_t *__restrict__ lstart, const float *__restrict__ frac,
    const uint32_t *__restrict__ frac_off, const float *__restrict__ alive, float *w3, uint32_t n,
    uint32_t buf_floats) {
    extern __shared__ __align__(16) float lds[];
    const uint32_t z = phase + 2 * blockIdx.x;
    if (z + 1 >= a.nz) return;  // uniform per workgroup
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    float *global = w3 + (size_t)blockIdx.y * n;
    float *buf = lds + wave * buf_floats + kBufFront;
    const SlicePair pair = slice_pair(a, z, n);
    float *resident = lds + kChainWaves * buf_floats;
    float *w = RESIDENT ? resident - pair.first : global;
    if (RESIDENT) {
        for (uint32_t i = threadIdx.x; i < pair.count; i += kChainThreads)
            resident[i] = global[pair.first + i];
        __syncthreads();
    }
    auto next_step = [&] {
        // LDS is all that the waves share: nothing waits for the fractions
        // in flight
        if (RESIDENT)
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        else
            __syncthreads();
    };
    const uint32_t *cells = list + (size_t)z * steps * M;
    uint32_t p = __builtin_amdgcn_readfirstlane(lstart[(kChainWaves + 1) * z + wave]);
    const uint32_t end =
        __builtin_amdgcn_readfirstlane(lstart[(kChainWaves + 1) * z + wave + 1]);
    // the list's last cell stands in for those after it
    auto entry_at = [&](uint32_t i) {
        return __builtin_amdgcn_readfirstlane(cells[min(i, end - 1)]);
    };
    auto load = [&](uint32_t entry) {
        const uint32_t t = entry >> 16, y = entry & 0xffffu;
        return chain_cell_load(a, (t - 2 * y) + a.nx * (y + a.ny * z), frac_off, lane);
    };
    uint32_t now = 0;  // barriers passed: the current wavefront step
    if (p < end) {
        uint32_t entry = entry_at(p), entry1 = entry_at(p + 1), entry2 = cells[min(p + 2, end - 1)];
        ChainCell cell = chain_cell(load(entry), frac);
        uint32_t v1 = load(entry1);
        ChainLead lead, lead1;
        lead_load(lead, cell, cell.F, 0, alive, lane);
        for (; p < end; ++p) {
            const ChainCell cell1 = chain_cell(v1, frac);
            const uint32_t e2 = __builtin_amdgcn_readfirstlane(entry2);
            v1 = load(e2);
            entry2 = cells[min(p + 3, end - 1)];
            lead_load(lead1, cell1, cell1.F, 0, alive, lane);
            for (; now < (entry >> 16); ++now) next_step();
            const uint32_t np = cell.cp.pre[8];
            for (uint32_t j0 = 0; j0 < np; j0 += 256) {
                float v[4];
#pragma unroll
                for (uint32_t r = 0; r < 4; ++r) {
                    const uint32_t j = j0 + 64 * r + lane;
                    if (j < np) v[r] = w[partner_index(cell.cp.base, cell.cp.pre, j)];
                }
#pragma unroll
                for (uint32_t r = 0; r < 4; ++r) {
                    const uint32_t j = j0 + 64 * r + lane;
                    if (j < np) buf[j] = v[r];
                }
            }
            wave_lds_fence();
            pse_cell_chain(a, cell, lead, alive, w, buf);
            lead = lead1;
            cell = cell1;
            entry = entry1;
            entry1 = e2;
        }
    }
    for (; now < steps; ++now) next_step();
    if (RESIDENT)
        for (uint32_t i = threadIdx.x; i < pair.count; i += kChainThreads)
            global[pair.first + i] = resident[i];
}

// perm / wstart: the schedule of k_pse_schedule, or null for round robin by
// row (steps of more than kSchedSlots * 64 cells).
__global__ __launch_bounds__(kPseThreads) void k_pse_phase(PseArgs a, uint32_t phase,
                                                           const uint32_t *__restrict__ perm,
                                                           const uint32_t *__restrict__ wstart,
                                                           uint32_t M) {
    const uint32_t z = phase + 2 * blockIdx.x;
    if (z + 1 >= a.nz) return;  // uniform per workgroup
    const int wave = (int)(threadIdx.x >> 6);
    const int cx = (int)a.nx - 1, cy = (int)a.ny - 1;  // cells per axis
    const int steps = (cx - 1) + 2 * (cy - 1) + 1;
    for (int t = 0; t < steps; ++t) {
        int ylo, yhi;
        step_rows(t, cx, cy, ylo, yhi);
        if (perm) {
            const size_t sched = (size_t)z * (size_t)steps + (size_t)t;
            const uint32_t b = wstart[(kPseWaves + 1) * sched + (size_t)wave];
            const uint32_t e = wstart[(kPseWaves + 1) * sched + (size_t)wave + 1];
            for (uint32_t i = b; i < e; ++i) {
                const int y = (int)perm[sched * M + i];
                pse_cell_wave(a, (uint32_t)(t - 2 * y), (uint32_t)y, z);
            }
        } else {
            for (int y = ylo + wave; y <= yhi; y += kPseWaves)
                pse_cell_wave(a, (uint32_t)(t - 2 * y), (uint32_t)y, z);
        }
        __syncthreads();
    }
}

// Simultaneous exchange (no reference counterpart): one thread per vorton
// in cell-sorted order, every exchange from the starting values w0, summed
// in the order of vgo_pse_diffuse_simultaneous: received from the live
// vortons of the 7 backward cells, from the live earlier vortons of the own
// cell, then (if alive) given to the later vortons of the own cell and the
// vortons of the 7 forward cells.
__device__ __forceinline__ void pse_pair(const float4 ph, float r2h, const float4 wh,
                                         const float4 pt, const float4 wt, float nu_dt2,
                                         float &ex, float &ey, float &ez) {
#pragma clang fp contract(off)
    const float sx = ph.x - pt.x, sy = ph.y - pt.y, sz = ph.z - pt.z;
    const float d2 = sx * sx + sy * sy + sz * sz;
    float f = nu_dt2 * pse_exp(-d2 / r2h);
    f = f < -0.5f ? -0.5f : (f > 0.5f ? 0.5f : f);
    ex = (wh.x - wt.x) * f;
    ey = (wh.y - wt.y) * f;
    ez = (wh.z - wt.z) * f;
}

__global__ void k_pse_simultaneous(PseArgs a, const vg_grid_desc g, const float4 *__restrict__ w0,
                                   float4 *__restrict__ w1, uint32_t n) {
#pragma clang fp contract(off)
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float4 pi = a.p[i], wi = w0[i];
    const int ix = cell_of(pi.x, g.min[0], g.cpe[0], (int)g.np[0] - 1);
    const int iy = cell_of(pi.y, g.min[1], g.cpe[1], (int)g.np[1] - 1);
    const int iz = cell_of(pi.z, g.min[2], g.cpe[2], (int)g.np[2] - 1);
    const uint32_t nx = a.nx, nxy = a.nx * a.ny;
    const uint32_t c = (uint32_t)ix + nx * (uint32_t)iy + nxy * (uint32_t)iz;
    const int d[7][3] = {{1, 0, 0}, {0, 1, 0}, {1, 1, 0}, {0, 0, 1}, {1, 0, 1}, {0, 1, 1}, {1, 1, 1}};
    float ax = 0.f, ay = 0.f, az = 0.f, ex, ey, ez;
#pragma unroll
    for (int k = 0; k < 7; ++k) {
        if (ix < d[k][0] || iy < d[k][1] || iz < d[k][2]) continue;
        const uint32_t cb = c - ((uint32_t)d[k][0] + nx * d[k][1] + nxy * d[k][2]);
        const uint32_t b = a.start[cb], e = b + a.count[cb];
        for (uint32_t j = b; j < e; ++j) {
            const float4 wh = w0[j];
            if (wh.w == 0.f) continue;
            const float4 ph = a.p[j];
            const float sh = 4.0f * ph.w;
            pse_pair(ph, sh * sh, wh, pi, wi, a.nu_dt2, ex, ey, ez);
            ax += ex;
            ay += ey;
            az += ez;
        }
    }
    const uint32_t b = a.start[c], e = b + a.count[c];
    for (uint32_t j = b; j < i; ++j) {
        const float4 wh = w0[j];
        if (wh.w == 0.f) continue;
        const float4 ph = a.p[j];
        const float sh = 4.0f * ph.w;
        pse_pair(ph, sh * sh, wh, pi, wi, a.nu_dt2, ex, ey, ez);
        ax += ex;
        ay += ey;
        az += ez;
    }
    const bool live = wi.w != 0.f;
    if (live) {
        const float si = 4.0f * pi.w;
        const float r2 = si * si;
        for (uint32_t j = i + 1; j < e; ++j) {
            pse_pair(pi, r2, wi, a.p[j], w0[j], a.nu_dt2, ex, ey, ez);
            ax -= ex;
            ay -= ey;
            az -= ez;
        }
#pragma unroll
        for (int k = 0; k < 7; ++k) {
            const uint32_t cf = c + ((uint32_t)d[k][0] + nx * d[k][1] + nxy * d[k][2]);
            const uint32_t bf = a.start[cf], ef = bf + a.count[cf];
            for (uint32_t j = bf; j < ef; ++j) {
                pse_pair(pi, r2, wi, a.p[j], w0[j], a.nu_dt2, ex, ey, ez);
                ax -= ex;
                ay -= ey;
                az -= ez;
            }
        }
    }
    float4 o = make_float4(wi.x + ax, wi.y + ay, wi.z + az, wi.w);
    if (live) {
        o.x -= o.x * a.dissipation;
        o.y -= o.y * a.dissipation;
        o.z -= o.z * a.dissipation;
    }
    w1[i] = o;
}

__global__ void k_pse_gather(const uint32_t *__restrict__ idx, const float *__restrict__ angvel,
                             size_t ang_stride, const int32_t *__restrict__ birth,
                             size_t birth_stride, size_t n, float4 *__restrict__ w) {
    const size_t j = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    const size_t i = idx[j];
    const float *o = angvel + i * ang_stride;
    const bool alive = birth ? birth[i * birth_stride] >= 0 : true;
    w[j] = make_float4(o[0], o[1], o[2], alive ? 1.f : 0.f);
}

__global__ void k_pse_scatter(const uint32_t *__restrict__ idx, const float4 *__restrict__ w,
                              size_t n, float *__restrict__ angvel, size_t ang_stride) {
    const size_t j = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    float *o = angvel + (size_t)idx[j] * ang_stride;
    const float4 v = w[j];
    o[0] = v.x;
    o[1] = v.y;
    o[2] = v.z;
}

// One array per component, and which vortons are alive.
__global__ void k_pse_gather3(const uint32_t *__restrict__ idx, const float *__restrict__ angvel,
                              size_t ang_stride, const int32_t *__restrict__ birth,
                              size_t birth_stride, size_t n, float *__restrict__ w3,
                              float *__restrict__ alive) {
    const size_t j = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    const size_t i = idx[j];
    const float *o = angvel + i * ang_stride;
    w3[j] = o[0];
    w3[n + j] = o[1];
    w3[2 * n + j] = o[2];
    alive[j] = !birth || birth[i * birth_stride] >= 0 ? 1.f : 0.f;
}

__global__ void k_pse_scatter3(const uint32_t *__restrict__ idx, const float *__restrict__ w3,
                               size_t n, float *__restrict__ angvel, size_t ang_stride) {
    const size_t j = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    float *o = angvel + (size_t)idx[j] * ang_stride;
    o[0] = w3[j];
    o[1] = w3[n + j];
    o[2] = w3[2 * n + j];
}

}  // namespace

vg_status pse_diffuse(const vg_tree *t, float *angvel, size_t ang_stride, const int32_t *birth,
                      size_t birth_stride, float viscosity, float dt, int order, hipStream_t s) {
    TreeView tv;
    VG_TRY(tree_checked_view(t, &tv));
    const size_t n = tv.n;
    if (n == 0) return VG_OK;
    const vg_grid_desc &g = tv.layer[0];
    VG_REQUIRE(g.np[0] >= 2 && g.np[1] >= 2 && g.np[2] >= 2, "leaf grid is degenerate");
    VG_REQUIRE(capacity(g) < (size_t(1) << 32), "leaf grid has 2^32 points or more");
    VG_REQUIRE(order == VG_PSE_REFERENCE_ORDER || order == VG_PSE_SIMULTANEOUS, "bad PSE order");
    const bool sim = order == VG_PSE_SIMULTANEOUS;
    float4 *w = nullptr;
    VG_TRY(salloc((void **)&w, (sim ? 2 : 1) * n * sizeof(float4), s));
    PseArgs a;
    a.nx = g.np[0];
    a.ny = g.np[1];
    a.nz = g.np[2];
    a.start = tv.cell_start;
    a.count = tv.cell_count;
    a.p = tv.sorted_p;
    a.w = w;
    a.nu_dt2 = 2.0f * viscosity * dt;   // 2.0f * mViscosity * timeStep
    a.dissipation = viscosity * dt;     // mViscosity * timeStep
    a.frac = nullptr;
    a.frac_off = nullptr;
    if (sim) {
        vg_status st = launch("vg_pse_gather", k_pse_gather, dim3(ceil_div(n, 256)), dim3(256), 0,
                              s, tv.sorted_idx, (const float *)angvel, ang_stride, birth,
                              birth_stride, n, w);
        if (st == VG_OK)
            st = launch("vg_pse_simultaneous", k_pse_simultaneous, dim3(ceil_div(n, 256)),
                        dim3(256), 0, s, a, g, (const float4 *)w, w + n, (uint32_t)n);
        if (st == VG_OK)
            st = launch("vg_pse_scatter", k_pse_scatter, dim3(ceil_div(n, 256)), dim3(256), 0, s,
                        tv.sorted_idx, (const float4 *)(w + n), n, angvel, ang_stride);
        sfree(w, s);
        return st;
    }
    const uint32_t slices = a.nz - 1;  // cell slices 0 .. nz-2
    const uint32_t cx = a.nx - 1, cy = a.ny - 1;
    const uint32_t steps = (cx - 1) + 2 * (cy - 1) + 1;
    // cells per wavefront step are at most min(cy, (cx + 1) / 2)
    const uint32_t M = cy < (cx + 1) / 2 ? cy : (cx + 1) / 2;
    const size_t nsched = (size_t)slices * steps, cells = capacity(g);
    // (An allocation and its release are 8 us of the host's: what is needed at
    // one time is one.  100 vortons in 16x16x16 cells: 227 us a call with ten
    // allocations, 105 with four.)
    uint32_t *sizes = nullptr, *sched = nullptr, *wide = nullptr;
    float *frac = nullptr;
    // The fractions' sizes are read back to size their buffer: one stream
    // synchronisation.
    constexpr size_t kTotals = 4;
    vg_status st = salloc((void **)&sizes,
                          kTotals * sizeof(unsigned long long) +
                              (2 * cells + scan_scratch_elems(cells)) * sizeof(uint32_t),
                          s);
    unsigned long long *dtot = reinterpret_cast<unsigned long long *>(sizes);
    uint32_t *fsize = reinterpret_cast<uint32_t *>(dtot + kTotals), *foff = fsize + cells,
             *stmp = foff + cells;
    if (st == VG_OK) st = launch("vg_pse_frac_size", k_pse_zero64, dim3(1), dim3(kTotals), 0, s,
                                  dtot);
    if (st == VG_OK)
        st = launch("vg_pse_frac_size", k_pse_frac_size,
                    dim3(min(ceil_div(cells, 256), 1024u)), dim3(256), 0, s, a, (uint32_t)cells,
                    (uint32_t)n, fsize, dtot);
    if (st == VG_OK) st = exclusive_scan_u32(fsize, foff, cells, stmp, s);
    unsigned long long totals[kTotals] = {0, 0, 0, 0};
    if (st == VG_OK) {
        hipError_t e = hipMemcpyAsync(totals, dtot, sizeof totals, hipMemcpyDeviceToHost, s);
        if (e == hipSuccess) e = hipStreamSynchronize(s);
        if (e != hipSuccess) {
            set_error(std::string("PSE fraction sizes: ") + hipGetErrorString(e));
            st = VG_EDEVICE;
        }
    }
    // One cell whose partners do not fit a wave's LDS, a wavefront step of more
    // cells than the schedule deals, or 2^31 floats of fractions or more keep
    // the whole call in the form without the chain; it reads its fractions by
    // rows, unless those are 2^31 floats or more, too.  VG_PSE_FRACTIONS=0 in
    // the environment keeps them in the serial exchange (the same bits any
    // way; the switch keeps that path testable).
    const char *env = getenv("VG_PSE_FRACTIONS");
    const bool precompute = !(env && env[0] == '0');
    const bool scheduled = M <= 64u * kSchedSlots && nsched * M < (size_t(1) << 28);
    const bool chain = precompute && totals[0] > 0 && totals[0] < (1ull << 31) &&
                       totals[1] <= kChainPartners && scheduled && steps < (1u << 16);
    const uint32_t waves = chain ? kChainWaves : kPseWaves;
    uint32_t *perm = nullptr, *wstart = nullptr, *list = nullptr, *lstart = nullptr;
    if (st == VG_OK && scheduled) {
        const size_t deal = nsched * M, starts = nsched * (waves + 1);
        const size_t lists = chain ? deal + slices * (kChainWaves + 1) : 0;
        st = salloc((void **)&sched, (deal + starts + lists) * sizeof(uint32_t), s);
        perm = sched;
        wstart = perm + deal;
        list = wstart + starts;
        lstart = list + deal;
        if (st == VG_OK)
            st = launch("vg_pse_schedule",
                        chain ? k_pse_schedule<kChainWaves, true> : k_pse_schedule<kPseWaves, false>,
                        dim3(steps, slices), dim3(64), 0, s, a, steps, M, perm, wstart);
    }
    if (chain) {
        float *w3 = reinterpret_cast<float *>(w), *alive = w3 + 3 * n;
        if (st == VG_OK)
            st = launch("vg_pse_schedule", k_pse_lists, dim3(slices), dim3(kChainThreads), 0, s,
                        steps, M, (const uint32_t *)perm, (const uint32_t *)wstart, list, lstart);
        if (st == VG_OK) st = salloc((void **)&frac, totals[0] * sizeof(float), s);
        if (st == VG_OK)
            st = launch("vg_pse_gather", k_pse_gather3, dim3(ceil_div(n, 256)), dim3(256), 0, s,
                        tv.sorted_idx, (const float *)angvel, ang_stride, birth, birth_stride, n,
                        w3, alive);
        if (st == VG_OK)
            st = launch("vg_pse_fractions", k_pse_fractions, dim3(ceil_div(cells, 4)), dim3(256), 0, s,
                        a, (uint32_t)cells, (const float *)alive, (const uint32_t *)foff, frac);
        const uint32_t buf_floats = kBufFront + (((uint32_t)totals[1] + 3u) & ~3u) + kBufBack;
        size_t lds = kChainWaves * buf_floats * sizeof(float);
        const bool resident = lds + totals[2] * sizeof(float) <= kLdsBytes;
        if (resident) lds += totals[2] * sizeof(float);
        const auto kernel = resident ? k_pse_phase_chain<true> : k_pse_phase_chain<false>;
        if (st == VG_OK) {
            const hipError_t e =
                hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLdsBytes);
            if (e != hipSuccess) st = device_error(e, "PSE LDS size", __FILE__, __LINE__);
        }
        for (uint32_t phase = 0; phase < 2 && st == VG_OK; ++phase) {
            const uint32_t groups = (slices - phase + 1) / 2;
            if (groups)
                st = launch("vg_pse_phase", kernel, dim3(groups, 3), dim3(kChainThreads), lds, s,
                            a, phase, steps, M, (const uint32_t *)list, (const uint32_t *)lstart,
                            (const float *)frac, (const uint32_t *)foff, (const float *)alive, w3,
                            (uint32_t)n, buf_floats);
        }
        if (st == VG_OK)
            st = launch("vg_pse_scatter", k_pse_scatter3, dim3(ceil_div(n, 256)), dim3(256), 0, s,
                        tv.sorted_idx, (const float *)w3, n, angvel, ang_stride);
    } else {
        if (st == VG_OK)
            st = launch("vg_pse_gather", k_pse_gather, dim3(ceil_div(n, 256)), dim3(256), 0, s,
                        tv.sorted_idx, (const float *)angvel, ang_stride, birth, birth_stride, n,
                        w);
        if (st == VG_OK && precompute && totals[3] > 0 && totals[3] < (1ull << 31)) {
            // (the cells past one wave's share: fewer than the fractions hold of it)
            const size_t most = 1 + totals[3] / kRowsPerWave;
            st = salloc((void **)&wide, (1 + most) * sizeof(uint32_t), s);
            if (st == VG_OK) st = zero_fill(wide, sizeof(uint32_t), s);
            if (st == VG_OK)
                st = launch("vg_pse_frac_size", k_pse_row_size, dim3(ceil_div(cells, 256)),
                            dim3(256), 0, s, a, (uint32_t)cells, fsize, wide);
            if (st == VG_OK) st = exclusive_scan_u32(fsize, foff, cells, stmp, s);
            if (st == VG_OK) st = salloc((void **)&frac, totals[3] * sizeof(float), s);
            a.frac = frac;
            a.frac_off = foff;
            if (st == VG_OK)
                st = launch("vg_pse_fractions", k_pse_row_fractions, dim3(ceil_div(cells, 4)),
                            dim3(256), 0, s, a, (uint32_t)cells, frac);
            if (st == VG_OK && totals[1] * totals[1] > kRowsPerWave)
                st = launch("vg_pse_fractions", k_pse_row_fractions_wide, dim3(32 * kWideParts),
                            dim3(256), 0, s, a, (const uint32_t *)wide, frac);
        }
        for (uint32_t phase = 0; phase < 2 && st == VG_OK; ++phase) {
            const uint32_t groups = (slices - phase + 1) / 2;
            if (groups)
                st = launch("vg_pse_phase", k_pse_phase, dim3(groups), dim3(kPseThreads), 0, s, a,
                            phase, (const uint32_t *)perm, (const uint32_t *)wstart, M);
        }
        if (st == VG_OK)
            st = launch("vg_pse_scatter", k_pse_scatter, dim3(ceil_div(n, 256)), dim3(256), 0, s,
                        tv.sorted_idx, (const float4 *)w, n, angvel, ang_stride);
    }
    sfree(sched, s);
    sfree(wide, s);
    sfree(frac, s);
    sfree(sizes, s);
    sfree(w, s);
    return st;
}

}  // namespace vg

using namespace vg;

VG_API vg_status vg_tree_partition(const vg_tree *t, const uint32_t **cell_start,
                                   const uint32_t **cell_count, const uint32_t **vorton_index,
                                   size_t *cells) {
    VG_REQUIRE(cell_start && cell_count && vorton_index && cells, "null argument");
    TreeView tv;
    VG_TRY(tree_checked_view(t, &tv));
    *cell_start = tv.cell_start;
    *cell_count = tv.cell_count;
    *vorton_index = tv.sorted_idx;
    *cells = capacity(tv.layer[0]);
    return VG_OK;
}

VG_API vg_status vg_tree_pse_diffuse(const vg_tree *t, float *angvel, size_t ang_stride,
                                     const int32_t *birth, size_t birth_stride, float viscosity,
                                     float dt, int order, vg_stream s) {
    VG_REQUIRE(angvel && ang_stride >= 3, "bad angular velocity array");
    VG_REQUIRE(!birth || birth_stride >= 1, "bad birth stride");
    VG_REQUIRE(viscosity * dt <= 1.0f, "viscosity * dt exceeds 1 (vorticity would flip)");
    return pse_diffuse(t, angvel, ang_stride, birth, birth_stride, viscosity, dt, order,
                       (hipStream_t)s);
}
