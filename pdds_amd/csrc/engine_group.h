// engine_group.h -- the group path kernel: G neighbouring lanes of a wave carry one path.
//
// A path's steps follow one another, so a launch with few paths -- or the last paths of a large
// one -- lasts as long as its longest path times the time of one step, whatever the card could do
// beside it; one wave issues a step's 400-700 instructions one after another.  Most of a step does
// not depend on the steps before it: the normals of a step are a function of its number, and what
// the functionals Z and xi add is a function of the position it starts from.  Here lane l of a
// group draws the normals of step st + l; the positions then follow by the only part that is
// serial, which every lane of the group repeats (for a constant sigma without drift one addition
// per coordinate and step, else the coefficients that move X; with reflecting sides also distance,
// side and push); each lane evaluates f, grad u and the stopping test of its own step; and the sums
// Z and xi are formed in step order again.  Every value is formed by the operations of
// Walker::step in their order, so a path's record is the same bit for bit.
//
// FP32 lanes carry two steps each (one Philox call gives the normals of two).
//
// What it costs and gains: the step-ordered sums are repeated by every lane of a group, 6 (FP64, DPP
// broadcasts of both halves of a double) to 12 instructions a step, so a group of one lane is the
// cheapest per step (FP32 Helmholtz: about 280 VALU instructions for two steps of 64 paths, 377 for
// eight steps of 16) and one of 16 has the shortest step (a path of the FP64 recorded run: 1.9 us a
// step with one path per lane, 0.15 us here).  A launch starts as wide as its path count asks for
// (group_lanes) and widens where a wave's last paths leave room.  Against one path per lane, whole
// calls: 4 points x 1000 paths 2.4 -> 0.29 ms, one knot of the recorded run 7.0 -> 0.55, the whole
// run 11.2 -> 3.4, Poisson FP32 (0.6 M paths) 13.0 -> 3.4, server burst 129 -> 73; per-path records
// of 1e5 two-phase paths 10.9 -> 4.3, 16 Robin points x 4096 paths 10.6 -> 4.2.
#pragma once
#include <type_traits>
#include <utility>
#include "engine_kernels.h"

namespace pdds {

template <class F, int... K> __device__ __forceinline__ void static_for_seq(F &&f, std::integer_sequence<int, K...>) {
    (f(std::integral_constant<int, K>{}), ...);
}
template <int N, class F> __device__ __forceinline__ void static_for(F &&f) {
    static_for_seq(f, std::make_integer_sequence<int, N>{});
}

// 64-bit form of __builtin_amdgcn_update_dpp (the builtin takes 32 bits only)
__device__ long long update_dpp_i64(long long old, long long src, int ctrl, int row_mask, int bank_mask,
                                    bool bound_ctrl) __asm("llvm.amdgcn.update.dpp.i64");

// lane K's value in every lane of its group of G lanes: a DPP row (row_newbcast:K) or a
// quad (quad_perm).  Every lane of the wave is active where these are used.
template <int G, int K> constexpr int group_ctrl() {
    static_assert(G == 16 || G == 4, "groups are DPP rows or quads");
    return G == 16 ? 0x150 + K : K * 0x55;
}
template <int G, int K> __device__ __forceinline__ float group_bcast(float v) {
    if constexpr (G == 1) return v;
    else return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), group_ctrl<G, K>(), 0xf, 0xf, true));
}
template <int G, int K> __device__ __forceinline__ double group_bcast(double v) {
    if constexpr (G == 1) {
        return v;
    } else if constexpr (G == 16) {
        // v_mov_b64_dpp takes row_newbcast only
        return __builtin_bit_cast(double, update_dpp_i64(0ll, __builtin_bit_cast(long long, v), group_ctrl<G, K>(), 0xf, 0xf, true));
    } else {
        const uint64_t u = __builtin_bit_cast(uint64_t, v);
        const uint32_t lo = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)u, group_ctrl<G, K>(), 0xf, 0xf, true);
        const uint32_t hi = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)(u >> 32), group_ctrl<G, K>(), 0xf, 0xf, true);
        return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
    }
}
// whether the lane is lane K of its group, as a constant mask
template <int G, int K> __device__ __forceinline__ bool group_lane() {
    if constexpr (G == 1) return true;
    constexpr unsigned long long first = G == 16 ? 0x0001000100010001ULL : 0x1111111111111111ULL;
    return __builtin_amdgcn_inverse_ballot_w64(first << K);
}

// Problems whose Y changes along a path (c not zero)
template <int PDE> constexpr bool has_c() { return PDE != PDE_SINSIN && PDE != PDE_MONEGROS; }

// The widest group of a problem: where the coefficients decide the motion, every lane of a group
// repeats their evaluation step by step, and past four lanes a step hardly gets shorter.
template <int PDE> constexpr int group_widest() { return const_motion<PDE>() ? 16 : 4; }

// waves per SIMD of the register budget
template <class R, int PDE> constexpr int group_waves() { return sizeof(R) == 8 || !const_motion<PDE>() ? 2 : 4; }

// What a group carries: its path, the same values in each of its lanes, and the lane's step counts.
template <class R> struct GroupState {
    // nzc, nxc: the negated compensations of the FP32 sums, so that em_step's fma(.., -zc) can take
    // their register
    R x, y, Y, Z, xi, nzc, nxc;
    R x0, y0;               // start point of the group's knot
    RectC<R> rect;
    R h, sqrth, k2;
    uint32_t strm, st, poff, kid, g;
    int gmask;
    bool active;
    LaneSteps ks;
    R s00, s11, b0, b1, c;  // varying motion: the coefficients at X that move it (and Y)
    R rd, lt;               // reflecting sides: distance of the nearest side at X, pending local time
    int rk, rmask;          //   that side, and the reflecting sides of the domain
    uint32_t st0;           // records: steps of the first phase, once it has ended
    bool second;            //   the path is in its second phase
};

// an assembly's launch: exits go to the batch's records
struct NoOut {};

// the coefficients that move X and Y (the others are not formed)
template <class R, int PDE> __device__ __forceinline__ void group_motion(const PathKernelArgs &a, GroupState<R> &p) {
    const LutTile none{nullptr, 0, 0, 0, 0, 0, 0, 0};
    Coef<R> co;
    pde_coef_t<PDE, R, false>(p.x, p.y, a.pp, none, p.k2, co);
    p.s00 = co.s00; p.s11 = co.s11; p.b0 = co.b0; p.b1 = co.b1; p.c = co.c;
}

// distance, side and projection of rect_dist from the rectangle's centre form
template <class R> __device__ __forceinline__ R group_dist(const RectC<R> &p, R x, R y, R &ex, R &ey, int &kind) {
    const R ax = RM<R>::fabs(x - p.cx) - p.hx, ay = RM<R>::fabs(y - p.cy) - p.hy;
    rect_exit<R>(p, x, y, ex, ey, kind);
    R d = kind == 2 || kind == 3 ? ax : ay;
    if (__any(kind > 3)) {
        const R r = RM<R>::sqrt(ax * ax + ay * ay);
        d = kind > 3 ? r : d;
    }
    return d;
}
// the outward normal of side or corner `kind`
template <class R> __device__ __forceinline__ void group_normal(int kind, R &nx, R &ny) {
    const R diag = (R)0.70710678118f;
    const bool corner = kind > 3;
    nx = corner ? (kind == 4 || kind == 6 ? diag : -diag) : kind == 2 ? (R)1 : kind == 3 ? (R)-1 : (R)0;
    ny = corner ? (kind == 4 || kind == 5 ? diag : -diag) : kind == 0 ? (R)1 : kind == 1 ? (R)-1 : (R)0;
}

// value v of lane `from`
template <class T> __device__ __forceinline__ T lane_value(T v, int from) {
    static_assert(sizeof(T) == 4 || sizeof(T) == 8, "one or two registers");
    if constexpr (sizeof(T) == 4) {
        return __builtin_bit_cast(T, __shfl(__builtin_bit_cast(int, v), from));
    } else {
        const uint64_t u = __builtin_bit_cast(uint64_t, v);
        const uint32_t lo = (uint32_t)__shfl((int)(uint32_t)u, from), hi = (uint32_t)__shfl((int)(uint32_t)(u >> 32), from);
        return __builtin_bit_cast(T, ((uint64_t)hi << 32) | lo);
    }
}

// G steps (FP32: 2 G) of every group of the wave
template <class R, int PDE, int G, bool REFL, class OUT>
__device__ __forceinline__ void group_advance(const PathKernelArgs &a, const OUT &out, GroupState<R> &p) {
    constexpr bool VAR = !const_motion<PDE>(), HAS_C = has_c<PDE>(), REC = std::is_same<OUT, PathOut>::value;
    constexpr int NS = sizeof(R) == 8 ? 1 : 2;    // steps a lane carries
    static_assert(!REFL || NS == 1, "reflecting sides: FP64");
    const int lane = __lane_id();
    const int sub = lane & (G - 1);
    const int base = lane & ~(G - 1);
    const LutTile none{nullptr, 0, 0, 0, 0, 0, 0, 0};
    const R beta = REC && p.second ? (R)0 : (R)a.beta;
    const R h = p.h, sqrth = p.sqrth;
    R x = p.x, y = p.y, Y = p.Y, Z = p.Z, xi = p.xi, nzc = p.nzc, nxc = p.nxc;
    // (an FP64 group without a path reads one texel's lines of a table; with that test the compiler
    // issues the FP32 reads one by one: 40 points x 30 paths of the LUT 0.7 ms, 1.7 so)
    const bool live = sizeof(R) == 4 || p.active;
    // normals of the lane's steps, and the moves they make
    R n1[NS], n2[NS];
    const uint32_t st_l = p.st + (uint32_t)(sub * NS);
    if constexpr (NS == 1) {
        normals_f64(a.seed, p.strm, p.kid, p.g - p.poff, st_l, n1[0], n2[0]);
    } else {
        float n[4];
        normals4_f32(st_l >> 1, p.g - p.poff, p.kid, a.seed, p.strm, n);
        n1[0] = n[0]; n2[0] = n[1]; n1[1] = n[2]; n2[1] = n[3];
    }
    Coef<R> co;
    if constexpr (VAR) {
        co.s00 = p.s00; co.s11 = p.s11; co.b0 = p.b0; co.b1 = p.b1; co.c = p.c;
    } else {
        pde_coef_t<PDE, R, false>(x, y, a.pp, none, p.k2, co, live);   // sigma, b and c are constants
    }
    R i0[NS], i1[NS], dx[NS], dy[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        i0[s] = sqrth * n1[s];
        i1[s] = sqrth * n2[s];
        if constexpr (!VAR) {
            dx[s] = em_scale(co.s00, i0[s]);
            dy[s] = em_scale(co.s11, i1[s]);
        }
    }
    // the serial part: where (and, its Y not waiting for local time, with which Y) each lane's first
    // step starts; the coefficients, or distance and side, where its last one ends
    R px = x, py = y, pY = Y;
    R qs00 = co.s00, qs11 = co.s11;
    R pd = 0, pLt = 0, qx = 0, qy = 0, qd = 0, qlt = 0, d = p.rd, lt = p.lt;
    int pk = 0, qk = 0, kind = p.rk;
    R E = 0;
    // constant motion: the root of the lane's own Lepingle step for a side in x and one in y (a side's
    // normal has one component, +-1), which so leaves the serial part (5 points x 500 paths
    // 2.34 -> 2.13 ms, 20 x 20000 18.9 -> 17.6).  A corner's has two, and its root is formed in place.  A
    // path steps from a corner only where it starts past one, or was put back onto one (below) and
    // the projection rounded outwards: corner says whether a path of the wave may do so.
    R Sx = 0, Sy = 0;
    bool corner = false;
    if constexpr (REFL) {
        E = draw_exponential<R>(st_l, p.g - p.poff, a.seed, p.strm, p.kid);
        if constexpr (!VAR) {
            corner = __any(p.active && kind > 3);
            const R hE = ((R)2.0 * h) * E;
            Sx = RM<R>::sqrt((co.s00 * co.s00) * hE + dx[0] * dx[0]);
            Sy = RM<R>::sqrt((co.s11 * co.s11) * hE + dy[0] * dy[0]);
        }
    }
    static_for<G>([&](auto kk) {
        constexpr int K = decltype(kk)::value;
        const bool me = group_lane<G, K>();
        if constexpr (K > 0) {
            px = me ? x : px;
            py = me ? y : py;
            if constexpr (HAS_C && !REFL) pY = me ? Y : pY;
        }
        if constexpr (REFL) {
            // refl_step's move: the Lepingle step while the nearest side reflects (within rho of it)
            R nx, ny, L = (R)0;
            group_normal<R>(kind, nx, ny);
            const bool lep = refl_kind(kind, p.rmask) && (a.pp.rho <= 0.0 || d > -(R)a.pp.rho);
            R mx, my;
            auto push = [&](R j0, R j1) {
                const R ga = nx * co.s00, gb = ny * co.s11;
                const R uc = (ga * j0 + gb * j1) + (nx * co.b0 + ny * co.b1) * h;
                const R M = (R)0.5 * (uc + RM<R>::sqrt((ga * ga + gb * gb) * (((R)2.0 * h) * group_bcast<G, K>(E)) + uc * uc));
                return RM<R>::fmax((R)0, M + d);
            };
            if constexpr (VAR) {
                const R j0 = group_bcast<G, K>(i0[0]), j1 = group_bcast<G, K>(i1[0]);
                if (__any(lep)) {
                    const R Lp = push(j0, j1);
                    L = lep ? Lp : (R)0;
                }
                mx = em_move(co.b0, h, co.s00, j0);
                my = em_move(co.b1, h, co.s11, j1);
            } else {
                mx = group_bcast<G, K>(dx[0]);
                my = group_bcast<G, K>(dy[0]);
                const R sx = group_bcast<G, K>(Sx), sy = group_bcast<G, K>(Sy);
                const R S = nx != (R)0 ? sx : sy;
                const R M = (R)0.5 * (nx * mx + ny * my + S);
                L = lep ? RM<R>::fmax((R)0, M + d) : (R)0;
                if (__builtin_expect(corner, 0)) {
                    const R Lp = push(group_bcast<G, K>(i0[0]), group_bcast<G, K>(i1[0]));
                    L = lep && kind > 3 ? Lp : L;
                    corner = false;
                }
            }
            pd = me ? d : pd;
            pk = me ? kind : pk;
            pLt = me ? L + lt : pLt;
            x = x + mx;
            y = y + my;
            x = lep ? x - L * nx : x;
            y = lep ? y - L * ny : y;
            R ex, ey;
            d = group_dist<R>(p.rect, x, y, ex, ey, kind);
            // past a reflecting side: back onto it, the distance becoming local time
            const bool past = refl_kind(kind, p.rmask) && d > (R)0;
            lt = past ? d : (R)0;
            if (__any(past)) {
                x = past ? ex : x;
                y = past ? ey : y;
                int k2;
                const R d2 = group_dist<R>(p.rect, x, y, ex, ey, k2);
                d = past ? d2 : d;
                kind = past ? k2 : kind;
                if constexpr (!VAR) corner = __any(past && kind > 3);
            }
            if constexpr (VAR) pde_coef_t<PDE, R, false>(x, y, a.pp, none, p.k2, co, live);
            qx = me ? x : qx;
            qy = me ? y : qy;
            qd = me ? d : qd;
            qk = me ? kind : qk;
            if constexpr (REC) qlt = me ? lt : qlt;
        } else {
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                if constexpr (VAR) {
                    const R j0 = group_bcast<G, K>(i0[s]), j1 = group_bcast<G, K>(i1[s]);
                    x = x + em_move(co.b0, h, co.s00, j0);
                    y = y + em_move(co.b1, h, co.s11, j1);
                } else {
                    x = x + group_bcast<G, K>(dx[s]);
                    y = y + group_bcast<G, K>(dy[s]);
                }
                if constexpr (HAS_C) {
                    const R dY = co.c * Y * h;
                    Y = Y + dY;
                }
                if constexpr (VAR) pde_coef_t<PDE, R, false>(x, y, a.pp, none, p.k2, co, live);
            }
        }
        if constexpr (VAR) {
            qs00 = me ? co.s00 : qs00;
            qs11 = me ? co.s11 : qs11;
        }
    });
    p.s00 = co.s00; p.s11 = co.s11; p.b0 = co.b0; p.b1 = co.b1; p.c = co.c;
    p.rd = d; p.rk = kind; p.lt = lt;
    // each lane's own steps: what they add to Z and xi, and where they stop
    R fY[NS], vi[NS], Yb[NS], ex[NS], ey[NS], eY[NS], lz = 0;
    bool stop[NS], cap[NS], go[NS];
    if constexpr (REFL) {
        pde_coef_t<PDE, R, false>(px, py, a.pp, none, p.k2, co, live);
        vi[0] = em_dot(-(co.s11 * co.g1), i1[0], -(co.s00 * co.g0), i0[0]);
        // local time of the step: boundary data at X's projection, the growth factor of Y
        R psi = (R)0, w = (R)0;
        const R phi = (R)a.pp.robin;
        if (__any(pLt > (R)0)) {
            R nx, ny;
            group_normal<R>(pk, nx, ny);
            const R ps = pde_psi<PDE, R>(px - pd * nx, py - pd * ny, nx, ny, phi, a.pp);
            const R pw = pLt * RM<R>::exprel(phi * pLt);
            psi = pLt > (R)0 ? ps : (R)0;
            w = pLt > (R)0 ? pw : (R)0;
        }
        // Y in step order
        const R c = co.c;
        static_for<G>([&](auto kk) {
            constexpr int K = decltype(kk)::value;
            const bool me = group_lane<G, K>();
            pY = me ? Y : pY;
            const R dY = group_bcast<G, K>(c) * Y * h + (phi * Y) * group_bcast<G, K>(w);
            Y = Y + dY;
        });
        Yb[0] = pY;
        fY[0] = co.f * pY;
        lz = (psi * pY) * w;
        ex[0] = qx; ey[0] = qy;
        {
            const R dY = c * pY * h + (phi * pY) * w;
            eY[0] = pY + dY;
        }
        R nx, ny;
        group_normal<R>(qk, nx, ny);
        if constexpr (VAR) { co.s00 = qs00; co.s11 = qs11; }
        const R nrm = normal_sigma<R, PDE, STEP_CV, REFL>(nx, ny, co);
        go[0] = refl_kind(qk, p.rmask) || qd < beta * nrm * sqrth;
        cap[0] = st_l + 1u - p.st0 >= a.max_steps;
        stop[0] = !go[0] || cap[0];
    } else {
        R tx = px, ty = py, tY = pY;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            pde_coef_t<PDE, R, false>(tx, ty, a.pp, none, p.k2, co, live);
            const R v0 = -(co.s00 * co.g0);
            const R v1 = -(co.s11 * co.g1);
            vi[s] = em_dot(v1, i1[s], v0, i0[s]);
            Yb[s] = tY;
            fY[s] = co.f * tY;
            if constexpr (VAR) {
                tx = tx + em_move(co.b0, h, co.s00, i0[s]);
                ty = ty + em_move(co.b1, h, co.s11, i1[s]);
            } else {
                tx = tx + dx[s];
                ty = ty + dy[s];
            }
            if constexpr (HAS_C) {
                const R dY = co.c * tY * h;
                tY = tY + dY;
            }
            ex[s] = tx; ey[s] = ty; eY[s] = tY;
            R s00 = co.s00, s11 = co.s11;      // sigma where the step ends
            if constexpr (VAR) {
                if (s + 1 < NS) {
                    Coef<R> cm;
                    pde_coef_t<PDE, R, false>(tx, ty, a.pp, none, p.k2, cm, live);
                    s00 = cm.s00; s11 = cm.s11;
                } else {
                    s00 = qs00; s11 = qs11;
                }
            }
            bool xside;
            const R dd = rect_dist_inside<R>(p.rect, tx, ty, xside);
            go[s] = dd < beta * side_norm(xside, s00, s11) * sqrth;
            cap[s] = st_l + (uint32_t)s + 1u - (REC ? p.st0 : 0u) >= a.max_steps;
            stop[s] = !go[s] || cap[s];
        }
    }
    // the group's first stopping step ends its path
    bool any_stop = stop[0];
    if constexpr (NS == 2) any_stop = any_stop || stop[1];
    const unsigned long long sm = __ballot(p.active && any_stop);
    const unsigned row = (unsigned)(sm >> base) & ((1u << G) - 1u);
    const int last = row != 0u ? __builtin_ctz(row) : G;
    // Z and xi in step order
    R eZ[NS], exi[NS];
    if constexpr (NS == 1) {
        // the steps after the stop add 0
        R dz = fY[0] * h;
        if constexpr (REFL) dz = dz + lz;
        dz = sub <= last ? dz : (R)0;
        const R dxi = sub <= last ? Yb[0] * vi[0] : (R)0;
        static_for<G>([&](auto kk) {
            constexpr int K = decltype(kk)::value;
            xi = xi + group_bcast<G, K>(dxi);
            Z = Z + group_bcast<G, K>(dz);
        });
        eZ[0] = Z; exi[0] = xi;
    } else {
        // Kahan-compensated sums with em_step's fused products; a lane keeps the sums after each
        // of its own steps
#pragma unroll
        for (int s = 0; s < NS; ++s) { eZ[s] = Z; exi[s] = xi; }
        static_for<G>([&](auto kk) {
            constexpr int K = decltype(kk)::value;
            const bool me = group_lane<G, K>();
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                const R t = group_bcast<G, K>(vi[s]);
                R yk;
                if constexpr (HAS_C) yk = __builtin_fmaf(t, group_bcast<G, K>(Yb[s]), nxc);
                else yk = t + nxc;
                const R tk = xi + yk;
                nxc = yk - (tk - xi);
                xi = tk;
                const R yz = __builtin_fmaf(group_bcast<G, K>(fY[s]), h, nzc);
                const R tz = Z + yz;
                nzc = yz - (tz - Z);
                Z = tz;
                eZ[s] = me ? Z : eZ[s];
                exi[s] = me ? xi : exi[s];
            }
        });
    }
    if (p.active && sub == last) {
        constexpr int L = NS - 1;
        const bool first = stop[0];
        PathState<R> s;
        s.x = first ? ex[0] : ex[L]; s.y = first ? ey[0] : ey[L]; s.Y = first ? eY[0] : eY[L];
        s.Z = first ? eZ[0] : eZ[L]; s.xi = first ? exi[0] : exi[L];
        const uint32_t st = st_l + (first ? 1u : (unsigned)NS);
        R px2, py2;
        int kd;
        rect_exit<R>(p.rect, s.x, s.y, px2, py2, kd);
        if constexpr (REC) {
            const int f = p.second ? 1 : 0;
            if (out.xt[f]) out.xt[f][p.g] = (double)px2;
            if (out.yt[f]) out.yt[f][p.g] = (double)py2;
            if (out.Y[f]) out.Y[f][p.g] = (double)s.Y;
            if (out.Z[f]) out.Z[f][p.g] = (double)s.Z;
            if (out.xi[f]) out.xi[f][p.g] = (double)s.xi;
            if (out.steps[f]) out.steps[f][p.g] = (int64_t)(st - p.st0);
        } else {
            write_exit<R, PDE, GeomRect>(a, p.g, s, p.gmask, px2, py2, kd);
            p.ks.st += st;
            p.ks.cap += (first ? cap[0] && go[0] : cap[L] && go[L]) ? 1u : 0u;
        }
    }
    p.x = x; p.y = y; p.Y = Y; p.Z = Z; p.xi = xi; p.nzc = nzc; p.nxc = nxc;
    const uint32_t st_was = p.st;
    p.st += (uint32_t)(G * NS);
    bool ended = row != 0u;
    if constexpr (REC && NS == 1) {
        // the second phase goes on from the first one's last step
        const bool next = p.active && ended && !p.second && out.phase2 != 0;
        if (__any(next)) {
            const int from = next ? base + last : lane;
            const R nx = lane_value(ex[0], from), ny = lane_value(ey[0], from), nY = lane_value(eY[0], from);
            const R nd = lane_value(qd, from), nlt = lane_value(qlt, from);
            const int nk = lane_value(qk, from);
            if (next) {
                p.x = nx; p.y = ny; p.Y = nY;
                p.st = st_was + (uint32_t)last + 1u;
                p.st0 = p.st;
                p.second = true;
                if constexpr (REFL) { p.rd = nd; p.lt = nlt; p.rk = nk; }
                if constexpr (VAR) group_motion<R, PDE>(a, p);
            }
            ended = ended && !next;
        }
    }
    p.active = p.active && !ended;
}

// The paths of the lanes m (at most 64 / G) go on with G lanes each, path i of them in the wave's
// group i.
template <class R, int G, bool VAR, bool REFL, bool REC>
__device__ __forceinline__ void group_widen(const PathKernelArgs &a, GroupState<R> &p, unsigned long long m) {
    const int lane = __lane_id();
    const int n = __popcll(m), row = lane / G;
    for (int i = 0; i < row; ++i) m &= m - 1;
    const int from = row < n ? __builtin_ctzll(m) : lane;   // a lane of the group's path
    const int k = lane_value(p.ks.k, from);
    p.x = lane_value(p.x, from); p.y = lane_value(p.y, from); p.Y = lane_value(p.Y, from);
    p.Z = lane_value(p.Z, from); p.xi = lane_value(p.xi, from);
    p.nzc = lane_value(p.nzc, from); p.nxc = lane_value(p.nxc, from);
    p.rect.cx = lane_value(p.rect.cx, from); p.rect.cy = lane_value(p.rect.cy, from);
    p.rect.hx = lane_value(p.rect.hx, from); p.rect.hy = lane_value(p.rect.hy, from);
    p.h = lane_value(p.h, from); p.sqrth = lane_value(p.sqrth, from); p.k2 = lane_value(p.k2, from);
    p.strm = lane_value(p.strm, from); p.st = lane_value(p.st, from); p.poff = lane_value(p.poff, from);
    p.kid = lane_value(p.kid, from); p.g = lane_value(p.g, from); p.gmask = lane_value(p.gmask, from);
    if constexpr (VAR) {
        p.s00 = lane_value(p.s00, from); p.s11 = lane_value(p.s11, from);
        p.b0 = lane_value(p.b0, from); p.b1 = lane_value(p.b1, from); p.c = lane_value(p.c, from);
    }
    if constexpr (REFL) {
        p.rd = lane_value(p.rd, from); p.lt = lane_value(p.lt, from);
        p.rk = lane_value(p.rk, from); p.rmask = lane_value(p.rmask, from);
    }
    if constexpr (REC) {
        p.st0 = lane_value(p.st0, from);
        p.second = lane_value(p.second ? 1 : 0, from) != 0;
    }
    p.active = row < n;
    if (p.active && k != p.ks.k) p.ks.enter(a, k);
}

// The last paths of a wave (one lane of each in left, at most 16 / G) to their end, in groups four
// times as wide as they were and then wider still.
template <class R, int PDE, int G, bool REFL, class OUT>
__device__ __forceinline__ void group_finish(const PathKernelArgs &a, const OUT &out, GroupState<R> &p, unsigned long long left) {
    if (!left) return;
    constexpr int W = 4 * G;
    static_assert(W <= group_widest<PDE>(), "a kernel does not widen past its widest form");
    group_widen<R, W, !const_motion<PDE>(), REFL, std::is_same<OUT, PathOut>::value>(a, p, left);
    while (true) {
        left = __ballot(p.active && (__lane_id() & (W - 1)) == 0);
        if constexpr (W < group_widest<PDE>()) {
            if (__popcll(left) <= 16 / W) {
                group_finish<R, PDE, W, REFL>(a, out, p, left);
                return;
            }
        } else {
            if (!left) return;
        }
        group_advance<R, PDE, W, REFL>(a, out, p);
    }
}

template <class R, int PDE, bool MIXED, int G, bool REFL = false, class OUT = NoOut>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(group_waves<R, PDE>()))) group_kernel(PathKernelArgs a, OUT out) {
    const int lane = __lane_id();
    const int sub = lane & (G - 1);
    const int base = lane & ~(G - 1);
    GroupState<R> p{};
    p.rect = RectC<R>{0, 0, 1, 1};
    p.h = (R)a.h; p.sqrth = (R)a.sqrth; p.k2 = (R)a.pp.k2;
    p.strm = a.stream;
    p.ks.init();
    bool done = false;
    PathQueues qs;
    qs.init(a);
    while (true) {
        while (true) {
            const bool need = !p.active && !done;
            const unsigned long long m = __ballot(need && sub == 0);
            if (!m) break;
            qs.refill(a, lane);
            WavePool &pool = qs.pool;
            const int64_t avail = pool.end > pool.next ? pool.end - pool.next : 0;
            const int rank = __popcll(m & ((1ULL << base) - 1ULL));
            if (need) {
                if (rank < avail) {
                    const int64_t gg = pool.next + rank;
                    const int k = pool.knot_of(a, gg);
                    if (k != p.ks.k) {
                        p.ks.enter(a, k);
                        const KnotDesc &kd = a.knots[k];
                        const R d[4] = {(R)kd.dom[0], (R)kd.dom[1], (R)kd.dom[2], (R)kd.dom[3]};
                        p.rect = rect_centre<R>(d);
                        p.gmask = kd.gmask;
                        p.kid = kd.knot_id;
                        p.poff = (uint32_t)kd.path_off;
                        p.x0 = (R)kd.x0; p.y0 = (R)kd.y0;
                        if constexpr (REFL) {
                            p.rmask = kd.gmask & a.pp.refl;
                            loaded(p.rmask);
                        }
                        if constexpr (MIXED) {
                            p.strm = kd.stream; p.k2 = (R)kd.k2; p.h = (R)kd.h; p.sqrth = (R)kd.sqrth;
                            loaded(p.strm); loaded(p.k2); loaded(p.h); loaded(p.sqrth);
                        }
                        loaded(p.x0); loaded(p.y0); loaded(p.poff); loaded(p.kid); loaded(p.gmask);
                        loaded(p.rect.cx); loaded(p.rect.cy); loaded(p.rect.hx); loaded(p.rect.hy);
                    }
                    p.g = (uint32_t)gg;
                    p.x = p.x0; p.y = p.y0;
                    p.Y = (R)1; p.Z = (R)0; p.xi = (R)0; p.nzc = (R)0; p.nxc = (R)0;
                    p.st = 0;
                    p.active = true;
                    if constexpr (!const_motion<PDE>()) group_motion<R, PDE>(a, p);
                    if constexpr (REFL) {
                        R ex, ey;
                        p.rd = group_dist<R>(p.rect, p.x, p.y, ex, ey, p.rk);
                        p.lt = (R)0;
                    }
                    if constexpr (std::is_same<OUT, PathOut>::value) {
                        p.st0 = 0;
                        p.second = false;
                    }
                } else if (qs.drained) {
                    done = true;
                }
            }
            const int64_t cnt = __popcll(m);
            pool.next += cnt < avail ? cnt : avail;
        }
        const unsigned long long left = __ballot(p.active && sub == 0);
        if constexpr (G < group_widest<PDE>()) {
            // none to start and no more left than wider groups hold (none at all among them)
            if (qs.drained && qs.pool.next >= qs.pool.end && __popcll(left) <= 16 / G) {
                group_finish<R, PDE, G, REFL>(a, out, p, left);
                break;
            }
        } else {
            if (!left) break;
        }
        group_advance<R, PDE, G, REFL>(a, out, p);
    }
    p.ks.flush(a);
}

}  // namespace pdds
