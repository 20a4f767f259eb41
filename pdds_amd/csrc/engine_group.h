// engine_group.h -- the group path kernel: G neighbouring lanes of a wave carry one path.
//
// A path's steps follow one another, so a launch with few paths -- or the last paths of a large
// one -- lasts as long as its longest path times the time of one step, whatever the card could do
// beside it; one wave issues a step's 400-700 instructions one after another.  Most of a step does
// not depend on the steps before it: the normals of a step are a function of its number, and what
// the functionals Z and xi add is a function of the position it starts from.  Here lane l of a
// group draws the normals of step st + l; the positions then follow by the only part that is
// serial (for a constant sigma without drift one addition per coordinate and step); each lane
// evaluates f, grad u and the stopping test of its own step; and the sums Z and xi are formed in
// step order again.  Every value is formed by the operations of Walker::step in their order, so a
// path's record is the same bit for bit.
//
// FP32 lanes carry two steps each (one Philox call gives the normals of two).
//
// What it costs and gains: the step-ordered part is repeated by every lane of a group, 6 (FP64, DPP
// broadcasts of both halves of a double) to 12 instructions a step, so a group of one lane is the
// cheapest per step (FP32 Helmholtz: about 280 VALU instructions for two steps of 64 paths, 377 for
// eight steps of 16) and one of 16 has the shortest step (a path of the FP64 recorded run: 1.9 us a
// step with one path per lane, 0.15 us here).  A launch starts as wide as its path count asks for
// and widens where a wave's last paths leave room.  Measured against the persistent kernel with one
// path per lane: 4 points x 1000 paths 1.9 -> 0.29 ms, one knot of the recorded run 4.7 -> 0.58,
// the whole run 8.0 -> 3.6, Poisson FP32 (0.6 M paths) 8.2 -> 3.4, server burst 139 -> 83 ms.
#pragma once
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

// Problems whose paths move by a constant multiple of the increments (sigma constant and diagonal,
// no drift): the serial part of a step is one addition per coordinate.
template <int PDE> constexpr bool const_motion() { return PDE == PDE_SINSIN || PDE == PDE_HELMHOLTZ || PDE == PDE_MONEGROS; }
// ... and whose Y changes along a path (c not zero)
template <int PDE> constexpr bool has_c() { return PDE != PDE_SINSIN && PDE != PDE_MONEGROS; }

template <class R, int PDE> constexpr int group_waves() { return sizeof(R) == 8 ? 2 : 4; }

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
    KnotSteps ks;
};

// G steps (FP32: 2 G) of every group of the wave
template <class R, int PDE, int G> __device__ __forceinline__ void group_advance(const PathKernelArgs &a, GroupState<R> &p) {
    constexpr int NS = sizeof(R) == 8 ? 1 : 2;    // steps a lane carries
    const int lane = __lane_id();
    const int sub = lane & (G - 1);
    const int base = lane & ~(G - 1);
    const LutTile none{nullptr, 0, 0, 0, 0};
    const R beta = (R)a.beta;
    const R h = p.h, sqrth = p.sqrth;
    R x = p.x, y = p.y, Y = p.Y, Z = p.Z, xi = p.xi, nzc = p.nzc, nxc = p.nxc;
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
    Coef<R> co;                       // sigma, b and c are constants of the problem
    pde_coef_t<PDE, R, false>(x, y, a.pp, none, p.k2, co);
    R i0[NS], i1[NS], dx[NS], dy[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        i0[s] = sqrth * n1[s];
        i1[s] = sqrth * n2[s];
        dx[s] = em_scale(co.s00, i0[s]);
        dy[s] = em_scale(co.s11, i1[s]);
    }
    // the serial part: where (and with which Y) each lane's first step starts
    R px = x, py = y, pY = Y;
    static_for<G>([&](auto kk) {
        constexpr int K = decltype(kk)::value;
        if constexpr (K > 0) {
            const bool me = group_lane<G, K>();
            px = me ? x : px;
            py = me ? y : py;
            if constexpr (has_c<PDE>()) pY = me ? Y : pY;
        }
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            x = x + group_bcast<G, K>(dx[s]);
            y = y + group_bcast<G, K>(dy[s]);
            if constexpr (has_c<PDE>()) {
                const R dY = co.c * Y * h;
                Y = Y + dY;
            }
        }
    });
    // each lane's own steps: what they add to Z and xi, and where they stop
    R fY[NS], vi[NS], Yb[NS], ex[NS], ey[NS], eY[NS];
    bool stop[NS], cap[NS], go[NS];
    {
        R qx = px, qy = py, qY = pY;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            pde_coef_t<PDE, R, false>(qx, qy, a.pp, none, p.k2, co);
            const R v0 = -(co.s00 * co.g0);
            const R v1 = -(co.s11 * co.g1);
            vi[s] = em_dot(v1, i1[s], v0, i0[s]);
            Yb[s] = qY;
            fY[s] = co.f * qY;
            qx = qx + dx[s];
            qy = qy + dy[s];
            if constexpr (has_c<PDE>()) {
                const R dY = co.c * qY * h;
                qY = qY + dY;
            }
            ex[s] = qx; ey[s] = qy; eY[s] = qY;
            bool xside;
            const R d = rect_dist_inside<R>(p.rect, qx, qy, xside);
            go[s] = d < beta * side_norm(xside, co.s00, co.s11) * sqrth;
            cap[s] = st_l + (uint32_t)s + 1u >= a.max_steps;
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
        const R dz = sub <= last ? fY[0] * h : (R)0, dxi = sub <= last ? Yb[0] * vi[0] : (R)0;
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
                if constexpr (has_c<PDE>()) yk = __builtin_fmaf(t, group_bcast<G, K>(Yb[s]), nxc);
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
        R px2, py2;
        int kind;
        rect_exit<R>(p.rect, s.x, s.y, px2, py2, kind);
        write_exit<R, PDE, GeomRect>(a, p.g, s, p.gmask, px2, py2, kind);
        p.ks.st += st_l + (first ? 1u : (unsigned)NS);
        p.ks.cap += (first ? cap[0] && go[0] : cap[L] && go[L]) ? 1u : 0u;
    }
    p.x = x; p.y = y; p.Y = Y; p.Z = Z; p.xi = xi; p.nzc = nzc; p.nxc = nxc;
    p.active = p.active && row == 0u;
    p.st += (uint32_t)(G * NS);
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

// The paths of the lanes m (at most 64 / G) go on with G lanes each, path i of them in the wave's
// group i.
template <class R, int G>
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
    p.active = row < n;
    if (p.active && k != p.ks.k) p.ks.enter(a, k);
}

// The last paths of a wave (one lane of each in left, at most 16 / G) to their end, in groups four
// times as wide as they were and then wider still.
template <class R, int PDE, int G>
__device__ __forceinline__ void group_finish(const PathKernelArgs &a, GroupState<R> &p, unsigned long long left) {
    if (!left) return;
    constexpr int W = 4 * G;
    group_widen<R, W>(a, p, left);
    while (true) {
        left = __ballot(p.active && (__lane_id() & (W - 1)) == 0);
        if constexpr (W < 16) {
            if (__popcll(left) <= 16 / W) {
                group_finish<R, PDE, W>(a, p, left);
                return;
            }
        } else {
            if (!left) return;
        }
        group_advance<R, PDE, W>(a, p);
    }
}

template <class R, int PDE, bool MIXED, int G>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(group_waves<R, PDE>()))) group_kernel(PathKernelArgs a) {
    static_assert(const_motion<PDE>(), "the serial part is a plain addition");
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
                } else if (qs.drained) {
                    done = true;
                }
            }
            const int64_t cnt = __popcll(m);
            pool.next += cnt < avail ? cnt : avail;
        }
        const unsigned long long left = __ballot(p.active && sub == 0);
        if constexpr (G < 16) {
            // none to start and no more left than wider groups hold (none at all among them)
            if (qs.drained && qs.pool.next >= qs.pool.end && __popcll(left) <= 16 / G) {
                group_finish<R, PDE, G>(a, p, left);
                break;
            }
        } else {
            if (!left) break;
        }
        group_advance<R, PDE, G>(a, p);
    }
    p.ks.flush(a);
}

}  // namespace pdds
