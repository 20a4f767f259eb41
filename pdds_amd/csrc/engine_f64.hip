// engine_f64.hip -- FP64 instantiations of the path kernels, and the reduction,
// finalize and LUT-evaluation kernels (shared by both path precisions).  Built
// with -ffp-contract=off so that the only fused multiply-adds are the explicit
// fma() calls: every FP64 path and every reduction is then bit-identical to the
// FP64 CPU restatement on the same Philox stream.
#include "../../include/pdds_engine.h"
#include "engine_kernels.h"

namespace pdds {

__constant__ double kExp2TabDev[64] = PDDS_EXP2_TAB;   // 2^(j/64), j = 0..63

template <int PDE, int GEOM, int FAM>
static hipError_t path_f64_gf(bool persistent, bool mixed, const PathLaunch &l, const PathKernelArgs &a) {
    if (!persistent) return l.go(plain_kernel<double, PDE, GEOM, FAM>, a);
    return mixed ? l.go(path_kernel<double, PDE, true, GEOM, FAM>, a) : l.go(path_kernel<double, PDE, false, GEOM, FAM>, a);
}

// the default control-variate step has kernels of its own, without a family test in the loop
template <int PDE, int GEOM>
static hipError_t path_f64_g(bool persistent, bool mixed, const PathLaunch &l, const PathKernelArgs &a) {
    if (a.pp.step != STEP_CV) return path_f64_gf<PDE, GEOM, STEP_ANY>(persistent, mixed, l, a);
    if constexpr (GEOM == GeomRect && group_only<PDE, double>()) {
        // (its persistent form is the group kernel)
        return persistent ? hipErrorInvalidValue : l.go(plain_kernel<double, PDE, GEOM, STEP_CV>, a);
    } else {
        return path_f64_gf<PDE, GEOM, STEP_CV>(persistent, mixed, l, a);
    }
}

template <int PDE>
static hipError_t path_f64(int geom, bool persistent, bool mixed, const PathLaunch &l, const PathKernelArgs &a) {
    if (a.pp.refl) {
        // reflecting sides: rectangles, one stream and k2 per launch, every step family
        if (mixed || geom != GeomRect) return hipErrorInvalidValue;
        return persistent ? l.go(path_kernel<double, PDE, false, GeomRect, STEP_ANY, true>, a)
                          : l.go(plain_kernel<double, PDE, GeomRect, STEP_ANY, true>, a);
    }
    return geom == GeomDisc ? path_f64_g<PDE, GeomDisc>(persistent, mixed, l, a)
                            : path_f64_g<PDE, GeomRect>(persistent, mixed, l, a);
}

hipError_t launch_path_f64(int pde, int geom, bool persistent, bool mixed, const PathLaunch &l, const PathKernelArgs &a) {
    switch (pde) {
        case PDE_MONEGROS: return path_f64<PDE_MONEGROS>(geom, persistent, mixed, l, a);
        case PDE_SINSIN: return path_f64<PDE_SINSIN>(geom, persistent, mixed, l, a);
        case PDE_VARCOEF: return path_f64<PDE_VARCOEF>(geom, persistent, mixed, l, a);
        case PDE_VARCOEF_LUT: return path_f64<PDE_VARCOEF_LUT>(geom, persistent, mixed, l, a);
        case PDE_HELMHOLTZ: return path_f64<PDE_HELMHOLTZ>(geom, persistent, mixed, l, a);
        case PDE_TABLE: return path_f64<PDE_TABLE>(geom, persistent, mixed, l, a);
        default: return hipErrorInvalidValue;
    }
}

template <int PDE, int GEOM> static int path_tiled_wg_g(int precision, int step) {
    if (step == STEP_CV)
        return precision == PDDS_FP64 ? tiled_wg<double, PDE, STEP_CV, GEOM>() : tiled_wg<float, PDE, STEP_CV, GEOM>();
    return precision == PDDS_FP64 ? tiled_wg<double, PDE, STEP_ANY, GEOM>() : tiled_wg<float, PDE, STEP_ANY, GEOM>();
}

int path_tiled_wg(int pde, int precision, int step, int geom) {
    if (pde == PDE_TABLE) return path_tiled_wg_g<PDE_TABLE, GeomRect>(precision, step);
    return geom == GeomDisc ? path_tiled_wg_g<PDE_VARCOEF_LUT, GeomDisc>(precision, step)
                            : path_tiled_wg_g<PDE_VARCOEF_LUT, GeomRect>(precision, step);
}

template <int PDE, bool MIXED, int GEOM, int FAM>
static hipError_t path_tiled_f64_f(int grid, size_t lds, hipStream_t s, const PathKernelArgs &a) {
    if (lds > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute((const void *)path_kernel_tiled<double, PDE, MIXED, GEOM, FAM>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL((path_kernel_tiled<double, PDE, MIXED, GEOM, FAM>), dim3(grid), dim3(tiled_wg<double, PDE, FAM, GEOM>()), lds, s, a);
    return hipGetLastError();
}

template <int PDE, bool MIXED, int GEOM>
static hipError_t path_tiled_f64(int grid, size_t lds, hipStream_t s, const PathKernelArgs &a) {
    return a.pp.step == STEP_CV ? path_tiled_f64_f<PDE, MIXED, GEOM, STEP_CV>(grid, lds, s, a)
                                : path_tiled_f64_f<PDE, MIXED, GEOM, STEP_ANY>(grid, lds, s, a);
}

template <int PDE, int GEOM> static hipError_t path_tiled_f64_m(bool mixed, int grid, size_t lds, hipStream_t s, const PathKernelArgs &a) {
    return mixed ? path_tiled_f64<PDE, true, GEOM>(grid, lds, s, a) : path_tiled_f64<PDE, false, GEOM>(grid, lds, s, a);
}

hipError_t launch_path_tiled_f64(int pde, int geom, bool mixed, int grid, size_t lds, hipStream_t s, const PathKernelArgs &a) {
    if (pde == PDE_TABLE) return geom == GeomRect ? path_tiled_f64_m<PDE_TABLE, GeomRect>(mixed, grid, lds, s, a) : hipErrorInvalidValue;
    return geom == GeomDisc ? path_tiled_f64_m<PDE_VARCOEF_LUT, GeomDisc>(mixed, grid, lds, s, a)
                            : path_tiled_f64_m<PDE_VARCOEF_LUT, GeomRect>(mixed, grid, lds, s, a);
}

template <int PDE>
static hipError_t paths_f64(int grid, int wg, hipStream_t s, const PathsArgs &a) {
    if (a.pp.refl)
        hipLaunchKernelGGL((paths_kernel<double, PDE, STEP_ANY, true>), dim3(grid), dim3(wg), 0, s, a);
    else if (a.pp.step == STEP_CV)
        hipLaunchKernelGGL((paths_kernel<double, PDE, STEP_CV>), dim3(grid), dim3(wg), 0, s, a);
    else
        hipLaunchKernelGGL((paths_kernel<double, PDE, STEP_ANY>), dim3(grid), dim3(wg), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_paths_f64(int pde, int grid, int wg, hipStream_t s, const PathsArgs &a) {
    switch (pde) {
        case PDE_MONEGROS: return paths_f64<PDE_MONEGROS>(grid, wg, s, a);
        case PDE_SINSIN: return paths_f64<PDE_SINSIN>(grid, wg, s, a);
        case PDE_VARCOEF: return paths_f64<PDE_VARCOEF>(grid, wg, s, a);
        case PDE_VARCOEF_LUT: return paths_f64<PDE_VARCOEF_LUT>(grid, wg, s, a);
        case PDE_HELMHOLTZ: return paths_f64<PDE_HELMHOLTZ>(grid, wg, s, a);
        case PDE_TABLE: return paths_f64<PDE_TABLE>(grid, wg, s, a);
        default: return hipErrorInvalidValue;
    }
}

// The reduction of stencils and sub-batches that reduce16_kernel does not take (more than 32 tiles of
// 16 side entries, or a group's records and moments too large for two work-groups on a CU): one
// work-group per work item.  Per-side RBF moments per sub-batch, G_beta = -Psi^-T Phi per
// CSR column, sums in fixed order (sub-batch -> item), B sums per sub-batch.  A group of kNBG
// sub-batches is staged in LDS with, per (sub-batch, side), the list of its paths that exit
// through that side in path order (built with wave ballots, each exit's side read from its
// record's Y bits or found from its exit point, and counted per side).  A thread then owns one stencil
// entry e and, for each sub-batch b, adds Y phi_e(X) over the list of e's side in path order
// (the order of the per-exit loop it replaces), four exits per iteration so that four exp chains
// are in flight; Phi is kept [entry][sub-batch] so that the Psi^-T pass reads a row of kNBG
// values with two 16-byte LDS reads per pair of sub-batches.
// EQ: the launch carries reference values (ReduceArgs::wref) and also sums the knot equations
// SIDE (ReduceSide): how the exit side of a record is found
template <bool EQ, int SIDE>
__global__ void __launch_bounds__(kReduceWG) __attribute__((amdgpu_waves_per_eu(4))) reduce_kernel(ReduceArgs a) {
    extern __shared__ __align__(16) double smem[];
    __shared__ double s_bsb[kNBG], s_bbsb[kNBG];
    __shared__ double s_wsum[(kReduceWG / 64) * kNBG];
    __shared__ double s_exp2[64];
    __shared__ int s_lcnt[kNBG * 4];
    __shared__ unsigned int s_cnt[8];
    const int tid = threadIdx.x;
    const int WG = blockDim.x;
    const int lane = tid & 63, wave = tid >> 6, nwaves = WG >> 6;
    const int64_t item = a.items[a.item_base + (int64_t)blockIdx.x].span_first;
    const ItemDesc it = a.items[item];
    const KnotDesc kd = a.knots[it.knot];
    const TableDesc tb = a.tables[kd.table];
    const StencilDesc &sd = tb.sten[kd.stencil];
    const int64_t g0 = kd.path_off + it.p_begin;
    const ExitRec *rr = a.rec.r + g0;
    const int S = a.S;
    const int GS = kNBG * S;
    double *Phi = smem;                                     // [ne_cap][kNBG]
    double *accS = smem + kNBG * a.ne_cap;
    double *accQ = accS + a.nnz_cap;
    double *gx = accQ + a.nnz_cap;
    double *gy = gx + GS;
    double *gY = gy + GS;
    double *gs = gY + GS;
    uint16_t *lst = (uint16_t *)(gs + GS);
    if (tid == 0)
        for (int q = 0; q < 8; ++q) s_cnt[q] = 0u;
    if (tid < 64) s_exp2[tid] = kExp2TabDev[tid];
    __syncthreads();
    // exit side of a record (stencil side 0..3, 4 global boundary, -1 none) and its Y
    auto side_of = [&](double x, double y, double Yr, double &Y) -> int {
        if constexpr (SIDE == SIDE_BITS) {
            const uint64_t yb = __builtin_bit_cast(uint64_t, Yr);
            Y = __builtin_bit_cast(double, yb & ~kSideBitsMask);
            return (int)(yb & kSideBitsMask) - 1;
        }
        Y = Yr;
        if constexpr (SIDE == SIDE_DISC) return classify_sector(sd.geo, a.gc[0], x, y);
        else return classify_coord_c(sd.rect, a.gc, x, y);
    };
    const int ne = sd.msz[0] + sd.msz[1] + sd.msz[2] + sd.msz[3];
    const int nnz = sd.csr_nnz;
    const int nsb = (it.n + S - 1) / S;
    // per-side sizes, first entries and Psi^-1 offsets as scalars picked by selects: a private
    // array indexed by a per-lane side would live in scratch memory
    const int ms0 = sd.msz[0], ms1 = sd.msz[1], ms2 = sd.msz[2], ms3 = sd.msz[3];
    const int64_t io0 = sd.ipsi_off[0], io1 = sd.ipsi_off[1], io2 = sd.ipsi_off[2], io3 = sd.ipsi_off[3];
    auto pick = [](int s, auto v0, auto v1, auto v2, auto v3) { return s == 0 ? v0 : s == 1 ? v1 : s == 2 ? v2 : v3; };
    auto msz_of = [&](int s) { return pick(s, ms0, ms1, ms2, ms3); };
    auto eoff_of = [&](int s) { return pick(s, 0, ms0, ms0 + ms1, ms0 + ms1 + ms2); };
    auto ipsi_of = [&](int s) { return pick(s, io0, io1, io2, io3); };
    for (int c = tid; c < nnz; c += WG) { accS[c] = 0.0; accQ[c] = 0.0; }
    double Bs = 0.0, BBs = 0.0, Rs = 0.0, RQs = 0.0;
    // (holding the next group's records in registers while a group is reduced, to overlap their
    // loads with the work, takes 8 more registers than the four-wave budget leaves: with the
    // exit side found below it spills and runs the reduction 35 % slower)
    for (int g = 0; g < nsb; g += kNBG) {
        const int nb = (nsb - g) < kNBG ? (nsb - g) : kNBG;
        const int q0 = g * S;                                   // first path of the group
        const int gn = (it.n - q0) < nb * S ? (it.n - q0) : nb * S;
        for (int p = tid; p < gn; p += WG) {
            const ExitRec rc = rr[q0 + p];
            gx[p] = rc.x;
            gy[p] = rc.y;
            gY[p] = rc.Y;
            gs[p] = rc.score;
        }
        __syncthreads();
        // per (sub-batch, side) lists in path order: a wave per sub-batch, 64 paths per ballot
        for (int b = wave; b < nb; b += nwaves) {
            const int p0 = b * S, p1 = (p0 + S) < gn ? (p0 + S) : gn;
            int cnt0 = 0, cnt1 = 0, cnt2 = 0, cnt3 = 0, cnt4 = 0;
            const unsigned long long below = (1ULL << lane) - 1ULL;
            for (int c0 = p0; c0 < p1; c0 += 64) {
                const int p = c0 + lane;
                // the exit side (FP32 records' Y loses its side bits here)
                int sdp = -2;
                if (p < p1) {
                    double Y;
                    sdp = side_of(gx[p], gy[p], gY[p], Y);
                    if constexpr (SIDE == SIDE_BITS) gY[p] = Y;
                }
                uint16_t *Lb = lst + (b * 4) * S;
                const unsigned long long m0 = __ballot(sdp == 0), m1 = __ballot(sdp == 1);
                const unsigned long long m2 = __ballot(sdp == 2), m3 = __ballot(sdp == 3);
                if (sdp == 0) Lb[0 * S + cnt0 + __popcll(m0 & below)] = (uint16_t)(p - p0);
                if (sdp == 1) Lb[1 * S + cnt1 + __popcll(m1 & below)] = (uint16_t)(p - p0);
                if (sdp == 2) Lb[2 * S + cnt2 + __popcll(m2 & below)] = (uint16_t)(p - p0);
                if (sdp == 3) Lb[3 * S + cnt3 + __popcll(m3 & below)] = (uint16_t)(p - p0);
                cnt0 += __popcll(m0); cnt1 += __popcll(m1); cnt2 += __popcll(m2); cnt3 += __popcll(m3);
                cnt4 += __popcll(__ballot(sdp == 4));
            }
            if (lane == 0) {
                s_lcnt[b * 4 + 0] = cnt0; s_lcnt[b * 4 + 1] = cnt1;
                s_lcnt[b * 4 + 2] = cnt2; s_lcnt[b * 4 + 3] = cnt3;
                // the item's exits per side
                atomicAdd(&s_cnt[0], (unsigned)cnt0); atomicAdd(&s_cnt[1], (unsigned)cnt1);
                atomicAdd(&s_cnt[2], (unsigned)cnt2); atomicAdd(&s_cnt[3], (unsigned)cnt3);
                atomicAdd(&s_cnt[4], (unsigned)cnt4);
                atomicAdd(&s_cnt[5], (unsigned)((p1 - p0) - (cnt0 + cnt1 + cnt2 + cnt3 + cnt4)));
            } else if (lane == 1) {
                // B sums of the sub-batch in path order
                double bs = 0.0, bb = 0.0;
                for (int p = p0; p < p1; ++p) { const double v = gs[p]; bs = bs + v; bb = __builtin_fma(v, v, bb); }
                s_bsb[b] = bs;
                s_bbsb[b] = bb;
            }
        }
        __syncthreads();
        // moments Phi[e][b] = sum over the exits of e's side in sub-batch b of Y phi_e(X)
        if (a.side_rbf) {
            // rectangle sides: a thread per (sub-batch, side, chunk of kRbfChunk entries) walks the
            // side's exits of the sub-batch in path order, forms the chunk's RBF values of each
            // (rbf_side_chunk) and adds Y phi into one register sum per entry -- per entry the
            // order of the direct form.  (Without the sums of the knot equations the branch of
            // rbf_side_chunk is the faster: 4 x 4 subdomains of 70 knots a side, sub-batches of 100, 8000
            // paths a knot 6.7 ms, 8.6 without it; with them the other is, 7.6 ms and 12.2)
            const int cb1 = (ms0 + kRbfChunk - 1) / kRbfChunk;
            const int cb2 = cb1 + (ms1 + kRbfChunk - 1) / kRbfChunk;
            const int cb3 = cb2 + (ms2 + kRbfChunk - 1) / kRbfChunk;
            const int cb4 = cb3 + (ms3 + kRbfChunk - 1) / kRbfChunk;
            for (int t = tid; t < nb * cb4; t += WG) {
                const int b = t / cb4, r = t - b * cb4;
                const int s = r < cb1 ? 0 : r < cb2 ? 1 : r < cb3 ? 2 : 3;
                const int m = msz_of(s);
                const int j0 = (r - pick(s, 0, cb1, cb2, cb3)) * kRbfChunk;
                const int len = (m - j0) < kRbfChunk ? (m - j0) : kRbfChunk;
                const int e0 = sd.ent_off + eoff_of(s);
                const double *px = tb.entx + e0, *py = tb.enty + e0;
                const double ic2 = tb.entic2[e0];
                double sx = 0.0, sy = 0.0, ss = 1.0;
                if (m > 1) {
                    sx = px[1] - px[0];
                    sy = py[1] - py[0];
                    ss = sx * sx + sy * sy;
                }
                const double q = dexp_tab_nonpos(-(2.0 * ss) * ic2, s_exp2);
                const uint16_t *L = lst + (b * 4 + s) * S;
                const int nl = s_lcnt[b * 4 + s];
                const int pb = b * S;
                double acc[kRbfChunk];
#pragma unroll
                for (int k = 0; k < kRbfChunk; ++k) acc[k] = 0.0;
                for (int l = 0; l < nl; ++l) {
                    const int p = pb + L[l];
                    rbf_side_chunk<!EQ>(px, py, j0, sx, sy, ss, q, gx[p], gy[p], ic2, s_exp2, gY[p], acc);
                }
#pragma unroll
                for (int k = 0; k < kRbfChunk; ++k)
                    if (k < len) Phi[(eoff_of(s) + j0 + k) * kNBG + b] = acc[k];
            }
        } else
        for (int e = tid; e < ne; e += WG) {
            const int se = tb.ents[sd.ent_off + e];
            const double pxe = tb.entx[sd.ent_off + e], pye = tb.enty[sd.ent_off + e];
            const double ic2 = tb.entic2[sd.ent_off + e];
            for (int b = 0; b < nb; ++b) {
                const uint16_t *L = lst + (b * 4 + se) * S;
                const int nl = s_lcnt[b * 4 + se];
                const int pb = b * S;
                double acc = 0.0;
                int l = 0;
                for (; l + 3 < nl; l += 4) {
                    const int pa = pb + L[l], pc = pb + L[l + 1], pd = pb + L[l + 2], pe = pb + L[l + 3];
                    const double fa = rbf_tab(pxe, pye, gx[pa], gy[pa], ic2, s_exp2);
                    const double fc = rbf_tab(pxe, pye, gx[pc], gy[pc], ic2, s_exp2);
                    const double fd = rbf_tab(pxe, pye, gx[pd], gy[pd], ic2, s_exp2);
                    const double fe = rbf_tab(pxe, pye, gx[pe], gy[pe], ic2, s_exp2);
                    acc = __builtin_fma(gY[pa], fa, acc);
                    acc = __builtin_fma(gY[pc], fc, acc);
                    acc = __builtin_fma(gY[pd], fd, acc);
                    acc = __builtin_fma(gY[pe], fe, acc);
                }
                for (; l < nl; ++l) {
                    const int pa = pb + L[l];
                    acc = __builtin_fma(gY[pa], rbf_tab(pxe, pye, gx[pa], gy[pa], ic2, s_exp2), acc);
                }
                Phi[e * kNBG + b] = acc;
            }
        }
        __syncthreads();
        double tp[kNBG];   // this thread's columns' sum of G_b,c u_ref (equation residual)
#pragma unroll
        for (int b = 0; b < kNBG; ++b) tp[b] = 0.0;
        for (int c = tid; c < nnz; c += WG) {
            double G[kNBG];
#pragma unroll
            for (int b = 0; b < kNBG; ++b) G[b] = 0.0;
            const int ec[2] = {tb.e1[sd.csr_off + c], tb.e2[sd.csr_off + c]};
            for (int q = 0; q < 2; ++q) {
                const int e = ec[q];
                if (e < 0) continue;
                const int se = tb.ents[sd.ent_off + e];
                const int m = msz_of(se);
                const int es = eoff_of(se);
                const int el = e - es;
                const double *A = tb.ipsi + ipsi_of(se) + el;
                const double2 *ph = (const double2 *)(Phi + es * kNBG);
                double H[kNBG];
#pragma unroll
                for (int b = 0; b < kNBG; ++b) H[b] = 0.0;
                // Psi^-1 column el, eight rows per batch of loads so that their latency overlaps
                int j = 0;
                for (; j + 8 <= m; j += 8) {
                    double av[8];
#pragma unroll
                    for (int u = 0; u < 8; ++u) av[u] = A[(int64_t)(j + u) * m];
#pragma unroll
                    for (int u = 0; u < 8; ++u) {
#pragma unroll
                        for (int b2 = 0; b2 < kNBG / 2; ++b2) {
                            const double2 v = ph[(j + u) * (kNBG / 2) + b2];
                            H[2 * b2] = __builtin_fma(av[u], v.x, H[2 * b2]);
                            H[2 * b2 + 1] = __builtin_fma(av[u], v.y, H[2 * b2 + 1]);
                        }
                    }
                }
                for (; j < m; ++j) {
                    const double aj = A[(int64_t)j * m];
#pragma unroll
                    for (int b2 = 0; b2 < kNBG / 2; ++b2) {
                        const double2 v = ph[j * (kNBG / 2) + b2];
                        H[2 * b2] = __builtin_fma(aj, v.x, H[2 * b2]);
                        H[2 * b2 + 1] = __builtin_fma(aj, v.y, H[2 * b2 + 1]);
                    }
                }
#pragma unroll
                for (int b = 0; b < kNBG; ++b) G[b] = G[b] + (-H[b]);
            }
            double sum = accS[c], q2 = accQ[c];
            for (int b = 0; b < nb; ++b) {
                const int p0 = (g + b) * S;
                const int p1 = (p0 + S) < it.n ? (p0 + S) : it.n;
                sum = sum + G[b];
                q2 = q2 + (G[b] * G[b]) / (double)(p1 - p0);
            }
            accS[c] = sum;
            accQ[c] = q2;
            if constexpr (EQ) {
                const double wc = a.wref[kd.out_off + c];
#pragma unroll
                for (int b = 0; b < kNBG; ++b) tp[b] = __builtin_fma(G[b], wc, tp[b]);
            }
        }
        if constexpr (EQ) {
            // sum over the columns: a butterfly over each wave, then the waves in order
#pragma unroll
            for (int b = 0; b < kNBG; ++b) {
                double v = tp[b];
                for (int off = 32; off > 0; off >>= 1) v = v + __shfl_xor(v, off);
                if (lane == 0) s_wsum[wave * kNBG + b] = v;
            }
            __syncthreads();
        }
        if (tid == 0) {
            for (int b = 0; b < nb; ++b) { Bs = Bs + s_bsb[b]; BBs = BBs + s_bbsb[b]; }
            if constexpr (EQ)
                for (int b = 0; b < nb; ++b) {
                    double T = 0.0;
                    for (int w = 0; w < nwaves; ++w) T = T + s_wsum[w * kNBG + b];
                    const int p0 = (g + b) * S;
                    const int p1 = (p0 + S) < it.n ? (p0 + S) : it.n;
                    const double R = s_bsb[b] - T;
                    Rs = Rs + R;
                    RQs = RQs + (R * R) / (double)(p1 - p0);
                }
        }
        __syncthreads();
    }
    for (int c = tid; c < nnz; c += WG) {
        a.partials[it.part_off + c] = accS[c];
        a.partials[it.part_off + nnz + c] = accQ[c];
    }
    if (tid == 0) {
        ItemStat st;
        st.Bs = Bs;
        st.BBs = BBs;
        st.Rs = Rs;
        st.RQs = RQs;
        for (int q = 0; q < 6; ++q) st.cnt[q] = s_cnt[q];
        a.stats[item] = st;
    }
}

template <bool EQ, int SIDE> static hipError_t launch_reduce_t(int grid, int wg, size_t shmem, hipStream_t s,
                                                            const ReduceArgs &a) {
    if (shmem > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute((const void *)reduce_kernel<EQ, SIDE>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)shmem);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL((reduce_kernel<EQ, SIDE>), dim3(grid), dim3(wg), shmem, s, a);
    return hipGetLastError();
}

template <bool EQ> static hipError_t launch_reduce_eq(int grid, int wg, size_t shmem, hipStream_t s, const ReduceArgs &a) {
    switch (a.side_mode) {
        case SIDE_BITS: return launch_reduce_t<EQ, SIDE_BITS>(grid, wg, shmem, s, a);
        case SIDE_RECT: return launch_reduce_t<EQ, SIDE_RECT>(grid, wg, shmem, s, a);
        case SIDE_DISC: return launch_reduce_t<EQ, SIDE_DISC>(grid, wg, shmem, s, a);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_reduce(int grid, int wg, size_t shmem, hipStream_t s, const ReduceArgs &a) {
    return a.wref ? launch_reduce_eq<true>(grid, wg, shmem, s, a) : launch_reduce_eq<false>(grid, wg, shmem, s, a);
}

// v / n for a whole n >= 1 that is the same for the whole wave: a power of two divides exactly by a
// multiplication, a tenth of a division's time
__device__ __forceinline__ double over_count(double v, int n) {
    if ((n & (n - 1)) == 0) return v * __builtin_bit_cast(double, (uint64_t)(1023 - __builtin_ctz(n)) << 52);
    return v / (double)n;
}

typedef double d4 __attribute__((ext_vector_type(4)));

// Values and pointers read from descriptors, the same for the whole wave, moved to scalar registers
// (the compiler keeps a value loaded behind a store in vector registers, and loads through it flat).
template <class T> __device__ __forceinline__ T wave_uniform(T v) {
    if constexpr (sizeof(T) == 4) {
        return __builtin_bit_cast(T, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, v)));
    } else {
        const uint64_t b = __builtin_bit_cast(uint64_t, v);
        const uint32_t lo = __builtin_amdgcn_readfirstlane((int)(uint32_t)b), hi = __builtin_amdgcn_readfirstlane((int)(uint32_t)(b >> 32));
        return __builtin_bit_cast(T, (uint64_t)hi << 32 | lo);
    }
}
template <class T> using global_ptr = const __attribute__((address_space(1))) T *;
template <class T> __device__ __forceinline__ global_ptr<T> wave_global(const T *p) {
    return (global_ptr<T>)wave_uniform((uint64_t)p);
}

// The reduction by groups of 16 sub-batches, for the stencils and sub-batches of reduce16_fits: the
// same sums in the same order as reduce_kernel's, so the same bits.  A work-group takes a span of
// items of one knot (ItemDesc::span_first), which need not end where a group does.
//  * records are read once, a wave 64 consecutive paths at a time and two such pieces ahead; the side
//    of each exit is found in registers and its place in the list of its (sub-batch, side) by ballots.
//  * moments: as in reduce_kernel, with the 16 sub-batches of one side chunk on neighbouring lanes,
//    whose lists are about equally long.
//  * H = Psi^-T Phi is a matrix product, 16 side entries x 16 sub-batches x the side's entries, on
//    v_mfma_f64_16x16x4: its four products are added one after another, each with one rounding, as
//    the ascending fma chain of reduce_kernel (the vector units' rate is no lower, but a chain of
//    fma's needs an LDS read of 16 bytes a lane for every two, and the LDS bounded it).
//  * H goes back through the LDS, in Phi's place, to a thread per CSR column.
// Phi and H lie in the LDS as [entry][16 sub-batches], the sub-batches of a row permuted by its
// number (phi_at), so that rows and columns are both read without bank conflicts.
// Bound by issuing the exponentials and recurrences of the moments (about 180 instructions per exit
// and 16 entries, on lanes whose lists are of unequal length), then the matrix product.  344 10^6
// paths (S = 32, 3437 knots of about 260 entries, FP32
// records): 39 ms, reduce_kernel 57 ms; 9807 knots of a disc with 32 10^6 paths and equation sums:
// 9.9 ms, reduce_kernel 27 ms.  Work-groups of 4 waves: of 5 to 8, fewer stay on a CU at once
// (1.4 instead of 2, 60 ms).  Up to 16 tiles three of them fit a CU; more tiles, and equation sums,
// take the registers of two.
__device__ __forceinline__ int phi_at(int e, int b) { return e * kGroup16 + (b ^ (e & 15)); }

template <bool EQ, int SIDE, int TW>
__global__ void __launch_bounds__(kReduceWG) __attribute__((amdgpu_waves_per_eu(EQ || TW > kSmallTiles / 4 ? 2 : 3))) reduce16_kernel(ReduceArgs a) {
    constexpr int NB = kGroup16, WG = kReduceWG, NW = WG / 64;
    static_assert(kRbfChunk == 16, "a chunk of the recurrence is a tile");
    // 16 entries of a side: the side's entries m, the first of the tile j0 and of the side e0 (in the
    // stencil), the side s
    struct Tile { int m, j0, e0, s; };
    extern __shared__ __align__(16) double smem[];
    __shared__ double s_bsb[NB], s_bbsb[NB];
    __shared__ double s_wsum[EQ ? NW * NB : 1];
    __shared__ double s_exp2[64];
    __shared__ int s_lcnt[NB * 6];               // exits per (sub-batch, side 0..4), and with no side
    __shared__ ItemStat s_stat[kSpanItems];      // the items' sums
    __shared__ Tile s_tile[TW * NW];
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const ItemDesc *items = a.items;
    const int64_t item0 = wave_uniform(items[a.item_base + (int64_t)blockIdx.x].span_first);
    const int n_items = wave_uniform(items[a.item_base + (int64_t)blockIdx.x].span_count);
    const int it_n = wave_uniform(items[item0].n);
    const int64_t part_off = wave_uniform(items[item0].part_off);
    const KnotDesc &kd = a.knots[wave_uniform(items[item0].knot)];
    const TableDesc &tb = a.tables[wave_uniform(kd.table)];
    const StencilDesc &sd = wave_uniform(tb.sten)[wave_uniform(kd.stencil)];
    const global_ptr<double> entx = wave_global(tb.entx), enty = wave_global(tb.enty), entic2 = wave_global(tb.entic2);
    const global_ptr<double> ipsi = wave_global(tb.ipsi);
    const int ent = wave_uniform(sd.ent_off), nnz = wave_uniform(sd.csr_nnz);
    const global_ptr<int32_t> ce1 = wave_global(tb.e1 + sd.csr_off), ce2 = wave_global(tb.e2 + sd.csr_off);
    const global_ptr<double> wref = wave_global(EQ ? a.wref + kd.out_off : nullptr);
    const global_ptr<ExitRec> rr = wave_global(a.rec.r + (kd.path_off + items[item0].p_begin));
    double dom[6];
#pragma unroll
    for (int i = 0; i < (SIDE == SIDE_DISC ? 6 : 4); ++i) dom[i] = wave_uniform(kd.dom[i]);
    const int ms0 = wave_uniform(sd.msz[0]), ms1 = wave_uniform(sd.msz[1]), ms2 = wave_uniform(sd.msz[2]);
    const int ms3 = wave_uniform(sd.msz[3]);
    const int S = a.S;
    const int np = n_items > 1 ? it_n * (n_items - 1) + wave_uniform(items[item0 + n_items - 1].n) : it_n;
    const int nsb = (np + S - 1) / S;                        // sub-batches of the span
    const int qi = n_items > 1 ? it_n / S : nsb;             // of an item (the last may have fewer)
    const int ne = ms0 + ms1 + ms2 + ms3;
    // tiles up to and with each side
    const int t1 = (ms0 + 15) >> 4, t2 = t1 + ((ms1 + 15) >> 4), t3 = t2 + ((ms2 + 15) >> 4), t4 = t3 + ((ms3 + 15) >> 4);
    double *Phi = smem;                                      // [ne][NB], then H
    double *gx = smem + NB * a.ne_cap;
    double *gy = gx + NB * S;
    double *gY = gy + NB * S;
    double *gs = gY + NB * S;                                // [NB][S + 1]
    uint8_t *lst = (uint8_t *)(gs + NB * (S + 1));           // [NB][S], the sides' lists one behind another
    if (tid < 64) s_exp2[tid] = kExp2TabDev[tid];
    if (tid < t4) {
        const int s = tid < t1 ? 0 : tid < t2 ? 1 : tid < t3 ? 2 : 3;
        Tile t;
        t.s = s;
        t.m = s == 0 ? ms0 : s == 1 ? ms1 : s == 2 ? ms2 : ms3;
        t.j0 = (tid - (s == 0 ? 0 : s == 1 ? t1 : s == 2 ? t2 : t3)) * 16;
        t.e0 = s == 0 ? 0 : s == 1 ? ms0 : s == 2 ? ms0 + ms1 : ms0 + ms1 + ms2;
        s_tile[tid] = t;
    }
    if (tid < kSpanItems) {
        const ItemStat z = {0.0, 0.0, 0.0, 0.0, {0, 0, 0, 0, 0, 0}};
        s_stat[tid] = z;
    }
    auto side_of = [&](double x, double y, double Yr, double &Y) -> int {
        if constexpr (SIDE == SIDE_BITS) {
            const uint64_t yb = __builtin_bit_cast(uint64_t, Yr);
            Y = __builtin_bit_cast(double, yb & ~kSideBitsMask);
            return (int)(yb & kSideBitsMask) - 1;
        }
        Y = Yr;
        if constexpr (SIDE == SIDE_DISC) return classify_sector(dom, a.gc[0], x, y);
        else return classify_coord_c(dom, a.gc, x, y);
    };
    // a piece of records: 64 paths, whole sub-batches of them (S divides 64) or a sub-batch's next 64
    const bool whole = S <= 64 && 64 % S == 0;
    const int usb = whole ? 64 / S : 1;                      // sub-batches of a piece
    const int uS = whole ? 64 : S;                           // paths of them
    const int chunks = (uS + 63) >> 6;                       // pieces of a sub-batch
    const int seg = whole ? lane / S : 0;                    // this lane's sub-batch of the piece
    const unsigned long long segm = whole && S < 64 ? ((1ULL << S) - 1ULL) << (seg * S) : ~0ULL;
    const unsigned long long before = segm & ((1ULL << lane) - 1ULL);
    // piece v of this wave: chunk v % chunks of the sub-batches from usb (wave + NW (v / chunks))
    auto load_piece = [&](int q0, int gn, int v) -> ExitRec {
        const int u = chunks == 1 ? v : v / chunks, c = v - u * chunks;
        const int o = c * 64 + lane, p = (wave + NW * u) * uS + o;
        ExitRec r = {0.0, 0.0, 0.0, 0.0};
        if (o < uS && p < gn) {
            const global_ptr<ExitRec> q = rr + q0 + p;
            r.x = q->x; r.y = q->y; r.Y = q->Y; r.score = q->score;
        }
        return r;
    };
    ExitRec recA = load_piece(0, np < NB * S ? np : NB * S, 0), recB = load_piece(0, np < NB * S ? np : NB * S, 1);
    __syncthreads();
    int il = 0, left = qi;                                   // item of the next sub-batch, its sub-batches left
    for (int g = 0; g < nsb; g += NB) {
        const int nb = (nsb - g) < NB ? (nsb - g) : NB;
        const int q0 = g * S;                                // first path of the group
        const int gn = (np - q0) < nb * S ? (np - q0) : nb * S;
        const int units = (nb + usb - 1) / usb;
        const int nv = units > wave ? (units - wave + NW - 1) / NW * chunks : 0;
        int n0 = 0, n1 = 0, n2 = 0, n3 = 0, n4 = 0, nn = 0;
        auto piece = [&](const ExitRec &rc, int v) {
            const int u = chunks == 1 ? v : v / chunks, c = v - u * chunks;
            const int o = c * 64 + lane, b = (wave + NW * u) * usb + seg, p = (wave + NW * u) * uS + o;
            double Y = 0.0;
            int s = -2;
            if (o < uS && p < gn) {
                s = side_of(rc.x, rc.y, rc.Y, Y);
                gx[p] = rc.x;
                gy[p] = rc.y;
                gY[p] = Y;
                gs[p + b] = rc.score;
            }
            const unsigned long long m0 = __ballot(s == 0) & segm, m1 = __ballot(s == 1) & segm;
            const unsigned long long m2 = __ballot(s == 2) & segm, m3 = __ballot(s == 3) & segm;
            const unsigned long long m4 = __ballot(s == 4) & segm, mn = __ballot(s == -1) & segm;
            const int c0 = __popcll(m0), c1 = __popcll(m1), c2 = __popcll(m2), c3 = __popcll(m3);
            if (s >= 0 && s < 4) {
                const unsigned long long ms = s == 0 ? m0 : s == 1 ? m1 : s == 2 ? m2 : m3;
                int at = __popcll(ms & before);
                // (the lists of longer sub-batches, whose lengths come out at their end, lie S apart)
                if (whole) at += s == 0 ? 0 : s == 1 ? c0 : s == 2 ? c0 + c1 : c0 + c1 + c2;
                else at += s == 0 ? n0 : s == 1 ? S + n1 : s == 2 ? 2 * S + n2 : 3 * S + n3;
                lst[b * (whole ? S : 4 * S) + at] = (uint8_t)(p - b * S);
            }
            n0 += c0;
            n1 += c1;
            n2 += c2;
            n3 += c3;
            n4 += __popcll(m4);
            nn += __popcll(mn);
            if (c == chunks - 1) {
                if (b < nb && lane == seg * S) {
                    int *lc = s_lcnt + b * 6;
                    lc[0] = n0; lc[1] = n1; lc[2] = n2; lc[3] = n3; lc[4] = n4; lc[5] = nn;
                }
                n0 = n1 = n2 = n3 = n4 = nn = 0;
            }
        };
        for (int v = 0; v < nv; v += 2) {
            piece(recA, v);
            if (v + 2 < nv) recA = load_piece(q0, gn, v + 2);
            if (v + 1 < nv) {
                piece(recB, v + 1);
                if (v + 3 < nv) recB = load_piece(q0, gn, v + 3);
            }
        }
        if (g + NB < nsb) {
            const int q1 = q0 + NB * S, rest = np - q1 < NB * S ? np - q1 : NB * S;
            recA = load_piece(q1, rest, 0);
            recB = load_piece(q1, rest, 1);
        }
        __syncthreads();
        if (wave == NW - 1 && lane < nb) {
            // B sums of a sub-batch in path order
            const int n = gn - lane * S < S ? gn - lane * S : S;
            const double *v = gs + lane * (S + 1);
            double bs = 0.0, bb = 0.0;
#pragma unroll 8
            for (int p = 0; p < n; ++p) { bs = bs + v[p]; bb = __builtin_fma(v[p], v[p], bb); }
            s_bsb[lane] = bs;
            s_bbsb[lane] = bb;
        }
        // list of a (sub-batch, side)
        auto list_of = [&](int b, int s) -> const uint8_t * {
            const int *lc = s_lcnt + b * 6;
            if (!whole) return lst + (b * 4 + s) * S;
            return lst + b * S + (s > 0 ? lc[0] : 0) + (s > 1 ? lc[1] : 0) + (s > 2 ? lc[2] : 0);
        };
        // moments Phi[e][b]
        if (a.side_rbf) {
            // (the wave that takes a remainder differs between neighbouring work-groups: each sits on
            // a SIMD of its own)
            for (int t = (tid + 64 * blockIdx.x) & (WG - 1); t < nb * t4; t += WG) {
                const int r = nb == NB ? t / NB : t / nb, b = t - r * nb;
                const Tile ti = s_tile[r];
                const int len = ti.m - ti.j0;
                const global_ptr<double> px = entx + ent, py = enty + ent;
                const double ic2 = entic2[ent + ti.e0];
                const double x0 = px[ti.e0 + ti.j0], y0 = py[ti.e0 + ti.j0];
                double sx = 0.0, sy = 0.0, ss = 1.0;
                if (ti.m > 1) {
                    sx = px[ti.e0 + 1] - px[ti.e0];
                    sy = py[ti.e0 + 1] - py[ti.e0];
                    ss = sx * sx + sy * sy;
                }
                const double q = dexp_tab_nonpos(-(2.0 * ss) * ic2, s_exp2);
                const uint8_t *L = list_of(b, ti.s);
                const int nl = s_lcnt[b * 6 + ti.s];
                const int pb = b * S;
                double acc[kRbfChunk];
#pragma unroll
                for (int k = 0; k < kRbfChunk; ++k) acc[k] = 0.0;
                for (int l = 0; l < nl; ++l) {
                    const int p = pb + L[l];
                    rbf_side_chunk(&x0, &y0, 0, sx, sy, ss, q, gx[p], gy[p], ic2, s_exp2, gY[p], acc);
                }
                const int e = ti.e0 + ti.j0;
#pragma unroll
                for (int k = 0; k < kRbfChunk; ++k)
                    if (k < len) Phi[phi_at(e + k, b)] = acc[k];
            }
        } else {
            const int ec = (ne + 63) >> 6;
            for (int t = wave; t < ec * nb; t += NW) {
                // (64 entries of a sub-batch; each wave goes through all the 64's, whose exits differ)
                const int b = t / ec, e = (t + b) % ec * 64 + lane;
                if (e >= ne) continue;
                const int s = e < ms0 ? 0 : e < ms0 + ms1 ? 1 : e < ms0 + ms1 + ms2 ? 2 : 3;
                const double pxe = entx[ent + e], pye = enty[ent + e], ic2 = entic2[ent + e];
                const uint8_t *L = list_of(b, s);
                const int nl = s_lcnt[b * 6 + s];
                const int pb = b * S;
                double acc = 0.0;
                int l = 0;
                for (; l + 3 < nl; l += 4) {
                    int p[4];
                    double x[4], y[4], f[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u) p[u] = pb + L[l + u];
#pragma unroll
                    for (int u = 0; u < 4; ++u) { x[u] = gx[p[u]]; y[u] = gy[p[u]]; }
                    rbf_tab4(pxe, pye, x, y, ic2, s_exp2, f);
#pragma unroll
                    for (int u = 0; u < 4; ++u) acc = __builtin_fma(gY[p[u]], f[u], acc);
                }
                for (; l < nl; ++l) {
                    const int pa = pb + L[l];
                    acc = __builtin_fma(gY[pa], rbf_tab(pxe, pye, gx[pa], gy[pa], ic2, s_exp2), acc);
                }
                Phi[phi_at(e, b)] = acc;
            }
        }
        // H = Psi^-T Phi: lane (mi, mk) holds row mk of column mi of Psi^-1's 4 x 16 piece and row mk
        // of Phi's sub-batch mi; register r of the result is entry 4 r + mk of sub-batch mi.  A batch
        // is 16 rows; the next one, also a tile's first, is loaded while the last is multiplied
        const int mi = lane & 15, mk = lane >> 4;
        d4 H[TW];
        int wt = wave;                                       // (opaque: no tile's addresses are kept over the groups)
        asm volatile("" : "+s"(wt));
        // batch j of the tile r: 16 rows from 16 j on, four base addresses and one offset for Psi^-1
        double av[4], bv[4], an[4], bn[4];
        int m = 1, nbat = 0;
        uint32_t ao = 0;
        global_ptr<double> A = ipsi;
        const double *ph[4];
        auto open_tile = [&](int r) {
            m = wave_uniform(s_tile[r].m);
            nbat = (m + 15) >> 4;
            const int j0 = wave_uniform(s_tile[r].j0), e = wave_uniform(s_tile[r].e0) + mk;
            A = ipsi + wave_uniform(sd.ipsi_off[wave_uniform(s_tile[r].s)]);
            ao = (uint32_t)(mk * m + (j0 + mi < m ? j0 + mi : m - 1));
#pragma unroll
            for (int q = 0; q < 4; ++q) ph[q] = Phi + phi_at(e + 4 * q, mi);
        };
        auto load_a = [&](int j, double (&x)[4]) {
            const uint32_t o = ao + (uint32_t)(16 * j) * (uint32_t)m;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t w = o + (uint32_t)(4 * q) * (uint32_t)m;
                x[q] = A[j + 1 < nbat || 16 * j + 4 * q + mk < m ? w : 0u];
            }
        };
        auto load_b = [&](int j, double (&x)[4]) {
#pragma unroll
            for (int q = 0; q < 4; ++q) x[q] = *(j + 1 < nbat || 16 * j + 4 * q + mk < m ? ph[q] + 256 * j : Phi);
        };
        d4 h;
        auto multiply = [&](int j, const double (&x)[4], const double (&y)[4]) {
            if (j + 1 < nbat) {
#pragma unroll
                for (int q = 0; q < 4; ++q) h = __builtin_amdgcn_mfma_f64_16x16x4f64(x[q], y[q], h, 0, 0, 0);
            } else {
                // the side's last rows; those past its end are zeros
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    if (16 * j + 4 * q >= m) break;
                    const bool in = 16 * j + 4 * q + mk < m;
                    h = __builtin_amdgcn_mfma_f64_16x16x4f64(in ? x[q] : 0.0, in ? y[q] : 0.0, h, 0, 0, 0);
                }
            }
        };
        if (wt < t4) {
            open_tile(wt);
            load_a(0, av);
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < TW; ++u) {
            const int r = wt + u * NW;
            if (r >= t4) break;
            h = d4{0.0, 0.0, 0.0, 0.0};
            if (u > 0) {
                open_tile(r);
                load_a(0, av);
            }
            load_b(0, bv);
            for (int j = 0;;) {
                if (j + 1 < nbat) { load_a(j + 1, an); load_b(j + 1, bn); }
                multiply(j, av, bv);
                if (++j == nbat) break;
                if (j + 1 < nbat) { load_a(j + 1, av); load_b(j + 1, bv); }
                multiply(j, an, bn);
                if (++j == nbat) break;
            }
            H[u] = h;
        }
        if (wave == NW - 1) {
            // the group's scores and exits join their items, an item per lane
            const int b0 = lane == il ? 0 : left + (lane - il - 1) * qi, b1 = lane == il ? left : b0 + qi;
            if (lane >= il && lane < n_items && b0 < nb) {
                ItemStat &st = s_stat[lane];
                for (int b = b0; b < b1 && b < nb; ++b) {
                    st.Bs = st.Bs + s_bsb[b];
                    st.BBs = st.BBs + s_bbsb[b];
                    for (int q = 0; q < 6; ++q) st.cnt[q] += (uint32_t)s_lcnt[b * 6 + q];
                }
            }
        }
        // a column's two entries, and its sums so far of the item that the last group ended in (this
        // thread's first column's are loaded before they are waited for)
        double *part = a.partials + part_off;
        int r1 = -1, r2 = -1;
        double aS = 0.0, aQ = 0.0;
        auto load_col = [&](int c) {
            if (c < nnz) {
                r1 = ce1[c];
                r2 = ce2[c];
                if (left < qi) {
                    aS = part[(int64_t)il * 2 * nnz + c];
                    aQ = part[(int64_t)il * 2 * nnz + nnz + c];
                }
            }
        };
        load_col(tid);
        __syncthreads();
        asm volatile("" : "+s"(wt));
#pragma unroll
        for (int u = 0; u < TW; ++u) {
            const int r = wt + u * NW;
            if (r >= t4) break;
            const Tile ti = s_tile[r];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int el = ti.j0 + mk + 4 * q;
                if (el < ti.m) Phi[phi_at(ti.e0 + el, mi)] = H[u][q];
            }
        }
        __syncthreads();
        const bool full = gn == NB * S && (S & (S - 1)) == 0;
        const double invS = __builtin_bit_cast(double, (uint64_t)(1023 - __builtin_ctz(S)) << 52);
        double tp[EQ ? NB : 1];    // this thread's columns' sum of G_b,c u_ref (equation residual)
        if constexpr (EQ)
#pragma unroll
            for (int b = 0; b < NB; ++b) tp[b] = 0.0;
        for (int c = tid; c < nnz; c += WG) {
            if (c >= WG) load_col(c);
            auto g_of = [&](int b) -> double {
                double G = 0.0;
                if (r1 >= 0) G = G + (-Phi[phi_at(r1, b)]);
                if (r2 >= 0) G = G + (-Phi[phi_at(r2, b)]);
                return G;
            };
            for (int b = 0, i = il, lf = left; b < nb; ++i, lf = qi) {
                const int b1 = b + lf < nb ? b + lf : nb;
                if (b1 - b == NB && full) {                  // a group of full sub-batches of one item
                    double G[NB];
#pragma unroll
                    for (int bb = 0; bb < NB; ++bb) G[bb] = g_of(bb);
#pragma unroll
                    for (int bb = 0; bb < NB; ++bb) {
                        aS = aS + G[bb];
                        aQ = aQ + G[bb] * G[bb] * invS;
                    }
                    b = NB;
                }
#pragma unroll 4
                for (int bb = b; bb < b1; ++bb) {
                    const double G = g_of(bb);
                    const int n = gn - bb * S < S ? gn - bb * S : S;
                    aS = aS + G;
                    aQ = aQ + over_count(G * G, n);
                }
                double *out = part + (int64_t)i * 2 * nnz + c;
                out[0] = aS;
                out[nnz] = aQ;
                aS = aQ = 0.0;
                b = b1;
            }
            if constexpr (EQ) {
                const double wc = wref[c];
#pragma unroll
                for (int b = 0; b < NB; ++b) tp[b] = __builtin_fma(g_of(b), wc, tp[b]);
            }
        }
        if constexpr (EQ) {
            // sum over the columns: a butterfly over each wave, then the waves in order.  The
            // butterfly's first four stages halve the sub-batches a lane still sums: lane 4 b has
            // sub-batch b's
#pragma unroll
            for (int off = 32, hb = NB / 2; off >= 4; off >>= 1, hb >>= 1) {
                const bool hi = (lane & off) != 0;
#pragma unroll
                for (int b = 0; b < hb; ++b) {
                    const double send = hi ? tp[b] : tp[b + hb], keep = hi ? tp[b + hb] : tp[b];
                    tp[b] = keep + __shfl_xor(send, off);
                }
            }
            double v = tp[0];
            v = v + __shfl_xor(v, 2);
            v = v + __shfl_xor(v, 1);
            if ((lane & 3) == 0) s_wsum[wave * NB + (lane >> 2)] = v;
            __syncthreads();
            if (wave == 0) {
                double R = 0.0, RQ = 0.0;
                if (lane < nb) {
                    double T = 0.0;
                    for (int w = 0; w < NW; ++w) T = T + s_wsum[w * NB + lane];
                    R = s_bsb[lane] - T;
                    const int n = gn - lane * S;
                    RQ = n < S ? (R * R) / (double)n : over_count(R * R, S);
                }
                const int b0 = lane == il ? 0 : left + (lane - il - 1) * qi, b1 = lane == il ? left : b0 + qi;
                const bool own = lane >= il && lane < n_items;
                double r = own ? s_stat[lane].Rs : 0.0, rq = own ? s_stat[lane].RQs : 0.0;
                for (int b = 0; b < nb; ++b) {
                    const double r1 = __shfl(R, b), r2 = __shfl(RQ, b);
                    if (own && b >= b0 && b < b1) { r = r + r1; rq = rq + r2; }
                }
                if (own) { s_stat[lane].Rs = r; s_stat[lane].RQs = rq; }
            }
        }
        // (the next group's moments are written behind its first barrier)
        if (nb < left) {
            left -= nb;
        } else {
            const int over = nb - left;
            il += 1 + over / qi;
            left = qi - over % qi;
        }
    }
    __syncthreads();
    if (tid < n_items) a.stats[item0 + tid] = s_stat[tid];
}

template <bool EQ, int SIDE, int TW> static hipError_t launch_reduce16_t(int grid, size_t shmem, hipStream_t s, const ReduceArgs &a) {
    if (shmem > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute((const void *)reduce16_kernel<EQ, SIDE, TW>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)shmem);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL((reduce16_kernel<EQ, SIDE, TW>), dim3(grid), dim3(kReduceWG), shmem, s, a);
    return hipGetLastError();
}

template <bool EQ, int TW> static hipError_t launch_reduce16_eq(int grid, size_t shmem, hipStream_t s, const ReduceArgs &a) {
    switch (a.side_mode) {
        case SIDE_BITS: return launch_reduce16_t<EQ, SIDE_BITS, TW>(grid, shmem, s, a);
        case SIDE_RECT: return launch_reduce16_t<EQ, SIDE_RECT, TW>(grid, shmem, s, a);
        case SIDE_DISC: return launch_reduce16_t<EQ, SIDE_DISC, TW>(grid, shmem, s, a);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_reduce16(bool small, int grid, size_t shmem, hipStream_t s, const ReduceArgs &a) {
    constexpr int SMALL = kSmallTiles * 64 / kReduceWG, LARGE = kMaxTiles * 64 / kReduceWG;
    if (small) return a.wref ? launch_reduce16_eq<true, SMALL>(grid, shmem, s, a) : launch_reduce16_eq<false, SMALL>(grid, shmem, s, a);
    return a.wref ? launch_reduce16_eq<true, LARGE>(grid, shmem, s, a) : launch_reduce16_eq<false, LARGE>(grid, shmem, s, a);
}

// One block per knot: sum the knot's items in item order.
__global__ void __launch_bounds__(256) finalize_kernel(FinalizeArgs f) {
    const int k = blockIdx.x;
    if (k >= f.n_knots) return;
    const KnotDesc kd = f.knots[k];
    const StencilDesc &sd = f.tables[kd.table].sten[kd.stencil];
    const int nnz = sd.csr_nnz;
    const int64_t w0 = kd.item_begin, w1 = kd.item_begin + kd.item_count;
    const double N = (double)kd.n_paths;
    const int64_t nb = (kd.n_paths + f.S - 1) / f.S;
    for (int c = threadIdx.x; c < nnz; c += blockDim.x) {
        double sum = 0.0, q2 = 0.0;
        for (int64_t w = w0; w < w1; ++w) {
            const int64_t off = f.items[w].part_off;
            sum = sum + f.partials[off + c];
            q2 = q2 + f.partials[off + nnz + c];
        }
        const double G = sum / N;
        f.G[kd.out_off + c] = G;
        f.Gvar[kd.out_off + c] = nb > 1 ? (q2 - N * G * G) / (double)(nb - 1) : 0.0;
    }
    if (threadIdx.x == 0) {
        double Bs = 0.0, BBs = 0.0, Rs = 0.0, RQs = 0.0;
        KnotStat ks;
        ks.steps = f.kacc[2 * (int64_t)k];
        ks.capped = f.kacc[2 * (int64_t)k + 1];
        for (int q = 0; q < 6; ++q) ks.cnt[q] = 0;
        for (int64_t w = w0; w < w1; ++w) {
            const ItemStat st = f.stats[w];
            Bs = Bs + st.Bs;
            BBs = BBs + st.BBs;
            Rs = Rs + st.Rs;
            RQs = RQs + st.RQs;
            for (int q = 0; q < 6; ++q) ks.cnt[q] += st.cnt[q];
        }
        ks.B = Bs / N;
        ks.BB = BBs / N;
        ks.Rm = Rs / N;
        ks.Rv = nb > 1 ? (RQs - N * ks.Rm * ks.Rm) / (double)(nb - 1) : 0.0;
        f.kstats[k] = ks;
    }
}

hipError_t launch_finalize(int grid, int wg, hipStream_t s, const FinalizeArgs &f) {
    hipLaunchKernelGGL(finalize_kernel, dim3(grid), dim3(wg), 0, s, f);
    return hipGetLastError();
}

// Sets n 64-bit words to v: the path queues' counters are cleared by a kernel rather than a
// memset node, so the sequence stays capturable in a HIP graph.
__global__ void fill_u64_kernel(unsigned long long *p, int64_t n, unsigned long long v) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

hipError_t launch_fill_u64(unsigned long long *p, int64_t n, unsigned long long v, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    const int wg = 256;
    hipLaunchKernelGGL(fill_u64_kernel, dim3((unsigned)((n + wg - 1) / wg)), dim3(wg), 0, s, p, n, v);
    return hipGetLastError();
}

__global__ void lut_eval_kernel(LutView L, int field, int64_t n, const double *x, const double *y, double *out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double v[8];
    if (L.nf > 5) lut_eval<double, 8>(L, x[i], y[i], v);
    else if (L.nf == 5) lut_eval<double, 5>(L, x[i], y[i], v);
    else lut_eval<double, 4>(L, x[i], y[i], v);
    out[i] = v[field];
}

hipError_t launch_lut_eval(const LutView &L, int field, int64_t n, const double *x, const double *y, double *out,
                           hipStream_t s) {
    int wg = 256;
    int64_t grid = (n + wg - 1) / wg;
    hipLaunchKernelGGL(lut_eval_kernel, dim3((unsigned)grid), dim3(wg), 0, s, L, field, n, x, y, out);
    return hipGetLastError();
}

}  // namespace pdds
