// engine_types.h -- device-resident descriptors shared by host and kernels.
#pragma once
#include <stdint.h>
#include "pdds_pde.h"

namespace pdds {

constexpr int kNBG = 8;                    // sub-batches reduced per pass over Psi^-1
constexpr int kReduceWG = 256;            // reduction work-group
constexpr int kRbfChunk = 16;             // side entries per direct exponential (rectangle sides)

// LDS of the reduction kernel: Phi [ne_cap][kNBG], accS/accQ [nnz_cap] (FP64), the group's
// records x, y, Y and score [kNBG*S] (FP64) and per-(sub-batch, side) path lists [kNBG][4][S]
// (uint16)
inline size_t reduce_lds_bytes(int ne_cap, int nnz_cap, int S) {
    const size_t g = (size_t)kNBG * S;
    size_t b = ((size_t)kNBG * ne_cap + 2 * (size_t)nnz_cap + 4 * g) * sizeof(double);
    b += g * 4 * sizeof(uint16_t);
    return (b + 15) & ~(size_t)15;
}

// The reduction of groups of 16 sub-batches (reduce16_kernel): its LDS holds Phi [ne_cap][16], the
// group's x, y, Y [16 S] and score [16 (S + 1)] (FP64) and the path lists (bytes: [16][S], or
// [16][4][S] where S does not divide 64).  It takes stencils of at most kMaxTiles tiles of 16 side
// entries, and sub-batches whose group leaves room for two work-groups on a CU; stencils of up to
// kSmallTiles leave room for three.
constexpr int kGroup16 = 16;
constexpr int kSmallTiles = 16, kMaxTiles = 32;
constexpr int kSpanItems = 16;            // work items of one knot a work-group may take
inline size_t reduce16_lds_bytes(int ne_cap, int S) {
    const size_t g = (size_t)kGroup16 * S;
    const size_t b = ((size_t)kGroup16 * ne_cap + 4 * g + kGroup16) * sizeof(double) + (S <= 64 && 64 % S == 0 ? g : 4 * g);
    return (b + 15) & ~(size_t)15;
}
inline bool reduce16_fits(int ne, int tiles, int S) {
    return S <= 256 && reduce16_lds_bytes(ne, S) <= 76 * 1024 && tiles <= kMaxTiles;
}
// The reduction of a stencil: by reduce16_kernel, of up to kSmallTiles tiles or more, or by reduce_kernel
enum ReduceClass { REDUCE16_SMALL = 0, REDUCE16_LARGE = 1, REDUCE_ANY = 2, REDUCE_CLASSES = 3 };
// FP32 exit records carry the exit side + 1 (0 = none, 1..5 = sides -1..4) in the low bits of
// Y: a float widened to double leaves the low 29 bits of its mantissa zero.
constexpr uint64_t kSideBitsMask = 7ULL;
constexpr int kMaxQueues = 8;              // path queues: one per XCD of an MI355X (8 XCDs x 32 CUs)
// 64-bit words between two queue counters: atomics of one cache line wait for each other across the
// XCDs (about 130 ns each)
constexpr int kQueueStride = 32;

// One Monte Carlo knot of an assembly batch.
struct KnotDesc {
    double x0, y0;          // start point
    uint32_t knot_id;       // Philox counter word 2 (knot index within its request / mesh)
    uint32_t stream;        // Philox key word 1 (the run's stream, or the serving request's)
    int32_t table;          // stencil table of the knot (TableDesc index of the launch)
    int32_t stencil;        // index into that table's stencils
    int64_t n_paths;
    int64_t path_off;       // global index of the knot's first path in the batch (ascending)
    int64_t out_off;        // first value of the knot's G row in the CSR value array
    int64_t item_begin;     // first work item of the knot
    int64_t item_count;
    double k2;              // Helmholtz parameter of the knot's problem
    double h, sqrth;        // Euler-Maruyama step of the knot's paths (the run's, or its adaptive h)
    // the knot's stopping domain and the sides of it on the global boundary, copied from its
    // stencil (StencilDesc rect or geo, gmask): a lane starts a path with one load instead of three
    // that wait for each other
    double dom[6];
    int32_t gmask, pad;
};

// One distinct stencil: stopping rectangle, four side lists (N,S,E,W), Psi^-1 per side,
// and for each CSR column of the row up to two contributing side entries.
struct StencilDesc {
    double rect[4];         // rectangular stopping domain x0, y0, x1, y1
    double geo[6];          // annular-sector stopping domain r0, r1, cos/sin ray a, cos/sin ray b
    double bbox[4];         // bounding box of the stopping domain (host: LUT tiles)
    double inv_c2[4];       // 1 / c^2 of the Gaussian shape c per side
    int64_t ipsi_off[4];    // row-major m x m blocks in the ipsi array
    int32_t msz[4];
    int32_t ent_off;        // first side entry in ent_x / ent_y / ent_side
    int32_t csr_nnz;        // columns in the CSR row
    int32_t csr_off;        // first column map entry in csr_e1 / csr_e2
    int32_t gmask;          // bit s set: side s lies on the global boundary
};

// The device stencil tables of one mesh: a launch may carry knots of several meshes (serving),
// each knot naming its table.
struct TableDesc {
    const StencilDesc *sten;
    const double *entx, *enty;     // side-entry positions
    const int8_t *ents;            // side of each entry
    const double *entic2;          // 1 / c^2 of each entry's Gaussian (its side's c, or its own)
    const int32_t *e1, *e2;        // contributing entries of each CSR column
    const double *ipsi;            // Psi^-1 blocks
};

struct ItemDesc {
    int32_t knot;           // index into the knot table
    int32_t n;              // paths in the item
    int64_t p_begin;        // first path index within the knot
    int64_t part_off;       // 2*nnz partials (sum, sum of squares / n_beta)
    // the reduction's w-th work-group (of its launches' one after another) takes items span_first ..
    // + span_count of one knot, as entry w of the item table says: these two are not about the
    // entry's own item
    int32_t span_first, span_count;
};

struct ItemStat {
    double Bs, BBs;
    double Rs, RQs;         // equation residual sums (ReduceArgs::wref set): sum R_b, sum R_b^2 / n_b
    uint32_t cnt[6];        // exits per side 0..4, and paths stopped inside (no side)
};

struct KnotStat {
    double B, BB;
    double Rm, Rv;          // mean and per-path variance of the knot's equation estimator
    unsigned long long steps;
    unsigned long long capped;
    unsigned long long cnt[6];
};

// Bytes of a knot's descriptor where a call's device memory is estimated ahead of it (serving
// admission, pdds_point_eval_noalloc).  What a descriptor has beyond them and the block table of the
// knots are launch-side copies of a few dozen bytes a knot and stay out of these limits.
constexpr int64_t kKnotDescQuota = 96;
constexpr int64_t kItemDescQuota = 24;     // of a work item's, in the same estimates

// Per-path exit records, indexed by global path index: the FP64 exit values as one aligned
// 32-byte record (a lane stores it with two 16-byte writes when its path stops, so a record
// reaches memory as one 32-byte piece).  The exit side is not stored for FP64 paths: the
// reduction classifies the exit point again, with the same test on the same doubles.  Step
// counts are not stored per path: a wave sums the steps and step-cap stops of its stopped paths
// per knot (KnotSteps, LaneSteps) and adds them to the knot's counters kacc[2k] (steps) and
// kacc[2k + 1] (capped).
struct alignas(32) ExitRec {
    double x, y, Y, score;
};
struct Records {
    ExitRec *r;
    unsigned long long *kacc;   // 2 per knot of the launch, zero before the path kernel
};

// A patch: knots whose LUT tile (the plane-a texels their stencil rectangle can touch) is the
// same; their paths are [pbeg, pend) of the batch.  tiled == 0: the tile does not fit in LDS
// and the patch reads the LUT from global memory.
struct PatchDesc {
    int64_t pbeg, pend;
    int32_t c0, r0, tw, th;
    int32_t tiled, pitch;   // tiled: planes in the tile (coefficient LUT: 1, tabulated problem: 2, or 3
                            // with mu and F), 0: none; pitch: texels per LDS tile row (tw plus the run's lut_pad)
};

struct PathKernelArgs {
    const KnotDesc *knots;
    int32_t n_knots;
    // knot of the first path of every block of 2^kshift paths, and of the last path at the end:
    // bounds of the search for a path's knot
    int32_t kshift;
    const int32_t *kblk;
    const TableDesc *tables;
    int64_t total;          // paths in the batch
    int64_t base;           // plain launches: first path of this launch
    // persistent launches: queue q serves paths [q queue_len, (q + 1) queue_len) of the batch;
    // work-group b starts on queue b % n_queues (the XCD it is dispatched to) and moves to the next
    // queue when its own is drained.  The first pool_first paths of each wave of a queue are its own
    // (no atomic where a launch starts, with every wave at once); those behind them are handed out
    // pool_chunk at a time through counter[q kQueueStride].
    unsigned long long *counter;
    int32_t n_queues;
    int32_t pool_first;
    int64_t queue_len;
    int64_t pool_chunk;     // paths a wave takes from a queue at once
    // LDS-tiled launches: one queue per patch (counter[p kQueueStride] counts paths handed out of patch p)
    const struct PatchDesc *patches;
    int32_t n_patches;
    Records rec;
    double gc[4];           // the global rectangle's centre and half-sides, or the disc's radius
    double h, sqrth, beta;
    uint32_t seed, stream;
    uint32_t max_steps;     // below 2^27
    PdeParams pp;
};

struct ReduceArgs {
    const KnotDesc *knots;
    const TableDesc *tables;
    const ItemDesc *items;
    int64_t item_base;
    Records rec;
    ItemStat *stats;
    double *partials;
    // optional: per CSR value (out_off + c), the reference interface value u_ref of the column's
    // knot; the reduction then also sums R_b = B_b - sum_c G_b,c u_ref per sub-batch b
    const double *wref;
    int32_t ne_cap, nnz_cap;
    int32_t S;
    // 1: every stencil side is straight and uniformly spaced with one Gaussian width (rectangle
    // meshes), and the RBF values of a side come from rbf_side_chunk
    int32_t side_rbf;
    // exit sides (ReduceSide): from the low bits of the records' Y (FP32 paths), or by
    // classifying the exit point as write_exit does for FP64 paths, on the global
    // rectangle of centre and half-sides gc (classify_coord_c) or the disc of radius gc[0]
    int32_t side_mode;
    double gc[4];
};
enum ReduceSide { SIDE_BITS = 0, SIDE_RECT = 1, SIDE_DISC = 2 };

struct FinalizeArgs {
    const KnotDesc *knots;
    const TableDesc *tables;
    const ItemDesc *items;
    const ItemStat *stats;
    const double *partials;
    int32_t n_knots;
    int32_t S;
    double *G, *Gvar;
    KnotStat *kstats;
    const unsigned long long *kacc;   // steps and capped paths per knot (Records::kacc)
};

struct PathsArgs {
    double x0, y0;
    double rect[4];
    uint32_t knot, seed, stream;
    int32_t phase2;
    int64_t path0, n;
    double h, sqrth, beta;
    int64_t max_steps;
    PdeParams pp;
    double *xt, *yt, *Y, *Z, *xi;
    int64_t *steps;
    double *xt2, *yt2, *Y2, *Z2, *xi2;
    int64_t *steps2;
};

// Where pdds_paths has a path's exit values written (null: not asked for), per phase.
struct PathOut {
    double *xt[2], *yt[2], *Y[2], *Z[2], *xi[2];
    int64_t *steps[2];
    int32_t phase2;
};
// A path launch: with per_cu set nothing is launched, and the work-groups of the kernel that a CU
// holds at once are put there (a persistent grid is sized by them).
struct PathLaunch {
    int grid, wg;
    hipStream_t stream;
    int *per_cu;
    template <class K, class... A> hipError_t go(K kernel, const A &...args) const {
        if (per_cu) return hipOccupancyMaxActiveBlocksPerMultiprocessor(per_cu, kernel, wg, 0);
        hipLaunchKernelGGL(kernel, dim3(grid), dim3(wg), 0, stream, args...);
        return hipGetLastError();
    }
};

// Launchers (defined in engine_f64.hip / engine_f32.hip)
hipError_t launch_path_tiled_f64(int pde, int geom, bool mixed, int grid, size_t lds, hipStream_t s, const PathKernelArgs &a);
hipError_t launch_path_tiled_f32(int pde, int geom, bool mixed, int grid, size_t lds, hipStream_t s, const PathKernelArgs &a);
// Whether a launch of the tabulated problem takes the LDS-tiled kernel, by its paths, the lanes of the
// tiled grid (131072 on 256 CUs) and the share of paths whose tile fits.  Where all fit, from four paths a
// lane on: 357 knots of 8 x 8 or 4 x 4 subdomains, 128 x 128 texels, FP64, h = 2e-4 and 2e-3 of the
// subdomain: 5.2 10^5 paths 9.2 and 1.15 ms, persistent kernel 8.7 and 1.08 (VR + CV 14.4 and 1.83,
// 13.7 and 2.02; FP32 6.4 and 0.73, 8.1 and 1.0); 10^6 10.0 and 1.18, 11.1 and 1.33; 3 10^5 8.6 and 1.14,
// 6.3 and 0.85.  The patch without a tile is worked on last, by all, with the tiled kernel's thin grid: where
// 3 of 100 paths have none, 2.5 10^6 paths take 2.9 ms (2.7), 8 10^6 5.1 (6.9); where none fits (512 x 512
// texels) 4.7 (3.0) and 11.0 (8.8).
inline bool tabulated_tiles(int64_t paths, int64_t lanes, double fitting) {
    return fitting >= 1.0 ? paths >= 4 * lanes : fitting >= 0.9 && paths >= 32 * lanes;
}
// The same of the coefficient LUT (lanes: 131072, FP32 rectangles 196608).  Each pair: tiled and persistent
// kernel, at h = 1e-2 of the subdomain's size squared, and where two follow, at 1e-3.  FP64: 2 10^6 paths
// 4.9 and 4.8 ms, 47 and 44 (8 x 8 subdomains of 32 knots, 256 x 256 samples, all tiles fit), 7.0 and 5.8,
// 60 and 59 (512 x 512, a few tiles do not); 6 10^6 paths 9.8 and 9.7, 11.4 and 13.0 (64 x 64: 9.8 and 8.9);
// 1.5 10^7 18.3 and 21.5, 18.5 and 27.4; where none fits (4 x 4) 6 10^6 take 14.1 and 14.2, 1.5 10^7 32.0 and
// 33.3.  FP32 (4 x 4, 128 x 128, at 5e-3 and 1e-3): 5.4 10^5 paths 4.6 and 3.7, 23 and 21, 7.7 10^5 4.8 and
// 4.8, 24 and 24, 10^6 4.5 and 5.0, 20 and 26 (256 x 256 on 8 x 8 4.3 and 5.5, 22 and 24); where a few tiles
// do not fit 2 10^6 7.0 and 5.2, 55 and 47, 6 10^6 8.5 and 12.1; where none fits 15.5 and 13.1 (6 10^6), 34.1
// and 31.2 (1.5 10^7).  Discs of 24 and 144 sectors, 64 x 64: FP32 2 10^6 paths 1.0 and 1.4, 1.6 and 1.2, 6 10^6
// 1.9 and 2.6, 2.0 and 2.1; FP64 2 10^6 2.2 and 2.0, 2.2 and 1.7, 6 10^6 3.9 and 3.6, 3.4 and 2.9, 1.5 10^7 7.8
// and 6.9, 6.1 and 5.8.
inline bool lut_tiles(bool fp64, bool rect, int64_t paths, int64_t lanes, double fitting) {
    if (fp64) return paths >= 24 * lanes;
    return fitting >= 0.75 && paths >= (rect && fitting >= 1.0 ? 4 : 16) * lanes;
}
int path_tiled_wg(int pde, int precision, int step, int geom);   // block size of the LDS-tiled kernel
hipError_t launch_path_f64(int pde, int geom, bool persistent, bool mixed, const PathLaunch &l, const PathKernelArgs &a);
hipError_t launch_path_f32(int pde, int geom, bool persistent, bool mixed, const PathLaunch &l, const PathKernelArgs &a);
// Group kernel (rectangles, control-variate step): lanes that carry one path of a launch of that many
// paths, 1, 4 or 16; 0 where the launch is the other path kernels'
int group_lanes(int pde, int precision, bool refl, int n_cu, int64_t paths);
hipError_t launch_group_f64(int pde, bool mixed, int lanes, const PathLaunch &l, const PathKernelArgs &a);
hipError_t launch_group_f32(int pde, bool mixed, int lanes, const PathLaunch &l, const PathKernelArgs &a);
// ... with each path's exit values written out (4 lanes to a path)
hipError_t launch_group_records_f64(int pde, const PathLaunch &l, const PathKernelArgs &a, const PathOut &o);
hipError_t launch_group_records_f32(int pde, const PathLaunch &l, const PathKernelArgs &a, const PathOut &o);
hipError_t launch_reduce(int grid, int wg, size_t shmem, hipStream_t s, const ReduceArgs &a);
hipError_t launch_reduce16(bool small, int grid, size_t shmem, hipStream_t s, const ReduceArgs &a);
hipError_t launch_paths_f64(int pde, int grid, int wg, hipStream_t s, const PathsArgs &a);
hipError_t launch_paths_f32(int pde, int grid, int wg, hipStream_t s, const PathsArgs &a);
hipError_t launch_finalize(int grid, int wg, hipStream_t s, const FinalizeArgs &f);
hipError_t launch_lut_eval(const LutView &L, int field, int64_t n, const double *x, const double *y, double *out,
                           hipStream_t s);
hipError_t launch_fill_u64(unsigned long long *p, int64_t n, unsigned long long v, hipStream_t s);

}  // namespace pdds
