// walsh.hip -- kernel and launcher of the Walsh-basis elastic and conduction operators
// (device code in walsh.h).
#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>
#include <math.h>

#include <algorithm>

#include "batch.h"
#include "walsh.h"

namespace chfem {

__device__ __forceinline__ float wave_uniform(float v)
{
    return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(v)));
}
__device__ __forceinline__ double wave_uniform(double v)
{
    return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(v)),
                            __builtin_amdgcn_readfirstlane(__double2loint(v)));
}

template <typename T, int ND, int TR, int TC, bool DOT, int FM, bool HALO, bool SDF>
__device__ __forceinline__ void walsh_block(const T *__restrict__ v, T *__restrict__ q,
                                            const uint16_t *__restrict__ keys, const T *__restrict__ lamu, int ebe,
                                            int ny, int nx, int nz, int LZ, const Reduce &red, DirFuse<T> fz)
{
    constexpr bool FUSE = FM == 1 || FM == 2;
    // the scalars are read together, before the stop flag is tested: one
    // read latency at the head of the launch instead of two
    double done = 0.0, iter = 0.0;
    if (FM == 2 && DOT && red.prev) {
        const Cg1Scalars c = cg1_chain(red, gridDim.x);
        if (c.done != 0.0) return;
        fz.beta = (T)(c.delta / c.delta_old);
        fz.alpha = fz.zpend ? (T)c.alpha : T(0);
        if (fz.zring) fz.bprev = (T)c.bprev;
        iter = c.iter;
    } else {
        done = DOT && red.guard ? red.S[S_DONE] : 0.0;
        // beta of the fused direction update, as k_kj_pcg_dir forms it
        if (FUSE && !fz.first) fz.beta = (T)(red.S[S_DELTA] / red.S[S_DELTA_OLD]);
        // single-kernel CG: alpha of the previous iteration for the deferred z
        // update
        if (FM == 2) fz.alpha = fz.zpend ? (T)red.S[S_ALPHA] : T(0);
        // single-kernel CG with z recovered from the ring: the beta that formed
        // d_old
        if (FM == 2 && fz.zring) fz.bprev = (T)red.S[S_BPREV];
        // lean z update: alpha of this iteration
        if (FM == 3) fz.alpha = fz.lean == LEAN_ZUPD ? (T)red.S[S_ALPHA] : T(0);
        if (FM == 2 && DOT && red.guard) iter = red.S[S_ITER];
    }
    if (done != 0.0) return;
    if (FM == 2) {
        // the same in every lane: kept in scalar registers (with them in
        // vector registers the FP64 thermal tiles lose a wavefront per SIMD)
        fz.beta = wave_uniform(fz.beta);
        fz.alpha = wave_uniform(fz.alpha);
        fz.bprev = wave_uniform(fz.bprev);
    }
    // 1-D grid; blocks are dispatched to the 8 XCDs round-robin (block b to
    // XCD b % 8), so each XCD is given one contiguous range of tiles (rows of
    // tiles fastest): tiles that share halo nodes then run on the same XCD at
    // about the same time and meet each other's halo lines in its L2.
    // Single-kernel CG iterations of a guarded loop walk each XCD's range
    // backwards on odd iterations: an iteration then starts with the tiles
    // whose d and q the previous one wrote last, some of which the
    // memory-side cache still holds (1.7 % off the 256^3 FP32 launch).
    constexpr int OR = HALO ? TR : TR - 1;  // node rows per tile
    const unsigned gx = (unsigned)(ny + OR - 1) / OR, gy = (unsigned)(nx + TC - 2) / (TC - 1);
    const unsigned b = blockIdx.x, nb = gridDim.x, per = nb / 8u, rem = nb % 8u, xcd = b % 8u;
    unsigned k = b / 8u;
    if (FM == 2 && DOT && red.guard && ((unsigned)iter & 1u)) k = (xcd < rem ? per + 1u : per) - 1u - k;
    const unsigned t = (xcd < rem ? xcd * (per + 1u) : rem * (per + 1u) + (xcd - rem) * per) + k;
    const TileSums ts = walsh_tile<T, ND, TR, TC, DOT, FM, HALO, SDF>(v, q, keys, lamu, ebe, ny, nx, nz, LZ,
                                                                      (int)(t % gx), (int)((t / gx) % gy),
                                                                      (int)(t / (gx * gy)), fz);
    if (DOT && FM == 2) {
        double vv[4] = {ts.dq, ts.zq, ts.qmq, ts.zdz};
        store_partials<4>(red, vv);
    } else if (DOT) {
        double vv[1] = {ts.dq};
        store_partials<1>(red, vv);
    }
}

template <typename T, int ND, int TR, int TC, bool DOT, int FM, bool HALO>
__global__ void __launch_bounds__(TR *TC + (HALO ? 64 : 0)) k_walsh(const T *__restrict__ v, T *__restrict__ q,
                                                   const uint16_t *__restrict__ keys, const T *__restrict__ lamu,
                                                   int ebe, int ny, int nx, int nz, int LZ, Reduce red, DirFuse<T> fz)
{
    walsh_block<T, ND, TR, TC, DOT, FM, HALO, false>(v, q, keys, lamu, ebe, ny, nx, nz, LZ, red, fz);
}

// with a scalar density field (op.sdf): 32x8 tiles, and the 65x7 ones where
// the rule prefers long rows
template <typename T, int ND, int TR, int TC, bool DOT, int FM, bool HALO>
__global__ void __launch_bounds__(TR *TC + (HALO ? 64 : 0)) k_walsh_sdf(const T *__restrict__ v, T *__restrict__ q,
                                                   const uint16_t *__restrict__ elems, const T *__restrict__ lamu,
                                                   int ny, int nx, int nz, int LZ, Reduce red, DirFuse<T> fz)
{
    walsh_block<T, ND, TR, TC, DOT, FM, HALO, true>(v, q, elems, lamu, 1, ny, nx, nz, LZ, red, fz);
}

// Chained iterations (Reduce::chain): even ones work on S, odd ones on the
// scalars and partials kept beside them.  Sets this launch's inputs in rr and
// returns the Reduce of its finishing kernel, which is launched unless
// rr.defer.  On grids of one block per CU or less an iteration is little but
// latency: without the finishing launch, CG iterations take 24^3 thermal FP64
// 11.2 -> 10.0 us, 32^3 11.9 -> 11.3, 32^3 elastic 14.9 -> 13.8, 64^3 23.7 ->
// 22.7.  With more blocks each would read more partials than the one
// finishing block saves.
static Reduce cg1_plan(Reduce &rr, unsigned grid)
{
    if (!rr.guard || grid > CHAIN_BLOCKS) rr.chain = rr.defer = 0;
    double *const P[2] = {rr.partials, rr.partials + 4 * CHAIN_BLOCKS}, *const S[2] = {rr.S, rr.S + S_CHAIN};
    const int odd = rr.chain & 1;
    if (rr.chain) {
        rr.prev = P[odd ^ 1];
        rr.Sin = S[odd ^ 1];
        rr.Sout = S[odd];
    }
    rr.partials = P[odd];
    Reduce fin = rr;
    fin.Sin = S[odd];
    return fin;
}

// Layers per block of a launch: those asked for, doubled until the blocks fit
// the reduction partials.  rows, cols: nodes owned by the tile that is
// launched.  It can be smaller than the one asked for: 65 x 15 runs as 65 x 7
// in FP64 and with a density field, other shapes without a kernel as 32 x 8.
static int layers_per_block(const OpDesc &op, int asked, int rows, int cols)
{
    int LZ = asked > 0 ? asked : 16;
    const long tiles = (long)((op.ny + rows - 1) / rows) * ((op.nx + cols - 1) / cols);
    while (tiles * ((op.nz + LZ - 1) / LZ) > MAX_PARTIAL_BLOCKS) LZ *= 2;
    return LZ;
}

template <typename T, int ND>
static void launch_walsh_nd(const OpDesc &op, const T *lamu, const T *v, T *q, const Reduce *red, WalshTiles t,
                            hipStream_t s, const DirFuse<T> *fz, const hipEvent_t *ev)
{
    Reduce rr = red ? *red : NO_REDUCE;
    DirFuse<T> f = {nullptr, nullptr, T(0), T(0), 1, 0, nullptr, nullptr, nullptr, 0, T(0), 0, {}, nullptr};
    if (fz) f = *fz;
    f.sdf = op.sdf;
    f.dnode = (const T *)op.dnode;
    // lean forms of the memory-lean solvers: one tile shape (32 x 8)
    const bool lean = fz && fz->lean;
    // single-kernel CG form: the dinv table given (only launch_apply_cg1
    // sets it; its z output may be absent)
    const bool cg1 = fz && (fz->kinv || (op.sdf.d && fz->dnew));
    // ev: a start and a stop event bound to the k_walsh dispatch itself
    // (hipExtLaunchKernel), so their interval is the kernel's own run time
#define WALSH_GO(TRv, TCv, H, DOTv, FMv)                                                                \
    if (ev) hipExtLaunchKernelGGL(k_walsh<T, ND, TRv, TCv, DOTv, FMv, H>, dim3(grid), dim3(nt), 0, s, ev[0], ev[1], \
                                  0, v, q, op.keys, lamu, op.ebe, op.ny, op.nx, op.nz, LZ, rr, f);               \
    else k_walsh<T, ND, TRv, TCv, DOTv, FMv, H><<<grid, nt, 0, s>>>(v, q, op.keys, lamu, op.ebe, op.ny, op.nx,   \
                                                                     op.nz, LZ, rr, f);
    // H: the halo-wavefront variant (tiles own all TRv rows; one more
    // wavefront per block)
#define WALSH_LAUNCH(TRv, TCv, H)                                                                       \
    {                                                                                                   \
        constexpr int orows = H ? TRv : TRv - 1, nt = TRv * TCv + (H ? 64 : 0);                         \
        const int LZ = layers_per_block(op, t.LZ, orows, TCv - 1);                                      \
        const unsigned grid = (unsigned)((op.ny + orows - 1) / orows) * ((op.nx + TCv - 2) / (TCv - 1)) * \
                              ((op.nz + LZ - 1) / LZ);                                                  \
        if (cg1) {                                                                                      \
            const Reduce fin = cg1_plan(rr, grid);                                                      \
            WALSH_GO(TRv, TCv, H, true, 2)                                                              \
            if (!rr.defer) launch_reduce_finish(fin, grid, 4, s);                                       \
        } else if (fz) {                                                                                \
            WALSH_GO(TRv, TCv, H, true, 1)                                                              \
            launch_reduce_finish(rr, grid, 1, s);                                                       \
        } else if (red) {                                                                               \
            WALSH_GO(TRv, TCv, H, true, 0)                                                              \
            launch_reduce_finish(rr, grid, 1, s);                                                       \
        } else {                                                                                        \
            WALSH_GO(TRv, TCv, H, false, 0)                                                             \
        }                                                                                               \
        return;                                                                                         \
    }
    // tile rows 65: 65 element rows per column (64 owned + the row above),
    // the halo-wavefront variant of 64-row tiles.  15 columns (1024
    // work-items) only in FP32: the FP64 planes of the single-kernel CG
    // iteration would not fit in LDS.
    if (lean) {
#define WALSH_LAUNCH_LEAN(TRv, TCv)                                                                     \
    {                                                                                                   \
        constexpr int nt = TRv * TCv;                                                                   \
        const int LZ = layers_per_block(op, t.LZ, TRv - 1, TCv - 1);                                    \
        const unsigned grid = (unsigned)((op.ny + TRv - 2) / (TRv - 1)) * ((op.nx + TCv - 2) / (TCv - 1)) * \
                              ((op.nz + LZ - 1) / LZ);                                                  \
        WALSH_GO(TRv, TCv, false, true, 3)                                                              \
        launch_reduce_finish(rr, grid, 1, s);                                                           \
        return;                                                                                         \
    }
        WALSH_LAUNCH_LEAN(32, 8)
#undef WALSH_LAUNCH_LEAN
    }
    if (op.sdf.d) {
#define WALSH_GO_SDF(TRv, TCv, H, DOTv, FMv)                                                            \
    if (ev) hipExtLaunchKernelGGL(k_walsh_sdf<T, ND, TRv, TCv, DOTv, FMv, H>, dim3(grid), dim3(nt), 0, s, ev[0], \
                                  ev[1], 0, v, q, op.keys, lamu, op.ny, op.nx, op.nz, LZ, rr, f);       \
    else k_walsh_sdf<T, ND, TRv, TCv, DOTv, FMv, H><<<grid, nt, 0, s>>>(v, q, op.keys, lamu, op.ny, op.nx, op.nz, \
                                                                        LZ, rr, f);
#define WALSH_LAUNCH_SDF(TRv, TCv, H)                                                                   \
    {                                                                                                   \
        constexpr int orows = H ? TRv : TRv - 1, nt = TRv * TCv + (H ? 64 : 0);                         \
        const int LZ = layers_per_block(op, t.LZ, orows, TCv - 1);                                      \
        const unsigned grid = (unsigned)((op.ny + orows - 1) / orows) * ((op.nx + TCv - 2) / (TCv - 1)) * \
                              ((op.nz + LZ - 1) / LZ);                                                  \
        if (cg1) {                                                                                      \
            const Reduce fin = cg1_plan(rr, grid);                                                      \
            WALSH_GO_SDF(TRv, TCv, H, true, 2)                                                          \
            if (!rr.defer) launch_reduce_finish(fin, grid, 4, s);                                       \
        } else if (red) {                                                                               \
            WALSH_GO_SDF(TRv, TCv, H, true, 0)                                                          \
            launch_reduce_finish(rr, grid, 1, s);                                                       \
        } else {                                                                                        \
            WALSH_GO_SDF(TRv, TCv, H, false, 0)                                                         \
        }                                                                                               \
        return;                                                                                         \
    }
        if (t.TR == 65) WALSH_LAUNCH_SDF(64, 7, true)
        WALSH_LAUNCH_SDF(32, 8, false)
#undef WALSH_LAUNCH_SDF
#undef WALSH_GO_SDF
    }
    if constexpr (sizeof(T) == 4) {
        if (t.TR == 65 && t.TC == 15) WALSH_LAUNCH(64, 15, true)
    }
    if (t.TR == 65) WALSH_LAUNCH(64, 7, true)
    if (t.TR == 16 && t.TC == 16) WALSH_LAUNCH(16, 16, false)
    if (t.TR == 64 && t.TC == 4) WALSH_LAUNCH(64, 4, false)
    if (t.TR == 64 && t.TC == 8) WALSH_LAUNCH(64, 8, false)
    if (t.TR == 32 && t.TC == 16) WALSH_LAUNCH(32, 16, false)
    WALSH_LAUNCH(32, 8, false)
#undef WALSH_LAUNCH
#undef WALSH_GO
}

template <typename T>
void launch_walsh(const OpDesc &op, const T *lamu, const T *v, T *q, const Reduce *red, WalshTiles t, hipStream_t s,
                  const DirFuse<T> *fz, const hipEvent_t *ev)
{
    if (op.physics == PHY_ELASTIC) launch_walsh_nd<T, 3>(op, lamu, v, q, red, t, s, fz, ev);
    else launch_walsh_nd<T, 1>(op, lamu, v, q, red, t, s, fz, ev);
}

template <typename T>
void launch_walsh_lean(const OpDesc &op, int form, const T *v, T *z, const void *kinv, const Reduce *red,
                       hipStream_t s)
{
    DirFuse<T> f = {nullptr, nullptr, T(0), T(0), 1, 0, nullptr, nullptr, (const T *)kinv, 0, T(0), form, {}, nullptr};
    const WalshTiles t = {32, 8, op.tile_lz};
    launch_walsh<T>(op, (const T *)op.lamu, v, z, red, t, s, &f, nullptr);
}
template void launch_walsh_lean<float>(const OpDesc &, int, const float *, float *, const void *, const Reduce *,
                                       hipStream_t);
template void launch_walsh_lean<double>(const OpDesc &, int, const double *, double *, const void *,
                                        const Reduce *, hipStream_t);

// Tile and layers per block of a grid.  What bounds a launch changes with the
// grid: a block walks its layers one after the other, with two barriers and a
// load latency per layer, so a grid of few blocks is bound by that chain (a
// 32^3 FP64 conduction iteration took 24.5 us with 16 layers per block, 12
// blocks on 256 CUs, and takes 13.9 us with 1 or 2), and a grid of many
// rounds of blocks by what they load, halos included (256^3 FP32 elastic:
// 347 us with 65x7x32, 394 with 32x8x16).  The cost of a candidate in us is
//   rounds of blocks x (LZ + 2) steps x (d + work-items on a CU x c)
//   + h x n / (n + 20) x the million values its planes load, every column run
//     rounded up by one 128-byte line, n million nodes
// with the CU's resident blocks from the kernels' registers and LDS, and h, d
// (by block size) and c (by tile: their halo shares and latencies differ)
// fitted to which candidate of timed solves was the fastest; halo loads cost
// little while the vectors stay in the caches, hence n / (n + 20).  Fitted to
// 65 grids in both precisions and physics, cubes of 16 to 400 nodes and
// slabs, columns and odd sizes, every tile, LZ 1 to 32: the pick is 0.7 %
// behind the fastest candidate on average, within 3 % on 94 of 100, at the
// worst 9 % (50x20x100) and 8 % (400^3), both FP32 elastic.  With one c and d
// for all tiles, no 65x15 and no 32x16 it was 18 % behind on 192^3 (FP32
// elastic 166.6 us against 141.0) and 7.5 % on 128^3 (59.8 against 55.7).
// Timing every candidate before the first solve cost as much as 30 (256^3) to
// 150 (32^3) iterations.
struct TileFit {
    double h, d[3];  // see above; d of blocks of 256, 512 and 1024 work-items
    double c[7];     // ns per work-item and step, of each tile
};
static const int TILES[7][2] = {{32, 8}, {16, 16}, {64, 4}, {64, 8}, {65, 7}, {32, 16}, {65, 15}};

static int size_class(int nt) { return nt <= 256 ? 0 : (nt <= 512 ? 1 : 2); }

// blocks of nt work-items resident on a CU
static int resident_blocks(bool dbl, bool el, int nt)
{
    static const int blocks[2][2][3] = {{{8, 4, 2}, {5, 2, 1}}, {{6, 3, 1}, {3, 1, 1}}};
    return blocks[dbl][el][size_class(nt)];
}

// values loaded per step by a tile of rows x cols owned nodes
static double step_loads(int rows, int cols, double bytes_per_node)
{
    return (cols + 2) * ((rows + 2) + 128.0 / bytes_per_node) * 1e-6;
}

// (lean: the memory-lean forms, whose steps have twice the latency d)
template <typename T>
static double tile_cost(const OpDesc &op, int tile, int lz, int lean)
{
    static const TileFit fit[2][2] = {  // [precision][physics]
        {{5.19, {0.503, 0.289, 0.575}, {1.044, 1.268, 0.908, 1.126, 1.180, 1.303, 1.428}},
         {8.74, {0.772, 0.813, 0.675}, {2.166, 3.064, 2.247, 1.972, 1.890, 2.568, 2.835}}},
        {{3.87, {0.340, 0.340, 0}, {1.945, 2.040, 1.814, 1.852, 1.838, 2.041, 0}},
         {17.78, {0.776, 0.776, 0}, {3.967, 4.329, 3.446, 3.957, 3.863, 4.210, 0}}}};
    const bool dbl = sizeof(T) == 8, el = op.physics == PHY_ELASTIC, halo = TILES[tile][0] == 65;
    const int rows = halo ? 64 : TILES[tile][0] - 1, tc = TILES[tile][1];
    const int nt = halo ? 64 * tc + 64 : TILES[tile][0] * tc;
    const TileFit &f = fit[dbl][el];
    const double c = f.c[tile] * 1e-3, d = (lean ? 2 : 1) * f.d[size_class(nt)];
    const int resident = resident_blocks(dbl, el, nt);
    const double tiles = (double)((op.ny + rows - 1) / rows) * ((op.nx + tc - 2) / (tc - 1));
    if (tiles > MAX_PARTIAL_BLOCKS) return 1e300;
    const double nb = tiles * ((op.nz + lz - 1) / lz);
    const double slots = 256.0 * resident, full = floor(nb / slots), rest = nb - full * slots;
    const double steps = std::min(lz, op.nz) + 2;
    const double chain = full * (d + resident * nt * c) + (rest > 0 ? d + ceil(rest / 256.0) * nt * c : 0.0);
    const double n = (double)op.ny * op.nx * op.nz * 1e-6;
    return steps * (chain + f.h * n / (n + 20.0) * nb * step_loads(rows, tc - 1, sizeof(T) * (el ? 3 : 1)));
}

// The same for a batch (FP32), summed over its samples: rounds of blocks
// become the layer steps of all blocks over the resident slots, and w marches
// of one last block run alone after them.  Fitted to 36 batches of 1 to 32
// samples of 24 to 288 nodes: the pick is 0.8 % behind the fastest of the 18
// candidates on average and 8 % at the worst (one 96^3 elastic sample), and
// on none slower than 64 x 7 x 32 for every batch (8 elastic samples of edges
// 48-80 217 -> 179 ms, 4 of 20-32 23.7 -> 10.1, 3 of 90-130 515 -> 454).  The
// coefficients of the rule before made conduction of one 256^3 sample 5 %
// slower than that, one of 233x190x251 6 % (64 x 7 x 16).
int batch_tile_rule(bool elastic, const batch::Shape *shapes, int nshapes, const std::vector<std::array<int, 3>> &dims,
                    int loads, int &lz_out)
{
    struct BatchFit { double d, h, w, c[3]; };
    static const BatchFit fit[2] = {{2.72, 8.06, 0.216, {0.234, 0.289, 0.223}},
                                    {1.53, 12.6, 0.518, {0.246, 0.501, 0.286}}};
    const BatchFit &f = fit[elastic];
    int best = 0;
    double least = 1e300, n = 0;
    for (const auto &g : dims) n += (double)g[0] * g[1] * g[2] * loads * 1e-6;
    for (int sh = 0; sh < nshapes && sh < 3; sh++) {
        const batch::Shape &t = shapes[sh];
        const int nt = t.tr == 65 ? 64 * t.tc + 64 : t.tr * t.tc;
        const int resident = resident_blocks(false, elastic, nt);
        auto step = [&](double on_cu) { return f.d + on_cu * nt * f.c[sh] * 1e-3; };
        for (int lz = 1; lz <= 32; lz *= 2) {
            double nb = 0, steps = 0, longest = 0;
            for (const auto &g : dims) {  // {ny, nx, nz}
                const double cols = (double)((g[0] + t.rows - 1) / t.rows) * ((g[1] + t.cols - 1) / t.cols) * loads;
                const int chunks = (g[2] + lz - 1) / lz;
                nb += cols * chunks;
                steps += cols * (g[2] + 2 * chunks);
                longest = std::max(longest, std::min(lz, g[2]) + 2.0);
            }
            const double all = steps / (256.0 * resident) * step(resident);
            const double last = f.w * longest * step(std::min((double)resident, ceil(nb / 256.0)));
            const double loads_cost = f.h * n / (n + 400.0) * steps * step_loads(t.rows, t.cols, elastic ? 12 : 4);
            if (all + last + loads_cost < least) {
                least = all + last + loads_cost;
                best = sh;
                lz_out = lz;
            }
        }
    }
    return best;
}

template <typename T>
WalshTiles walsh_tile_rule(const OpDesc &op, int lean)
{
    WalshTiles best = {32, 8, 16};
    double least = 1e300;
    for (int tile = 0; tile < 7; tile++) {
        const int tr = TILES[tile][0], tc = TILES[tile][1];
        if (lean && tile != 0) continue;
        if (op.sdf.d && tile != 0 && tile != 4) continue;
        if (sizeof(T) == 8 && tc == 15) continue;  // does not fit in LDS
        // (memory-lean forms: 32 layers were slower than 16 on every grid, up
        // to 6 % at 192^3 FP64 elastic, 447 us per CG3 iteration against 421)
        for (int lz = 1; lz <= (lean ? 16 : 32); lz *= 2) {
            const double c = tile_cost<T>(op, tile, lz, lean);
            if (c < least) {
                least = c;
                best = {tr, tc, lz};
            }
        }
    }
    return best;
}
template WalshTiles walsh_tile_rule<float>(const OpDesc &, int);
template WalshTiles walsh_tile_rule<double>(const OpDesc &, int);

bool apply_dir_ok(const OpDesc &op)
{
    // the operators launch_apply sends to the Walsh kernel, with key-Jacobi on
    // or a stored one per node (scalar density field; single-kernel form only)
    return op.physics != PHY_FLUID && op.lamu && (op.sdf.d ? op.dnode != nullptr : !op.ebe && op.kinv);
}

template <typename T>
void launch_apply_dir(const OpDesc &op, const T *z, const T *dold, T *dnew, T *q, const Reduce *red, hipStream_t s,
                      const hipEvent_t *ev)
{
    const DirFuse<T> f = {z, dnew, T(0), T(0), dold ? 0 : 1, 0, nullptr, nullptr, nullptr, 0, T(0), 0, {},
                          nullptr};
    const WalshTiles t = {op.tile_tr, op.tile_tc, op.tile_lz};
    launch_walsh<T>(op, (const T *)op.lamu, dold, q, red, t, s, &f, ev);
}

template <typename T>
void launch_apply_cg1(const OpDesc &op, const T *zold, const T *qold, const T *dold, T *znew, T *dnew, T *qnew,
                      int pend, const Reduce *red, hipStream_t s, const hipEvent_t *ev, const T *dold2)
{
    const int first = dold ? 0 : 1, p = dold && pend ? 1 : 0;
    // dold2: z_old recovered from the directions (needs d_old and the
    // pending update)
    const int zr = dold2 && p ? 1 : 0;
    const DirFuse<T> f = {zr ? dold2 : zold, dnew, T(0), T(0), first, p, p ? qold : zold, znew, (const T *)op.kinv,
                          zr, T(0), 0, {}, nullptr};
    const WalshTiles t = {op.tile_tr, op.tile_tc, op.tile_lz};
    launch_walsh<T>(op, (const T *)op.lamu, dold, qnew, red, t, s, &f, ev);
}

template void launch_apply_cg1<float>(const OpDesc &, const float *, const float *, const float *, float *, float *,
                                      float *, int, const Reduce *, hipStream_t, const hipEvent_t *, const float *);
template void launch_apply_cg1<double>(const OpDesc &, const double *, const double *, const double *, double *,
                                       double *, double *, int, const Reduce *, hipStream_t, const hipEvent_t *,
                                       const double *);

template void launch_apply_dir<float>(const OpDesc &, const float *, const float *, float *, float *, const Reduce *,
                                      hipStream_t, const hipEvent_t *);
template void launch_apply_dir<double>(const OpDesc &, const double *, const double *, double *, double *,
                                       const Reduce *, hipStream_t, const hipEvent_t *);
template void launch_walsh<float>(const OpDesc &, const float *, const float *, float *, const Reduce *, WalshTiles,
                                  hipStream_t, const DirFuse<float> *, const hipEvent_t *);
template void launch_walsh<double>(const OpDesc &, const double *, const double *, double *, const Reduce *,
                                   WalshTiles, hipStream_t, const DirFuse<double> *, const hipEvent_t *);

}  // namespace chfem
