// guess.hip -- kernels of the learned initial guess: a periodic 3D
// convolutional encoder-decoder over the voxel grid whose products run on the
// matrix cores (v_mfma_f32_16x16x16_bf16: BF16 operands, FP32 accumulation),
// and the kernels that train it (input and weight gradients, loss, Adam).
//
// Convolutions are implicit GEMMs: rows are output voxels, columns output
// channels, and the reduction runs over (tap, input channel).  One wavefront
// owns 4 groups of 16 output voxels and all (<= 64) output channels; its A
// operands are gathered straight from the channels-last input (8 bytes = 4
// channels per lane), its B operand is the packed BF16 weight row, loaded
// once for the 4 groups (37-47 % faster than one group per wavefront for
// the full-resolution layers at 256^3).  The products are the 16x16x16 BF16
// shape: these layers are bound by their operand gathers, not by the matrix
// cores (a 16 -> 16 channel layer at 256^3 runs about 230 GFLOP in 2.2 ms),
// so the 16x16x32 shape of gfx950 would not shorten them.
#include <hip/hip_runtime.h>
#include <stdio.h>
#include "guess.h"

namespace chfem {
namespace nn {

typedef short short4_t __attribute__((ext_vector_type(4)));
typedef float float4_t __attribute__((ext_vector_type(4)));

#define NB 256

__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// FP32 -> BF16, round to nearest even
__device__ __forceinline__ uint16_t f2bf(float f)
{
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7f800000u) == 0x7f800000u) return (uint16_t)((u >> 16) | ((u & 0xffffu) ? 0x40u : 0u));
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

__device__ __forceinline__ float4_t mfma16(short4_t a, short4_t b, float4_t c)
{
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ int wrap(int a, int n) { return a < 0 ? a + n : (a >= n ? a - n : a); }

// input voxel feeding tap t of the output row at (r, c, l)
template <int MODE>
__device__ __forceinline__ size_t in_index(int r, int c, int l, int t, const Grid3 &gi, const Grid3 &go)
{
    if (MODE == CONV_SAME) {
        const int rr = wrap(r + t % 3 - 1, gi.ny), cc = wrap(c + (t / 3) % 3 - 1, gi.nx), ll = wrap(l + t / 9 - 1, gi.nz);
        return (size_t)rr + (size_t)cc * gi.ny + (size_t)ll * gi.ny * gi.nx;
    } else if (MODE == CONV_DOWN) {
        const int rr = 2 * r + (t & 1), cc = 2 * c + ((t >> 1) & 1), ll = 2 * l + (t >> 2);
        return (size_t)rr + (size_t)cc * gi.ny + (size_t)ll * gi.ny * gi.nx;
    } else if (MODE == CONV_UP) {
        const int rr = wrap(r + t % 3 - 1, go.ny), cc = wrap(c + (t / 3) % 3 - 1, go.nx), ll = wrap(l + t / 9 - 1, go.nz);
        return (size_t)(rr >> 1) + (size_t)(cc >> 1) * gi.ny + (size_t)(ll >> 1) * gi.ny * gi.nx;
    } else {
        return (size_t)r + (size_t)c * gi.ny + (size_t)l * gi.ny * gi.nx;
    }
}

// Each wavefront owns CG groups of 16 consecutive output voxels (64): a
// weight operand, loaded once per (tap, 16 input channels, 16 output
// channels), feeds CG products, and the CG input gathers of a step are in
// flight together.
constexpr int CG = 4;

template <int MODE, int NT, bool OUTF>
__global__ void __launch_bounds__(NB) k_conv(const uint16_t *__restrict__ in, Grid3 gi, int Ci,
                                             const uint16_t *__restrict__ W, int taps, const float *__restrict__ bias,
                                             const uint16_t *__restrict__ skip, int relu, void *out, int accumulate,
                                             Grid3 go)
{
    constexpr int Co = NT * 16;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int i = lane & 15, kg = lane >> 4;
    const Grid3 rg = MODE == CONV_PARITY ? gi : go;  // grid of the output rows
    const size_t V = (size_t)rg.ny * rg.nx * rg.nz;
    const size_t vb = ((size_t)blockIdx.x * 4 + wave) * 16 * CG;
    if (vb >= V) return;  // no barriers in this kernel
    const int par = MODE == CONV_PARITY ? (int)blockIdx.y : 0;
    const uint16_t *Wp = W + (size_t)par * Co * taps * Ci;
    bool okA[CG];
    int r[CG], c[CG], l[CG];
#pragma unroll
    for (int gq = 0; gq < CG; gq++) {
        size_t va = vb + 16 * gq + i;
        okA[gq] = va < V;
        if (!okA[gq]) va = V - 1;
        r[gq] = (int)(va % rg.ny);
        c[gq] = (int)((va / rg.ny) % rg.nx);
        l[gq] = (int)(va / ((size_t)rg.ny * rg.nx));
    }
    float4_t acc[CG][NT];
#pragma unroll
    for (int gq = 0; gq < CG; gq++)
#pragma unroll
        for (int nt = 0; nt < NT; nt++) acc[gq][nt] = float4_t{0.f, 0.f, 0.f, 0.f};
    const size_t Ktot = (size_t)taps * Ci;
    for (int t = 0; t < taps; t++) {
        const uint16_t *src[CG];
#pragma unroll
        for (int gq = 0; gq < CG; gq++) src[gq] = in + in_index<MODE>(r[gq], c[gq], l[gq], t, gi, go) * Ci + 4 * kg;
        const uint16_t *wsrc = Wp + (size_t)i * Ktot + (size_t)t * Ci + 4 * kg;
        for (int c0 = 0; c0 < Ci; c0 += 16) {
            short4_t a[CG];
#pragma unroll
            for (int gq = 0; gq < CG; gq++) {
                a[gq] = *(const short4_t *)(src[gq] + c0);
                if (!okA[gq]) a[gq] = short4_t{0, 0, 0, 0};
            }
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                const short4_t bw = *(const short4_t *)(wsrc + (size_t)nt * 16 * Ktot + c0);
#pragma unroll
                for (int gq = 0; gq < CG; gq++) acc[gq][nt] = mfma16(a[gq], bw, acc[gq][nt]);
            }
        }
    }
    // D[row][col]: this lane holds column i, rows 4*kg + e of each group
#pragma unroll
    for (int gq = 0; gq < CG; gq++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const size_t vr = vb + 16 * gq + 4 * kg + e;
            if (vr >= V) continue;
            size_t vo = vr;
            if (MODE == CONV_PARITY) {
                const int rr = (int)(vr % rg.ny), cc = (int)((vr / rg.ny) % rg.nx),
                          ll = (int)(vr / ((size_t)rg.ny * rg.nx));
                vo = (size_t)(2 * rr + (par & 1)) + (size_t)(2 * cc + ((par >> 1) & 1)) * go.ny +
                     (size_t)(2 * ll + (par >> 2)) * go.ny * go.nx;
            }
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                const int co = nt * 16 + i;
                float val = acc[gq][nt][e];
                if (bias) val += bias[co];
                if (skip) val += bf2f(skip[vo * Co + co]);
                if (relu) val = fmaxf(val, 0.f);
                if (OUTF) {
                    float *o = (float *)out + vo * Co + co;
                    *o = accumulate ? *o + val : val;
                } else {
                    ((uint16_t *)out)[vo * Co + co] = f2bf(val);
                }
            }
        }
}

// Small grids: a wavefront takes 16 output voxels and 16 output channels, and
// issues the loads of STEPS (tap, 16 input channels) steps before their
// products, which keep k_conv's order (the same bits).  A 16^3 layer of 48
// channels gave k_conv 64 wavefronts of 81 dependent steps each, bound by one
// load latency per step: 115 us; here 23 us (8^3: 120 -> 23, 32^3
// up-convolution 48 -> 32: 98 -> 47).  With enough voxels k_conv's 4 groups
// per weight operand win.
template <int MODE, bool OUTF>
__global__ void __launch_bounds__(NB) k_conv_small(const uint16_t *__restrict__ in, Grid3 gi, int Ci,
                                                   const uint16_t *__restrict__ W, int taps,
                                                   const float *__restrict__ bias, const uint16_t *__restrict__ skip,
                                                   int relu, void *out, int accumulate, Grid3 go, int Co)
{
    constexpr int STEPS = 9;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int i = lane & 15, kg = lane >> 4;
    const uint32_t V = (uint32_t)go.ny * go.nx * go.nz, NT = (uint32_t)Co / 16u;
    const uint32_t job = blockIdx.x * 4u + wave, vb = job / NT * 16u, nt = job % NT;
    if (vb >= V) return;  // no barriers in this kernel
    const bool okA = vb + i < V;
    const uint32_t va = okA ? vb + i : V - 1;
    const int r = (int)(va % (uint32_t)go.ny), c = (int)(va / (uint32_t)go.ny % (uint32_t)go.nx),
              l = (int)(va / ((uint32_t)go.ny * go.nx));
    const int kc = Ci / 16, steps = taps * kc;
    const uint16_t *wrow = W + (size_t)(nt * 16 + i) * ((size_t)taps * Ci) + 4 * kg;
    float4_t acc = {0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < steps; s0 += STEPS) {
        short4_t a[STEPS], b[STEPS];
#pragma unroll
        for (int k = 0; k < STEPS; k++) {
            // (steps past the last re-read it; their products are left out)
            const int st = min(s0 + k, steps - 1), t = st / kc, c0 = (st - t * kc) * 16;
            a[k] = *(const short4_t *)(in + in_index<MODE>(r, c, l, t, gi, go) * Ci + c0 + 4 * kg);
            b[k] = *(const short4_t *)(wrow + (size_t)t * Ci + c0);
            if (!okA) a[k] = short4_t{0, 0, 0, 0};
        }
#pragma unroll
        for (int k = 0; k < STEPS; k++)
            if (s0 + k < steps) acc = mfma16(a[k], b[k], acc);
    }
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const uint32_t vo = vb + 4 * kg + e;
        if (vo >= V) continue;
        const int co = nt * 16 + i;
        float val = acc[e];
        if (bias) val += bias[co];
        if (skip) val += bf2f(skip[(size_t)vo * Co + co]);
        if (relu) val = fmaxf(val, 0.f);
        if (OUTF) {
            float *o = (float *)out + (size_t)vo * Co + co;
            *o = accumulate ? *o + val : val;
        } else {
            ((uint16_t *)out)[(size_t)vo * Co + co] = f2bf(val);
        }
    }
}
constexpr size_t CONV_SMALL = 65536;  // output voxels: 32^3 is faster here, 64^3 in k_conv

void conv(int mode, const uint16_t *in, Grid3 gi, int Ci, const uint16_t *W, const float *bias, const uint16_t *skip,
          int relu, void *out, int out_f32, int accumulate, Grid3 go, int Co, hipStream_t s)
{
    const int taps = mode == CONV_DOWN ? 8 : (mode == CONV_PARITY ? 1 : 27);
    const Grid3 rg = mode == CONV_PARITY ? gi : go;
    const size_t V = (size_t)rg.ny * rg.nx * rg.nz;
    dim3 grid((unsigned)((V + 64 * CG - 1) / (64 * CG)), mode == CONV_PARITY ? 8 : 1);
    if (mode != CONV_PARITY && V <= CONV_SMALL && Co % 16 == 0) {
        const unsigned sgrid = (unsigned)(((V + 15) / 16 * (Co / 16) + 3) / 4);
#define CONV_SMALL_CASE(M)                                                                             \
    if (mode == M) {                                                                                   \
        if (out_f32)                                                                                   \
            k_conv_small<M, true><<<sgrid, NB, 0, s>>>(in, gi, Ci, W, taps, bias, skip, relu, out, accumulate, go, Co); \
        else                                                                                           \
            k_conv_small<M, false><<<sgrid, NB, 0, s>>>(in, gi, Ci, W, taps, bias, skip, relu, out, accumulate, go, Co); \
        return;                                                                                        \
    }
        CONV_SMALL_CASE(CONV_SAME)
        CONV_SMALL_CASE(CONV_DOWN)
        CONV_SMALL_CASE(CONV_UP)
#undef CONV_SMALL_CASE
    }
#define CONV_CASE(M, NTv)                                                                              \
    if (mode == M && Co == NTv * 16) {                                                                 \
        if (out_f32)                                                                                   \
            k_conv<M, NTv, true><<<grid, NB, 0, s>>>(in, gi, Ci, W, taps, bias, skip, relu, out, accumulate, go); \
        else                                                                                           \
            k_conv<M, NTv, false><<<grid, NB, 0, s>>>(in, gi, Ci, W, taps, bias, skip, relu, out, accumulate, go); \
        return;                                                                                        \
    }
#define CONV_MODE(M) CONV_CASE(M, 1) CONV_CASE(M, 2) CONV_CASE(M, 3) CONV_CASE(M, 4)
    CONV_MODE(CONV_SAME)
    CONV_MODE(CONV_DOWN)
    CONV_MODE(CONV_UP)
    CONV_MODE(CONV_PARITY)
#undef CONV_MODE
#undef CONV_CASE
    fprintf(stderr, "chfem guess: no convolution kernel for mode %d, %d -> %d channels\n", mode, Ci, Co);
}

// ---------------------------------------------------------------------------
// weight gradients
// ---------------------------------------------------------------------------
// output voxels per block.  3x3x3 layers: about 256 chunks, in multiples of
// the 64 voxels that a block's wavefronts take per step.  DOWN: 2048, halved
// (down to 256) while the launch would have fewer than 2048 blocks, so the
// coarse levels' few voxels are still spread over the GPU.
static int wchunk(size_t V, int taps)
{
    if (taps == 27) {
        const size_t c = ((V + 255) / 256 + 63) / 64 * 64;
        return (int)(c < 64 ? 64 : c);
    }
    int c = 2048;
    while (c > 256 && ((V + c - 1) / c) * (size_t)taps < 2048) c /= 2;
    return c;
}

// 3x3x3 layers (SAME, UP).  A block takes a chunk of output voxels, one layer
// offset dl of the taps (blockIdx.y) and 16 input channels (blockIdx.z); a
// wavefront keeps the products of its 9 taps and all NCO * 16 output channels
// in registers, so a voxel's output gradients are read once for 9 taps, and
// per column offset the 6 rows around 4 consecutive voxels once for the 3 row
// offsets (for row counts that are multiples of 4: 4 consecutive voxels share
// a column).  The wavefronts take every fourth 16 voxels and add up through
// LDS.  Bound by its 2-byte gathers: 54 input loads per 27 products, where a
// block per tap read 27 x 8 and formed every voxel's position for every tap.
// 64^3, 16 -> 16: 39 us, up-convolution 32 -> 16: 56 us (403, 463 before).
template <int MODE, int NCO>
__global__ void __launch_bounds__(NB) k_convw27(const uint16_t *__restrict__ in, Grid3 gi, int Ci,
                                                const uint16_t *__restrict__ dz, Grid3 go, int chunk,
                                                float *__restrict__ part)
{
    constexpr int Co = NCO * 16;
    __shared__ float4_t red[3][9][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int i = lane & 15, kg = lane >> 4;
    const int dl = (int)blockIdx.y - 1, cit = blockIdx.z;
    const uint32_t V = (uint32_t)go.ny * go.nx * go.nz;
    const uint32_t v0 = blockIdx.x * (uint32_t)chunk, v1 = v0 + chunk < V ? v0 + chunk : V;
    float4_t acc[9][NCO];
#pragma unroll
    for (int t = 0; t < 9; t++)
#pragma unroll
        for (int m = 0; m < NCO; m++) acc[t][m] = float4_t{0.f, 0.f, 0.f, 0.f};
    for (uint32_t vk = v0 + 16 * (uint32_t)wave; vk < v1; vk += 64) {
        // this lane's 4 voxels (all in the chunk or all past it)
        const uint32_t vq = vk + 4 * kg;
        const bool ok = vq < v1;
        const uint32_t v = ok ? vq : v0;
        const uint32_t cl = v / (uint32_t)go.ny;
        const int r = (int)(v - cl * (uint32_t)go.ny), l = (int)(cl / (uint32_t)go.nx), c = (int)(cl - (uint32_t)l * go.nx);
        short4_t az[NCO];
#pragma unroll
        for (int m = 0; m < NCO; m++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const short g = (short)dz[(size_t)(v + e) * Co + m * 16 + i];
                az[m][e] = ok ? g : (short)0;
            }
        const int ll = wrap(l + dl, go.nz);
        uint32_t row[6];
#pragma unroll
        for (int e = 0; e < 6; e++) {
            const int rr = wrap(r + e - 1, go.ny);
            row[e] = (uint32_t)(MODE == CONV_UP ? rr >> 1 : rr);
        }
#pragma unroll
        for (int dc = 0; dc < 3; dc++) {
            const int cc = wrap(c + dc - 1, go.nx);
            const uint32_t col = MODE == CONV_UP ? ((uint32_t)(ll >> 1) * gi.nx + (uint32_t)(cc >> 1)) * gi.ny
                                                 : ((uint32_t)ll * gi.nx + (uint32_t)cc) * gi.ny;
            short x[6];
#pragma unroll
            for (int e = 0; e < 6; e++) x[e] = (short)in[(size_t)(col + row[e]) * Ci + cit * 16 + i];
#pragma unroll
            for (int dr = 0; dr < 3; dr++) {
                const short4_t bx = {x[dr], x[dr + 1], x[dr + 2], x[dr + 3]};
#pragma unroll
                for (int m = 0; m < NCO; m++) acc[3 * dc + dr][m] = mfma16(az[m], bx, acc[3 * dc + dr][m]);
            }
        }
    }
#pragma unroll
    for (int m = 0; m < NCO; m++) {
        if (wave > 0)
#pragma unroll
            for (int t = 0; t < 9; t++) red[wave - 1][t][lane] = acc[t][m];
        __syncthreads();
        if (wave == 0)
#pragma unroll
            for (int t = 0; t < 9; t++) {
                const float4_t sum = (acc[t][m] + red[0][t][lane]) + (red[1][t][lane] + red[2][t][lane]);
                const int tap = 9 * (int)blockIdx.y + t;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int co = m * 16 + 4 * kg + e, ci = cit * 16 + i;
                    part[(((size_t)blockIdx.x * 27 + tap) * Co + co) * Ci + ci] = sum[e];
                }
            }
        __syncthreads();
    }
}

// DOWN layers, and 3x3x3 ones on grids whose row count is no multiple of 4:
// block (chunk of output voxels, tap); the Co x Ci tile of the tap is split into 16x16 products spread over the 4 wavefronts
template <int MODE>
__global__ void __launch_bounds__(NB) k_convw(const uint16_t *__restrict__ in, Grid3 gi, int Ci,
                                              const uint16_t *__restrict__ dz, Grid3 go, int Co, int taps,
                                              int chunk, float *__restrict__ part)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int i = lane & 15, kg = lane >> 4;
    const int t = blockIdx.y;
    const size_t V = (size_t)go.ny * go.nx * go.nz;
    const size_t v0 = (size_t)blockIdx.x * chunk;
    const size_t v1 = v0 + chunk < V ? v0 + chunk : V;
    const int nci = Ci / 16, ntiles = (Co / 16) * nci;
    // With 4 tiles or more, wavefront w takes tiles w, w + 4, .. over all the
    // chunk's voxels.  With fewer, the wavefronts split the voxels as well:
    // wavefront w takes tile w % ntiles on every nsplit-th step of 16 voxels
    // from step w / ntiles, and the shares are added through LDS.
    const bool few = ntiles < 4;
    const int nsplit = few ? 4 / ntiles : 1;
    const int grp = few ? wave / ntiles : 0;
    const int wt = few ? wave % ntiles : wave;
    const int mmax = few ? 1 : 4;
    float4_t acc[4];
#pragma unroll
    for (int m = 0; m < 4; m++) acc[m] = float4_t{0.f, 0.f, 0.f, 0.f};
    if (grp < nsplit) {
        for (size_t vk = v0 + 16 * (size_t)grp; vk < v1; vk += 16 * (size_t)nsplit) {
            size_t u[4];
            bool ok[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const size_t v = vk + 4 * kg + e;
                ok[e] = v < v1;
                const size_t vv = ok[e] ? v : v0;
                const int r = (int)(vv % go.ny), c = (int)((vv / go.ny) % go.nx), l = (int)(vv / ((size_t)go.ny * go.nx));
                u[e] = in_index<MODE>(r, c, l, t, gi, go);
            }
#pragma unroll
            for (int m = 0; m < 4; m++) {
                const int tt = wt + 4 * m;
                if (m >= mmax || tt >= ntiles) break;
                const int cot = tt / nci, cit = tt % nci;
                short4_t a, b;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const size_t v = vk + 4 * kg + e;
                    a[e] = ok[e] ? (short)dz[v * Co + cot * 16 + i] : (short)0;
                    b[e] = ok[e] ? (short)in[u[e] * Ci + cit * 16 + i] : (short)0;
                }
                acc[m] = mfma16(a, b, acc[m]);
            }
        }
    }
    if (few && nsplit > 1) {
        __shared__ float4_t red[4][64];
        red[wave][lane] = acc[0];
        __syncthreads();
        if (wave >= ntiles) return;
        for (int k = 1; k < nsplit; k++) acc[0] += red[wave + ntiles * k][lane];
    }
    if (few && wave >= ntiles) return;
#pragma unroll
    for (int m = 0; m < 4; m++) {
        const int tt = wt + 4 * m;
        if (m >= mmax || tt >= ntiles) break;
        const int cot = tt / nci, cit = tt % nci;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int co = cot * 16 + 4 * kg + e, ci = cit * 16 + i;
            part[(((size_t)blockIdx.x * taps + t) * Co + co) * Ci + ci] = acc[m][e];
        }
    }
}

// Adds the chunks' partials: 32 outputs per block, the chunks shared by its 8
// groups of 32 work-items, 8 reads of each in flight (one work-item per
// output reading chunk after chunk took 42 us on 128 chunks of 6912; now
// 4.6 on 256).
__global__ void __launch_bounds__(NB) k_wsum(const float *__restrict__ part, int nchunk, int taps, int Co, int Ci,
                                             float *__restrict__ grad)
{
    constexpr int OUTS = 32, GROUPS = NB / OUTS, TURN = 8;
    __shared__ float red[GROUPS][OUTS];
    const size_t n = (size_t)taps * Co * Ci;
    const int o = threadIdx.x % OUTS, g = threadIdx.x / OUTS;
    // p enumerates the partials' layout (t, co, ci)
    const size_t p = (size_t)blockIdx.x * OUTS + o;
    float sum = 0.f;
    if (p < n)
        for (int c0 = g; c0 < nchunk; c0 += GROUPS * TURN) {
            float a[TURN];
#pragma unroll
            for (int k = 0; k < TURN; k++) {
                const int ch = c0 + k * GROUPS;
                a[k] = ch < nchunk ? part[(size_t)ch * n + p] : 0.f;
            }
#pragma unroll
            for (int k = 0; k < TURN; k++) sum += a[k];
        }
    red[g][o] = sum;
    __syncthreads();
    if (g != 0 || p >= n) return;
#pragma unroll
    for (int k = 1; k < GROUPS; k++) sum += red[k][o];
    const int ci = (int)(p % Ci), co = (int)((p / Ci) % Co), t = (int)(p / ((size_t)Ci * Co));
    grad[((size_t)co * taps + t) * Ci + ci] += sum;
}

// (an upper bound that grows with the grid: the scratch of a grid also serves
// every smaller one)
size_t wpart_size(Grid3 go, int Co, int Ci, int taps)
{
    const size_t V = (size_t)go.ny * go.nx * go.nz;
    const size_t most = taps == 27 ? 256 : V / 2048 + 512, all = (V + 63) / 64;
    return (most < all ? most : all) * taps * Co * Ci;
}

void conv_wgrad(int mode, const uint16_t *in, Grid3 gi, int Ci, const uint16_t *dz, Grid3 go, int Co, float *part,
                float *grad, hipStream_t s)
{
    const int taps = mode == CONV_DOWN ? 8 : 27;
    const size_t V = (size_t)go.ny * go.nx * go.nz;
    const int chunk = wchunk(V, taps);
    const int nchunk = (int)((V + chunk - 1) / chunk);
    if (mode == CONV_DOWN) {
        k_convw<CONV_DOWN><<<dim3(nchunk, taps), NB, 0, s>>>(in, gi, Ci, dz, go, Co, taps, chunk, part);
    } else if (go.ny % 4) {
        // (4 consecutive voxels straddle columns: the coarse levels of row
        // counts like 24 or 40)
        if (mode == CONV_SAME) k_convw<CONV_SAME><<<dim3(nchunk, taps), NB, 0, s>>>(in, gi, Ci, dz, go, Co, taps, chunk, part);
        else k_convw<CONV_UP><<<dim3(nchunk, taps), NB, 0, s>>>(in, gi, Ci, dz, go, Co, taps, chunk, part);
    } else {
        const dim3 grid(nchunk, 3, Ci / 16);
#define CONVW_CASE(M, N) \
    if (mode == M && Co == N * 16) k_convw27<M, N><<<grid, NB, 0, s>>>(in, gi, Ci, dz, go, chunk, part);
        CONVW_CASE(CONV_SAME, 1) CONVW_CASE(CONV_SAME, 2) CONVW_CASE(CONV_SAME, 3)
        CONVW_CASE(CONV_UP, 1) CONVW_CASE(CONV_UP, 2) CONVW_CASE(CONV_UP, 3)
#undef CONVW_CASE
        if (Co > 48) fprintf(stderr, "chfem guess: no weight-gradient kernel for %d output channels\n", Co);
    }
    const size_t n = (size_t)taps * Co * Ci;
    k_wsum<<<(unsigned)((n + 31) / 32), NB, 0, s>>>(part, nchunk, taps, Co, Ci, grad);
}

// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(NB) k_pack(const float *__restrict__ Wm, uint16_t *__restrict__ out, int Co, int Ci,
                                             int taps, int how)
{
    const size_t n = (size_t)Co * Ci * taps;
    for (size_t j = (size_t)blockIdx.x * NB + threadIdx.x; j < n; j += (size_t)gridDim.x * NB) {
        const int ci = (int)(j % Ci), t = (int)((j / Ci) % taps), co = (int)(j / ((size_t)Ci * taps));
        const uint16_t w = f2bf(Wm[j]);
        size_t o;
        if (how == 0) o = j;
        else if (how == 1) o = ((size_t)ci * taps + (taps - 1 - t)) * Co + co;
        else o = ((size_t)t * Ci + ci) * Co + co;
        out[o] = w;
    }
}

void pack_weights(const float *Wm, uint16_t *out, int Co, int Ci, int taps, int how, hipStream_t s)
{
    const size_t n = (size_t)Co * Ci * taps;
    k_pack<<<(unsigned)((n + NB - 1) / NB), NB, 0, s>>>(Wm, out, Co, Ci, taps, how);
}

// ---------------------------------------------------------------------------
// voxels per block of the activation backward: 256, on the coarse levels 32
// (16^3, 48 channels: 16 blocks of 51 serial steps took 25 us)
static int achunk(size_t V) { return V >= 65536 ? 256 : 32; }

__global__ void __launch_bounds__(NB) k_act_bwd(const float *__restrict__ dy, const uint16_t *__restrict__ y, int relu,
                                                uint16_t *__restrict__ dz, float *__restrict__ skip_grad,
                                                float *__restrict__ bpart, size_t V, int C, int chunk)
{
    __shared__ float red[NB];
    const int c = threadIdx.x % C, lanes = NB / C, vl = threadIdx.x / C;
    const size_t v0 = (size_t)blockIdx.x * chunk, v1 = v0 + chunk < V ? v0 + chunk : V;
    float bsum = 0.f;
    if (vl < lanes) {
        for (size_t v = v0 + vl; v < v1; v += lanes) {
            const size_t j = v * C + c;
            float g = dy[j];
            if (relu && !(bf2f(y[j]) > 0.f)) g = 0.f;
            const uint16_t gb = f2bf(g);
            dz[j] = gb;
            if (skip_grad) skip_grad[j] += g;
            bsum += bf2f(gb);
        }
    }
    red[threadIdx.x] = (vl < lanes) ? bsum : 0.f;
    __syncthreads();
    if (threadIdx.x < C) {
        float s = 0.f;
        for (int k = 0; k < lanes; k++) s += red[k * C + threadIdx.x];
        bpart[(size_t)blockIdx.x * C + threadIdx.x] = s;
    }
}

// one block per channel (one work-item per channel adding block after block
// took 65 us on 1024 blocks; now 4.6)
__global__ void __launch_bounds__(NB) k_bsum(const float *__restrict__ bpart, int nb, int C,
                                             float *__restrict__ bias_grad)
{
    __shared__ float red[NB / 64];
    const int c = blockIdx.x;
    float s = 0.f;
#pragma unroll 4
    for (int b = threadIdx.x; b < nb; b += NB) s += bpart[(size_t)b * C + c];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) bias_grad[c] += (red[0] + red[1]) + (red[2] + red[3]);
}

// (an upper bound that grows with V, as wpart_size)
size_t bias_part_size(size_t V, int C) { return ((V < 65536 ? V : 65536) / 32 + V / 256 + 2) * (size_t)C; }

void act_backward(const float *dy, const uint16_t *y, int relu, uint16_t *dz, float *skip_grad, float *bias_part,
                  float *bias_grad, size_t V, int C, hipStream_t s)
{
    const int chunk = achunk(V), nb = (int)((V + chunk - 1) / chunk);
    k_act_bwd<<<nb, NB, 0, s>>>(dy, y, relu, dz, skip_grad, bias_part, V, C, chunk);
    k_bsum<<<C, NB, 0, s>>>(bias_part, nb, C, bias_grad);
}

// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(NB) k_pool(const float *__restrict__ fine, Grid3 gf, float *__restrict__ coarse, int C,
                                             int accumulate)
{
    const int ny = gf.ny / 2, nx = gf.nx / 2, nz = gf.nz / 2;
    const size_t n = (size_t)ny * nx * nz * C;
    for (size_t j = (size_t)blockIdx.x * NB + threadIdx.x; j < n; j += (size_t)gridDim.x * NB) {
        const int c = (int)(j % C);
        const size_t w = j / C;
        const int r = (int)(w % ny), cc = (int)((w / ny) % nx), l = (int)(w / ((size_t)ny * nx));
        float s = 0.f;
#pragma unroll
        for (int t = 0; t < 8; t++) {
            const size_t u = (size_t)(2 * r + (t & 1)) + (size_t)(2 * cc + ((t >> 1) & 1)) * gf.ny +
                             (size_t)(2 * l + (t >> 2)) * gf.ny * gf.nx;
            s += fine[u * C + c];
        }
        coarse[j] = accumulate ? coarse[j] + s : s;
    }
}

void pool_children(const float *fine, Grid3 gf, float *coarse, int C, int accumulate, hipStream_t s)
{
    const size_t n = (size_t)(gf.ny / 2) * (gf.nx / 2) * (gf.nz / 2) * C;
    unsigned b = (unsigned)((n + NB - 1) / NB);
    if (b > 65536) b = 65536;
    k_pool<<<b, NB, 0, s>>>(fine, gf, coarse, C, accumulate);
}

// ---------------------------------------------------------------------------
#define LCHUNK 128

__global__ void __launch_bounds__(NB) k_mse(const float *__restrict__ y, int Cp, const float *__restrict__ target, int nt,
                                            size_t V, double scale, float *__restrict__ dy, double *__restrict__ part)
{
    __shared__ double red[NB];
    const size_t j0 = (size_t)blockIdx.x * LCHUNK * Cp, j1 = j0 + (size_t)LCHUNK * Cp < V * Cp ? j0 + (size_t)LCHUNK * Cp : V * Cp;
    double acc = 0;
    for (size_t j = j0 + threadIdx.x; j < j1; j += NB) {
        const int c = (int)(j % Cp);
        const size_t v = j / Cp;
        float g = 0.f;
        if (c < nt) {
            const float d = y[j] - target[v * nt + c];
            acc += (double)d * (double)d;
            g = (float)(2.0 * scale) * d;
        }
        dy[j] = g;
    }
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int w = NB / 2; w > 0; w >>= 1) {
        if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = red[0] * scale;
}

__global__ void __launch_bounds__(64) k_dsum(const double *__restrict__ part, int nb, double *__restrict__ out)
{
    double s = 0;
#pragma unroll 8
    for (int b = threadIdx.x; b < nb; b += 64) s += part[b];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    if (threadIdx.x == 0) *out += s;
}

size_t loss_part_size(size_t V) { return (V + LCHUNK - 1) / LCHUNK; }

void mse(const float *y, int Cp, const float *target, int nt, size_t V, double scale, float *dy, double *part,
         double *loss, hipStream_t s)
{
    const int nb = (int)loss_part_size(V);
    k_mse<<<nb, NB, 0, s>>>(y, Cp, target, nt, V, scale, dy, part);
    k_dsum<<<1, 64, 0, s>>>(part, nb, loss);
}

// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(NB) k_adam(float *__restrict__ w, const float *__restrict__ g, float *__restrict__ m,
                                             float *__restrict__ v, size_t n, float lr, float b1, float b2, float eps,
                                             float c1, float c2, float gscale)
{
    for (size_t j = (size_t)blockIdx.x * NB + threadIdx.x; j < n; j += (size_t)gridDim.x * NB) {
        const float gj = g[j] * gscale;
        const float mj = b1 * m[j] + (1.f - b1) * gj;
        const float vj = b2 * v[j] + (1.f - b2) * gj * gj;
        m[j] = mj;
        v[j] = vj;
        w[j] -= lr * (mj / c1) / (sqrtf(vj / c2) + eps);
    }
}

void adam(float *w, const float *g, float *m, float *v, size_t n, float lr, float b1, float b2, float eps, int step,
          float gscale, hipStream_t s)
{
    const float c1 = 1.f - powf(b1, (float)step), c2 = 1.f - powf(b2, (float)step);
    unsigned b = (unsigned)((n + NB - 1) / NB);
    if (b > 4096) b = 4096;
    k_adam<<<b, NB, 0, s>>>(w, g, m, v, n, lr, b1, b2, eps, c1, c2, gscale);
}

// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(NB) k_features(const uint16_t *__restrict__ elem, const float *__restrict__ table,
                                                 int nf, uint16_t *__restrict__ in, int C, size_t V)
{
    const size_t n = V * C;
    for (size_t j = (size_t)blockIdx.x * NB + threadIdx.x; j < n; j += (size_t)gridDim.x * NB) {
        const int c = (int)(j % C);
        const size_t v = j / C;
        in[j] = c < nf ? f2bf(table[(size_t)elem[v] * nf + c]) : (uint16_t)0;
    }
}

void features(const uint16_t *elem, const float *table, int nf, uint16_t *in, int C, size_t V, hipStream_t s)
{
    unsigned b = (unsigned)((V * C + NB - 1) / NB);
    if (b > 65536) b = 65536;
    k_features<<<b, NB, 0, s>>>(elem, table, nf, in, C, V);
}

// out[v * n + k] = y[v * C + k], k < n: the network's real outputs, packed for
// the copy to the host (the padded channels are 14 of 32, and repacking on
// the host cost as much again as the copy)
__global__ void __launch_bounds__(NB) k_outputs(const float *__restrict__ y, int C, int n, size_t V,
                                                float *__restrict__ out)
{
    const size_t all = V * n;
    for (size_t j = (size_t)blockIdx.x * NB + threadIdx.x; j < all; j += (size_t)gridDim.x * NB) {
        const size_t v = j / n;
        out[j] = y[v * C + (j - v * n)];
    }
}

void outputs(const float *y, int C, int n, size_t V, float *out, hipStream_t s)
{
    size_t b = (V * n + NB - 1) / NB;
    if (b > 65536) b = 65536;
    k_outputs<<<(unsigned)b, NB, 0, s>>>(y, C, n, V, out);
}

// load cases (seam axis, jumping component): X, Y, Z, YZ, XZ, XY
__constant__ int cLoadAxis[6] = {0, 1, 2, 1, 2, 1};
__constant__ int cLoadComp[6] = {0, 1, 2, 2, 0, 0};

__global__ void __launch_bounds__(NB) k_guess_x0(const float *__restrict__ y, int Cp, int load, int nd, Grid3 g,
                                                 float scale, double *__restrict__ x0)
{
    const size_t N = (size_t)g.ny * g.nx * g.nz;
    const int axis = cLoadAxis[load], comp = nd == 3 ? cLoadComp[load] : 0;
    for (size_t i = (size_t)blockIdx.x * NB + threadIdx.x; i < N; i += (size_t)gridDim.x * NB) {
        const int r = (int)(i % g.ny), c = (int)((i / g.ny) % g.nx), l = (int)(i / ((size_t)g.ny * g.nx));
        // total field of the homogeneous medium: ramp with the jump on the seam
        const double ramp = axis == 0 ? (double)c : (axis == 1 ? (double)((g.ny - r) % g.ny) : (double)((g.nz - l) % g.nz));
        for (int a = 0; a < nd; a++)
            x0[nd * i + a] = (a == comp ? ramp : 0.0) + (double)(scale * y[i * Cp + load * nd + a]);
    }
}

void guess_to_x0(const float *y, int Cp, int load, int nd, Grid3 g, float scale, double *x0, hipStream_t s)
{
    const size_t N = (size_t)g.ny * g.nx * g.nz;
    unsigned b = (unsigned)((N + NB - 1) / NB);
    if (b > 65536) b = 65536;
    k_guess_x0<<<b, NB, 0, s>>>(y, Cp, load, nd, g, scale, x0);
}

struct X0Set {
    double *x[6];
};

__global__ void __launch_bounds__(NB) k_guess_x0_all(const float *__restrict__ y, int Cp, int nd, Grid3 g, float scale,
                                                     X0Set xs)
{
    const size_t N = (size_t)g.ny * g.nx * g.nz;
    const int nloads = nd == 3 ? 6 : 3;
    for (size_t i = (size_t)blockIdx.x * NB + threadIdx.x; i < N; i += (size_t)gridDim.x * NB) {
        const int r = (int)(i % g.ny), c = (int)((i / g.ny) % g.nx), l = (int)(i / ((size_t)g.ny * g.nx));
        const double ramps[3] = {(double)c, (double)((g.ny - r) % g.ny), (double)((g.nz - l) % g.nz)};
        const float *yi = y + i * Cp;
        for (int load = 0; load < nloads; load++) {
            double *x0 = xs.x[load];
            if (!x0) continue;
            const int comp = nd == 3 ? cLoadComp[load] : 0;
            const double ramp = ramps[cLoadAxis[load]];
            for (int a = 0; a < nd; a++)
                x0[nd * i + a] = (a == comp ? ramp : 0.0) + (double)(scale * yi[load * nd + a]);
        }
    }
}

void guess_to_x0_all(const float *y, int Cp, int nd, Grid3 g, float scale, double *const x0[6], hipStream_t s)
{
    const size_t N = (size_t)g.ny * g.nx * g.nz;
    unsigned b = (unsigned)((N + NB - 1) / NB);
    if (b > 65536) b = 65536;
    X0Set xs;
    for (int k = 0; k < 6; k++) xs.x[k] = x0[k];
    k_guess_x0_all<<<b, NB, 0, s>>>(y, Cp, nd, g, scale, xs);
}

__global__ void k_fill_f32(float *p, float v, size_t n)
{
    for (size_t j = (size_t)blockIdx.x * NB + threadIdx.x; j < n; j += (size_t)gridDim.x * NB) p[j] = v;
}
__global__ void k_add_f32(float *d, const float *src, size_t n)
{
    for (size_t j = (size_t)blockIdx.x * NB + threadIdx.x; j < n; j += (size_t)gridDim.x * NB) d[j] += src[j];
}
void fill_f32(float *p, float v, size_t n, hipStream_t s)
{
    unsigned b = (unsigned)((n + NB - 1) / NB);
    if (b > 65536) b = 65536;
    if (b) k_fill_f32<<<b, NB, 0, s>>>(p, v, n);
}
void add_f32(float *dst, const float *src, size_t n, hipStream_t s)
{
    unsigned b = (unsigned)((n + NB - 1) / NB);
    if (b > 65536) b = 65536;
    if (b) k_add_f32<<<b, NB, 0, s>>>(dst, src, n);
}

__global__ void k_mfma_check(const uint16_t *__restrict__ A, const uint16_t *__restrict__ B, float *__restrict__ D)
{
    const int lane = threadIdx.x, i = lane & 15, kg = lane >> 4;
    short4_t a, b;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        a[e] = (short)A[i * 16 + 4 * kg + e];  // A[row i][k]
        b[e] = (short)B[(4 * kg + e) * 16 + i];  // B[k][col i]
    }
    const float4_t d = mfma16(a, b, float4_t{0.f, 0.f, 0.f, 0.f});
#pragma unroll
    for (int e = 0; e < 4; e++) D[(4 * kg + e) * 16 + i] = d[e];
}

void mfma_check(const uint16_t *A, const uint16_t *B, float *D, hipStream_t s)
{
    k_mfma_check<<<1, 64, 0, s>>>(A, B, D);
}

}  // namespace nn
}  // namespace chfem
