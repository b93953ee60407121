// BF16 MFMA kernels of the learned warm start's U-Net: 3x3x3 convolutions
// with any channel counts that are multiples of 16 (forward, data gradient
// through transposed weights, weight gradient), the grid transfers between
// node-coincident levels (full-weighting restriction, trilinear
// interpolation, each the other's adjoint up to a factor 8), a BF16 sum and
// a weighted mean-squared-error loss.  No counterpart in the reference.
//
// Layouts: activations X[b][v][C] bf16 (channels fastest, C a multiple of
// 16), v = k + nz*(i + nx*j); weights W[o][t][c] bf16 (FP32 masters kept by
// the caller); tap t = (dz+1) + 3(dx+1) + 9(dy+1).  Operand layout of one
// v_mfma_f32_16x16x16_bf16 on a wavefront: lane l holds A[l%16][4(l/16)+i],
// B[4(l/16)+i][l%16] and D[4(l/16)+i][l%16], i = 0..3.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdint>

#include "../../include/citcom_learn.h"
#include "learn_common.h"

using namespace learn;

namespace {

constexpr int TAPS = 27;

// ---- forward: Y[v][o] = act(sum_t sum_c X[v+off_t][c] W[o][t][c] + bias[o] + R[v][o])
//
// A workgroup takes a block of TZ x TX x TY voxels and NBO*16 output channels.
// The block with its one-voxel halo is staged in LDS, zero outside the grid,
// as [16-channel block][voxel][16]: along a plane of the block the voxels of
// consecutive lines (of TZ + 2) are consecutive, so a tap is one constant
// offset and 16 consecutive positions are one MFMA operand read of 512
// consecutive bytes, without a test or a conflict; positions on the halo are
// computed and dropped (2 in TZ + 2).  The weights are the A operand (rows:
// output channels), so a lane holds four channels of one voxel and stores them
// together.  K runs over the taps and, within a tap, the 16-channel blocks:
// each output is the same chain of 16x16x16 products whatever the block.
//
// WREG: all 27 taps' weights in registers (one or two channel blocks), any
// number of tiles per wavefront; else the weights of nine taps at a time in
// LDS, the next nine in flight during the products, CONV_M tiles per wavefront.
// A workgroup stages, multiplies and stores in turn, two or four of them to a
// CU.  At 16 -> 16 channels bound by the issue of vector instructions (indexes
// of the staging and the outputs, rounding; an MFMA in seven): they take 65 %
// of the time, LDS 39 % (18 % bank conflicts), MFMA 35 %.  At 32 -> 16 by waits
// for the staged loads, two workgroups to a CU: 46 % of a wavefront's cycles
// (vector instructions 40 %, LDS 31 %, MFMA 26 %).  129x129x65 nodes: 16 -> 16
// channels 52 us (1.3 TB/s of
// activations, 290 TFLOP/s), 32 -> 16 119 us; 65x65x33, 32 -> 32 25 us; with
// 8-byte loads of both operands per MFMA and no staging (the general kernel
// below) these took 228, 228 and 98 us.
constexpr int CONV_M = 4;             // 16-voxel tiles a wavefront has in flight
constexpr int CONV_WAVES = 4, CONV_TPB = CONV_WAVES * 64;
constexpr int CONV_PAD = 32;          // voxels before (1) and past the region that dropped positions read
constexpr int CONV_BATCH = 6;         // 16-byte loads a lane has in flight while the region is staged

struct ConvBlock {
    int TZ, TX, TY, LZ, LX, LY;       // outputs and staged region
    int nbz, nbx, nby;                // blocks of the grid
    int tpp, tiles;                   // 16-voxel tiles of a plane, of the block
    int region;                       // staged voxels and pad
};

// A block's region of NCB 16-channel blocks into LDS: 64 units of 16 bytes of a
// line to a wavefront at a time, CONV_BATCH of them requested before the first
// is stored (no branch: off the grid the nearest voxel is read and zero
// stored).  X: the batch's first voxel and channel, ci its voxels' stride.
template <int NCB>
__device__ __forceinline__ void stage_region(const Vol &g, const ConvBlock &cb, const uint16_t *__restrict__ X, int ci,
                                             int k0, int i0, int j0, unsigned char *smem, int lane, int w) {
    constexpr int UPV = 2 * NCB;   // 16-byte units of a voxel
    const int nlines = cb.LX * cb.LY, upl = cb.LZ * UPV, nch = (upl + 63) >> 6, total = nlines * nch;
    const unsigned mch = 65536u / nch + 1, mlx = 65536u / cb.LX + 1;   // exact for the few hundred chunks here
    for (int ch = w; ch < total; ch += CONV_WAVES * CONV_BATCH) {
        uint4 v[CONV_BATCH];
        int at[CONV_BATCH];
#pragma unroll
        for (int q = 0; q < CONV_BATCH; q++) {
            const int cq = min(ch + q * CONV_WAVES, total - 1), ln = (int)(cq * mch >> 16);
            const int ly = (int)(ln * mlx >> 16), lx = ln - ly * cb.LX;
            const int gi = i0 - 1 + lx, gj = j0 - 1 + ly;
            const int u = min((cq - ln * nch) * 64 + lane, upl - 1), z = u / UPV, c = u - z * UPV, gk = k0 - 1 + z;
            const int gic = min(max(gi, 0), g.nx - 1), gjc = min(max(gj, 0), g.ny - 1), gkc = min(max(gk, 0), g.nz - 1);
            v[q] = *reinterpret_cast<const uint4 *>(X + (size_t)(gkc + g.nz * (gic + g.nx * gjc)) * ci + c * 8);
            const bool in = gi == gic && gj == gjc && gk == gkc;
            at[q] = (((c >> 1) * cb.region + 1 + ln * cb.LZ + z) * 32 + (c & 1) * 16) | (in ? 0 : 1);
        }
#pragma unroll
        for (int q = 0; q < CONV_BATCH; q++) {
            const unsigned keep = at[q] & 1 ? 0u : ~0u;
            *reinterpret_cast<uint4 *>(smem + (at[q] & ~1)) =
                make_uint4(v[q].x & keep, v[q].y & keep, v[q].z & keep, v[q].w & keep);
        }
    }
}

template <int NCB, int NBO, bool WREG>
__global__ void __launch_bounds__(CONV_TPB) k_conv_block(Vol g, ConvBlock cb, int co, const uint16_t *__restrict__ X,
                                                         const uint16_t *__restrict__ W, int wtrans,
                                                         const float *__restrict__ bias, const uint16_t *__restrict__ R,
                                                         int relu, int mirror, uint16_t *__restrict__ Y,
                                                         float *__restrict__ Yf) {
    constexpr int CI = 16 * NCB;
    extern __shared__ __align__(16) unsigned char smem[];
    unsigned char *ws = smem + (size_t)NCB * cb.region * 32;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int b = blockIdx.x;
    const int k0 = (b % cb.nbz) * cb.TZ;
    b /= cb.nbz;
    const int i0 = (b % cb.nbx) * cb.TX;
    b /= cb.nbx;
    const int j0 = (b % cb.nby) * cb.TY, batch = b / cb.nby;
    const int o0 = blockIdx.y * NBO * 16;
    const uint16_t *Xb = X + (size_t)batch * g.nv * CI;
    const int m16 = lane & 15, kq = 4 * (lane >> 4);
    // weights of output channel o0 + 16 ob + m16, tap t, input channels 16 c + kq ..: A operand
    auto load_w = [&](int ob, int t, int c) -> bf16x4 {
        if (!wtrans) return load4(W + ((size_t)(o0 + ob * 16 + m16) * TAPS + t) * CI + c * 16 + kq);
        bf16x4 a;   // W[input][t][output]
#pragma unroll
        for (int i = 0; i < 4; i++) a[i] = (short)W[((size_t)(c * 16 + kq + i) * TAPS + t) * co + o0 + ob * 16 + m16];
        return a;
    };
    // all taps', or this wavefront's share of nine taps', requested ahead of the
    // region (and the next nine ahead of the products)
    constexpr int NF = 9 * NCB * NBO, NW = WREG ? TAPS * NCB * NBO : (NF + CONV_WAVES - 1) / CONV_WAVES;
    bf16x4 wr[NW];
    auto fetch_w = [&](int dy) {
#pragma unroll
        for (int n = 0; n < NW; n++) {
            const int f = min(w + n * CONV_WAVES, NF - 1);
            wr[n] = load_w(f % NBO, 9 * dy + f / (NBO * NCB), (f / NBO) % NCB);
        }
    };
    if constexpr (WREG)
#pragma unroll
        for (int f = 0; f < NW; f++) wr[f] = load_w(f % NBO, f / (NBO * NCB), (f / NBO) % NCB);
    else
        fetch_w(0);
    __builtin_amdgcn_sched_barrier(0);
    stage_region<NCB>(g, cb, Xb, CI, k0, i0, j0, smem, lane, w);
    float bo[NBO][4];
#pragma unroll
    for (int ob = 0; ob < NBO; ob++)
#pragma unroll
        for (int e = 0; e < 4; e++) bo[ob][e] = bias ? bias[o0 + ob * 16 + kq + e] : 0.f;
    if (WREG) __syncthreads();
    const int sgn = mirror ? -32 : 32;
    for (int q0 = w; q0 < (WREG ? cb.tiles : CONV_WAVES); q0 += CONV_WAVES * CONV_M) {
        f32x4 acc[CONV_M][NBO];
        int pos[CONV_M];   // LDS byte of the lane's voxel and channel quarter
#pragma unroll
        for (int m = 0; m < CONV_M; m++) {
            const int q = min(q0 + m * CONV_WAVES, cb.tiles - 1), y = q / cb.tpp, qq = q - y * cb.tpp;
            pos[m] = (1 + ((y + 1) * cb.LX + 1) * cb.LZ + 16 * qq + m16) * 32 + 2 * kq;
#pragma unroll
            for (int ob = 0; ob < NBO; ob++) acc[m][ob] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int dy = 0; dy < 3; dy++) {
            if constexpr (!WREG) {
                if (dy) __syncthreads();
#pragma unroll
                for (int n = 0; n < NW; n++)
                    *reinterpret_cast<bf16x4 *>(ws + (size_t)min(w + n * CONV_WAVES, NF - 1) * 512 + lane * 8) = wr[n];
                __syncthreads();
                if (dy < 2) fetch_w(dy + 1);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int t9 = 0; t9 < 9; t9++) {
                const int off = sgn * ((t9 % 3 - 1) + cb.LZ * ((t9 / 3 - 1) + cb.LX * (dy - 1)));
#pragma unroll
                for (int c = 0; c < NCB; c++) {
                    bf16x4 x[CONV_M];
#pragma unroll
                    for (int m = 0; m < CONV_M; m++)
                        x[m] = *reinterpret_cast<const bf16x4 *>(smem + pos[m] + off + c * cb.region * 32);
#pragma unroll
                    for (int ob = 0; ob < NBO; ob++) {
                        bf16x4 a;
                        if constexpr (WREG) a = wr[((9 * dy + t9) * NCB + c) * NBO + ob];
                        else a = *reinterpret_cast<const bf16x4 *>(ws + (size_t)((t9 * NCB + c) * NBO + ob) * 512 + lane * 8);
#pragma unroll
                        for (int m = 0; m < CONV_M; m++)
                            acc[m][ob] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, x[m], acc[m][ob], 0, 0, 0);
                    }
                }
            }
        }
        // D[4(l/16)+i][l%16]: output channels kq .. kq+3 of voxel m16 of the tile
#pragma unroll
        for (int m = 0; m < CONV_M; m++) {
            const int q = q0 + m * CONV_WAVES;
            if (q >= cb.tiles) break;
            const int y = q / cb.tpp, p = 16 * (q - y * cb.tpp) + m16, lx = p / cb.LZ, z = p - lx * cb.LZ - 1;
            const int k = k0 + z, i = i0 + lx, j = j0 + y;
            if ((unsigned)z >= (unsigned)cb.TZ || lx >= cb.TX || k >= g.nz || i >= g.nx || j >= g.ny) continue;
            const size_t at = ((size_t)batch * g.nv + k + (size_t)g.nz * (i + (size_t)g.nx * j)) * co + o0 + kq;
#pragma unroll
            for (int ob = 0; ob < NBO; ob++) {
                float y4[4];
                uint2 r = {0, 0};
                if (R) r = *reinterpret_cast<const uint2 *>(R + at + ob * 16);
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    float yv = acc[m][ob][e] + bo[ob][e];
                    if (R) yv += bf2f((uint16_t)((e < 2 ? r.x : r.y) >> (16 * (e & 1))));
                    if (relu) yv = yv > 0.f ? yv : 0.f;
                    y4[e] = yv;
                }
                uint2 o;
                o.x = f2bf(y4[0]) | ((uint32_t)f2bf(y4[1]) << 16);
                o.y = f2bf(y4[2]) | ((uint32_t)f2bf(y4[3]) << 16);
                *reinterpret_cast<uint2 *>(Y + at + ob * 16) = o;
                if (Yf) *reinterpret_cast<float4 *>(Yf + at + ob * 16) = make_float4(y4[0], y4[1], y4[2], y4[3]);
            }
        }
    }
}

// The block of a grid: of the shapes whose tiles (at most `most`) and region
// (at most `lds` bytes) fit, the one with the least positions computed and
// voxels staged per output (a staged voxel costs about as much as a quarter
// of a computed one at 16 channels, a block `start` tiles before its first),
// a grid of too few blocks for `wide` workgroups a group counting as work too.
ConvBlock conv_block(const Vol &g, int nb, int ncb, int most, long lds, long wide, double start) {
    ConvBlock best{};
    double cost = 0.0;
    const double turn = 1.0 / (CONV_WAVES * CONV_M), share = 1.0 / (double)wide;
    for (int cuts = 1; cuts <= g.nz && (cuts <= 8 || !best.TZ); cuts++) {
        const int TZ = (g.nz + cuts - 1) / cuts;
        if (cuts > 1 && TZ == (g.nz + cuts - 2) / (cuts - 1)) continue;
        const int nbz = (g.nz + TZ - 1) / TZ;
        for (int TX = 1, last = 0; TX <= 8 && TX <= g.nx; TX++) {
            const int nbx = (g.nx + TX - 1) / TX, tpp = ((TZ + 2) * TX + 15) / 16;
            if (nbx == last) continue;   // as many blocks, larger
            last = nbx;
            for (int TY = 1; TY <= 4 && TY <= g.ny; TY++) {
                const int tiles = TY * tpp, region = (TZ + 2) * (TX + 2) * (TY + 2) + CONV_PAD;
                if (tiles > most || (long)region * ncb * 32 > lds) break;
                const int nby = (g.ny + TY - 1) / TY;
                const double blocks = (double)nb * nbz * nbx * nby;
                // rounds of `wide` workgroups; each as long as its tiles (in whole turns of the wavefronts) and staging
                const double rounds = std::max(1.0, blocks * share);
                const double v = rounds * (16.0 * std::ceil(tiles * turn) + 0.25 / 16.0 * region + start);
                if (!best.TZ || v < cost) best = {TZ, TX, TY, TZ + 2, TX + 2, TY + 2, nbz, nbx, nby, tpp, tiles, region}, cost = v;
            }
        }
    }
    return best;
}

constexpr long CONV_LDS = 80 << 10;       // two workgroups to a CU

// a kernel's dynamic LDS limit raised to CONV_LDS, once per device (a bit of `raised`)
int raise_lds(const void *kern, std::atomic<uint64_t> &raised) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev > 63) return -1;
    if (!(raised.load() >> dev & 1)) {
        if (hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)CONV_LDS) != hipSuccess) return -1;
        raised.fetch_or(1ull << dev);
    }
    return 0;
}

template <int NCB, int NBO, bool WREG>
int conv_launch(const Vol &g, int nb, int co, const uint16_t *x, const uint16_t *w, int wtrans, const float *bias,
                const uint16_t *res, int relu, int mirror, uint16_t *y, float *yf, hipStream_t s) {
    auto kern = k_conv_block<NCB, NBO, WREG>;
    static std::atomic<uint64_t> raised{0};
    if (raise_lds((const void *)kern, raised)) return -1;
    const long wlds = WREG ? 0 : 9L * NCB * NBO * 512;
    const int groups = co / (16 * NBO);
    const ConvBlock cb = conv_block(g, nb, NCB, WREG ? 1 << 20 : CONV_WAVES * CONV_M,
                                    (NCB * NBO == 1 ? CONV_LDS / 2 : CONV_LDS) - wlds, std::max(1, 512 / groups), 4.0);
    if (!cb.TZ) return -1;
    const long blocks = (long)nb * cb.nbz * cb.nbx * cb.nby;
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks, groups), dim3(CONV_TPB), (size_t)NCB * cb.region * 32 + wlds, s, g, cb,
                       co, x, w, wtrans, bias, res, relu, mirror, y, yf);
    return 0;
}

bool aligned(const void *p, unsigned n) { return ((uintptr_t)p & (n - 1)) == 0; }

}  // namespace

namespace learn {

thread_local hipError_t g_launch_err = hipSuccess;
int ret() { return (g_launch_err = hipGetLastError()) == hipSuccess ? 0 : -1; }
hipError_t launch_error() { return g_launch_err; }

// the block kernel takes up to 64 input channels and pointers aligned to its
// vector loads and stores
bool conv_block_ok(int ci, const uint16_t *x, const uint16_t *w, const uint16_t *res, const uint16_t *y, const float *yf) {
    return ci <= 64 && aligned(x, 16) && aligned(w, 8) && aligned(res, 8) && aligned(y, 8) && aligned(yf, 16);
}

int conv_fwd(const Vol &g, int nb, int ci, int co, const uint16_t *x, const uint16_t *w, int wtrans, const float *bias,
             const uint16_t *res, int relu, int mirror, uint16_t *y, float *yf, hipStream_t s) {
#define CONV_CASE(NCB, NBO, WREG) conv_launch<NCB, NBO, WREG>(g, nb, co, x, w, wtrans, bias, res, relu, mirror, y, yf, s)
    // two output blocks a workgroup halve the staging and the operand reads;
    // on a grid of too few blocks one gives twice the workgroups
    const bool two = co % 32 == 0 && (long)nb * g.nv * co >= 32L * 16 * 4096;
    switch (ci / 16) {
    case 1: return two ? CONV_CASE(1, 2, true) : CONV_CASE(1, 1, true);
    case 2: return two ? CONV_CASE(2, 2, false) : CONV_CASE(2, 1, true);
    case 3: return two ? CONV_CASE(3, 2, false) : CONV_CASE(3, 1, false);
    default: return two ? CONV_CASE(4, 2, false) : CONV_CASE(4, 1, false);
    }
#undef CONV_CASE
}

}  // namespace learn

namespace {

// the same for more than 64 input channels or less aligned operands:
// one wavefront computes 16 voxels x (NBO*16) output channels; the K loop
// runs over the taps and the 16-channel blocks of the input.  mirror reads
// tap t at the mirrored offset -off_t (the data gradient, with transposed
// weights).
template <int NBO>
__global__ void __launch_bounds__(256) k_conv_fwd_c(Vol g, int ci, int co, const uint16_t *__restrict__ X,
                                                    const uint16_t *__restrict__ W, const float *__restrict__ bias,
                                                    const uint16_t *__restrict__ R, int relu, int mirror,
                                                    uint16_t *__restrict__ Y, float *__restrict__ Yf) {
    const int l = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int groups = co / (16 * NBO);
    const int b = blockIdx.y / groups, og = blockIdx.y % groups;
    const int v0 = (blockIdx.x * 4 + wv) * 16;
    if (v0 >= g.nv) return;
    const uint16_t *Xb = X + (size_t)b * g.nv * ci;
    const int m = v0 + (l & 15), kq = 4 * (l >> 4);
    const Cell cm = cell(g, m);
    const int ncb = ci >> 4;
    f32x4 acc[NBO];
#pragma unroll
    for (int ob = 0; ob < NBO; ob++) acc[ob] = f32x4{0.f, 0.f, 0.f, 0.f};
    // weight row of this lane's output channel (column l%16 of B) per block
    const uint16_t *Wl = W + (size_t)(og * NBO * 16 + (l & 15)) * TAPS * ci + kq;
    const size_t wstride = (size_t)16 * TAPS * ci;   // next block of 16 output channels
#pragma unroll 3
    for (int t = 0; t < TAPS; t++) {
        const int vn = nbr(g, cm, mirror ? 26 - t : t);
        const uint16_t *xa = Xb + (size_t)(vn < 0 ? 0 : vn) * ci + kq;
        for (int cb = 0; cb < ncb; cb++) {
            bf16x4 a = {0, 0, 0, 0};
            if (vn >= 0) a = load4(xa + cb * 16);
#pragma unroll
            for (int ob = 0; ob < NBO; ob++) {
                const bf16x4 w = load4(Wl + ob * wstride + (size_t)t * ci + cb * 16);
                acc[ob] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, w, acc[ob], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int ob = 0; ob < NBO; ob++) {
        const int o = (og * NBO + ob) * 16 + (l & 15);
        const float bo = bias ? bias[o] : 0.f;
        for (int i = 0; i < 4; i++) {
            const int v = v0 + kq + i;
            if (v >= g.nv) continue;
            const size_t at = ((size_t)b * g.nv + v) * co + o;
            float y = acc[ob][i] + bo;
            if (R) y += bf2f(R[at]);
            if (relu) y = y > 0.f ? y : 0.f;
            Y[at] = f2bf(y);
            if (Yf) Yf[at] = y;
        }
    }
}

// WT[c][t][o] = W[o][t][c]
__global__ void k_transpose_w(const uint16_t *__restrict__ W, int ci, int co, uint16_t *__restrict__ WT) {
    const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long)co * TAPS * ci) return;
    const int c = (int)(idx % ci), t = (int)((idx / ci) % TAPS), o = (int)(idx / ((long)ci * TAPS));
    WT[((size_t)c * TAPS + t) * co + o] = W[idx];
}

// ---- weight gradient: dW[o][t][c] = sum_b sum_v dY[b][v][o] X[b][v+off_t][c],
// db[o] = sum dY[b][v][o].
//
// A workgroup takes NOB*16 output and NCB*16 input channels and every
// nslots-th block of voxels: the block of X with its halo and the block of dY
// are staged in LDS voxel by voxel, and the MFMA operands, which need four
// voxels of one channel to a lane, are read with the transposing LDS read.  K
// runs over the block's voxels inside the grid, 16 at a time (a table in LDS
// holds each one's place in the region, so a tap is one offset); a wavefront
// keeps the sums of seven taps in registers over all its blocks, the last one
// the bias as a tap of ones, and writes them once into its slot.  A second
// kernel sums the slots in a fixed order.
//
// Bound by waits for the staged loads, which few products hide: 55 % of a
// wavefront's cycles at 16 x 16 channels, 59 % at 32 x 16 (vector instructions
// 40 and 37 % of the time, LDS 18 and 22 %, MFMA 18 and 21 %).  65^3 nodes,
// batch 4: 16 x 16 channels 83 us and
// its slots' sum 8; with 2-byte loads of single voxels and a slot for 512
// voxels these took 1715 and 502 us.
typedef short s16x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ bf16x4 lds_read_tr(const unsigned char *p) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)p);
}

constexpr double WG_START = 20.0;   // a block's staging and table, in 16-voxel tiles' time
constexpr int WG_TAPS = 7;   // taps of a wavefront: 0-6, 7-13, 14-20, 21-26 and the bias

template <int NCB, int NOB>
__global__ void __launch_bounds__(CONV_TPB) k_wgrad_block(Vol g, ConvBlock cb, int nblocks, int ci, int co,
                                                          const uint16_t *__restrict__ X, const uint16_t *__restrict__ dY,
                                                          float *__restrict__ part) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int most = (cb.TZ * cb.TX * cb.TY + 15) & ~15;
    unsigned char *ys = smem + (size_t)NCB * cb.region * 32;                     // [NOB][voxel][16]
    int *table = reinterpret_cast<int *>(ys + (size_t)NOB * most * 32);          // [voxel] byte of its place
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ngc = ci / (16 * NCB), c0 = (blockIdx.y % ngc) * NCB * 16, o0 = (blockIdx.y / ngc) * NOB * 16;
    const int t0 = w * WG_TAPS;
    int off[WG_TAPS];
#pragma unroll
    for (int n = 0; n < WG_TAPS; n++) {
        const int t = min(t0 + n, TAPS - 1);
        off[n] = 32 * ((t % 3 - 1) + cb.LZ * (((t / 3) % 3 - 1) + cb.LX * (t / 9 - 1)));
    }
    f32x4 acc[WG_TAPS][NCB][NOB];
#pragma unroll
    for (int n = 0; n < WG_TAPS; n++)
#pragma unroll
        for (int c = 0; c < NCB; c++)
#pragma unroll
            for (int o = 0; o < NOB; o++) acc[n][c][o] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int blk = blockIdx.x; blk < nblocks; blk += gridDim.x) {
        int b = blk;
        const int k0 = (b % cb.nbz) * cb.TZ;
        b /= cb.nbz;
        const int i0 = (b % cb.nbx) * cb.TX;
        b /= cb.nbx;
        const int j0 = (b % cb.nby) * cb.TY, batch = b / cb.nby;
        const int tz = min(cb.TZ, g.nz - k0), tx = min(cb.TX, g.nx - i0), ty = min(cb.TY, g.ny - j0);
        const int count = tz * tx * ty;   // the block's voxels inside the grid, z fastest
        if (blk != (int)blockIdx.x) __syncthreads();   // the last block's reads
        stage_region<NCB>(g, cb, X + (size_t)batch * g.nv * ci + c0, ci, k0, i0, j0, smem, lane, w);
        for (int v = threadIdx.x; v < ((count + 15) & ~15); v += CONV_TPB) {
            const int vc = min(v, count - 1), z = vc % tz, x = (vc / tz) % tx, y = vc / (tz * tx);
            table[v] = (1 + ((y + 1) * cb.LX + x + 1) * cb.LZ + z + 1) * 32;
            const uint16_t *src = dY + ((size_t)batch * g.nv + k0 + z + (size_t)g.nz * (i0 + x + (size_t)g.nx * (j0 + y))) * co + o0;
#pragma unroll
            for (int o = 0; o < NOB; o++)
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    uint4 q = *reinterpret_cast<const uint4 *>(src + o * 16 + h * 8);
                    if (v >= count) q = make_uint4(0, 0, 0, 0);
                    *reinterpret_cast<uint4 *>(ys + ((size_t)o * most + v) * 32 + h * 16) = q;
                }
        }
        __syncthreads();
        const int row = 4 * (lane >> 4) + ((lane & 15) >> 2), quad = (lane & 3) * 8;   // what this lane reads of 16 voxels
        const bf16x4 one = {0x3F80, 0x3F80, 0x3F80, 0x3F80};
        for (int v0 = 0; v0 < count; v0 += 16) {
            const unsigned char *xp = smem + table[v0 + row] + quad;
            bf16x4 y[NOB];
#pragma unroll
            for (int o = 0; o < NOB; o++) y[o] = lds_read_tr(ys + ((size_t)o * most + v0 + row) * 32 + quad);
            const bool whole = v0 + 16 <= count;
#pragma unroll
            for (int n = 0; n < WG_TAPS; n++) {
                const bool bias = t0 + n == TAPS;   // uniform; more taps than that are not there
#pragma unroll
                for (int c = 0; c < NCB; c++) {
                    bf16x4 x = lds_read_tr(xp + off[n] + (size_t)c * cb.region * 32);
                    if (bias) x = one;
                    if (!whole)   // past the block: neither operand counts, whatever the region holds there
#pragma unroll
                        for (int e = 0; e < 4; e++) x[e] = v0 + 4 * (lane >> 4) + e < count ? x[e] : (short)0;
#pragma unroll
                    for (int o = 0; o < NOB; o++)
                        acc[n][c][o] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(y[o], x, acc[n][c][o], 0, 0, 0);
                }
            }
        }
    }
    // D[4(l/16)+i][l%16] = dW[o0 + 16 o + 4(l/16)+i][t][c0 + 16 c + l%16]
    const int r = lane & 15, kq = 4 * (lane >> 4);
    float *P = part + (size_t)blockIdx.x * ((size_t)co * TAPS * ci + co);
#pragma unroll
    for (int n = 0; n < WG_TAPS; n++) {
        const int t = t0 + n;
#pragma unroll
        for (int o = 0; o < NOB; o++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const size_t oc = o0 + o * 16 + kq + i;
                if (t < TAPS)
#pragma unroll
                    for (int c = 0; c < NCB; c++) P[(oc * TAPS + t) * ci + c0 + c * 16 + r] = acc[n][c][o][i];
                else if (t == TAPS && c0 == 0 && r == 0)
                    P[(size_t)co * TAPS * ci + oc] = acc[n][0][o][i];
            }
    }
}

// out[i] = sum of the slots' i: 64 entries to a workgroup, a quarter of the slots to a wavefront
__global__ void __launch_bounds__(256) k_sum_slots(const float *__restrict__ part, int nslots, long slot,
                                                   float *__restrict__ out) {
    __shared__ float sh[4][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const long i = (long)blockIdx.x * 64 + lane;
    const int per = (nslots + 3) / 4, k1 = min(nslots, (w + 1) * per);
    float s = 0.f;
    if (i < slot)
#pragma unroll 8
        for (int k = w * per; k < k1; k++) s += part[(size_t)k * slot + i];
    sh[w][lane] = s;
    __syncthreads();
    if (w == 0 && i < slot) out[i] = (sh[0][lane] + sh[1][lane]) + (sh[2][lane] + sh[3][lane]);
}

template <int NCB, int NOB>
int wgrad_launch(const Vol &g, int nb, int ci, int co, const uint16_t *x, const uint16_t *dy, float *part, long slots,
                 hipStream_t s) {
    auto kern = k_wgrad_block<NCB, NOB>;
    static std::atomic<uint64_t> raised{0};
    if (raise_lds((const void *)kern, raised)) return -1;
    const int groups = (ci / (16 * NCB)) * (co / (16 * NOB));
    // dY and the table take less than NOB + 1/8 blocks' regions
    // two workgroups to a CU; no more slots than the workspace has, whose
    // workgroups take larger blocks where they are few
    const long wide = std::min(slots, std::max(1L, 512L / groups));
    const ConvBlock cb = conv_block(g, nb, NCB + NOB, 1 << 20, CONV_LDS * 8 / 9, wide, WG_START);
    if (!cb.TZ) return -1;
    const long blocks = (long)nb * cb.nbz * cb.nbx * cb.nby;
    if (blocks >= 1L << 31) return -1;
    const long nslots = std::min(blocks, wide);
    const long most = ((long)cb.TZ * cb.TX * cb.TY + 15) & ~15L;
    hipLaunchKernelGGL(kern, dim3((unsigned)nslots, groups), dim3(CONV_TPB),
                       (size_t)NCB * cb.region * 32 + NOB * most * 32 + most * 4, s, g, cb, (int)blocks, ci, co, x, dy, part);
    return (int)nslots;
}

}  // namespace

namespace learn {

// partial sums of at most `slots` slots of co*27*ci + co floats, then their
// sum; for 16-byte aligned operands, 0 or -1
int conv_wgrad(const Vol &g, int nb, int ci, int co, const uint16_t *x, const uint16_t *dy, float *part, long slots,
               float *grad, hipStream_t s) {
    if (!aligned(x, 16) || !aligned(dy, 16) || slots < 1) return -1;
    const int ncb = ci / 16, nob = co / 16;
    int n;
#define WGRAD_CASE(NCB, NOB) wgrad_launch<NCB, NOB>(g, nb, ci, co, x, dy, part, slots, s)
    if (ncb % 2 == 0) n = nob % 2 == 0 ? WGRAD_CASE(2, 2) : WGRAD_CASE(2, 1);
    else if (ncb % 3 == 0) n = WGRAD_CASE(3, 1);
    else n = nob % 2 == 0 ? WGRAD_CASE(1, 2) : WGRAD_CASE(1, 1);
#undef WGRAD_CASE
    if (n < 1) return -1;
    const long slot = (long)co * TAPS * ci + co;
    hipLaunchKernelGGL(k_sum_slots, dim3((unsigned)((slot + 63) / 64)), dim3(256), 0, s, part, n, slot, grad);
    return 0;
}

}  // namespace learn

namespace {

// the same for less aligned operands: one wavefront per (voxel chunk, 16 output
// channels, 16 input channels), its partial sums in its own slot
constexpr int WCH = 512;   // voxels per chunk
__global__ void __launch_bounds__(256) k_conv_bwd_weight_c(Vol g, int nb, int ci, int co,
                                                           const uint16_t *__restrict__ X,
                                                           const uint16_t *__restrict__ dY, float *__restrict__ part) {
    const int l = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int per = (g.nv + WCH - 1) / WCH;
    const int nob = co >> 4, ncb = ci >> 4;
    const long w = (long)blockIdx.x * 4 + wv;   // over nb * per * nob * ncb
    if (w >= (long)nb * per * nob * ncb) return;
    const int cb = (int)(w % ncb), ob = (int)((w / ncb) % nob);
    const long chunk = w / ((long)ncb * nob);
    const int b = (int)(chunk / per), vbeg = (int)(chunk % per) * WCH;
    const int vend = min(g.nv, vbeg + WCH);
    const size_t slot = (size_t)co * TAPS * ci + co;
    float *P = part + chunk * slot;
    const uint16_t *Xb = X + (size_t)b * g.nv * ci, *dYb = dY + (size_t)b * g.nv * co;
    const int r = l & 15, kq = 4 * (l >> 4);
    const int o = ob * 16 + r, c = cb * 16 + r;
    float dbias = 0.f;
    for (int t = 0; t < TAPS; t++) {
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        for (int v0 = vbeg; v0 < vend; v0 += 16) {
            bf16x4 a, bb;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int v = v0 + kq + i;
                uint16_t av = 0, bv = 0;
                if (v < vend) {
                    av = dYb[(size_t)v * co + o];
                    const int vn = nbr(g, cell(g, v), t);
                    if (vn >= 0) bv = Xb[(size_t)vn * ci + c];
                    if (t == 0) dbias += bf2f(av);
                }
                a[i] = (short)av;
                bb[i] = (short)bv;
            }
            acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, bb, acc, 0, 0, 0);
        }
        // D[4(l/16)+i][l%16] = dW[ob*16 + kq+i][t][cb*16 + l%16]
#pragma unroll
        for (int i = 0; i < 4; i++) P[((size_t)(ob * 16 + kq + i) * TAPS + t) * ci + c] = acc[i];
    }
    if (cb == 0) {   // lanes sharing r hold disjoint voxel quarters
        dbias += __shfl_xor(dbias, 16, 64);
        dbias += __shfl_xor(dbias, 32, 64);
        if (l < 16) P[(size_t)co * TAPS * ci + o] = dbias;
    }
}

// ---- grid transfers.  Coarse node c of a level lies on fine node 2c per
// axis (fine n = 2 (coarse n - 1) + 1).  Restriction (full weighting):
// coarse[c] = scale * sum_{d in {-1,0,1}^3} w(d) fine[2c+d], w = prod of
// 1/2 (d = 0) and 1/4 (d = +-1), neighbours outside the grid left out.
// Interpolation (trilinear): fine[f] = scale * sum_c p(f - 2c) coarse[c],
// p = prod of 1 (d = 0) and 1/2 (d = +-1).  The restriction's transpose is
// the interpolation / 8 and the interpolation's transpose 8 x the restriction.
__global__ void k_restrict(Vol fg, Vol cg, int ch, float scale, const uint16_t *__restrict__ F,
                           uint16_t *__restrict__ Cc, int nb) {
    const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long)nb * cg.nv * ch) return;
    const int c = (int)(idx % ch);
    const long bv = idx / ch;
    const int b = (int)(bv / cg.nv), v = (int)(bv % cg.nv);
    const int k = v % cg.nz, i = (v / cg.nz) % cg.nx, j = v / (cg.nz * cg.nx);
    const uint16_t *Fb = F + (size_t)b * fg.nv * ch;
    float s = 0.f;
    for (int dy = -1; dy <= 1; dy++) {
        const int jj = 2 * j + dy;
        if ((unsigned)jj >= (unsigned)fg.ny) continue;
        for (int dx = -1; dx <= 1; dx++) {
            const int ii = 2 * i + dx;
            if ((unsigned)ii >= (unsigned)fg.nx) continue;
            for (int dz = -1; dz <= 1; dz++) {
                const int kk = 2 * k + dz;
                if ((unsigned)kk >= (unsigned)fg.nz) continue;
                const float w = (dy ? 0.25f : 0.5f) * (dx ? 0.25f : 0.5f) * (dz ? 0.25f : 0.5f);
                s += w * bf2f(Fb[((size_t)kk + fg.nz * ((size_t)ii + fg.nx * jj)) * ch + c]);
            }
        }
    }
    Cc[idx] = f2bf(scale * s);
}

__global__ void k_interp(Vol cg, Vol fg, int ch, float scale, const uint16_t *__restrict__ Cc,
                         uint16_t *__restrict__ F, int nb) {
    const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long)nb * fg.nv * ch) return;
    const int c = (int)(idx % ch);
    const long bv = idx / ch;
    const int b = (int)(bv / fg.nv), v = (int)(bv % fg.nv);
    const int k = v % fg.nz, i = (v / fg.nz) % fg.nx, j = v / (fg.nz * fg.nx);
    const uint16_t *Cb = Cc + (size_t)b * cg.nv * ch;
    // per axis: even fine index -> one coarse node (weight 1), odd -> the two
    // coarse nodes either side (1/2 each)
    const int j0 = j >> 1, j1 = (j + 1) >> 1, i0 = i >> 1, i1 = (i + 1) >> 1, k0 = k >> 1, k1 = (k + 1) >> 1;
    const float wy = (j & 1) ? 0.5f : 1.f, wx = (i & 1) ? 0.5f : 1.f, wz = (k & 1) ? 0.5f : 1.f;
    float s = 0.f;
    for (int a = 0; a < ((j & 1) ? 2 : 1); a++) {
        const int jj = a ? j1 : j0;
        for (int e = 0; e < ((i & 1) ? 2 : 1); e++) {
            const int ii = e ? i1 : i0;
            for (int h = 0; h < ((k & 1) ? 2 : 1); h++) {
                const int kk = h ? k1 : k0;
                s += (wy * wx * wz) * bf2f(Cb[((size_t)kk + cg.nz * ((size_t)ii + cg.nx * jj)) * ch + c]);
            }
        }
    }
    F[idx] = f2bf(scale * s);
}

// The same, eight channels to a thread (one 16-byte load per neighbour; the
// sums in the same order), for channels and pointers that allow it.  Bound by
// the bytes: interpolation to 129x129x65 nodes of 32 channels 36 us (195 us
// with one channel to a thread, bound by its index arithmetic), restriction
// from there of 16 channels 16 us (45).
struct Ch8 {
    float v[8];
    __device__ __forceinline__ void add(float w, const uint16_t *p) {
        const uint4 r = *reinterpret_cast<const uint4 *>(p);
        const uint32_t q[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] += w * __uint_as_float(e & 1 ? q[e / 2] & 0xFFFF0000u : q[e / 2] << 16);
    }
    __device__ __forceinline__ void store(float scale, uint16_t *p) const {
        uint32_t q[4];
#pragma unroll
        for (int e = 0; e < 4; e++) q[e] = f2bf(scale * v[2 * e]) | ((uint32_t)f2bf(scale * v[2 * e + 1]) << 16);
        *reinterpret_cast<uint4 *>(p) = make_uint4(q[0], q[1], q[2], q[3]);
    }
};

__global__ void __launch_bounds__(256) k_restrict8(Vol fg, Vol cg, int ch8, float scale, const uint16_t *__restrict__ F,
                                                   uint16_t *__restrict__ Cc) {
    const int idx = blockIdx.x * blockDim.x + threadIdx.x, b = blockIdx.y;   // over cg.nv * ch8
    if (idx >= cg.nv * ch8) return;
    const int v = idx / ch8, c = 8 * (idx - v * ch8), ch = 8 * ch8;
    const int k = v % cg.nz, i = (v / cg.nz) % cg.nx, j = v / (cg.nz * cg.nx);
    const uint16_t *Fb = F + (size_t)b * fg.nv * ch + c;
    Ch8 s = {{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int dy = -1; dy <= 1; dy++) {
        const int jj = 2 * j + dy;
        if ((unsigned)jj >= (unsigned)fg.ny) continue;
#pragma unroll
        for (int dx = -1; dx <= 1; dx++) {
            const int ii = 2 * i + dx;
            if ((unsigned)ii >= (unsigned)fg.nx) continue;
#pragma unroll
            for (int dz = -1; dz <= 1; dz++) {
                const int kk = 2 * k + dz;
                if ((unsigned)kk >= (unsigned)fg.nz) continue;
                s.add((dy ? 0.25f : 0.5f) * (dx ? 0.25f : 0.5f) * (dz ? 0.25f : 0.5f),
                      Fb + ((size_t)kk + fg.nz * ((size_t)ii + fg.nx * jj)) * ch);
            }
        }
    }
    s.store(scale, Cc + ((size_t)b * cg.nv + v) * ch + c);
}

__global__ void __launch_bounds__(256) k_interp8(Vol cg, Vol fg, int ch8, float scale, const uint16_t *__restrict__ Cc,
                                                 uint16_t *__restrict__ F) {
    const int idx = blockIdx.x * blockDim.x + threadIdx.x, b = blockIdx.y;   // over fg.nv * ch8
    if (idx >= fg.nv * ch8) return;
    const int v = idx / ch8, c = 8 * (idx - v * ch8), ch = 8 * ch8;
    const int k = v % fg.nz, i = (v / fg.nz) % fg.nx, j = v / (fg.nz * fg.nx);
    const uint16_t *Cb = Cc + (size_t)b * cg.nv * ch + c;
    const float w = ((j & 1) ? 0.5f : 1.f) * ((i & 1) ? 0.5f : 1.f) * ((k & 1) ? 0.5f : 1.f);
    Ch8 s = {{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}};
    for (int a = j >> 1; a <= (j + 1) >> 1; a++)
        for (int e = i >> 1; e <= (i + 1) >> 1; e++)
            for (int h = k >> 1; h <= (k + 1) >> 1; h++)
                s.add(w, Cb + ((size_t)h + cg.nz * ((size_t)e + cg.nx * a)) * ch);
    s.store(scale, F + ((size_t)b * fg.nv + v) * ch + c);
}

__global__ void k_add_bf16(uint16_t *__restrict__ a, const uint16_t *__restrict__ b, long n) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] = f2bf(bf2f(a[i]) + bf2f(b[i]));
}

// weighted mean squared error over the first nout of ystride channels:
// loss = sum_v sum_c wch[c] (Y[v][c] - T[v][c])^2 / (nvox nout); dY (bf16,
// ystride channels, zero beyond nout) = d loss / d Y; part[block] = block sums
__global__ void k_wmse(const float *__restrict__ Y, int ystride, const float *__restrict__ T, long nvox, int nout,
                       const float *__restrict__ wch, uint16_t *__restrict__ dY, float *__restrict__ part) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    float e2 = 0.f;
    if (i < nvox * ystride) {
        const int c = (int)(i % ystride);
        const long v = i / ystride;
        float gr = 0.f;
        if (c < nout) {
            const float e = Y[i] - T[v * nout + c];
            e2 = wch[c] * e * e;
            gr = 2.f * wch[c] * e / (float)(nvox * nout);
        }
        dY[i] = f2bf(gr);
    }
    for (int w = 32; w >= 1; w >>= 1) e2 += __shfl_xor(e2, w, 64);
    __shared__ float sh[4];
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = e2;
    __syncthreads();
    if (threadIdx.x == 0) part[blockIdx.x] = (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

hipStream_t st(void *s) { return static_cast<hipStream_t>(s); }
unsigned nblk(long n) { return (unsigned)((n + 255) / 256); }
bool chan_ok(int c) { return c >= 16 && c <= 256 && c % 16 == 0; }

// eight channels to a thread: whole groups of them, 16-byte aligned, indexes within int and the grid's y limit
bool ch8_ok(const Vol &g, int nb, int ch, const void *a, const void *b) {
    return ch % 8 == 0 && aligned(a, 16) && aligned(b, 16) && (long)g.nv * (ch / 8) < (1L << 31) - 256 && nb < 65536;
}

// ---- the U-Net of the warm start (4 levels, 16/32/48/64 channels, 15
// convolutions; additive skip connections; 594,432 weights + 528 biases).
// Level l has (n - 1) / 2^l + 1 nodes per axis.  Encoder: two convolutions
// per level (ReLU), the second's output kept as the level's skip, then a
// full-weighting restriction to the next level; bottom: two convolutions;
// decoder: trilinear interpolation to the finer level, a convolution plus
// that level's skip (ReLU), a second convolution (ReLU); a last 16 -> 16
// convolution without activation gives the output (FP32, channels 0..3
// used).
struct UConv {
    int ci, co;
};
constexpr UConv UNET[15] = {{16, 16}, {16, 16}, {16, 32}, {32, 32}, {32, 48}, {48, 48}, {48, 64}, {64, 64},
                            {64, 48}, {48, 48}, {48, 32}, {32, 32}, {32, 16}, {16, 16}, {16, 16}};
constexpr int UNET_LEVELS = 4;
// channels of the forward pass's buffers per level: A, B, S (skip)
constexpr int UA[UNET_LEVELS] = {32, 48, 64, 64}, UB[UNET_LEVELS] = {16, 32, 48, 64}, US[UNET_LEVELS] = {16, 32, 48, 0};

long unet_level_nv(int nx, int ny, int nz, int lev) {
    const int s = 1 << lev;
    return (long)((nx - 1) / s + 1) * ((ny - 1) / s + 1) * ((nz - 1) / s + 1);
}

}  // namespace

extern "C" {

int cl_conv3d_fwd_c(const uint16_t *x, int nb, int nx, int ny, int nz, int ci, int co, const uint16_t *w,
                    const float *bias, const uint16_t *res, int relu, int mirror, uint16_t *y, float *yf,
                    void *stream) {
    const Vol g{nx, ny, nz, nx * ny * nz};
    if (nb <= 0 || g.nv <= 0 || !chan_ok(ci) || !chan_ok(co)) return -1;
    if (conv_block_ok(ci, x, w, res, y, yf) &&
        conv_fwd(g, nb, ci, co, x, w, 0, bias, res, relu, mirror, y, yf, st(stream)) == 0)
        return ret();
    const int nbo = (co % 64 == 0) ? 4 : (co % 48 == 0) ? 3 : (co % 32 == 0) ? 2 : 1;
    const dim3 grid((g.nv + 63) / 64, nb * (co / (16 * nbo)));
    switch (nbo) {
    case 4: hipLaunchKernelGGL(k_conv_fwd_c<4>, grid, dim3(256), 0, st(stream), g, ci, co, x, w, bias, res, relu, mirror, y, yf); break;
    case 3: hipLaunchKernelGGL(k_conv_fwd_c<3>, grid, dim3(256), 0, st(stream), g, ci, co, x, w, bias, res, relu, mirror, y, yf); break;
    case 2: hipLaunchKernelGGL(k_conv_fwd_c<2>, grid, dim3(256), 0, st(stream), g, ci, co, x, w, bias, res, relu, mirror, y, yf); break;
    default: hipLaunchKernelGGL(k_conv_fwd_c<1>, grid, dim3(256), 0, st(stream), g, ci, co, x, w, bias, res, relu, mirror, y, yf); break;
    }
    return ret();
}

int cl_conv3d_transpose_w(const uint16_t *w, int ci, int co, uint16_t *wt, void *stream) {
    if (!chan_ok(ci) || !chan_ok(co)) return -1;
    const long n = (long)co * TAPS * ci;
    hipLaunchKernelGGL(k_transpose_w, dim3(nblk(n)), dim3(256), 0, st(stream), w, ci, co, wt);
    return ret();
}

int cl_conv3d_bwd_data_c(const uint16_t *dy, int nb, int nx, int ny, int nz, int ci, int co, const uint16_t *wt,
                         uint16_t *dx, void *stream) {
    // dX[v][c] = sum_t sum_o dY[v - off_t][o] W[o][t][c]: the forward
    // convolution of dY (co channels in, ci out) with WT[c][t][o] and the
    // mirrored taps
    return cl_conv3d_fwd_c(dy, nb, nx, ny, nz, co, ci, wt, nullptr, nullptr, 0, 1, dx, nullptr, stream);
}

long cl_conv3d_bwd_weight_c_workspace(int nb, int nx, int ny, int nz, int ci, int co) {
    const long nv = (long)nx * ny * nz, chunks = (long)nb * ((nv + WCH - 1) / WCH);
    return chunks * ((long)co * TAPS * ci + co) * (long)sizeof(float);
}

int cl_conv3d_bwd_weight_c(const uint16_t *x, const uint16_t *dy, int nb, int nx, int ny, int nz, int ci, int co,
                           float *grad, float *workspace, void *stream) {
    const Vol g{nx, ny, nz, nx * ny * nz};
    if (nb <= 0 || g.nv <= 0 || !chan_ok(ci) || !chan_ok(co)) return -1;
    const long chunks = (long)nb * ((g.nv + WCH - 1) / WCH);
    if (conv_wgrad(g, nb, ci, co, x, dy, workspace, chunks, grad, st(stream)) == 0) return ret();
    const long waves = chunks * (co / 16) * (ci / 16);
    const long slot = (long)co * TAPS * ci + co;
    if (chunks >= 1L << 31) return -1;
    hipLaunchKernelGGL(k_conv_bwd_weight_c, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, st(stream), g, nb, ci,
                       co, x, dy, workspace);
    hipLaunchKernelGGL(k_sum_slots, dim3((unsigned)((slot + 63) / 64)), dim3(256), 0, st(stream), workspace, (int)chunks,
                       slot, grad);
    return ret();
}

int cl_restrict(const uint16_t *fine, int nb, int nx, int ny, int nz, int ch, float scale, uint16_t *coarse,
                void *stream) {
    if (nb <= 0 || nx < 3 || ny < 3 || nz < 3 || !(nx & ny & nz & 1) || ch <= 0) return -1;
    const Vol fg{nx, ny, nz, nx * ny * nz};
    const Vol cg{(nx - 1) / 2 + 1, (ny - 1) / 2 + 1, (nz - 1) / 2 + 1, ((nx - 1) / 2 + 1) * ((ny - 1) / 2 + 1) * ((nz - 1) / 2 + 1)};
    if (ch8_ok(fg, nb, ch, fine, coarse)) {
        hipLaunchKernelGGL(k_restrict8, dim3(nblk((long)cg.nv * (ch / 8)), nb), dim3(256), 0, st(stream), fg, cg, ch / 8,
                           scale, fine, coarse);
        return ret();
    }
    const long n = (long)nb * cg.nv * ch;
    hipLaunchKernelGGL(k_restrict, dim3(nblk(n)), dim3(256), 0, st(stream), fg, cg, ch, scale, fine, coarse, nb);
    return ret();
}

int cl_interp(const uint16_t *coarse, int nb, int nx, int ny, int nz, int ch, float scale, uint16_t *fine,
              void *stream) {
    if (nb <= 0 || nx < 3 || ny < 3 || nz < 3 || !(nx & ny & nz & 1) || ch <= 0) return -1;
    const Vol fg{nx, ny, nz, nx * ny * nz};
    const Vol cg{(nx - 1) / 2 + 1, (ny - 1) / 2 + 1, (nz - 1) / 2 + 1, ((nx - 1) / 2 + 1) * ((ny - 1) / 2 + 1) * ((nz - 1) / 2 + 1)};
    if (ch8_ok(fg, nb, ch, coarse, fine)) {
        hipLaunchKernelGGL(k_interp8, dim3(nblk((long)fg.nv * (ch / 8)), nb), dim3(256), 0, st(stream), cg, fg, ch / 8,
                           scale, coarse, fine);
        return ret();
    }
    const long n = (long)nb * fg.nv * ch;
    hipLaunchKernelGGL(k_interp, dim3(nblk(n)), dim3(256), 0, st(stream), cg, fg, ch, scale, coarse, fine, nb);
    return ret();
}

int cl_add_bf16(uint16_t *a, const uint16_t *b, long n, void *stream) {
    hipLaunchKernelGGL(k_add_bf16, dim3(nblk(n)), dim3(256), 0, st(stream), a, b, n);
    return ret();
}

int cl_wmse(const float *y, int ystride, const float *target, long nvox, int nout, const float *wch, uint16_t *dy,
            float *partial, void *stream) {
    if (nout <= 0 || nout > ystride) return -1;
    hipLaunchKernelGGL(k_wmse, dim3(nblk(nvox * ystride)), dim3(256), 0, st(stream), y, ystride, target, nvox, nout, wch,
                       dy, partial);
    return ret();
}

}  // extern "C"

extern "C" {

int cl_unet_params(long *n_weights, long *n_biases) {
    long nw = 0, nb = 0;
    for (const UConv &c : UNET) {
        nw += (long)c.co * TAPS * c.ci;
        nb += c.co;
    }
    if (n_weights) *n_weights = nw;
    if (n_biases) *n_biases = nb;
    return 0;
}

long cl_unet_workspace(int nb, int nx, int ny, int nz) {
    long bytes = 0;
    for (int l = 0; l < UNET_LEVELS; l++) {
        const long nv = (long)nb * unet_level_nv(nx, ny, nz, l);
        // bf16 buffers A, B, S of the level, 256-byte aligned
        for (int ch : {UA[l], UB[l], US[l]}) bytes += (nv * ch * 2 + 255) / 256 * 256;
    }
    return bytes;
}

int cl_unet_forward(const uint16_t *x, int nb, int nx, int ny, int nz, const uint16_t *w, const float *bias,
                    float *out, void *workspace, void *stream) {
    for (int n : {nx, ny, nz})
        if (n < 17 || (n - 1) % 8) return -1;   // four levels of at least 3 nodes per axis
    if (nb <= 0 || !x || !w || !bias || !out || !workspace) return -1;
    // carve the buffers in the order cl_unet_workspace counts them
    uint16_t *A[UNET_LEVELS], *B[UNET_LEVELS], *Sk[UNET_LEVELS];
    char *p = static_cast<char *>(workspace);
    for (int l = 0; l < UNET_LEVELS; l++) {
        const long nv = (long)nb * unet_level_nv(nx, ny, nz, l);
        uint16_t **slots[3] = {&A[l], &B[l], &Sk[l]};
        const int chs[3] = {UA[l], UB[l], US[l]};
        for (int q = 0; q < 3; q++) {
            *slots[q] = reinterpret_cast<uint16_t *>(p);
            p += (nv * chs[q] * 2 + 255) / 256 * 256;
        }
    }
    int d[UNET_LEVELS][3];
    for (int l = 0; l < UNET_LEVELS; l++) {
        const int s = 1 << l;
        d[l][0] = (nx - 1) / s + 1;
        d[l][1] = (ny - 1) / s + 1;
        d[l][2] = (nz - 1) / s + 1;
    }
    const uint16_t *wl[15];
    const float *bl[15];
    {
        long ow = 0, ob = 0;
        for (int i = 0; i < 15; i++) {
            wl[i] = w + ow;
            bl[i] = bias + ob;
            ow += (long)UNET[i].co * TAPS * UNET[i].ci;
            ob += UNET[i].co;
        }
    }
    int li = 0;
    auto conv = [&](int lev, const uint16_t *in, const uint16_t *res, int relu, uint16_t *y, float *yf) {
        const UConv &c = UNET[li];
        const int r = cl_conv3d_fwd_c(in, nb, d[lev][0], d[lev][1], d[lev][2], c.ci, c.co, wl[li], bl[li], res, relu, 0,
                                      y, yf, stream);
        li++;
        return r;
    };
    int rc = 0;
    // encoder
    rc |= conv(0, x, nullptr, 1, B[0], nullptr);
    rc |= conv(0, B[0], nullptr, 1, Sk[0], nullptr);
    rc |= cl_restrict(Sk[0], nb, d[0][0], d[0][1], d[0][2], 16, 1.f, B[1], stream);
    rc |= conv(1, B[1], nullptr, 1, A[1], nullptr);
    rc |= conv(1, A[1], nullptr, 1, Sk[1], nullptr);
    rc |= cl_restrict(Sk[1], nb, d[1][0], d[1][1], d[1][2], 32, 1.f, B[2], stream);
    rc |= conv(2, B[2], nullptr, 1, A[2], nullptr);
    rc |= conv(2, A[2], nullptr, 1, Sk[2], nullptr);
    rc |= cl_restrict(Sk[2], nb, d[2][0], d[2][1], d[2][2], 48, 1.f, B[3], stream);
    // bottom
    rc |= conv(3, B[3], nullptr, 1, A[3], nullptr);
    rc |= conv(3, A[3], nullptr, 1, B[3], nullptr);
    // decoder
    rc |= cl_interp(B[3], nb, d[2][0], d[2][1], d[2][2], 64, 1.f, A[2], stream);
    rc |= conv(2, A[2], Sk[2], 1, B[2], nullptr);
    rc |= conv(2, B[2], nullptr, 1, A[2], nullptr);
    rc |= cl_interp(A[2], nb, d[1][0], d[1][1], d[1][2], 48, 1.f, A[1], stream);
    rc |= conv(1, A[1], Sk[1], 1, B[1], nullptr);
    rc |= conv(1, B[1], nullptr, 1, A[1], nullptr);
    rc |= cl_interp(A[1], nb, d[0][0], d[0][1], d[0][2], 32, 1.f, A[0], stream);
    rc |= conv(0, A[0], Sk[0], 1, B[0], nullptr);
    rc |= conv(0, B[0], nullptr, 1, A[0], nullptr);
    rc |= conv(0, A[0], nullptr, 0, B[0], out);
    return rc ? -1 : 0;
}

}  // extern "C"
