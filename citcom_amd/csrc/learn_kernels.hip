// BF16 MFMA kernels of the learned warm start: a 3-D convolutional network
// (3x3x3 kernels, 16 channels, zero padding) trained on the GPU by these
// forward and backward kernels.  No counterpart in the reference.
//
// Layouts: activations X[b][v][16] bf16, v = k + nz*(i + nx*j) (z fastest,
// the solver's node order); weights W[o][t][c] bf16 with FP32 master copies,
// tap t = (dz+1) + 3(dx+1) + 9(dy+1).  Every product runs on
// v_mfma_f32_16x16x16_bf16 with FP32 accumulation.  Operand layout of one
// 16x16x16 MFMA on a wavefront (checked on the device): lane l holds
// A[l%16][4(l/16)+i], B[4(l/16)+i][l%16] and D[4(l/16)+i][l%16], i = 0..3.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <mutex>
#include <string>

#include "../../include/citcom_learn.h"
#include "learn_common.h"

using namespace learn;

namespace {

constexpr int CH = 16;   // channels (padded)
constexpr int TAPS = 27;

// ---- backward through the activation: dYp = dY * (Y > 0)
__global__ void k_relu_bwd(const uint16_t *__restrict__ Y, uint16_t *__restrict__ dY, long n) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && !(bf2f(Y[i]) > 0.f)) dY[i] = 0;
}

// Up to this many voxels a wavefront that takes 16 of them and all their loads
// at once beats the staged blocks (unet_kernels.hip): four layers and their
// launches at 16 x 11^3 voxels 37.6 us against 42.3, 17^3 31.9 and 36.1, but
// 4 x 24x30x20 54.5 and 47.2, 40^3 58.7 and 47.5.
constexpr long SMALL_VOXELS = 32768;

// ---- forward, small volumes: Y[v][o] = act(sum_t sum_c X[v+off_t][c] W[o][t][c] + bias[o])
__global__ void __launch_bounds__(256) k_conv_fwd(Vol g, const uint16_t *__restrict__ X, const uint16_t *__restrict__ W,
                                                  const float *__restrict__ bias, int relu, uint16_t *__restrict__ Y,
                                                  float *__restrict__ Yf) {
    const int l = threadIdx.x & 63, wv = threadIdx.x >> 6, b = blockIdx.y;
    const int v0 = (blockIdx.x * 4 + wv) * 16;
    if (v0 >= g.nv) return;
    const uint16_t *Xb = X + (size_t)b * g.nv * CH;
    const int m = v0 + (l & 15), kq = 4 * (l >> 4);
    const Cell cm = cell(g, m);
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < TAPS; t++) {
        const int vn = nbr(g, cm, t);
        bf16x4 a = {0, 0, 0, 0};
        if (vn >= 0) a = load4(Xb + (size_t)vn * CH + kq);
        const bf16x4 w = load4(W + ((size_t)(l & 15) * TAPS + t) * CH + kq);
        acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, w, acc, 0, 0, 0);
    }
    const int o = l & 15;
    for (int i = 0; i < 4; i++) {
        const int v = v0 + kq + i;
        if (v >= g.nv) continue;
        float y = acc[i] + bias[o];
        if (relu) y = y > 0.f ? y : 0.f;
        Y[((size_t)b * g.nv + v) * CH + o] = f2bf(y);
        if (Yf) Yf[((size_t)b * g.nv + v) * CH + o] = y;
    }
}

// ---- backward data, small volumes or less aligned operands: dX[v][c] = sum_t sum_o dY[v-off_t][o] W[o][t][c]
__global__ void __launch_bounds__(256) k_conv_bwd_data(Vol g, const uint16_t *__restrict__ dY,
                                                       const uint16_t *__restrict__ W, uint16_t *__restrict__ dX) {
    __shared__ __align__(16) uint16_t Wt[TAPS][CH][CH];   // [t][c][o]
    for (int idx = threadIdx.x; idx < TAPS * CH * CH; idx += blockDim.x) {
        const int o = idx % CH, c = (idx / CH) % CH, t = idx / (CH * CH);
        Wt[t][c][o] = W[((size_t)o * TAPS + t) * CH + c];
    }
    __syncthreads();
    const int l = threadIdx.x & 63, wv = threadIdx.x >> 6, b = blockIdx.y;
    const int v0 = (blockIdx.x * 4 + wv) * 16;
    if (v0 >= g.nv) return;
    const uint16_t *dYb = dY + (size_t)b * g.nv * CH;
    const int m = v0 + (l & 15), kq = 4 * (l >> 4);
    const Cell cm = cell(g, m);
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < TAPS; t++) {
        // the output voxel u with u + off_t = m is the neighbour of m at the
        // mirrored tap 26 - t
        const int u = nbr(g, cm, 26 - t);
        bf16x4 a = {0, 0, 0, 0};
        if (u >= 0) a = load4(dYb + (size_t)u * CH + kq);
        const bf16x4 w = load4(&Wt[t][l & 15][kq]);
        acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, w, acc, 0, 0, 0);
    }
    const int c = l & 15;
    for (int i = 0; i < 4; i++) {
        const int v = v0 + kq + i;
        if (v < g.nv) dX[((size_t)b * g.nv + v) * CH + c] = f2bf(acc[i]);
    }
}

// chunks of voxels whose partial sums a caller's workspace has slots for
constexpr int WCHUNK = 256;

// mean squared error over the first nout channels; dY = d loss / d Y in bf16
__global__ void k_mse(const float *__restrict__ Y, const float *__restrict__ T, long nvox, int nout,
                      uint16_t *__restrict__ dY, float *__restrict__ part) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    float e2 = 0.f;
    if (i < nvox * CH) {
        const int c = (int)(i % CH);
        float g = 0.f;
        if (c < nout) {
            const float e = Y[i] - T[i];
            e2 = e * e;
            g = 2.f * e / (float)(nvox * nout);
        }
        dY[i] = f2bf(g);
    }
    for (int w = 32; w >= 1; w >>= 1) e2 += __shfl_xor(e2, w, 64);
    __shared__ float sh[4];
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = e2;
    __syncthreads();
    if (threadIdx.x == 0) part[blockIdx.x] = (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

// Adam on the FP32 master weights, then the BF16 copy
__global__ void k_adam(float *__restrict__ w, const float *__restrict__ gr, float *__restrict__ m, float *__restrict__ v,
                       long n, float lr, float b1, float b2, float eps, float c1, float c2, uint16_t *__restrict__ wbf,
                       const unsigned char *__restrict__ mask) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (mask && !mask[i]) return;
    const float g = gr[i];
    m[i] = b1 * m[i] + (1.f - b1) * g;
    v[i] = b2 * v[i] + (1.f - b2) * g * g;
    const float mh = m[i] / c1, vh = v[i] / c2;
    w[i] -= lr * mh / (sqrtf(vh) + eps);
    if (wbf) wbf[i] = f2bf(w[i]);
}

__global__ void k_to_bf16(const float *__restrict__ a, uint16_t *__restrict__ b, long n) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) b[i] = f2bf(a[i]);
}

hipStream_t st(void *s) { return static_cast<hipStream_t>(s); }

// ---- the weight gradient's partial sums without a workspace argument: a
// file-scope device array, one copy per GPU, held until the process ends.
// Host code never passes `scratch` itself to a kernel (its host-side name is
// not a device address): the device address comes from hipGetSymbolAddress,
// once per device with that device current, and is kept in scratch_ptr.
constexpr long SCRATCH_FLOATS = 4L << 20;   // 16 MiB
__device__ __align__(256) float scratch[SCRATCH_FLOATS];
constexpr int MAX_DEVICES = 64;
float *scratch_ptr[MAX_DEVICES];
std::once_flag scratch_once[MAX_DEVICES];
hipError_t scratch_err[MAX_DEVICES];

// the device address of this device's scratch array (nullptr on failure,
// with the message in *why)
float *scratch_on_current_device(const char **why) {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES) {
        *why = "no current HIP device (or more devices than the library tracks)";
        return nullptr;
    }
    std::call_once(scratch_once[dev], [dev] {
        void *p = nullptr;
        scratch_err[dev] = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        scratch_ptr[dev] = scratch_err[dev] == hipSuccess ? static_cast<float *>(p) : nullptr;
    });
    if (!scratch_ptr[dev]) *why = "hipGetSymbolAddress of the scratch array failed";
    return scratch_ptr[dev];
}

thread_local std::string g_learn_err;

}  // namespace

extern "C" {

int cl_conv3d_fwd(const uint16_t *x, int nb, int nx, int ny, int nz, const uint16_t *w, const float *bias, int relu,
                  uint16_t *y, float *yf, void *stream) {
    const Vol g{nx, ny, nz, nx * ny * nz};
    if (bias && nb > 0 && g.nv > 0 && (long)nb * g.nv <= SMALL_VOXELS) {
        hipLaunchKernelGGL(k_conv_fwd, dim3((g.nv + 63) / 64, nb), dim3(256), 0, st(stream), g, x, w, bias, relu, y, yf);
        return ret();
    }
    return cl_conv3d_fwd_c(x, nb, nx, ny, nz, CH, CH, w, bias, nullptr, relu, 0, y, yf, stream);
}

int cl_relu_bwd(const uint16_t *y, uint16_t *dy, long n, void *stream) {
    hipLaunchKernelGGL(k_relu_bwd, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st(stream), y, dy, n);
    return ret();
}

int cl_conv3d_bwd_data(const uint16_t *dy, int nb, int nx, int ny, int nz, const uint16_t *w, uint16_t *dx,
                       void *stream) {
    const Vol g{nx, ny, nz, nx * ny * nz};
    // the forward convolution of dy with the weights read transposed and the
    // taps mirrored
    if (nb > 0 && g.nv > 0 && (long)nb * g.nv > SMALL_VOXELS && conv_block_ok(CH, dy, w, nullptr, dx, nullptr) &&
        conv_fwd(g, nb, CH, CH, dy, w, 1, nullptr, nullptr, 0, 1, dx, nullptr, st(stream)) == 0)
        return ret();
    hipLaunchKernelGGL(k_conv_bwd_data, dim3((g.nv + 63) / 64, nb), dim3(256), 0, st(stream), g, dy, w, dx);
    return ret();
}

long cl_conv3d_bwd_weight_workspace(int nb, int nx, int ny, int nz) {
    const long nv = (long)nx * ny * nz, chunks = nb * ((nv + WCHUNK - 1) / WCHUNK);
    return ((chunks + 3) / 4 * 4) * (TAPS * CH * CH + CH) * (long)sizeof(float);
}

int cl_conv3d_bwd_weight(const uint16_t *x, const uint16_t *dy, int nb, int nx, int ny, int nz, float *grad,
                         float *workspace, void *stream) {
    const Vol g{nx, ny, nz, nx * ny * nz};
    const long slots = cl_conv3d_bwd_weight_workspace(nb, nx, ny, nz) / ((TAPS * CH * CH + CH) * (long)sizeof(float));
    if (nb > 0 && g.nv > 0 && conv_wgrad(g, nb, CH, CH, x, dy, workspace, slots, grad, st(stream)) == 0) return ret();
    // (a slot for 256 voxels holds at least as many as the general call's for 512)
    return cl_conv3d_bwd_weight_c(x, dy, nb, nx, ny, nz, CH, CH, grad, workspace, stream);
}

long cl_scratch_bytes(void) { return SCRATCH_FLOATS * (long)sizeof(float); }

const char *cl_last_error(void) { return g_learn_err.c_str(); }

int cl_conv3d_bwd_weight_noalloc(const uint16_t *x, const uint16_t *dy, int nb, int nx, int ny, int nz, float *grad,
                                 void *stream) {
    const Vol g{nx, ny, nz, nx * ny * nz};
    if (nb <= 0 || nx <= 0 || ny <= 0 || nz <= 0) {
        g_learn_err = "cl_conv3d_bwd_weight_noalloc: empty volume";
        return -1;
    }
    const long need = cl_conv3d_bwd_weight_workspace(nb, nx, ny, nz);
    if (need > cl_scratch_bytes()) {
        g_learn_err = "cl_conv3d_bwd_weight_noalloc: " + std::to_string(nb) + " volumes of " + std::to_string(g.nv) +
                      " voxels need " + std::to_string(need) + " bytes of partial sums, more than the " +
                      std::to_string(cl_scratch_bytes()) + "-byte scratch array";
        return -1;
    }
    const char *why = "";
    float *part = scratch_on_current_device(&why);
    if (!part) {
        g_learn_err = std::string("cl_conv3d_bwd_weight_noalloc: ") + why;
        return -1;
    }
    // every slot of partial sums that is summed is written in full before, so
    // nothing is cleared
    if (cl_conv3d_bwd_weight(x, dy, nb, nx, ny, nz, grad, part, stream) == 0) return 0;
    // sizes that fit the scratch array are refused by HIP only
    g_learn_err = std::string("cl_conv3d_bwd_weight_noalloc: ") + hipGetErrorString(launch_error());
    return -1;
}

int cl_mse(const float *y, const float *target, long nvox, int nout, uint16_t *dy, float *partial, void *stream) {
    hipLaunchKernelGGL(k_mse, dim3((unsigned)((nvox * CH + 255) / 256)), dim3(256), 0, st(stream), y, target, nvox, nout,
                       dy, partial);
    return ret();
}

int cl_adam(float *w, const float *g, float *m, float *v, long n, float lr, float b1, float b2, float eps, int step,
            uint16_t *wbf, const unsigned char *mask, void *stream) {
    const float c1 = 1.f - powf(b1, (float)step), c2 = 1.f - powf(b2, (float)step);
    hipLaunchKernelGGL(k_adam, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st(stream), w, g, m, v, n, lr, b1, b2,
                       eps, c1, c2, wbf, mask);
    return ret();
}

int cl_to_bf16(const float *a, uint16_t *b, long n, void *stream) {
    hipLaunchKernelGGL(k_to_bf16, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st(stream), a, b, n);
    return ret();
}

}  // extern "C"
