// gfx950 kernels of the CitcomCU hot path.
//
// Every scatter-add of the reference (element loops adding into nodes) is
// written here as a per-node gather over the node's elements in increasing
// element number, which reproduces the reference's summation order and
// rounding points, so these kernels agree bit for bit with the reference
// wherever the reference itself is deterministic.  Built with
// -ffp-contract=off for that reason.  The stiffness operator is bandwidth
// bound (2 flops per 4-byte coefficient): coefficient streams are read once,
// coalesced, 256-byte aligned; vectors are gathered through L2.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <cfloat>
#include <cmath>
#include <type_traits>

#include "chip_kernels.h"

namespace chip {

__constant__ double cNv[64];   // N.vpt   (Shape_functions.c:104-110)
__constant__ double cNp[8];    // N.ppt at the element centre
__constant__ double cMv[16];   // M.vpt   (2-D surface shape functions)
__constant__ double cMxv[32];  // Mx.vpt
__constant__ int cOffz[9] = {0, 0, 0, 0, 0, 1, 1, 1, 1};
__constant__ int cOffx[9] = {0, 0, 1, 1, 0, 0, 1, 1, 0};
__constant__ int cOffy[9] = {0, 0, 0, 1, 1, 0, 0, 1, 1};
// local node of offsets (dz, dx, dy): cLoc[dz + 2 dx + 4 dy]
__constant__ int cLoc[8] = {1, 5, 2, 6, 4, 8, 3, 7};

namespace {
constexpr int TPB = 256;
inline int nblk(long n, int tpb = TPB) { return (int)std::max<long>(1, (n + tpb - 1) / tpb); }
}  // namespace

int upload_constants() {
    const double B = 0.57735026918962576451;
    const float b = (float)B;
    const float gp[9][3] = {{0, 0, 0}, {-b, -b, -b}, {b, -b, -b}, {b, b, -b}, {-b, b, -b},
                            {-b, -b, b}, {b, -b, b}, {b, b, b}, {-b, b, b}};
    const float sp[5][2] = {{0, 0}, {-b, -b}, {b, -b}, {b, b}, {-b, b}};
    const int bbv[3][9] = {{0, 1, 2, 2, 1, 1, 2, 2, 1}, {0, 1, 1, 2, 2, 1, 1, 2, 2}, {0, 1, 1, 1, 1, 2, 2, 2, 2}};
    auto lp = [](int p, double y) { return p == 1 ? 0.5 * (1 - y) : (p == 2 ? 0.5 * (1 + y) : 0.0); };
    auto ld = [](int p) { return p == 1 ? -0.5 : (p == 2 ? 0.5 : 0.0); };
    double Nv[64], Np[8], Mv[16], Mxv[32];
    for (int i = 1; i <= 8; i++) {
        for (int j = 1; j <= 8; j++) {
            double v = 1.0;
            for (int d = 1; d <= 3; d++) v *= lp(bbv[d - 1][i], gp[j][d - 1]);
            Nv[8 * (i - 1) + j - 1] = v;
        }
        double v = 1.0;
        for (int d = 1; d <= 3; d++) v *= lp(bbv[d - 1][i], 0.0);
        Np[i - 1] = v;
    }
    // construct_shape_functions, surface part (Shape_functions.c:130-158)
    for (int j = 1; j <= 4; j++)
        for (int k = 1; k <= 4; k++) {
            Mv[4 * (j - 1) + k - 1] = lp(bbv[0][j], sp[k][0]) * lp(bbv[1][j], sp[k][1]);
            Mxv[4 * (j - 1) + k - 1] = ld(bbv[0][j]) * lp(bbv[1][j], sp[k][1]);
            Mxv[16 + 4 * (j - 1) + k - 1] = ld(bbv[1][j]) * lp(bbv[0][j], sp[k][0]);
        }
    if (hipMemcpyToSymbol(HIP_SYMBOL(cNv), Nv, sizeof Nv) != hipSuccess) return -1;
    if (hipMemcpyToSymbol(HIP_SYMBOL(cNp), Np, sizeof Np) != hipSuccess) return -1;
    if (hipMemcpyToSymbol(HIP_SYMBOL(cMv), Mv, sizeof Mv) != hipSuccess) return -1;
    if (hipMemcpyToSymbol(HIP_SYMBOL(cMxv), Mxv, sizeof Mxv) != hipSuccess) return -1;
    return 0;
}

// ---------------------------------------------------------------------------
// index helpers

__device__ __forceinline__ int nid(const Geo &g, int k, int i, int j) { return k + g.noz * (i + g.nox * j); }

__device__ __forceinline__ void node_kij(const Geo &g, int n, int &k, int &i, int &j) {
    k = n % g.noz;
    const int t = n / g.noz;
    i = t % g.nox;
    j = t / g.nox;
}

__device__ __forceinline__ void colour_kij(const Geo &g, int c, int q, int &k, int &i, int &j) {
    const int r = q - g.cs[c];
    const int nz = g.cz[c], nx = g.cx[c];
    const int kk = r % nz, t = r / nz;
    k = 2 * kk + (c & 1);
    i = 2 * (t % nx) + ((c >> 1) & 1);
    j = 2 * (t / nx) + ((c >> 2) & 1);
}

// colour-ordered index of node (k, i, j) of colour c (inverse of colour_kij)
__device__ __forceinline__ int colour_index(const Geo &g, int c, int k, int i, int j) {
    return g.cs[c] + (k >> 1) + g.cz[c] * ((i >> 1) + g.cx[c] * (j >> 1));
}

__device__ __forceinline__ int colour_of(const Geo &g, int q) {
    int c = 0;
#pragma unroll
    for (int m = 1; m < 8; m++) c += (q >= g.cs[m]);
    return c;
}

// colour of q, or -1 for a padding slot
__device__ __forceinline__ int colour_valid(const Geo &g, int q) {
    if (q >= g.pitch) return -1;
    const int c = colour_of(g, q);
    return (q - g.cs[c] < g.cn[c]) ? c : -1;
}

// Stiffness storage: 64-node tiles in colour order, each tile holding its
// 243 coefficient runs of 64 floats back to back, so one wavefront reads
// 243 contiguous 256-byte lines (62 KB) per row product.
__device__ __forceinline__ size_t ktile(int q) { return (size_t)(q >> 6) * (KROW * 64) + (q & 63); }

// Workgroups are dispatched to the 8 XCDs round-robin.  This gives XCD x a
// contiguous range of the grid's tiles, so the vector entries that
// neighbouring tiles share are fetched into one L2 rather than several.
__device__ __forceinline__ int xcd_tile(int b, int nb) {
    const int x = b & 7, y = b >> 3, qn = nb >> 3, rn = nb & 7;
    return (x < rn ? x * (qn + 1) : rn * (qn + 1) + (x - rn) * qn) + y;
}

// full-row product of the node at colour index q, (k,i,j), with u.  The
// neighbour order (dy, dx, dz ascending) and the per-block expression are
// those of the CPU restatement.  Loads are issued one dy-plane (9 blocks) at
// a time so that each thread keeps 81 coefficients and 27 vector entries in
// flight.  Missing neighbours carry zero coefficients and read the node's
// own entries instead.
template <typename A, typename KA, typename UA>
__device__ __forceinline__ void row_product_t(const Geo &g, KA kat, int k, int i, int j, UA u, A out[3]) {
    const int self = nid(g, k, i, j);
    out[0] = out[1] = out[2] = A(0);
#pragma unroll
    for (int dy = -1; dy <= 1; dy++) {
        const bool oy = (unsigned)(j + dy) < (unsigned)g.noy;
        float kv[81];
        A uv[27];
#pragma unroll
        for (int dx = -1; dx <= 1; dx++) {
            const bool ox = oy && (unsigned)(i + dx) < (unsigned)g.nox;
#pragma unroll
            for (int dz = -1; dz <= 1; dz++) {
                const int b = (dz + 1) + 3 * (dx + 1);
                const bool ok = ox && (unsigned)(k + dz) < (unsigned)g.noz;
                const int m = ok ? self + dz + g.noz * (dx + g.nox * dy) : self;
                uv[3 * b] = u(3 * m);
                uv[3 * b + 1] = u(3 * m + 1);
                uv[3 * b + 2] = u(3 * m + 2);
                const int s0 = 9 * (b + 9 * (dy + 1));
#pragma unroll
                for (int t = 0; t < 9; t++) kv[9 * b + t] = kat(s0 + t);
            }
        }
#pragma unroll
        for (int b = 0; b < 9; b++)
#pragma unroll
            for (int r = 0; r < 3; r++)
                out[r] += kv[9 * b + 3 * r] * uv[3 * b] + kv[9 * b + 3 * r + 1] * uv[3 * b + 1] +
                          kv[9 * b + 3 * r + 2] * uv[3 * b + 2];
    }
}

template <typename V>
__device__ __forceinline__ void strip3(unsigned f, V v[3]) {
    if (f & VBX) v[0] = V(0);
    if (f & VBY) v[1] = V(0);
    if (f & VBZ) v[2] = V(0);
}

// ---------------------------------------------------------------------------
// Smoother row sums.  The 8-colour smoother sums a row in a fixed order: the
// block terms t[b] = k0*u0 + k1*u1 + k2*u2 of each y-plane p = dy+1
// (b = (dz+1) + 3(dx+1); absent neighbours and b >= 9 give 0) are summed in a
// pairwise tree over 16 slots (t[q] += t[q+w], w = 1, 2, 4, 8, q a multiple
// of 2w) into P[p], and the row sum is (P[0] + P[1]) + P[2].  A thread forms
// a plane's tree in registers (PairSum16); a 16-lane row of a wavefront
// forms the same tree with DPP row shifts (IEEE addition is commutative, so
// both give the same bits).  The matvec keeps row_product_t's sequential order.

// tree over 16 slots formed term by term: push<B>(t[B]) for B = 0..15 keeps
// one partial sum per tree level; after B = 15, total is t[0] of the tree
template <typename V>
struct PairSum16 {
    V st[4];
    V total;
    template <int B>
    __device__ __forceinline__ void push(V v) {
#pragma unroll
        for (int l = 0; l < 4; l++) {
            if (B & (1 << l)) {
                v = st[l] + v;
            } else {
                st[l] = v;
                return;
            }
        }
        total = v;
    }
};

// lane i of each 16-lane row receives lane i+W's value (row_shl:W)
template <int W>
__device__ __forceinline__ double dpp_row_shl(double v) {
    const int lo = __double2loint(v), hi = __double2hiint(v);
    const int rlo = __builtin_amdgcn_update_dpp(0, lo, 0x100 + W, 0xF, 0xF, false);
    const int rhi = __builtin_amdgcn_update_dpp(0, hi, 0x100 + W, 0xF, 0xF, false);
    return __hiloint2double(rhi, rlo);
}

// PairSum16 over the 16 lanes of a DPP row; lane 16k holds the row's total
__device__ __forceinline__ double tree16_lanes(double v) {
    v = v + dpp_row_shl<1>(v);
    v = v + dpp_row_shl<2>(v);
    v = v + dpp_row_shl<4>(v);
    v = v + dpp_row_shl<8>(v);
    return v;
}

__device__ __forceinline__ double lane_value(double v, int lane) {
    const int lo = __builtin_amdgcn_readlane(__double2loint(v), lane);
    const int hi = __builtin_amdgcn_readlane(__double2hiint(v), lane);
    return __hiloint2double(hi, lo);
}

// a vector entry: a plain load, or (COHERENT) one that reads the copy in L2
// rather than the CU's L1, for values other workgroups of the same kernel
// have written (k_gs_xcd)
template <bool COHERENT, typename V>
__device__ __forceinline__ V vload(const V *__restrict__ p) {
    if constexpr (COHERENT)
        return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else
        return *p;
}

// a coefficient of a stream read once: kept out of the caches that hold the
// vectors where the level's coefficients do not fit them anyway (streamed)
template <bool STREAM, typename KT>
__device__ __forceinline__ KT kload(const KT *__restrict__ p) {
    if constexpr (STREAM)
        return __builtin_nontemporal_load(p);
    else
        return *p;
}

// Plane P = dy+1 of the three rows of node (k, i, j), coefficients kp (its
// tile column), into P[r]; arithmetic in the vector type V.
// The three parts of plane_rows: the neighbours' vector entries (and which
// neighbours exist), the plane's 81 coefficients, and the tree sums
template <int P, typename V, bool COHERENT>
__device__ __forceinline__ void plane_gather(const Geo &g, int k, int i, int j, int self, const V *__restrict__ u,
                                             V uv[27], bool okb[9]) {
    constexpr int DY = P - 1;
    const bool oy = (unsigned)(j + DY) < (unsigned)g.noy;
#pragma unroll
    for (int dx = -1; dx <= 1; dx++) {
        const bool ox = oy && (unsigned)(i + dx) < (unsigned)g.nox;
#pragma unroll
        for (int dz = -1; dz <= 1; dz++) {
            const int b = (dz + 1) + 3 * (dx + 1);
            const bool ok = ox && (unsigned)(k + dz) < (unsigned)g.noz;
            const int m = ok ? self + dz + g.noz * (dx + g.nox * DY) : self;
            okb[b] = ok;
            uv[3 * b] = vload<COHERENT>(u + 3 * m);
            uv[3 * b + 1] = vload<COHERENT>(u + 3 * m + 1);
            uv[3 * b + 2] = vload<COHERENT>(u + 3 * m + 2);
        }
    }
}

template <int P, bool STREAM, typename KT>
__device__ __forceinline__ void plane_coefs(const KT *__restrict__ kp, float kv[81]) {
#pragma unroll
    for (int c = 0; c < 81; c++) kv[c] = (float)kload<STREAM>(kp + (81 * P + c) * 64);
}

template <typename V>
__device__ __forceinline__ void plane_sums(const float kv[81], const V uv[27], const bool okb[9], V out[3]) {
    PairSum16<V> ps[3];
#define CHIP_TERM(B, R)                                                                                            \
    (okb[B] ? kv[9 * (B) + 3 * (R)] * uv[3 * (B)] + kv[9 * (B) + 3 * (R) + 1] * uv[3 * (B) + 1] +                  \
                  kv[9 * (B) + 3 * (R) + 2] * uv[3 * (B) + 2]                                                      \
            : V(0))
#define CHIP_PUSH(B)                                  \
    ps[0].template push<B>(CHIP_TERM(B, 0));          \
    ps[1].template push<B>(CHIP_TERM(B, 1));          \
    ps[2].template push<B>(CHIP_TERM(B, 2))
    CHIP_PUSH(0); CHIP_PUSH(1); CHIP_PUSH(2); CHIP_PUSH(3); CHIP_PUSH(4);
    CHIP_PUSH(5); CHIP_PUSH(6); CHIP_PUSH(7); CHIP_PUSH(8);
#undef CHIP_PUSH
#undef CHIP_TERM
#pragma unroll
    for (int r = 0; r < 3; r++) {
        ps[r].template push<9>(V(0));
        ps[r].template push<10>(V(0));
        ps[r].template push<11>(V(0));
        ps[r].template push<12>(V(0));
        ps[r].template push<13>(V(0));
        ps[r].template push<14>(V(0));
        ps[r].template push<15>(V(0));
        out[r] = ps[r].total;
    }
}

template <int P, bool STREAM, typename V, typename KT>
__device__ __forceinline__ void plane_rows(const Geo &g, const KT *__restrict__ kp, int k, int i, int j, int self,
                                           const V *__restrict__ u, V out[3]) {
    float kv[81];
    V uv[27];
    bool okb[9];
    plane_gather<P, V, false>(g, k, i, j, self, u, uv, okb);
    plane_coefs<P, STREAM, KT>(kp, kv);
    plane_sums<V>(kv, uv, okb, out);
}

// matvec of large levels: n_assemble_del2_u (Element_calculations.c:552-621)
// with strip, optionally res = rhs - Au; three wavefronts per 64-node tile: wavefront
// p loads y-plane p's 81 coefficients (coalesced 256-byte runs over the
// tile) and 27 vector entries and forms its 27 block terms (the expression
// of row_product_t); planes 1 and 2 hand their terms to wavefront 0 through
// LDS, which adds all 27 terms in row_product_t's sequential order, so the
// result has the reference's bits while three planes' loads are in
// flight at once.  Four wavefronts a SIMD: at most 128 registers (FP64 needs 129
// left alone, and ran three).
template <typename V, typename KT, bool STREAM>
__global__ void __launch_bounds__(192, 4) k_matvec3(Geo g, const KT *__restrict__ K, const unsigned *__restrict__ NODE,
                                                 const V *__restrict__ u, V *__restrict__ Au,
                                                 const V *__restrict__ rhs, V *__restrict__ res,
                                                 const V *__restrict__ BIs, V *__restrict__ ucopy) {
    __shared__ V Ts[2][27][64];   // [plane - 1][block * 3 + row][lane]
    const int lane = threadIdx.x & 63, P = threadIdx.x >> 6;
    const int q = xcd_tile(blockIdx.x, gridDim.x) * 64 + lane;
    const int col = colour_valid(g, q);
    int k = 0, i = 0, j = 0;
    if (col >= 0) colour_kij(g, col, q, k, i, j);
    const int self = nid(g, k, i, j);
    V T[27];
    if (col >= 0) {
        const KT *kp = K + ktile(q);
        const int dy = P - 1;
        const bool oy = (unsigned)(j + dy) < (unsigned)g.noy;
        float kv[81];
        V uv[27];
#pragma unroll
        for (int dx = -1; dx <= 1; dx++) {
            const bool ox = oy && (unsigned)(i + dx) < (unsigned)g.nox;
#pragma unroll
            for (int dz = -1; dz <= 1; dz++) {
                const int b = (dz + 1) + 3 * (dx + 1);
                const bool ok = ox && (unsigned)(k + dz) < (unsigned)g.noz;
                const int m = ok ? self + dz + g.noz * (dx + g.nox * dy) : self;
                uv[3 * b] = u[3 * m];
                uv[3 * b + 1] = u[3 * m + 1];
                uv[3 * b + 2] = u[3 * m + 2];
            }
        }
#pragma unroll
        for (int c = 0; c < 81; c++) kv[c] = (float)kload<STREAM>(kp + (81 * P + c) * 64);
#pragma unroll
        for (int b = 0; b < 9; b++)
#pragma unroll
            for (int r = 0; r < 3; r++)
                T[3 * b + r] = kv[9 * b + 3 * r] * uv[3 * b] + kv[9 * b + 3 * r + 1] * uv[3 * b + 1] +
                               kv[9 * b + 3 * r + 2] * uv[3 * b + 2];
        if (P > 0)
#pragma unroll
            for (int t = 0; t < 27; t++) Ts[P - 1][t][lane] = T[t];
    }
    __syncthreads();
    if (P == 1 && col >= 0 && ucopy) {   // u copied to ucopy in the same launch
        ucopy[3 * self] = u[3 * self];
        ucopy[3 * self + 1] = u[3 * self + 1];
        ucopy[3 * self + 2] = u[3 * self + 2];
    }
    if (P != 0 || col < 0) return;
    V out[3] = {V(0), V(0), V(0)};
#pragma unroll
    for (int b = 0; b < 9; b++)
#pragma unroll
        for (int r = 0; r < 3; r++) out[r] += T[3 * b + r];
#pragma unroll
    for (int pl = 0; pl < 2; pl++)
#pragma unroll
        for (int b = 0; b < 9; b++)
#pragma unroll
            for (int r = 0; r < 3; r++) out[r] += Ts[pl][3 * b + r][lane];
    const int n = self;
    if (BIs) {  // rows stored scaled by BI: K d = (BI K) d / BI
        out[0] = out[0] / BIs[3 * n];
        out[1] = out[1] / BIs[3 * n + 1];
        out[2] = out[2] / BIs[3 * n + 2];
    }
    strip3(NODE[n], out);
    Au[3 * n] = out[0];
    Au[3 * n + 1] = out[1];
    Au[3 * n + 2] = out[2];
    if (res) {
        res[3 * n] = rhs[3 * n] - out[0];
        res[3 * n + 1] = rhs[3 * n + 1] - out[1];
        res[3 * n + 2] = rhs[3 * n + 2] - out[2];
    }
}

// The same product with all three planes' coefficients and vector entries
// loaded before the first addition (one memory round trip instead of
// three; the sums keep row_product_t's order).  For small levels, whose
// matvec is latency-bound: 243 + 81 live values per thread, one wavefront
// per workgroup.
template <typename V>
__device__ __forceinline__ void row_product_all(const Geo &g, const float *__restrict__ kp, int k, int i, int j,
                                                const V *__restrict__ u, V out[3]) {
    const int self = nid(g, k, i, j);
    float kv[243];
    V uv[81];
#pragma unroll
    for (int dy = -1; dy <= 1; dy++) {
        const int P = dy + 1;
        const bool oy = (unsigned)(j + dy) < (unsigned)g.noy;
#pragma unroll
        for (int dx = -1; dx <= 1; dx++) {
            const bool ox = oy && (unsigned)(i + dx) < (unsigned)g.nox;
#pragma unroll
            for (int dz = -1; dz <= 1; dz++) {
                const int b = (dz + 1) + 3 * (dx + 1);
                const bool ok = ox && (unsigned)(k + dz) < (unsigned)g.noz;
                const int m = ok ? self + dz + g.noz * (dx + g.nox * dy) : self;
                uv[27 * P + 3 * b] = u[3 * m];
                uv[27 * P + 3 * b + 1] = u[3 * m + 1];
                uv[27 * P + 3 * b + 2] = u[3 * m + 2];
                const int s0 = 9 * (b + 9 * P);
#pragma unroll
                for (int t = 0; t < 9; t++) kv[s0 + t] = kp[(s0 + t) * 64];
            }
        }
    }
    out[0] = out[1] = out[2] = V(0);
#pragma unroll
    for (int P = 0; P < 3; P++)
#pragma unroll
        for (int b = 0; b < 9; b++)
#pragma unroll
            for (int r = 0; r < 3; r++) {
                const float *kb = kv + 81 * P + 9 * b + 3 * r;
                const V *ub = uv + 27 * P + 3 * b;
                out[r] += kb[0] * ub[0] + kb[1] * ub[1] + kb[2] * ub[2];
            }
}

// Levels whose coefficients are read past the caches: a sweep of a level of
// more than the 256 MB of the Infinity Cache finds none of them there again,
// and read plainly they put out the vectors, which the next colours read again
// (129x129x65 nodes, 1042 MB: a colour pass in FP64 35.4 us -> 33.4, the FP64
// residual 242 -> 232; 521 MB in FP16 19.1 -> 17.2; 65x65x65 nodes, 267 MB:
// 11.6 -> 11.2).  The product after a sweep still finds a part of a level not
// much larger (267 MB: 54 us, past the caches 60).  Levels that fit lose
// (65x65x33 nodes, 136 MB: 7.4 -> 8.1 us, product 28 -> 33).
constexpr double GS_STREAM = 256e6, MV_STREAM = 400e6;
template <typename KT>
static bool streamed(const Level &L, double limit) {
    return L.stream < 0 ? (double)L.g.pitch * KROW * sizeof(KT) > limit : L.stream != 0;
}

constexpr int MV_SMALL_NNO = 20000;   // levels up to this size use k_matvec_small

template <typename V>
__global__ void __launch_bounds__(64) k_matvec_small(Geo g, const float *__restrict__ K,
                                                     const unsigned *__restrict__ NODE, const V *__restrict__ u,
                                                     V *__restrict__ Au, const V *__restrict__ rhs,
                                                     V *__restrict__ res, V *__restrict__ ucopy) {
    const int q = xcd_tile(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    const int col = colour_valid(g, q);
    if (col < 0) return;
    int k, i, j;
    colour_kij(g, col, q, k, i, j);
    V out[3];
    row_product_all(g, K + ktile(q), k, i, j, u, out);
    const int n = nid(g, k, i, j);
    strip3(NODE[n], out);
    Au[3 * n] = out[0];
    Au[3 * n + 1] = out[1];
    Au[3 * n + 2] = out[2];
    if (res) {
        res[3 * n] = rhs[3 * n] - out[0];
        res[3 * n + 1] = rhs[3 * n + 1] - out[1];
        res[3 * n + 2] = rhs[3 * n + 2] - out[2];
    }
    if (ucopy) {   // u copied to ucopy in the same launch
        ucopy[3 * n] = u[3 * n];
        ucopy[3 * n + 1] = u[3 * n + 1];
        ucopy[3 * n + 2] = u[3 * n + 2];
    }
}

template <typename V>
void matvec(hipStream_t s, const Level &L, const V *u, V *Au, const V *rhs, V *res, hipEvent_t e0, hipEvent_t e1,
            V *ucopy) {
    if (!L.Kh && L.g.nno <= MV_SMALL_NNO) {
        auto kern = k_matvec_small<V>;
        const float *K = L.K;
        if (e0)
            hipExtLaunchKernelGGL(kern, dim3(nblk(L.g.pitch, 64)), dim3(64), 0, s, e0, e1, 0, L.g, K, L.NODE, u, Au,
                                  rhs, res, ucopy);
        else
            hipLaunchKernelGGL(kern, dim3(nblk(L.g.pitch, 64)), dim3(64), 0, s, L.g, K, L.NODE, u, Au, rhs, res,
                               ucopy);
        return;
    }
    const int tiles = L.g.pitch / 64;   // the colour index space is whole 64-node tiles
    auto launch = [&](auto kern, const auto *K, const V *BIs) {
        if (e0)
            hipExtLaunchKernelGGL(kern, dim3(tiles), dim3(192), 0, s, e0, e1, 0, L.g, K, L.NODE, u, Au, rhs, res, BIs, ucopy);
        else
            hipLaunchKernelGGL(kern, dim3(tiles), dim3(192), 0, s, L.g, K, L.NODE, u, Au, rhs, res, BIs, ucopy);
    };
    if constexpr (sizeof(V) == 4) {
        if (L.Kh) {
            const _Float16 *Kh = (const _Float16 *)L.Kh;
            if (streamed<_Float16>(L, MV_STREAM)) launch(k_matvec3<V, _Float16, true>, Kh, (const V *)L.BIf);
            else launch(k_matvec3<V, _Float16, false>, Kh, (const V *)L.BIf);
            return;
        }
    }
    const V *none = nullptr;
    const float *K = L.K;
    if (streamed<float>(L, MV_STREAM)) launch(k_matvec3<V, float, true>, K, none);
    else launch(k_matvec3<V, float, false>, K, none);
}
template void matvec<double>(hipStream_t, const Level &, const double *, double *, const double *, double *,
                             hipEvent_t, hipEvent_t, double *);
template void matvec<float>(hipStream_t, const Level &, const float *, float *, const float *, float *, hipEvent_t,
                            hipEvent_t, float *);

// Gauss-Seidel: gauss_seidel (General_matrix_functions.c:1160-1361) as eight
// colour passes; the node-block update t = (F - (K d)_node) * BI, rounded to
// float as the reference's temp[] is, then d += t.  One workgroup per 64-node
// tile of one colour: wavefront p forms y-plane p of the three rows of its 64
// nodes (81 coalesced coefficient loads and 27 vector gathers, all issued
// together), the partial sums meet in LDS, and wavefront r updates row r.
// Every row is formed before any unknown is written (workgroup barrier), as
// the reference updates all three unknowns of a node from the same Ad.
template <typename V, typename KT, bool STREAM>
__global__ void __launch_bounds__(192) k_gs_colour(Geo g, int c, const KT *__restrict__ K,
                                                   const V *__restrict__ BI, V *d, const V *__restrict__ F) {
    __shared__ V Ps[3][3][64];   // [plane][row][node]
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int q = g.cs[c] + xcd_tile(blockIdx.x, gridDim.x) * 64 + lane;
    const bool act = q < g.cs[c] + g.cn[c];
    int k = 0, i = 0, j = 0;
    if (act) colour_kij(g, c, q, k, i, j);
    const int self = nid(g, k, i, j);
    // row w's F, BI and d, read before the barrier: only this thread
    // writes d[3 self + w] in this pass
    V Fr = V(0), Br = V(0), dr = V(0);
    if (act) {
        Fr = F[3 * self + w];
        Br = BI[3 * self + w];
        dr = d[3 * self + w];
    }
    if (act) {
        V out[3];
        const KT *kp = K + ktile(q);
        if (w == 0)
            plane_rows<0, STREAM>(g, kp, k, i, j, self, (const V *)d, out);
        else if (w == 1)
            plane_rows<1, STREAM>(g, kp, k, i, j, self, (const V *)d, out);
        else
            plane_rows<2, STREAM>(g, kp, k, i, j, self, (const V *)d, out);
        Ps[w][0][lane] = out[0];
        Ps[w][1][lane] = out[1];
        Ps[w][2][lane] = out[2];
    }
    __syncthreads();
    if (act) {
        const int r = w;
        const V o = (Ps[0][r][lane] + Ps[1][r][lane]) + Ps[2][r][lane];
        // FP16 rows are stored scaled by BI: t = BI F - (BI K) d
        const float t = sizeof(KT) == 2 ? (float)(Fr * Br - o) : (float)((Fr - o) * Br);
        d[3 * self + r] = dr + t;
    }
}

template <typename V>
void gs_colour(hipStream_t s, const Level &L, const V *BI, int colour, V *d, const V *F, hipEvent_t e0, hipEvent_t e1) {
    const int tiles = (L.g.cn[colour] + 63) / 64;
    auto launch = [&](auto kern, const auto *K) {
        if (e0)
            hipExtLaunchKernelGGL(kern, dim3(tiles), dim3(192), 0, s, e0, e1, 0, L.g, colour, K, BI, d, F);
        else
            hipLaunchKernelGGL(kern, dim3(tiles), dim3(192), 0, s, L.g, colour, K, BI, d, F);
    };
    if constexpr (sizeof(V) == 4) {
        if (L.Kh) {
            const _Float16 *Kh = (const _Float16 *)L.Kh;
            if (streamed<_Float16>(L, GS_STREAM)) launch(k_gs_colour<V, _Float16, true>, Kh);
            else launch(k_gs_colour<V, _Float16, false>, Kh);
            return;
        }
    }
    const float *K = L.K;
    if (streamed<float>(L, GS_STREAM)) launch(k_gs_colour<V, float, true>, K);
    else launch(k_gs_colour<V, float, false>, K);
}
template void gs_colour<double>(hipStream_t, const Level &, const double *, int, double *, const double *, hipEvent_t,
                                hipEvent_t);
template void gs_colour<float>(hipStream_t, const Level &, const float *, int, float *, const float *, hipEvent_t,
                               hipEvent_t);

// ---------------------------------------------------------------------------
// Colour passes of one sweep joined into two launches, with the bits of the
// 8-colour order.  Colour = (k&1) | (i&1) << 1 | (j&1) << 2 and a node couples
// to its 26 neighbours only, so nodes two apart along any axis are
// independent: all of colours 0-3 lie on even y-planes, where a plane sees
// its two neighbours as they were before the sweep, and colours 4-7 on odd
// ones; within a plane, colours 0-1 (4-5) lie on even x-lines and 2-3 (6-7)
// on odd ones.
//
// A workgroup of k_gs_rect takes a strip of W lines of one plane, cut along k
// into segments of Wz nodes, through the plane's four colours.  The odd lines
// need the even line on either side updated, so it also updates the even line
// past its strip and, at a cut, the nodes that later colours read, from the
// sweep's input (din); it writes its own nodes only, to dout.
//
// A lane forms one row of one node.  Its 81 coefficients are requested at the
// start, packed for the launch (k_rect_pack; as nine-node pieces of the tiles'
// lines they took 81 loads and a third of the time); the sums of the planes
// dy = -1 and +1, whose entries no colour of the launch changes, are formed by
// all wavefronts at once, as are the blocks of the plane dy = 0; in its turn a
// colour only forms the blocks again whose entries have changed, one workgroup
// barrier a colour.  A node's own entries are kept in registers, so its three
// rows need no barrier between reading and writing them.
//
// Bound by latency (launch, one load, four colours of LDS reads and sums) and,
// in the wide shape, by the coefficients' bytes, the nodes computed twice among
// them.  FP64 vectors, a half sweep (four colours) against four launches of
// k_gs_colour: 4913 nodes (17x17x17) 5.6 us against 18.4, 18513 (33x33x17) 7.6
// against 18.5, 35937 (33x33x33) 9.6 against 18.9, 79233 (49x33x49) 19 against
// 20, 139425 (65x65x33) 27 against 28, 194481 (81x49x49) 42 against 29: past one
// workgroup per CU the nodes computed twice cost what the launches save, and
// the level stays with k_gs_colour.
// Shapes: narrow, a colour's 21 nodes in one wavefront, three lanes each (four
// wavefronts, one a SIMD), while there are at most two workgroups to a CU
// (18513 nodes: 7.6 us, wide 8.7; 35937 nodes, three to a CU: 14, wide 9.6);
// wide, a colour's 64 nodes in three wavefronts, one a row.

// row r of one plane's tree (absent neighbours have zero coefficients and
// zero entries; adding the tree's empty slots changes no bit but a zero's sign)
template <typename V>
__device__ __forceinline__ V plane_sum_row(const float kv[27], const V uv[27]) {
    V t[9];
#pragma unroll
    for (int b = 0; b < 9; b++) t[b] = kv[3 * b] * uv[3 * b] + kv[3 * b + 1] * uv[3 * b + 1] + kv[3 * b + 2] * uv[3 * b + 2];
    return (((t[0] + t[1]) + (t[2] + t[3])) + ((t[4] + t[5]) + (t[6] + t[7]))) + t[8];
}

// Coefficients packed for the joined passes and the box smoother: a lane's 81
// in 16-byte groups of G = 4 (FP32) or 8 (FP16), [cc / G][lane][cc % G], so
// that a wavefront reads them in 21 or 11 coalesced loads per lane.  The
// padding past cc = 80 (and the boxes' lanes without a node) hold zeros; in a
// joined pass's run the lanes with a node come first and the others read the
// last one's.
template <typename KT>
struct Pack {
    static constexpr int G = 16 / (int)sizeof(KT);
    static constexpr int NG = (81 + G - 1) / G;
    static constexpr size_t WAVE = (size_t)NG * 64 * G;   // entries of a wavefront
    uint4 q[NG];
    __device__ __forceinline__ void load(const uint4 *__restrict__ p, int lanes = 64) {
#pragma unroll
        for (int t = 0; t < NG; t++) q[t] = p[t * lanes];
    }
    template <int P>
    __device__ __forceinline__ void hold_plane() {
#pragma unroll
        for (int t = 27 * P / G; t <= (27 * P + 26) / G; t++)
            asm volatile("" : "+v"(q[t].x), "+v"(q[t].y), "+v"(q[t].z), "+v"(q[t].w));
    }
    template <int FROM, int TO>
    __device__ __forceinline__ void load_part(const uint4 *__restrict__ p) {
#pragma unroll
        for (int t = FROM; t < TO; t++) q[t] = p[t * 64];
    }
    // the values as loaded up to here: widened earlier they would not fit the registers
    __device__ __forceinline__ void hold() {
#pragma unroll
        for (int t = 0; t < NG; t++) asm volatile("" : "+v"(q[t].x), "+v"(q[t].y), "+v"(q[t].z), "+v"(q[t].w));
    }
    template <int FROM, int N>
    __device__ __forceinline__ void widen(float kv[N]) const {
        const KT *e = reinterpret_cast<const KT *>(q);
#pragma unroll
        for (int ci = 0; ci < N; ci++) kv[ci] = (float)e[FROM + ci];
    }
};

// the shape of a workgroup: nodes of a colour, W lines, HZ entries of one k
// parity in the staged region
template <bool WIDE_, int W_, int HZ_>
struct RectShape {
    static constexpr bool WIDE = WIDE_;
    static constexpr int W = W_, HZ = HZ_, NL = W + 3, NODES = WIDE ? 64 : 21, WAVES = WIDE ? 12 : 4;
    static constexpr int CH = (2 * HZ + 20) / 21;           // chunks of a staged line, 21 nodes each
    static constexpr int BATCH = (3 * NL + WAVES - 1) / WAVES * CH;
    static constexpr int LINE = 3 * 2 * HZ;                 // [component][k parity][k/2]
};

// what a wavefront of a workgroup (seg, strip, plane j) and its lane take:
// colour phase ph, row r of node (k, i) (act: if there is one), lines and
// nodes stepping two, nodes past the segment that later colours read
template <class S>
struct RectLane {
    int ph, r, k, i, lanes, slot;   // slot: the lane's place among the `lanes` with a node
    bool act;
    __device__ __forceinline__ RectLane(const Geo &g, const RectPart &rp, int seg, int strip, int w, int lane) {
        ph = S::WIDE ? w / 3 : w;
        const int i0 = strip * S::W, k0 = seg * rp.Wz, k1 = k0 + rp.Wz;
        const int kp = ph & 1, ip = ph >> 1, grow = 2 - ph;
        const int klo = max(kp, k0 - grow), khi = min(g.noz - 1, k1 + grow);
        const int ilo = i0 + ip, ihi = min(g.nox - 1, i0 + S::W - ip);
        const int nk = khi >= klo ? ((khi - klo) >> 1) + 1 : 0, ni = ihi >= ilo ? ((ihi - ilo) >> 1) + 1 : 0;
        r = S::WIDE ? w - 3 * ph : lane / 21;
        const int t = S::WIDE ? lane : lane - 21 * r;
        act = r < 3 && t < nk * ni;
        int ii = 0;   // t / nk, of at most W/2 + 1 lines
#pragma unroll
        for (int m = 1; m <= S::W / 2; m++) ii += t >= m * nk;
        k = klo + 2 * (t - ii * nk);
        i = ilo + 2 * ii;
        lanes = (S::WIDE ? 1 : 3) * nk * ni;
        slot = max(0, act ? (S::WIDE ? t : r * nk * ni + t) : lanes - 1);
    }
};

// the plane staged for plane j beside a workgroup's own: past the mesh, where
// its entries count as zero, the plane on the other side, since the own plane's
// buffer may be the one being written (dout, in the odd planes' launch)
__host__ __device__ constexpr int rect_side(int j, int noy) { return j < 0 ? 1 : j >= noy ? noy - 2 : j; }

// no launch stages a plane that it writes, beside its own
constexpr bool rect_side_clear(int most) {
    for (int noy = 2; noy <= most; noy++)
        for (int j = 0; j < noy; j++)
            for (int d = -1; d <= 1; d += 2) {
                const int s = rect_side(j + d, noy);
                if (s < 0 || s >= noy || (s - j) % 2 == 0) return false;
            }
    return true;
}
static_assert(rect_side_clear(16), "the joined passes' side planes");

// the packed coefficients of wavefront w of workgroup (seg, strip, j)
template <class S>
__device__ __forceinline__ size_t rect_wave(const RectPart &rp, int seg, int strip, int j, int w) {
    return (((size_t)j * rp.nstrip + strip) * rp.ns + seg) * S::WAVES + w;
}

template <typename KT, class S>
__global__ void __launch_bounds__(S::WAVES * 64) k_rect_pack(Geo g, RectPart rp, const KT *__restrict__ K,
                                                             KT *__restrict__ Kr) {
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int seg = blockIdx.x, strip = blockIdx.y, j = blockIdx.z;
    const RectLane<S> rl(g, rp, seg, strip, w, lane);
    const KT *kq = K + (rl.act ? ktile(colour_index(g, rl.ph | (j & 1) << 2, rl.k, rl.i, j)) + 3 * 64 * rl.r : 0);
    KT v[Pack<KT>::NG * Pack<KT>::G];
#pragma unroll
    for (int cc = 0; cc < Pack<KT>::NG * Pack<KT>::G; cc++)
        v[cc] = rl.act && cc < 81 ? kq[(81 * (cc / 27) + 9 * (cc % 27 / 3) + cc % 3) * 64] : KT(0);
    uint4 *dst = reinterpret_cast<uint4 *>(Kr) + rect_wave<S>(rp, seg, strip, j, w) * (Pack<KT>::NG * 64) + rl.slot;
    if (!rl.act) return;
#pragma unroll
    for (int t = 0; t < Pack<KT>::NG; t++) dst[t * rl.lanes] = reinterpret_cast<const uint4 *>(v)[t];
}

template <typename V, typename KT, class S>
__global__ void __launch_bounds__(S::WAVES * 64, sizeof(V) == 8 || sizeof(KT) == 2 ? 3 : 4) k_gs_rect(Geo g, RectPart rp, int jpar, const KT *__restrict__ Kr,
                                                           const V *__restrict__ BI, const V *__restrict__ F,
                                                           const V *__restrict__ dself, const V *__restrict__ dside,
                                                           V *__restrict__ dout) {
    constexpr int W = S::W, HZ = S::HZ, NL = S::NL, LINE = S::LINE;
    __shared__ __align__(16) V sd[3 * NL * LINE];   // [plane][line]
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int seg = blockIdx.x, strip = blockIdx.y, j = 2 * blockIdx.z + jpar;
    const int i0 = strip * W, k0 = seg * rp.Wz, k1 = k0 + rp.Wz;
    const RectLane<S> rl(g, rp, seg, strip, w, lane);
    const int ph = rl.ph, r = rl.r, k = rl.k, i = rl.i, kp = ph & 1;
    const bool act = rl.act;
    const int fself = act ? 3 * nid(g, k, i, j) + r : 0;
    // staged region: lines i0-1 .. i0+W+1 of three planes, nodes kr0 .. (kr0
    // even), zero outside the mesh.  A wavefront takes whole lines, 21 nodes
    // at a time (a lane keeps its component), all requested before the first
    // is stored; past its last line it repeats it.
    const int l3 = min(lane, 62) / 3, comp = min(lane, 62) - 3 * l3;
    const int kr0 = max(k0 - 4, -2);
    V stage[S::BATCH];
    const V *side = dside ? dside : F, *same = dself ? dself : F;
#pragma unroll
    for (int q = 0; q < S::BATCH; q++) {
        const int ln = min(w + q / S::CH * S::WAVES, 3 * NL - 1), pl = ln / NL;
        const int gi = min(max(i0 - 1 + ln - pl * NL, 0), g.nox - 1), gj = rect_side(j + pl - 1, g.noy);
        const int gk = min(max(kr0 + q % S::CH * 21 + l3, 0), g.noz - 1);
        stage[q] = (pl == 1 ? same : side)[3 * nid(g, gk, gi, gj) + comp];
    }
    const V Fr = F[fself], Br = BI[fself];
    Pack<KT> pk;
    pk.load(reinterpret_cast<const uint4 *>(Kr) + rect_wave<S>(rp, seg, strip, j, w) * (Pack<KT>::NG * 64) + rl.slot, rl.lanes);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < S::BATCH; q++) {
        const int ln = min(w + q / S::CH * S::WAVES, 3 * NL - 1), kq = q % S::CH * 21 + l3, pl = ln / NL;
        const bool in = (pl == 1 ? dself : dside) && (unsigned)(i0 - 1 + ln - pl * NL) < (unsigned)g.nox &&
                        (unsigned)(j + pl - 1) < (unsigned)g.noy && (unsigned)(kr0 + kq) < (unsigned)g.noz;
        if (kq < 2 * HZ) sd[ln * LINE + comp * 2 * HZ + (kq & 1) * HZ + (kq >> 1)] = in ? stage[q] : V(0);
    }
    __syncthreads();
    // this node's component 0 on its own plane (an idle lane's: any inner
    // one), and its neighbours along k, which lie in the other parity's run
    const int own = act ? (NL + i - i0 + 1) * LINE + kp * HZ + ((k - kr0) >> 1) : (NL + 1) * LINE + kp * HZ + 1;
    const V *u0 = sd + own, *um = u0 + (kp ? -HZ : HZ - 1), *up = u0 + (kp ? 1 - HZ : HZ);
    auto gather = [&](int pl, V uv[27]) {
#pragma unroll
        for (int dx = -1; dx <= 1; dx++)
#pragma unroll
            for (int e = 0; e < 3; e++) {
                const int p = (pl * NL + dx) * LINE + e * 2 * HZ;
                uv[9 * (dx + 1) + e] = um[p];
                uv[9 * (dx + 1) + 3 + e] = u0[p];
                uv[9 * (dx + 1) + 6 + e] = up[p];
            }
    };
    V uv[27];
    float kv[27];
    pk.hold();
    pk.template widen<0, 27>(kv);
    gather(-1, uv);
    const V s0 = plane_sum_row<V>(kv, uv);
    __builtin_amdgcn_sched_barrier(0);   // one plane's entries live at a time
    pk.hold();
    pk.template widen<54, 27>(kv);
    gather(1, uv);
    const V s2 = plane_sum_row<V>(kv, uv);
    __builtin_amdgcn_sched_barrier(0);
    pk.hold();
    pk.template widen<27, 27>(kv);
    // the plane's nine blocks from the entries before the launch; in its turn a
    // colour forms again those whose entries have changed: odd k the two along
    // k, odd lines the six on the lines beside
    V tb[9];
    auto block = [&](int bb) {
        const V *v = bb % 3 == 0 ? um : bb % 3 == 1 ? u0 : up;
        const int p = (bb / 3 - 1) * LINE;
        return kv[3 * bb] * v[p] + kv[3 * bb + 1] * v[p + 2 * HZ] + kv[3 * bb + 2] * v[p + 4 * HZ];
    };
#pragma unroll
    for (int bb = 0; bb < 9; bb++) tb[bb] = block(bb);
    const V dr = u0[r < 3 ? r * 2 * HZ : 0];
#pragma unroll 1
    for (int p = 0; p < 4; p++) {
        __syncthreads();
        if (ph == p) {
            if (ph & 1) {
                tb[3] = block(3);
                tb[5] = block(5);
            }
            if (ph & 2) {
#pragma unroll
                for (int dz = 0; dz < 3; dz++) {
                    tb[dz] = block(dz);
                    tb[6 + dz] = block(6 + dz);
                }
            }
            const V o = (s0 + ((((tb[0] + tb[1]) + (tb[2] + tb[3])) + ((tb[4] + tb[5]) + (tb[6] + tb[7]))) + tb[8])) + s2;
            // FP16 rows are stored scaled by BI: t = BI F - (BI K) d
            const float tt = sizeof(KT) == 2 ? (float)(Fr * Br - o) : (float)((Fr - o) * Br);
            if (act) sd[own + r * 2 * HZ] = dr + tt;
        }
    }
    __syncthreads();
    // the workgroup's own nodes, a line to a wavefront
    const int ie = strip == rp.nstrip - 1 ? g.nox : i0 + W;
    const int onk = (seg == rp.ns - 1 ? g.noz : k1) - k0, rel = (k0 - kr0) >> 1;   // k0 - kr0 is even
    for (int gi = i0 + w; gi < ie; gi += S::WAVES) {
        V *out = dout + 3L * nid(g, k0, gi, j) + comp;
        const V *row = sd + (NL + gi - i0 + 1) * LINE + comp * 2 * HZ + rel;
        for (int kq = lane < 63 ? l3 : onk; kq < onk; kq += 21) out[3 * kq] = row[(kq & 1) * HZ + (kq >> 1)];
    }
}

using RectNarrow = RectShape<false, 2, 10>;
using RectWide = RectShape<true, 4, 23>;

template <class S>
static RectPart rect_part(const Geo &g, int shape) {
    const int most = S::NODES / (S::W / 2 + 1);   // nodes of a colour along k
    for (int ns = 1; ns <= (g.noz + 1) / 2; ns++) {
        RectPart rp{};
        rp.shape = shape;
        rp.Wz = std::max(2, ((g.noz - 1 + ns - 1) / ns + 1) / 2 * 2);
        rp.ns = std::max(1, (g.noz - 1 + rp.Wz - 1) / rp.Wz);
        if (rp.ns != ns) continue;
        const int nk = ns == 1 ? (g.noz + 1) / 2 : std::min((g.noz + 1) / 2, rp.Wz / 2 + 3);
        if (nk > most || std::min(rp.Wz + 7, g.noz + 2) + 1 > 2 * S::HZ) continue;
        rp.nstrip = std::max(1, (g.nox - 1 + S::W - 1) / S::W);
        return rp;
    }
    return RectPart{};
}

// the narrow shape while there are at most two workgroups to a CU, else the
// wide one with at most one (measured above); larger levels pass colour by colour
RectPart rect_planes(const Geo &g) {
    constexpr long CUS = 256;
    for (const RectPart &rp : {rect_part<RectNarrow>(g, 1), rect_part<RectWide>(g, 2)})
        if (rp.shape && (long)(g.noy + 1) / 2 * rp.nstrip * rp.ns <= (rp.shape == 1 ? 2 : 1) * CUS) return rp;
    return RectPart{};
}

template <typename V, typename KT>
static void rect_launch(hipStream_t s, const Level &L, const KT *Kr, const V *BI, const V *F, int jpar, const V *dself,
                        const V *dside, V *dout, hipEvent_t e0, hipEvent_t e1) {
    const RectPart &rp = L.planes;
    const dim3 grid(rp.ns, rp.nstrip, (L.g.noy - jpar + 1) / 2);
    if (grid.z == 0) return;
    auto launch = [&](auto kern, int waves) {
        if (e0)
            hipExtLaunchKernelGGL(kern, grid, dim3(64 * waves), 0, s, e0, e1, 0, L.g, rp, jpar, Kr, BI, F, dself, dside, dout);
        else
            hipLaunchKernelGGL(kern, grid, dim3(64 * waves), 0, s, L.g, rp, jpar, Kr, BI, F, dself, dside, dout);
    };
    if (rp.shape == 1) launch(k_gs_rect<V, KT, RectNarrow>, RectNarrow::WAVES);
    else launch(k_gs_rect<V, KT, RectWide>, RectWide::WAVES);
}

size_t rect_pack_elems(const Level &L, bool half) {
    const RectPart &rp = L.planes;
    return (size_t)L.g.noy * rp.nstrip * rp.ns * (rp.shape == 1 ? RectNarrow::WAVES : RectWide::WAVES) *
           (half ? Pack<_Float16>::WAVE : Pack<float>::WAVE);
}

// the levels' packed coefficients, after the stiffness (and its FP16 rows)
void rect_pack(hipStream_t s, const Level &L) {
    const RectPart &rp = L.planes;
    const dim3 grid(rp.ns, rp.nstrip, L.g.noy);
    auto launch = [&](auto *K, auto *Kr) {
        using KT = std::remove_const_t<std::remove_pointer_t<decltype(Kr)>>;
        if (rp.shape == 1)
            hipLaunchKernelGGL((k_rect_pack<KT, RectNarrow>), grid, dim3(64 * RectNarrow::WAVES), 0, s, L.g, rp, K, Kr);
        else
            hipLaunchKernelGGL((k_rect_pack<KT, RectWide>), grid, dim3(64 * RectWide::WAVES), 0, s, L.g, rp, K, Kr);
    };
    if (L.Kr) launch((const float *)L.K, L.Kr);
    if (L.Krh) launch((const _Float16 *)L.Kh, (_Float16 *)L.Krh);
}

template <typename V>
void gs_rect(hipStream_t s, const Level &L, const V *BI, const V *F, int jpar, const V *dself, const V *dside, V *dout,
             hipEvent_t e0, hipEvent_t e1) {
    if constexpr (sizeof(V) == 4) {
        if (L.Kh) {
            rect_launch<V, _Float16>(s, L, (const _Float16 *)L.Krh, BI, F, jpar, dself, dside, dout, e0, e1);
            return;
        }
    }
    rect_launch<V, float>(s, L, (const float *)L.Kr, BI, F, jpar, dself, dside, dout, e0, e1);
}
template void gs_rect<double>(hipStream_t, const Level &, const double *, const double *, int, const double *,
                              const double *, double *, hipEvent_t, hipEvent_t);
template void gs_rect<float>(hipStream_t, const Level &, const float *, const float *, int, const float *, const float *,
                             float *, hipEvent_t, hipEvent_t);

// the FP16 stiffness of the mixed = 2 form: each row scaled by its BI, so
// the coefficients are O(1) (the diagonal block's diagonal is 1) whatever the
// viscosity, then rounded to FP16.  Same tiling as K.
__global__ void __launch_bounds__(TPB) k_scale_half(Geo g, const float *__restrict__ K, const double *__restrict__ BI,
                                                    _Float16 *__restrict__ Kh) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= g.pitch) return;
    const int col = colour_valid(g, q);
    const size_t base = ktile(q);
    if (col < 0) {
        for (int ci = 0; ci < KROW; ci++) Kh[base + (size_t)ci * 64] = (_Float16)0.0f;
        return;
    }
    int k, i, j;
    colour_kij(g, col, q, k, i, j);
    const int n = nid(g, k, i, j);
    const float b[3] = {(float)BI[3 * n], (float)BI[3 * n + 1], (float)BI[3 * n + 2]};
    for (int ci = 0; ci < KROW; ci++) Kh[base + (size_t)ci * 64] = (_Float16)(K[base + (size_t)ci * 64] * b[(ci / 3) % 3]);
}

void scale_half(hipStream_t s, const Level &L) {
    hipLaunchKernelGGL(k_scale_half, dim3(nblk(L.g.pitch)), dim3(TPB), 0, s, L.g, (const float *)L.K,
                       (const double *)L.BI, (_Float16 *)L.Kh);
}

// ---------------------------------------------------------------------------
// A level whose stiffness fits in LDS (the coarsest, 4x4x2 elements at the
// workloads here) runs every sweep of a gauss_seidel call, and the final
// Ad = K d, in one workgroup.  One wavefront per node: lane 16p + b forms
// block b of y-plane p for the three rows, each 16-lane row sums its plane
// with DPP shifts, lane 0 combines the planes, lanes 0..2 update.

constexpr int SMALL_TPB = 1024;

__host__ __device__ inline size_t kstage_bytes(int nno) { return (((size_t)KROW * nno * 4 + 15) / 16) * 16; }
__host__ __device__ inline size_t vstage_bytes(int nno) { return (size_t)9 * nno * 8 + (size_t)27 * nno * 4; }

__device__ __forceinline__ int compact_base(const Geo &g, int col) {
    int base = 0;
    for (int m = 0; m < col; m++) base += g.cn[m];
    return base;
}

// unit = 1: workgroup j smooths the unit right-hand side e_j into column j
// of the row-major [3 nno][3 nno] matrix d (the coarse operator), without Ad.
__global__ void __launch_bounds__(SMALL_TPB) k_gs_lds(Geo g, const float *__restrict__ K, const double *__restrict__ BI,
                                                      const unsigned *__restrict__ NODE, double *d,
                                                      const double *__restrict__ F, double *__restrict__ Ad, int sweeps,
                                                      int guess, int unit) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int nno = g.nno, tid = threadIdx.x, lane = tid & 63, w = tid >> 6, nw = blockDim.x >> 6;
    float *Ks = (float *)smem;                                   // [243][nno], compact colour order
    double *ds = (double *)(smem + kstage_bytes(nno));           // [3 nno] natural order
    double *Fs = ds + 3 * nno, *Bs = Fs + 3 * nno;
    int *nb = (int *)(Bs + 3 * nno);                             // [nno][27] neighbour node or -1
    for (int q = tid; q < g.pitch; q += blockDim.x) {
        const int col = colour_valid(g, q);
        if (col < 0) continue;
        const int cq = compact_base(g, col) + (q - g.cs[col]);
        int k, i, j;
        colour_kij(g, col, q, k, i, j);
        const int self = nid(g, k, i, j);
        const float *kp = K + ktile(q);
#pragma unroll 27
        for (int ci = 0; ci < KROW; ci++) Ks[ci * nno + cq] = kp[ci * 64];
        for (int sl = 0; sl < 27; sl++) {
            const int dz = sl % 3 - 1, dx = (sl / 3) % 3 - 1, dy = sl / 9 - 1;
            const bool ok = (unsigned)(k + dz) < (unsigned)g.noz && (unsigned)(i + dx) < (unsigned)g.nox &&
                            (unsigned)(j + dy) < (unsigned)g.noy;
            nb[cq * 27 + sl] = ok ? self + dz + g.noz * (dx + g.nox * dy) : -1;
        }
    }
    for (int idx = tid; idx < 3 * nno; idx += blockDim.x) {
        ds[idx] = guess ? d[idx] : 0.0;
        Fs[idx] = unit ? (idx == (int)blockIdx.x ? 1.0 : 0.0) : F[idx];
        Bs[idx] = BI[idx];
    }
    __syncthreads();
    const int p = lane >> 4, b = lane & 15;
    const int sl = (p < 3 && b < 9) ? 9 * p + b : -1;   // neighbour slot of this lane
    for (int cyc = 0; cyc < sweeps; cyc++) {
        int cb = 0;
        for (int c = 0; c < 8; c++) {
            const int cn = g.cn[c];
            for (int t = w; t < cn; t += nw) {   // wave-uniform
                const int cq = cb + t;
                double v0 = 0.0, v1 = 0.0, v2 = 0.0;
                if (sl >= 0) {
                    const int m = nb[cq * 27 + sl];
                    if (m >= 0) {
                        const double u0 = ds[3 * m], u1 = ds[3 * m + 1], u2 = ds[3 * m + 2];
                        const float *kc = Ks + (sl * 9) * nno + cq;
                        v0 = kc[0] * u0 + kc[nno] * u1 + kc[2 * nno] * u2;
                        v1 = kc[3 * nno] * u0 + kc[4 * nno] * u1 + kc[5 * nno] * u2;
                        v2 = kc[6 * nno] * u0 + kc[7 * nno] * u1 + kc[8 * nno] * u2;
                    }
                }
                v0 = tree16_lanes(v0);
                v1 = tree16_lanes(v1);
                v2 = tree16_lanes(v2);
                const double o0 = (lane_value(v0, 0) + lane_value(v0, 16)) + lane_value(v0, 32);
                const double o1 = (lane_value(v1, 0) + lane_value(v1, 16)) + lane_value(v1, 32);
                const double o2 = (lane_value(v2, 0) + lane_value(v2, 16)) + lane_value(v2, 32);
                if (lane < 3) {
                    const int n = nb[cq * 27 + 13];
                    const double o = lane == 0 ? o0 : (lane == 1 ? o1 : o2);
                    const float tt = (float)((Fs[3 * n + lane] - o) * Bs[3 * n + lane]);
                    ds[3 * n + lane] += tt;
                }
            }
            cb += cn;
            __syncthreads();
        }
    }
    // Ad = K d in row_product_t's sequential order, BC rows stripped
    for (int cq = tid; Ad && cq < nno; cq += blockDim.x) {
        const int n = nb[cq * 27 + 13];
        double out[3] = {0.0, 0.0, 0.0};
        for (int s2 = 0; s2 < 27; s2++) {
            const int m = nb[cq * 27 + s2];
            const int mm = m >= 0 ? m : n;   // absent neighbours have zero coefficients
            const double u0 = ds[3 * mm], u1 = ds[3 * mm + 1], u2 = ds[3 * mm + 2];
            const float *kc = Ks + (s2 * 9) * nno + cq;
#pragma unroll
            for (int r = 0; r < 3; r++)
                out[r] += kc[(3 * r) * nno] * u0 + kc[(3 * r + 1) * nno] * u1 + kc[(3 * r + 2) * nno] * u2;
        }
        strip3(NODE[n], out);
        Ad[3 * n] = out[0];
        Ad[3 * n + 1] = out[1];
        Ad[3 * n + 2] = out[2];
    }
    __syncthreads();
    if (unit)
        for (int idx = tid; idx < 3 * nno; idx += blockDim.x) d[(size_t)idx * 3 * nno + blockIdx.x] = ds[idx];
    else
        for (int idx = tid; idx < 3 * nno; idx += blockDim.x) d[idx] = ds[idx];
}

// the coarsest level's smoother call is a matrix on levels of at most this many
// dofs, and with it the calls of the levels above it of at most MAP_MAX_DOF
// (their rule beside k_map_columns)
constexpr long AFFINE_MAX_DOF = 1500, MAP_MAX_DOF = 3300;

bool affine_ok(const Level &L) { return 3L * L.g.nno <= AFFINE_MAX_DOF; }

bool map_ok(const Level &L) { return 3L * L.g.nno <= MAP_MAX_DOF; }

// largest level of the one-XCD smoother (k_gs_xcd, below): its FP32
// stiffness (972 B a node) stays within about one XCD's 4 MB L2; polls per
// barrier before a launch gives up
constexpr int XCD_MAX_NNO = 6000;
constexpr unsigned XCD_SPIN = 1u << 20;

size_t lds_limit() {
    static size_t lim = 0;
    if (!lim) {
        int dev = 0, v = 0;
        if (hipGetDevice(&dev) == hipSuccess &&
            hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) == hipSuccess && v > 0)
            lim = (size_t)v;
        else
            lim = 65536;
        if (lim > 65536) {
            (void)hipFuncSetAttribute((const void *)k_gs_lds, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lim);
        }
    }
    return lim;
}

int gs_small_kind(const Level &L) {
    const size_t nno = L.g.nno;
    return kstage_bytes(nno) + vstage_bytes(nno) <= lds_limit() ? 1 : 0;
}

void gs_small(hipStream_t s, const Level &L, double *d, const double *F, double *Ad, int sweeps, int guess) {
    const int nno = L.g.nno;
    hipLaunchKernelGGL(k_gs_lds, dim3(1), dim3(SMALL_TPB), kstage_bytes(nno) + vstage_bytes(nno), s, L.g, L.K, L.BI,
                       L.NODE, d, F, Ad, sweeps, guess, 0);
}

// ---------------------------------------------------------------------------
// A mid-size level (a few thousand nodes, a few MB of stiffness) runs a
// whole gauss_seidel call as one launch of nwg workgroups that share one XCD.
// Workgroups are dispatched to the XCDs round-robin, so blocks 8m (m = 0 ..
// nwg-1) sit on one XCD and share its L2; the grid's other blocks return at
// once.  Each colour pass is k_gs_colour's (same trees, same update
// expression; workgroup m takes the colour's tiles m, m + nwg, ...), and a
// barrier through that L2 stands in for each kernel boundary: every wave
// waits until its stores are acknowledged, then one thread per workgroup
// adds one to a 64-bit arrival counter and polls it (relaxed device-scope
// atomics).  Vector entries that other workgroups write are read with
// device-scope loads, which take the L2 copy rather than the CU's L1; the
// stiffness, F and BI are read-only and stay cached.  The counter is never
// reset: every launch adds a multiple of nwg, so a launch's first arrival
// returns base + (arrivals before it) with base a multiple of nwg.  The first
// barrier also checks that the workgroups share an XCD (the XCC_ID hardware
// register); if they do not, or a poll runs past its limit, the launch stops
// early and writes a nonzero status (2: not on one XCD, 1: poll limit) for
// the host, which reports the multigrid call as failed.  Then Ad = K d in
// row_product_t's order (and res = rhs - Ad), as after the per-colour passes.

__device__ __forceinline__ unsigned xcc_id() { return __builtin_amdgcn_s_getreg((3 << 11) | 20); }

// polls until the counter reaches target; false past the poll limit
__device__ __forceinline__ bool xcd_wait(unsigned long long *cnt, unsigned long long target) {
    for (unsigned s = 0; __hip_atomic_load(cnt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < target; s++)
        if (s >= XCD_SPIN) return false;
    return true;
}

template <typename V>
__global__ void __launch_bounds__(192) k_gs_xcd(Geo g, const float *__restrict__ K, const unsigned *__restrict__ NODE,
                                                const V *__restrict__ BI, V *d, const V *__restrict__ F,
                                                V *__restrict__ Ad, const V *__restrict__ rhs, V *__restrict__ res,
                                                int sweeps, int guess, XcdBar *bar, double *status) {
    if (blockIdx.x & 7) return;
    const int me = blockIdx.x >> 3, nwg = gridDim.x >> 3;
    __shared__ V Ps[3][3][64];   // [plane][row][node]
    __shared__ unsigned long long base_s;
    __shared__ int stop_s;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    if (!guess)
        for (int idx = me * 192 + tid; idx < 3 * g.nno; idx += nwg * 192) d[idx] = V(0);
    // first barrier: the launch's base and the one-XCD check
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (tid == 0) {
        const unsigned seen = __hip_atomic_fetch_or(&bar->mask, 1u << xcc_id(), __ATOMIC_RELAXED,
                                                    __HIP_MEMORY_SCOPE_AGENT);
        (void)seen;
        __builtin_amdgcn_s_waitcnt(0);   // the mask bit lands before the arrival
        const unsigned long long old =
            __hip_atomic_fetch_add(&bar->count, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const unsigned long long base = old - old % (unsigned long long)nwg;
        base_s = base;
        int stop = xcd_wait(&bar->count, base + nwg) ? 0 : 1;
        if (!stop) {
            const unsigned m = __hip_atomic_load(&bar->mask, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (m & (m - 1)) stop = 2;
        }
        stop_s = stop;
    }
    __syncthreads();
    if (stop_s) {
        if (tid == 0) *status = (double)stop_s;
        return;
    }
    unsigned long long target = base_s + nwg;
    for (int cyc = 0; cyc < sweeps; cyc++)
        for (int c = 0; c < 8; c++) {
            const int tiles = (g.cn[c] + 63) >> 6;
            for (int t = me; t < tiles; t += nwg) {   // uniform over the workgroup
                const int q = g.cs[c] + t * 64 + lane;
                const bool act = q < g.cs[c] + g.cn[c];
                int k = 0, i = 0, j = 0;
                if (act) colour_kij(g, c, q, k, i, j);
                const int self = nid(g, k, i, j);
                V Fr = V(0), Br = V(0), dr = V(0);
                if (act) {
                    Fr = F[3 * self + w];
                    Br = BI[3 * self + w];
                    dr = vload<true>(d + 3 * self + w);
                    const float *kp = K + ktile(q);
                    float kv[81];
                    V uv[27], out[3];
                    bool okb[9];
                    if (w == 0) {
                        plane_gather<0, V, true>(g, k, i, j, self, d, uv, okb);
                        plane_coefs<0, false, float>(kp, kv);
                    } else if (w == 1) {
                        plane_gather<1, V, true>(g, k, i, j, self, d, uv, okb);
                        plane_coefs<1, false, float>(kp, kv);
                    } else {
                        plane_gather<2, V, true>(g, k, i, j, self, d, uv, okb);
                        plane_coefs<2, false, float>(kp, kv);
                    }
                    plane_sums<V>(kv, uv, okb, out);
                    Ps[w][0][lane] = out[0];
                    Ps[w][1][lane] = out[1];
                    Ps[w][2][lane] = out[2];
                }
                __syncthreads();
                if (act) {
                    const int r = w;
                    const V o = (Ps[0][r][lane] + Ps[1][r][lane]) + Ps[2][r][lane];
                    const float tt = (float)((Fr - o) * Br);
                    d[3 * self + r] = dr + tt;
                }
                __syncthreads();
            }
            // every wave's updates are acknowledged before the arrival
            __builtin_amdgcn_s_waitcnt(0);
            __syncthreads();
            target += nwg;
            if (tid == 0) {
                __hip_atomic_fetch_add(&bar->count, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                stop_s = xcd_wait(&bar->count, target) ? 0 : 1;
            }
            __syncthreads();
            if (stop_s) {
                if (tid == 0) *status = 1.0;
                return;
            }
        }
    // every workgroup has read the mask (after the first barrier) and passed
    // the last barrier: clear it for the next launch
    if (me == 0 && tid == 0) __hip_atomic_store(&bar->mask, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (int q = me * 192 + tid; q < g.pitch; q += nwg * 192) {
        const int col = colour_valid(g, q);
        if (col < 0) continue;
        int k, i, j;
        colour_kij(g, col, q, k, i, j);
        const float *kp = K + ktile(q);
        V out[3];
        row_product_t<V>(
            g, [kp](int ci) { return kp[ci * 64]; }, k, i, j, [d](int idx) { return vload<true>(d + idx); }, out);
        const int n = nid(g, k, i, j);
        strip3(NODE[n], out);
        Ad[3 * n] = out[0];
        Ad[3 * n + 1] = out[1];
        Ad[3 * n + 2] = out[2];
        if (res) {
            res[3 * n] = rhs[3 * n] - out[0];
            res[3 * n + 1] = rhs[3 * n + 1] - out[1];
            res[3 * n + 2] = rhs[3 * n + 2] - out[2];
        }
    }
}

// workgroups of a level's k_gs_xcd launch: one per tile of its largest
// colour (at most 16, which gs_xcd_ok checks)
int xcd_groups(const Level &L) {
    int t = 1;
    for (int c = 0; c < 8; c++) t = std::max(t, (L.g.cn[c] + 63) / 64);
    return std::min(t, 16);
}

bool gs_xcd_ok(const Level &L) {
    int t = 1;
    for (int c = 0; c < 8; c++) t = std::max(t, (L.g.cn[c] + 63) / 64);
    return !L.Kh && L.xbar && L.g.nno > SMALL_NNO && L.g.nno <= XCD_MAX_NNO && t <= 16;
}

template <typename V>
void gs_xcd(hipStream_t s, const Level &L, const V *BI, V *d, const V *F, V *Ad, const V *rhs, V *res, int sweeps,
            int guess, double *status, hipEvent_t e0, hipEvent_t e1) {
    auto kern = k_gs_xcd<V>;
    const dim3 grid(8 * xcd_groups(L));
    if (e0)
        hipExtLaunchKernelGGL(kern, grid, dim3(192), 0, s, e0, e1, 0, L.g, (const float *)L.K, L.NODE, BI, d, F, Ad,
                              rhs, res, sweeps, guess, L.xbar, status);
    else
        hipLaunchKernelGGL(kern, grid, dim3(192), 0, s, L.g, (const float *)L.K, L.NODE, BI, d, F, Ad, rhs, res,
                           sweeps, guess, L.xbar, status);
}
template void gs_xcd<double>(hipStream_t, const Level &, const double *, double *, const double *, double *,
                             const double *, double *, int, int, double *, hipEvent_t, hipEvent_t);
template void gs_xcd<float>(hipStream_t, const Level &, const float *, float *, const float *, float *, const float *,
                            float *, int, int, double *, hipEvent_t, hipEvent_t);

// The XCC_ID of the active blocks of a k_gs_xcd-shaped launch (8 nwg
// blocks, every eighth one active), for the set-up check that they share
// one XCD.
__global__ void k_xcd_ids(unsigned *ids) {
    if ((blockIdx.x & 7) == 0 && threadIdx.x == 0) ids[blockIdx.x >> 3] = xcc_id();
}

int xcd_colocated(hipStream_t s, int nwg, unsigned *ids_dev, bool *same) {
    *same = false;
    if (nwg < 1 || nwg > 16) return -1;
    unsigned h[16];
    for (int rep = 0; rep < 4; rep++) {
        hipLaunchKernelGGL(k_xcd_ids, dim3(8 * nwg), dim3(64), 0, s, ids_dev);
        if (hipGetLastError() != hipSuccess) return -1;
        if (hipMemcpyAsync(h, ids_dev, nwg * sizeof(unsigned), hipMemcpyDeviceToHost, s) != hipSuccess ||
            hipStreamSynchronize(s) != hipSuccess)
            return -1;
        for (int m = 1; m < nwg; m++)
            if (h[m] != h[0]) return 0;
    }
    *same = true;
    return 0;
}

// ---------------------------------------------------------------------------
// Box smoother of the FP32 cycles.  A level's nodes are cut into boxes of at
// most BOX nodes a side; one workgroup takes one box, copies it with its
// one-node halo from din into LDS, runs the 8 colour passes of the
// node-block update on the box's own nodes in LDS (the update and row sums
// of k_gs_colour), and writes the box to dout.  Inside a box each colour
// sees the colours before it as updated; across a box face the neighbour's
// values are those of din.  One launch replaces the 8 colour launches of a
// sweep, whose cost on the small levels is launch latency, not bytes.

// segments of at most BOX nodes, as equal as they come
static bool axis_split(int n, int &nseg, unsigned short *s) {
    nseg = (n + BOX - 1) / BOX;
    if (nseg < 1 || nseg > BOX_MAXSEG) return false;
    int pos = 0;
    for (int t = 0; t < nseg; t++) {
        s[t] = (unsigned short)pos;
        pos += n / nseg + (t < n % nseg ? 1 : 0);
    }
    s[nseg] = (unsigned short)n;
    return true;
}

bool box_part(int nz, int nx, int ny, BoxPart &bp) {
    return axis_split(nz, bp.n[0], bp.s[0]) && axis_split(nx, bp.n[1], bp.s[1]) && axis_split(ny, bp.n[2], bp.s[2]);
}

// the nodes of colour c in box (bz, bx, by): first index and count per axis
struct BoxColour {
    int k0, i0, j0, nz, nx, ny;
};
__device__ __forceinline__ BoxColour box_colour(const BoxPart &bp, int bz, int bx, int by, int c) {
    BoxColour r;
    const int z0 = bp.s[0][bz], z1 = bp.s[0][bz + 1];
    const int x0 = bp.s[1][bx], x1 = bp.s[1][bx + 1];
    const int y0 = bp.s[2][by], y1 = bp.s[2][by + 1];
    r.k0 = z0 + ((z0 ^ c) & 1);
    r.i0 = x0 + ((x0 ^ (c >> 1)) & 1);
    r.j0 = y0 + ((y0 ^ (c >> 2)) & 1);
    r.nz = max(0, (z1 - r.k0 + 1) >> 1);
    r.nx = max(0, (x1 - r.i0 + 1) >> 1);
    r.ny = max(0, (y1 - r.j0 + 1) >> 1);
    return r;
}

// Box tiles: for the (box, colour) tile b 8 + c and row r, each node's 81
// coefficients of that row, plane by plane, packed.
size_t box_tile_elems(const Level &L) {
    return (size_t)L.nbox * 8 * 3 * (L.Kbox_half ? Pack<_Float16>::WAVE : Pack<float>::WAVE);
}

template <typename KT>
__global__ void __launch_bounds__(64) k_box_tiles(Geo g, BoxPart bp, const KT *__restrict__ K, KT *__restrict__ Kb) {
    using BT = Pack<KT>;
    const int tile = blockIdx.x, lane = threadIdx.x;
    const int b = tile >> 3, c = tile & 7;
    const int bz = b % bp.n[0], bx = (b / bp.n[0]) % bp.n[1], by = b / (bp.n[0] * bp.n[1]);
    const BoxColour bc = box_colour(bp, bz, bx, by, c);
    KT *dst = Kb + (size_t)tile * (3 * BT::WAVE) + lane * BT::G;
    const bool act = lane < bc.nz * bc.nx * bc.ny;
    const KT *src = K;
    if (act) {
        const int kk = lane % bc.nz, t = lane / bc.nz;
        const int k = bc.k0 + 2 * kk, i = bc.i0 + 2 * (t % bc.nx), j = bc.j0 + 2 * (t / bc.nx);
        src = K + ktile(colour_index(g, c, k, i, j));
    }
    for (int r = 0; r < 3; r++)
        for (int cc = 0; cc < BT::NG * BT::G; cc++)
            dst[r * BT::WAVE + (size_t)(cc / BT::G) * 64 * BT::G + cc % BT::G] =
                act && cc < 81 ? src[(81 * (cc / 27) + 9 * (cc % 27 / 3) + 3 * r + cc % 3) * 64] : KT(0);
}

void box_tiles(hipStream_t s, const Level &L) {
    if (!L.Kbox) return;
    const dim3 grid(8 * L.nbox);
    if (L.Kbox_half)
        hipLaunchKernelGGL(k_box_tiles<_Float16>, grid, dim3(64), 0, s, L.g, L.bp, (const _Float16 *)L.Kh,
                           (_Float16 *)L.Kbox);
    else
        hipLaunchKernelGGL(k_box_tiles<float>, grid, dim3(64), 0, s, L.g, L.bp, (const float *)L.K, (float *)L.Kbox);
}

constexpr int BOXH = BOX + 2;   // box side with its halo
static_assert(BOX <= 8, "a box holds at most 64 nodes of one colour");
constexpr int BOX_TPB = 768;

// One sweep, a workgroup per box.  ZIN: din is zero (not read).
//
// Twelve wavefronts: a row of a colour each, four colours (those of the even
// or of the odd y-planes) at a time, as k_gs_rect: no colour of the four
// changes the planes beside, so all wavefronts form these sums and the blocks
// of the own plane at once, and in its turn a colour only forms the blocks
// again whose entries have changed, one barrier a colour.  The coefficients of
// the second four are requested when the first four's have been used but for
// the own plane's (FP16: as many as 80 registers hold, two workgroups to a CU).
// A sweep, before (a y-plane of the three rows to each of three wavefronts, two
// barriers a colour) -> now: 33x33x17 nodes in FP32 16.7 us -> 13.8, 17x17x17 in
// FP16 14.0 -> 9.8; 65x65x33 in FP16 24.9 -> 24.4.  Bound by latency, eight
// colours in turn, on 75 or 27 boxes for 256 CUs; on the last, 405 boxes of
// which two share a CU, a wavefront waits for operands in 48 % of its cycles
// and for its turn to issue in 38 % (vector instructions 37 % of the time, LDS
// 29 %, of which 12 % bank conflicts).
template <typename KT, bool ZIN>
__global__ void __launch_bounds__(BOX_TPB, sizeof(KT) == 2 ? 6 : 3) k_gs_box(Geo g, BoxPart bp, const KT *__restrict__ Kb,
                                                    const float *__restrict__ BI, const float *__restrict__ F,
                                                    const float *__restrict__ din, float *__restrict__ dout) {
    using BT = Pack<KT>;
    // [component][y][x][parity of z][z / 2]: a colour's nodes 1, 20 and 260
    // words apart, all but twelve in banks of their own
    constexpr int EARLY = sizeof(KT) == 2 ? 6 : BT::NG;   // FP16: what 80 registers hold
    constexpr int HS = BOXH / 2, XS = BOXH, YS = 130, CS = BOXH * YS;
    __shared__ float sd[3 * CS];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ph = w / 3, r = w - 3 * ph, b = blockIdx.x;
    const int bz = b % bp.n[0], bx = (b / bp.n[0]) % bp.n[1], by = b / (bp.n[0] * bp.n[1]);
    const int z0 = bp.s[0][bz], x0 = bp.s[1][bx], y0 = bp.s[2][by];
    const int hz = bp.s[0][bz + 1] - z0 + 2, hx = bp.s[1][bx + 1] - x0 + 2, hy = bp.s[2][by + 1] - y0 + 2;
    auto place = [](int lz, int lx, int ly) { return ly * YS + lx * XS + (lz & 1) * HS + (lz >> 1); };
    // this wavefront's colour of either half: the lane's node (an idle lane's: the box's first)
    int own[2], fg[2];
    bool act[2];
    Pack<KT> pk;
    auto tile = [&](int h) {
        return reinterpret_cast<const uint4 *>(Kb + ((size_t)b * 8 + ph + 4 * h) * (3 * BT::WAVE) + r * BT::WAVE) + lane;
    };
    pk.load(tile(0));
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const BoxColour bc = box_colour(bp, bz, bx, by, ph + 4 * h);
        act[h] = lane < bc.nz * bc.nx * bc.ny;
        const int nz = max(bc.nz, 1), nx = max(bc.nx, 1), kk = lane % nz, t = lane / nz;
        const int k = act[h] ? bc.k0 + 2 * kk : z0, i = act[h] ? bc.i0 + 2 * (t % nx) : x0, j = act[h] ? bc.j0 + 2 * (t / nx) : y0;
        own[h] = place(k - z0 + 1, i - x0 + 1, j - y0 + 1);
        fg[h] = 3 * nid(g, k, i, j) + r;
    }
    const float Fr[2] = {F[fg[0]], F[fg[1]]}, Br[2] = {BI[fg[0]], BI[fg[1]]};
    // the box and its halo, zero outside the mesh
    constexpr int BATCH = (BOXH * BOXH * BOXH + BOX_TPB - 1) / BOX_TPB;
#pragma unroll
    for (int q = 0; q < BATCH; q++) {
        const int t = threadIdx.x + q * BOX_TPB;
        const int lz = t % hz, u = t / hz, lx = u % hx, ly = u / hx;
        const int k = z0 - 1 + lz, i = x0 - 1 + lx, j = y0 - 1 + ly;
        float v[3] = {0.0f, 0.0f, 0.0f};
        if (!ZIN && ly < hy && (unsigned)k < (unsigned)g.noz && (unsigned)i < (unsigned)g.nox && (unsigned)j < (unsigned)g.noy) {
            const int n = nid(g, k, i, j);
#pragma unroll
            for (int e = 0; e < 3; e++) v[e] = din[3 * n + e];
        }
        if (ly < hy)
#pragma unroll
            for (int e = 0; e < 3; e++) sd[e * CS + place(lz, lx, ly)] = v[e];
    }
    __syncthreads();
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const bool odd = (((ph & 1) ^ z0) & 1) == 0;   // parity of the nodes' place along z
        float *u0 = sd + own[h];
        const float *um = u0 + (odd ? -HS : HS - 1), *up = u0 + (odd ? 1 - HS : HS);
        auto block = [&](const Pack<KT> &c, int P, int bb) {
            const KT *e = reinterpret_cast<const KT *>(c.q) + 27 * P + 3 * bb;
            const float *v = (bb % 3 == 0 ? um : bb % 3 == 1 ? u0 : up) + (P - 1) * YS + (bb / 3 - 1) * XS;
            return (float)e[0] * v[0] + (float)e[1] * v[CS] + (float)e[2] * v[2 * CS];
        };
        auto tree = [](const float t[9]) { return (((t[0] + t[1]) + (t[2] + t[3])) + ((t[4] + t[5]) + (t[6] + t[7]))) + t[8]; };
        // FP16: two workgroups to a CU, for which a line's entries are live at a time
        auto narrow = [](float &v, int bb) {
            asm volatile("" : "+v"(v));
            if (sizeof(KT) == 2 && bb % 3 == 2) __builtin_amdgcn_sched_barrier(0);
        };
        auto side = [&](int P) {
            float t[9];
#pragma unroll
            for (int bb = 0; bb < 9; bb++) {
                t[bb] = block(pk, P, bb);
                narrow(t[bb], bb);
            }
            float v = tree(t);
            asm volatile("" : "+v"(v));
            __builtin_amdgcn_sched_barrier(0);   // one plane's entries live at a time
            return v;
        };
        pk.template hold_plane<0>();
        const float s0 = side(0);
        pk.template hold_plane<2>();
        const float s2 = side(2);
        const Pack<KT> mid = pk;   // of which the own plane's are still needed
        float tb[9];
#pragma unroll
        for (int bb = 0; bb < 9; bb++) {
            tb[bb] = block(mid, 1, bb);
            narrow(tb[bb], bb);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (h == 0) pk.template load_part<0, EARLY>(tile(1));
        const float dr = u0[r * CS];
#pragma unroll 1
        for (int p = 0; p < 4; p++) {
            __syncthreads();
            if (ph == p) {
                if (ph & 1) {
                    tb[3] = block(mid, 1, 3);
                    tb[5] = block(mid, 1, 5);
                }
                if (ph & 2) {
#pragma unroll
                    for (int dz = 0; dz < 3; dz++) {
                        tb[dz] = block(mid, 1, dz);
                        tb[6 + dz] = block(mid, 1, 6 + dz);
                    }
                }
                const float o = (s0 + tree(tb)) + s2;
                // FP16 rows are stored scaled by BI: t = BI F - (BI K) d
                const float t = sizeof(KT) == 2 ? Fr[h] * Br[h] - o : (Fr[h] - o) * Br[h];
                if (act[h]) u0[r * CS] = dr + t;
            }
        }
        if (h == 0) pk.template load_part<EARLY, BT::NG>(tile(1));
        __syncthreads();
    }
    // the box's own nodes
    const int nz = hz - 2, nx = hx - 2, ny = hy - 2;
    if (const int t = threadIdx.x; t < nz * nx * ny) {
        const int lz = t % nz, u = t / nz, lx = u % nx, ly = u / nx;
        const int n = nid(g, z0 + lz, x0 + lx, y0 + ly), m = place(lz + 1, lx + 1, ly + 1);
#pragma unroll
        for (int e = 0; e < 3; e++) dout[3 * n + e] = sd[e * CS + m];
    }
}

void gs_box(hipStream_t s, const Level &L, const float *BI, const float *din, float *dout, const float *F,
            hipEvent_t e0, hipEvent_t e1) {
    const dim3 grid(L.nbox), block(BOX_TPB);
    auto launch = [&](auto kern, const auto *Kb) {
        if (e0)
            hipExtLaunchKernelGGL(kern, grid, block, 0, s, e0, e1, 0, L.g, L.bp, Kb, BI, F, din, dout);
        else
            hipLaunchKernelGGL(kern, grid, block, 0, s, L.g, L.bp, Kb, BI, F, din, dout);
    };
    if (L.Kbox_half) {
        const _Float16 *Kb = (const _Float16 *)L.Kbox;
        if (din) launch(k_gs_box<_Float16, false>, Kb);
        else launch(k_gs_box<_Float16, true>, Kb);
    } else {
        const float *Kb = (const float *)L.Kbox;
        if (din) launch(k_gs_box<float, false>, Kb);
        else launch(k_gs_box<float, true>, Kb);
    }
}

// ---------------------------------------------------------------------------
// Coarsest level as a matrix.  The gauss_seidel call on the coarsest level of
// ---------------------------------------------------------------------------
// Exact solve on the FP32 cycles' coarsest level (mixed forms): the level's
// stiffness as a dense symmetric matrix, factored and inverted in FP64 by
// rocSOLVER (potrf, potri) when the operators are rebuilt, applied as FP16
// rows scaled by their largest entry (FP64 sums).
// Fixed components (the rows strip3 zeroes) get an identity row and column,
// so the matrix is SPD and the solve leaves them at the right-hand side's
// value, which the restriction has already zeroed.

// A (column-major n x n, zeroed) <- K of the level: node q's row r, block
// of neighbour m, column cc at A[(3n+r) + (3m+cc) n]
__global__ void __launch_bounds__(TPB) k_dense_assemble(Geo g, const float *__restrict__ K,
                                                        const unsigned *__restrict__ NODE, double *A) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    const int col = colour_valid(g, q);
    if (col < 0) return;
    int k, i, j;
    colour_kij(g, col, q, k, i, j);
    const long n3 = 3L * g.nno;
    const int self = nid(g, k, i, j);
    const unsigned fs = NODE[self];
    const unsigned fixbit[3] = {VBX, VBY, VBZ};
    const float *kp = K + ktile(q);
    for (int dy = -1; dy <= 1; dy++)
        for (int dx = -1; dx <= 1; dx++)
            for (int dz = -1; dz <= 1; dz++) {
                if ((unsigned)(j + dy) >= (unsigned)g.noy || (unsigned)(i + dx) >= (unsigned)g.nox ||
                    (unsigned)(k + dz) >= (unsigned)g.noz)
                    continue;
                const int m = self + dz + g.noz * (dx + g.nox * dy);
                const unsigned fm = NODE[m];
                const int b = (dz + 1) + 3 * (dx + 1), P = dy + 1;
                for (int r = 0; r < 3; r++)
                    for (int cc = 0; cc < 3; cc++) {
                        const long row = 3L * self + r, cl = 3L * m + cc;
                        double v = (double)kp[(81 * P + 9 * b + 3 * r + cc) * 64];
                        if ((fs & fixbit[r]) || (fm & fixbit[cc])) v = (row == cl) ? 1.0 : 0.0;
                        A[row + cl * n3] = v;
                    }
            }
}

// M (row-major, full) <- the inverse held in A's lower triangle, in FP32
__global__ void __launch_bounds__(TPB) k_sym_to_f32(const double *__restrict__ A, float *__restrict__ M, int n) {
    const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long)n * n) return;
    const long r = idx / n, c = idx % n;
    const long lo = r > c ? r : c, hi = r > c ? c : r;   // lower triangle: row >= column
    M[idx] = (float)A[lo + hi * (long)n];
}

// H, s <- M (row-major FP32) with each row scaled by its largest entry and
// rounded to FP16 (entries within 1, half the bytes to apply), one
// wavefront per row.  H's rows are in blocks of 256 columns, [lane][4]: lane t
// holds the columns t, t+64, t+128, t+192, which k_dense_apply adds in that
// order, as 8 bytes; the last block's places past n stay zero as allocated.
__global__ void __launch_bounds__(256) k_rowscale_f16(const float *__restrict__ M, _Float16 *__restrict__ H,
                                                      float *__restrict__ s, int n) {
    const int t = threadIdx.x & 63, i = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (i >= n) return;
    const float *row = M + (size_t)i * n;
    float m = 0.0f;
    for (int j = t; j < n; j += 64) m = fmaxf(m, fabsf(row[j]));
#pragma unroll
    for (int w = 1; w < 64; w *= 2) m = fmaxf(m, __shfl_xor(m, w, 64));
    const float sc = m > 0.0f ? m : 1.0f;
    for (int j = t; j < n; j += 64) H[(size_t)i * dense_pitch(n) + (j & ~255) + (j & 63) * 4 + (j >> 6 & 3)] = (_Float16)(row[j] / sc);
    if (t == 0) s[i] = sc;
}

// out = s M' F (M' the scaled FP16 rows), one wavefront per row, FP64 sums in a
// fixed order (lane t the terms j = t, t+64, ..., then a butterfly over the
// wavefront).  With FP32 entries a product is exact in FP64 (11 + 24 bits), so
// the fused form rounds as the sum does.  Bound by reading the
// rows: 7803 unknowns (124 MB) 41.5 us -> 34.2, with 8 bytes a load instead of 2
// (two rows to a wavefront, to share F: 44.8, half the wavefronts).
template <typename V>
__global__ void __launch_bounds__(256) k_dense_apply(const _Float16 *__restrict__ H, const float *__restrict__ s,
                                                     const V *__restrict__ F, V *__restrict__ out, int n) {
    typedef _Float16 half4 __attribute__((ext_vector_type(4)));
    const int t = threadIdx.x & 63, i = blockIdx.x * 4 + (threadIdx.x >> 6), np = dense_pitch(n);
    if (i >= n) return;
    const half4 *row = reinterpret_cast<const half4 *>(H + (size_t)i * np) + t;
    double S = 0.0;
    constexpr int UN = 6;   // 4 / 6 / 8: 33.5 / 34.2 / 32.4 us at 7803 unknowns, 6.4 / 5.8 / 7.3 at 2187
    for (int j0 = 0; j0 < np; j0 += 256 * UN) {
        half4 a[UN];
        V f[4 * UN];
#pragma unroll
        for (int q = 0; q < UN; q++) a[q] = row[min(j0 + 256 * q, np - 256) / 4];
#pragma unroll
        for (int e = 0; e < 4 * UN; e++) f[e] = F[min(j0 + 64 * e + t, n - 1)];
#pragma unroll
        for (int e = 0; e < 4 * UN; e++) {
            const double fe = j0 + 64 * e + t < n ? (double)f[e] : 0.0, h = (double)(float)a[e / 4][e % 4];
            if constexpr (sizeof(V) == 4) S = fma(h, fe, S);
            else S = S + h * fe;
        }
    }
#pragma unroll
    for (int w = 1; w < 64; w *= 2) S = S + __shfl_xor(S, w, 64);
    if (t == 0) out[i] = (V)(S * (double)s[i]);
}

void dense_assemble(hipStream_t s, const Level &L, double *A) {
    const long n3 = 3L * L.g.nno;
    (void)hipMemsetAsync(A, 0, sizeof(double) * n3 * n3, s);
    hipLaunchKernelGGL(k_dense_assemble, dim3(nblk(L.g.pitch)), dim3(TPB), 0, s, L.g, L.K, L.NODE, A);
}

void sym_to_f32(hipStream_t s, const double *A, float *M, int n) {
    hipLaunchKernelGGL(k_sym_to_f32, dim3((unsigned)(((long)n * n + TPB - 1) / TPB)), dim3(TPB), 0, s, A, M, n);
}

void rowscale_f16(hipStream_t s, const float *M, uint16_t *H, float *sc, int n) {
    hipLaunchKernelGGL(k_rowscale_f16, dim3((n + 3) / 4), dim3(256), 0, s, M, (_Float16 *)H, sc, n);
}

template <typename V>
void dense_apply(hipStream_t s, const uint16_t *H, const float *sc, const V *F, V *out, int n) {
    hipLaunchKernelGGL(k_dense_apply<V>, dim3((n + 3) / 4), dim3(256), 0, s, (const _Float16 *)H, sc, F, out, n);
}
template void dense_apply<double>(hipStream_t, const uint16_t *, const float *, const double *, double *, int);
template void dense_apply<float>(hipStream_t, const uint16_t *, const float *, const float *, float *, int);

// interp_vector + un_inject_vector (Solver_multigrid.c:173-298, 581-634):
// injection, then linear fills along x, z, y in the reference's order; at(cn, d)
// is component d of coarse node cn
template <typename V, typename At>
__device__ __forceinline__ void interp_node(const Geo &gc, const Geo &gf, const float *__restrict__ iw, int k, int i, int j,
                                            At at, V v[3]) {
    const float *wx = iw, *wz = iw + 2 * gf.nox, *wy = iw + 2 * (gf.nox + gf.noz);
    // the (up to) 8 coarse nodes around the fine node are loaded together,
    // then the linear fills along x, then z, then y: an odd fine index
    // interpolates its two coarse neighbours n1 a + n2 b, an even one takes
    // its single coarse value
    const int kc[2] = {k >> 1, (k + 1) >> 1}, ic[2] = {i >> 1, (i + 1) >> 1}, jc[2] = {j >> 1, (j + 1) >> 1};
    V c[2][2][2][3];   // [y][z][x][component]
#pragma unroll
    for (int yy = 0; yy < 2; yy++)
#pragma unroll
        for (int zz = 0; zz < 2; zz++)
#pragma unroll
            for (int xx = 0; xx < 2; xx++) {
                const int cn = nid(gc, kc[zz], ic[xx], jc[yy]);
#pragma unroll
                for (int d = 0; d < 3; d++) c[yy][zz][xx][d] = at(cn, d);
            }
    const float nx1 = wx[2 * i], nx2 = wx[2 * i + 1], nz1 = wz[2 * k], nz2 = wz[2 * k + 1];
    const float ny1 = wy[2 * j], ny2 = wy[2 * j + 1];
#pragma unroll
    for (int d = 0; d < 3; d++) {
        V lx[2][2];
#pragma unroll
        for (int yy = 0; yy < 2; yy++)
#pragma unroll
            for (int zz = 0; zz < 2; zz++)
                lx[yy][zz] = (i & 1) ? nx1 * c[yy][zz][0][d] + nx2 * c[yy][zz][1][d] : c[yy][zz][0][d];
        V pz[2];
#pragma unroll
        for (int yy = 0; yy < 2; yy++) pz[yy] = (k & 1) ? nz1 * lx[yy][0] + nz2 * lx[yy][1] : lx[yy][0];
        v[d] = (j & 1) ? ny1 * pz[0] + ny2 * pz[1] : pz[0];
    }
}

constexpr int MAP_PAD = 2;

// ---------------------------------------------------------------------------
// Smoother calls of multi_grid as matrices.  On the coarsest level a call
// (v_steps_low sweeps from a zero guess, General_matrix_functions.c:574, :613)
// is linear in its right-hand side apart from the FP32 rounding of each
// increment, and its Ad is not read afterwards: d = Mc F.  On the levels above
// it (down_heavy = up_heavy sweeps) a call is likewise d = Ma d_in + Mb F, or
// Mb F from a zero guess; and on the level right above the coarsest the way up
// (restriction, coarsest call, prolongation, call with that guess) is one
// matrix of the residual, Mu = Ma (P Mc R) + Mb.  The columns are the smoother's
// results for unit vectors, formed when the stiffness is rebuilt.  The FP32
// cycles read Ma and Mb rounded to FP32, with FP64 sums: on 441 to 1089 nodes
// 2.9e-8 to 4.5e-8 from the call in FP64, where FP32 sweeps are 4.6e-8 to
// 7.4e-8; Mc and Mu, whose sums hold Mc's, stay FP64.
//
// A sweep of such a level is bound by latency (two launches of 8 us whatever
// its size), a map by reading 8 n^2 bytes; the FP64 cycle, three sweeps: 405
// nodes 46 us -> 5.8, 729 nodes 47 us -> 11 to 12.  The line: a Stokes solve on
// 20x20x16 elements (level of 1089 nodes) 41.7 ms with sweeps, 34.7 with maps;
// on 20x20x20 (1331 nodes) 40.7 and 39.0, and with a rebuild a step 68.3 and
// 69.2.  The columns are formed NC at a time by a workgroup that keeps them in
// LDS; lanes are columns by nodes, so a stiffness entry is fetched once for NC
// columns (one column a workgroup -> NC: 462 nodes, 20 sweeps 1.27 ms -> 1.02;
// 405 nodes, two maps of three sweeps 0.29 -> 0.30; 729 nodes, three maps 0.9).

// share of fine node (2k-1 + t%3, ...) in coarse node (k, i, j) by project_vector
__device__ double project_share(const Geo &gc, const float *__restrict__ TWW, const float *__restrict__ MASS, int k,
                                int i, int j, int t) {
    const int tz = t % 3, tx = t / 3 % 3, ty = t / 9;
    double w = 0.0;
    for (int m = 0; m < 8; m++) {
        const int oz = m & 1, ox = (m >> 1) & 1, oy = m >> 2;
        const int ez = k - 1 + oz, ex = i - 1 + ox, ey = j - 1 + oy;
        if ((unsigned)ez >= (unsigned)gc.elz || (unsigned)ex >= (unsigned)gc.elx || (unsigned)ey >= (unsigned)gc.ely) continue;
        if ((unsigned)(tz - oz) > 1u || (unsigned)(tx - ox) > 1u || (unsigned)(ty - oy) > 1u) continue;
        w += TWW[(size_t)(ez + gc.elz * (ex + gc.elx * ey)) * TWW_SZ + cLoc[(k - ez) + 2 * (i - ex) + 4 * (j - ey)]];
    }
    return w * MASS[nid(gc, k, i, j)];
}

// X = Mc R, R the restriction with multi_grid's strip: column j (a fine dof)
// has the up to eight coarse nodes around it.  X [3 coarse nno][3 fine nno].
__global__ void __launch_bounds__(256) k_map_restrict(Geo gf, Geo gc, const float *__restrict__ TWW,
                                                      const float *__restrict__ MASS, const unsigned *__restrict__ NODE,
                                                      const double *__restrict__ Mc, double *__restrict__ X) {
    const int j = blockIdx.x * 256 + threadIdx.x, n3f = 3 * gf.nno, n3c = 3 * gc.nno;
    if (j >= n3f) return;
    const int d = j % 3;
    int kf, xf, yf;
    node_kij(gf, j / 3, kf, xf, yf);
    const unsigned fixed = d == 0 ? VBX : d == 1 ? VBY : VBZ;
    double wt[8];
    int col[8];
#pragma unroll
    for (int m = 0; m < 8; m++) {
        const int k = (kf + (m & 1)) >> 1, i = (xf + ((m >> 1) & 1)) >> 1, y = (yf + (m >> 2)) >> 1;
        // an even index has one coarse node, counted once
        const bool twice = ((m & 1) && !(kf & 1)) || ((m & 2) && !(xf & 1)) || ((m & 4) && !(yf & 1));
        const int n = nid(gc, k, i, y);
        const int t = (kf - 2 * k + 1) + 3 * (xf - 2 * i + 1) + 9 * (yf - 2 * y + 1);
        col[m] = 3 * n + d;
        wt[m] = twice || (NODE[n] & fixed) ? 0.0 : project_share(gc, TWW, MASS, k, i, y, t);
    }
    for (int r = blockIdx.y; r < n3c; r += gridDim.y) {
        double v = 0.0;
#pragma unroll
        for (int m = 0; m < 8; m++) v += Mc[(size_t)r * n3c + col[m]] * wt[m];
        X[(size_t)r * n3f + j] = v;
    }
}

// Map blockIdx.y + kind0 (0: Ma, 1: Mb, 2: Mu, whose first rows hold X on
// entry), columns blockIdx.x NC ..: a level of one colour pass after the
// other, each thread the three rows of a (node, column), in the order of
// k_gs_colour.  The kinds below `rounded` take the increments rounded to FP32,
// as the reference's sweeps do (Mc, and Ma and Mb of at most AFFINE_MAX_DOF
// unknowns); the others are the call in FP64, since a map of columns with
// rounded increments may be further from it than the sweeps are (729 nodes,
// three sweeps from a random guess: 3.0e-8, the sweeps 2.0e-8).
template <int NC>
__global__ void __launch_bounds__(1024) k_map_columns(Geo g, Geo gc, const float *__restrict__ K,
                                                      const double *__restrict__ BI, const float *__restrict__ iw,
                                                      const unsigned *__restrict__ NODE, int sweeps, int kind0, int rounded,
                                                      MapSet ms) {
    extern __shared__ __align__(16) unsigned char smem[];
    double *ds = (double *)smem;   // [nno][3][NC], a node's run MAP_PAD longer against bank conflicts
    constexpr int ST = 3 * NC + MAP_PAD;
    const int n3 = 3 * g.nno, kind = blockIdx.y + kind0, j0 = blockIdx.x * NC;
    double *M = ms.m[kind];
    for (int idx = threadIdx.x; idx < g.nno * NC; idx += 1024) {
        const int n = idx / NC, col = idx % NC, jc = j0 + col;
        double v[3] = {0.0, 0.0, 0.0};
        if (kind == 0) {
            if (jc / 3 == n) v[jc % 3] = 1.0;
        } else if (kind == 2 && jc < n3) {
            int k, i, j;
            node_kij(g, n, k, i, j);
            interp_node<double>(gc, g, iw, k, i, j, [&](int cn, int d) { return M[(size_t)(3 * cn + d) * n3 + jc]; }, v);
            strip3(NODE[n], v);
        }
#pragma unroll
        for (int e = 0; e < 3; e++) ds[n * ST + e * NC + col] = v[e];
    }
    __syncthreads();
    for (int cyc = 0; cyc < sweeps; cyc++)
        for (int c = 0; c < 8; c++) {
            for (int idx = threadIdx.x; idx < g.cn[c] * NC; idx += 1024) {
                const int q = g.cs[c] + idx / NC, col = idx % NC;
                int k, i, j;
                colour_kij(g, c, q, k, i, j);
                const int self = nid(g, k, i, j);
                const float *kp = K + ktile(q);
                double o[3] = {0.0, 0.0, 0.0};
#pragma unroll 1
                for (int P = 0; P < 3; P++) {
                    double uv[27];
#pragma unroll
                    for (int b = 0; b < 9; b++) {
                        const int dz = b % 3 - 1, dx = b / 3 - 1, dy = P - 1;
                        const bool ok = (unsigned)(k + dz) < (unsigned)g.noz && (unsigned)(i + dx) < (unsigned)g.nox &&
                                        (unsigned)(j + dy) < (unsigned)g.noy;   // else a zero block of the row
                        const double *u = ds + (ok ? nid(g, k + dz, i + dx, j + dy) : self) * ST + col;
#pragma unroll
                        for (int e = 0; e < 3; e++) uv[3 * b + e] = u[e * NC];
                    }
#pragma unroll
                    for (int r = 0; r < 3; r++) {
                        float kv[27];
#pragma unroll
                        for (int b = 0; b < 9; b++)
#pragma unroll
                            for (int e = 0; e < 3; e++) kv[3 * b + e] = kp[(81 * P + 9 * b + 3 * r + e) * 64];
                        o[r] += plane_sum_row<double>(kv, uv);
                        __builtin_amdgcn_sched_barrier(0);   // one row's entries live at a time
                    }
                }
                double *u = ds + self * ST + col;
#pragma unroll
                for (int r = 0; r < 3; r++) {
                    const double F = kind != 0 && 3 * self + r == j0 + col ? 1.0 : 0.0;
                    const double t = (F - o[r]) * BI[3 * self + r];
                    u[r * NC] += kind < rounded ? (double)(float)t : t;
                }
            }
            __syncthreads();
        }
    float *Mf = ms.f[kind];
    for (int idx = threadIdx.x; idx < n3 * NC; idx += 1024) {
        const int row = idx / NC, col = idx % NC;
        if (j0 + col >= n3) continue;
        const double v = ds[row / 3 * ST + row % 3 * NC + col];
        M[(size_t)row * n3 + j0 + col] = v;
        if (Mf) Mf[(size_t)row * n3 + j0 + col] = (float)v;   // the FP32 cycles read half the bytes
    }
}

// as many columns a workgroup as its LDS takes
static int map_columns(hipStream_t s, const Level &L, const Geo &gc, int sweeps, int kind0, int kinds, int rounded,
                       const MapSet &ms) {
    const int n3 = 3 * L.g.nno;
    auto launch = [&](auto kern, int nc) {
        const size_t lds = (size_t)L.g.nno * (3 * nc + MAP_PAD) * 8;
        if (lds > lds_limit()) return false;
        if (lds > 65536 && hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
            return false;
        hipLaunchKernelGGL(kern, dim3((n3 + nc - 1) / nc, kinds), dim3(1024), lds, s, L.g, gc, L.K, L.BI, L.iw, L.NODE,
                           sweeps, kind0, rounded, ms);
        return true;
    };
    if (launch(k_map_columns<8>, 8) || launch(k_map_columns<4>, 4) || launch(k_map_columns<1>, 1)) return 0;
    set_error("the smoother's maps do not fit the workgroup memory");
    return -1;
}

int coarse_build(hipStream_t s, const Level &L, int sweeps) {
    const int nno = L.g.nno;
    if (gs_small_kind(L)) {
        hipLaunchKernelGGL(k_gs_lds, dim3(3 * nno), dim3(SMALL_TPB), kstage_bytes(nno) + vstage_bytes(nno), s, L.g,
                           L.K, L.BI, L.NODE, L.Mc, nullptr, nullptr, sweeps, 0, 1);
        return 0;
    }
    return map_columns(s, L, L.g, sweeps, 1, 1, 2, MapSet{{nullptr, L.Mc, nullptr}, {}});
}

int affine_build(hipStream_t s, const Level &L, const Level &coarse) {
    const MapSet ms{{L.Ma, L.Mb, L.Mu}, {L.Maf, L.Mbf, nullptr}};
    if (L.Mu)
        hipLaunchKernelGGL(k_map_restrict, dim3(nblk(3L * L.g.nno), std::min(3 * coarse.g.nno, 64)), dim3(256), 0, s, L.g,
                           coarse.g, coarse.TWW, coarse.MASS, coarse.NODE, coarse.Mc, L.Mu);
    return map_columns(s, L, coarse.g, L.affine_sweeps, 0, L.Mu ? 3 : 2, affine_ok(L) ? 2 : 0, ms);
}

// out = A din + B F (A may be null): LANES lanes a row; lane t sums A's terms
// j = t, t + LANES, ... in order, then B's likewise, into S[t]; the S[t] meet in
// a pairwise tree (S[q] += S[q+w], w = 1, 2, ...) formed by a butterfly.  Bound
// by the latency of its loads: up to NB terms of a lane are requested together
// (past the row's end the last one again, counted as 0), a whole row where it
// fits (729 nodes, rows of 2187: 15.8 us -> 11.0 a call; eight terms at a time
// and the rest one by one before).
template <typename V, typename M, int LANES, int NB>
__global__ void __launch_bounds__(64) k_map_apply(const M *A, const M *B, const V *__restrict__ din,
                                                  const V *__restrict__ F, V *__restrict__ out, int n3) {
    const int t = threadIdx.x % LANES, i = blockIdx.x * (64 / LANES) + threadIdx.x / LANES;
    double S = 0.0;
    if (i < n3) {
#pragma unroll 1
        for (int h = A ? 0 : 1; h < 2; h++) {
            const M *row = (h ? B : A) + (size_t)i * n3;
            const V *x = h ? F : din;
#pragma unroll 1
            for (int b = t; b < n3; b += NB * LANES) {
                M m[NB];
                V v[NB];
#pragma unroll
                for (int q = 0; q < NB; q++) {
                    const int j = min(b + q * LANES, n3 - 1);
                    m[q] = row[j];
                    v[q] = x[j];
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int q = 0; q < NB; q++) S = S + (b + q * LANES < n3 ? (double)m[q] * (double)v[q] : 0.0);
            }
        }
    }
#pragma unroll
    for (int w = 1; w < LANES; w *= 2) S = S + __shfl_xor(S, w, 64);
    if (i < n3 && t == 0) out[i] = (V)S;
}

template <typename V, typename M>
static void map_apply(hipStream_t s, const M *A, const M *B, const V *din, const V *F, V *out, int n3) {
    const int terms = (n3 + 63) / 64;
    auto kern = terms <= 8 ? k_map_apply<V, M, 64, 8> : terms <= 20 ? k_map_apply<V, M, 64, 20> : k_map_apply<V, M, 64, 36>;
    hipLaunchKernelGGL(kern, dim3(n3), dim3(64), 0, s, A, B, din, F, out, n3);
}

template <typename V>
void affine_apply(hipStream_t s, const Level &L, const V *din, const V *F, V *out) {
    const int n3 = 3 * L.g.nno;
    if (sizeof(V) == 4 && L.Maf)
        map_apply<V, float>(s, din ? L.Maf : nullptr, L.Mbf, din, F, out, n3);
    else
        map_apply<V, double>(s, din ? L.Ma : nullptr, L.Mb, din, F, out, n3);
}
template void affine_apply<double>(hipStream_t, const Level &, const double *, const double *, double *);
template void affine_apply<float>(hipStream_t, const Level &, const float *, const float *, float *);

// the way up to the level above the coarsest: out = Mu res.  FP64 in the FP32
// cycles too: its sums hold the coarsest level's call, whose matrix is FP64.
template <typename V>
void up_apply(hipStream_t s, const Level &L, const V *res, V *out) {
    map_apply<V, double>(s, nullptr, L.Mu, nullptr, res, out, 3 * L.g.nno);
}
template void up_apply<double>(hipStream_t, const Level &, const double *, double *);
template void up_apply<float>(hipStream_t, const Level &, const float *, float *);

// d = Mc F, sixteen lanes a row
template <typename V>
void coarse_apply(hipStream_t s, const Level &L, const V *F, V *d) {
    const int n3 = 3 * L.g.nno;
    hipLaunchKernelGGL((k_map_apply<V, double, 16, 24>), dim3((n3 + 3) / 4), dim3(64), 0, s, nullptr, L.Mc, nullptr, F, d, n3);
}
template void coarse_apply<double>(hipStream_t, const Level &, const double *, double *);
template void coarse_apply<float>(hipStream_t, const Level &, const float *, float *);

// ---------------------------------------------------------------------------
// grid transfers

// project_vector (Solver_multigrid.c:72-159), optionally followed by the
// strip_bcs_from_residual that multi_grid applies to its result
template <typename V>
__global__ void __launch_bounds__(TPB) k_project(Geo gf, Geo gc, const float *__restrict__ TWW,
                                                 const float *__restrict__ MASS, const unsigned *__restrict__ NODE,
                                                 const V *__restrict__ AU, V *__restrict__ AD, int do_strip,
                                                 V *__restrict__ zero) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= gc.nno) return;
    int k, i, j;
    node_kij(gc, n, k, i, j);
    // every load first: the 27 fine nodes 2k-1..2k+1 (x, y likewise) that the
    // coarse node's elements reach, and the element weights; then the sums
    // in the reference's order (elements ascending, their 8 fine nodes in
    // local order)
    V fv[27][3];
#pragma unroll
    for (int t = 0; t < 27; t++) {
        const int fz = 2 * k - 1 + t % 3, fx = 2 * i - 1 + (t / 3) % 3, fy = 2 * j - 1 + t / 9;
        const bool in = (unsigned)fz < (unsigned)gf.noz && (unsigned)fx < (unsigned)gf.nox &&
                        (unsigned)fy < (unsigned)gf.noy;
        const int fn = in ? nid(gf, fz, fx, fy) : nid(gf, 2 * k, 2 * i, 2 * j);
        fv[t][0] = AU[3 * fn];
        fv[t][1] = AU[3 * fn + 1];
        fv[t][2] = AU[3 * fn + 2];
    }
    float w[8];
    bool ok[8];
#pragma unroll
    for (int m = 0; m < 8; m++) {
        const int ez = k - 1 + (m & 1), ex = i - 1 + ((m >> 1) & 1), ey = j - 1 + (m >> 2);
        ok[m] = (unsigned)ez < (unsigned)gc.elz && (unsigned)ex < (unsigned)gc.elx && (unsigned)ey < (unsigned)gc.ely;
        const int a = cLoc[(k - ez) + 2 * (i - ex) + 4 * (j - ey)];
        w[m] = ok[m] ? TWW[(size_t)(ez + gc.elz * (ex + gc.elx * ey)) * TWW_SZ + a] : 0.0f;
    }
    // offsets of local node b (the cOff tables, as compile-time constants)
    constexpr int OZ[9] = {0, 0, 0, 0, 0, 1, 1, 1, 1};
    constexpr int OX[9] = {0, 0, 1, 1, 0, 0, 1, 1, 0};
    constexpr int OY[9] = {0, 0, 0, 1, 1, 0, 0, 1, 1};
    V acc[3] = {V(0), V(0), V(0)};
#pragma unroll
    for (int m = 0; m < 8; m++) {
        if (!ok[m]) continue;
        // element m = (k-1+mz, i-1+mx, j-1+my) holds the coarse node at local
        // offset (1-mz, 1-mx, 1-my); its fine node b is 2 e + that offset +
        // off(b), i.e. (mz + OZ[b], ...) from 2k - 1
        const int oz = m & 1, ox = (m >> 1) & 1, oy = m >> 2;
        V av0 = V(0), av1 = V(0), av2 = V(0);
#pragma unroll
        for (int b = 1; b <= 8; b++) {
            const int t = (oz + OZ[b]) + 3 * (ox + OX[b]) + 9 * (oy + OY[b]);
            av0 += fv[t][0];
            av1 += fv[t][1];
            av2 += fv[t][2];
        }
        acc[0] += w[m] * av0;
        acc[1] += w[m] * av1;
        acc[2] += w[m] * av2;
    }
    const float m = MASS[n];
    acc[0] = acc[0] * m;
    acc[1] = acc[1] * m;
    acc[2] = acc[2] * m;
    if (do_strip) strip3(NODE[n], acc);
    AD[3 * n] = acc[0];
    AD[3 * n + 1] = acc[1];
    AD[3 * n + 2] = acc[2];
    if (zero) {   // the coarse level's smoother starts from zero
        zero[3 * n] = V(0);
        zero[3 * n + 1] = V(0);
        zero[3 * n + 2] = V(0);
    }
}

template <typename V>
void project(hipStream_t s, const Level &fine, const Level &coarse, const V *AU, V *AD, bool do_strip, V *zero) {
    hipLaunchKernelGGL(k_project<V>, dim3(nblk(coarse.g.nno)), dim3(TPB), 0, s, fine.g, coarse.g, coarse.TWW,
                       coarse.MASS, coarse.NODE, AU, AD, (int)do_strip, zero);
}
template void project<double>(hipStream_t, const Level &, const Level &, const double *, double *, bool, double *);
template void project<float>(hipStream_t, const Level &, const Level &, const float *, float *, bool, float *);

// optionally followed by multi_grid's strip_bcs_from_residual
template <typename V>
__global__ void __launch_bounds__(TPB) k_interp(Geo gc, Geo gf, const float *__restrict__ iw,
                                                const unsigned *__restrict__ NODE, const V *__restrict__ AD,
                                                V *__restrict__ AU, int do_strip) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= gf.nno) return;
    int k, i, j;
    node_kij(gf, n, k, i, j);
    V v[3];
    interp_node<V>(gc, gf, iw, k, i, j, [&](int cn, int d) { return AD[3 * cn + d]; }, v);
    if (do_strip) strip3(NODE[n], v);
    AU[3 * n] = v[0];
    AU[3 * n + 1] = v[1];
    AU[3 * n + 2] = v[2];
}

template <typename V>
void interp(hipStream_t s, const Level &coarse, const Level &fine, const V *AD, V *AU, bool do_strip) {
    hipLaunchKernelGGL(k_interp<V>, dim3(nblk(fine.g.nno)), dim3(TPB), 0, s, coarse.g, fine.g, fine.iw, fine.NODE, AD,
                       AU, (int)do_strip);
}
template void interp<double>(hipStream_t, const Level &, const Level &, const double *, double *, bool);
template void interp<float>(hipStream_t, const Level &, const Level &, const float *, float *, bool);

// ---------------------------------------------------------------------------
// divergence and gradient (Element_calculations.c:691-769)

__global__ void __launch_bounds__(TPB) k_div(Geo g, const float *__restrict__ EG, const double *__restrict__ U,
                                             double *__restrict__ divU) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= g.nel) return;
    const int ez = e % g.elz, ex = (e / g.elz) % g.elx, ey = e / (g.elz * g.elx);
    const float *eg = EG + (size_t)e * EG_SZ;
    double acc = 0.0;
#pragma unroll
    for (int a = 1; a <= 8; a++) {
        const int n = nid(g, ez + cOffz[a], ex + cOffx[a], ey + cOffy[a]);
        const int p = 3 * (a - 1);
        acc += eg[p] * U[3 * n] + eg[p + 1] * U[3 * n + 1] + eg[p + 2] * U[3 * n + 2];
    }
    divU[e] = acc;
}

void div(hipStream_t s, const Level &L, const double *U, double *divU) {
    hipLaunchKernelGGL(k_div, dim3(nblk(L.g.nel)), dim3(TPB), 0, s, L.g, L.EG, U, divU);
}

__global__ void __launch_bounds__(TPB) k_grad(Geo g, const float *__restrict__ EG, const unsigned *__restrict__ NODE,
                                              const double *__restrict__ P, double *__restrict__ gradP) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= g.nno) return;
    int k, i, j;
    node_kij(g, n, k, i, j);
    // all eight elements' P and g entries are loaded first (absent elements
    // read element 0 and are masked), then summed in ascending element order
    double pe[8];
    float eg[8][3];
    bool ok[8];
#pragma unroll
    for (int m = 0; m < 8; m++) {
        const int ez = k - 1 + (m & 1), ex = i - 1 + ((m >> 1) & 1), ey = j - 1 + (m >> 2);
        ok[m] = (unsigned)ez < (unsigned)g.elz && (unsigned)ex < (unsigned)g.elx && (unsigned)ey < (unsigned)g.ely;
        const int e = ok[m] ? ez + g.elz * (ex + g.elx * ey) : 0;
        const int a = cLoc[(k - ez) + 2 * (i - ex) + 4 * (j - ey)];
        const float *ge = EG + (size_t)e * EG_SZ + 3 * ((ok[m] ? a : 1) - 1);
        pe[m] = P[e];
        eg[m][0] = ge[0];
        eg[m][1] = ge[1];
        eg[m][2] = ge[2];
    }
    double acc[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int m = 0; m < 8; m++) {
        if (!ok[m] || 0.0 == pe[m]) continue;   // assemble_grad_p skips P[e] == 0 (:746)
        acc[0] += eg[m][0] * pe[m];
        acc[1] += eg[m][1] * pe[m];
        acc[2] += eg[m][2] * pe[m];
    }
    strip3(NODE[n], acc);
    gradP[3 * n] = acc[0];
    gradP[3 * n + 1] = acc[1];
    gradP[3 * n + 2] = acc[2];
}

void grad(hipStream_t s, const Level &L, const double *P, double *gradP) {
    hipLaunchKernelGGL(k_grad, dim3(nblk(L.g.nno)), dim3(TPB), 0, s, L.g, L.EG, L.NODE, P, gradP);
}

__global__ void k_strip(Geo g, const unsigned *__restrict__ NODE, double *v) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= g.nno) return;
    const unsigned f = NODE[n];
    if (f & VBX) v[3 * n] = 0.0;
    if (f & VBY) v[3 * n + 1] = 0.0;
    if (f & VBZ) v[3 * n + 2] = 0.0;
}

void strip(hipStream_t s, const Level &L, double *v) {
    hipLaunchKernelGGL(k_strip, dim3(nblk(L.g.nno)), dim3(TPB), 0, s, L.g, L.NODE, v);
}

// ---------------------------------------------------------------------------
// reductions: one launch, per-block partial sums, the last block to finish
// sums the partials in block order (deterministic for a given size)

constexpr int DOT_TPB = 256;
// at most 256 workgroups: the last-workgroup handoff is one atomic per
// workgroup on a single counter
constexpr int DOT_MAXB = 256;

template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    return v;
}

template <int ND>
__device__ void block_sum(double v[ND], double *sh /* [ND][DOT_TPB/64] */) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
#pragma unroll
    for (int m = 0; m < ND; m++) v[m] = wave_sum(v[m]);
    if (lane == 0)
#pragma unroll
        for (int m = 0; m < ND; m++) sh[m * 16 + w] = v[m];
    __syncthreads();
    if (threadIdx.x == 0)
#pragma unroll
        for (int m = 0; m < ND; m++) {
            double t = 0.0;
            for (int q = 0; q < nw; q++) t += sh[m * 16 + q];
            v[m] = t;
        }
}

template <int ND, typename V>
__global__ void __launch_bounds__(DOT_TPB) k_dots(int n, const V *__restrict__ a0, const V *__restrict__ b0,
                                                  const V *__restrict__ a1, const V *__restrict__ b1,
                                                  const V *__restrict__ a2, const V *__restrict__ b2,
                                                  const V *__restrict__ a3, const V *__restrict__ b3,
                                                  double *partial, unsigned *counter, double *out) {
    __shared__ double sh[4 * 16];
    __shared__ bool last;
    // four independent partial sums per thread (u = 0..3 over consecutive
    // grid strides), combined as (s0 + s1) + (s2 + s3)
    double v[ND], w[ND][4];
#pragma unroll
    for (int m = 0; m < ND; m++)
#pragma unroll
        for (int u = 0; u < 4; u++) w[m][u] = 0.0;
    const int stride = gridDim.x * blockDim.x;
    long i1 = blockIdx.x * blockDim.x + threadIdx.x;
    // BATCH grid strides at a time with all their loads in flight, the sums in
    // the same order (one pair of 3.2 M entries in FP64 21.6 us -> 14.3)
    constexpr int BATCH = ND == 1 ? 16 : 8;
    const V *const pa[4] = {a0, a1, a2, a3}, *const pb[4] = {b0, b1, b2, b3};
    for (; i1 + (long)(BATCH - 1) * stride < n; i1 += (long)BATCH * stride) {
        V x[ND][BATCH], y[ND][BATCH];
#pragma unroll
        for (int q = 0; q < BATCH; q++)
#pragma unroll
            for (int m = 0; m < ND; m++) {
                x[m][q] = pa[m][i1 + (long)q * stride];
                y[m][q] = pb[m][i1 + (long)q * stride];
            }
#pragma unroll
        for (int q = 0; q < BATCH; q++)
#pragma unroll
            for (int m = 0; m < ND; m++) w[m][q & 3] += (double)x[m][q] * (double)y[m][q];
    }
    for (int i0 = (int)i1; i0 < n; i0 += 4 * stride) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int i = i0 + u * stride;
            if (i < n) {
                w[0][u] += (double)a0[i] * (double)b0[i];
                if (ND > 1) w[1][u] += (double)a1[i] * (double)b1[i];
                if (ND > 2) w[2][u] += (double)a2[i] * (double)b2[i];
                if (ND > 3) w[3][u] += (double)a3[i] * (double)b3[i];
            }
        }
    }
#pragma unroll
    for (int m = 0; m < ND; m++) v[m] = (w[m][0] + w[m][1]) + (w[m][2] + w[m][3]);
    block_sum<ND>(v, sh);
    if (threadIdx.x == 0) {
#pragma unroll
        for (int m = 0; m < ND; m++) partial[blockIdx.x * 4 + m] = v[m];
        __threadfence();
        const unsigned t = atomicAdd(counter, 1u);
        last = (t == gridDim.x - 1);
    }
    __syncthreads();
    if (!last) return;
    __threadfence();
#pragma unroll
    for (int m = 0; m < ND; m++) v[m] = 0.0;
    for (int b = threadIdx.x; b < (int)gridDim.x; b += blockDim.x)
#pragma unroll
        for (int m = 0; m < ND; m++) v[m] += __builtin_nontemporal_load(&partial[b * 4 + m]);
    __syncthreads();
    block_sum<ND>(v, sh);
    if (threadIdx.x == 0) {
#pragma unroll
        for (int m = 0; m < ND; m++) out[m] = v[m];
        *counter = 0u;
    }
}

template <typename V>
void dots(hipStream_t s, chip_ctx *c, int n, int nd, const V *a0, const V *b0, typename same_t<const V *>::type a1,
          typename same_t<const V *>::type b1, typename same_t<const V *>::type a2, typename same_t<const V *>::type b2,
          typename same_t<const V *>::type a3, typename same_t<const V *>::type b3, double *out) {
    const int nb = std::min(DOT_MAXB, std::max(1, (n + DOT_TPB * 4 - 1) / (DOT_TPB * 4)));
    switch (nd) {
    case 1: hipLaunchKernelGGL((k_dots<1, V>), dim3(nb), dim3(DOT_TPB), 0, s, n, a0, b0, a1, b1, a2, b2, a3, b3, c->partial, c->counter, out); break;
    case 2: hipLaunchKernelGGL((k_dots<2, V>), dim3(nb), dim3(DOT_TPB), 0, s, n, a0, b0, a1, b1, a2, b2, a3, b3, c->partial, c->counter, out); break;
    case 3: hipLaunchKernelGGL((k_dots<3, V>), dim3(nb), dim3(DOT_TPB), 0, s, n, a0, b0, a1, b1, a2, b2, a3, b3, c->partial, c->counter, out); break;
    default: hipLaunchKernelGGL((k_dots<4, V>), dim3(nb), dim3(DOT_TPB), 0, s, n, a0, b0, a1, b1, a2, b2, a3, b3, c->partial, c->counter, out); break;
    }
}
template void dots<double>(hipStream_t, chip_ctx *, int, int, const double *, const double *, const double *,
                           const double *, const double *, const double *, const double *, const double *, double *);
template void dots<float>(hipStream_t, chip_ctx *, int, int, const float *, const float *, const float *,
                          const float *, const float *, const float *, const float *, const float *, double *);

// multi_grid's line search on a small level in one launch of one workgroup
// (General_matrix_functions.c:626-638): sc = (AU.AU, AU.res), alpha =
// sc[1] / sc[0], vel += alpha del and, with resout, resout -= alpha AU
// (resout may be res: every read of res precedes the barrier).  In place of
// dots + mg_update where the level's vectors are short enough that the two
// launches, not the bytes, set the time: one CU streams about 100 GB/s, so
// at 8192 entries (about 160 KB moved) the one launch takes 2 us.
constexpr int LS_TPB = 1024;
constexpr long LS_MAX_N = 8192;

template <typename V>
__global__ void __launch_bounds__(LS_TPB) k_line_search(long n, V *__restrict__ vel, const V *__restrict__ del,
                                                        V *resout, const V *__restrict__ AU, const V *res,
                                                        double *__restrict__ sc) {
    __shared__ double sh[4 * 16];
    __shared__ double alpha_s;
    double v[2] = {0.0, 0.0};
    for (long i = threadIdx.x; i < n; i += LS_TPB) {
        const double a = (double)AU[i];
        v[0] += a * a;
        v[1] += a * (double)res[i];
    }
    block_sum<2>(v, sh);
    if (threadIdx.x == 0) {
        sc[0] = v[0];
        sc[1] = v[1];
        alpha_s = v[1] / v[0];
    }
    __syncthreads();
    const V alpha = (V)alpha_s;
    for (long i = threadIdx.x; i < n; i += LS_TPB) {
        vel[i] += alpha * del[i];
        if (resout) resout[i] -= alpha * AU[i];
    }
}

bool line_search_ok(long n) { return n <= LS_MAX_N; }

template <typename V>
void line_search(hipStream_t s, long n, V *vel, const V *del, V *resout, const V *AU, const V *res, double *sc) {
    hipLaunchKernelGGL(k_line_search<V>, dim3(1), dim3(LS_TPB), 0, s, n, vel, del, resout, AU, res, sc);
}
template void line_search<double>(hipStream_t, long, double *, const double *, double *, const double *,
                                  const double *, double *);
template void line_search<float>(hipStream_t, long, float *, const float *, float *, const float *, const float *,
                                 double *);

// ---------------------------------------------------------------------------
// elementwise

template <typename V>
__global__ void k_fill(V *v, V val, long n) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) v[i] = val;
}
void fill(hipStream_t s, double *v, double val, long n) { hipLaunchKernelGGL(k_fill<double>, dim3(nblk(n)), dim3(TPB), 0, s, v, val, n); }
void fill(hipStream_t s, float *v, float val, long n) { hipLaunchKernelGGL(k_fill<float>, dim3(nblk(n)), dim3(TPB), 0, s, v, val, n); }

// FP64 -> FP32 (the residual handed to the FP32 multigrid)
__global__ void k_to_f32(float *d, const double *a, long n) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) d[i] = (float)a[i];
}
void to_f32(hipStream_t s, float *dst, const double *src, long n) { hipLaunchKernelGGL(k_to_f32, dim3(nblk(n)), dim3(TPB), 0, s, dst, src, n); }

// y += x with an FP32 correction x (FP64 accumulation of the refinement)
__global__ void k_add_f32(double *y, const float *x, long n) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] += (double)x[i];
}
void add_f32(hipStream_t s, double *y, const float *x, long n) { hipLaunchKernelGGL(k_add_f32, dim3(nblk(n)), dim3(TPB), 0, s, y, x, n); }

__global__ void k_copy(double *d, const double *a, long n) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) d[i] = a[i];
}
void copy(hipStream_t s, double *dst, const double *src, long n) { hipLaunchKernelGGL(k_copy, dim3(nblk(n)), dim3(TPB), 0, s, dst, src, n); }

__global__ void k_fcopy(float *d, const float *a, long n) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) d[i] = a[i];
}
void fcopy(hipStream_t s, float *dst, const float *src, long n) { hipLaunchKernelGGL(k_fcopy, dim3(nblk(n)), dim3(TPB), 0, s, dst, src, n); }

__global__ void k_axpy(double *y, const double *x, double a, long n) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] += a * x[i];
}
void axpy_scalar(hipStream_t s, double *y, const double *x, double a, long n) { hipLaunchKernelGGL(k_axpy, dim3(nblk(n)), dim3(TPB), 0, s, y, x, a, n); }

// the warm start's extrapolation along the sequence of solves: with x the
// last solution and h1, h2 the two before it, x <- x + r1 (x - h1) +
// r2 (h1 - h2); d2 (optional) <- x - 2 h1 + h2, the second difference; then
// h2 <- h1, h1 <- the old x
__global__ void k_extrapolate(double *x, double *h1, double *h2, double r1, double r2, double *d2, long n) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double xn = x[i], a = h1[i], b = h2[i];
    x[i] = xn + r1 * (xn - a) + r2 * (a - b);
    if (d2) d2[i] = (xn - a) - (a - b);
    h2[i] = a;
    h1[i] = xn;
}
void extrapolate(hipStream_t s, double *x, double *h1, double *h2, double r1, double r2, double *d2, long n) {
    hipLaunchKernelGGL(k_extrapolate, dim3(nblk(n)), dim3(TPB), 0, s, x, h1, h2, r1, r2, d2, n);
}

template <typename V>
__global__ void k_sub(V *r, const V *a, const V *b, long n) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) r[i] = a[i] - b[i];
}
void sub(hipStream_t s, double *r, const double *a, const double *b, long n) { hipLaunchKernelGGL(k_sub<double>, dim3(nblk(n)), dim3(TPB), 0, s, r, a, b, n); }
void sub(hipStream_t s, float *r, const float *a, const float *b, long n) { hipLaunchKernelGGL(k_sub<float>, dim3(nblk(n)), dim3(TPB), 0, s, r, a, b, n); }

// multi_grid line search update (General_matrix_functions.c:626-638)
template <typename V>
__global__ void k_mg_update(V *vel, const V *del, V *res, const V *AU, const double *sc, long n) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const V alpha = (V)(sc[1] / sc[0]);
    vel[i] += alpha * del[i];
    if (res) res[i] -= alpha * AU[i];
}
void mg_update(hipStream_t s, double *vel, const double *del, double *res, const double *AU, const double *sc, long n) {
    hipLaunchKernelGGL(k_mg_update<double>, dim3(nblk(n)), dim3(TPB), 0, s, vel, del, res, AU, sc, n);
}
void mg_update(hipStream_t s, float *vel, const float *del, float *res, const float *AU, const double *sc, long n) {
    hipLaunchKernelGGL(k_mg_update<float>, dim3(nblk(n)), dim3(TPB), 0, s, vel, del, res, AU, sc, n);
}

__global__ void k_uz_z(double *z1, const double *BPI, const double *r1, long n) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) z1[i] = BPI[i] * r1[i];
}
void uz_z(hipStream_t s, double *z1, const double *BPI, const double *r1, long n) { hipLaunchKernelGGL(k_uz_z, dim3(nblk(n)), dim3(TPB), 0, s, z1, BPI, r1, n); }

// s2 = z1 + delta s1, delta = *num / *den (Stokes_flow_Incomp.c:401-411)
__global__ void k_uz_search(double *s2, const double *z1, const double *s1, const double *num, const double *den,
                            int first, long n) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (first) s2[i] = z1[i];
    else {
        const double delta = *num / *den;
        s2[i] = z1[i] + delta * s1[i];
    }
}
void uz_search(hipStream_t s, double *s2, const double *z1, const double *s1, const double *num, const double *den,
               int first, long n) {
    hipLaunchKernelGGL(k_uz_search, dim3(nblk(n)), dim3(TPB), 0, s, s2, z1, s1, num, den, first, n);
}

// r2 = r1 - alpha Ah, P += alpha s2 with alpha = valid ? *num / *den : 0
// (Stokes_flow_Incomp.c:420-431)
__global__ void k_uz_pupdate(double *r2, const double *r1, const double *Ah, double *P, const double *s2,
                             const double *num, const double *den, int valid, long n) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double alpha = valid ? *num / *den : 0.0;
    r2[i] = r1[i] - alpha * Ah[i];
    P[i] += alpha * s2[i];
}
void uz_pupdate(hipStream_t s, double *r2, const double *r1, const double *Ah, double *P, const double *s2,
                const double *num, const double *den, int valid, long n) {
    hipLaunchKernelGGL(k_uz_pupdate, dim3(nblk(n)), dim3(TPB), 0, s, r2, r1, Ah, P, s2, num, den, valid, n);
}

// V -= alpha u1 (Stokes_flow_Incomp.c:433-434)
__global__ void k_uz_vupdate(double *V, const double *u1, const double *num, const double *den, int valid, long n) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double alpha = valid ? *num / *den : 0.0;
    V[i] -= alpha * u1[i];
}
void uz_vupdate(hipStream_t s, double *V, const double *u1, const double *num, const double *den, int valid, long n) {
    hipLaunchKernelGGL(k_uz_vupdate, dim3(nblk(n)), dim3(TPB), 0, s, V, u1, num, den, valid, n);
}

// Ah = F - gradP - K V (Stokes_flow_Incomp.c:357-358)
__global__ void k_init_residual(double *Ah, const double *F, const double *gP, const double *KV, long n) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) Ah[i] = F[i] - gP[i] - KV[i];
}
void init_residual(hipStream_t s, double *Ah, const double *F, const double *gradP, const double *KV, long n) {
    hipLaunchKernelGGL(k_init_residual, dim3(nblk(n)), dim3(TPB), 0, s, Ah, F, gradP, KV, n);
}

// v_from_vector (Stokes_flow_Incomp.c:530-552); prescribed velocities are zero
__global__ void k_v_from_vector(Geo g, const unsigned *__restrict__ NODE, const double *__restrict__ U, float *V) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= g.nno) return;
    const unsigned f = NODE[n];
    V[n] = (f & VBX) ? 0.0f : (float)U[3 * n];
    V[g.nno + n] = (f & VBY) ? 0.0f : (float)U[3 * n + 1];
    V[2 * g.nno + n] = (f & VBZ) ? 0.0f : (float)U[3 * n + 2];
}
void v_from_vector(hipStream_t s, const Level &L, const double *U, float *V) {
    hipLaunchKernelGGL(k_v_from_vector, dim3(nblk(L.g.nno)), dim3(TPB), 0, s, L.g, L.NODE, U, V);
}

// velocities_conform_bcs (Boundary_conditions.c:993-1023) with VB = 0
void conform_velocity(hipStream_t s, const Level &L, double *U) { strip(s, L, U); }

// ---------------------------------------------------------------------------
// stiffness rebuild

// visc_from_T (Viscosity_structures.c:491-737, rheol 0, 3 and 11) or
// visc_from_mat (:477-489), then the MAX / MIN clip of get_system_viscosity
struct ViscLaw {
    int rheol, tdepv, vmin_on, vmax_on;
    float visc0[4], viscE[4], viscT[4];
    float visc_min, visc_max;
};

__global__ void __launch_bounds__(TPB) k_visc_from_T(Geo g, ViscLaw law, const int *__restrict__ mat,
                                                     const float *__restrict__ T, float *__restrict__ evi) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= g.nel) return;
    const int ez = e % g.elz, ex = (e / g.elz) % g.elx, ey = e / (g.elz * g.elx);
    const int l = mat[e] - 1;
    const float tempa = law.visc0[l];
    float TT[9];
#pragma unroll
    for (int a = 1; a <= 8; a++) TT[a] = T[nid(g, ez + cOffz[a], ex + cOffx[a], ey + cOffy[a])];
    for (int jj = 1; jj <= 8; jj++) {
        float v;
        if (!law.tdepv) {
            v = tempa;
        } else {
            float temp = 1.0e-32f;
#pragma unroll
            for (int kk = 1; kk <= 8; kk++) temp = (float)(temp + fmaxf(0.0f, TT[kk]) * cNv[8 * (kk - 1) + jj - 1]);
            if (law.rheol == 11) {
                // eta0 exp(E/(T+T0) - E/(0.5+T0)): the first quotient in
                // float, the second in double (the literal 0.5), :697-719
                const double arg = (double)(law.viscE[l] / (temp + law.viscT[l])) -
                                   (double)law.viscE[l] / (0.5 + (double)law.viscT[l]);
                v = (float)(tempa * exp(arg));
            } else {
                float arg;
                if (law.rheol == 3) arg = law.viscE[l] * (law.viscT[l] - temp);
                else arg = law.viscE[l] * (1.0f - temp);
                v = (float)(tempa * exp((double)arg));
            }
        }
        if (law.vmax_on && v > law.visc_max) v = law.visc_max;
        if (law.vmin_on && v < law.visc_min) v = law.visc_min;
        evi[e * 8 + jj - 1] = v;
    }
}

void visc_from_T(hipStream_t s, const chip_ctx *c, const float *T, float *evi) {
    ViscLaw law{};
    law.rheol = c->p.rheol;
    law.tdepv = c->p.tdepv;
    law.vmin_on = c->p.vmin_on;
    law.vmax_on = c->p.vmax_on;
    law.visc_min = c->p.visc_min;
    law.visc_max = c->p.visc_max;
    for (int i = 0; i < 4; i++) {
        law.visc0[i] = c->p.visc0[i];
        law.viscE[i] = c->p.viscE[i];
        law.viscT[i] = c->p.viscT[i];
    }
    const Geo &g = c->L[c->levmax].g;
    hipLaunchKernelGGL(k_visc_from_T, dim3(nblk(g.nel)), dim3(TPB), 0, s, g, law, c->mat, T, evi);
}

// visc_from_gint_to_nodes (Nodal_mesh.c:583-615)
__global__ void __launch_bounds__(TPB) k_visc_to_nodes(Geo g, const float *__restrict__ EVI,
                                                       const float *__restrict__ TWW, const float *__restrict__ MASS,
                                                       float *__restrict__ VN) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= g.nno) return;
    int k, i, j;
    node_kij(g, n, k, i, j);
    float acc = 0.0f;
    for (int ey = j - 1; ey <= j; ey++) {
        if ((unsigned)ey >= (unsigned)g.ely) continue;
        for (int ex = i - 1; ex <= i; ex++) {
            if ((unsigned)ex >= (unsigned)g.elx) continue;
            for (int ez = k - 1; ez <= k; ez++) {
                if ((unsigned)ez >= (unsigned)g.elz) continue;
                const int e = ez + g.elz * (ex + g.elx * ey);
                double tv = 0.0;
#pragma unroll
                for (int q = 0; q < 8; q++) tv += EVI[e * 8 + q];
                tv = tv / 8;
                const int a = cLoc[(k - ez) + 2 * (i - ex) + 4 * (j - ey)];
                acc = (float)(acc + TWW[(size_t)e * TWW_SZ + a] * tv);
            }
        }
    }
    VN[n] = acc * MASS[n];
}

// project_scalar (Solver_multigrid.c:344-388), result into the coarse VN
__global__ void __launch_bounds__(TPB) k_visc_project(Geo gf, Geo gc, const float *__restrict__ VNf,
                                                      const float *__restrict__ TWW, const float *__restrict__ MASS,
                                                      float *__restrict__ VNc) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= gc.nno) return;
    int k, i, j;
    node_kij(gc, n, k, i, j);
    float acc = 0.0f;
    for (int ey = j - 1; ey <= j; ey++) {
        if ((unsigned)ey >= (unsigned)gc.ely) continue;
        for (int ex = i - 1; ex <= i; ex++) {
            if ((unsigned)ex >= (unsigned)gc.elx) continue;
            for (int ez = k - 1; ez <= k; ez++) {
                if ((unsigned)ez >= (unsigned)gc.elz) continue;
                const int a = cLoc[(k - ez) + 2 * (i - ex) + 4 * (j - ey)];
                const int el = ez + gc.elz * (ex + gc.elx * ey);
                const int fz = 2 * ez + cOffz[a], fx = 2 * ex + cOffx[a], fy = 2 * ey + cOffy[a];
                float average = 0.0f;
#pragma unroll
                for (int b = 1; b <= 8; b++) average += VNf[nid(gf, fz + cOffz[b], fx + cOffx[b], fy + cOffy[b])];
                const float w = (float)((1.0 / 8) * average);
                acc += w * TWW[(size_t)el * TWW_SZ + a];
            }
        }
    }
    VNc[n] = acc * MASS[n];
}

// visc_from_nodes_to_gint (Nodal_mesh.c:617-640)
__global__ void __launch_bounds__(TPB) k_visc_to_gint(Geo g, const float *__restrict__ VN, float *__restrict__ EVI) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= g.nel) return;
    const int ez = e % g.elz, ex = (e / g.elz) % g.elx, ey = e / (g.elz * g.elx);
    float vn[9];
#pragma unroll
    for (int a = 1; a <= 8; a++) vn[a] = VN[nid(g, ez + cOffz[a], ex + cOffx[a], ey + cOffy[a])];
#pragma unroll
    for (int i = 1; i <= 8; i++) {
        double tv = 0.0;
#pragma unroll
        for (int j = 1; j <= 8; j++) tv += cNv[8 * (j - 1) + i - 1] * vn[j];
        EVI[e * 8 + i - 1] = (float)tv;
    }
}

void project_viscosity(hipStream_t s, const Level &fine, const Level &coarse) {
    hipLaunchKernelGGL(k_visc_to_nodes, dim3(nblk(fine.g.nno)), dim3(TPB), 0, s, fine.g, fine.EVI, fine.TWW, fine.MASS,
                       fine.VN);
    hipLaunchKernelGGL(k_visc_project, dim3(nblk(coarse.g.nno)), dim3(TPB), 0, s, fine.g, coarse.g, fine.VN,
                       coarse.TWW, coarse.MASS, coarse.VN);
    hipLaunchKernelGGL(k_visc_to_gint, dim3(nblk(coarse.g.nel)), dim3(TPB), 0, s, coarse.g, coarse.VN, coarse.EVI);
}

// get_elt_g (Element_calculations.c:831-934, CART3D)
__global__ void k_elt_g(Geo g, const float *__restrict__ GNX, const float *__restrict__ GDA, float *__restrict__ EG) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= g.nel) return;
    const float *gnx = GNX + (size_t)e * GNX_SZ + 192;
    const float tf = 8.0f * GDA[(size_t)e * GDA_SZ + 10];
    const double temp = tf;
#pragma unroll
    for (int a = 1; a <= 8; a++) {
        const int p = 3 * (a - 1);
        EG[(size_t)e * EG_SZ + p] = (float)(-gnx[a - 1] * temp);
        EG[(size_t)e * EG_SZ + p + 1] = (float)(-gnx[8 + a - 1] * temp);
        EG[(size_t)e * EG_SZ + p + 2] = (float)(-gnx[16 + a - 1] * temp);
    }
}

void elt_g(hipStream_t s, const Level &L) {
    hipLaunchKernelGGL(k_elt_g, dim3(nblk(L.g.nel)), dim3(TPB), 0, s, L.g, L.GNX, L.GDA, L.EG);
}

// 3x3 block of the element stiffness elt_k (get_elt_k, Element_calculations.c:
// 133-293, cartesian isotropic) plus get_aug_k (:1127-1163): rows of local
// node ar, columns of local node bc.  The reference evaluates the (a,b) block
// for a <= b and stores its transpose below the diagonal; the aug term is
// added per entry in the (row, column) orientation.
__device__ void elt_block(const float *__restrict__ gnx, const float *__restrict__ gda, const float *__restrict__ evi,
                          const float *__restrict__ eg, int aug_on, double aug, int ar, int bc, double blk[3][3]) {
    const int a = ar < bc ? ar : bc, b = ar < bc ? bc : ar;
    double m[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}}, temp = 0.0;
#pragma unroll
    for (int k = 1; k <= 8; k++) {
        float wf = 1.0f * gda[k];
        wf = wf * evi[k - 1];
        const double W = wf;
        const float ax = gnx[8 * (a - 1) + k - 1], ay = gnx[64 + 8 * (a - 1) + k - 1], az = gnx[128 + 8 * (a - 1) + k - 1];
        const float bx = gnx[8 * (b - 1) + k - 1], by = gnx[64 + 8 * (b - 1) + k - 1], bz = gnx[128 + 8 * (b - 1) + k - 1];
        m[0][0] += W * ax * bx;
        m[0][1] += W * ay * bx;
        m[0][2] += W * az * bx;
        m[1][0] += W * ax * by;
        m[1][1] += W * ay * by;
        m[1][2] += W * az * by;
        m[2][0] += W * ax * bz;
        m[2][1] += W * ay * bz;
        m[2][2] += W * az * bz;
    }
#pragma unroll
    for (int k = 1; k <= 8; k++) {
        float wf = 1.0f * gda[k];
        wf = wf * evi[k - 1];
        const double W = wf;
        const float s = gnx[8 * (a - 1) + k - 1] * gnx[8 * (b - 1) + k - 1] +
                        gnx[64 + 8 * (a - 1) + k - 1] * gnx[64 + 8 * (b - 1) + k - 1] +
                        gnx[128 + 8 * (a - 1) + k - 1] * gnx[128 + 8 * (b - 1) + k - 1];
        temp += W * s;
    }
    m[0][0] += temp;
    m[1][1] += temp;
    m[2][2] += temp;
    const bool tr = ar > bc;
#pragma unroll
    for (int r = 0; r < 3; r++)
#pragma unroll
        for (int c = 0; c < 3; c++) blk[r][c] = tr ? m[c][r] : m[r][c];
    if (aug_on) {
        double visc = 0.0;
#pragma unroll
        for (int q = 0; q < 8; q++) visc += evi[q];
        visc = visc / 8;
#pragma unroll
        for (int r = 0; r < 3; r++)
#pragma unroll
            for (int c = 0; c < 3; c++) blk[r][c] += visc * aug * eg[3 * (ar - 1) + r] * eg[3 * (bc - 1) + c];
    }
}

// ---------------------------------------------------------------------------
// Compact geometry of brick elements.  On a mesh given by one coordinate array
// per axis every element is a brick, and its 192 shape-function derivatives
// are twelve numbers: the derivative along an axis of node a at Gauss point q
// depends on whether a and q lie on the same side along the other two axes,
// and its sign on a's side along this one; the eight Jacobians are one, and
// the 24 entries of elt_del three.  k_brick gathers them, entry by entry of
// the arrays as the reference computes them, [BRICK_SZ][nel] so that elements
// side by side are read side by side, and counts the elements whose arrays are
// not reproduced bit for bit (those levels keep the arrays).  The kernels that
// read the derivatives are bound by these bytes: 908 B an element as arrays
// (a cache line per lane and entry), 80 B so.
constexpr int CORNER_X[8] = {0, 1, 1, 0, 0, 1, 1, 0}, CORNER_Y[8] = {0, 0, 1, 1, 0, 0, 1, 1},
              CORNER_Z[8] = {0, 0, 0, 0, 1, 1, 1, 1};
constexpr int BRICK_B = 0, BRICK_J = 12, BRICK_E = 13, BRICK_SIZE = 16, BRICK_AREA = 19;

// which of the four values of axis d: sides of a and q along the other axes
__device__ constexpr int brick_idx(int d, int a, int q) {
    const int x = CORNER_X[a] ^ CORNER_X[q], y = CORNER_Y[a] ^ CORNER_Y[q], z = CORNER_Z[a] ^ CORNER_Z[q];
    return d == 0 ? y + 2 * z : d == 1 ? x + 2 * z : x + 2 * y;
}
__device__ constexpr bool brick_up(int d, int a) {
    return (d == 0 ? CORNER_X[a] : d == 1 ? CORNER_Y[a] : CORNER_Z[a]) != 0;
}

__global__ void __launch_bounds__(64) k_brick(Geo g, const float *__restrict__ GNX, const float *__restrict__ GDA,
                                              const float *__restrict__ ECO, float *__restrict__ GB, int *bad) {
    const int e = blockIdx.x * 64 + threadIdx.x;
    if (e >= g.nel) return;
    const float *gnx = GNX + (size_t)e * GNX_SZ, *gda = GDA + (size_t)e * GDA_SZ, *eco = ECO + (size_t)e * ECO_SZ;
    bool ok = true;
#pragma unroll
    for (int d = 0; d < 3; d++) {
        float b[4];
#pragma unroll
        for (int q = 0; q < 8; q++) b[brick_idx(d, 6, q)] = gnx[64 * d + 8 * 6 + q];   // node 6: the far corner
#pragma unroll
        for (int a = 0; a < 8; a++) {
#pragma unroll
            for (int q = 0; q < 8; q++) {
                const float v = b[brick_idx(d, a, q)];
                ok = ok && isfinite(v) && __float_as_uint(gnx[64 * d + 8 * a + q]) == __float_as_uint(brick_up(d, a) ? v : -v);
            }
            const float c = gnx[192 + 8 * d + 6];
            ok = ok && __float_as_uint(gnx[192 + 8 * d + a]) == __float_as_uint(brick_up(d, a) ? c : -c);
        }
#pragma unroll
        for (int q = 0; q < 4; q++) GB[(size_t)(BRICK_B + 4 * d + q) * g.nel + e] = b[q];
        // get_elt_g: -(derivative at the centre) x weight, rounded once
        const float ed = (float)(gnx[192 + 8 * d + 6] * (double)(8.0f * gda[10]));
        ok = ok && isfinite(ed);
        GB[(size_t)(BRICK_E + d) * g.nel + e] = ed;
        GB[(size_t)(BRICK_SIZE + d) * g.nel + e] = eco[5 + d];
    }
#pragma unroll
    for (int q = 2; q <= 8; q++) ok = ok && __float_as_uint(gda[q]) == __float_as_uint(gda[1]);
    ok = ok && isfinite(gda[1]);   // elements outside the mesh count as 0 times these
    GB[(size_t)BRICK_J * g.nel + e] = gda[1];
    GB[(size_t)BRICK_AREA * g.nel + e] = eco[12];
    if (!ok) atomicAdd(bad, 1);
}

void brick(hipStream_t s, const Level &L, int *bad) {
    hipLaunchKernelGGL(k_brick, dim3(nblk(L.g.nel, 64)), dim3(64), 0, s, L.g, L.GNX, L.GDA, L.ECO, L.GB, bad);
}

// one element's geometry, from the compact form or from the arrays (d: axis,
// a: node, q: Gauss point, from 0)
template <bool BRICK>
struct ElemGeo {
    const float *gnx, *gda, *eco;
    float b[12], j, size[3];
    __device__ __forceinline__ ElemGeo(const Geo &g, const float *GB, const float *GNX, const float *GDA,
                                       const float *ECO, int e) {
        if constexpr (BRICK) {
#pragma unroll
            for (int f = 0; f < 12; f++) b[f] = GB[(size_t)(BRICK_B + f) * g.nel + e];
            j = GB[(size_t)BRICK_J * g.nel + e];
#pragma unroll
            for (int d = 0; d < 3; d++) size[d] = GB[(size_t)(BRICK_SIZE + d) * g.nel + e];
        } else {
            gnx = GNX + (size_t)e * GNX_SZ, gda = GDA + (size_t)e * GDA_SZ, eco = ECO + (size_t)e * ECO_SZ;
        }
    }
    __device__ __forceinline__ float dN(int d, int a, int q) const {
        if constexpr (BRICK) return brick_up(d, a) ? b[4 * d + brick_idx(d, a, q)] : -b[4 * d + brick_idx(d, a, q)];
        else return gnx[64 * d + 8 * a + q];
    }
    // values derived from these are formed anew after this point
    __device__ __forceinline__ void hold() {
        if constexpr (BRICK)
#pragma unroll
            for (int f = 0; f < 12; f++) asm volatile("" : "+v"(b[f]));
    }
    __device__ __forceinline__ float dA(int q) const { return BRICK ? j : gda[q + 1]; }
    __device__ __forceinline__ float len(int d) const { return BRICK ? size[d] : eco[5 + d]; }
};

// k_node_ks (below) from the compact geometry: three wavefronts per 64-node
// tile, wavefront P the 81 coefficients of y-plane dy = P - 1, through the two or
// four elements times two planes of elements that hold them in ascending element
// order.  The same products and sums: with self the
// node, m its neighbour, row r, column c, an element adds
//   sum over the Gauss points of (W lo) hi, lo and hi the derivatives (self
//   along c, m along r) of the node with the smaller and the larger local
//   number, + the Laplacian term on the diagonal, + visc aug e e
// (the reference forms one of each pair and transposes; a node's own block is
// read transposed).  Elements outside the mesh have weight 0.
// Bound by waits: 256 registers, 148 more spilled (388 B of scratch a lane), two
// wavefronts a SIMD that wait in 63 % of their cycles; vector instructions take
// 47 % of the time, and the 17000 FP64 operations a node would take a seventh
// at their full rate.  128x128x64 elements, finest level 1.7 ms, from the
// arrays (one thread a node) 12 to 17.
__global__ void __launch_bounds__(192, 2) k_node_ks_brick(Geo g, const float *__restrict__ GB, const float *__restrict__ EVI,
                                                          const unsigned *__restrict__ NODE, int aug_on, double aug,
                                                          float *__restrict__ K, double *__restrict__ BI) {
    const int lane = threadIdx.x & 63, P = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int q = blockIdx.x * 64 + lane;
    const int col = colour_valid(g, q);
    int k = 0, i = 0, j = 0;
    if (col >= 0) colour_kij(g, col, q, k, i, j);
    const int self = nid(g, k, i, j);
    float acc[9][3][3];
    double diag[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int b = 0; b < 9; b++)
#pragma unroll
        for (int r = 0; r < 3; r++)
#pragma unroll
            for (int c = 0; c < 3; c++) acc[b][r][c] = 0.0f;
#pragma unroll 1
    for (int my = P == 2; my <= (P >= 1); my++) {   // element rows ey = j - 1 + my
        const int by = P - my, ay = 1 - my;          // sides of m and of the node along y
#pragma unroll
        for (int mx = 0; mx < 2; mx++)
#pragma unroll
            for (int mz = 0; mz < 2; mz++) {
                const int ez = k - 1 + mz, ex = i - 1 + mx, ey = j - 1 + my;
                const bool ok = (unsigned)ez < (unsigned)g.elz && (unsigned)ex < (unsigned)g.elx &&
                                (unsigned)ey < (unsigned)g.ely;
                const int e = ok ? ez + g.elz * (ex + g.elx * ey) : 0;
                const int ax = 1 - mx, az = 1 - mz;
                const float *gb = GB + e;
                float B[3][4], E[3];
#pragma unroll
                for (int f = 0; f < 12; f++) B[f / 4][f % 4] = gb[(size_t)(BRICK_B + f) * g.nel];
#pragma unroll
                for (int d = 0; d < 3; d++) E[d] = gb[(size_t)(BRICK_E + d) * g.nel];
                const float jv = gb[(size_t)BRICK_J * g.nel];
                float evi[8];
                {
                    const float4 v0 = *reinterpret_cast<const float4 *>(EVI + (size_t)e * 8);
                    const float4 v1 = *reinterpret_cast<const float4 *>(EVI + (size_t)e * 8 + 4);
                    evi[0] = v0.x, evi[1] = v0.y, evi[2] = v0.z, evi[3] = v0.w;
                    evi[4] = v1.x, evi[5] = v1.y, evi[6] = v1.z, evi[7] = v1.w;
                }
                double W[8], visc = 0.0;
#pragma unroll
                for (int p = 0; p < 8; p++) {
                    const float wf = (1.0f * jv) * evi[p];
                    W[p] = ok ? (double)wf : 0.0;
                    visc += evi[p];
                }
                visc = visc / 8;
                const double va = ok && aug_on ? visc * aug : 0.0;
                // values of the node (side ay) and of m (side by) along y: x and z
                // derivatives by the Gauss point's y side, y derivatives' sign
                float Sx[2][2], Sz[2][2], Sy[4], Mx[2][2], Mz[2][2], My[4];   // [y side][z side], [y side][x side]
#pragma unroll
                for (int y = 0; y < 2; y++)
#pragma unroll
                    for (int o = 0; o < 2; o++) {
                        Sx[y][o] = ay ? B[0][(1 - y) + 2 * o] : B[0][y + 2 * o];
                        Mx[y][o] = by ? B[0][(1 - y) + 2 * o] : B[0][y + 2 * o];
                        Sz[y][o] = ay ? B[2][o + 2 * (1 - y)] : B[2][o + 2 * y];
                        Mz[y][o] = by ? B[2][o + 2 * (1 - y)] : B[2][o + 2 * y];
                    }
#pragma unroll
                for (int o = 0; o < 4; o++) {
                    Sy[o] = ay ? B[1][o] : -B[1][o];
                    My[o] = by ? B[1][o] : -B[1][o];
                }
                float S[3][8];
#pragma unroll
                for (int p = 0; p < 8; p++) {
                    const int qx = CORNER_X[p], qy = CORNER_Y[p], qz = CORNER_Z[p];
                    const float sx = Sx[qy][az ^ qz], sz = Sz[qy][ax ^ qx];
                    S[0][p] = ax ? sx : -sx;
                    S[1][p] = Sy[(ax ^ qx) + 2 * (az ^ qz)];
                    S[2][p] = az ? sz : -sz;
                }
                const double ES[3] = {ax ? -E[0] : E[0], ay ? -E[1] : E[1], az ? -E[2] : E[2]};
#pragma unroll
                for (int bx = 0; bx < 2; bx++)
#pragma unroll
                    for (int bz = 0; bz < 2; bz++) {
                        const int b = (mz + bz) + 3 * (mx + bx);
                        // formed anew in each block: shared over the blocks the
                        // products would not fit the registers
#pragma unroll
                        for (int p = 0; p < 8; p++) {
                            asm volatile("" : "+v"(W[p]));
#pragma unroll
                            for (int d = 0; d < 3; d++) asm volatile("" : "+v"(S[d][p]));
                        }
                        double T[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}}, temp = 0.0;
                        // local numbers: z first, then (x, y) in the order 00 10 11 01
                        const int oa = ax ? 1 + ay : 3 * ay, ob = bx ? 1 + by : 3 * by;
                        const bool self_lo = az != bz ? az == 0 : oa <= ob;
                        auto sum = [&](auto lo) {
#pragma unroll
                            for (int p = 0; p < 8; p++) {
                                const int qx = CORNER_X[p], qy = CORNER_Y[p], qz = CORNER_Z[p];
                                const float mxv = Mx[qy][bz ^ qz], mzv = Mz[qy][bx ^ qx];
                                const float M[3] = {bx ? mxv : -mxv, My[(bx ^ qx) + 2 * (bz ^ qz)], bz ? mzv : -mzv};
                                double wl[3];   // W times the lower node's derivatives
#pragma unroll
                                for (int d = 0; d < 3; d++) wl[d] = W[p] * (lo.value ? S[d][p] : M[d]);
#pragma unroll
                                for (int r = 0; r < 3; r++)
#pragma unroll
                                    for (int c = 0; c < 3; c++) T[r][c] += lo.value ? wl[c] * M[r] : wl[r] * S[c][p];
                                const float s = S[0][p] * M[0] + S[1][p] * M[1] + S[2][p] * M[2];
                                temp += W[p] * s;
                            }
                        };
                        if (self_lo) sum(std::true_type{});
                        else sum(std::false_type{});
                        T[0][0] += temp;
                        T[1][1] += temp;
                        T[2][2] += temp;
                        if (aug_on) {
                            const double EM[3] = {bx ? -E[0] : E[0], by ? -E[1] : E[1], bz ? -E[2] : E[2]};
                            // m <= the node (in node order): the node's rows are the larger node's
                            const int dx = mx + bx - 1, dz = mz + bz - 1;
                            const bool nbig = P == 0 || (P == 1 && (dx < 0 || (dx == 0 && dz <= 0)));
#pragma unroll
                            for (int r = 0; r < 3; r++)
#pragma unroll
                                for (int c = 0; c < 3; c++) T[r][c] += nbig ? va * ES[r] * EM[c] : va * EM[c] * ES[r];
                        }
                        if (b == 4 && P == 1) {
                            diag[0] += T[0][0];
                            diag[1] += T[1][1];
                            diag[2] += T[2][2];
                        }
#pragma unroll
                        for (int r = 0; r < 3; r++)
#pragma unroll
                            for (int c = 0; c < 3; c++) {
                                acc[b][r][c] = (float)(acc[b][r][c] + T[r][c]);
                                asm volatile("" : "+v"(acc[b][r][c]));   // added here, not kept for the loop's end
                            }
                        __builtin_amdgcn_sched_barrier(0);
                    }
            }
    }
    if (col < 0) return;
    float *kq = K + ktile(q) + (size_t)(81 * P) * 64;
    const unsigned fs = NODE[self];
    const float wr[3] = {(fs & VBX) ? 0.0f : 1.0f, (fs & VBY) ? 0.0f : 1.0f, (fs & VBZ) ? 0.0f : 1.0f};
#pragma unroll
    for (int b = 0; b < 9; b++) {
        const int km = k + b % 3 - 1, im = i + b / 3 - 1, jm = j + P - 1;
        const bool ok = (unsigned)km < (unsigned)g.noz && (unsigned)im < (unsigned)g.nox && (unsigned)jm < (unsigned)g.noy;
        const unsigned fm = NODE[ok ? nid(g, km, im, jm) : self];
        const float wc[3] = {(fm & VBX) ? 0.0f : 1.0f, (fm & VBY) ? 0.0f : 1.0f, (fm & VBZ) ? 0.0f : 1.0f};
        const bool own = b == 4 && P == 1;
#pragma unroll
        for (int r = 0; r < 3; r++)
#pragma unroll
            for (int c = 0; c < 3; c++) kq[(b * 9 + r * 3 + c) * 64] = (own ? acc[b][c][r] : acc[b][r][c]) * (wr[r] * wc[c]) + 0.0f;
    }
    if (P == 1) {
        BI[3 * self] = (float)1.0 / diag[0];
        BI[3 * self + 1] = (float)1.0 / diag[1];
        BI[3 * self + 2] = (float)1.0 / diag[2];
    }
}

// construct_node_ks (Construct_arrays.c:359-535) restated per node: the block
// coupling node n with neighbour m is the float accumulation, in element
// order, of w_r ww_c elt_k[rows of max(n,m)][cols of min(n,m)] (BC weights
// zero the prescribed rows and columns), transposed when m > n; also
// build_diagonal_of_K (Element_calculations.c:624-652) into BI = 1/diag.
__global__ void __launch_bounds__(128) k_node_ks(Geo g, const float *__restrict__ GNX, const float *__restrict__ GDA,
                                                 const float *__restrict__ EVI, const float *__restrict__ EG,
                                                 const unsigned *__restrict__ NODE, int aug_on, double aug,
                                                 float *__restrict__ K, double *__restrict__ BI) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    const int col = colour_valid(g, q);
    if (col < 0) return;
    int k, i, j;
    colour_kij(g, col, q, k, i, j);
    const int n = nid(g, k, i, j);
    float *kq = K + ktile(q);
    double diag[3] = {0.0, 0.0, 0.0};
    for (int dy = -1; dy <= 1; dy++)
        for (int dx = -1; dx <= 1; dx++)
            for (int dz = -1; dz <= 1; dz++) {
                const int s = (dz + 1) + 3 * (dx + 1) + 9 * (dy + 1);
                const int km = k + dz, im = i + dx, jm = j + dy;
                float acc[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
                const bool ok = (unsigned)km < (unsigned)g.noz && (unsigned)im < (unsigned)g.nox &&
                                (unsigned)jm < (unsigned)g.noy;
                if (ok) {
                    const int m = nid(g, km, im, jm);
                    const bool nbig = (m <= n);
                    const int big = nbig ? n : m, small = nbig ? m : n;
                    const unsigned fb = NODE[big], fs = NODE[small];
                    const double w[3] = {(fb & VBX) ? 0.0 : 1.0, (fb & VBY) ? 0.0 : 1.0, (fb & VBZ) ? 0.0 : 1.0};
                    const double ww[3] = {(fs & VBX) ? 0.0 : 1.0, (fs & VBY) ? 0.0 : 1.0, (fs & VBZ) ? 0.0 : 1.0};
                    const int kb = nbig ? k : km, ib = nbig ? i : im, jb = nbig ? j : jm;
                    const int ks = nbig ? km : k, is = nbig ? im : i, js = nbig ? jm : j;
                    // elements holding both nodes, ascending element number
                    for (int ey = max(j, jm) - 1; ey <= min(j, jm); ey++) {
                        if ((unsigned)ey >= (unsigned)g.ely) continue;
                        for (int ex = max(i, im) - 1; ex <= min(i, im); ex++) {
                            if ((unsigned)ex >= (unsigned)g.elx) continue;
                            for (int ez = max(k, km) - 1; ez <= min(k, km); ez++) {
                                if ((unsigned)ez >= (unsigned)g.elz) continue;
                                const int e = ez + g.elz * (ex + g.elx * ey);
                                const int ab = cLoc[(kb - ez) + 2 * (ib - ex) + 4 * (jb - ey)];
                                const int as = cLoc[(ks - ez) + 2 * (is - ex) + 4 * (js - ey)];
                                double blk[3][3];
                                elt_block(GNX + (size_t)e * GNX_SZ, GDA + (size_t)e * GDA_SZ, EVI + (size_t)e * 8,
                                          EG + (size_t)e * EG_SZ, aug_on, aug, ab, as, blk);
                                if (s == 13) {
                                    diag[0] += blk[0][0];
                                    diag[1] += blk[1][1];
                                    diag[2] += blk[2][2];
                                }
                                // reference order: column direction outer, row inner
#pragma unroll
                                for (int c = 0; c < 3; c++)
#pragma unroll
                                    for (int r = 0; r < 3; r++)
                                        acc[r][c] = (float)(acc[r][c] + w[r] * ww[c] * blk[r][c]);
                            }
                        }
                    }
                    // m > n: the lower node's stored block, transposed.  m == n:
                    // the reference's matvec and smoother read a node's own block
                    // through the column loop (Element_calculations.c:604-605,
                    // General_matrix_functions.c:1254-1255), i.e. transposed too
                    if (!nbig || s == 13) {
                        float t[3][3];
#pragma unroll
                        for (int r = 0; r < 3; r++)
#pragma unroll
                            for (int c = 0; c < 3; c++) t[r][c] = acc[c][r];
#pragma unroll
                        for (int r = 0; r < 3; r++)
#pragma unroll
                            for (int c = 0; c < 3; c++) acc[r][c] = t[r][c];
                    }
                }
#pragma unroll
                for (int r = 0; r < 3; r++)
#pragma unroll
                    for (int c = 0; c < 3; c++) kq[(s * 9 + r * 3 + c) * 64] = acc[r][c];
            }
    BI[3 * n] = (float)1.0 / diag[0];
    BI[3 * n + 1] = (float)1.0 / diag[1];
    BI[3 * n + 2] = (float)1.0 / diag[2];
}

void node_ks(hipStream_t s, const Level &L, const chip_problem &p) {
    if (L.brick && L.eg_brick) {
        hipLaunchKernelGGL(k_node_ks_brick, dim3(L.g.pitch / 64), dim3(192), 0, s, L.g, L.GB, L.EVI, L.NODE, p.aug_lagr,
                           p.aug_number, L.K, L.BI);
        return;
    }
    hipLaunchKernelGGL(k_node_ks, dim3(nblk(L.g.pitch, 128)), dim3(128), 0, s, L.g, L.GNX, L.GDA, L.EVI, L.EG, L.NODE,
                       p.aug_lagr, p.aug_number, L.K, L.BI);
}

// assemble_dAhatp_entry / build_diagonal_of_Ahat (Element_calculations.c:654-685, 771-824)
__global__ void k_bpi(Geo g, const float *__restrict__ EG, const double *__restrict__ BI, int precond,
                      double *__restrict__ BPI) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= g.nel) return;
    if (!precond) {
        BPI[e] = 1.0;
        return;
    }
    const int ez = e % g.elz, ex = (e / g.elz) % g.elx, ey = e / (g.elz * g.elx);
    const float *eg = EG + (size_t)e * EG_SZ;
    double divU = 0.0;
#pragma unroll
    for (int a = 1; a <= 8; a++) {
        const int n = nid(g, ez + cOffz[a], ex + cOffx[a], ey + cOffy[a]);
#pragma unroll
        for (int d = 0; d < 3; d++) {
            const double gp = BI[3 * n + d] * eg[3 * (a - 1) + d];
            divU += eg[3 * (a - 1) + d] * gp;
        }
    }
    BPI[e] = (divU != 0.0) ? 1.0 / divU : 1.0;
}

void build_bpi(hipStream_t s, const Level &L, int precond) {
    hipLaunchKernelGGL(k_bpi, dim3(nblk(L.g.nel)), dim3(TPB), 0, s, L.g, L.EG, L.BI, precond, L.BPI);
}

// ---------------------------------------------------------------------------
// energy equation

// order-preserving float <-> unsigned maps for atomic min / max
__device__ __forceinline__ unsigned ford(float f) {
    const unsigned b = __float_as_uint(f);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}

// std_timestep (Advection_diffusion.c:737-810): per-element advective limit
// min into minmax[0]; Tmax (Global_operations.c:394-406) into minmax[1].
// The sizes lie ECO_SZ apart in ECO and side by side in the compact geometry
// (stride nel).  One atomic per wavefront on the same two words was the whole
// of it (387 us at 128x128x64 elements, so 21): up to 1024 workgroups go over
// the mesh, and one adds only what the words do not hold already.
__global__ void __launch_bounds__(TPB) k_timestep_tmax(Geo g, const float *__restrict__ size, int se, long sd,
                                                       const float *__restrict__ V, const float *__restrict__ T,
                                                       unsigned *minmax) {
    __shared__ unsigned sh[2][TPB / 64];
    unsigned mn = ford(1.0e8f), mx = ford(-10.0f);
    for (int t = blockIdx.x * TPB + threadIdx.x; t < max(g.nel, g.nno); t += gridDim.x * TPB) {
        if (V && t < g.nel) {
            const int e = t;
            const int ez = e % g.elz, ex = (e / g.elz) % g.elx, ey = e / (g.elz * g.elx);
            float uc1 = 0.0f, uc2 = 0.0f, uc3 = 0.0f;
#pragma unroll
            for (int a = 1; a <= 8; a++) {
                const int nd = nid(g, ez + cOffz[a], ex + cOffx[a], ey + cOffy[a]);
                uc1 = (float)(uc1 + cNp[a - 1] * V[nd]);
                uc2 = (float)(uc2 + cNp[a - 1] * V[g.nno + nd]);
                uc3 = (float)(uc3 + cNp[a - 1] * V[2 * g.nno + nd]);
            }
            const float *h = size + (size_t)e * se;
            const float uc = (float)(fabs((double)uc1) / h[0] + fabs((double)uc2) / h[sd] + fabs((double)uc3) / h[2 * sd]);
            const float step = (float)(0.5 / uc);
            mn = min(mn, ford(step));
        }
        if (t < g.nno) mx = max(mx, ford(T[t]));
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        mn = min(mn, (unsigned)__shfl_down((int)mn, o, 64));
        mx = max(mx, (unsigned)__shfl_down((int)mx, o, 64));
    }
    if ((threadIdx.x & 63) == 0) {
        sh[0][threadIdx.x >> 6] = mn;
        sh[1][threadIdx.x >> 6] = mx;
    }
    __syncthreads();
    if (threadIdx.x) return;
    for (int w = 1; w < TPB / 64; w++) {
        mn = min(mn, sh[0][w]);
        mx = max(mx, sh[1][w]);
    }
    if (mn < __hip_atomic_load(&minmax[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMin(&minmax[0], mn);
    if (mx > __hip_atomic_load(&minmax[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(&minmax[1], mx);
}

__global__ void k_minmax_init(unsigned *minmax) {
    minmax[0] = ford(1.0e8f);
    minmax[1] = ford(-10.0f);
}

void timestep_tmax(hipStream_t s, chip_ctx *c, const float *V, const float *T) {
    const Level &L = c->L[c->levmax];
    hipLaunchKernelGGL(k_minmax_init, dim3(1), dim3(1), 0, s, c->minmax);
    const int nb = std::min(nblk(std::max(L.g.nel, L.g.nno)), 1024);
    if (L.brick)
        hipLaunchKernelGGL(k_timestep_tmax, dim3(nb), dim3(TPB), 0, s, L.g, L.GB + (size_t)BRICK_SIZE * L.g.nel, 1,
                           (long)L.g.nel, V, T, c->minmax);
    else
        hipLaunchKernelGGL(k_timestep_tmax, dim3(nb), dim3(TPB), 0, s, L.g, L.ECO + 5, ECO_SZ, 1L, V, T, c->minmax);
}

void tmax(hipStream_t s, chip_ctx *c, const float *T) { timestep_tmax(s, c, nullptr, T); }

// predictor (Advection_diffusion.c:352-366)
__global__ void k_predictor(Geo g, const unsigned *__restrict__ NODE, float *T, float *Tdot, float mult) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= g.nno) return;
    if (!(NODE[n] & (TBX | TBZ | TBY))) T[n] += mult * Tdot[n];
    Tdot[n] = 0.0f;
}

void predictor(hipStream_t s, const Level &L, float *T, float *Tdot, float mult) {
    hipLaunchKernelGGL(k_predictor, dim3(nblk(L.g.nno)), dim3(TPB), 0, s, L.g, L.NODE, T, Tdot, mult);
}

// pg_shape_fn + element_residual (Advection_diffusion.c:448-727, CART3D,
// diffusion on, no FBZ flux nodes): Eres[a][e] for the 8 nodes of element e
// (elements side by side, for this store and the gather's reads).  Bound by
// FP64 arithmetic with the compact geometry; by the arrays' reads without it
// (128x128x64 elements 105 us, from the arrays, every entry a cache line per
// lane, 713).
template <bool BRICK>
__global__ void __launch_bounds__(TPB, 3) k_pg_residual(Geo g, const float *__restrict__ GB, const float *__restrict__ GNX,
                                                     const float *__restrict__ GDA, const float *__restrict__ ECO,
                                                     const unsigned *__restrict__ NODE,
                                                     const float *__restrict__ diffusivity, double Q,
                                                     const float *__restrict__ T, const float *__restrict__ Tdot,
                                                     const float *__restrict__ V, double *__restrict__ Eres) {
    const int el = blockIdx.x * blockDim.x + threadIdx.x;
    if (el >= g.nel) return;
    const int ez = el % g.elz, ex = (el / g.elz) % g.elx, ey = el / (g.elz * g.elx);
    const float diff = (float)((diffusivity[ez] + diffusivity[ez + 1]) * 0.5);
    ElemGeo<BRICK> eg(g, GB, GNX, GDA, ECO, el);
    int nodes[9];
    float v1n[9], v2n[9], v3n[9];
#pragma unroll
    for (int a = 1; a <= 8; a++) {
        nodes[a] = nid(g, ez + cOffz[a], ex + cOffx[a], ey + cOffy[a]);
        v1n[a] = V[nodes[a]];
        v2n[a] = V[g.nno + nodes[a]];
        v3n[a] = V[2 * g.nno + nodes[a]];
    }
    // pg_shape_fn
    double uc1 = 0.0, uc2 = 0.0, uc3 = 0.0;
#pragma unroll
    for (int a = 1; a <= 8; a++) {
        uc1 += cNp[a - 1] * v1n[a];
        uc2 += cNp[a - 1] * v2n[a];
        uc3 += cNp[a - 1] * v3n[a];
    }
    const double twodiff = 2.0 * diff;
    const double uxse = fabs(uc1 * (double)eg.len(0)), ueta = fabs(uc2 * (double)eg.len(1)), ufai = fabs(uc3 * (double)eg.len(2));
    const double xse = (uxse > twodiff) ? (1.0 - twodiff / uxse) : 0.0;
    const double eta = (ueta > twodiff) ? (1.0 - twodiff / ueta) : 0.0;
    const double fai = (ufai > twodiff) ? (1.0 - twodiff / ufai) : 0.0;
    const double unorm = uc1 * uc1 + uc2 * uc2 + uc3 * uc3;
    const double adiff = (unorm > 0.000001) ? ((uxse * xse + ueta * eta + ufai * fai) / (2.0 * unorm)) : 0.0;
    // element_residual, one Gauss point after the other
    float Tn[9], DT[9];
    double r[9];
#pragma unroll
    for (int j = 1; j <= 8; j++) {
        Tn[j] = T[nodes[j]];
        DT[j] = Tdot[nodes[j]];
        if (NODE[nodes[j]] & (TBX | TBY | TBZ)) DT[j] = 0.0f;
        r[j] = 0.0;
    }
#pragma unroll
    for (int i = 1; i <= 8; i++) {
        eg.hold();
        double dT = 0.0, tx1 = 0.0, tx2 = 0.0, tx3 = 0.0, v1 = 0.0, v2 = 0.0, v3 = 0.0;
#pragma unroll
        for (int j = 1; j <= 8; j++) asm volatile("" : "+v"(Tn[j]), "+v"(DT[j]), "+v"(v1n[j]), "+v"(v2n[j]), "+v"(v3n[j]));
#pragma unroll
        for (int j = 1; j <= 8; j++) {
            const double sfn = cNv[8 * (j - 1) + i - 1];
            dT += DT[j] * sfn;
            tx1 += eg.dN(0, j - 1, i - 1) * (double)Tn[j];
            tx2 += eg.dN(1, j - 1, i - 1) * (double)Tn[j];
            tx3 += eg.dN(2, j - 1, i - 1) * (double)Tn[j];
            v1 += v1n[j] * sfn;
            v2 += v2n[j] * sfn;
            v3 += v3n[j] * sfn;
        }
        const float w = eg.dA(i - 1), dl = diff * 1.0f * w;
        const double val = dT - Q + v1 * tx1 + v2 * tx2 + v3 * tx3;
#pragma unroll
        for (int j = 1; j <= 8; j++) {
            const float gx = eg.dN(0, j - 1, i - 1), gy = eg.dN(1, j - 1, i - 1), gz = eg.dN(2, j - 1, i - 1);
            const double prod1 = (v1 * gx + v2 * gy + v3 * gz);
            const double PG = cNv[8 * (j - 1) + i - 1] + adiff * prod1;
            r[j] -= PG * w * val + dl * (gx * tx1 + gy * tx2 + gz * tx3);
        }
        __builtin_amdgcn_sched_barrier(0);   // else the next points' values take the registers of four wavefronts
    }
#pragma unroll
    for (int j = 1; j <= 8; j++) Eres[(size_t)(j - 1) * g.nel + el] = r[j];
}

void pg_residual(hipStream_t s, const chip_ctx *c, const float *T, const float *Tdot, const float *V, double *Eres) {
    const Level &L = c->L[c->levmax];
    // heating_adi = heating_visc = 0 and heating_latent = 1 (Instructions.c:376-381)
    const double Q = (c->p.Q0 - 0.0f + 0.0f) * 1.0f;
    hipLaunchKernelGGL(L.brick ? k_pg_residual<true> : k_pg_residual<false>, dim3(nblk(L.g.nel)), dim3(TPB), 0, s, L.g,
                       L.GB, L.GNX, L.GDA, L.ECO, L.NODE, c->diffusivity, Q, T, Tdot, V, Eres);
}

// pg_solver's scatter and lumped-mass scaling (Advection_diffusion.c:423-437)
// fused with corrector (:369-387)
__global__ void __launch_bounds__(TPB) k_pg_gather(Geo g, const unsigned *__restrict__ NODE,
                                                   const float *__restrict__ MASS, const double *__restrict__ Eres,
                                                   float *T, float *Tdot, float mult) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= g.nno) return;
    int k, i, j;
    node_kij(g, n, k, i, j);
    float dt = 0.0f;
    for (int ey = j - 1; ey <= j; ey++) {
        if ((unsigned)ey >= (unsigned)g.ely) continue;
        for (int ex = i - 1; ex <= i; ex++) {
            if ((unsigned)ex >= (unsigned)g.elx) continue;
            for (int ez = k - 1; ez <= k; ez++) {
                if ((unsigned)ez >= (unsigned)g.elz) continue;
                const int e = ez + g.elz * (ex + g.elx * ey);
                const int a = cLoc[(k - ez) + 2 * (i - ex) + 4 * (j - ey)];
                dt = (float)(dt + Eres[(size_t)(a - 1) * g.nel + e]);
            }
        }
    }
    dt *= MASS[n];
    if (!(NODE[n] & (TBX | TBZ | TBY))) T[n] += mult * dt;
    Tdot[n] += dt;
}

void pg_gather_correct(hipStream_t s, const chip_ctx *c, const double *Eres, float *T, float *Tdot, float mult) {
    const Level &L = c->L[c->levmax];
    hipLaunchKernelGGL(k_pg_gather, dim3(nblk(L.g.nno)), dim3(TPB), 0, s, L.g, L.NODE, L.MASS, Eres, T, Tdot, mult);
}

// temperatures_conform_bcs (Boundary_conditions.c:949-990); the side walls
// carry zero-flux flags, so only TBZ nodes are set
__global__ void k_conform_T(Geo g, const unsigned *__restrict__ NODE, const float *__restrict__ TB, float *T) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= g.nno) return;
    if (NODE[n] & TBZ) T[n] = TB[n];
}

void conform_temperature(hipStream_t s, const chip_ctx *c, float *T) {
    const Level &L = c->L[c->levmax];
    hipLaunchKernelGGL(k_conform_T, dim3(nblk(L.g.nno)), dim3(TPB), 0, s, L.g, L.NODE, c->TB, T);
}

// thermal_buoyancy (Pan_problem_misc_functions.c:83-153) with remove_horiz_ave
// / return_horiz_ave (Global_operations.c:55-80, 133-251)
__global__ void k_buoy_raw(Geo g, float Ra, const float *__restrict__ expansivity, const float *__restrict__ T,
                           float *__restrict__ b) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= g.nno) return;
    b[n] = Ra * T[n] * expansivity[n % g.noz];
}

// horizontal averages of a nodal field, with the bilinear surface quadrature of
// get_global_1d_shape_fn gathered into one weight a column (its corners' shares
// of the faces around it).  A workgroup takes 64 columns, a thread one face's
// share of a weight and then a lane one node layer, so that a column is read
// as it lies; k_horiz_fin adds the workgroups' sums.  Bound by launches (16 us
// at 129x129x65 nodes; one workgroup a layer, a cache line per value, 64).
constexpr int HA_COLS = 64;

__global__ void __launch_bounds__(256) k_horiz_part(Geo g, const float *__restrict__ xc, const float *__restrict__ yc,
                                                    const float *__restrict__ X, double *__restrict__ part) {
    __shared__ double share[4][HA_COLS], sum[4][64];
    const int ncol = g.nox * g.noy, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    {
        const int q = blockIdx.x * HA_COLS + lane, i = q % g.nox, j = q / g.nox;
        const int ex = i - 1 + (w & 1), ey = j - 1 + (w >> 1);
        double t = 0.0;
        if (q < ncol && (unsigned)ex < (unsigned)g.elx && (unsigned)ey < (unsigned)g.ely) {
            const int d = i == ex ? (j == ey ? 1 : 4) : (j == ey ? 2 : 3);   // the column's corner of the face
            const double xx1[5] = {0, xc[ex], xc[ex + 1], xc[ex + 1], xc[ex]};
            const double xx2[5] = {0, yc[ey], yc[ey], yc[ey + 1], yc[ey + 1]};
#pragma unroll
            for (int nint = 1; nint <= 4; nint++) {
                double d11 = 0, d12 = 0, d21 = 0, d22 = 0;
#pragma unroll
                for (int ii = 1; ii <= 4; ii++) {
                    const double mx0 = cMxv[4 * (ii - 1) + nint - 1], mx1 = cMxv[16 + 4 * (ii - 1) + nint - 1];
                    d11 += xx1[ii] * mx0;
                    d12 += xx2[ii] * mx0;
                    d21 += xx1[ii] * mx1;
                    d22 += xx2[ii] * mx1;
                }
                t += cMv[4 * (d - 1) + nint - 1] * (d11 * d22 - d12 * d21);
            }
        }
        share[w][lane] = t;
    }
    __syncthreads();
    const int k = blockIdx.y * 64 + lane;
    const float *x = X + (size_t)blockIdx.x * HA_COLS * g.noz + k;
    double v = 0.0, wt = 0.0;
#pragma unroll 4
    for (int q = w; q < HA_COLS; q += 4) {
        const double c = share[0][q] + share[1][q] + share[2][q] + share[3][q];
        if (blockIdx.x * HA_COLS + q < ncol) {
            wt += c;
            if (k < g.noz) v += c * x[(size_t)q * g.noz];
        }
    }
    sum[w][lane] = v;
    __syncthreads();
    share[0][w] = wt;   // read above by all before the barrier
    __syncthreads();
    double *p = part + (size_t)blockIdx.x * (g.noz + 1);
    if (w == 0 && k < g.noz) p[k] = sum[0][lane] + sum[1][lane] + sum[2][lane] + sum[3][lane];
    if (threadIdx.x == 0 && blockIdx.y == 0) p[g.noz] = share[0][0] + share[0][1] + share[0][2] + share[0][3];
}

__global__ void __launch_bounds__(64) k_horiz_fin(Geo g, int nb, const double *__restrict__ part, float *__restrict__ H) {
    double v = 0.0, w = 0.0;
    for (int b = threadIdx.x; b < nb; b += 64) {
        v += part[(size_t)b * (g.noz + 1) + blockIdx.x];
        w += part[(size_t)b * (g.noz + 1) + g.noz];
    }
    v = wave_sum(v);
    w = wave_sum(w);
    if (threadIdx.x == 0 && w != 0.0) H[blockIdx.x] = (float)(v / w);
}

// part: noz + 1 doubles per 64 columns, of the element scratch
void horiz_ave(hipStream_t s, const chip_ctx *c, const float *X, float *H) {
    const Geo &g = c->L[c->levmax].g;
    const int nb = nblk((long)g.nox * g.noy, HA_COLS);
    hipLaunchKernelGGL(k_horiz_part, dim3(nb, nblk(g.noz, 64)), dim3(256), 0, s, g, c->xc_d, c->yc_d, X, c->Eres);
    hipLaunchKernelGGL(k_horiz_fin, dim3(g.noz), dim3(64), 0, s, g, nb, c->Eres, H);
}

// averages (Process_velocity.c:179-224): per-layer horizontal averages of
// T, of |V|^2 (square-rooted on the host) and of the nodal viscosity
// (visc_from_gint_to_nodes of the finest EVI); |V|^2 in FP32 as the
// reference forms it
__global__ void k_vsq(long nno, const float *__restrict__ V, float *__restrict__ out) {
    const long n = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= nno) return;
    const float a = V[n], b = V[nno + n], c = V[2 * nno + n];
    out[n] = a * a + b * b + c * c;
}

void averages(hipStream_t s, chip_ctx *c, float *Have /* [3 noz] */, float *scratch /* [nno] */) {
    Level &L = c->L[c->levmax];
    horiz_ave(s, c, c->T, Have);
    hipLaunchKernelGGL(k_vsq, dim3(nblk(L.g.nno)), dim3(TPB), 0, s, (long)L.g.nno, c->V, scratch);
    horiz_ave(s, c, scratch, Have + L.g.noz);
    hipLaunchKernelGGL(k_visc_to_nodes, dim3(nblk(L.g.nno)), dim3(TPB), 0, s, L.g, L.EVI, L.TWW, L.MASS, scratch);
    horiz_ave(s, c, scratch, Have + 2 * L.g.noz);
}

__global__ void k_sub_layer(Geo g, const float *__restrict__ H, float *b) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= g.nno) return;
    b[n] -= H[n % g.noz];
}

void thermal_buoyancy(hipStream_t s, const chip_ctx *c, const float *T, float *buoy) {
    const Level &L = c->L[c->levmax];
    hipLaunchKernelGGL(k_buoy_raw, dim3(nblk(L.g.nno)), dim3(TPB), 0, s, L.g, c->p.rayleigh, c->expansivity, T, buoy);
    horiz_ave(s, c, buoy, c->H);
    hipLaunchKernelGGL(k_sub_layer, dim3(nblk(L.g.nno)), dim3(TPB), 0, s, L.g, c->H, buoy);
}

// assemble_forces + get_elt_f (Element_calculations.c:74-125, 989-1121,
// CART3D, no imposed velocities): element z-forces, then a per-node gather
__global__ void __launch_bounds__(TPB) k_elt_f(Geo g, const float *__restrict__ GDA, const float *__restrict__ buoy,
                                               double *__restrict__ Ef) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= g.nel) return;
    const int ez = e % g.elz, ex = (e / g.elz) % g.elx, ey = e / (g.elz * g.elx);
    const float *gda = GDA + (size_t)e * GDA_SZ;
    double force[9], fg[9];
#pragma unroll
    for (int a = 1; a <= 8; a++) force[a] = buoy[nid(g, ez + cOffz[a], ex + cOffx[a], ey + cOffy[a])];
#pragma unroll
    for (int j = 1; j <= 8; j++) {
        double t = 0.0;
#pragma unroll
        for (int k = 1; k <= 8; k++) t += force[k] * cNv[8 * (k - 1) + j - 1];
        fg[j] = t;
    }
#pragma unroll
    for (int a = 1; a <= 8; a++) {
        double f = 0.0;
#pragma unroll
        for (int j = 1; j <= 8; j++) f += fg[j] * cNv[8 * (a - 1) + j - 1] * gda[j] * 1.0f;
        Ef[(size_t)(a - 1) * g.nel + e] = f;
    }
}

__global__ void __launch_bounds__(TPB) k_forces_gather(Geo g, const unsigned *__restrict__ NODE,
                                                       const double *__restrict__ Ef, double *__restrict__ F) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= g.nno) return;
    int k, i, j;
    node_kij(g, n, k, i, j);
    double acc = 0.0;
    for (int ey = j - 1; ey <= j; ey++) {
        if ((unsigned)ey >= (unsigned)g.ely) continue;
        for (int ex = i - 1; ex <= i; ex++) {
            if ((unsigned)ex >= (unsigned)g.elx) continue;
            for (int ez = k - 1; ez <= k; ez++) {
                if ((unsigned)ez >= (unsigned)g.elz) continue;
                const int e = ez + g.elz * (ex + g.elx * ey);
                acc += Ef[(size_t)(cLoc[(k - ez) + 2 * (i - ex) + 4 * (j - ey)] - 1) * g.nel + e];
            }
        }
    }
    const unsigned f = NODE[n];
    F[3 * n] = 0.0;
    F[3 * n + 1] = 0.0;
    F[3 * n + 2] = (f & VBZ) ? 0.0 : acc;
}

void assemble_forces(hipStream_t s, const chip_ctx *c, const float *buoy, double *F) {
    const Level &L = c->L[c->levmax];
    hipLaunchKernelGGL(k_elt_f, dim3(nblk(L.g.nel)), dim3(TPB), 0, s, L.g, L.GDA, buoy, c->Eres);
    hipLaunchKernelGGL(k_forces_gather, dim3(nblk(L.g.nno)), dim3(TPB), 0, s, L.g, L.NODE, c->Eres, F);
}

// heat_flux (Process_buoyancy.c:63-203).  The surface values extrapolate from
// the two node layers at each end of the columns, so only the element layers
// that these touch (two at each end, all where there are fewer than four) are
// integrated, only those nodes averaged (k_hf_columns: one thread a column and
// end) and the columns summed by one workgroup (k_hf_surface).  Bound by launches
// and latency: over the whole mesh 268 us at 128x128x64 elements, 140 of them one
// workgroup on strided columns; so 30.
template <bool BRICK>
__global__ void __launch_bounds__(TPB) k_hf_elem(Geo g, int nl, const float *__restrict__ GB,
                                                 const float *__restrict__ GNX, const float *__restrict__ GDA,
                                                 const float *__restrict__ ECO, const float *__restrict__ diffusivity,
                                                 const float *__restrict__ T, const float *__restrict__ V,
                                                 double *__restrict__ uTe) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nl * g.elx * g.ely) return;
    const int ec = t / nl, l = t - ec * nl;
    const int ez = l < 2 ? l : g.elz - nl + l, ex = ec % g.elx, ey = ec / g.elx;
    const int e = ez + g.elz * ec;
    const double diff = (diffusivity[ez] + diffusivity[ez + 1]) * 0.5;
    const ElemGeo<BRICK> eg(g, GB, GNX, GDA, ECO, e);
    double VZ[9];
    float Tn[9];
#pragma unroll
    for (int a = 1; a <= 8; a++) {
        const int n = nid(g, ez + cOffz[a], ex + cOffx[a], ey + cOffy[a]);
        VZ[a] = V[2 * g.nno + n];
        Tn[a] = T[n];
    }
    double uT = 0.0;
#pragma unroll
    for (int i = 1; i <= 8; i++) {
        double u = 0.0, Tg = 0.0, dTdz = 0.0;
#pragma unroll
        for (int j = 1; j <= 8; j++) {
            u += VZ[j] * cNv[8 * (j - 1) + i - 1];
            Tg += Tn[j] * cNv[8 * (j - 1) + i - 1];
            dTdz = dTdz + Tn[j] * eg.dN(2, j - 1, i - 1);
        }
        uT = uT + (u * Tg - diff * dTdz) * eg.dA(i - 1);
    }
    uTe[e] = uT / (BRICK ? GB[(size_t)BRICK_AREA * g.nel + e] : ECO[(size_t)e * ECO_SZ + 12]);
}

// Volume-RMS velocity (no counterpart in the reference): per element the Q1
// quadrature of v.v and of 1 with the reference's shape functions and
// Jacobian weights (Shape_function_dA), in FP64.
__global__ void __launch_bounds__(TPB) k_vrms_elem(Geo g, const float *__restrict__ GDA, const float *__restrict__ V,
                                                   double *__restrict__ num, double *__restrict__ den,
                                                   double *__restrict__ ones) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= g.nel) return;
    const int ez = e % g.elz, ex = (e / g.elz) % g.elx, ey = e / (g.elz * g.elx);
    const float *gda = GDA + (size_t)e * GDA_SZ;
    double Vn[3][9];
#pragma unroll
    for (int a = 1; a <= 8; a++) {
        const int n = nid(g, ez + cOffz[a], ex + cOffx[a], ey + cOffy[a]);
#pragma unroll
        for (int d = 0; d < 3; d++) Vn[d][a] = V[d * g.nno + n];
    }
    double vv = 0.0, vol = 0.0;
#pragma unroll
    for (int i = 1; i <= 8; i++) {
        double s2 = 0.0;
#pragma unroll
        for (int d = 0; d < 3; d++) {
            double u = 0.0;
#pragma unroll
            for (int j = 1; j <= 8; j++) u += Vn[d][j] * cNv[8 * (j - 1) + i - 1];
            s2 += u * u;
        }
        vv += s2 * gda[i];
        vol += gda[i];
    }
    num[e] = vv;
    den[e] = vol;
    ones[e] = 1.0;
}

void vrms(hipStream_t s, chip_ctx *c, const float *V, double *out2) {
    const Level &L = c->L[c->levmax];
    const long nel = L.g.nel;
    double *num = c->Eres, *den = c->Eres + nel, *one = c->Eres + 2 * nel;
    hipLaunchKernelGGL(k_vrms_elem, dim3(nblk(nel)), dim3(TPB), 0, s, L.g, L.GDA, V, num, den, one);
    dots(s, c, (int)nel, 2, (const double *)num, (const double *)one, (const double *)den, (const double *)one,
         nullptr, nullptr, nullptr, nullptr, out2);
}

// out: [2][ncol] surface values (bottom, top), then [2][nface] element areas
__global__ void __launch_bounds__(TPB) k_hf_columns(Geo g, const float *__restrict__ TWW, const float *__restrict__ MASS,
                                                    const float *__restrict__ ECO, const double *__restrict__ uTe,
                                                    float *__restrict__ out) {
    const int ncol = g.nox * g.noy, t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= 2 * ncol) return;
    const int top = t >= ncol, q = t - top * ncol, i = q % g.nox, j = q / g.nox;
    float hf[2];
#pragma unroll
    for (int l = 0; l < 2; l++) {   // the surface node, the next one inwards
        const int k = top ? g.noz - 1 - l : l;
        float acc = 0.0f;
        for (int ey = j - 1; ey <= j; ey++) {
            if ((unsigned)ey >= (unsigned)g.ely) continue;
            for (int ex = i - 1; ex <= i; ex++) {
                if ((unsigned)ex >= (unsigned)g.elx) continue;
                for (int ez = k - 1; ez <= k; ez++) {
                    if ((unsigned)ez >= (unsigned)g.elz) continue;
                    const int e = ez + g.elz * (ex + g.elx * ey);
                    const int a = cLoc[(k - ez) + 2 * (i - ex) + 4 * (j - ey)];
                    acc = (float)(acc + TWW[(size_t)e * TWW_SZ + a] * uTe[e]);
                }
            }
        }
        hf[l] = acc * MASS[nid(g, k, i, j)];
    }
    out[t] = 2 * hf[0] - hf[1];
    if (i < g.elx && j < g.ely) {
        const int f = i + g.elx * j, nface = g.elx * g.ely;
        out[2 * ncol + top * nface + f] = ECO[(size_t)(g.elz * f + (top ? g.elz - 1 : 0)) * ECO_SZ + 12];
    }
}

// surface-element sums (Process_buoyancy.c:158-193)
__global__ void __launch_bounds__(1024) k_hf_surface(Geo g, const float *__restrict__ col, double *__restrict__ out) {
    __shared__ double sh[4 * 16];
    const int ncol = g.nox * g.noy, nface = g.elx * g.ely;
    const float *area = col + 2 * ncol;
    double v[4] = {0, 0, 0, 0};
    for (int f = threadIdx.x; f < nface; f += blockDim.x) {
        const int ex = f % g.elx, ey = f / g.elx;
        const int cols[4] = {ex + g.nox * ey, ex + 1 + g.nox * ey, ex + 1 + g.nox * (ey + 1), ex + g.nox * (ey + 1)};
        double tb = 0.0, tt = 0.0;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            tb += col[cols[q]];
            tt += col[ncol + cols[q]];
        }
        const float ab = area[f], at = area[nface + f];
        v[0] += tb * ab;
        v[1] += ab;
        v[2] += tt * at;
        v[3] += at;
    }
    block_sum<4>(v, sh);
    if (threadIdx.x == 0)
        for (int m = 0; m < 4; m++) out[m] = v[m];
}

void heat_flux(hipStream_t s, chip_ctx *c, const float *T, const float *V) {
    const Level &L = c->L[c->levmax];
    const Geo &g = L.g;
    const int nl = std::min(g.elz, 4);
    float *col = reinterpret_cast<float *>(c->Eres + g.nel);   // at most 6.5 values a face, of the scratch's 14 an element
    hipLaunchKernelGGL(L.brick ? k_hf_elem<true> : k_hf_elem<false>, dim3(nblk((long)nl * g.elx * g.ely)), dim3(TPB), 0, s,
                       g, nl, L.GB, L.GNX, L.GDA, L.ECO, c->diffusivity, T, V, c->Eres);
    hipLaunchKernelGGL(k_hf_columns, dim3(nblk(2L * g.nox * g.noy)), dim3(TPB), 0, s, g, L.TWW, L.MASS, L.ECO, c->Eres,
                       col);
    hipLaunchKernelGGL(k_hf_surface, dim3(1), dim3(1024), 0, s, g, col, c->dots + 24);
}

// ---------------------------------------------------------------------------
// Learned coarse-level correction (no reference counterpart).  The coarsest
// level's smoother call of multi_grid (General_matrix_functions.c:574, :613)
// is replaced by a small 3-D CNN (trained by the BF16 MFMA kernels of
// learn_kernels.hip): inputs F / rms(F) (three channels) and log10
// viscosity, output the correction / rms(F).  The inner solve still
// iterates to its own residual criterion.

// one workgroup of CNET_TPB threads runs the whole correction; its two
// activation buffers ([nv][16] bf16 each) take 64 nv bytes of LDS
constexpr int CNET_TPB = 512;
constexpr int CNET_MAX_NV = 1024;
typedef short bf16x4_t __attribute__((ext_vector_type(4)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

__global__ void __launch_bounds__(TPB) k_cnet_logeta(Geo g, const float *__restrict__ EVI, float *__restrict__ out) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= g.nno) return;
    const int k = n % g.noz, i = (n / g.noz) % g.nox, j = n / (g.noz * g.nox);
    float acc = 0.f;
    int cnt = 0;
    for (int dj = -1; dj <= 0; dj++)
        for (int di = -1; di <= 0; di++)
            for (int dk = -1; dk <= 0; dk++) {
                const int ez = k + dk, ex = i + di, ey = j + dj;
                if (ez < 0 || ex < 0 || ey < 0 || ez >= g.elz || ex >= g.elx || ey >= g.ely) continue;
                const size_t e = (size_t)ez + (size_t)g.elz * (ex + (size_t)g.elx * ey);
                float m = 0.f;
                for (int q = 0; q < 8; q++) m += log10f(EVI[e * 8 + q]);
                acc += 0.125f * m;
                cnt++;
            }
    out[n] = acc / (float)cnt;
}

void cnet_logeta(hipStream_t s, const Level &L, float *out) {
    hipLaunchKernelGGL(k_cnet_logeta, dim3(nblk(L.g.nno)), dim3(TPB), 0, s, L.g, (const float *)L.EVI, out);
}

// round to the nearest bf16, ties to even (finite values)
__device__ __forceinline__ uint16_t bf16_rne(float f) {
    const unsigned u = __float_as_uint(f);
    return (uint16_t)((u + 0x7FFFu + ((u >> 16) & 1u)) >> 16);
}


__device__ __forceinline__ bf16x4_t cnet_load4(const uint16_t *p) {
    const uint2 r = *reinterpret_cast<const uint2 *>(p);
    bf16x4_t a;
    a[0] = (short)(r.x & 0xFFFF);
    a[1] = (short)(r.x >> 16);
    a[2] = (short)(r.y & 0xFFFF);
    a[3] = (short)(r.y >> 16);
    return a;
}

// The whole correction in one workgroup: rms(F) and the input (F / rms,
// log10 eta) into LDS, the layers with activations in LDS (the products,
// operand layout and rounding of k_conv_fwd in learn_kernels.hip: one
// 16x16x16 bf16 MFMA per tap, FP32 accumulation, bias, ReLU, bf16), the
// last layer's three output channels times out_scale times rms into d,
// BC rows zero.
template <typename V>
__global__ void __launch_bounds__(CNET_TPB) k_cnet(Geo g, const V *__restrict__ F, const float *__restrict__ logeta,
                                                   const uint16_t *__restrict__ W, const float *__restrict__ bias,
                                                   int layers, const float *__restrict__ ys,
                                                   const unsigned *__restrict__ NODE, V *__restrict__ d) {
    extern __shared__ __align__(16) uint16_t act[];   // [2][nv][16]
    __shared__ double sh[16];
    __shared__ double sc_sh[2];
    const int nv = g.nno, l = threadIdx.x & 63, wv = threadIdx.x >> 6, nw = blockDim.x >> 6;
    double v[1] = {0.0};
    for (int i = threadIdx.x; i < 3 * nv; i += blockDim.x) v[0] += (double)F[i] * (double)F[i];
    block_sum<1>(v, sh);
    if (threadIdx.x == 0) {
        const double rms = sqrt(v[0] / (3.0 * nv));
        sc_sh[0] = rms;
        sc_sh[1] = rms > 0.0 ? 1.0 / rms : 0.0;
    }
    __syncthreads();
    const double rms = sc_sh[0], inv = sc_sh[1];
    for (int idx = threadIdx.x; idx < nv * 16; idx += blockDim.x) {
        const int n = idx >> 4, ch = idx & 15;
        float x = 0.f;
        if (ch < 3)
            x = (float)((double)F[3 * n + ch] * inv);
        else if (ch == 3)
            x = logeta[n];
        act[idx] = bf16_rne(x);
    }
    __syncthreads();
    const int o = l & 15, kq = 4 * (l >> 4);
    for (int li = 0; li < layers; li++) {
        const uint16_t *X = act + (size_t)(li & 1) * nv * 16;
        uint16_t *Y = act + (size_t)((li + 1) & 1) * nv * 16;
        const uint16_t *Wl = W + (size_t)li * 16 * 27 * 16;
        const float bo = bias[li * 16 + o];
        const bool last = li == layers - 1;
        for (int v0 = wv * 16; v0 < nv; v0 += nw * 16) {   // uniform per wavefront
            const int m = v0 + (l & 15);
            const bool in = m < nv;
            const int k = m % g.noz, i = (m / g.noz) % g.nox, j = m / (g.noz * g.nox);
            f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int t = 0; t < 27; t++) {   // tap t = (dz+1) + 3(dx+1) + 9(dy+1)
                const int dz = t % 3 - 1, dx = (t / 3) % 3 - 1, dy = t / 9 - 1;
                const bool ok = in && (unsigned)(k + dz) < (unsigned)g.noz && (unsigned)(i + dx) < (unsigned)g.nox &&
                                (unsigned)(j + dy) < (unsigned)g.noy;
                bf16x4_t a = {0, 0, 0, 0};
                if (ok) a = cnet_load4(X + (size_t)(m + dz + g.noz * (dx + g.nox * dy)) * 16 + kq);
                const bf16x4_t w = cnet_load4(Wl + ((size_t)o * 27 + t) * 16 + kq);
                acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, w, acc, 0, 0, 0);
            }
            for (int i = 0; i < 4; i++) {
                const int vv = v0 + kq + i;
                if (vv >= nv) continue;
                float y = acc[i] + bo;
                if (!last) {
                    Y[(size_t)vv * 16 + o] = bf16_rne(y > 0.f ? y : 0.f);
                } else if (o < 3) {
                    V out = (V)((double)y * (double)ys[o] * rms);
                    const unsigned f = NODE[vv];
                    if ((o == 0 && (f & VBX)) || (o == 1 && (f & VBY)) || (o == 2 && (f & VBZ))) out = V(0);
                    d[3 * vv + o] = out;
                }
            }
        }
        __syncthreads();
    }
}

bool cnet_fits(const Geo &g) { return g.nno <= CNET_MAX_NV; }

template <typename V>
int cnet_apply(hipStream_t s, const chip_ctx *c, const Level &L, const V *F, V *d) {
    if (!cnet_fits(L.g)) return -1;
    auto kern = k_cnet<V>;
    hipLaunchKernelGGL(kern, dim3(1), dim3(CNET_TPB), (size_t)2 * L.g.nno * 16 * sizeof(uint16_t), s, L.g, F,
                       (const float *)c->cnet_logeta, (const uint16_t *)c->cnet_w, (const float *)c->cnet_b,
                       c->cnet_layers, (const float *)c->cnet_ys, L.NODE, d);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}
template int cnet_apply<double>(hipStream_t, const chip_ctx *, const Level &, const double *, double *);
template int cnet_apply<float>(hipStream_t, const chip_ctx *, const Level &, const float *, float *);

}  // namespace chip

// ---------------------------------------------------------------------------
// the learned warm start's inputs and outputs on the finest level (no
// counterpart in the reference: the network's output is only the Uzawa
// solve's initial guess)

namespace chip {

__device__ __forceinline__ uint16_t warm_bf16(float f) {
    const unsigned u = __float_as_uint(f);
    return (uint16_t)((u + 0x7FFFu + ((u >> 16) & 1u)) >> 16);
}

// dT = T - (2 Th0 - Th1): the temperature's departure from its own linear
// extrapolation over the last two solves
__global__ void k_warm_dT(const float *__restrict__ T, const float *__restrict__ Th0, const float *__restrict__ Th1,
                          long n, float *__restrict__ dT) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dT[i] = T[i] - (2.0f * Th0[i] - Th1[i]);
}
void warm_dT(hipStream_t s, const float *T, const float *Th0, const float *Th1, long n, float *dT) {
    hipLaunchKernelGGL(k_warm_dT, dim3(nblk(n)), dim3(TPB), 0, s, T, Th0, Th1, n, dT);
}

// nodal value of an element field: the mean of (Pa - Pb) over the node's
// elements (Pb optional)
__global__ void k_e2n(Geo g, const double *__restrict__ Pa, const double *__restrict__ Pb, float *__restrict__ out) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= g.nno) return;
    const int k = n % g.noz, i = (n / g.noz) % g.nox, j = n / (g.noz * g.nox);
    double acc = 0.0;
    int cnt = 0;
    for (int dj = -1; dj <= 0; dj++)
        for (int di = -1; di <= 0; di++)
            for (int dk = -1; dk <= 0; dk++) {
                const int ez = k + dk, ex = i + di, ey = j + dj;
                if (ez < 0 || ex < 0 || ey < 0 || ez >= g.elz || ex >= g.elx || ey >= g.ely) continue;
                const size_t e = (size_t)ez + (size_t)g.elz * (ex + (size_t)g.elx * ey);
                acc += Pb ? Pa[e] - Pb[e] : Pa[e];
                cnt++;
            }
    out[n] = (float)(acc / cnt);
}
void e2n(hipStream_t s, const Level &L, const double *Pa, const double *Pb, float *out) {
    hipLaunchKernelGGL(k_e2n, dim3(nblk(L.g.nno)), dim3(TPB), 0, s, L.g, Pa, Pb, out);
}

// the network's input, 16 bf16 channels per node: T - 1/2, dT / s_dT,
// log10(eta) / 2.5, the extrapolated U / s_u (3) and nodal P / s_p, the
// last step's increments U - U_prev / s_u (3) and nodal P - P_prev / s_p,
// the second differences of U / s_2u (3) and of the nodal P / s_2p, z
// (node index over noz - 1).  U_prev here is the last solution.
__global__ void k_warm_features(Geo g, const float *__restrict__ T, const float *__restrict__ dT,
                                const float *__restrict__ logeta, const double *__restrict__ U,
                                const double *__restrict__ Uprev, const double *__restrict__ D2,
                                const float *__restrict__ pn, const float *__restrict__ dpn,
                                const float *__restrict__ d2pn, float inv_dT, float inv_u, float inv_p,
                                float inv_2u, float inv_2p, uint16_t *__restrict__ x) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= g.nno) return;
    float f[16];
    f[0] = T[n] - 0.5f;
    f[1] = dT[n] * inv_dT;
    f[2] = logeta[n] * 0.4f;
    for (int d = 0; d < 3; d++) {
        const size_t i = 3 * (size_t)n + d;
        f[3 + d] = (float)U[i] * inv_u;
        f[7 + d] = (float)(U[i] - Uprev[i]) * inv_u;
        f[11 + d] = (float)D2[i] * inv_2u;
    }
    f[6] = pn[n] * inv_p;
    f[10] = dpn[n] * inv_p;
    f[14] = d2pn[n] * inv_2p;
    f[15] = (float)(n % g.noz) / (float)(g.noz - 1);
    uint4 *o = reinterpret_cast<uint4 *>(x + (size_t)n * 16);
    for (int q = 0; q < 2; q++) {
        uint4 w;
        w.x = warm_bf16(f[8 * q + 0]) | ((uint32_t)warm_bf16(f[8 * q + 1]) << 16);
        w.y = warm_bf16(f[8 * q + 2]) | ((uint32_t)warm_bf16(f[8 * q + 3]) << 16);
        w.z = warm_bf16(f[8 * q + 4]) | ((uint32_t)warm_bf16(f[8 * q + 5]) << 16);
        w.w = warm_bf16(f[8 * q + 6]) | ((uint32_t)warm_bf16(f[8 * q + 7]) << 16);
        o[q] = w;
    }
}
void warm_features(hipStream_t s, const Level &L, const float *T, const float *dT, const float *logeta,
                   const double *U, const double *Uprev, const double *D2, const float *pn, const float *dpn,
                   const float *d2pn, float inv_dT, float inv_u, float inv_p, float inv_2u, float inv_2p,
                   uint16_t *x) {
    hipLaunchKernelGGL(k_warm_features, dim3(nblk(L.g.nno)), dim3(TPB), 0, s, L.g, T, dT, logeta, U, Uprev, D2, pn,
                       dpn, d2pn, inv_dT, inv_u, inv_p, inv_2u, inv_2p, x);
}

// the network's correction: U += s_eu out[n][0..2] at every node; P[e] +=
// s_ep (mean of out[.][3] over the element's eight nodes)
__global__ void k_warm_apply(Geo g, const float *__restrict__ out, double s_eu, double s_ep, double *__restrict__ U,
                             double *__restrict__ P) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < 3L * g.nno) U[i] += s_eu * (double)out[(i / 3) * 16 + i % 3];
    if (i < g.nel) {
        const int ez = (int)(i % g.elz), ex = (int)((i / g.elz) % g.elx), ey = (int)(i / ((long)g.elz * g.elx));
        double m = 0.0;
        for (int q = 0; q < 8; q++) {
            const int k = ez + (q & 1), ii = ex + ((q >> 1) & 1), j = ey + (q >> 2);
            m += (double)out[((size_t)k + (size_t)g.noz * (ii + (size_t)g.nox * j)) * 16 + 3];
        }
        P[i] += s_ep * 0.125 * m;
    }
}
void warm_apply(hipStream_t s, const Level &L, const float *out, double s_eu, double s_ep, double *U, double *P) {
    hipLaunchKernelGGL(k_warm_apply, dim3(nblk(3L * L.g.nno)), dim3(TPB), 0, s, L.g, out, s_eu, s_ep, U, P);
}

// the training target of one solve: (U - Ue) / s_eu per node (3 channels)
// and the nodal mean of (P - Pe) / s_ep, Ue, Pe the extrapolated guess
__global__ void k_warm_target(Geo g, const double *__restrict__ U, const double *__restrict__ Ue,
                              const float *__restrict__ dpn, double inv_eu, double inv_ep, float *__restrict__ y) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= g.nno) return;
    for (int d = 0; d < 3; d++) y[4 * (size_t)n + d] = (float)((U[3 * (size_t)n + d] - Ue[3 * (size_t)n + d]) * inv_eu);
    y[4 * (size_t)n + 3] = (float)(dpn[n] * inv_ep);
}
void warm_target(hipStream_t s, const Level &L, const double *U, const double *Ue, const float *dpn, double inv_eu,
                 double inv_ep, float *y) {
    hipLaunchKernelGGL(k_warm_target, dim3(nblk(L.g.nno)), dim3(TPB), 0, s, L.g, U, Ue, dpn, inv_eu, inv_ep, y);
}

}  // namespace chip
