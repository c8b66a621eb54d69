// Learned offset proposal: a small 3D CNN that scores, per 32x8x8 filter
// tile, how much weight mass each search offset carries, trained on the GPU
// with these kernels.
//
// Network (per voxel, "same" zero padding, ReLU after every conv):
//   conv1 1->16 (3^3)  conv2..4 16->16 (3^3)  mean-pool per tile -> 16 features
//   head 16 -> N_s logits, softmax over the search offsets.
// Loss: cross-entropy of the softmax against the tile's measured weight-mass
// distribution over offsets (mass / total), averaged over tiles.
//
// Activations are channels-last BF16 with a one-voxel zero halo:
// act[((z+1)*(ny+2) + (y+1))*(nx+2) + (x+1)][16].  Convolutions 2..4 (forward
// and the gradient with respect to their input) are implicit GEMMs on
// v_mfma_f32_16x16x32_bf16 with FP32 accumulation: 16 consecutive voxels x
// 16 output channels, K = 27 taps x 16 channels in 14 chunks of two taps.
// Their weight gradients (a reduction over all voxels) run there too; the
// first layer (one input channel) runs on the vector ALUs in FP32.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <string>
#include <vector>

#include "inlm_kernels.hpp"
#include "inlm_learn.hpp"

namespace inlm {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int C = 16;      // channels
constexpr int NTAP = 27;
constexpr int PTX = 32, PTY = 8, PTZ = 8;  // proposal tile = filter tile

struct ActGeom {
    int nx, ny, nz;       // unpadded
    long sx, sy;          // padded strides in voxels: x 1, y (nx+2), z (nx+2)(ny+2)
    __device__ __host__ long vox(int x, int y, int z) const { return (long)(z + 1) * sy + (long)(y + 1) * sx + (x + 1); }
};

__device__ __host__ inline long tap_off(const ActGeom &g, int tap)
{
    const int dz = tap / 9 - 1, dy = (tap / 3) % 3 - 1, dx = tap % 3 - 1;
    return (long)dz * g.sy + (long)dy * g.sx + dx;
}

__device__ __forceinline__ float bf2f(__bf16 v) { return (float)v; }

// ---------------------------------------------------------------------------
// layer 1: input (FP32, padded with zero halo, one channel) -> 16 channels
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void conv1_fwd(const float *__restrict__ in, const float *__restrict__ w,
                                                 const float *__restrict__ b, __bf16 *__restrict__ out, ActGeom g)
{
    const long n = (long)g.nx * g.ny * g.nz;
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const int x = (int)(i % g.nx), y = (int)((i / g.nx) % g.ny), z = (int)(i / ((long)g.nx * g.ny));
    const long v = g.vox(x, y, z);
    float acc[C];
#pragma unroll
    for (int c = 0; c < C; c++) acc[c] = b[c];
    for (int t = 0; t < NTAP; t++) {
        const float xv = in[v + tap_off(g, t)];
#pragma unroll
        for (int c = 0; c < C; c++) acc[c] = __builtin_fmaf(w[t * C + c], xv, acc[c]);
    }
    __bf16 o[C];
#pragma unroll
    for (int c = 0; c < C; c++) o[c] = (__bf16)__builtin_fmaxf(acc[c], 0.f);
    __builtin_memcpy(out + v * C, o, sizeof o);
}

// ---------------------------------------------------------------------------
// 16 -> 16 channel 3^3 convolution on MFMA.  wk is [27 tap][16 n][16 k] BF16
// (n = output channel, k = input channel).  MODE 0: forward,
// out = relu(acc + bias).  MODE 1: input gradient, out = acc * (mask > 0)
// with mask the forward input activation of this layer.
//
// A 16x16x32 product takes 16 voxels of an x row and two taps of 16 channels:
// A is the taps' weights (row = output channel), B the voxels' input, so a
// lane ends with four consecutive channels of one voxel and a wave writes 512
// contiguous bytes.  The 14 weight operands stay in 56 registers over all
// tiles of a block (at most kConvBlocks, two per CU); the input comes from a
// 32x8x4 tile with its halo staged in LDS (2 voxels per output, 65 KB), where
// a 16-byte read at 32-byte voxel pitch hits 16 distinct bank groups in each
// 16-lane service group.  One wave per 16 voxels reading the input and the
// weights of every product from global memory took 1.22 ms a layer on a
// 256^3 volume, bound by the L1; this takes 0.43 ms forward (535 TFLOP/s)
// and 0.56 ms backward, where each row's mask is loaded one row ahead.
// ---------------------------------------------------------------------------
constexpr int kConvBlocks = 512;
constexpr int CTX = 32, CTY = 8, CTZ = 4;
constexpr int CRX = CTX + 2, CRY = CTY + 2, CRZ = CTZ + 2;
template <int MODE>
__global__ __launch_bounds__(256, 2) void conv16_mfma(const __bf16 *__restrict__ X, const __bf16 *__restrict__ wk,
                                                      const float *__restrict__ bias, const __bf16 *__restrict__ mask,
                                                      __bf16 *__restrict__ out, ActGeom g)
{
    constexpr int XCH = CRX * CRY * CRZ * 2, XPT = (XCH + 255) / 256;  // 16-byte chunks
    __shared__ __attribute__((aligned(16))) __bf16 xs[CRZ * CRY * CRX * C + 8];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int m = lane & 15, q = lane >> 4, k0 = 8 * (q & 1);
    // the tap past the last: zero weights on a zero input (on a voxel of the
    // tile they would make a NaN of an infinite activation)
    __bf16 *const none = xs + CRZ * CRY * CRX * C;
    if (t < 8) none[t] = (__bf16)0.f;
    const int ntx = (g.nx + CTX - 1) / CTX, nty = (g.ny + CTY - 1) / CTY, ntz = (g.nz + CTZ - 1) / CTZ;
    const long tiles = (long)ntx * nty * ntz;
    const long t0 = tiles * blockIdx.x / gridDim.x, t1 = tiles * (blockIdx.x + 1) / gridDim.x;
    const long last = g.vox(g.nx, g.ny, g.nz);  // the last voxel of the padded volume

    bf16x8 w[14];
    int xoff[14];  // LDS offset of this lane's tap and channels
#pragma unroll
    for (int c = 0; c < 14; c++) {
        const int tap = 2 * c + (q >> 1);
        if (tap < NTAP) __builtin_memcpy(&w[c], wk + ((long)tap * C + m) * C + k0, 16);
        else
#pragma unroll
            for (int e = 0; e < 8; e++) w[c][e] = (__bf16)0.f;
        const int tp = tap < NTAP ? tap : NTAP - 1;
        xoff[c] = ((tp / 9) * CRY * CRX + (tp / 3 % 3) * CRX + tp % 3 + m) * C + k0;
    }
    float bs[4] = {0.f, 0.f, 0.f, 0.f};
    if constexpr (MODE == 0)
#pragma unroll
        for (int i = 0; i < 4; i++) bs[i] = bias[4 * q + i];

    for (long tile = t0; tile < t1; tile++) {
        const int x0 = (int)(tile % ntx) * CTX, y0 = (int)(tile / ntx % nty) * CTY, z0 = (int)(tile / ((long)ntx * nty)) * CTZ;
        // region voxel (rx, ry, rz) is the padded voxel (x0 + rx, y0 + ry, z0 + rz); those past the padded
        // volume feed only outputs that are dropped and read some voxel inside it
        const long origin = (long)z0 * g.sy + (long)y0 * g.sx + x0;
        __bf16 mk[2][4], mn[2][4];
        auto load_mask = [&](int r) __attribute__((always_inline)) {
            const int y = y0 + r % CTY, z = z0 + r / CTY;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int x = x0 + 16 * h + m;
                if (x < g.nx && y < g.ny && z < g.nz) __builtin_memcpy(mn[h], mask + g.vox(x, y, z) * C + 4 * q, 8);
            }
        };
        if constexpr (MODE == 1) load_mask(wave);
        __syncthreads();  // the tile before this one has been read
#pragma unroll
        for (int i = 0; i < XPT; i++) {
            const int ch = t + i * 256, v = ch >> 1;
            if (XCH % 256 == 0 || ch < XCH) {
                const int rx = v % CRX, ry = v / CRX % CRY, rz = v / (CRX * CRY);
                const long at = origin + (long)rz * g.sy + (long)ry * g.sx + rx;
                *reinterpret_cast<uint4 *>(xs + 8 * ch) =
                    *reinterpret_cast<const uint4 *>(X + (at < last ? at : last) * C + 8 * (ch & 1));
            }
        }
        __syncthreads();
#pragma unroll 1
        for (int r = wave; r < CTY * CTZ; r += 4) {
            const int ry = r % CTY, rz = r / CTY, y = y0 + ry, z = z0 + rz;
            const __bf16 *xrow = xs + (rz * CRY + ry) * CRX * C;
            const bool row = y < g.ny && z < g.nz;
            if constexpr (MODE == 1) {  // this row's mask has landed under the products before it
#pragma unroll
                for (int h = 0; h < 2; h++)
#pragma unroll
                    for (int i = 0; i < 4; i++) mk[h][i] = mn[h][i];
                if (r + 4 < CTY * CTZ) load_mask(r + 4);
            }
            floatx4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
            for (int c = 0; c < 14; c++)
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    bf16x8 b;
                    const __bf16 *p = xrow + xoff[c] + h * 16 * C;
                    if (c == 13 && q >= 2) p = none;
                    __builtin_memcpy(&b, __builtin_assume_aligned(p, 16), 16);
                    acc[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[c], b, acc[h], 0, 0, 0);
                }
            if (!row) continue;
            // C[row 4q+i][col m]: channel 4q + i of voxel x0 + 16 h + m
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int x = x0 + 16 * h + m;
                if (x >= g.nx) continue;
                const long v = g.vox(x, y, z) * C + 4 * q;
                __bf16 o[4];
                if constexpr (MODE == 0) {
#pragma unroll
                    for (int i = 0; i < 4; i++) o[i] = (__bf16)__builtin_fmaxf(acc[h][i] + bs[i], 0.f);
                } else {
#pragma unroll
                    for (int i = 0; i < 4; i++) o[i] = (__bf16)(bf2f(mk[h][i]) > 0.f ? acc[h][i] : 0.f);
                }
                __builtin_memcpy(out + v, o, 8);
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Weight gradients: dW[tap][k][n] = sum_v X[v + tap][k] * G[v][n] and
// dB[n] = sum_v G[v][n].  Each of at most kWgradBlocks blocks writes its
// partial sums (part[block][tap][k][n], then part[block][NTAP CIN C + n] for
// the bias) and wgrad_reduce adds them in a fixed order, so training repeats
// bit for bit.
// ---------------------------------------------------------------------------
constexpr int kWgradBlocks = 512;               // two per CU
constexpr int kWgradStride = NTAP * C * C + C;  // floats per block's partials
constexpr int kHeadShares = 64;                 // partials of the head's gradient
static_assert(kHeadShares * (C + 1) * (long)kMaxProposalOffsets <= (long)kWgradBlocks * kWgradStride,
              "the head's partials fit the same buffer");

// 16 -> 16 channels on v_mfma_f32_16x16x32_bf16: per tap a 16x16 product
// whose K dimension runs over 32 voxels of an x row, A[k][v] = X[v + tap][k]
// and B[v][n] = G[v][n], summed in FP32.  A wave keeps the 27 products and
// the bias (A = 1) in registers over all rows it visits.  Both operands need
// eight voxels of one channel per lane, the transpose of the channels-last
// layout: ds_read_b64_tr_b16 reads four voxels of 16 channels per 16 lanes
// that way, so a shift in x is a shift of 32 bytes and every read of a wave
// covers 512 contiguous bytes.  (The order of the 32 voxels within K is free:
// lane group q holds voxels 4q..4q+3 and 16+4q..16+4q+3 in both operands.)
//
// A block stages X over a 32x4x4 tile and its halo (2.4 voxels per output,
// 39 KB) and G (16 KB) per tile, two blocks per CU.  The form before it, one
// thread per (k, n) pair with 27 shifted copies of X in LDS, read one LDS
// dword per multiply-add and one block filled a CU's LDS: 37.7 ms a layer on
// a 256^3 volume against 0.37 ms (630 TFLOP/s), which the tiles' loads
// through L2 (1.8 GB) and the LDS reads (56 per 28 MFMAs) bound together.
constexpr int WTX = 32, WTY = 4, WTZ = 4;
constexpr int WRX = WTX + 2, WRY = WTY + 2, WRZ = WTZ + 2;
typedef short short4v __attribute__((ext_vector_type(4)));

// eight voxels of this lane's channel: p is the LDS address of the first of
// 32 voxels of a row, the lane's share of it included
__device__ __forceinline__ bf16x8 read_voxels(const __bf16 *p)
{
    typedef __attribute__((address_space(3))) short4v lds4;
    const short4v a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4 *)p);
    const short4v b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4 *)(p + 16 * C));
    bf16x8 r;
    __builtin_memcpy(&r, &a, 8);
    __builtin_memcpy(reinterpret_cast<char *>(&r) + 8, &b, 8);
    return r;
}

__global__ __launch_bounds__(256, 2) void conv16_wgrad(const __bf16 *__restrict__ X, const __bf16 *__restrict__ G,
                                                       float *__restrict__ part, ActGeom g)
{
    constexpr int XCH = WRX * WRY * WRZ * 2, GCH = WTX * WTY * WTZ * 2;  // 16-byte chunks
    constexpr int XPT = (XCH + 255) / 256, GPT = GCH / 256;
    static_assert(GCH % 256 == 0 && WTY * WTZ % 4 == 0, "whole chunks and rows per thread and wave");
    __shared__ __attribute__((aligned(16))) __bf16 xs[WRZ * WRY * WRX * C];
    __shared__ __attribute__((aligned(16))) __bf16 gs[WTZ * WTY * WTX * C];
    static_assert(sizeof(xs) >= NTAP * C * C * sizeof(float), "the block's sums reuse the X tile");
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int ntx = (g.nx + WTX - 1) / WTX, nty = (g.ny + WTY - 1) / WTY, ntz = (g.nz + WTZ - 1) / WTZ;
    const long tiles = (long)ntx * nty * ntz;
    const long t0 = tiles * blockIdx.x / gridDim.x, t1 = tiles * (blockIdx.x + 1) / gridDim.x;

    floatx4 acc[NTAP], accb = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < NTAP; i++) acc[i] = floatx4{0.f, 0.f, 0.f, 0.f};
    bf16x8 ones;
#pragma unroll
    for (int e = 0; e < 8; e++) ones[e] = (__bf16)1.f;
    // this lane's share of a 32-voxel read: voxel 4 q + (lane % 16) / 4, channels 4 (lane % 4) ..
    const int share = (4 * (lane >> 4) + ((lane & 15) >> 2)) * C + 4 * (lane & 3);

    for (long tile = t0; tile < t1; tile++) {
        const int x0 = (int)(tile % ntx) * WTX, y0 = (int)(tile / ntx % nty) * WTY, z0 = (int)(tile / ((long)ntx * nty)) * WTZ;
        // region voxel (rx, ry, rz) is the padded voxel (x0 + rx, y0 + ry, z0 + rz); past the padded volume it is zero
        const __bf16 *xo = X + ((long)z0 * g.sy + (long)y0 * g.sx + x0) * C;
        const __bf16 *go = G + g.vox(x0, y0, z0) * C;
        uint4 xr[XPT], gr[GPT];
#pragma unroll
        for (int i = 0; i < XPT; i++) {
            const int ch = t + i * 256, v = ch >> 1;
            const int rx = v % WRX, ry = v / WRX % WRY, rz = v / (WRX * WRY);
            xr[i] = uint4{0, 0, 0, 0};
            if (ch < XCH && x0 + rx < g.nx + 2 && y0 + ry < g.ny + 2 && z0 + rz < g.nz + 2)
                xr[i] = *reinterpret_cast<const uint4 *>(xo + ((long)rz * g.sy + (long)ry * g.sx + rx) * C + 8 * (ch & 1));
        }
#pragma unroll
        for (int i = 0; i < GPT; i++) {
            const int ch = t + i * 256, v = ch >> 1;
            const int rx = v % WTX, ry = v / WTX % WTY, rz = v / (WTX * WTY);
            gr[i] = uint4{0, 0, 0, 0};
            if (x0 + rx < g.nx && y0 + ry < g.ny && z0 + rz < g.nz)
                gr[i] = *reinterpret_cast<const uint4 *>(go + ((long)rz * g.sy + (long)ry * g.sx + rx) * C + 8 * (ch & 1));
        }
        __syncthreads();  // the tile before this one has been read
#pragma unroll
        for (int i = 0; i < XPT; i++)
            if (t + i * 256 < XCH) *reinterpret_cast<uint4 *>(xs + 8 * (t + i * 256)) = xr[i];
#pragma unroll
        for (int i = 0; i < GPT; i++) *reinterpret_cast<uint4 *>(gs + 8 * (t + i * 256)) = gr[i];
        __syncthreads();
        for (int r = wave; r < WTY * WTZ; r += 4) {
            const int ry = r % WTY, rz = r / WTY;
            const bf16x8 b = read_voxels(gs + r * WTX * C + share);
            accb = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, b, accb, 0, 0, 0);
            const __bf16 *xrow = xs + ((rz * WRY + ry) * WRX) * C + share;
#pragma unroll
            for (int tap = 0; tap < NTAP; tap++) {
                const bf16x8 a = read_voxels(xrow + ((tap / 9) * WRY * WRX + (tap / 3 % 3) * WRX + tap % 3) * C);
                acc[tap] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc[tap], 0, 0, 0);
            }
        }
    }
    // the block's sums, wave after wave: lane l holds rows k = 4 (l / 16) + i of column n = l % 16
    float *sum = reinterpret_cast<float *>(xs), *sumb = reinterpret_cast<float *>(gs);
    const int n = lane & 15, q = lane >> 4;
    for (int w = 0; w < 4; w++) {
        __syncthreads();
        if (wave == w) {
#pragma unroll
            for (int tap = 0; tap < NTAP; tap++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    float *d = sum + (tap * C + 4 * q + i) * C + n;
                    *d = w == 0 ? acc[tap][i] : *d + acc[tap][i];
                }
            if (q == 0) sumb[n] = w == 0 ? accb[0] : sumb[n] + accb[0];
        }
    }
    __syncthreads();
    float *pb = part + (long)blockIdx.x * kWgradStride;
    for (int i = t; i < NTAP * C * C; i += 256) pb[i] = sum[i];
    if (t < C) pb[NTAP * C * C + t] = sumb[t];
}

// The first layer (one FP32 input channel): dW[tap][n] = sum_v X[v + tap] G[v][n]
// in FP32.  A wave takes 64 voxels of a row, one a lane, and one dz: nine X
// values and 16 G values a lane feed 144 multiply-adds into registers, so the
// vector ALUs bound it (14.5 GFLOP on a 256^3 volume: 0.18 ms at their rate);
// the loads of the next 64 voxels are in flight meanwhile, two waves a SIMD.
// A thread per channel with X in LDS read one dword per multiply-add and used
// 16 of 256 threads: 4.2 ms with 2048 blocks there, 0.89 ms here.
__global__ __launch_bounds__(192, 2) void conv1_wgrad(const float *__restrict__ X, const __bf16 *__restrict__ G,
                                                      float *__restrict__ part, ActGeom g)
{
    const int lane = threadIdx.x & 63, dz = (threadIdx.x >> 6) - 1;
    const int nxc = (g.nx + 63) / 64;
    const long units = (long)nxc * g.ny * g.nz;
    const long u0 = units * blockIdx.x / gridDim.x, u1 = units * (blockIdx.x + 1) / gridDim.x;
    int xc = (int)(u0 % nxc), y = (int)(u0 / nxc % g.ny), z = (int)(u0 / ((long)nxc * g.ny));
    float acc[9][C], accb[C];
#pragma unroll
    for (int i = 0; i < 9; i++)
#pragma unroll
        for (int c = 0; c < C; c++) acc[i][c] = 0.f;
#pragma unroll
    for (int c = 0; c < C; c++) accb[c] = 0.f;
    float xv[9];
    uint4 gr[2];
    // lanes past the row read its last voxel against a zero gradient
    auto load = [&](float (&xo)[9], uint4 (&go)[2]) __attribute__((always_inline)) {
        const int x = xc * 64 + lane;
        const long v = g.vox(x < g.nx ? x : g.nx - 1, y, z);
        const float *p = X + v + (long)dz * g.sy;
#pragma unroll
        for (int i = 0; i < 9; i++) xo[i] = p[(i / 3 - 1) * g.sx + i % 3 - 1];
        const uint4 *q = reinterpret_cast<const uint4 *>(G + v * C);
        const uint4 zero = {0, 0, 0, 0};
        go[0] = x < g.nx ? q[0] : zero;
        go[1] = x < g.nx ? q[1] : zero;
    };
    if (u0 < u1) load(xv, gr);
    for (long u = u0; u < u1; u++) {
        if (++xc == nxc) {
            xc = 0;
            if (++y == g.ny) {
                y = 0;
                z++;
            }
        }
        float xn[9];
        uint4 gn[2];
        if (u + 1 < u1) load(xn, gn);
        unsigned w[8];
        __builtin_memcpy(w, gr, sizeof w);
        float gv[C];
#pragma unroll
        for (int c = 0; c < C; c++)
            gv[c] = __builtin_bit_cast(float, (c & 1) != 0 ? w[c >> 1] & 0xffff0000u : w[c >> 1] << 16);
#pragma unroll
        for (int i = 0; i < 9; i++)
#pragma unroll
            for (int c = 0; c < C; c++) acc[i][c] = __builtin_fmaf(xv[i], gv[c], acc[i][c]);
        if (dz == 0)
#pragma unroll
            for (int c = 0; c < C; c++) accb[c] += gv[c];
#pragma unroll
        for (int i = 0; i < 9; i++) xv[i] = xn[i];
        gr[0] = gn[0];
        gr[1] = gn[1];
    }
    auto wave_total = [](float v) __attribute__((always_inline)) {
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
        return v;
    };
    float *pb = part + (long)blockIdx.x * kWgradStride;
#pragma unroll
    for (int i = 0; i < 9; i++)
#pragma unroll
        for (int c = 0; c < C; c++) {
            const float s = wave_total(acc[i][c]);
            if (lane == 0) pb[((dz + 1) * 9 + i) * C + c] = s;
        }
    if (dz == 0)
#pragma unroll
        for (int c = 0; c < C; c++) {
            const float s = wave_total(accb[c]);
            if (lane == 0) pb[NTAP * C + c] = s;
        }
}

// out[e] = sum over blocks of part[block][e], e < n, blocks `stride` floats
// apart (weights and biases lie side by side in both).  Four threads share an
// element (blocks b, b + 4, ...), 64 consecutive elements a block, so a
// block's reads are 256 contiguous bytes and the chain of one thread is a
// quarter of the partials: 0.68 -> 0.01 ms for 512 partials of a 16 -> 16
// layer.
__global__ __launch_bounds__(256) void wgrad_reduce(const float *__restrict__ part, long stride, int nblocks, int n,
                                                    float *__restrict__ out)
{
    __shared__ float sh[4][64];
    const int e = blockIdx.x * 64 + (threadIdx.x & 63), w = threadIdx.x >> 6;
    float s = 0.f;
    if (e < n) {
#pragma unroll 8
        for (int b = w; b < nblocks; b += 4) s += part[(long)b * stride + e];
    }
    sh[w][threadIdx.x & 63] = s;
    __syncthreads();
    if (w == 0 && e < n) out[e] = (sh[0][e & 63] + sh[1][e & 63]) + (sh[2][e & 63] + sh[3][e & 63]);
}

// ---------------------------------------------------------------------------
// Mean pool per 32x8x8 tile (tiles x-fastest, partial tiles at the edges).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void pool_fwd(const __bf16 *__restrict__ A, float *__restrict__ feat, ActGeom g,
                                                int ntx, int nty)
{
    const int t = blockIdx.x;
    const int bx = t % ntx, by = (t / ntx) % nty, bz = t / (ntx * nty);
    __shared__ float part[256][C + 1];
    float s[C];
#pragma unroll
    for (int c = 0; c < C; c++) s[c] = 0.f;
    for (int i = threadIdx.x; i < PTX * PTY * PTZ; i += 256) {
        const int x = bx * PTX + i % PTX, y = by * PTY + (i / PTX) % PTY, z = bz * PTZ + i / (PTX * PTY);
        if (x < g.nx && y < g.ny && z < g.nz) {
            __bf16 v[C];
            __builtin_memcpy(v, A + g.vox(x, y, z) * C, sizeof v);
#pragma unroll
            for (int c = 0; c < C; c++) s[c] += bf2f(v[c]);
        }
    }
#pragma unroll
    for (int c = 0; c < C; c++) part[threadIdx.x][c] = s[c];
    __syncthreads();
    if (threadIdx.x < C) {
        float tot = 0.f;
        for (int i = 0; i < 256; i++) tot += part[i][threadIdx.x];
        const int nxv = min(PTX, g.nx - bx * PTX), nyv = min(PTY, g.ny - by * PTY), nzv = min(PTZ, g.nz - bz * PTZ);
        feat[(long)t * C + threadIdx.x] = tot / (float)(nxv * nyv * nzv);
    }
}

// gradient of the pool (times the ReLU mask of the pooled activation)
__global__ __launch_bounds__(256) void pool_bwd(const float *__restrict__ dfeat, const __bf16 *__restrict__ A,
                                                __bf16 *__restrict__ G, ActGeom g, int ntx, int nty)
{
    const long n = (long)g.nx * g.ny * g.nz;
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const int x = (int)(i % g.nx), y = (int)((i / g.nx) % g.ny), z = (int)(i / ((long)g.nx * g.ny));
    const int bx = x / PTX, by = y / PTY, bz = z / PTZ;
    const int t = (bz * nty + by) * ntx + bx;
    const int nxv = min(PTX, g.nx - bx * PTX), nyv = min(PTY, g.ny - by * PTY), nzv = min(PTZ, g.nz - bz * PTZ);
    const float inv = 1.f / (float)(nxv * nyv * nzv);
    const long v = g.vox(x, y, z);
    __bf16 a[C], o[C];
    __builtin_memcpy(a, A + v * C, sizeof a);
#pragma unroll
    for (int c = 0; c < C; c++) o[c] = (__bf16)(bf2f(a[c]) > 0.f ? dfeat[(long)t * C + c] * inv : 0.f);
    __builtin_memcpy(G + v * C, o, sizeof o);
}

// ---------------------------------------------------------------------------
// Head: logits = bh + feat . Wh, softmax over the N_s offsets (one block per
// tile).  With a target mass it writes the tile's cross-entropy and
// dlogits = (q - p) / ntiles.
// ---------------------------------------------------------------------------
__device__ __forceinline__ float block_reduce(float v, float *sh, bool is_max)
{
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        const float u = __shfl_xor(v, o, 64);
        v = is_max ? __builtin_fmaxf(v, u) : v + u;
    }
    __syncthreads();
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    float r = sh[0];
    for (int w = 1; w < 4; w++) r = is_max ? __builtin_fmaxf(r, sh[w]) : r + sh[w];
    return r;
}

__global__ __launch_bounds__(256) void head_fwd(const float *__restrict__ feat, const float *__restrict__ Wh,
                                                const float *__restrict__ bh, int ns, const float *__restrict__ mass,
                                                float *__restrict__ probs, float *__restrict__ dlogits,
                                                float *__restrict__ tile_loss, float inv_tiles)
{
    extern __shared__ float lg[];  // ns logits
    __shared__ float sh[4];
    const int t = blockIdx.x;
    float f[C];
#pragma unroll
    for (int c = 0; c < C; c++) f[c] = feat[(long)t * C + c];
    float mx = -3.0e38f;
    for (int s = threadIdx.x; s < ns; s += 256) {
        float l = bh[s];
#pragma unroll
        for (int c = 0; c < C; c++) l = __builtin_fmaf(f[c], Wh[(long)c * ns + s], l);
        lg[s] = l;
        mx = __builtin_fmaxf(mx, l);
    }
    mx = block_reduce(mx, sh, true);
    float se = 0.f;
    for (int s = threadIdx.x; s < ns; s += 256) se += expf(lg[s] - mx);
    se = block_reduce(se, sh, false);
    const float lse = mx + logf(se);
    float tm = 0.f;
    if (mass)
        for (int s = threadIdx.x; s < ns; s += 256) tm += mass[(long)t * ns + s];
    if (mass) tm = block_reduce(tm, sh, false);
    float ce = 0.f;
    for (int s = threadIdx.x; s < ns; s += 256) {
        const float lq = lg[s] - lse;
        const float qv = expf(lq);
        if (probs) probs[(long)t * ns + s] = qv;
        if (mass) {
            const float p = tm > 0.f ? mass[(long)t * ns + s] / tm : 1.f / (float)ns;
            ce -= p * lq;
            dlogits[(long)t * ns + s] = (qv - p) * inv_tiles;
        }
    }
    if (mass) {
        ce = block_reduce(ce, sh, false);
        if (threadIdx.x == 0) tile_loss[t] = ce * inv_tiles;
    }
}

// loss = sum of the tiles' terms, in a fixed order (strided per thread,
// then the block's fixed reduction tree)
__global__ __launch_bounds__(256) void loss_reduce(const float *__restrict__ tile_loss, int ntiles,
                                                   float *__restrict__ loss)
{
    __shared__ float sh[4];
    float v = 0.f;
    for (int t = threadIdx.x; t < ntiles; t += 256) v += tile_loss[t];
    v = block_reduce(v, sh, false);
    if (threadIdx.x == 0) loss[0] = v;
}

// dWh[c][s] = sum_t feat[t][c] dl[t][s]; dbh[s] = sum_t dl[t][s]:
// partial sums over a share of the tiles (blockIdx.y of gridDim.y), added by
// wgrad_reduce: part[share][c * ns + s], then part[share][C ns + s] for the
// bias.  kHeadShares blocks along the tiles keep the chip busy where ns / 256
// blocks alone did not: 2.6 ms for 8192 tiles and 1326 offsets against
// 0.03 ms.
__global__ __launch_bounds__(256) void head_bwd_w(const float *__restrict__ feat, const float *__restrict__ dl,
                                                  int ntiles, int ns, float *__restrict__ part)
{
    const int s = blockIdx.x * 256 + threadIdx.x;
    if (s >= ns) return;
    const int t0 = (int)((long)ntiles * blockIdx.y / gridDim.y), t1 = (int)((long)ntiles * (blockIdx.y + 1) / gridDim.y);
    float acc[C], ab = 0.f;
#pragma unroll
    for (int c = 0; c < C; c++) acc[c] = 0.f;
#pragma unroll 4
    for (int t = t0; t < t1; t++) {
        const float d = dl[(long)t * ns + s];
        ab += d;
#pragma unroll
        for (int c = 0; c < C; c++) acc[c] = __builtin_fmaf(feat[(long)t * C + c], d, acc[c]);
    }
    float *pb = part + (long)blockIdx.y * (C + 1) * ns;
#pragma unroll
    for (int c = 0; c < C; c++) pb[(long)c * ns + s] = acc[c];
    pb[(long)C * ns + s] = ab;
}

// dfeat[t][c] = sum_s dl[t][s] Wh[c][s]  (one block per tile)
__global__ __launch_bounds__(256) void head_bwd_x(const float *__restrict__ dl, const float *__restrict__ Wh, int ns,
                                                  float *__restrict__ dfeat)
{
    __shared__ float sh[4];
    const int t = blockIdx.x;
    float acc[C];
#pragma unroll
    for (int c = 0; c < C; c++) acc[c] = 0.f;
    for (int s = threadIdx.x; s < ns; s += 256) {
        const float d = dl[(long)t * ns + s];
#pragma unroll
        for (int c = 0; c < C; c++) acc[c] = __builtin_fmaf(d, Wh[(long)c * ns + s], acc[c]);
    }
    for (int c = 0; c < C; c++) {
        const float r = block_reduce(acc[c], sh, false);
        if (threadIdx.x == 0) dfeat[(long)t * C + c] = r;
    }
}

__global__ __launch_bounds__(256) void adam_kernel(float *__restrict__ p, const float *__restrict__ gr,
                                                   float *__restrict__ m1, float *__restrict__ m2, long n, float lr,
                                                   float b1, float b2, float eps, float c1, float c2)
{
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const float g = gr[i];
    const float a = b1 * m1[i] + (1.f - b1) * g;
    const float b = b2 * m2[i] + (1.f - b2) * g * g;
    m1[i] = a;
    m2[i] = b;
    p[i] -= lr * (a * c1) / (sqrtf(b * c2) + eps);
}

// BF16 copies of the conv weights for the MFMA kernel: forward layout
// [tap][cout][cin] and input-gradient layout [tap][cin][cout] with the taps
// mirrored (tap -> 26 - tap).
__global__ __launch_bounds__(256) void pack_weights(const float *__restrict__ w, __bf16 *__restrict__ wf,
                                                    __bf16 *__restrict__ wb)
{
    const int i = blockIdx.x * 256 + threadIdx.x;  // over [tap][cin][cout]
    if (i >= NTAP * C * C) return;
    const int t = i / (C * C), ci = (i / C) % C, co = i % C;
    const __bf16 v = (__bf16)w[i];
    wf[((long)t * C + co) * C + ci] = v;
    wb[((long)(NTAP - 1 - t) * C + ci) * C + co] = v;
}

// volume (float, unpadded) -> normalised FP32 input with zero halo
__global__ __launch_bounds__(256) void prep_input(const float *__restrict__ vol, float *__restrict__ in, ActGeom g,
                                                  float shift, float scale)
{
    const long n = (long)g.nx * g.ny * g.nz;
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const int x = (int)(i % g.nx), y = (int)((i / g.nx) % g.ny), z = (int)(i / ((long)g.nx * g.ny));
    in[g.vox(x, y, z)] = (vol[i] - shift) * scale;
}

// Top-K offsets per tile by predicted probability (bitonic sort of up to
// 2048 (probability, index) pairs in LDS), then the fallback decision: the
// tile keeps its K offsets (sorted by search index, i.e. in reference order)
// when their predicted mass reaches `threshold` and the tile is not drawn
// for the audit; otherwise it visits the full search.
__global__ __launch_bounds__(256) void topk_kernel(const float *__restrict__ probs, int ns, int K, float threshold,
                                                   float audit_frac, uint64_t seed, int *__restrict__ lists,
                                                   int *__restrict__ counts, float *__restrict__ stats)
{
    __shared__ float key[2048];
    __shared__ int idx[2048];
    __shared__ float sh[4];
    const int t = blockIdx.x;
    for (int i = threadIdx.x; i < 2048; i += 256) {
        // probabilities lie in [0, 1]; a NaN from a diverged network ranks
        // as 0 and the padding below every real key
        const float pv = i < ns ? probs[(long)t * ns + i] : -1.f;
        key[i] = pv == pv ? pv : 0.f;
        idx[i] = i;
    }
    __syncthreads();
    for (int size = 2; size <= 2048; size <<= 1)
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            for (int i = threadIdx.x; i < 1024; i += 256) {
                const int lo = 2 * i - (i & (stride - 1));
                const int hi = lo + stride;
                const bool desc = (lo & size) == 0;  // sort descending overall
                const bool swap = desc ? key[lo] < key[hi] : key[lo] > key[hi];
                if (swap) {
                    const float tk = key[lo];
                    key[lo] = key[hi];
                    key[hi] = tk;
                    const int ti = idx[lo];
                    idx[lo] = idx[hi];
                    idx[hi] = ti;
                }
            }
            __syncthreads();
        }
    float cap = 0.f;
    for (int i = threadIdx.x; i < K; i += 256) cap += key[i];
    cap = block_reduce(cap, sh, false);
    // audit draw: SplitMix64 of (seed, tile)
    uint64_t zz = seed + 0x9E3779B97F4A7C15ull * (uint64_t)(t + 1);
    zz = (zz ^ (zz >> 30)) * 0xBF58476D1CE4E5B9ull;
    zz = (zz ^ (zz >> 27)) * 0x94D049BB133111EBull;
    zz ^= zz >> 31;
    const bool audit = (double)(zz >> 11) * (1.0 / 9007199254740992.0) < (double)audit_frac;
    const bool keep = cap >= threshold && !audit && K < ns;
    if (threadIdx.x == 0) {
        counts[t] = keep ? K : ns;
        atomicAdd(&stats[0], keep ? 0.f : 1.f);
        atomicAdd(&stats[1], audit ? 1.f : 0.f);
        atomicAdd(&stats[2], cap);
        atomicAdd(&stats[3], (float)(keep ? K : ns));
    }
    __syncthreads();
    if (keep) {
        // the K kept indices in ascending order (rank by counting)
        for (int i = threadIdx.x; i < K; i += 256) {
            int rank = 0;
            const int me = idx[i];
            for (int j = 0; j < K; j++) rank += idx[j] < me;
            lists[(long)t * K + rank] = me;
        }
    }
}

}  // namespace

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
struct ProposalNet::Impl {
    int ns = 0;
    int device = 0;
    hipStream_t st = nullptr;
    // parameters, FP32 master copies, in one buffer:
    // w1[27][16] b1[16] | w2[27][16][16] b2[16] | w3 ... | w4 ... | Wh[16][ns] bh[ns]
    long n_params = 0;
    float *params = nullptr, *grads = nullptr, *m1 = nullptr, *m2 = nullptr;
    long off_w1 = 0, off_b1 = 0, off_w[3] = {0, 0, 0}, off_b[3] = {0, 0, 0}, off_wh = 0, off_bh = 0;
    __bf16 *wf[3] = {nullptr, nullptr, nullptr}, *wb[3] = {nullptr, nullptr, nullptr};
    // activations: act[0..1] always (inference ping-pongs between them);
    // act[2..3] and the two gradient planes only for training
    long cap_vox = 0, cap_train = 0;
    float *in = nullptr;
    __bf16 *act[4] = {nullptr, nullptr, nullptr, nullptr};
    __bf16 *gbuf[2] = {nullptr, nullptr};
    int halo[7][3] = {};  // shape whose zero halo in, act and gbuf hold (0: none)
    long cap_tiles = 0;
    float *feat = nullptr, *dfeat = nullptr, *dl = nullptr, *probs = nullptr, *loss = nullptr;
    float *tile_loss = nullptr;  // per tile, summed by loss_reduce
    double *moments = nullptr;
    float *wpart = nullptr;  // weight-gradient partials, kWgradBlocks x kWgradStride
    int steps = 0;
};

namespace {

hipError_t ensure_acts(ProposalNet::Impl &m, const int shape[3], bool training)
{
    const long pv = (long)(shape[0] + 2) * (shape[1] + 2) * (shape[2] + 2);
    const long tiles = (long)((shape[0] + PTX - 1) / PTX) * ((shape[1] + PTY - 1) / PTY) * ((shape[2] + PTZ - 1) / PTZ);
    const size_t ab = (size_t)pv * C * sizeof(__bf16);
    hipError_t e;
    if (pv > m.cap_vox) {
        (void)hipFree(m.in);
        (void)hipFree(m.act[0]);
        (void)hipFree(m.act[1]);
        m.in = nullptr;
        m.act[0] = m.act[1] = nullptr;
        m.cap_vox = 0;
        std::memset(m.halo, 0, 3 * sizeof m.halo[0]);
        if ((e = hipMalloc(&m.in, pv * sizeof(float))) != hipSuccess) return e;
        if ((e = hipMalloc(&m.act[0], ab)) != hipSuccess) return e;
        if ((e = hipMalloc(&m.act[1], ab)) != hipSuccess) return e;
        m.cap_vox = pv;
    }
    if (training && pv > m.cap_train) {
        for (int i = 2; i < 4; i++) {
            (void)hipFree(m.act[i]);
            m.act[i] = nullptr;
        }
        for (auto &a : m.gbuf) {
            (void)hipFree(a);
            a = nullptr;
        }
        m.cap_train = 0;
        std::memset(m.halo[3], 0, 4 * sizeof m.halo[0]);
        for (int i = 2; i < 4; i++)
            if ((e = hipMalloc(&m.act[i], ab)) != hipSuccess) return e;
        for (auto &a : m.gbuf)
            if ((e = hipMalloc(&a, ab)) != hipSuccess) return e;
        m.cap_train = pv;
    }
    // the zero halos: no kernel writes them, so a buffer is cleared (its used
    // extent) when it is new or last held another shape
    auto halo = [&](int k, void *p, size_t bytes) {
        if (std::memcmp(m.halo[k], shape, sizeof m.halo[k]) == 0) return hipSuccess;
        std::memset(m.halo[k], 0, sizeof m.halo[k]);
        const hipError_t r = hipMemsetAsync(p, 0, bytes, m.st);
        if (r == hipSuccess) std::memcpy(m.halo[k], shape, sizeof m.halo[k]);
        return r;
    };
    if ((e = halo(0, m.in, pv * sizeof(float))) != hipSuccess) return e;
    for (int i = 0; i < (training ? 4 : 2); i++)
        if ((e = halo(1 + i, m.act[i], ab)) != hipSuccess) return e;
    if (training)
        for (int i = 0; i < 2; i++)
            if ((e = halo(5 + i, m.gbuf[i], ab)) != hipSuccess) return e;
    if (tiles > m.cap_tiles) {
        (void)hipFree(m.feat);
        (void)hipFree(m.dfeat);
        (void)hipFree(m.dl);
        (void)hipFree(m.probs);
        (void)hipFree(m.tile_loss);
        m.feat = m.dfeat = m.dl = m.probs = m.tile_loss = nullptr;
        m.cap_tiles = 0;
        if ((e = hipMalloc(&m.feat, tiles * C * sizeof(float))) != hipSuccess) return e;
        if ((e = hipMalloc(&m.dfeat, tiles * C * sizeof(float))) != hipSuccess) return e;
        if ((e = hipMalloc(&m.dl, tiles * (long)m.ns * sizeof(float))) != hipSuccess) return e;
        if ((e = hipMalloc(&m.probs, tiles * (long)m.ns * sizeof(float))) != hipSuccess) return e;
        if ((e = hipMalloc(&m.tile_loss, tiles * sizeof(float))) != hipSuccess) return e;
        m.cap_tiles = tiles;
    }
    return hipSuccess;
}

}  // namespace

ProposalNet::ProposalNet() : d(new Impl()) {}

ProposalNet::~ProposalNet()
{
    (void)hipSetDevice(d->device);
    if (d->st) (void)hipStreamSynchronize(d->st);
    for (float *p : {d->params, d->grads, d->m1, d->m2, d->in, d->feat, d->dfeat, d->dl, d->probs, d->loss,
                     d->tile_loss})
        (void)hipFree(p);
    for (int l = 0; l < 3; l++) {
        (void)hipFree(d->wf[l]);
        (void)hipFree(d->wb[l]);
    }
    for (auto &a : d->act) (void)hipFree(a);
    for (auto &a : d->gbuf) (void)hipFree(a);
    (void)hipFree(d->moments);
    (void)hipFree(d->wpart);
    if (d->st) (void)hipStreamDestroy(d->st);
    delete d;
}

long ProposalNet::num_params() const { return d->n_params; }
int ProposalNet::num_offsets() const { return d->ns; }
const float *ProposalNet::probs() const { return d->probs; }

hipError_t ProposalNet::init(int ns, int device, uint64_t seed)
{
    if (ns < 1 || ns > kMaxProposalOffsets) return hipErrorInvalidValue;
    d->ns = ns;
    d->device = device;
    hipError_t e;
    if ((e = hipSetDevice(device)) != hipSuccess) return e;
    if ((e = hipStreamCreateWithFlags(&d->st, hipStreamNonBlocking)) != hipSuccess) return e;
    long o = 0;
    d->off_w1 = o;
    o += NTAP * C;
    d->off_b1 = o;
    o += C;
    for (int l = 0; l < 3; l++) {
        d->off_w[l] = o;
        o += (long)NTAP * C * C;
        d->off_b[l] = o;
        o += C;
    }
    d->off_wh = o;
    o += (long)C * ns;
    d->off_bh = o;
    o += ns;
    d->n_params = o;
    const size_t bytes = o * sizeof(float);
    if ((e = hipMalloc(&d->params, bytes)) != hipSuccess) return e;
    if ((e = hipMalloc(&d->grads, bytes)) != hipSuccess) return e;
    if ((e = hipMalloc(&d->m1, bytes)) != hipSuccess) return e;
    if ((e = hipMalloc(&d->m2, bytes)) != hipSuccess) return e;
    if ((e = hipMalloc(&d->loss, sizeof(float))) != hipSuccess) return e;
    if ((e = hipMalloc(&d->moments, kMomentDoubles * sizeof(double))) != hipSuccess) return e;
    if ((e = hipMalloc(&d->wpart, (size_t)kWgradBlocks * kWgradStride * sizeof(float))) != hipSuccess) return e;
    for (int l = 0; l < 3; l++) {
        if ((e = hipMalloc(&d->wf[l], NTAP * C * C * sizeof(__bf16))) != hipSuccess) return e;
        if ((e = hipMalloc(&d->wb[l], NTAP * C * C * sizeof(__bf16))) != hipSuccess) return e;
    }
    // He-uniform initialisation from a SplitMix64 stream; zero biases; a
    // small head so the first predictions are near uniform
    std::vector<float> h(o, 0.f);
    uint64_t s = seed;
    auto rnd = [&]() {
        uint64_t z = (s += 0x9E3779B97F4A7C15ull);
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        z ^= z >> 31;
        return (double)(z >> 11) * (1.0 / 9007199254740992.0) * 2.0 - 1.0;
    };
    const double a1 = std::sqrt(6.0 / NTAP), a2 = std::sqrt(6.0 / (NTAP * C)), ah = std::sqrt(6.0 / C) * 0.1;
    for (int i = 0; i < NTAP * C; i++) h[d->off_w1 + i] = (float)(a1 * rnd());
    for (int l = 0; l < 3; l++)
        for (long i = 0; i < (long)NTAP * C * C; i++) h[d->off_w[l] + i] = (float)(a2 * rnd());
    for (long i = 0; i < (long)C * ns; i++) h[d->off_wh + i] = (float)(ah * rnd());
    if ((e = hipMemcpy(d->params, h.data(), bytes, hipMemcpyHostToDevice)) != hipSuccess) return e;
    if ((e = hipMemset(d->m1, 0, bytes)) != hipSuccess) return e;
    if ((e = hipMemset(d->m2, 0, bytes)) != hipSuccess) return e;
    return hipDeviceSynchronize();
}

hipError_t ProposalNet::set_params(const float *host, long n)
{
    if (n != d->n_params) return hipErrorInvalidValue;
    hipError_t e;
    if ((e = hipSetDevice(d->device)) != hipSuccess) return e;
    if ((e = hipMemcpy(d->params, host, n * sizeof(float), hipMemcpyHostToDevice)) != hipSuccess) return e;
    if ((e = hipMemset(d->m1, 0, n * sizeof(float))) != hipSuccess) return e;
    if ((e = hipMemset(d->m2, 0, n * sizeof(float))) != hipSuccess) return e;
    d->steps = 0;
    return hipDeviceSynchronize();
}

hipError_t ProposalNet::get_params(float *host, long n) const
{
    if (n != d->n_params) return hipErrorInvalidValue;
    hipError_t e;
    if ((e = hipSetDevice(d->device)) != hipSuccess) return e;
    return hipMemcpy(host, d->params, n * sizeof(float), hipMemcpyDeviceToHost);
}

hipError_t ProposalNet::get_grads(float *host, long n) const
{
    if (n != d->n_params) return hipErrorInvalidValue;
    hipError_t e;
    if ((e = hipSetDevice(d->device)) != hipSuccess) return e;
    return hipMemcpy(host, d->grads, n * sizeof(float), hipMemcpyDeviceToHost);
}

hipError_t ProposalNet::run(const float *vol, const int shape[3], const float *mass, bool backward, float *loss_host)
{
    Impl &m = *d;
    hipError_t e;
    if (shape[0] < 1 || shape[1] < 1 || shape[2] < 1) return hipErrorInvalidValue;
    if ((e = hipSetDevice(m.device)) != hipSuccess) return e;
    const bool training = mass && backward;
    if ((e = ensure_acts(m, shape, training)) != hipSuccess) return e;
    ActGeom g;
    g.nx = shape[0];
    g.ny = shape[1];
    g.nz = shape[2];
    g.sx = g.nx + 2;
    g.sy = (long)(g.nx + 2) * (g.ny + 2);
    const long nv = (long)g.nx * g.ny * g.nz;
    const unsigned vb = (unsigned)((nv + 255) / 256);
    const int ntx = (g.nx + PTX - 1) / PTX, nty = (g.ny + PTY - 1) / PTY, ntz = (g.nz + PTZ - 1) / PTZ;
    const int ntiles = ntx * nty * ntz;
    const long ctiles = (long)((g.nx + CTX - 1) / CTX) * ((g.ny + CTY - 1) / CTY) * ((g.nz + CTZ - 1) / CTZ);
    const unsigned cb = (unsigned)std::min<long>(ctiles, kConvBlocks);

    // input normalisation: (v - mean) / std of this volume (FP64 moments)
    if ((e = launch_moments(vol, nv, m.moments, m.st)) != hipSuccess) return e;
    double mom[2];
    if ((e = hipMemcpyAsync(mom, m.moments, sizeof mom, hipMemcpyDeviceToHost, m.st)) != hipSuccess) return e;
    if ((e = hipStreamSynchronize(m.st)) != hipSuccess) return e;
    const double mean = mom[0] / (double)nv;
    const double var = std::max(mom[1] / (double)nv - mean * mean, 0.0);
    const float shift = (float)mean, scale = var > 0 ? (float)(1.0 / std::sqrt(var)) : 1.f;

    const float *P = m.params;
    for (int l = 0; l < 3; l++)
        hipLaunchKernelGGL(pack_weights, dim3((NTAP * C * C + 255) / 256), dim3(256), 0, m.st, P + m.off_w[l],
                           m.wf[l], m.wb[l]);
    hipLaunchKernelGGL(prep_input, dim3(vb), dim3(256), 0, m.st, vol, m.in, g, shift, scale);
    hipLaunchKernelGGL(conv1_fwd, dim3(vb), dim3(256), 0, m.st, m.in, P + m.off_w1, P + m.off_b1, m.act[0], g);
    // training keeps every layer's activation for the backward pass;
    // inference alternates between two planes
    auto A = [&](int l) { return training ? m.act[l] : m.act[l & 1]; };
    for (int l = 0; l < 3; l++)
        hipLaunchKernelGGL(conv16_mfma<0>, dim3(cb), dim3(256), 0, m.st, A(l), m.wf[l], P + m.off_b[l],
                           (const __bf16 *)nullptr, A(l + 1), g);
    hipLaunchKernelGGL(pool_fwd, dim3(ntiles), dim3(256), 0, m.st, A(3), m.feat, g, ntx, nty);
    hipLaunchKernelGGL(head_fwd, dim3(ntiles), dim3(256), m.ns * sizeof(float), m.st, m.feat, P + m.off_wh,
                       P + m.off_bh, m.ns, mass, m.probs, mass ? m.dl : nullptr, m.tile_loss, 1.f / (float)ntiles);
    if (mass) hipLaunchKernelGGL(loss_reduce, dim3(1), dim3(256), 0, m.st, m.tile_loss, ntiles, m.loss);
    else if ((e = hipMemsetAsync(m.loss, 0, sizeof(float), m.st)) != hipSuccess) return e;
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if (training) {
        float *G = m.grads;
        auto reduce = [&](long stride, int nblocks, int n, float *out) {
            hipLaunchKernelGGL(wgrad_reduce, dim3((unsigned)((n + 63) / 64)), dim3(256), 0, m.st, m.wpart, stride,
                               nblocks, n, out);
        };
        const int shares = std::min(ntiles, kHeadShares);
        hipLaunchKernelGGL(head_bwd_w, dim3((m.ns + 255) / 256, shares), dim3(256), 0, m.st, m.feat, m.dl, ntiles,
                           m.ns, m.wpart);
        reduce((long)(C + 1) * m.ns, shares, (C + 1) * m.ns, G + m.off_wh);
        hipLaunchKernelGGL(head_bwd_x, dim3(ntiles), dim3(256), 0, m.st, m.dl, P + m.off_wh, m.ns, m.dfeat);
        // gradient at the pre-activation of the last convolution
        hipLaunchKernelGGL(pool_bwd, dim3(vb), dim3(256), 0, m.st, m.dfeat, m.act[3], m.gbuf[0], g, ntx, nty);
        const long wtiles = (long)((g.nx + WTX - 1) / WTX) * ((g.ny + WTY - 1) / WTY) * ((g.nz + WTZ - 1) / WTZ);
        const int wtb = (int)std::min<long>(wtiles, kWgradBlocks);
        int cur = 0;
        for (int l = 2; l >= 0; l--) {
            // convolution l+2: input act[l], gradient at its output gbuf[cur]
            hipLaunchKernelGGL(conv16_wgrad, dim3(wtb), dim3(256), 0, m.st, m.act[l], m.gbuf[cur], m.wpart, g);
            reduce(kWgradStride, wtb, NTAP * C * C + C, G + m.off_w[l]);
            hipLaunchKernelGGL(conv16_mfma<1>, dim3(cb), dim3(256), 0, m.st, m.gbuf[cur], m.wb[l],
                               (const float *)nullptr, m.act[l], m.gbuf[cur ^ 1], g);
            cur ^= 1;
        }
        const int w1b = (int)std::min<long>((long)((g.nx + 63) / 64) * g.ny * g.nz, kWgradBlocks);
        hipLaunchKernelGGL(conv1_wgrad, dim3(w1b), dim3(192), 0, m.st, m.in, m.gbuf[cur], m.wpart, g);
        reduce(kWgradStride, w1b, NTAP * C + C, G + m.off_w1);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    if (loss_host) {
        if ((e = hipMemcpyAsync(loss_host, m.loss, sizeof(float), hipMemcpyDeviceToHost, m.st)) != hipSuccess)
            return e;
    }
    return hipStreamSynchronize(m.st);
}

hipError_t ProposalNet::adam(float lr)
{
    Impl &m = *d;
    hipError_t e;
    if ((e = hipSetDevice(m.device)) != hipSuccess) return e;
    m.steps++;
    const double b1 = 0.9, b2 = 0.999;
    const float c1 = (float)(1.0 / (1.0 - std::pow(b1, (double)m.steps)));
    const float c2 = (float)(1.0 / (1.0 - std::pow(b2, (double)m.steps)));
    hipLaunchKernelGGL(adam_kernel, dim3((unsigned)((m.n_params + 255) / 256)), dim3(256), 0, m.st, m.params,
                       m.grads, m.m1, m.m2, m.n_params, lr, (float)b1, (float)b2, 1e-8f, c1, c2);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    return hipStreamSynchronize(m.st);
}

hipError_t launch_topk(const float *probs, int ntiles, int ns, int K, float threshold, float audit_frac,
                       uint64_t seed, int *lists, int *counts, float *stats, hipStream_t st)
{
    if (ns < 1 || ns > kMaxProposalOffsets || K < 1 || K > ns) return hipErrorInvalidValue;
    hipLaunchKernelGGL(topk_kernel, dim3(ntiles), dim3(256), 0, st, probs, ns, K, threshold, audit_frac, seed, lists,
                       counts, stats);
    return hipGetLastError();
}

}  // namespace inlm
