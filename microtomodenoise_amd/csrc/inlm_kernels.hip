// iterNLM filter, padding and noise kernels for gfx950 (MI355X).
//
// The filter pass computes, per voxel x of slice z (sigma = sigma[z],
// m = -1/(sigma^2*beta)):
//   d_s(x) = sum_p W_p * (P[x+s+p] - P[x+p])^2       (taps p in reference order)
//   w_s    = pade(d_s*m) if d_s*m > -3.56648 else 0   (or expf)
//   num += w_s*R[x+s]; den += w_s; wmax = max(wmax, w_s)
//   out    = (num + wmax*R[x]) / (den + wmax)          (R[x] when wmax == 0)
// which restates Denoiser/iternlm_cpu.cpp:758-843 and the specialised
// Denoiser/iternlm_cpu_kernels.cpp:7-1108 of the reference.
//
// The tiled kernels are offset-major: a workgroup owns a 32x8x8 output tile
// (32x64x1 for flat patches);
// for each search offset s it stages D_s(y) = (P(y+s) - P(y))^2 over the tile
// plus the patch halo in LDS (double buffered, one barrier per offset) and
// every thread sums the stencil for a run of 4 voxels along x from LDS
// windows.  D_s(x+p) is the very float the reference computes as tmp*tmp for
// tap p, and every voxel adds its taps in the reference order with separate
// multiply and add (this file is compiled with -ffp-contract=off), so the
// result is bit-identical to the reference CPU path.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "inlm_kernels.hpp"

namespace inlm {
namespace {

constexpr int NT = 256;   // threads per workgroup of the helper kernels
constexpr int NTF = 512;  // threads per workgroup of the tiled filter (8 wavefronts)
constexpr int TX = 32, VX = 4;  // tile width; each thread sums a 4-voxel x-run
constexpr float kPadeCut = -3.56648f;

// ---------------------------------------------------------------------------
// Compile-time patch rows of an ellipsoid of radii (RX, RY, RZ), in the
// reference scan order z -> y -> x (iternlm_prepare.cpp:152-203).  Each row
// (dz,dy) holds the taps dx = -j..j; tap0 is the reference index of its first
// tap (index 0 is the centre, which leads the list).  Every tap also carries a
// weight class: the centre is class 0, other taps are grouped by
// (dx^2+dy^2, dz^2), which fixes 1/(2d+1)^2 for any z anisotropy, so the
// kernel needs one scalar weight per class instead of one per tap.
// ---------------------------------------------------------------------------
struct Row {
    int dz, dy, j, tap0;
};
constexpr int kMaxClasses = 48;
template <int RX, int RY, int RZ>
struct Rows {
    Row r[(2 * RY + 1) * (2 * RZ + 1)];
    int n, ntaps, nclass;
    int key_rho[kMaxClasses], key_z[kMaxClasses];
    static constexpr bool inside(int x, int y, int z)
    {
        const float fx = (float)x / (float)(RX > 1 ? RX : 1), fy = (float)y / (float)(RY > 1 ? RY : 1),
                    fz = (float)z / (float)(RZ > 1 ? RZ : 1);
        float e = fx * fx;
        e = e + fy * fy;
        e = e + fz * fz;
        return e <= 1.f;
    }
    constexpr int class_of(int dx, int dy, int dz) const
    {
        if (dx == 0 && dy == 0 && dz == 0) return 0;
        for (int c = 1; c < nclass; c++)
            if (key_rho[c] == dx * dx + dy * dy && key_z[c] == dz * dz) return c;
        return -1;
    }
    constexpr Rows() : r(), n(0), ntaps(0), nclass(1), key_rho(), key_z()
    {
        int tap = 1;
        for (int z = -RZ; z <= RZ; ++z)
            for (int y = -RY; y <= RY; ++y) {
                int j = -1;
                for (int x = 0; x <= RX; ++x)
                    if (inside(x, y, z)) j = x;
                if (j < 0) continue;
                r[n] = Row{z, y, j, tap};
                n++;
                tap += 2 * j + 1 - ((z == 0 && y == 0) ? 1 : 0);
                for (int x = -j; x <= j; ++x) {
                    if (x == 0 && y == 0 && z == 0) continue;
                    if (class_of(x, y, z) < 0) {
                        key_rho[nclass] = x * x + y * y;
                        key_z[nclass] = z * z;
                        nclass++;
                    }
                }
            }
        ntaps = tap;
    }
};
// A patch shape of the tiled kernel.
template <int RX_, int RY_, int RZ_>
struct Patch {
    static constexpr int RX = RX_, RY = RY_, RZ = RZ_;
    static constexpr Rows<RX, RY, RZ> rows{};
    static_assert(rows.nclass <= kMaxClasses, "too many weight classes");
    // one weight for every tap (1/7, or 1/9 in a plane): the staged squares
    // are multiplied by it once instead of once per tap
    static constexpr bool kUniform = RX == 1 && RY == 1 && RZ <= 1;
    // large patches leave whole wavefronts without a weight above the cutoff
    static constexpr bool kSkip = rows.ntaps > 50;
    // A NaN weight (an exp weight of a NaN distance): isotropic patches take it
    // for the largest, and the voxel keeps its value; the others pass it over
    // in the maximum and it reaches the sums, as in the per-voxel kernel.
    static constexpr bool kNanIsLargest = RX == RY && RX == RZ;
};

// Compiler fence that also pins the running sums: the row's arithmetic must
// complete before it and no memory access moves across it.
__device__ __forceinline__ void pin(float (&d)[4])
{
    asm volatile("" : "+v"(d[0]), "+v"(d[1]), "+v"(d[2]), "+v"(d[3])::"memory");
}

template <int I, int N, class F>
__device__ __forceinline__ void static_for(F &&f)
{
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}

// LDS layout of the parity kernel: rows of 40 floats.  gfx950 serves a
// ds_read_b128 in four groups of 16 lanes ({0-3, 12-15, 20-27},
// {4-11, 16-19, 28-31} and the same +32), each group one 256-byte pass over
// 64 banks.  A lane reads the 16 bytes at row ty, float 4*xr, i.e. 16-byte
// bank group (10*ty + xr) mod 16; with a 40-float pitch every bank group
// occurs exactly four times over the 8x8 (xr, ty) cells of a wavefront, and
// kLaneCell hands each hardware group 16 cells with 16 distinct bank groups,
// so the window reads are conflict-free for every row shift.
constexpr int kPitch = 40;
__constant__ const unsigned char kLaneCell[64] = {
    0,  1,  2,  3,  14, 15, 28, 29, 16, 17, 18, 19, 4,  5,  6,  7,  32, 33, 22, 23, 20, 21,
    8,  9,  10, 11, 12, 13, 36, 37, 24, 25, 26, 27, 40, 41, 52, 53, 54, 55, 42, 43, 56, 57,
    30, 31, 44, 45, 58, 59, 60, 61, 46, 47, 34, 35, 48, 49, 38, 39, 62, 63, 50, 51};  // xr | ty << 3

template <class PT>
struct Tile {
    static constexpr int TZ = PT::RZ == 0 ? 1 : 8, TY = PT::RZ == 0 ? 64 : 8;  // a flat patch takes flat tiles
    static constexpr int RY = TY + 2 * PT::RY, RZ = TZ + 2 * PT::RZ;
    // LDS column of a tile's first voxel.  Patches of one tap per row outside
    // the middle one (RX = 1) keep each 4-voxel run on one 16-byte read.
    static constexpr int O = PT::RX == 1 ? 4 : PT::RX;
    static constexpr int PITCH = kPitch;  // LDS row pitch in floats
    static_assert(O + TX + PT::RX <= kPitch, "patch radius too large for the LDS row");
    static constexpr int CPR = PITCH / 4;        // 4-float chunks per row
    static constexpr int NCHUNK = RZ * RY * CPR;
    static constexpr int CPT = (NCHUNK + NTF - 1) / NTF;  // chunks staged per thread
    static constexpr int LDS = CPT * NTF * 4;  // floats per buffer: slots past NCHUNK write behind the region
    // chunks a run reads of a row of half-width j: columns O - j .. O + 3 + j
    static constexpr int lo(int j) { return (O - j) / 4; }
    static constexpr int hi(int j) { return (O + 3 + j) / 4; }
    static constexpr int WIN = 4 * (hi(PT::RX) - lo(PT::RX) + 1);
};

struct TiledArgs {
    const float *R;
    const float *P;
    float *out;
    const float *sigma;
    const SearchEntry *search;
    int n_search;
    float beta;
    FilterGeom g;
    int ntx, nty, ntz;
    float wc[kMaxClasses];  // weight per class (class 0 = centre)
    float *mass;            // optional: [tile][offset] sum of the weights over the tile's voxels
};

// Correctly rounded n/d for the operands the Pade weight produces
// (n in [0, 120], d in [120, 600]: no overflow, underflow or special value):
// the quotient by the hardware reciprocal and one correction with the exact
// fused remainder.  Both are functions of one float, and
// selftest_div_kernel compares the weight with IEEE division on every float
// of its domain, so neither a refined reciprocal nor a second correction
// (four more instructions, as a general division needs) is kept.
__device__ __forceinline__ float div_pade(float n, float d)
{
    const float y = __builtin_amdgcn_rcpf(d);
    const float q = n * y;
    const float r = __builtin_fmaf(-d, q, n);
    return __builtin_fmaf(r, y, q);
}

// (120 + 60a + 12a^2 + a^3) / (120 - 60a + 12a^2 - a^3), evaluated left to
// right with every product and sum rounded, as Denoiser/iternlm_cpu.h:125
// writes it, and zero at or below the cutoff of iternlm_cpu.h:126.
template <bool IEEE_DIV>
__device__ __forceinline__ float pade_cut(float a)
{
    const float t60 = 60.f * a;
    const float t12 = (12.f * a) * a;
    const float t3 = (a * a) * a;
    float num = 120.f + t60;
    num = num + t12;
    num = num + t3;
    float den = 120.f - t60;
    den = den + t12;
    den = den - t3;
    const float q = IEEE_DIV ? num / den : div_pade(num, den);
    return (a > kPadeCut) ? q : 0.0f;
}

template <int WFN>
__device__ __forceinline__ float weight_of(float a)
{
    if constexpr (WFN == 0) return pade_cut<false>(a);
    else return expf(a);
}

// Workgroup id -> tile, so that the tiles one XCD runs are contiguous (the
// hardware deals workgroups to the 8 XCDs round-robin, and neighbouring tiles
// share their halo in that XCD's L2), for any number of workgroups: the first
// nwg % 8 XCDs take one more.  Where the count is no
// multiple of 8, dealing tiles in order (as before) cost 8% at r = 2 on
// 301x333x131 (37.6 against 34.8 ms) and 66% on a 1200x900 colour image (1.63
// against 0.98 ms), whose tiles then came from the other XCDs' side of memory.
__device__ __forceinline__ int xcd_swizzle(int wg, int nwg)
{
    const int xcd = wg & 7, more = nwg & 7;
    return xcd * (nwg >> 3) + (xcd < more ? xcd : more) + (wg >> 3);
}

// Chunks lo..hi of a row of half-width J: whole 16-byte reads (one
// ds_read_b128 with an immediate offset), not the narrowed pieces the compiler
// would pick.
template <class PT, int J>
__device__ __forceinline__ void load_window(const float *row, float (&win)[Tile<PT>::WIN])
{
    using T = Tile<PT>;
    typedef float f4v __attribute__((ext_vector_type(4)));
#pragma unroll
    for (int i = T::lo(J); i <= T::hi(J); i++) {
        f4v q = *reinterpret_cast<const f4v *>(row + 4 * i);
        asm("" : "+v"(q));
#pragma unroll
        for (int e = 0; e < 4; e++) win[4 * (i - T::lo(J)) + e] = q[e];
    }
}

// The distances of a 4-voxel run: the taps of the squares staged around LDS
// row L in reference order, every product and sum rounded.
template <class PT>
__device__ __forceinline__ void patch_sums(const float *L, const float *wc, float (&d)[VX])
{
    using T = Tile<PT>;
    float win[2][T::WIN];
    {
        // the centre tap leads the sum (iternlm_prepare.cpp:176-177)
        load_window<PT, 0>(L, win[1]);
        const float w0 = wc[0];
#pragma unroll
        for (int v = 0; v < VX; v++) {
            const float c = win[1][T::O + v - 4 * T::lo(0)];
            d[v] = PT::kUniform ? c : c * w0;
        }
    }
    // Rows in reference order; the window of row i+1 is read while row i
    // is summed.  A compiler barrier per row keeps the optimiser from
    // hoisting every window above the arithmetic (which exhausts the
    // register budget and spills).
    constexpr int NR = PT::rows.n;
    constexpr Row first = PT::rows.r[0];
    load_window<PT, first.j>(L + (first.dz * T::RY + first.dy) * T::PITCH, win[0]);
    static_for<0, NR>([&](auto ri) __attribute__((always_inline)) {
        constexpr int i = decltype(ri)::value;
        constexpr Row rw = PT::rows.r[i];
        if constexpr (i + 1 < NR) {
            constexpr Row nx = PT::rows.r[i + 1];
            load_window<PT, nx.j>(L + (nx.dz * T::RY + nx.dy) * T::PITCH, win[(i + 1) & 1]);
        }
        static_for<0, 2 * rw.j + 1>([&](auto kk) __attribute__((always_inline)) {
            constexpr int dx = decltype(kk)::value - rw.j;
            if constexpr (!(rw.dz == 0 && rw.dy == 0 && dx == 0)) {
                constexpr int cls = PT::rows.class_of(dx, rw.dy, rw.dz);
                const float wt = PT::kUniform ? 0.f : wc[cls];
#pragma unroll
                for (int v = 0; v < VX; v++) {
                    const float q = win[i & 1][T::O + v + dx - 4 * T::lo(rw.j)];
                    d[v] = d[v] + (PT::kUniform ? q : q * wt);
                }
            }
        });
        pin(d);
    });
}

// Occupancy is bounded by LDS to 4, 3 or 2 workgroups of 8 waves per CU (2, 3
// or 4 chunks per thread); the register budget is capped to match so that
// the scheduler does not trade occupancy for hoisted loads.
template <class PT, bool MASS>
constexpr int waves_per_eu() { return Tile<PT>::CPT <= 2 && PT::RX <= 2 && !MASS ? 8 : Tile<PT>::CPT <= 3 ? 6 : 4; }

// Vector issue bounds this kernel (no fused multiply-add, no packed FP32: at
// most one instruction every two cycles per SIMD).  Per offset and output it
// needs two instructions per tap, 21 issue slots for the weight and 4 for the
// sums.  The offsets of 62 steps lie in one register per lane, so a step
// has its addresses at once and issues its loads (R of this offset, the chunks
// of the next) before anything else; with the offsets read from memory each
// step waited for three loads one after the other.  Before (with the longer
// division, a multiply per tap at r = 1 and two reads per row there) and now:
// r = 1, 3102 offsets of 256^3: 54 and 43 ms; r = 2, 1326 offsets of
// 301x333x131: 41.6 and 34.8 ms (37.6 before xcd_swizzle took any number of
// workgroups); r = 3, 256x256x96: 40.2 and 38.1 ms.
template <class PT, int WFN, bool MASS>
__global__ __launch_bounds__(NTF) __attribute__((amdgpu_waves_per_eu(waves_per_eu<PT, MASS>(), waves_per_eu<PT, MASS>()))) void
filter_tiled_fp32(TiledArgs a)
{
    using T = Tile<PT>;
    __shared__ __attribute__((aligned(16))) float lds[2][T::LDS];
    __shared__ float red[2][NTF / 64];

    const int t = threadIdx.x;
    const int wg = xcd_swizzle(blockIdx.x, gridDim.x);
    const int bx = wg % a.ntx;
    const int rem = wg / a.ntx;
    const int by = rem % a.nty;
    const int bz = rem / a.nty;
    const int X0 = bx * TX, Y0 = by * T::TY, Z0 = bz * T::TZ;
    const FilterGeom g = a.g;
    const long sp = (long)g.nxp * g.nyp;
    const float w0 = a.wc[0];

    // Staging: LDS column 0 of region row 0 is voxel (X0 - O, Y0 - RY, Z0 - RZ).
    const float *pc[T::CPT];
    float p0[T::CPT][4];
#pragma unroll
    for (int c = 0; c < T::CPT; c++) {
        const int ci = t + c * NTF < T::NCHUNK ? t + c * NTF : 0;  // slots past the region repeat chunk 0
        const int cx = ci % T::CPR, row = ci / T::CPR;
        const int ry = row % T::RY, rz = row / T::RY;
        pc[c] = a.P + ((long)(Z0 + g.pz - PT::RZ + rz) * sp + (long)(Y0 + g.py - PT::RY + ry) * g.nxp +
                       (X0 + g.px - T::O + 4 * cx));
        __builtin_memcpy(p0[c], pc[c], 16);
    }

    // This thread's 4-voxel run.
    const int cell = kLaneCell[t & 63];
    const int xr = cell & 7, ty = (cell >> 3) + (T::TZ == 1 ? 8 * (t >> 6) : 0), tz = T::TZ == 1 ? 0 : t >> 6;
    const int x0 = X0 + VX * xr, y = Y0 + ty, z = Z0 + tz;
    const float *Rv = a.R + ((long)(z + g.pz) * sp + (long)(y + g.py) * g.nxp + (x0 + g.px));
    const int zc = z < g.nz ? z : g.nz - 1;
    const float sig = a.sigma[zc];
    const float m = -1.f / (sig * sig * a.beta);
    const bool valid = y < g.ny && z < g.nz;

    // wmax as the bits of a non-negative float: the integer max orders those
    // like floats (== (wt > wmax ? wt : wmax)) without NaN canonicalisation
    float fv[VX], fw[VX];
    unsigned wmax_bits[VX];
#pragma unroll
    for (int v = 0; v < VX; v++) {
        fv[v] = fw[v] = 0.f;
        wmax_bits[v] = 0u;
    }

    const int ldsrow = ((tz + PT::RZ) * T::RY + (ty + PT::RY)) * T::PITCH + VX * xr;
    const int nS = a.n_search;

    auto stage = [&](const float (&pn)[T::CPT][4], float *buf) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < T::CPT; c++) {
            float dv[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float q = pn[c][e] - p0[c][e];
                dv[e] = q * q;
                if constexpr (PT::kUniform) dv[e] = dv[e] * w0;
            }
            __builtin_memcpy(__builtin_assume_aligned(buf + 4 * (t + c * NTF), 16), dv, 16);
        }
    };
    auto load_chunks = [&](float (&pn)[T::CPT][4], int lin) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < T::CPT; c++) __builtin_memcpy(pn[c], pc[c] + lin, 16);
    };
    auto lin_at = [&](int k) __attribute__((always_inline)) { return a.search[k < nS ? k : nS - 1].lin; };

    // offset k from LDS buffer rd, while the chunks of offset k + 1 (the last
    // offset again past the end) go to wr
    int linv = 0, kb = 0;
    auto step = [&](int k, const float *rd, float *wr) __attribute__((always_inline)) {
        float rs[VX], pn[T::CPT][4];
        __builtin_memcpy(rs, Rv + __builtin_amdgcn_readlane(linv, k - kb), 16);
        load_chunks(pn, __builtin_amdgcn_readlane(linv, k + 1 - kb));
        const float *L = rd + ldsrow;
        float d[VX];
        patch_sums<PT>(L, a.wc, d);
        float sw = 0.f;
        bool some = true;
        if constexpr (PT::kSkip && WFN == 0) {
            bool any = false;
#pragma unroll
            for (int v = 0; v < VX; v++) any = any || d[v] * m > kPadeCut;
            some = __builtin_amdgcn_ballot_w64(any) != 0;
        }
        if (some) {
#pragma unroll
            for (int v = 0; v < VX; v++) {
                const float wt = weight_of<WFN>(d[v] * m);
                fv[v] = fv[v] + wt * rs[v];
                fw[v] = fw[v] + wt;
                if constexpr (PT::kNanIsLargest)
                    wmax_bits[v] = __builtin_elementwise_max(wmax_bits[v], __builtin_bit_cast(unsigned, wt));
                else  // the other operand of a NaN; the builtin would first quiet wmax, an instruction more
                    asm("v_max_f32 %0, %0, %1" : "+v"(wmax_bits[v]) : "v"(wt));
                if constexpr (MASS) sw += (valid && x0 + v < g.nx) ? wt : 0.f;
            }
        } else {
            // every weight of the wavefront is zero: only an infinite or NaN
            // value still reaches the sum
#pragma unroll
            for (int v = 0; v < VX; v++) fv[v] = fv[v] + 0.f * rs[v];
        }
        if constexpr (MASS) {
            // weight mass of this offset over the tile: wave sums into LDS,
            // thread 0 adds the 8 wave sums after the barrier below
#pragma unroll
            for (int o = 32; o >= 1; o >>= 1) sw += __shfl_xor(sw, o, 64);
            if ((t & 63) == 0) red[k & 1][t >> 6] = sw;
        }
        // the chunks are in flight until here: without the fence their first
        // use moves up among the window sums and waits for them
        __builtin_amdgcn_sched_barrier(0);
        stage(pn, wr);
        __syncthreads();
        if constexpr (MASS) {
            if (t == 0) {
                float tot = 0.f;
#pragma unroll
                for (int w = 0; w < NTF / 64; w++) tot += red[k & 1][w];
                a.mass[(long)wg * nS + k] = tot;
            }
        }
    };
    {
        float pn[T::CPT][4];
        load_chunks(pn, lin_at(0));
        stage(pn, lds[0]);
    }
    __syncthreads();
    constexpr int kBlock = 62;  // even; a step looks one offset ahead
    for (kb = 0; kb < nS; kb += kBlock) {
        linv = lin_at(kb + (t & 63));
        const int ke = kb + kBlock < nS ? kb + kBlock : nS;
        for (int k = kb; k < ke; k += 2) {
            step(k, lds[0], lds[1]);
            if (k + 1 < ke) step(k + 1, lds[1], lds[0]);
        }
    }

    float wmax[VX];
#pragma unroll
    for (int v = 0; v < VX; v++) wmax[v] = __builtin_bit_cast(float, wmax_bits[v]);
    if (y < g.ny && z < g.nz) {
        float *o = a.out + ((long)z * g.ny + y) * g.nx + x0;
#pragma unroll
        for (int v = 0; v < VX; v++) {
            if (x0 + v < g.nx) {
                const float r0 = Rv[v];
                float res;
                if (wmax[v] > 0.0f) {
                    const float num = fv[v] + wmax[v] * r0;
                    const float den = fw[v] + wmax[v];
                    res = num / den;
                } else
                    res = r0;
                o[v] = res;
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Per-voxel kernel for any tap table without a tiled kernel, and for volumes
// too thin for the tiles (tiled_pays): one thread per voxel, gathers straight
// from global memory, the same operation sequence as the tiled kernel.
// ---------------------------------------------------------------------------
struct VoxelArgs {
    const float *R;
    const float *P;
    float *out;
    const float *sigma;
    const SearchEntry *search;
    int n_search;
    float beta;
    FilterGeom g;
    TapTable taps;
};

template <int WFN>
__global__ __launch_bounds__(NT) void filter_pervoxel_fp32(VoxelArgs a)
{
    const FilterGeom g = a.g;
    const long nvox = (long)g.nx * g.ny * g.nz;
    const long idx = (long)blockIdx.x * NT + threadIdx.x;
    if (idx >= nvox) return;
    const int x = (int)(idx % g.nx);
    const int y = (int)((idx / g.nx) % g.ny);
    const int z = (int)(idx / ((long)g.nx * g.ny));
    const long sp = (long)g.nxp * g.nyp;
    const long i0 = (long)(z + g.pz) * sp + (long)(y + g.py) * g.nxp + (x + g.px);
    const float sig = a.sigma[z];
    const float m = -1.f / (sig * sig * a.beta);
    float fv = 0.f, fw = 0.f, wmax = 0.f;
    for (int k = 0; k < a.n_search; k++) {
        const long i1 = i0 + a.search[k].lin;
        float d = 0.f;
        for (int p = 0; p < a.taps.n; p++) {
            const float q = a.P[i1 + a.taps.lin[p]] - a.P[i0 + a.taps.lin[p]];
            d = d + (q * q) * a.taps.w[p];
        }
        const float wt = weight_of<WFN>(d * m);
        fv = fv + wt * a.R[i1];
        fw = fw + wt;
        wmax = __builtin_fmaxf(wmax, wt);
    }
    const float r0 = a.R[i0];
    float res = r0;
    if (wmax > 0.0f) {
        const float num = fv + wmax * r0;
        const float den = fw + wmax;
        res = num / den;
    }
    a.out[idx] = res;
}

// ---------------------------------------------------------------------------
// Three-channel filter of the colour path (iternlm_cpu.cpp:932-1075): one
// thread per output pixel, the three channels' distances in patch order,
// each scaled by its channel's multiplier.  Joint weights (the default) take
// the mean of the three scaled distances and weight all channels alike,
// the centre counted once with the largest weight; independent channels
// weigh each channel by its own distance and, as the reference does, leave
// the centre out.  Every product and sum rounds as the reference's float code
// does (no contraction, IEEE division).
// ---------------------------------------------------------------------------
struct RgbArgs {
    const float *R[3];  // padded originals
    const float *P[3];  // padded previous iterates
    float *out[3];      // unpadded results
    const SearchEntry *search;
    int n_search;
    float mult[3];  // -1 / (sigma_c^2 beta)
    int independent;
    FilterGeom g;
    TapTable taps;
};

template <int WFN>
__global__ __launch_bounds__(NT) void filter_rgb_fp32(RgbArgs a)
{
    const FilterGeom g = a.g;
    const long nvox = (long)g.nx * g.ny * g.nz;
    const long idx = (long)blockIdx.x * NT + threadIdx.x;
    if (idx >= nvox) return;
    const int x = (int)(idx % g.nx);
    const int y = (int)((idx / g.nx) % g.ny);
    const int z = (int)(idx / ((long)g.nx * g.ny));
    const long sp = (long)g.nxp * g.nyp;
    const long i0 = (long)(z + g.pz) * sp + (long)(y + g.py) * g.nxp + (x + g.px);
    const float *P0 = a.P[0], *P1 = a.P[1], *P2 = a.P[2];
    float fv0 = 0.f, fv1 = 0.f, fv2 = 0.f, fw0 = 0.f, fw1 = 0.f, fw2 = 0.f, wm0 = 0.f, wm1 = 0.f, wm2 = 0.f;
    for (int k = 0; k < a.n_search; k++) {
        const long i1 = i0 + a.search[k].lin;
        float d0 = 0.f, d1 = 0.f, d2 = 0.f;
        for (int p = 0; p < a.taps.n; p++) {
            const int pp = a.taps.lin[p];
            const float dw = a.taps.w[p];
            float t = P0[i1 + pp] - P0[i0 + pp];
            d0 = d0 + (t * t) * dw;
            t = P1[i1 + pp] - P1[i0 + pp];
            d1 = d1 + (t * t) * dw;
            t = P2[i1 + pp] - P2[i0 + pp];
            d2 = d2 + (t * t) * dw;
        }
        d0 = d0 * a.mult[0];
        d1 = d1 * a.mult[1];
        d2 = d2 * a.mult[2];
        if (!a.independent) {
            const float ds = ((d0 + d1) + d2) / 3.f;
            const float w = weight_of<WFN>(ds);
            fv0 = fv0 + w * a.R[0][i1];
            fv1 = fv1 + w * a.R[1][i1];
            fv2 = fv2 + w * a.R[2][i1];
            fw0 = fw0 + w;
            wm0 = w > wm0 ? w : wm0;
        } else {
            const float w0 = weight_of<WFN>(d0), w1 = weight_of<WFN>(d1), w2 = weight_of<WFN>(d2);
            fv0 = fv0 + w0 * a.R[0][i1];
            fv1 = fv1 + w1 * a.R[1][i1];
            fv2 = fv2 + w2 * a.R[2][i1];
            fw0 = fw0 + w0;
            fw1 = fw1 + w1;
            fw2 = fw2 + w2;
            wm0 = w0 > wm0 ? w0 : wm0;
            wm1 = w1 > wm1 ? w1 : wm1;
            wm2 = w2 > wm2 ? w2 : wm2;
        }
    }
    const float r0 = a.R[0][i0], r1 = a.R[1][i0], r2 = a.R[2][i0];
    float o0 = r0, o1 = r1, o2 = r2;
    if (!a.independent) {
        if (wm0 > 0.f) {
            fv0 = fv0 + wm0 * r0;
            fv1 = fv1 + wm0 * r1;
            fv2 = fv2 + wm0 * r2;
            fw0 = fw0 + wm0;
            o0 = fv0 / fw0;
            o1 = fv1 / fw0;
            o2 = fv2 / fw0;
        }
    } else {
        if (wm0 > 0.f) o0 = fv0 / fw0;
        if (wm1 > 0.f) o1 = fv1 / fw1;
        if (wm2 > 0.f) o2 = fv2 / fw2;
    }
    a.out[0][idx] = o0;
    a.out[1][idx] = o1;
    a.out[2][idx] = o2;
}

// x / 3, correctly rounded: the product with the rounded reciprocal and one
// correction with the exact fused remainder (only -0 gives +0, which weighs
// alike; selftest_third_kernel checks every float), about half the
// instructions of a general division; infinities stay as they are.
__device__ __forceinline__ float third(float x)
{
    constexpr float r3 = 1.f / 3.f;
    const float q = x * r3;
    const float e = __builtin_fmaf(-3.f, q, x);
    const float c = __builtin_fmaf(e, r3, q);
    return __builtin_fabsf(x) < __builtin_inff() ? c : q;
}

// The same filter on 32x64 tiles for disks of radius 1 to 3: per offset the
// squares of the three channels are staged together, and every thread sums
// three stencils of a 4-pixel run and shares one weight (or takes three).  The
// kernel above gathers two values per tap, channel and offset from global
// memory: 2.71 ms a pass on 1200x900 at r = 1 and 316 offsets, 0.98 ms here
// (vector issue: three times the tap and staging work of the grey kernel per
// weight; 1.1 rounds of workgroups at that size).
template <class PT>
struct RgbTile {
    using T = Tile<PT>;
    static constexpr int NCHUNK = 3 * T::NCHUNK;
    static constexpr int CPT = (NCHUNK + NTF - 1) / NTF;
    static constexpr int LDS = CPT * NTF * 4;
};
struct RgbTiledArgs {
    RgbArgs f;
    int ntx;
    float wc[kMaxClasses];
};

template <class PT, int WFN, bool INDEP>
__global__ __launch_bounds__(NTF) __attribute__((amdgpu_waves_per_eu(4, 4))) void filter_rgb_tiled_fp32(RgbTiledArgs a)
{
    using T = Tile<PT>;
    using RT = RgbTile<PT>;
    static_assert(T::TZ == 1, "one slice");
    __shared__ __attribute__((aligned(16))) float lds[2][RT::LDS];
    const int t = threadIdx.x;
    const int wg = xcd_swizzle(blockIdx.x, gridDim.x);
    const int X0 = (wg % a.ntx) * TX, Y0 = (wg / a.ntx) * T::TY;
    const FilterGeom g = a.f.g;
    const float w0 = a.wc[0];

    const float *pc[RT::CPT];
    float p0[RT::CPT][4];
#pragma unroll
    for (int c = 0; c < RT::CPT; c++) {
        const int ci = t + c * NTF < RT::NCHUNK ? t + c * NTF : 0;  // slots past the region repeat chunk 0
        const int ch = ci / T::NCHUNK, row = ci % T::NCHUNK / T::CPR, cx = ci % T::CPR;
        const float *P = ch == 0 ? a.f.P[0] : ch == 1 ? a.f.P[1] : a.f.P[2];
        pc[c] = P + ((long)(Y0 + g.py - PT::RY + row) * g.nxp + (X0 + g.px - T::O + 4 * cx));
        __builtin_memcpy(p0[c], pc[c], 16);
    }
    const int cell = kLaneCell[t & 63];
    const int xr = cell & 7, ty = (cell >> 3) + 8 * (t >> 6);
    const int x0 = X0 + VX * xr, y = Y0 + ty;
    const long at = (long)(y + g.py) * g.nxp + (x0 + g.px);
    const float *R0 = a.f.R[0] + at, *R1 = a.f.R[1] + at, *R2 = a.f.R[2] + at;
    constexpr int NWT = INDEP ? 3 : 1;
    float fv[3][VX], fw[NWT][VX], wm[NWT][VX];
#pragma unroll
    for (int v = 0; v < VX; v++) {
#pragma unroll
        for (int c = 0; c < 3; c++) fv[c][v] = 0.f;
#pragma unroll
        for (int c = 0; c < NWT; c++) fw[c][v] = wm[c][v] = 0.f;
    }
    const int ldsrow = (ty + PT::RY) * T::PITCH + VX * xr;
    const int nS = a.f.n_search;
    auto load_chunks = [&](float (&pn)[RT::CPT][4], int lin) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < RT::CPT; c++) __builtin_memcpy(pn[c], pc[c] + lin, 16);
    };
    auto stage = [&](const float (&pn)[RT::CPT][4], float *buf) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < RT::CPT; c++) {
            float dv[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float q = pn[c][e] - p0[c][e];
                dv[e] = q * q;
                if constexpr (PT::kUniform) dv[e] = dv[e] * w0;
            }
            __builtin_memcpy(__builtin_assume_aligned(buf + 4 * (t + c * NTF), 16), dv, 16);
        }
    };
    auto lin_at = [&](int k) __attribute__((always_inline)) { return a.f.search[k < nS ? k : nS - 1].lin; };
    int linv = 0, kb = 0;
    auto step = [&](int k, const float *rd, float *wr) __attribute__((always_inline)) {
        const int l0 = __builtin_amdgcn_readlane(linv, k - kb);
        float rs[3][VX], pn[RT::CPT][4], d[3][VX];
        __builtin_memcpy(rs[0], R0 + l0, 16);
        __builtin_memcpy(rs[1], R1 + l0, 16);
        __builtin_memcpy(rs[2], R2 + l0, 16);
        load_chunks(pn, __builtin_amdgcn_readlane(linv, k + 1 - kb));
#pragma unroll
        for (int c = 0; c < 3; c++) {
            patch_sums<PT>(rd + c * T::NCHUNK * 4 + ldsrow, a.wc, d[c]);
#pragma unroll
            for (int v = 0; v < VX; v++) d[c][v] = d[c][v] * a.f.mult[c];
        }
#pragma unroll
        for (int v = 0; v < VX; v++) {
            float w[NWT];
            if constexpr (INDEP) {
#pragma unroll
                for (int c = 0; c < NWT; c++) w[c] = weight_of<WFN>(d[c][v]);
            } else {
                w[0] = weight_of<WFN>(third((d[0][v] + d[1][v]) + d[2][v]));
            }
#pragma unroll
            for (int c = 0; c < 3; c++) fv[c][v] = fv[c][v] + w[INDEP ? c : 0] * rs[c][v];
#pragma unroll
            for (int c = 0; c < NWT; c++) {
                fw[c][v] = fw[c][v] + w[c];
                wm[c][v] = w[c] > wm[c][v] ? w[c] : wm[c][v];
            }
        }
        __builtin_amdgcn_sched_barrier(0);  // the chunks are in flight until here
        stage(pn, wr);
        __syncthreads();
    };
    {
        float pn[RT::CPT][4];
        load_chunks(pn, lin_at(0));
        stage(pn, lds[0]);
    }
    __syncthreads();
    constexpr int kBlock = 62;  // even; a step looks one offset ahead
    for (kb = 0; kb < nS; kb += kBlock) {
        linv = lin_at(kb + (t & 63));
        const int ke = kb + kBlock < nS ? kb + kBlock : nS;
        for (int k = kb; k < ke; k += 2) {
            step(k, lds[0], lds[1]);
            if (k + 1 < ke) step(k + 1, lds[1], lds[0]);
        }
    }
    if (y >= g.ny) return;
#pragma unroll
    for (int v = 0; v < VX; v++) {
        if (x0 + v >= g.nx) continue;
        const long o = (long)y * g.nx + x0 + v;
        const float r[3] = {R0[v], R1[v], R2[v]};
#pragma unroll
        for (int c = 0; c < 3; c++) {
            float res = r[c];
            if constexpr (INDEP) {
                if (wm[c][v] > 0.f) res = fv[c][v] / fw[c][v];
            } else if (wm[0][v] > 0.f) {
                res = (fv[c][v] + wm[0][v] * r[c]) / (fw[0][v] + wm[0][v]);
            }
            a.f.out[c][o] = res;
        }
    }
}

// ---------------------------------------------------------------------------
// Reflective padding (iternlm_prepare.cpp:6-48): mirror without repeating the
// edge, iterated until in range.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(NT) void pad_reflect_kernel(const float *__restrict__ in, float *__restrict__ out,
                                                         FilterGeom g)
{
    const long n = (long)g.nxp * g.nyp * g.nzp;
    const long idx = (long)blockIdx.x * NT + threadIdx.x;
    if (idx >= n) return;
    const int x1 = (int)(idx % g.nxp);
    const int y1 = (int)((idx / g.nxp) % g.nyp);
    const int z1 = (int)(idx / ((long)g.nxp * g.nyp));
    int x = x1 - g.px, y = y1 - g.py, z = z1 - g.pz;
    while (x < 0 || x >= g.nx) x = (x < 0) ? -x : 2 * g.nx - x - 2;
    while (y < 0 || y >= g.ny) y = (y < 0) ? -y : 2 * g.ny - y - 2;
    while (z < 0 || z >= g.nz) z = (z < 0) ? -z : 2 * g.nz - z - 2;
    out[idx] = in[((long)z * g.ny + y) * g.nx + x];
}

// ---------------------------------------------------------------------------
// Anscombe transform of the colour path and its algebraic inverse
// (Color/colorspace.h:87-123): the same float operations as anscombe() and
// inverse_anscombe() on the host, which took 5 of the 15 ms of a 1200x900
// image's call.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(NT) void anscombe_kernel(float *__restrict__ v, long n, int inverse)
{
    const long i = (long)blockIdx.x * NT + threadIdx.x;
    if (i >= n) return;
    const float x = v[i];
    v[i] = inverse ? (x / 2.f) * (x / 2.f) - 3.f / 8.f : 2.f * sqrtf(x + 3.f / 8.f);
}

// ---------------------------------------------------------------------------
// Noise: one wavefront per sample computes the population standard deviation
// of its patchsize x patchsize in-slice patch (noiselevel.cpp:235-283) with
// FP64 two-pass accumulation and a wavefront butterfly reduction.
// ---------------------------------------------------------------------------
__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

__global__ __launch_bounds__(NT) void patchstd_kernel(const float *__restrict__ origin, long row_pitch,
                                                      long slice_pitch, const int64_t *__restrict__ samples,
                                                      long n, int nx, long nslice, int ps, double *__restrict__ out)
{
    const int lane = threadIdx.x & 63;
    const long s = (long)blockIdx.x * (NT / 64) + (threadIdx.x >> 6);
    if (s >= n) return;  // whole wavefront leaves together
    const long idx = samples[s];
    const int z0 = (int)(idx / nslice);
    const int y0 = (int)((idx - z0 * nslice) / nx);
    const int x0 = (int)(idx - z0 * nslice - (long)y0 * nx);
    const float *base = origin + (long)z0 * slice_pitch + (long)y0 * row_pitch + x0;
    const int plen = ps * ps;
    double sum = 0.0;
    for (int i = lane; i < plen; i += 64) sum += (double)base[(long)(i / ps) * row_pitch + (i % ps)];
    const double mean = wave_sum(sum) / (double)plen;
    double sq = 0.0;
    for (int i = lane; i < plen; i += 64) {
        const double dv = (double)base[(long)(i / ps) * row_pitch + (i % ps)] - mean;
        sq += dv * dv;
    }
    const double var = wave_sum(sq) / (double)plen;
    if (lane == 0) out[s] = sqrt(var);
}

// ---------------------------------------------------------------------------
// Two-cluster hard EM (Noise/noiselevel.cpp:366-528) in FP64, one workgroup
// per window of the sample list: the steps of create2clusters, the sums in a
// fixed order over 1024 threads.  An assignment is one sweep over the window
// (values from the L2), the variances about the new means another; the
// assignment is kept as one bit per value in LDS, for the second sweep and for
// the next one's test for a change (a window beyond kClusterWords * 64 values
// derives it again from the parameters it was made with).
//
// p2 > p1 is decided from the difference of the logarithms, a quadratic in the
// value, wherever rounding (bounded for the whole interval in which the wider
// density is far from underflow) cannot reach its sign; the densities
// themselves decide the rest.  FP64 issue on the window's one CU bounds it.  On
// the host one thread took 35 ms for a window of 1e5 samples and 1.1 s for the
// 2 x 256 windows of a 256^3 volume with 2e4 samples; here that is 1.4 ms (0.5
// when spread, below) and 2 x 0.3 ms.
// ---------------------------------------------------------------------------
constexpr int NTC = 1024;
constexpr int kClusterRun = 4;          // 64-value words of a wavefront in flight
constexpr int kClusterWords = 1 << 14;  // at most this many words of bits (128 KB)

struct ClusterParams {
    double m1, m2, v1, v2;  // means and variances
    double a, b, c;         // log p2 - log p1 = (a x + b) x + c, x = v - m1
    double lo, hi, margin;  // the quadratic's sign decides between lo and hi beyond the margin
    bool first;             // the initial assignment: the nearer of m1, m2
};

// a value that is the same in every lane, in scalar registers
__device__ __forceinline__ double uniform(double v)
{
    const unsigned long b = __builtin_bit_cast(unsigned long, v);
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)b), hi = __builtin_amdgcn_readfirstlane((unsigned)(b >> 32));
    return __builtin_bit_cast(double, (unsigned long)hi << 32 | lo);
}
__device__ __forceinline__ unsigned long uniform(unsigned long v)
{
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)v), hi = __builtin_amdgcn_readfirstlane((unsigned)(v >> 32));
    return (unsigned long)hi << 32 | lo;
}

__device__ __forceinline__ ClusterParams cluster_params(double m1, double m2, double v1, double v2)
{
    const double PI = 3.14159265358979323846;
    const double h1 = 1.0 / (2 * v1), h2 = 1.0 / (2 * v2);
    const double k1 = -0.5 * log(v1 * 2 * PI), k2 = -0.5 * log(v2 * 2 * PI), d = m2 - m1;
    ClusterParams p;
    p.m1 = m1;
    p.m2 = m2;
    p.v1 = v1;
    p.v2 = v2;
    p.first = false;
    p.a = h1 - h2;
    p.b = 2 * d * h2;
    p.c = (k2 - k1) - d * d * h2;
    // exponents up to 600 of the wider density; no interval where the factors
    // leave the range in which a density of that exponent is a normal number
    const double h = fmin(h1, h2), r = sqrt(600.0 / h), mid = h1 < h2 ? m1 : m2;
    const bool plain = fabs(k1) < 50.0 && fabs(k2) < 50.0;
    p.lo = plain ? mid - r : 1e308;
    p.hi = plain ? mid + r : -1e308;
    const double x = fmax(fabs(p.lo - m1), fabs(p.hi - m1));
    p.margin = 1e-10 + 1e-12 * (fabs(p.a) * x * x + fabs(p.b) * x + fabs(p.c));
    for (double *q : {&p.a, &p.b, &p.c, &p.lo, &p.hi, &p.margin}) *q = uniform(*q);
    return p;
}

// not inlined: its divisions and exponentials would take the registers of the
// sweeps around it
__device__ __attribute__((noinline)) bool second_cluster_densities(double m1, double v1, double m2, double v2, double v)
{
    const double PI = 3.14159265358979323846;
    const double p1 = 1. / sqrt(v1 * 2 * PI) * exp(-((v - m1) * (v - m1) / (2 * v1)));
    const double p2 = 1. / sqrt(v2 * 2 * PI) * exp(-((v - m2) * (v - m2) / (2 * v2)));
    return p2 > p1;
}
// whether each of kClusterRun values belongs to the second cluster
__device__ __forceinline__ void second_cluster(const ClusterParams &c, const double (&v)[kClusterRun],
                                               bool (&r)[kClusterRun])
{
    if (c.first) {
#pragma unroll
        for (int j = 0; j < kClusterRun; j++) r[j] = !(fabs(v[j] - c.m1) < fabs(v[j] - c.m2));
        return;
    }
    bool ok = true;
#pragma unroll
    for (int j = 0; j < kClusterRun; j++) {
        const double x = v[j] - c.m1;
        const double l = __builtin_fma(__builtin_fma(c.a, x, c.b), x, c.c);
        r[j] = l > 0.0;
        ok = ok && (v[j] == 0.0 || (fabs(l) > c.margin && v[j] > c.lo && v[j] < c.hi));
    }
    if (__builtin_amdgcn_ballot_w64(!ok) == 0) return;
    unsigned m = 0;  // rare: one call in the code
#pragma unroll 1
    for (int j = 0; j < kClusterRun; j++) {
        const double x = j == 0 ? v[0] : j == 1 ? v[1] : j == 2 ? v[2] : v[3];
        m |= (second_cluster_densities(c.m1, c.v1, c.m2, c.v2, x) ? 1u : 0u) << j;
    }
#pragma unroll
    for (int j = 0; j < kClusterRun; j++) r[j] = (m >> j & 1) != 0;
}

// op over the block, the same value in every thread
template <class Op>
__device__ __forceinline__ double block_total(double v, double *sh, Op op)
{
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v = op(v, __shfl_xor(v, o, 64));
    __syncthreads();  // the values of the call before this one have been read
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    double r = sh[0];
    for (int w = 1; w < NTC / 64; w++) r = op(r, sh[w]);
    return uniform(r);
}

// KEPT: the windows' bits fit LDS (n <= 64 kClusterWords)
template <bool KEPT>
__global__ __launch_bounds__(NTC) void cluster_kernel(const double *__restrict__ values, long n,
                                                      const int64_t *__restrict__ bounds, double *__restrict__ out)
{
    extern __shared__ unsigned long bits[];  // the last assignment
    __shared__ double sh[4][NTC / 64];
    __shared__ unsigned long cnt[3][NTC / 64];
    const long fs = bounds ? bounds[2 * blockIdx.x] : 0, ls = bounds ? bounds[2 * blockIdx.x + 1] : n - 1;
    const long nword = (ls - fs + 64) / 64;  // 64-value words of the window (ls >= fs - 1)
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    constexpr int NW = NTC / 64;
    auto add = [](double a, double b) { return a + b; };
    // this lane's value of a word; 0 (never counted) past the window
    auto load = [&](long w, double (&v)[kClusterRun]) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < kClusterRun; j++) {
            const long i = fs + (w + (long)j * NW) * 64 + lane;
            v[j] = i <= ls ? values[i] : 0.0;
        }
    };
    double mn = 1e300, mx = -1e300;
    for (long i = fs + threadIdx.x; i <= ls; i += NTC) {
        const double v = values[i];
        mn = v < mn ? v : mn;
        mx = mx < v ? v : mx;
    }
    mn = block_total(mn, sh[0], [](double a, double b) { return b < a ? b : a; });
    mx = block_total(mx, sh[1], [](double a, double b) { return a < b ? b : a; });
    ClusterParams cur{}, prev{};
    cur.m1 = uniform(mn + 0.25 * (mx - mn));
    cur.m2 = uniform(mx - 0.25 * (mx - mn));
    cur.first = true;
    double m1 = cur.m1, m2 = cur.m2, v1 = 0.0, v2 = 0.0;
    // one assignment: counts, sums and means, then the variances about them
    auto assign = [&](bool test) -> bool {
        double c1 = 0, c2 = 0;
        unsigned long s1 = 0, s2 = 0, diff = 0;
        for (long w = wave; w < nword; w += kClusterRun * NW) {
            double v[kClusterRun];
            bool r[kClusterRun], was[kClusterRun];
            load(w, v);
            second_cluster(cur, v, r);
            if (!KEPT && test) second_cluster(prev, v, was);
#pragma unroll
            for (int j = 0; j < kClusterRun; j++) {
                const long word = w + (long)j * NW;
                const bool in = v[j] != 0.0, b = in && r[j], a = in && !r[j];
                const unsigned long mb = __builtin_amdgcn_ballot_w64(b);
                c1 += a ? v[j] : 0.0;
                c2 += b ? v[j] : 0.0;
                s1 += __builtin_popcountl(__builtin_amdgcn_ballot_w64(a));
                s2 += __builtin_popcountl(mb);
                if constexpr (KEPT) {
                    if (word < nword) {
                        if (test) diff |= uniform(bits[word]) ^ mb;
                        if (lane == 0) bits[word] = mb;
                    }
                } else if (test) {
                    diff |= __builtin_amdgcn_ballot_w64(in && r[j] != was[j]);
                }
            }
        }
        if (lane == 0) {
            cnt[0][wave] = s1;
            cnt[1][wave] = s2;
            cnt[2][wave] = diff;
        }
        c1 = block_total(c1, sh[0], add);  // its barriers also publish cnt
        c2 = block_total(c2, sh[1], add);
        s1 = s2 = diff = 0;
        for (int w = 0; w < NW; w++) {
            s1 += cnt[0][w];
            s2 += cnt[1][w];
            diff |= cnt[2][w];
        }
        if (s1 > 0) m1 = uniform(c1 / (double)s1);
        if (s2 > 0) m2 = uniform(c2 / (double)s2);
        double q1 = 0, q2 = 0;
        for (long w = wave; w < nword; w += kClusterRun * NW) {
            double v[kClusterRun];
            bool r[kClusterRun];
            load(w, v);
            if constexpr (KEPT) {
#pragma unroll
                for (int j = 0; j < kClusterRun; j++) {
                    const long word = w + (long)j * NW;
                    r[j] = word < nword && (bits[word] >> lane & 1) != 0;
                }
            } else {
                second_cluster(cur, v, r);
            }
#pragma unroll
            for (int j = 0; j < kClusterRun; j++) {
                const bool in = v[j] != 0.0;
                const double d = v[j] - (r[j] ? m2 : m1);
                const double d1 = in && !r[j] ? d : 0.0, d2 = in && r[j] ? d : 0.0;
                q1 += d1 * d1;
                q2 += d2 * d2;
            }
        }
        v1 = uniform(block_total(q1, sh[2], add) / fmax(1.0, (double)s1));
        v2 = uniform(block_total(q2, sh[3], add) / fmax(1.0, (double)s2));
        return test ? diff != 0 : s1 > 0 || s2 > 0;
    };
    double mean = 0.0, stdev = 0.0;
    if (assign(false)) {
        bool change = true;
        for (int iters = 1; change && v1 > 0 && v2 > 0; iters++) {
            prev = cur;
            cur = cluster_params(m1, m2, v1, v2);
            change = assign(true);
            if (iters == 1000) break;
        }
        const bool low = m1 <= m2 || v2 <= 0.0;
        mean = low ? m1 : m2;
        stdev = sqrt(low ? v1 : v2);
    }
    if (threadIdx.x == 0) {
        out[2 * blockIdx.x] = mean;
        out[2 * blockIdx.x + 1] = stdev;
    }
}

// One large window over many CUs: the same steps as two launches per
// iteration, each block taking a share of the values and first adding the
// partial sums that the launch before left (in block order, every block the
// same), so nothing is exchanged within a launch.  Launches behind the last
// iteration return at once.
constexpr int kSpreadBlocks = 64;
// From here on one window is spread.  One workgroup takes 0.13 ms for 4096
// samples and 0.52 ms for 16384, in proportion; spread, 16384 take 0.66 ms,
// 32768 take 0.51 ms and 1e5 0.53 ms (two launches an iteration, whatever the
// samples), where one workgroup takes 1.4 ms.
constexpr int64_t kSpreadSamples = 20480;
constexpr int kSpreadBatch = 16;  // iterations between looks at the end (about 20 are common)
constexpr int NTS = 256;
struct ClusterWork {
    ClusterParams params[2];          // of even and odd iterations
    double mean[2];                   // after the last assignment
    double minmax[kSpreadBlocks][2];
    double sums[2][kSpreadBlocks][5]; // c1, c2, s1, s2, changed values; of even and odd iterations
    double squares[kSpreadBlocks][2];
    int done;
};
static_assert(sizeof(ClusterWork) <= kClusterWorkBytes, "the callers' workspace");

// the sums of N columns of per-block partials
template <int N>
__device__ __forceinline__ void add_partials(const double (*p)[N], double (&t)[N])
{
#pragma unroll
    for (int e = 0; e < N; e++) t[e] = 0.0;
    for (int b = 0; b < kSpreadBlocks; b++)
#pragma unroll
        for (int e = 0; e < N; e++) t[e] += p[b][e];
}
// thread 0 gets the block's sums
template <int N>
__device__ __forceinline__ void block_sums(double (&v)[N])
{
    __shared__ double sh[N][NTS / 64];
#pragma unroll
    for (int e = 0; e < N; e++) {
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) v[e] += __shfl_xor(v[e], o, 64);
        if ((threadIdx.x & 63) == 0) sh[e][threadIdx.x >> 6] = v[e];
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < N; e++) v[e] = (sh[e][0] + sh[e][1]) + (sh[e][2] + sh[e][3]);
}
// this thread's next values of the block's share; 0 (never counted) past it
__device__ __forceinline__ void load_share(const double *values, long i, long end, double (&v)[kClusterRun])
{
#pragma unroll
    for (int j = 0; j < kClusterRun; j++) v[j] = i + j * NTS < end ? values[i + j * NTS] : 0.0;
}

__global__ __launch_bounds__(NTS) void spread_minmax_kernel(const double *__restrict__ values, long n, ClusterWork *w)
{
    __shared__ double sh[2][NTS / 64];
    const long end = n * (blockIdx.x + 1) / kSpreadBlocks;
    double mn = 1e300, mx = -1e300;
    for (long i = n * blockIdx.x / kSpreadBlocks + threadIdx.x; i < end; i += NTS) {
        const double v = values[i];
        mn = v < mn ? v : mn;
        mx = mx < v ? v : mx;
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        const double a = __shfl_xor(mn, o, 64), b = __shfl_xor(mx, o, 64);
        mn = a < mn ? a : mn;
        mx = mx < b ? b : mx;
    }
    if ((threadIdx.x & 63) == 0) {
        sh[0][threadIdx.x >> 6] = mn;
        sh[1][threadIdx.x >> 6] = mx;
    }
    __syncthreads();
    if (threadIdx.x != 0) return;
    for (int k = 1; k < NTS / 64; k++) {
        mn = sh[0][k] < mn ? sh[0][k] : mn;
        mx = mx < sh[1][k] ? sh[1][k] : mx;
    }
    w->minmax[blockIdx.x][0] = mn;
    w->minmax[blockIdx.x][1] = mx;
    if (blockIdx.x == 0) w->done = 0;
}

__global__ __launch_bounds__(NTS) void spread_assign_kernel(const double *__restrict__ values, long n, ClusterWork *w,
                                                            int it, double *__restrict__ out)
{
    if (w->done != 0) return;
    ClusterParams cur{}, prev{};
    if (it == 0) {
        double mn = 1e300, mx = -1e300;
        for (int b = 0; b < kSpreadBlocks; b++) {
            mn = w->minmax[b][0] < mn ? w->minmax[b][0] : mn;
            mx = mx < w->minmax[b][1] ? w->minmax[b][1] : mx;
        }
        cur.m1 = mn + 0.25 * (mx - mn);
        cur.m2 = mx - 0.25 * (mx - mn);
        cur.first = true;
    } else {
        double s[5], q[2];
        add_partials(w->sums[(it - 1) & 1], s);
        add_partials(w->squares, q);
        const double m1 = w->mean[0], m2 = w->mean[1], v1 = q[0] / fmax(1.0, s[2]), v2 = q[1] / fmax(1.0, s[3]);
        const bool any = it > 1 || s[2] > 0 || s[3] > 0, change = it == 1 || s[4] > 0;
        if (!any || !change || !(v1 > 0) || !(v2 > 0) || it > 1000) {
            if (blockIdx.x == 0 && threadIdx.x == 0) {
                const bool low = m1 <= m2 || v2 <= 0.0;
                out[0] = any ? (low ? m1 : m2) : 0.0;
                out[1] = any ? sqrt(low ? v1 : v2) : 0.0;
                w->done = 1;
            }
            return;
        }
        prev = w->params[(it - 1) & 1];
        cur = cluster_params(m1, m2, v1, v2);
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) w->params[it & 1] = cur;
    const long end = n * (blockIdx.x + 1) / kSpreadBlocks;
    double s[5] = {0, 0, 0, 0, 0};
    for (long i = n * blockIdx.x / kSpreadBlocks + threadIdx.x; i - (long)threadIdx.x < end; i += kClusterRun * NTS) {
        double v[kClusterRun];
        bool r[kClusterRun], was[kClusterRun];
        load_share(values, i, end, v);
        second_cluster(cur, v, r);
        if (it > 0) second_cluster(prev, v, was);
#pragma unroll
        for (int j = 0; j < kClusterRun; j++) {
            const bool in = v[j] != 0.0;
            s[0] += in && !r[j] ? v[j] : 0.0;
            s[1] += in && r[j] ? v[j] : 0.0;
            s[2] += in && !r[j] ? 1.0 : 0.0;
            s[3] += in && r[j] ? 1.0 : 0.0;
            s[4] += it > 0 && in && r[j] != was[j] ? 1.0 : 0.0;
        }
    }
    block_sums(s);
    if (threadIdx.x == 0)
        for (int e = 0; e < 5; e++) w->sums[it & 1][blockIdx.x][e] = s[e];
}

__global__ __launch_bounds__(NTS) void spread_squares_kernel(const double *__restrict__ values, long n, ClusterWork *w,
                                                             int it)
{
    if (w->done != 0) return;
    const ClusterParams cur = w->params[it & 1];
    double s[5];
    add_partials(w->sums[it & 1], s);
    const double m1 = s[2] > 0 ? s[0] / s[2] : cur.m1, m2 = s[3] > 0 ? s[1] / s[3] : cur.m2;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        w->mean[0] = m1;
        w->mean[1] = m2;
    }
    const long end = n * (blockIdx.x + 1) / kSpreadBlocks;
    double q[2] = {0, 0};
    for (long i = n * blockIdx.x / kSpreadBlocks + threadIdx.x; i - (long)threadIdx.x < end; i += kClusterRun * NTS) {
        double v[kClusterRun];
        bool r[kClusterRun];
        load_share(values, i, end, v);
        second_cluster(cur, v, r);
#pragma unroll
        for (int j = 0; j < kClusterRun; j++) {
            const bool in = v[j] != 0.0;
            const double d1 = in && !r[j] ? v[j] - m1 : 0.0, d2 = in && r[j] ? v[j] - m2 : 0.0;
            q[0] += d1 * d1;
            q[1] += d2 * d2;
        }
    }
    block_sums(q);
    if (threadIdx.x == 0)
        for (int e = 0; e < 2; e++) w->squares[blockIdx.x][e] = q[e];
}

// Every negative float from -0 down to the cutoff, as bit patterns
// 0x80000000 + [first, first + count): the Pade weight with the shortened
// division against the same weight with IEEE division.
__global__ __launch_bounds__(NT) void selftest_div_kernel(unsigned first, unsigned count,
                                                          unsigned long long *mismatch, unsigned *example)
{
    const unsigned stride = gridDim.x * NT;
    unsigned bad = 0;
    for (unsigned i = blockIdx.x * NT + threadIdx.x; i < count; i += stride) {
        const float a = __uint_as_float(0x80000000u + first + i);
        const float x = pade_cut<false>(a), y = pade_cut<true>(a);
        if (__float_as_uint(x) != __float_as_uint(y)) {
            bad++;
            *example = 0x80000000u + first + i;
        }
    }
    if (bad) atomicAdd(mismatch, (unsigned long long)bad);
}

// Every float, by bit pattern: the joint colour filter's division by three
// against IEEE division.
__global__ __launch_bounds__(NT) void selftest_third_kernel(unsigned long long *mismatch, unsigned *example)
{
    const unsigned long stride = (unsigned long)gridDim.x * NT;
    unsigned bad = 0;
    for (unsigned long i = (unsigned long)blockIdx.x * NT + threadIdx.x; i < (1ul << 32); i += stride) {
        const float x = __uint_as_float((unsigned)i), got = third(x), want = x / 3.f;
        const bool same = __float_as_uint(got) == __float_as_uint(want) || (got != got && want != want) ||
                          ((unsigned)i == 0x80000000u && got == 0.f);
        if (!same) {
            bad++;
            *example = (unsigned)i;
        }
    }
    if (bad) atomicAdd(mismatch, (unsigned long long)bad);
}

}  // namespace

hipError_t launch_selftest_third(unsigned long long *mismatch, unsigned *example, hipStream_t st)
{
    hipLaunchKernelGGL(selftest_third_kernel, dim3(8192), dim3(NT), 0, st, mismatch, example);
    return hipGetLastError();
}

hipError_t launch_selftest_div(unsigned first, unsigned count, unsigned long long *mismatch, unsigned *example,
                               hipStream_t st)
{
    hipLaunchKernelGGL(selftest_div_kernel, dim3(8192), dim3(NT), 0, st, first, count, mismatch, example);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Host launchers
// ---------------------------------------------------------------------------
// Per-class weights of the tiled kernel; false when two taps of one class
// carry different weights (then the per-voxel kernel must run).
template <class PT>
static bool class_weights(const int *dxyz, const float *w, int n, float *wc)
{
    bool seen[kMaxClasses] = {};
    for (int i = 0; i < n; i++) {
        const int c = PT::rows.class_of(dxyz[3 * i], dxyz[3 * i + 1], dxyz[3 * i + 2]);
        if (c < 0) return false;
        if (!seen[c]) {
            wc[c] = w[i];
            seen[c] = true;
        } else if (__builtin_memcmp(&wc[c], &w[i], sizeof(float)) != 0)
            return false;
        if (PT::kUniform && __builtin_memcmp(&w[0], &w[i], sizeof(float)) != 0) return false;
    }
    return true;
}

// Whether the kernel of this shape sums exactly these taps in this order.
template <class PT>
static bool taps_match(const int *dxyz, const float *w, int n)
{
    constexpr const auto &rows = PT::rows;
    if (n != rows.ntaps) return false;
    if (dxyz[0] != 0 || dxyz[1] != 0 || dxyz[2] != 0) return false;
    for (int ri = 0; ri < rows.n; ri++) {
        const Row rw = rows.r[ri];
        int tap = rw.tap0;
        for (int dx = -rw.j; dx <= rw.j; dx++) {
            if (rw.dz == 0 && rw.dy == 0 && dx == 0) continue;
            if (dxyz[3 * tap] != dx || dxyz[3 * tap + 1] != rw.dy || dxyz[3 * tap + 2] != rw.dz) return false;
            tap++;
        }
    }
    float wc[kMaxClasses];
    return class_weights<PT>(dxyz, w, n, wc);
}

// The patch shapes with a tiled kernel: radii as rx * 100 + ry * 10 + rz.
// The isotropic ones, those the reference has kernels for
// (iternlm_cpu_kernels.cpp), and the disks of a single slice.
#define INLM_TILED_SHAPES(X)                                                             \
    X(1, 1, 1) X(2, 2, 2) X(3, 3, 3) X(1, 1, 2) X(1, 1, 3) X(2, 2, 1) X(3, 3, 1) X(3, 3, 2) \
    X(1, 1, 0) X(2, 2, 0) X(3, 3, 0)

int tiled_shape(const int rp[3], const int *dxyz, const float *w, int n)
{
#define INLM_SHAPE(RX, RY, RZ)                                                                       \
    if (rp[0] == RX && rp[1] == RY && rp[2] == RZ)                                                    \
        return taps_match<Patch<RX, RY, RZ>>(dxyz, w, n) ? RX * 100 + RY * 10 + RZ : 0;
    INLM_TILED_SHAPES(INLM_SHAPE)
#undef INLM_SHAPE
    return 0;
}

// Tiles compute whole, so a volume thinner than its tiles pays for the rest;
// the per-voxel kernel does not.  Per-voxel against tiled, us:
//   221 of 1024x1024x2 (a quarter of each tile) 2109 / 2028, 332 of it 11032 /
//   5295; 220 of 256 slices of 1024x16 3501 / 3442, of 1024x8 (an eighth) 1835
//   / 3420; 330 of 1024x8 3757 / 5228.  Up to 512 tiles the waste costs
//   nothing, they run at once: 220 of 64 slices of 256x8 280 / 254.  Narrow
//   rows cost the per-voxel kernel as much: 220 of 64 slices of 2x4096 4734 /
//   1666.
//   The five taps of 110 leave the tiles less to share: 1024x16 1589 / 2413,
//   1024x32 3047 / 2420, 512 slices of 8x64 136 / 186, of 16x64 206 / 186, one
//   slice of 300x300 52.4 / 54.4, of 512x512 60.0 / 54.2.
bool tiled_pays(int shape, int nx, int ny, int nz)
{
    const int rx = shape / 100, ry = shape / 10 % 10, rz = shape % 10;
    if (rx == ry && rx == rz) return true;  // 32x8x8 tiles at every size
    const int tz = rz == 0 ? 1 : 8, ty = rz == 0 ? 64 : 8;
    auto tiles = [](long n, long t) { return (n + t - 1) / t; };
    auto fill = [&](long n, long t) { return (double)n / (double)(tiles(n, t) * t); };
    if (shape == 110) return (long)nx * ny * nz >= (1L << 17) && fill(nx, TX) >= 0.4 && fill(ny, ty) >= 0.4;
    return tiles(nx, TX) * tiles(ny, ty) * tiles(nz, tz) <= 512 || fill(ny, ty) * fill(nz, tz) >= 0.2;
}

hipError_t launch_pad_reflect(const float *in, float *out, const FilterGeom &g, hipStream_t st)
{
    const long n = (long)g.nxp * g.nyp * g.nzp;
    const unsigned blocks = (unsigned)((n + NT - 1) / NT);
    hipLaunchKernelGGL(pad_reflect_kernel, dim3(blocks), dim3(NT), 0, st, in, out, g);
    return hipGetLastError();
}

hipError_t launch_anscombe(float *v, long n, bool inverse, hipStream_t st)
{
    hipLaunchKernelGGL(anscombe_kernel, dim3((unsigned)((n + NT - 1) / NT)), dim3(NT), 0, st, v, n, inverse ? 1 : 0);
    return hipGetLastError();
}

template <class PT, int WFN>
static hipError_t launch_tiled(const float *Rv, const float *P, float *out, const float *sigma, float beta,
                               const SearchEntry *search, int n_search, const TapTable &taps, const FilterGeom &g,
                               float *mass, hipStream_t st)
{
    using T = Tile<PT>;
    TiledArgs a;
    a.mass = mass;
    a.R = Rv;
    a.P = P;
    a.out = out;
    a.sigma = sigma;
    a.search = search;
    a.n_search = n_search;
    a.beta = beta;
    a.g = g;
    a.ntx = (g.nx + TX - 1) / TX;
    a.nty = (g.ny + T::TY - 1) / T::TY;
    a.ntz = (g.nz + T::TZ - 1) / T::TZ;
    for (int i = 0; i < kMaxClasses; i++) a.wc[i] = 0.f;
    if (!class_weights<PT>(taps.dxyz, taps.w, taps.n, a.wc)) return hipErrorInvalidValue;
    const dim3 grid((unsigned)((long)a.ntx * a.nty * a.ntz)), block(NTF);
    if constexpr (PT::RX == PT::RY && PT::RX == PT::RZ) {
        if (mass) {
            hipLaunchKernelGGL((filter_tiled_fp32<PT, WFN, true>), grid, block, 0, st, a);
            return hipGetLastError();
        }
    }
    if (mass) return hipErrorInvalidValue;  // weight mass: isotropic patches, 32x8x8 tiles
    hipLaunchKernelGGL((filter_tiled_fp32<PT, WFN, false>), grid, block, 0, st, a);
    return hipGetLastError();
}

template <int WFN>
static hipError_t launch_pervoxel(const float *Rv, const float *P, float *out, const float *sigma, float beta,
                                  const SearchEntry *search, int n_search, const TapTable &taps,
                                  const FilterGeom &g, hipStream_t st)
{
    VoxelArgs a;
    a.R = Rv;
    a.P = P;
    a.out = out;
    a.sigma = sigma;
    a.search = search;
    a.n_search = n_search;
    a.beta = beta;
    a.g = g;
    a.taps = taps;
    const long n = (long)g.nx * g.ny * g.nz;
    hipLaunchKernelGGL((filter_pervoxel_fp32<WFN>), dim3((unsigned)((n + NT - 1) / NT)), dim3(NT), 0, st, a);
    return hipGetLastError();
}

template <class PT>
static hipError_t launch_rgb_tiled(int weight_fn, const RgbArgs &f, const TapTable &taps, hipStream_t st)
{
    using T = Tile<PT>;
    RgbTiledArgs a;
    a.f = f;
    a.ntx = (f.g.nx + TX - 1) / TX;
    for (int i = 0; i < kMaxClasses; i++) a.wc[i] = 0.f;
    if (!class_weights<PT>(taps.dxyz, taps.w, taps.n, a.wc)) return hipErrorInvalidValue;
    const dim3 grid((unsigned)((long)a.ntx * ((f.g.ny + T::TY - 1) / T::TY))), block(NTF);
    if (weight_fn == 0 && !f.independent) hipLaunchKernelGGL((filter_rgb_tiled_fp32<PT, 0, false>), grid, block, 0, st, a);
    else if (weight_fn == 0) hipLaunchKernelGGL((filter_rgb_tiled_fp32<PT, 0, true>), grid, block, 0, st, a);
    else if (!f.independent) hipLaunchKernelGGL((filter_rgb_tiled_fp32<PT, 1, false>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((filter_rgb_tiled_fp32<PT, 1, true>), grid, block, 0, st, a);
    return hipGetLastError();
}

hipError_t launch_filter_rgb(int shape, int weight_fn, const float *const R[3], const float *const P[3],
                             float *const out[3], const float mult[3], int independent, const SearchEntry *search,
                             int n_search, const TapTable &taps, const FilterGeom &g, hipStream_t st)
{
    RgbArgs a;
    for (int c = 0; c < 3; c++) {
        a.R[c] = R[c];
        a.P[c] = P[c];
        a.out[c] = out[c];
        a.mult[c] = mult[c];
    }
    a.search = search;
    a.n_search = n_search;
    a.independent = independent;
    a.g = g;
    a.taps = taps;
    // Few tiles leave each step's latency to show, which the three weights of
    // independent channels lengthen: a call of four iterations and 316 offsets
    // without noise estimate, us per pixel against tiled, joint (independent):
    //   110: 64x64 1376 / 1709 (1429 / 2280), 256x200 1608 / 1813 (1660 / 2385),
    //     4096x20 2010 / 1848 (2066 / 2400)
    //   220: 64x64 2704 / 2453 (2785 / 3140), 256x200 3261 / 2600 (3265 / 3268)
    //   330: 64x64 5.3 / 4.0 ms (5445 / 5683), 160x160 5.9 / 4.1 ms (5986 / 5710)
    const long pixels = (long)g.nx * g.ny;
    const long few = shape == 110 ? (independent ? 98304 : 65536) : !independent ? 0 : shape == 220 ? 32768 : 20480;
    if (g.nz == 1 && pixels >= few) {
        switch (shape) {
        case 110: return launch_rgb_tiled<Patch<1, 1, 0>>(weight_fn, a, taps, st);
        case 220: return launch_rgb_tiled<Patch<2, 2, 0>>(weight_fn, a, taps, st);
        case 330: return launch_rgb_tiled<Patch<3, 3, 0>>(weight_fn, a, taps, st);
        default: break;
        }
    }
    const long n = (long)g.nx * g.ny * g.nz;
    const dim3 grid((unsigned)((n + NT - 1) / NT)), block(NT);
    if (weight_fn == 0) hipLaunchKernelGGL((filter_rgb_fp32<0>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((filter_rgb_fp32<1>), grid, block, 0, st, a);
    return hipGetLastError();
}

hipError_t launch_filter(int form, int shape, int weight_fn, const float *R, const float *P, float *out,
                         const float *sigma, float beta, const SearchEntry *search, int n_search,
                         const TapTable &taps, const FilterGeom &g, hipStream_t st, float *mass)
{
    if (form != FORM_FP32) return hipErrorInvalidValue;
    switch (shape) {
#define INLM_SHAPE(RX, RY, RZ)                                                                                 \
    case RX * 100 + RY * 10 + RZ:                                                                              \
        return weight_fn == 0 ? launch_tiled<Patch<RX, RY, RZ>, 0>(R, P, out, sigma, beta, search, n_search, taps, \
                                                                   g, mass, st)                               \
                              : launch_tiled<Patch<RX, RY, RZ>, 1>(R, P, out, sigma, beta, search, n_search, taps, \
                                                                   g, mass, st);
        INLM_TILED_SHAPES(INLM_SHAPE)
#undef INLM_SHAPE
    default: break;
    }
    if (mass) return hipErrorInvalidValue;  // weight mass needs the tiled kernel
    return weight_fn == 0 ? launch_pervoxel<0>(R, P, out, sigma, beta, search, n_search, taps, g, st)
                          : launch_pervoxel<1>(R, P, out, sigma, beta, search, n_search, taps, g, st);
}

hipError_t launch_patchstd(const float *origin, int64_t row_pitch, int64_t slice_pitch, const int64_t *samples,
                           int64_t n, int nx, int64_t nslice, int patchsize, double *out, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    const unsigned blocks = (unsigned)((n + (NT / 64) - 1) / (NT / 64));
    hipLaunchKernelGGL(patchstd_kernel, dim3(blocks), dim3(NT), 0, st, origin, (long)row_pitch, (long)slice_pitch,
                       samples, (long)n, nx, (long)nslice, patchsize, out);
    return hipGetLastError();
}

hipError_t launch_clusters(const double *values, int64_t n, const int64_t *bounds, int nwin, double *out, void *work,
                           hipStream_t st)
{
    if (nwin < 1 || n < 1) return hipErrorInvalidValue;
    if (nwin == 1 && !bounds && work && n >= kSpreadSamples) {
        ClusterWork *w = static_cast<ClusterWork *>(work);
        hipLaunchKernelGGL(spread_minmax_kernel, dim3(kSpreadBlocks), dim3(NTS), 0, st, values, (long)n, w);
        for (int it = 0, done = 0; done == 0 && it <= 1001;) {
            // a batch of iterations, then a look whether the last has come
            for (const int end = std::min(it + kSpreadBatch, 1002); it < end; it++) {
                hipLaunchKernelGGL(spread_assign_kernel, dim3(kSpreadBlocks), dim3(NTS), 0, st, values, (long)n, w, it,
                                   out);
                hipLaunchKernelGGL(spread_squares_kernel, dim3(kSpreadBlocks), dim3(NTS), 0, st, values, (long)n, w, it);
            }
            hipError_t e = hipGetLastError();
            if (e == hipSuccess) e = hipMemcpyAsync(&done, &w->done, sizeof(int), hipMemcpyDeviceToHost, st);
            const hipError_t f = hipStreamSynchronize(st);  // also before `done` goes
            if (e != hipSuccess || f != hipSuccess) return e != hipSuccess ? e : f;
        }
        return hipSuccess;
    }
    if (n > 64L * kClusterWords) {
        hipLaunchKernelGGL(cluster_kernel<false>, dim3((unsigned)nwin), dim3(NTC), 0, st, values, (long)n, bounds, out);
        return hipGetLastError();
    }
    // beyond 64 KB of LDS a kernel has to ask for it
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(cluster_kernel<true>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize,
                                             kClusterWords * (int)sizeof(unsigned long));
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(cluster_kernel<true>, dim3((unsigned)nwin), dim3(NTC),
                       (size_t)((n + 63) / 64) * sizeof(unsigned long), st, values, (long)n, bounds, out);
    return hipGetLastError();
}

}  // namespace inlm
