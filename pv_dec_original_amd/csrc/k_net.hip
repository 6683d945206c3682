// k_net.hip — kernels of the warm-start network and the C ABI of include/pvnet.h (gfx950).
//
// The convolutions are implicit GEMMs on the CDNA4 matrix cores (v_mfma_f32_16x16x32_bf16):
//   forward / input gradient   C[m][n] = sum_k A[m][k] B[k][n],  m = voxel, n = output channel,
//                              k = tap * cin + ci, A gathered from the channels-last activations
//                              with zero padding, B the packed bf16 weights [n][k].
//   weight gradient            C[n][k] = sum_m dy[m][n] x[m + off(tap(k))][ci(k)], split over the
//                              voxels into FP32 partials that a second kernel sums in fixed order.
// Tiles are staged through LDS in rows of 32 k-values (one MFMA depth); the next tile's global
// loads are issued before the current tile's MFMAs so that their latency overlaps the math.
//
// MFMA 16x16x32 bf16 lane layout (64 lanes, g = lane / 16, c = lane % 16):
//   A operand: A[c][8g + j], j = 0..7      B operand: B[8g + j][c]
//   D:         D[4g + e][c], e = 0..3

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <string>
#include <type_traits>

#include "../../include/pvnet.h"
#include "march_plans.hpp"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

namespace {

thread_local std::string g_err;

int fail(int code, const std::string& msg) {
    g_err = msg;
    return code;
}

#define NET_HIP(x)                                                                      \
    do {                                                                                \
        hipError_t e_ = (x);                                                            \
        if (e_ != hipSuccess) return fail(2, std::string(#x) + ": " + hipGetErrorString(e_)); \
    } while (0)

#define NET_LAUNCH()                                                                    \
    do {                                                                                \
        hipError_t e_ = hipGetLastError();                                              \
        if (e_ != hipSuccess) return fail(2, std::string("launch: ") + hipGetErrorString(e_)); \
    } while (0)

constexpr int LP = 40;  // LDS row pitch in bf16 (32 + 8 padding: 80-byte rows)

__device__ __forceinline__ float bf2f(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }

// round to nearest even; NaN stays NaN
__device__ __forceinline__ uint16_t f2bf(float f) {
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

// two floats to bf16, the first in the low half: the conversion instruction rounds as f2bf does (equal on
// all 2^32 inputs, NaN included)
__device__ __forceinline__ uint32_t f2bf_pk(float lo, float hi) {
    const __bf16 v[2] = {(__bf16)lo, (__bf16)hi};
    return *reinterpret_cast<const uint32_t*>(v);
}

// bf16 bit pattern strictly greater than zero (NaN is not)
__device__ __forceinline__ bool bf_pos(uint16_t b) { return (b & 0x8000u) == 0 && b != 0 && b <= 0x7f80u; }

// Workgroups are dispatched to the 8 XCDs round-robin (block b to XCD b % 8), each XCD with its own
// L2.  Neighbouring output tiles share most of their input (the 3x3x3 halo), so block b works on
// tile xcd_tile(b, n): XCD x takes a contiguous run of tiles, and neighbours meet in one L2.
constexpr int NXCD = 8;

__device__ __forceinline__ int xcd_tile(int b, int n) {
    const int q = n / NXCD, r = n % NXCD, x = b % NXCD, i = b / NXCD;
    return (x < r ? x * (q + 1) : r * (q + 1) + (x - r) * q) + i;
}

__device__ __forceinline__ void tap_offset(int ntaps, int tap, int& dz, int& dy, int& dx) {
    if (ntaps == 27) {
        dz = tap / 9 - 1;
        dy = (tap / 3) % 3 - 1;
        dx = tap % 3 - 1;
    } else {
        dz = dy = dx = 0;
    }
}

// Inputs and outputs in two parts.  Input channels 0 .. cup - 1 are `up`, a tensor of half the size in each axis
// (nearest upsampling), the others x; output channels 0 .. c0 - 1 go to y0, the others to y.  All zero: one part.
struct NetParts {
    const uint16_t* up;
    uint16_t* y0;
    int32_t ldu, cup, ldy0, c0;
};

// ---------------------------------------------------------------------------------------------
// forward / input-gradient convolution: block tile 4*WM voxels x BN channels, 4 waves of WM x BN

template <int BN, int WM, bool PARTS = false>
__global__ __launch_bounds__(256) void k_conv_fwd(pvnet_conv a, int M, int K, NetParts pq) {
    constexpr int BM = 4 * WM;
    constexpr int NA = BM / 64;  // A rows loaded per thread and step
    __shared__ __attribute__((aligned(16))) uint16_t As[BM * LP];
    __shared__ __attribute__((aligned(16))) uint16_t Bs[BN * LP];
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const int g = lane >> 4, c16 = lane & 15;
    const int m0 = xcd_tile(blockIdx.x + blockIdx.z * gridDim.x, gridDim.x * gridDim.z) * BM, n0 = blockIdx.y * BN;
    const int d = a.s.d, h = a.s.h, w = a.s.w;

    // load roles: A rows r + 64 i, 8-wide k chunk q; B row bn (if < BN), same chunk.  Per row, a
    // mask of the taps whose neighbour lies in the box and the row's base pointer are set once;
    // the chunk's (tap, channel) advance by 32 k-values per step.
    const int q = t & 3, r = t >> 2, bn = t >> 2;
    uint32_t tmask[NA];
    const uint16_t* rowp[NA];
    int pz[NA], py[NA], px[NA];  // PARTS: the row's box and plane, y, x
    #pragma unroll
    for (int i = 0; i < NA; i++) {
        const int m = m0 + r + 64 * i;
        const int mm = m < M ? m : 0;
        const int xx = mm % w, tq = mm / w, yy = tq % h, zz = (tq / h) % d;
        pz[i] = tq / h, py[i] = yy, px[i] = xx;
        uint32_t mk = 0;
        if (m < M) {
            for (int tp = 0; tp < a.ntaps; tp++) {
                int dz, dy, dx;
                tap_offset(a.ntaps, tp, dz, dy, dx);
                if ((unsigned)(zz + dz) < (unsigned)d && (unsigned)(yy + dy) < (unsigned)h && (unsigned)(xx + dx) < (unsigned)w)
                    mk |= 1u << tp;
            }
        }
        tmask[i] = mk;
        rowp[i] = a.x + (int64_t)mm * a.ldx;
    }
    const bool brow = bn < BN && n0 + bn < a.cout;
    const uint16_t* wp = a.w + (int64_t)(n0 + (brow ? bn : 0)) * a.kpad + q * 8;
    const int nsteps = a.kpad / BK;
    uint4 ra[NA], rb;
    int tap = (q * 8) / a.cin, ci = q * 8 - tap * a.cin;  // chunk of step 0

    auto load = [&](int s) {
        const bool kin = tap < a.ntaps;  // k = s * 32 + 8 q < K
        int dz, dy, dx;
        tap_offset(a.ntaps, kin ? tap : 0, dz, dy, dx);
        const int64_t off = (((int64_t)dz * h + dy) * w + dx) * a.ldx + ci;
        #pragma unroll
        for (int i = 0; i < NA; i++) {
            ra[i] = make_uint4(0, 0, 0, 0);
            const uint16_t* src = rowp[i] + off;
            if constexpr (PARTS) {  // sizes are even where cup > 0: halving box * d + z halves both
                src -= pq.cup;
                if (ci < pq.cup)
                    src = pq.up + ((int64_t)((pz[i] + dz) >> 1) * (h >> 1) + ((py[i] + dy) >> 1)) * (w >> 1) * pq.ldu +
                          (int64_t)((px[i] + dx) >> 1) * pq.ldu + ci;
            }
            if (kin && ((tmask[i] >> tap) & 1u)) ra[i] = *(const uint4*)src;
        }
        rb = make_uint4(0, 0, 0, 0);
        if (brow) rb = *(const uint4*)(wp + s * BK);
        ci += BK;  // the chunk of the next step
        while (ci >= a.cin) {
            ci -= a.cin;
            tap++;
        }
    };

    f32x4 acc[WM / 16][BN / 16];
    #pragma unroll
    for (int i = 0; i < WM / 16; i++)
        for (int j = 0; j < BN / 16; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    load(0);
    for (int s = 0; s < nsteps; s++) {
        #pragma unroll
        for (int i = 0; i < NA; i++) *(uint4*)(As + (r + 64 * i) * LP + q * 8) = ra[i];
        if (bn < BN) *(uint4*)(Bs + bn * LP + q * 8) = rb;
        __syncthreads();
        if (s + 1 < nsteps) load(s + 1);
        bf16x8 af[WM / 16], bfr[BN / 16];
        #pragma unroll
        for (int i = 0; i < WM / 16; i++) af[i] = *(const bf16x8*)(As + (wv * WM + i * 16 + c16) * LP + g * 8);
        #pragma unroll
        for (int j = 0; j < BN / 16; j++) bfr[j] = *(const bf16x8*)(Bs + (j * 16 + c16) * LP + g * 8);
        #pragma unroll
        for (int i = 0; i < WM / 16; i++)
            for (int j = 0; j < BN / 16; j++)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i], bfr[j], acc[i][j], 0, 0, 0);
        __syncthreads();
    }

    const bool relu = a.flags & PVNET_RELU, f32out = a.flags & PVNET_F32OUT;
    #pragma unroll
    for (int i = 0; i < WM / 16; i++)
        for (int j = 0; j < BN / 16; j++) {
            const int n = n0 + j * 16 + c16;
            if (n >= a.cout) continue;
            const float b = a.bias ? a.bias[n] : 0.f;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int m = m0 + wv * WM + i * 16 + g * 4 + e;
                if (m >= M) continue;
                float v = acc[i][j][e] + b;
                if (relu) v = v < 0.f ? 0.f : v;
                if (a.relu_of && !bf_pos(a.relu_of[(int64_t)m * a.ldr + n])) v = 0.f;
                if (PARTS && n < pq.c0)
                    pq.y0[(int64_t)m * pq.ldy0 + n] = f2bf(v);
                else if (PARTS)
                    ((uint16_t*)a.y)[(int64_t)m * a.ldy + n - pq.c0] = f2bf(v);
                else if (f32out)
                    ((float*)a.y)[(int64_t)m * a.ldy + n] = v;
                else
                    ((uint16_t*)a.y)[(int64_t)m * a.ldy + n] = f2bf(v);
            }
        }
}

// ---------------------------------------------------------------------------------------------
// 1x1x1 convolutions with K = cin <= 32, one MFMA k-step: every wave takes PWT tiles of 16
// voxels and feeds the matrix core straight from global memory, with no LDS and no barrier.  Lane
// (c16, g) holds the input channels 8g .. 8g+7 of voxel c16 of a tile (zero beyond cin) and the
// weight row 16 j + c16 at the same k-values: the operands k_conv_fwd stages for the same
// convolution, so the outputs are the same bit for bit.  The weights are the MFMA's A operand, so that a lane holds
// four consecutive channels of one voxel and, where rows allow (vec), reads its mask and writes them at once.  Bound by memory: 8 x 96^3 voxels 16 -> 8 in FP32 and 8 -> 16 with a
// mask 156 us for both (6.4 TB/s of rows), 276 with one channel of four voxels a lane.
constexpr int PWT = 4;

template <int NJ>
__global__ __launch_bounds__(256) void k_conv_pw(pvnet_conv a, int M, bool vec) {
    const int lane = threadIdx.x & 63, g = lane >> 4, c16 = lane & 15;
    const int64_t tile0 = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * PWT;
    bf16x8 wf[NJ];
    float bias[NJ][4];
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        const int n = 16 * j + c16;
        uint4 v = make_uint4(0, 0, 0, 0);
        if (n < a.cout) v = *(const uint4*)(a.w + (int64_t)n * a.kpad + g * 8);
        wf[j] = *reinterpret_cast<const bf16x8*>(&v);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int c = 16 * j + 4 * g + e;
            bias[j][e] = (c < a.cout && a.bias) ? a.bias[c] : 0.f;
        }
    }
    uint4 ra[PWT];
    uint2 mk[PWT][NJ];
#pragma unroll
    for (int i = 0; i < PWT; i++) {
        const int64_t m = (tile0 + i) * 16 + c16;
        ra[i] = make_uint4(0, 0, 0, 0);
        if (m < M && g * 8 < a.cin) ra[i] = *(const uint4*)(a.x + m * a.ldx + g * 8);
        if (vec && a.relu_of) {
#pragma unroll
            for (int j = 0; j < NJ; j++)
                if (m < M && 16 * j + 4 * g < a.cout) mk[i][j] = *(const uint2*)(a.relu_of + m * a.ldr + 16 * j + 4 * g);
        }
    }
    const bool relu = a.flags & PVNET_RELU, f32out = a.flags & PVNET_F32OUT;
#pragma unroll
    for (int i = 0; i < PWT; i++) {
        const int64_t m = (tile0 + i) * 16 + c16;
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            const f32x4 acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[j], *reinterpret_cast<const bf16x8*>(&ra[i]),
                                                                      f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
            const int n = 16 * j + 4 * g;
            if (m >= M || n >= a.cout) continue;
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                v[e] = acc[e] + bias[j][e];
                if (relu) v[e] = v[e] < 0.f ? 0.f : v[e];
            }
            if (vec) {
                if (a.relu_of)
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        if (!bf_pos((uint16_t)((e < 2 ? mk[i][j].x : mk[i][j].y) >> (16 * (e & 1))))) v[e] = 0.f;
                if (f32out) *(float4*)((float*)a.y + m * a.ldy + n) = make_float4(v[0], v[1], v[2], v[3]);
                else *(uint2*)((uint16_t*)a.y + m * a.ldy + n) = make_uint2(f2bf_pk(v[0], v[1]), f2bf_pk(v[2], v[3]));
                continue;
            }
#pragma unroll
            for (int e = 0; e < 4; e++) {
                if (n + e >= a.cout) continue;
                if (a.relu_of && !bf_pos(a.relu_of[m * a.ldr + n + e])) v[e] = 0.f;
                if (f32out) ((float*)a.y)[m * a.ldy + n + e] = v[e];
                else ((uint16_t*)a.y)[m * a.ldy + n + e] = f2bf(v[e]);
            }
        }
    }
}

// ---------------------------------------------------------------------------------------------
// 3x3x3 convolutions on the matrix cores, plane by plane
#include "conv_march.hpp"
#include "wgrad_march.hpp"

// ---------------------------------------------------------------------------------------------
// weight gradient: block tile BN output channels x 64 k-values, reduction over its voxel chunk in
// LDS fills of 128 voxels.  Threads 0..127 each load an 8-voxel x 8-channel block of the gathered
// input (eight 16-byte loads), transpose it in registers and write eight 16-byte LDS rows of 8
// voxels; threads 128.. do the same for dy.  The MFMA reduction index is the voxel.
//
// The input's LDS rows are swizzled: the 16-byte chunk q of row r sits at chunk q ^ ((r >> 3) & 7).
// Eight consecutive x-role lanes write rows 8 kc + c (kc = 0..7) at one chunk, and any 16-byte row
// pitch puts rows eight apart on the same two bank groups (a 4-way conflict); the swizzle spreads
// them over eight, and the MFMA fragment reads (16 rows, one chunk) stay conflict-free.

// 8x8 transpose of bf16: r[i] = row i (8 channels, channel c in 16-bit half c); o[c] = column c
// (rows 0..7 in its halves)
__device__ __forceinline__ void transpose8(const uint4 (&r)[8], uint4 (&o)[8]) {
    const uint32_t* rw = reinterpret_cast<const uint32_t*>(r);
    uint32_t* ow = reinterpret_cast<uint32_t*>(o);
#pragma unroll
    for (int c = 0; c < 8; c++)
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const uint32_t lo = rw[(2 * k) * 4 + (c >> 1)], hi = rw[(2 * k + 1) * 4 + (c >> 1)];
            ow[c * 4 + k] = (c & 1) ? ((lo >> 16) | (hi & 0xffff0000u)) : ((lo & 0xffffu) | (hi << 16));
        }
}

template <int BN, bool PARTS = false>
__global__ __launch_bounds__(256) void k_conv_wgrad(pvnet_wgrad a, int M, int K, int mchunk, NetParts pq, int64_t dboff) {
    constexpr int BMW = 128;  // voxels per LDS fill
    constexpr int PW = BMW + 8;  // LDS row pitch in bf16 (272 bytes)
    __shared__ __attribute__((aligned(16))) uint16_t As[BN * PW];  // dy^T  [n][m]
    __shared__ __attribute__((aligned(16))) uint16_t Bs[64 * PW];  // x^T   [k][m]
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const int g = lane >> 4, c16 = lane & 15;
    const int k0 = blockIdx.x * 64, n0 = blockIdx.y * BN, split = blockIdx.z;
    // voxel numbers are unsigned: those of a fill's end may lie beyond 2^31
    const uint32_t mb = (uint32_t)split * (uint32_t)mchunk, me = min((uint32_t)M, mb + (uint32_t)mchunk);
    const int d = a.s.d, h = a.s.h, w = a.s.w;

    // roles: x blocks (t < 128): voxel group mg, k chunk kc; dy blocks (128 <= t < 128 + 2 BN)
    const bool xrole = t < 128;
    const int u = t - 128;
    const bool drole = !xrole && u < 2 * BN;
    const int mg = xrole ? (t >> 3) : drole ? u / (BN / 8) : 0;
    const int kc = t & 7, nc = drole ? u % (BN / 8) : 0;
    const int k = k0 + kc * 8;
    const bool kin = xrole && k < K;
    const int tap = kin ? k / a.cin : 0;
    const int ci = k - tap * a.cin;
    int dz, dy, dx;
    tap_offset(a.ntaps, tap, dz, dy, dx);
    const int64_t off = ((int64_t)dz * h + dy) * w + dx;
    const bool dcol = drole && n0 + nc * 8 < a.cout;

    f32x4 acc[BN / 16];
    for (int j = 0; j < BN / 16; j++) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    // the bias gradient: dy against ones, in the blocks of the first k-values, wave j taking the 16 channels j (a launch
    // of column sums before, 3.7 us: 4000 x 80 -> 32 pointwise, all three passes 32.1 -> 29.1 us).  One accumulator a
    // wave, and the ones made where they are used: with all four accumulators in one wave the kernel had 162 registers
    // instead of 104 (8 x 24^3, 27 taps, 64 -> 64: 139 us, 108 so; 224 -> 64: 426 and 332).
    const int bj = dboff >= 0 && blockIdx.x == 0 ? __builtin_amdgcn_readfirstlane(wv) : -1;
    f32x4 accb = f32x4{0.f, 0.f, 0.f, 0.f};

    uint4 r[8];
    auto load = [&](uint32_t mbase) {
        const uint32_t m0 = mbase + mg * 8;
        if (xrole) {
            const uint32_t tq = m0 / (uint32_t)w;
            int x = m0 % (uint32_t)w, y = tq % (uint32_t)h, z = (tq / (uint32_t)h) % (uint32_t)d;
            const bool up = PARTS && ci < pq.cup;
            int bz = (int)(tq / (uint32_t)h) - z;  // planes of the boxes before
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const uint32_t m = m0 + i;
                const int z2 = z + dz, y2 = y + dy, x2 = x + dx;
                const bool in = kin && m < me && (unsigned)z2 < (unsigned)d && (unsigned)y2 < (unsigned)h &&
                                (unsigned)x2 < (unsigned)w;
                r[i] = make_uint4(0, 0, 0, 0);
                if (in && up)
                    r[i] = *(const uint4*)(pq.up + (((int64_t)((bz + z2) >> 1) * (h >> 1) + (y2 >> 1)) * (w >> 1) + (x2 >> 1)) * pq.ldu + ci);
                else if (in)
                    r[i] = *(const uint4*)(a.x + ((int64_t)m + off) * a.ldx + ci - (PARTS ? pq.cup : 0));
                if (++x == w) {  // next voxel
                    x = 0;
                    if (++y == h) {
                        y = 0;
                        if (++z == d) z = 0, bz += d;
                    }
                }
            }
        } else {
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const uint32_t m = m0 + i;
                r[i] = make_uint4(0, 0, 0, 0);
                if (dcol && m < me) r[i] = *(const uint4*)(a.dy + (int64_t)m * a.lddy + n0 + nc * 8);
            }
        }
    };

    if (mb < me) load(mb);
    for (uint32_t mbase = mb; mbase < me; mbase += BMW) {
        if (xrole || drole) {
            uint4 o[8];
            transpose8(r, o);
            uint16_t* dst = xrole ? Bs + (kc * 8) * PW + (mg ^ kc) * 8 : As + (nc * 8) * PW + mg * 8;
#pragma unroll
            for (int c = 0; c < 8; c++) *(uint4*)(dst + c * PW) = o[c];
        }
        __syncthreads();
        if (mbase + BMW < me) load(mbase + BMW);
#pragma unroll
        for (int kk = 0; kk < BMW / 32; kk++) {
            const int brow = wv * 16 + c16;
            const bf16x8 bx = *(const bf16x8*)(Bs + brow * PW + ((kk * 4 + g) ^ ((brow >> 3) & 7)) * 8);
#pragma unroll
            for (int j = 0; j < BN / 16; j++) {
                const bf16x8 ad = *(const bf16x8*)(As + (j * 16 + c16) * PW + kk * 32 + g * 8);
                acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ad, bx, acc[j], 0, 0, 0);
                if (j == bj) {
                    uint4 ones = make_uint4(0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u);
                    asm volatile("" : "+v"(ones.x), "+v"(ones.y), "+v"(ones.z), "+v"(ones.w));  // not kept through the loop
                    accb = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ad, *reinterpret_cast<const bf16x8*>(&ones), accb, 0, 0, 0);
                }
            }
        }
        __syncthreads();
    }
    if (bj >= 0 && bj < BN / 16 && c16 == 0)  // every column holds the sum of its row's channel
        for (int e = 0; e < 4; e++) {
            const int n = n0 + bj * 16 + g * 4 + e;
            if (n < a.cout) a.ws[dboff + (int64_t)split * a.cout + n] = accb[e];
        }

    const int kk = k0 + wv * 16 + c16;
    if (kk >= K) return;
    for (int j = 0; j < BN / 16; j++)
        for (int e = 0; e < 4; e++) {
            const int n = n0 + j * 16 + g * 4 + e;
            if (n < a.cout) a.ws[((int64_t)split * a.cout + n) * K + kk] = acc[j][e];
        }
}

// dst[i] = sum_s src[s * len + i] in a fixed order: a block takes 16 columns, its 16 row groups
// sum the rows rg, rg + 16, ... in ascending order, and the 16 partials are added in ascending rg.  Bound
// by the latency of a row group's loads where the splits are many and the columns few: eight of them are in
// flight (768 splits of 6912 columns 16.9 us with one, 8.5 with eight; the order of the sum is the same).  The
// partials are summed in 64 bits: the rounding left is that of the partials' own chains and of the result.
constexpr int SUM_COLS = 16;

// One reduction of split partials: dst[(i / rowlen) ldd + i % rowlen] = sum_s src[s len + i].
struct SumJob {
    const float* src;
    float* dst;
    int64_t len, ldd, rowlen;
    int nsplit;
    int blocks;  // blocks_for(len, SUM_COLS)
};

// dw[n][k] over the voxels m0, m0 + 16, .. whose neighbour lies in the box
__device__ double wgrad_pairs(const pvnet_wgrad& a, const NetParts& q, int64_t i, uint32_t m0) {
    const int K = a.ntaps * a.cin, n = (int)(i / K), k = (int)(i - (int64_t)n * K), ci = k % a.cin;
    const uint32_t w = a.s.w, h = a.s.h, d = a.s.d, M = (uint32_t)a.s.nb * d * h * w;
    int dz, dy, dx;
    tap_offset(a.ntaps, k / a.cin, dz, dy, dx);
    double s = 0.0;
    for (uint32_t m = m0; m < M; m += 16) {
        const uint32_t row = m / w, pl = row / h, b = pl / d;
        const int x = (int)(m - row * w) + dx, y = (int)(row - pl * h) + dy, z = (int)(pl - b * d) + dz;
        if ((unsigned)x >= w || (unsigned)y >= h || (unsigned)z >= d) continue;
        const uint16_t v = ci < q.cup ? q.up[(((int64_t)(b * (d >> 1) + (z >> 1)) * (h >> 1) + (y >> 1)) * (w >> 1) + (x >> 1)) * q.ldu + ci]
                                      : a.x[(((int64_t)(b * d + z) * h + y) * w + x) * a.ldx + ci - q.cup];
        s += (double)bf2f(a.dy[(int64_t)m * a.lddy + n]) * (double)bf2f(v);
        if (s != s) break;
    }
    return s;
}

// Two reductions in one launch (the weight and bias gradients of a layer): blocks below
// a.blocks take job a, the others job b, each summing exactly as alone.
// REDO: the sums of the marching kernel, which hold every x also against the zeros around dy's box.  While x is finite
// that adds nothing; a column that is not finite is summed again over the pairs inside the box alone, in 64 bits.  A pass
// over x and dy for each 16 columns then, which ends where a sum is NaN; without, 0.1 to 2 us a call for looking (64 -> 64
// on 8 x 24^3 and 160 -> 160 on 480 voxels; a second body in the marching kernel cost that 2 to 9 %, for registers).
struct SumArgs {
    SumJob a, b;
    pvnet_wgrad g;
    NetParts q;
};

template <bool REDO>
__global__ __launch_bounds__(256, 8) void k_sum_splits(const SumArgs args) {
    const SumJob &a = args.a, &b = args.b;
    __shared__ double sp[16][SUM_COLS + 1];
    __shared__ uint32_t again[4];
    const bool second = (int)blockIdx.x >= a.blocks;
    const float* src = second ? b.src : a.src;
    float* dst = second ? b.dst : a.dst;
    const int64_t len = second ? b.len : a.len, ldd = second ? b.ldd : a.ldd, rowlen = second ? b.rowlen : a.rowlen;
    const int nsplit = second ? b.nsplit : a.nsplit;
    const int blk = second ? (int)blockIdx.x - a.blocks : (int)blockIdx.x;
    const int t = threadIdx.x, col = t % SUM_COLS, rg = t / SUM_COLS;
    const int64_t i = (int64_t)blk * SUM_COLS + col;
    double s = 0.0;
    if (i < len) {
#pragma unroll 8
        for (int p = rg; p < nsplit; p += 16) s += (double)src[(int64_t)p * len + i];
    }
    sp[rg][col] = s;
    if (REDO) again[t >> 6] = __any(!(fabs(s) < __builtin_inf()));
    __syncthreads();
    if (t < SUM_COLS && i < len) {
        double acc = 0.0;
        for (int k = 0; k < 16; k++) acc += sp[k][t];
        dst[(i / rowlen) * ldd + i % rowlen] = (float)acc;
    }
    if constexpr (REDO) {
        if (second || !(again[0] | again[1] | again[2] | again[3])) return;
        __syncthreads();
        // read anew: the launch's other arguments are not loaded unless they are needed
        auto* rest = (__attribute__((address_space(4))) const SumArgs*)__builtin_amdgcn_kernarg_segment_ptr();
        asm volatile("" : "+s"(rest));
        sp[rg][col] = i < len ? wgrad_pairs(*(const pvnet_wgrad*)&rest->g, *(const NetParts*)&rest->q, i, (uint32_t)rg) : 0.0;
        __syncthreads();
        if (t < SUM_COLS && i < len) {
            double acc = 0.0;
            for (int k = 0; k < 16; k++) acc += sp[k][t];
            dst[(i / rowlen) * ldd + i % rowlen] = (float)acc;
        }
    }
}

// ---------------------------------------------------------------------------------------------
// pooling, upsampling, ReLU backward, features

struct Coarse {
    int64_t b;
    int z, y, x;
};

__device__ __forceinline__ int64_t fine_index(const pvnet_shape& s, int64_t b, int z, int y, int x) {
    return ((b * s.d + z) * s.h + y) * (int64_t)s.w + x;
}

// coarse voxel and 8-channel chunk of thread i (32-bit arithmetic: the host keeps the coarse
// voxel count times the chunk count below 2^31)
__device__ __forceinline__ bool coarse_of(const pvnet_shape& s, int c8n, int64_t i, Coarse& o, int& ch) {
    const uint32_t d2 = s.d / 2, h2 = s.h / 2, w2 = s.w / 2;
    const int64_t n = (int64_t)s.nb * d2 * h2 * w2 * c8n;
    if (i >= n) return false;
    uint32_t v = (uint32_t)i;
    ch = (int)(v % (uint32_t)c8n) * 8;
    v /= (uint32_t)c8n;
    o.x = (int)(v % w2);
    v /= w2;
    o.y = (int)(v % h2);
    v /= h2;
    o.z = (int)(v % d2);
    o.b = v / d2;
    return true;
}

__device__ __forceinline__ int64_t coarse_index(const pvnet_shape& s, const Coarse& o) {
    return ((o.b * (s.d / 2) + o.z) * (s.h / 2) + o.y) * (int64_t)(s.w / 2) + o.x;
}

// fine voxel f and 8-channel chunk of thread i (consecutive threads: the chunks of one voxel, then
// the next voxel of the row), and the index of its parent coarse voxel; 32-bit arithmetic as above
__device__ __forceinline__ bool fine_of(const pvnet_shape& s, int c8n, int64_t i, int64_t& f, int64_t& cidx, int& ch) {
    const uint32_t w = s.w, h = s.h, d = s.d;
    const int64_t n = (int64_t)s.nb * d * h * w * c8n;
    if (i >= n) return false;
    uint32_t v = (uint32_t)i;
    ch = (int)(v % (uint32_t)c8n) * 8;
    v /= (uint32_t)c8n;
    f = v;
    const uint32_t x = v % w;
    v /= w;
    const uint32_t y = v % h;
    v /= h;
    const uint32_t z = v % d, b = v / d;
    cidx = (((int64_t)b * (d / 2) + z / 2) * (h / 2) + y / 2) * (int64_t)(w / 2) + x / 2;
    return true;
}

__global__ void k_pool2_fwd(pvnet_shape s, int c, const uint16_t* x, int ldx, uint16_t* y, int ldy) {
    Coarse o;
    int ch;
    if (!coarse_of(s, c / 8, (int64_t)blockIdx.x * blockDim.x + threadIdx.x, o, ch)) return;
    float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int k = 0; k < 8; k++) {
        const int64_t f = fine_index(s, o.b, 2 * o.z + (k >> 2), 2 * o.y + ((k >> 1) & 1), 2 * o.x + (k & 1));
        const uint4 v = *(const uint4*)(x + f * ldx + ch);
        const uint16_t* p = (const uint16_t*)&v;
        for (int j = 0; j < 8; j++) acc[j] += bf2f(p[j]);
    }
    uint4 out;
    uint16_t* po = (uint16_t*)&out;
    for (int j = 0; j < 8; j++) po[j] = f2bf(acc[j] * 0.125f);
    *(uint4*)(y + coarse_index(s, o) * ldy + ch) = out;
}

// one thread per fine voxel chunk: dx = dx (accumulate) + dy(parent) / 8.  relu_of (optional): the
// result is multiplied by (relu_of > 0), the backward of a ReLU whose output is relu_of, in the same
// pass
__global__ void k_pool2_bwd(pvnet_shape s, int c, const uint16_t* dy, int lddy, uint16_t* dx, int lddx, int accum,
                            const uint16_t* relu_of, int ldr) {
    int64_t f, ci;
    int ch;
    if (!fine_of(s, c / 8, (int64_t)blockIdx.x * blockDim.x + threadIdx.x, f, ci, ch)) return;
    const uint4 v = *(const uint4*)(dy + ci * lddy + ch);
    const uint16_t* p = (const uint16_t*)&v;
    uint4* dst = (uint4*)(dx + f * lddx + ch);
    uint4 out;
    uint16_t* po = (uint16_t*)&out;
    if (accum) {
        const uint4 old = *dst;
        const uint16_t* pold = (const uint16_t*)&old;
        for (int j = 0; j < 8; j++) po[j] = f2bf(bf2f(pold[j]) + bf2f(p[j]) * 0.125f);
    } else {
        for (int j = 0; j < 8; j++) po[j] = f2bf(bf2f(p[j]) * 0.125f);
    }
    if (relu_of) {
        const uint4 av = *(const uint4*)(relu_of + f * ldr + ch);
        const uint16_t* pa = (const uint16_t*)&av;
        for (int j = 0; j < 8; j++)
            if (!bf_pos(pa[j])) po[j] = 0;
    }
    *dst = out;
}

// one thread per fine voxel chunk, copying its parent's
__global__ void k_up2_fwd(pvnet_shape s, int c, const uint16_t* x, int ldx, uint16_t* y, int ldy) {
    int64_t f, ci;
    int ch;
    if (!fine_of(s, c / 8, (int64_t)blockIdx.x * blockDim.x + threadIdx.x, f, ci, ch)) return;
    *(uint4*)(y + f * ldy + ch) = *(const uint4*)(x + ci * ldx + ch);
}

// relu_of (optional) as in k_pool2_bwd
__global__ void k_up2_bwd(pvnet_shape s, int c, const uint16_t* dy, int lddy, uint16_t* dx, int lddx,
                          const uint16_t* relu_of, int ldr) {
    Coarse o;
    int ch;
    if (!coarse_of(s, c / 8, (int64_t)blockIdx.x * blockDim.x + threadIdx.x, o, ch)) return;
    float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int k = 0; k < 8; k++) {
        const int64_t f = fine_index(s, o.b, 2 * o.z + (k >> 2), 2 * o.y + ((k >> 1) & 1), 2 * o.x + (k & 1));
        const uint4 v = *(const uint4*)(dy + f * lddy + ch);
        const uint16_t* p = (const uint16_t*)&v;
        for (int j = 0; j < 8; j++) acc[j] += bf2f(p[j]);
    }
    uint4 out;
    uint16_t* po = (uint16_t*)&out;
    for (int j = 0; j < 8; j++) po[j] = f2bf(acc[j]);
    if (relu_of) {
        const uint4 av = *(const uint4*)(relu_of + coarse_index(s, o) * ldr + ch);
        const uint16_t* pa = (const uint16_t*)&av;
        for (int j = 0; j < 8; j++)
            if (!bf_pos(pa[j])) po[j] = 0;
    }
    *(uint4*)(dx + coarse_index(s, o) * lddx + ch) = out;
}

// grid.y: the 8-channel chunk
__global__ void k_relu_bwd(int64_t m, const uint16_t* a, int lda, uint16_t* dx, int lddx) {
    const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= m) return;
    const int ch = blockIdx.y * 8;
    const uint4 av = *(const uint4*)(a + v * lda + ch);
    uint4* dp = (uint4*)(dx + v * lddx + ch);
    uint4 dv = *dp;
    const uint16_t* pa = (const uint16_t*)&av;
    uint16_t* pd = (uint16_t*)&dv;
    for (int j = 0; j < 8; j++)
        if (!bf_pos(pa[j])) pd[j] = 0;
    *dp = dv;
}

// squared-distance transform along one axis: g(i) = min_j (g_in(j) + (i - j)^2); the first pass
// starts from g_in = 0 on solid voxels and "infinite" elsewhere.  The three passes take 35 us on a
// 96 x 96 x 192 box and 82 us on 8 x 96^3 (283 and 404 us with one thread per line).
constexpr float EDT_INF = 1e30f;

// First axis (binary input: 0 on solid voxels): the squared distance to the nearest solid voxel of the line.
// One wave per line: the solid voxels of each 64 are one ballot, and a lane finds its neighbours on both sides
// with bit scans (EDT_WORDS words cover the longest line).  Bound by memory: 1 byte in, 4 out per voxel.
constexpr int EDT_WORDS = PVNET_EDT_MAX / 64;

__global__ __launch_bounds__(256) void k_edt_row(int64_t nlines, int w, const uint8_t* code, float* g) {
    const int lane = threadIdx.x & 63;
    const int64_t line = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (line >= nlines) return;
    const int64_t base = line * w;
    uint64_t m[EDT_WORDS];
#pragma unroll
    for (int k = 0; k < EDT_WORDS; k++) {
        const int j = 64 * k + lane;
        m[k] = 64 * k < w ? __ballot(j < w && code[base + j] == 0) : 0;
    }
    int next[EDT_WORDS];  // the first solid voxel beyond word k
    int nx = 3 * w;
#pragma unroll
    for (int k = EDT_WORDS - 1; k >= 0; k--) {
        next[k] = nx;
        if (m[k]) nx = 64 * k + __builtin_ctzll(m[k]);
    }
    int last = -2 * w;  // the last solid voxel before word k
#pragma unroll
    for (int k = 0; k < EDT_WORDS; k++) {
        const int j = 64 * k + lane;
        if (64 * k >= w) break;
        const uint64_t lo = m[k] & (~0ull >> (63 - lane)), hi = m[k] >> lane;
        const int l = lo ? 64 * k + 63 - __builtin_clzll(lo) : last;
        const int r = hi ? j + __builtin_ctzll(hi) : next[k];
        const int dd = min(j - l, r - j);
        if (j < w) g[base + j] = dd >= w ? EDT_INF : (float)(dd * dd);
        if (m[k]) last = 64 * k + 63 - __builtin_clzll(m[k]);
    }
}

// The other axes: each voxel's min_j (f(j) + (i - j)^2), by scanning outward from i and stopping at the first r
// with r^2 >= the best value so far: f >= 0, so no farther j can lower it.  Every term is an exact integer in
// FP32 (or EDT_INF), so the result is that of the full scan bit for bit.  A block stages EDT_COLS neighbouring
// columns in LDS; its threads take one column and every EDT_ROWS-th row, so that a column's scans run side by
// side.  Bound by the longest scan of a wave (the vessel's radius).
constexpr int EDT_COLS = 32, EDT_ROWS = 16;

__global__ __launch_bounds__(EDT_COLS * EDT_ROWS) void k_edt_col(int ncols, int n, int64_t stride, int last_axis, float* g) {
    extern __shared__ float sh[];  // [n][EDT_COLS]
    const int c = threadIdx.x % EDT_COLS, r0 = threadIdx.x / EDT_COLS;
    const int col = blockIdx.x * EDT_COLS + c;  // columns of one slab are neighbours in memory
    const bool act = col < ncols;
    float* gb = g + (int64_t)blockIdx.y * stride * n + col;
    for (int j = r0; j < n; j += EDT_ROWS) sh[j * EDT_COLS + c] = act ? gb[j * stride] : 0.f;
    __syncthreads();
    if (!act) return;
    for (int i = r0; i < n; i += EDT_ROWS) {
        float best = sh[i * EDT_COLS + c];
        for (int r = 1; r < n; r++) {
            const float rr = (float)(r * r);
            if (rr >= best) break;
            if (i - r >= 0) best = fminf(best, sh[(i - r) * EDT_COLS + c] + rr);
            if (i + r < n) best = fminf(best, sh[(i + r) * EDT_COLS + c] + rr);
        }
        gb[i * stride] = last_axis ? fminf(sqrtf(best), 255.f) : best;
    }
}

__global__ void k_features(pvnet_shape s, const uint8_t* code, const float* prm, const float* dist, uint16_t* xo) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t n = (int64_t)s.nb * s.d * s.h * s.w;
    if (i >= n) return;
    const int x = (int)(i % s.w);
    const int64_t b = i / ((int64_t)s.w * s.h * s.d);
    const int cd = code[i];
    const float fl = cd > 0 ? 1.f : 0.f;
    float f[8];
    f[0] = fl;
    f[1] = cd == 2 ? 1.f : 0.f;
    f[2] = cd == 3 ? 1.f : 0.f;
    f[3] = fl * (prm[3 * b + 1] - 0.5f) / 0.4f;
    f[4] = fl * prm[3 * b] / 0.05f;
    f[5] = fl * ((float)x / (float)max(1, s.w - 1) - 0.5f);
    f[6] = fl * dist[i] / 16.f;
    f[7] = fl * prm[3 * b + 2] / 804.247719f;  // pi * 16^2
    uint4 out;
    uint16_t* po = (uint16_t*)&out;
    for (int j = 0; j < 8; j++) po[j] = f2bf(f[j]);
    *(uint4*)(xo + i * 8) = out;
}

// ---------------------------------------------------------------------------------------------
// masked MSE loss: per-block FP64 partials, one final block, then the gradient

constexpr int LOSS_BLOCK = 256;

// channel weights: in device memory, or (p null) with the launch
constexpr int LOSS_NC = 8;
struct LossWeights {
    const float* p;
    float w[LOSS_NC];
    __device__ __forceinline__ float operator[](int k) const { return p ? p[k] : w[k]; }
};

__global__ __launch_bounds__(LOSS_BLOCK) void k_loss_partial(int64_t M, int nc, const float* y, int ldy,
                                                             const uint16_t* t, const uint8_t* code,
                                                             const LossWeights wc, double* part) {
    __shared__ double ss[LOSS_BLOCK], sc[LOSS_BLOCK];
    const int64_t i = (int64_t)blockIdx.x * LOSS_BLOCK + threadIdx.x;
    double e = 0.0, c = 0.0;
    if (i < M && code[i] > 0) {
        c = 1.0;
        for (int k = 0; k < nc; k++) {
            const float r = y[i * ldy + k] - bf2f(t[i * nc + k]);
            e += (double)(wc[k] * r * r);
        }
    }
    ss[threadIdx.x] = e;
    sc[threadIdx.x] = c;
    __syncthreads();
    for (int st = LOSS_BLOCK / 2; st > 0; st >>= 1) {
        if ((int)threadIdx.x < st) {
            ss[threadIdx.x] += ss[threadIdx.x + st];
            sc[threadIdx.x] += sc[threadIdx.x + st];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        part[2 * blockIdx.x] = ss[0];
        part[2 * blockIdx.x + 1] = sc[0];
    }
}

__global__ __launch_bounds__(LOSS_BLOCK) void k_loss_final(int nblk, int nc, const double* part, double* loss) {
    __shared__ double ss[LOSS_BLOCK], sc[LOSS_BLOCK];
    double e = 0.0, c = 0.0;
#pragma unroll 8
    for (int b = threadIdx.x; b < nblk; b += LOSS_BLOCK) {
        e += part[2 * b];
        c += part[2 * b + 1];
    }
    ss[threadIdx.x] = e;
    sc[threadIdx.x] = c;
    __syncthreads();
    for (int st = LOSS_BLOCK / 2; st > 0; st >>= 1) {
        if ((int)threadIdx.x < st) {
            ss[threadIdx.x] += ss[threadIdx.x + st];
            sc[threadIdx.x] += sc[threadIdx.x + st];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        loss[0] = sc[0] > 0 ? ss[0] / (sc[0] * nc) : 0.0;
        loss[1] = sc[0];
    }
}

__global__ void k_loss_grad(int64_t M, int nc, const float* y, int ldy, const uint16_t* t, const uint8_t* code,
                            const LossWeights wc, const double* loss, uint16_t* dy, int lddy) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= M) return;
    const double cnt = loss[1];
    const float sc = cnt > 0 ? (float)(2.0 / (cnt * nc)) : 0.f;
    const bool fl = code[i] > 0;
    for (int k = 0; k < lddy; k++) {
        float gk = 0.f;
        if (fl && k < nc) gk = sc * wc[k] * (y[i * ldy + k] - bf2f(t[i * nc + k]));
        dy[i * lddy + k] = f2bf(gk);
    }
}

// ---------------------------------------------------------------------------------------------
// optimizer and weight packing

__global__ void k_adam(int64_t n, float* p, const float* g, float* m, float* v, float lr, float b1, float b2,
                       float eps, float c1, float c2) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

// Weight layouts of up to PACK_LAYERS layers in one launch: a block belongs to one layer, a thread writes eight
// values of a row (rows are multiples of 32).  wt follows w32's order; for wd neighbouring threads take
// neighbouring input channels, so that the reads of w32 are the contiguous ones.  Bound by the launch for small
// networks: 15 layers of at most 24 channels 4.3 us, 2.7 us and a launch gap each on their own.
constexpr int PACK_LAYERS = 32;

struct PackTable {
    pvnet_pack e[PACK_LAYERS];
    int32_t end[PACK_LAYERS];  // blocks up to and with this layer
};

__global__ __launch_bounds__(256) void k_pack(const PackTable T) {
    int l = 0;
    while ((int)blockIdx.x >= T.end[l]) l++;
    const pvnet_pack& e = T.e[l];
    const int64_t i = (int64_t)((int)blockIdx.x - (l ? T.end[l - 1] : 0)) * 256 + threadIdx.x;
    const int K = e.ntaps * e.cin, Kd = e.ntaps * e.cout, k8 = (K + BK - 1) / BK * (BK / 8), kd8 = (Kd + BK - 1) / BK * (BK / 8);
    const int64_t nt = (int64_t)e.cout * k8, nd = (int64_t)e.cin * kd8;
    float v[8];
    uint16_t* dst;
    if (i < nt) {
        const int n = (int)(i / k8), k = (int)(i - (int64_t)n * k8) * 8;
#pragma unroll
        for (int q = 0; q < 8; q++) v[q] = k + q < K ? e.w32[(int64_t)n * K + k + q] : 0.f;
        dst = e.wt + 8 * i;
    } else if (i < nt + nd) {
        const int64_t j = i - nt;
        const int kc = (int)(j / e.cin), ci = (int)(j - (int64_t)kc * e.cin);
#pragma unroll
        for (int q = 0; q < 8; q++) {
            const int k = 8 * kc + q, tapd = k / e.cout, co = k - tapd * e.cout;
            v[q] = k < Kd ? e.w32[(int64_t)co * K + (e.ntaps - 1 - tapd) * e.cin + ci] : 0.f;
        }
        dst = e.wd + ((int64_t)ci * kd8 + kc) * 8;
    } else {
        return;
    }
    const uint4 o = make_uint4(f2bf_pk(v[0], v[1]), f2bf_pk(v[2], v[3]), f2bf_pk(v[4], v[5]), f2bf_pk(v[6], v[7]));
    if (((uintptr_t)dst & 15) == 0) {
        *reinterpret_cast<uint4*>(dst) = o;
    } else {  // layouts that start anywhere
        const uint16_t* po = reinterpret_cast<const uint16_t*>(&o);
#pragma unroll
        for (int q = 0; q < 8; q++) dst[q] = po[q];
    }
}

// ---------------------------------------------------------------------------------------------
// host helpers

bool shape_ok(const pvnet_shape* s) { return s && s->nb > 0 && s->d > 0 && s->h > 0 && s->w > 0; }

bool al16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

int kpad_of(int ntaps, int c) { return (ntaps * c + BK - 1) / BK * BK; }

struct WgradPlan {
    TiledWgrad tiled;    // unless one of
    bool march;          // k_wgrad_march
    bool pw;             // k_wgrad_pw
    WgradMarch mp;
    int pw_chunks;       // per block
    int nsplit;
    int64_t ws_main, ws_total;
};

WgradPlan plan_wgrad(const pvnet_shape& s, int ntaps, int cin, int cout, int flags) {
    WgradPlan p{};
    const int64_t M = voxels(s);
    p.tiled = tiled_wgrad(M, ntaps, cin, cout);
    p.nsplit = p.tiled.nsplit;
    p.march = ntaps == 27 && !(flags & PVNET_GATHER) && wgrad_march_plan(s, cin, cout, p.mp);
    if (p.march) p.nsplit = p.mp.splits;
    p.pw = ntaps == 1 && cin <= 32 && cout <= 16 && !(flags & PVNET_GATHER);
    if (p.pw) {
        const int64_t chunks = (M + WPW_VOX - 1) / WPW_VOX;
        p.pw_chunks = 4 * (int)((chunks + 4 * WPW_BLOCKS - 1) / (4 * WPW_BLOCKS));  // whole rounds of the four waves
        p.nsplit = (int)((chunks + p.pw_chunks - 1) / p.pw_chunks);
    }
    p.ws_main = (int64_t)p.nsplit * cout * ntaps * cin;
    p.ws_total = p.ws_main + (int64_t)p.nsplit * cout;  // and the bias rows
    return p;
}

int blocks_for(int64_t n, int bs) { return (int)((n + bs - 1) / bs); }

int pool_args(const pvnet_shape* s, int c, const void* a, int lda, const void* b, int ldb, const char* who) {
    if (!shape_ok(s) || s->d % 2 || s->h % 2 || s->w % 2) return fail(1, std::string(who) + ": sizes must be even");
    if (c <= 0 || c % 8 || lda < c || ldb < c || lda % 8 || ldb % 8) return fail(1, std::string(who) + ": bad channels");
    if (!a || !b || !al16(a) || !al16(b)) return fail(1, std::string(who) + ": null or misaligned pointer");
    if (voxels(*s) * (c / 8) >= ((int64_t)1 << 31)) return fail(1, std::string(who) + ": too many voxels");
    return 0;
}

template <bool PARTS>
void conv_gather(const pvnet_conv& c, const NetParts& pq, int64_t M, hipStream_t st) {
    const GatherTile t = gather_tile(M, c.cout);
    const int K = c.ntaps * c.cin;
    // 2^24 blocks, which a full count of voxels needs, are 2^32 threads, and a launch has fewer along x
    const int mt = blocks_for(M, t.bm), nz = mt == 1 << 24 ? 2 : 1;
    const dim3 grid(mt / nz, (c.cout + t.bn - 1) / t.bn, nz);
    if (t.bm == 256)
        hipLaunchKernelGGL((k_conv_fwd<16, 64, PARTS>), grid, dim3(256), 0, st, c, (int)M, K, pq);
    else if (t.bn == 16)
        hipLaunchKernelGGL((k_conv_fwd<16, 32, PARTS>), grid, dim3(256), 0, st, c, (int)M, K, pq);
    else if (t.bn == 64)
        hipLaunchKernelGGL((k_conv_fwd<64, 32, PARTS>), grid, dim3(256), 0, st, c, (int)M, K, pq);
    else
        hipLaunchKernelGGL((k_conv_fwd<32, 32, PARTS>), grid, dim3(256), 0, st, c, (int)M, K, pq);
}

int conv_launch(const pvnet_conv* c, const NetParts& pq, void* stream, const char* who) {
    if (!c || !shape_ok(&c->s)) return fail(1, std::string(who) + ": bad shape");
    if (c->ntaps != 1 && c->ntaps != 27) return fail(1, std::string(who) + ": ntaps must be 1 or 27");
    if (c->cin <= 0 || c->cin % 8 || c->cout <= 0) return fail(1, std::string(who) + ": cin must be a positive multiple of 8");
    if (c->kpad != kpad_of(c->ntaps, c->cin)) return fail(1, std::string(who) + ": kpad must be roundup(ntaps*cin, 32)");
    if (c->ldx < c->cin - pq.cup || c->ldx % 8 || c->ldy < c->cout - pq.c0) return fail(1, std::string(who) + ": bad row lengths");
    if (!c->x || !c->w || !c->y || !al16(c->x) || !al16(c->w)) return fail(1, std::string(who) + ": null or misaligned pointer");
    if (c->relu_of && c->ldr < c->cout) return fail(1, std::string(who) + ": bad relu_of row length");
    const int64_t M = voxels(c->s);
    if (M >= (int64_t)1 << 31) return fail(1, std::string(who) + ": too many voxels");
    hipStream_t st = (hipStream_t)stream;
    const int K = c->ntaps * c->cin;
    const bool parts = pq.cup || pq.c0;
    MarchPlan mp;
    if (march_ok(*c, pq) && march_plan(c->s, c->cin, c->cout, mp)) {
        const unsigned nblk = (unsigned)mp.ntx * mp.nty * mp.nzs * mp.ng * c->s.nb;
        hipLaunchKernelGGL(march_kernel(mp), dim3(nblk), dim3(64 * (mp.wx * mp.wn + mp.roll)), mp.lds, st, *c, mp, pq);
    } else if (c->ntaps == 1 && K <= BK && c->cout <= 64 && !(c->flags & PVNET_GATHER)) {
        const dim3 gp((unsigned)((M + 64 * PWT - 1) / (64 * PWT)));
        const bool vec = rows_by_four(*c);
        switch ((c->cout + 15) / 16) {
            case 1: hipLaunchKernelGGL((k_conv_pw<1>), gp, dim3(256), 0, st, *c, (int)M, vec); break;
            case 2: hipLaunchKernelGGL((k_conv_pw<2>), gp, dim3(256), 0, st, *c, (int)M, vec); break;
            case 3: hipLaunchKernelGGL((k_conv_pw<3>), gp, dim3(256), 0, st, *c, (int)M, vec); break;
            default: hipLaunchKernelGGL((k_conv_pw<4>), gp, dim3(256), 0, st, *c, (int)M, vec); break;
        }
    } else if (parts) {
        conv_gather<true>(*c, pq, M, st);
    } else {
        conv_gather<false>(*c, pq, M, st);
    }
    NET_LAUNCH();
    return 0;
}

template <bool PARTS>
void wgrad_tiled(const pvnet_wgrad& a, const NetParts& pq, const TiledWgrad& p, int64_t M, int64_t dboff, hipStream_t st) {
    const int K = a.ntaps * a.cin;
    const dim3 grid(p.ktiles, p.ntiles, p.nsplit);
    if (p.bn == 16)
        hipLaunchKernelGGL((k_conv_wgrad<16, PARTS>), grid, dim3(256), 0, st, a, (int)M, K, p.mchunk, pq, dboff);
    else if (p.bn == 32)
        hipLaunchKernelGGL((k_conv_wgrad<32, PARTS>), grid, dim3(256), 0, st, a, (int)M, K, p.mchunk, pq, dboff);
    else
        hipLaunchKernelGGL((k_conv_wgrad<64, PARTS>), grid, dim3(256), 0, st, a, (int)M, K, p.mchunk, pq, dboff);
}

int wgrad_launch(const pvnet_wgrad* a, const NetParts& pq, void* stream, const char* who) {
    if (!a || !shape_ok(&a->s)) return fail(1, std::string(who) + ": bad shape");
    if (a->ntaps != 1 && a->ntaps != 27) return fail(1, std::string(who) + ": ntaps must be 1 or 27");
    if (a->cin <= 0 || a->cin % 8 || a->cout <= 0 || a->cout % 8)
        return fail(1, std::string(who) + ": cin and cout must be positive multiples of 8");
    if (a->ldx < a->cin - pq.cup || a->ldx % 8 || a->lddy < a->cout || a->lddy % 8) return fail(1, std::string(who) + ": bad row lengths");
    if (!a->x || !a->dy || !a->ws || !a->dw || !al16(a->x) || !al16(a->dy))
        return fail(1, std::string(who) + ": null or misaligned pointer");
    const int64_t M = voxels(a->s);
    if (M % 32) return fail(1, std::string(who) + ": voxel count must be a multiple of 32");
    if (M >= (int64_t)1 << 31) return fail(1, std::string(who) + ": too many voxels");
    if (a->db && a->cout > 256) return fail(1, std::string(who) + ": bias gradient needs cout <= 256");
    hipStream_t st = (hipStream_t)stream;
    const WgradPlan p = plan_wgrad(a->s, a->ntaps, a->cin, a->cout, a->flags | (wgrad_march_ok(*a, pq) ? 0 : PVNET_GATHER));
    const int K = a->ntaps * a->cin;
    const int64_t dboff = a->db ? p.ws_main : -1;  // the bias sums come with the weights'
    if (p.march) {
        hipLaunchKernelGGL(wgrad_march_kernel(p.mp), dim3(p.mp.splits * p.mp.ns * p.mp.nf), dim3(256), p.mp.lds, st, *a, p.mp, pq,
                           dboff);
    } else if (p.pw) {
        hipLaunchKernelGGL(wgrad_pw_kernel(a->cin, a->cout), dim3(p.nsplit), dim3(256), 0, st, *a, (int)M, p.pw_chunks, dboff);
    } else if (pq.cup) {
        wgrad_tiled<true>(*a, pq, p.tiled, M, dboff, st);
    } else {
        wgrad_tiled<false>(*a, pq, p.tiled, M, dboff, st);
    }
    NET_LAUNCH();
    const int64_t len = (int64_t)a->cout * K;
    const SumJob jw{a->ws, a->dw, len, (int64_t)K, (int64_t)K, p.nsplit, (int)blocks_for(len, SUM_COLS)};
    SumJob jb{nullptr, nullptr, 0, 1, 1, 0, 0};
    if (a->db)
        jb = SumJob{a->ws + p.ws_main, a->db, (int64_t)a->cout, (int64_t)a->cout, (int64_t)a->cout, p.nsplit,
                    (int)blocks_for(a->cout, SUM_COLS)};
    hipLaunchKernelGGL(p.march ? k_sum_splits<true> : k_sum_splits<false>, dim3(jw.blocks + jb.blocks), dim3(256), 0, st, SumArgs{jw, jb, *a, pq});
    NET_LAUNCH();
    return 0;
}

int up_args(const pvnet_shape* s, int ntaps, int cin, const void* up, int ldu, int cup, const char* who) {
    if (!shape_ok(s) || s->d % 2 || s->h % 2 || s->w % 2) return fail(1, std::string(who) + ": sizes must be even");
    if (ntaps != 27 || cup <= 0 || cup % 8 || cup >= cin || ldu < cup || ldu % 8 || !up || !al16(up))
        return fail(1, std::string(who) + ": bad upsampled part");
    return 0;
}

int loss_launch(int64_t m, int32_t nc, const float* y, int32_t ldy, const uint16_t* t, const uint8_t* code,
                const LossWeights& wc, uint16_t* dy, int32_t lddy, double* part, double* loss, void* stream,
                const char* who) {
    if (m <= 0 || nc <= 0 || ldy < nc || lddy < nc || !y || !t || !code || !dy || !part || !loss)
        return fail(1, std::string(who) + ": bad argument");
    hipStream_t st = (hipStream_t)stream;
    const int nblk = blocks_for(m, LOSS_BLOCK);
    hipLaunchKernelGGL(k_loss_partial, dim3(nblk), dim3(LOSS_BLOCK), 0, st, m, nc, y, ldy, t, code, wc, part);
    NET_LAUNCH();
    hipLaunchKernelGGL(k_loss_final, dim3(1), dim3(LOSS_BLOCK), 0, st, nblk, nc, part, loss);
    NET_LAUNCH();
    hipLaunchKernelGGL(k_loss_grad, dim3(blocks_for(m, 256)), dim3(256), 0, st, m, nc, y, ldy, t, code, wc, loss, dy, lddy);
    NET_LAUNCH();
    return 0;
}

}  // namespace

extern "C" {

const char* pvnet_last_error(void) { return g_err.c_str(); }

int pvnet_conv_fwd(const pvnet_conv* c, void* stream) { return conv_launch(c, NetParts{}, stream, "pvnet_conv_fwd"); }

int pvnet_conv_up_fwd(const pvnet_conv* c, const uint16_t* up, int32_t ldu, int32_t cup, void* stream) {
    if (int rc = up_args(c ? &c->s : nullptr, c ? c->ntaps : 0, c ? c->cin : 0, up, ldu, cup, "pvnet_conv_up_fwd")) return rc;
    if (c->flags & PVNET_F32OUT) return fail(1, "pvnet_conv_up_fwd: bf16 output only");
    return conv_launch(c, NetParts{up, nullptr, ldu, cup, 0, 0}, stream, "pvnet_conv_up_fwd");
}

int pvnet_conv_split_fwd(const pvnet_conv* c, uint16_t* y0, int32_t ldy0, int32_t c0, void* stream) {
    if (!c || c->ntaps != 27 || !y0 || c0 <= 0 || c0 >= c->cout || c0 % 8 || c->cout % 8 || ldy0 < c0)
        return fail(1, "pvnet_conv_split_fwd: bad argument");
    if (c->flags & PVNET_F32OUT) return fail(1, "pvnet_conv_split_fwd: bf16 output only");
    return conv_launch(c, NetParts{nullptr, y0, 0, 0, ldy0, c0}, stream, "pvnet_conv_split_fwd");
}

int64_t pvnet_wgrad_ws_floats(const pvnet_shape* s, int32_t ntaps, int32_t cin, int32_t cout) {
    if (!shape_ok(s) || cin <= 0 || cout <= 0) return -1;
    // either kernel's partials fit (the call's flags pick one)
    return std::max(plan_wgrad(*s, ntaps, cin, cout, 0).ws_total, plan_wgrad(*s, ntaps, cin, cout, PVNET_GATHER).ws_total);
}

int pvnet_conv_wgrad(const pvnet_wgrad* a, void* stream) { return wgrad_launch(a, NetParts{}, stream, "pvnet_conv_wgrad"); }

int pvnet_conv_up_wgrad(const pvnet_wgrad* a, const uint16_t* up, int32_t ldu, int32_t cup, void* stream) {
    if (int rc = up_args(a ? &a->s : nullptr, a ? a->ntaps : 0, a ? a->cin : 0, up, ldu, cup, "pvnet_conv_up_wgrad")) return rc;
    return wgrad_launch(a, NetParts{up, nullptr, ldu, cup, 0, 0}, stream, "pvnet_conv_up_wgrad");
}

int pvnet_pack_layers(const pvnet_pack* layers, int32_t n, void* stream) {
    if (!layers || n <= 0) return fail(1, "pvnet_pack_layers: bad argument");
    for (int32_t i = 0; i < n; i++) {
        const pvnet_pack& e = layers[i];
        if (!e.w32 || !e.wt || !e.wd || (e.ntaps != 1 && e.ntaps != 27) || e.cin <= 0 || e.cout <= 0)
            return fail(1, "pvnet_pack_weights: bad argument");
    }
    for (int32_t i0 = 0; i0 < n; i0 += PACK_LAYERS) {
        PackTable T{};
        const int32_t m = std::min(PACK_LAYERS, n - i0);
        int32_t end = 0;
        for (int32_t i = 0; i < m; i++) {
            const pvnet_pack& e = T.e[i] = layers[i0 + i];
            end += blocks_for(((int64_t)e.cout * kpad_of(e.ntaps, e.cin) + (int64_t)e.cin * kpad_of(e.ntaps, e.cout)) / 8, 256);
            T.end[i] = end;
        }
        hipLaunchKernelGGL(k_pack, dim3(end), dim3(256), 0, (hipStream_t)stream, T);
        NET_LAUNCH();
    }
    return 0;
}

int pvnet_pack_weights(const float* w32, int32_t ntaps, int32_t cin, int32_t cout, uint16_t* wt, uint16_t* wd,
                       void* stream) {
    const pvnet_pack e{w32, wt, wd, ntaps, cin, cout, 0};
    return pvnet_pack_layers(&e, 1, stream);
}

int pvnet_pool2_fwd(const pvnet_shape* s, int32_t c, const uint16_t* x, int32_t ldx, uint16_t* y, int32_t ldy,
                    void* stream) {
    if (int rc = pool_args(s, c, x, ldx, y, ldy, "pvnet_pool2_fwd")) return rc;
    const int64_t n = voxels(*s) / 8 * (c / 8);
    hipLaunchKernelGGL(k_pool2_fwd, dim3(blocks_for(n, 256)), dim3(256), 0, (hipStream_t)stream, *s, c, x, ldx, y, ldy);
    NET_LAUNCH();
    return 0;
}

int pvnet_pool2_bwd(const pvnet_shape* s, int32_t c, const uint16_t* dy, int32_t lddy, uint16_t* dx, int32_t lddx,
                    int32_t accumulate, void* stream) {
    if (int rc = pool_args(s, c, dy, lddy, dx, lddx, "pvnet_pool2_bwd")) return rc;
    const int64_t n = voxels(*s) * (c / 8);  // fine voxel chunks
    hipLaunchKernelGGL(k_pool2_bwd, dim3(blocks_for(n, 256)), dim3(256), 0, (hipStream_t)stream, *s, c, dy, lddy, dx,
                       lddx, accumulate ? 1 : 0, (const uint16_t*)nullptr, 0);
    NET_LAUNCH();
    return 0;
}

int pvnet_pool2_bwd_relu(const pvnet_shape* s, int32_t c, const uint16_t* dy, int32_t lddy, uint16_t* dx,
                         int32_t lddx, const uint16_t* relu_of, int32_t ldr, void* stream) {
    if (int rc = pool_args(s, c, dy, lddy, dx, lddx, "pvnet_pool2_bwd_relu")) return rc;
    if (!relu_of || !al16(relu_of) || ldr < c || ldr % 8) return fail(1, "pvnet_pool2_bwd_relu: bad relu_of");
    const int64_t n = voxels(*s) * (c / 8);  // fine voxel chunks
    hipLaunchKernelGGL(k_pool2_bwd, dim3(blocks_for(n, 256)), dim3(256), 0, (hipStream_t)stream, *s, c, dy, lddy, dx,
                       lddx, 1, relu_of, ldr);
    NET_LAUNCH();
    return 0;
}

int pvnet_up2_fwd(const pvnet_shape* s, int32_t c, const uint16_t* x, int32_t ldx, uint16_t* y, int32_t ldy,
                  void* stream) {
    if (int rc = pool_args(s, c, x, ldx, y, ldy, "pvnet_up2_fwd")) return rc;
    const int64_t n = voxels(*s) * (c / 8);  // fine voxel chunks
    hipLaunchKernelGGL(k_up2_fwd, dim3(blocks_for(n, 256)), dim3(256), 0, (hipStream_t)stream, *s, c, x, ldx, y, ldy);
    NET_LAUNCH();
    return 0;
}

int pvnet_up2_bwd(const pvnet_shape* s, int32_t c, const uint16_t* dy, int32_t lddy, uint16_t* dx, int32_t lddx,
                  void* stream) {
    if (int rc = pool_args(s, c, dy, lddy, dx, lddx, "pvnet_up2_bwd")) return rc;
    const int64_t n = voxels(*s) / 8 * (c / 8);
    hipLaunchKernelGGL(k_up2_bwd, dim3(blocks_for(n, 256)), dim3(256), 0, (hipStream_t)stream, *s, c, dy, lddy, dx, lddx,
                       (const uint16_t*)nullptr, 0);
    NET_LAUNCH();
    return 0;
}

int pvnet_up2_bwd_relu(const pvnet_shape* s, int32_t c, const uint16_t* dy, int32_t lddy, uint16_t* dx, int32_t lddx,
                       const uint16_t* relu_of, int32_t ldr, void* stream) {
    if (int rc = pool_args(s, c, dy, lddy, dx, lddx, "pvnet_up2_bwd_relu")) return rc;
    if (!relu_of || !al16(relu_of) || ldr < c || ldr % 8) return fail(1, "pvnet_up2_bwd_relu: bad relu_of");
    const int64_t n = voxels(*s) / 8 * (c / 8);
    hipLaunchKernelGGL(k_up2_bwd, dim3(blocks_for(n, 256)), dim3(256), 0, (hipStream_t)stream, *s, c, dy, lddy, dx, lddx,
                       relu_of, ldr);
    NET_LAUNCH();
    return 0;
}

int pvnet_relu_bwd(int64_t m, int32_t c, const uint16_t* a, int32_t lda, uint16_t* dx, int32_t lddx, void* stream) {
    if (m <= 0 || c <= 0 || c % 8 || lda < c || lddx < c || lda % 8 || lddx % 8 || !a || !dx || !al16(a) || !al16(dx))
        return fail(1, "pvnet_relu_bwd: bad argument");
    hipLaunchKernelGGL(k_relu_bwd, dim3(blocks_for(m, 256), c / 8), dim3(256), 0, (hipStream_t)stream, m, a, lda, dx, lddx);
    NET_LAUNCH();
    return 0;
}

int pvnet_wall_distance(const pvnet_shape* s, const uint8_t* code, float* dist, void* stream) {
    if (!shape_ok(s) || !code || !dist) return fail(1, "pvnet_wall_distance: bad argument");
    if (s->d > PVNET_EDT_MAX || s->h > PVNET_EDT_MAX || s->w > PVNET_EDT_MAX)
        return fail(1, "pvnet_wall_distance: box sizes are limited to PVNET_EDT_MAX");
    // axis y: slabs are the x-y planes, columns x; axis z: slabs are the boxes, columns the plane's voxels
    const int64_t plane = (int64_t)s->h * s->w, nlines = voxels(*s) / s->w, nslab[2] = {(int64_t)s->nb * s->d, s->nb};
    const int64_t ncol[2] = {s->w, plane};
    const int len[2] = {s->h, s->d};
    constexpr int64_t LINES = (int64_t)1 << 25;  // of one launch: 64 threads each, and a launch has fewer than 2^32
    for (int64_t l0 = 0; l0 < nlines; l0 += LINES) {
        const int64_t n = std::min(LINES, nlines - l0);
        hipLaunchKernelGGL(k_edt_row, dim3(blocks_for(n, 4)), dim3(256), 0, (hipStream_t)stream, n, s->w, code + l0 * s->w, dist + l0 * s->w);
        NET_LAUNCH();
    }
    for (int axis = 0; axis < 2; axis++)
        // slabs beyond the grid's y limit go in several launches
        for (int64_t s0 = 0; s0 < nslab[axis]; s0 += 65535) {
            const dim3 grid(blocks_for(ncol[axis], EDT_COLS), (unsigned)std::min<int64_t>(65535, nslab[axis] - s0));
            hipLaunchKernelGGL(k_edt_col, grid, dim3(EDT_COLS * EDT_ROWS), (size_t)len[axis] * EDT_COLS * sizeof(float),
                               (hipStream_t)stream, (int)ncol[axis], len[axis], ncol[axis], axis == 1 ? 1 : 0,
                               dist + s0 * ncol[axis] * len[axis]);
            NET_LAUNCH();
        }
    return 0;
}

int pvnet_features(const pvnet_shape* s, const uint8_t* code, const float* prm, const float* dist, uint16_t* x,
                   void* stream) {
    if (!shape_ok(s) || !code || !prm || !dist || !x || !al16(x)) return fail(1, "pvnet_features: bad argument");
    const int64_t n = voxels(*s);
    hipLaunchKernelGGL(k_features, dim3(blocks_for(n, 256)), dim3(256), 0, (hipStream_t)stream, *s, code, prm, dist,
                       x);
    NET_LAUNCH();
    return 0;
}

int64_t pvnet_loss_ws_doubles(int64_t m) { return m > 0 ? 2 * ((m + LOSS_BLOCK - 1) / LOSS_BLOCK) : -1; }

int pvnet_mse_loss(int64_t m, int32_t nc, const float* y, int32_t ldy, const uint16_t* t, const uint8_t* code,
                   const float* wc, uint16_t* dy, int32_t lddy, double* part, double* loss, void* stream) {
    if (!wc) return fail(1, "pvnet_mse_loss: bad argument");
    return loss_launch(m, nc, y, ldy, t, code, LossWeights{wc, {}}, dy, lddy, part, loss, stream, "pvnet_mse_loss");
}

int pvnet_mse_loss_host_weights(int64_t m, int32_t nc, const float* y, int32_t ldy, const uint16_t* t,
                                const uint8_t* code, const float* wc, uint16_t* dy, int32_t lddy, double* part,
                                double* loss, void* stream) {
    if (!wc || nc <= 0 || nc > LOSS_NC) return fail(1, "pvnet_mse_loss_host_weights: bad argument");
    LossWeights w{};
    for (int k = 0; k < nc; k++) w.w[k] = wc[k];
    return loss_launch(m, nc, y, ldy, t, code, w, dy, lddy, part, loss, stream, "pvnet_mse_loss_host_weights");
}

int pvnet_adam(int64_t n, float* p, const float* g, float* m, float* v, float lr, float b1, float b2, float eps,
               int32_t t, void* stream) {
    if (n <= 0 || !p || !g || !m || !v || t < 1) return fail(1, "pvnet_adam: bad argument");
    const float c1 = 1.f - powf(b1, (float)t), c2 = 1.f - powf(b2, (float)t);
    hipLaunchKernelGGL(k_adam, dim3(blocks_for(n, 256)), dim3(256), 0, (hipStream_t)stream, n, p, g, m, v, lr, b1, b2,
                       eps, c1, c2);
    NET_LAUNCH();
    return 0;
}

}  // extern "C"
