// wgrad_march.hpp — weight gradients of 3x3x3 convolutions that march through z (gfx950).
//
//   dw[n][tap][ci] = sum over voxels m of dy[m][n] x[m + off(tap)][ci]
//
// The reduction index is the voxel.  A block walks runs of planes of a tx x ty tile with the planes of both
// tensors copied straight into LDS, channels innermost as in memory, and reads the MFMA operands (eight
// voxels of one channel per lane) with the transposing LDS read, so nothing is transposed in registers.  The
// tensor with the fewer channels per block is the one that is shifted by the taps:
//   sum_m dy[m] x[m + off] = sum_m' dy[m' - off] x[m'],
// so a block takes 16 output channels of dy (planes z-1 .. z+1 with a halo) against 16 CF input channels of x
// (its own voxels only), and a wave reads CF + 7 fragments for 7 CF MFMAs.  Wave v owns the shifts v, v + 4, ..
// (7 of them; the 28th is a repeat that is not written), so every sum is complete within its wave.  Blocks are
// splits of the voxels, summed by k_sum_splits, which also sees to an x that is not finite (here it meets the zeros
// around dy's box).  The bias gradient is one more MFMA per dy fragment of the centre tap, with ones for x.
//
// What bounds it (counters of a training step on 8 x 96^3): at CF = 1 the LDS (8 KB of fragments for 7 MFMAs: busy 49 % of
// the time, matrix cores 26 %, waits 44 % of the waves'), at CF = 3 the matrix cores first (43 %; LDS 26 %, waits 40 %).
// Measured against the kernels it replaces (register transposes, one LDS copy of x per x shift or a gather per tap;
// split sums included), us per call, batch x grid, channels in -> out: 8 x 96^3 48->16 1032 -> 324, 16->16 346 -> 152,
// 8->16 200 -> 138; 8 x 48^3 96->32 301 -> 163, 32->32 114 -> 73; 8 x 24^3 224->64 339 -> 121, 64->64 115 -> 51;
// 8 x 12^3 160->160 111 -> 62; 3 x 20 x 18 x 28 64->160 92 -> 43.  With its input in two parts, in a training step,
// 48->16 takes 266 us (sums apart): the upsampled channels are read from a tensor an eighth the size.
#pragma once

typedef short tr4 __attribute__((ext_vector_type(4)));

// 4 voxels (rows of 16 channels, 32 bytes apart) x this lane's channel: lane 16 q + c of the wave addresses
// row 4 q + c / 4, channels 4 (c % 4) .. + 3, and receives channel c of rows 4 q .. 4 q + 3
__device__ __forceinline__ uint2 tr_read(const char* lds) {
    const tr4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) tr4*)(uintptr_t)(uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char*)lds);
    return *reinterpret_cast<const uint2*>(&v);
}

template <int CF>
__global__ __launch_bounds__(256, 3) void k_wgrad_march(const pvnet_wgrad a, const WgradMarch p, const NetParts q,
                                                        const int64_t dboff) {
    extern __shared__ uint4 wm_sm[];
    const int t = threadIdx.x, lane = t & 63, g = lane >> 4, c16 = lane & 15;
    const int wv = __builtin_amdgcn_readfirstlane(t >> 6);
    const int d = a.s.d, h = a.s.h, w = a.s.w, K = 27 * a.cin;
    const int slot = xcd_tile(blockIdx.x, gridDim.x);
    const int split = slot / (p.ns * p.nf), r0 = slot - split * (p.ns * p.nf);
    const int s0 = (r0 % p.ns) * 16, f0 = (r0 / p.ns) * 16 * CF;  // first channel of dy, of x
    const int vox = p.tx * p.ty, sl32 = p.gr * 32, nuS = 2 * p.hp, nuF = 2 * CF * sl32;
    uint4* Fs = wm_sm + 4 * p.su;
    int* vtab = reinterpret_cast<int*>(Fs + 2 * p.fu);
    int *soS = vtab + sl32, *soF = soS + nuS;
    const uint32_t ldsS = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint4*)wm_sm, ldsF = ldsS + 16u * 4u * (uint32_t)p.su;
    const char* smS = reinterpret_cast<const char*>(wm_sm);
    const char* smF = reinterpret_cast<const char*>(Fs);

    // slot -> byte offset of its own voxel in a dy plane (slots beyond the tile: the first voxel's)
    for (int i = t; i < sl32; i += 256) {
        const int v = i < vox ? i : 0, y = v / p.tx, x = v - y * p.tx;
        vtab[i] = 32 * ((y + 1) * p.hx + x + 1);
    }

    f32x4 acc[7][CF];
#pragma unroll
    for (int i = 0; i < 7; i++)
#pragma unroll
        for (int f = 0; f < CF; f++) acc[i][f] = f32x4{0.f, 0.f, 0.f, 0.f};
    // the bias gradient: wave 1 (it owns the centre tap), in the blocks of the first x channels
    const bool dob = dboff >= 0 && wv == 1 && f0 == 0;
    f32x4 accb = f32x4{0.f, 0.f, 0.f, 0.f};
    bf16x8 ones;
#pragma unroll
    for (int e = 0; e < 8; e++) ones[e] = (__bf16)1.0f;

    const int rowv = 4 * g + (c16 >> 2), colb = (c16 & 3) * 8;  // this lane's row within 16 voxels, byte column
    const int u1 = min(p.units, (split + 1) * p.per);
    for (int u = split * p.per; u < u1; u++) {
        int r = u;
        const int zq = r % p.nzs;
        r /= p.nzs;
        const int x0 = (r % p.ntx) * p.tx;
        r /= p.ntx;
        const int y0 = (r % p.nty) * p.ty;
        const int64_t box = r / p.nty;
        const int z0 = zq * p.zseg, z1 = min(d, z0 + p.zseg);
        __syncthreads();  // the previous run is done with the LDS
        // element offset of every unit within its plane (-1: zero; bit 0: x's half-size part, as in conv_march)
        for (int i = t; i < nuS; i += 256) {
            const int v = i >> 1, ch = s0 + 8 * (i & 1);
            const int hy = v / p.hx, x = x0 - 1 + v - hy * p.hx, y = y0 - 1 + hy;
            soS[i] = (unsigned)x < (unsigned)w && (unsigned)y < (unsigned)h && ch < a.cout ? (y * w + x) * a.lddy + ch : -1;
        }
        for (int i = t; i < nuF; i += 256) {
            const int cp = i / (2 * sl32), k = i - cp * 2 * sl32, v = k >> 1, ch = f0 + 16 * cp + 8 * (k & 1);
            const int yy = v / p.tx, y = y0 + yy, x = x0 + v - yy * p.tx;
            soF[i] = v >= vox || ch >= a.cin ? -1 : ch < q.cup ? ((y >> 1) * (w >> 1) + (x >> 1)) * q.ldu + ch + 1
                                                               : (y * w + x) * a.ldx + ch - q.cup;
        }
        __syncthreads();
        auto stage = [&](const uint16_t* base, int ld, int z, const int* so, int nu, uint32_t lds, bool parts) {
            const bool zin = (unsigned)z < (unsigned)d;
            const uint16_t* pb = base + (box * d + (zin ? z : 0)) * ((int64_t)h * w) * ld;
            const uint16_t* pu = parts && q.cup ? q.up + (box * (d >> 1) + (z >> 1)) * ((int64_t)(h >> 1) * (w >> 1)) * q.ldu - 1 : pb;
            for (int i = 64 * wv; i < nu; i += 256)
                if (i + lane < nu) {
                    const int o = so[i + lane];
                    lds_copy16(zin && o >= 0 ? (const void*)((o & 1 ? pu : pb) + o) : (const void*)g_march_zero,
                               __builtin_amdgcn_readfirstlane(lds + 16u * (uint32_t)i));
                }
        };
        for (int z = z0 - 1; z <= z0 + 1; z++) stage(a.dy, a.lddy, z, soS, nuS, ldsS + 16u * (uint32_t)((z & 3) * p.su), false);
        stage(a.x, a.ldx, z0, soF, nuF, ldsF + 16u * (uint32_t)((z0 & 1) * p.fu), true);
        march_wait();
        march_barrier();
        for (int z = z0; z < z1; z++) {
            if (z + 1 < z1) {
                stage(a.dy, a.lddy, z + 2, soS, nuS, ldsS + 16u * (uint32_t)(((z + 2) & 3) * p.su), false);
                stage(a.x, a.ldx, z + 1, soF, nuF, ldsF + 16u * (uint32_t)(((z + 1) & 1) * p.fu), true);
            }
            int toff[7];  // byte offset of each shift from a voxel's own unit, wave-uniform
#pragma unroll
            for (int i = 0; i < 7; i++) {
                const int s = min(wv + 4 * i, 26);
                const int dz = s / 9, dy = s / 3 % 3, dx = s % 3;
                toff[i] = 16 * (((z + dz - 1) & 3) * p.su) + 32 * ((dy - 1) * p.hx + dx - 1);
            }
            const char* fb = smF + 16 * ((z & 1) * p.fu) + 32 * rowv + colb;
            auto group = [&](int q, bool part) {
                const int v0 = vtab[32 * q + rowv] + colb, v1 = vtab[32 * q + 16 + rowv] + colb;
                // in the tile's last group, elements beyond the tile are zero in both operands
                uint2 m0 = make_uint2(~0u, ~0u), m1 = m0;
                if (part) {
                    auto keep = [&](int n) {
                        return make_uint2(n >= 2 ? ~0u : n == 1 ? 0xffffu : 0u, n >= 4 ? ~0u : n == 3 ? 0xffffu : 0u);
                    };
                    m0 = keep(vox - (32 * q + 4 * g));
                    m1 = keep(vox - (32 * q + 16 + 4 * g));
                }
                uint4 fr[CF];
#pragma unroll
                for (int f = 0; f < CF; f++) {
                    const char* pf = fb + 32 * (f * sl32 + 32 * q);
                    const uint2 lo = tr_read(pf), hi = tr_read(pf + 512);
                    fr[f] = make_uint4(lo.x, lo.y, hi.x, hi.y);
                }
#pragma unroll
                for (int i = 0; i < 7; i++) {
                    uint2 lo = tr_read(smS + toff[i] + v0), hi = tr_read(smS + toff[i] + v1);
                    if (part) {
                        lo.x &= m0.x, lo.y &= m0.y;
                        hi.x &= m1.x, hi.y &= m1.y;
                    }
                    const uint4 sv = make_uint4(lo.x, lo.y, hi.x, hi.y);
                    const bf16x8 sb = *reinterpret_cast<const bf16x8*>(&sv);
#pragma unroll
                    for (int f = 0; f < CF; f++)
                        acc[i][f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(sb, *reinterpret_cast<const bf16x8*>(&fr[f]), acc[i][f], 0, 0, 0);
                    if (i == 3 && dob) accb = __builtin_amdgcn_mfma_f32_16x16x32_bf16(sb, ones, accb, 0, 0, 0);
                }
            };
            const int whole = vox >> 5;
            for (int q = 0; q < whole; q++) group(q, false);
            if (whole < p.gr) group(whole, true);
            march_wait();
            if (z + 1 < z1) march_barrier();
        }
    }

    // D[4 g + e][c16] of a tile pair: channel 4 g + e of dy, channel c16 of x; shift s is tap 26 - s
#pragma unroll
    for (int i = 0; i < 7; i++) {
        const int tap = 26 - (wv + 4 * i);
        if (tap < 0) continue;
#pragma unroll
        for (int f = 0; f < CF; f++) {
            const int n = s0 + 4 * g, ci = f0 + 16 * f + c16;
            if (ci >= a.cin) continue;
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (n + e < a.cout) a.ws[((int64_t)split * a.cout + n + e) * K + tap * a.cin + ci] = acc[i][f][e];
        }
    }
    if (dob && c16 == 0)  // every column holds the sum of channel 4 g + e
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (s0 + 4 * g + e < a.cout) a.ws[dboff + (int64_t)split * a.cout + s0 + 4 * g + e] = accb[e];
}

typedef void (*WgradKernel)(const pvnet_wgrad, const WgradMarch, const NetParts, const int64_t);

inline WgradKernel wgrad_march_kernel(const WgradMarch& p) {
    return p.cf == 1 ? k_wgrad_march<1> : p.cf == 2 ? k_wgrad_march<2> : k_wgrad_march<3>;
}

// What one call needs beyond a plan: plane offsets fit 32 bits (as in conv_march, PVNET_GATHER and pointwise
// layers stay on k_conv_wgrad)
inline bool wgrad_march_ok(const pvnet_wgrad& a, const NetParts& q) {
    return (int64_t)a.s.h * a.s.w * std::max(std::max(a.ldx, a.lddy), q.ldu) < (int64_t)1 << 31;
}

// ---------------------------------------------------------------------------------------------
// Pointwise layers of at most 16 outputs and 32 inputs (the head): one pass over x and dy.  A wave copies chunks of
// 128 voxels of both into LDS of its own, one chunk ahead of its use and with no barrier, and reads the operands
// with the transposing LDS read as above; the bias gradient is one more MFMA against ones.  Bound by memory (48
// bytes a voxel for 16 -> 8 channels): 8 x 96^3 75 us (4.5 TB/s); the tiled kernel and its column sums took 149.
// Three blocks a CU, the LDS of 16 -> 8 channels, are one round of 768 blocks.
constexpr int WPW_VOX = 128, WPW_BLOCKS = 768;

constexpr int wpw_units(int cf, int nu) { return WPW_VOX * (2 * cf + nu); }  // one chunk, in 16-byte units

// CF: 16-channel tiles of x, NU: 8-channel units of dy
template <int CF, int NU>
__global__ __launch_bounds__(256) void k_wgrad_pw(const pvnet_wgrad a, const int M, const int per, const int64_t dboff) {
    constexpr int UN = wpw_units(CF, NU);
    __shared__ uint4 sm[4][2][UN];
    const int lane = threadIdx.x & 63, g = lane >> 4, c16 = lane & 15;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint4*)&sm[wv][0][0];
    // chunks wv, wv + 4, .. of the block's run (M + WPW_VOX may not fit 32 bits)
    const int c0 = blockIdx.x * per, c1 = min((M - 1) / WPW_VOX + 1, c0 + per);
    auto stage = [&](int c, int buf) {
#pragma unroll
        for (int i = 0; i < UN / 64; i++) {
            const bool ofx = i < 4 * CF;  // 64 units of x, or of dy
            const int u = 64 * (ofx ? i % 4 : i - 4 * CF) + lane;
            const int v = ofx ? u >> 1 : u / NU, ch = ofx ? 16 * (i / 4) + 8 * (u & 1) : 8 * (u % NU);
            const int64_t m = (int64_t)c * WPW_VOX + v;
            const bool in = m < M && ch < (ofx ? a.cin : a.cout);
            const uint16_t* src = (ofx ? a.x + m * a.ldx : a.dy + m * a.lddy) + ch;
            lds_copy16(in ? (const void*)src : (const void*)g_march_zero,
                       __builtin_amdgcn_readfirstlane(lds0 + 16u * (uint32_t)(buf * UN + 64 * i)));
        }
    };
    f32x4 acc[CF], accb = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int f = 0; f < CF; f++) acc[f] = accb;
    bf16x8 ones;
#pragma unroll
    for (int e = 0; e < 8; e++) ones[e] = (__bf16)1.0f;
    const int row = 4 * g + (c16 >> 2);
    const int xo = 32 * row + 8 * (c16 & 3);
    // dy rows of eight channels: the lanes of channels 8 .. 15 read 0 .. 7 again, for outputs that are not written
    const int dof = 16 * NU * row + 8 * (NU == 2 ? c16 & 3 : c16 & 1);
    auto frag = [&](const char* p, int step) {
        const uint2 lo = tr_read(p), hi = tr_read(p + step);
        return make_uint4(lo.x, lo.y, hi.x, hi.y);
    };
    if (c0 + wv < c1) stage(c0 + wv, 0);
    int buf = 0;
    for (int c = c0 + wv; c < c1; c += 4, buf ^= 1) {
        // the next chunk's copies stay in flight: the wait is for all but those
        if (c + 4 < c1) {
            stage(c + 4, buf ^ 1);
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(UN / 64) : "memory");
        } else {
            march_wait();
        }
        const char* xs = reinterpret_cast<const char*>(&sm[wv][buf][0]);
        const char* ds = xs + 16 * WPW_VOX * 2 * CF;
#pragma unroll
        for (int q = 0; q < WPW_VOX / 32; q++) {
            const uint4 dv = frag(ds + 16 * NU * 32 * q + dof, 16 * NU * 16);
            const bf16x8 db = *reinterpret_cast<const bf16x8*>(&dv);
#pragma unroll
            for (int f = 0; f < CF; f++) {
                const uint4 xv = frag(xs + 32 * (WPW_VOX * f + 32 * q) + xo, 512);
                acc[f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(db, *reinterpret_cast<const bf16x8*>(&xv), acc[f], 0, 0, 0);
            }
            accb = __builtin_amdgcn_mfma_f32_16x16x32_bf16(db, ones, accb, 0, 0, 0);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // read out before the slot is copied into again
    }
    // the four waves' sums, in order; [wave][channel of dy][channel of x, then the bias]
    constexpr int RW = 16 * CF + 1;
    float* red = reinterpret_cast<float*>(&sm[0][0][0]);
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 4; e++) {
        float* r = red + (wv * 16 + 4 * g + e) * RW;
#pragma unroll
        for (int f = 0; f < CF; f++) r[16 * f + c16] = acc[f][e];
        if (c16 == 0) r[16 * CF] = accb[e];
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 16 * RW; i += 256) {
        const int n = i / RW, ci = i - n * RW;
        if (n >= a.cout) continue;
        const float s = ((red[i] + red[16 * RW + i]) + red[32 * RW + i]) + red[48 * RW + i];
        if (ci < a.cin) a.ws[((int64_t)blockIdx.x * a.cout + n) * a.cin + ci] = s;
        else if (ci == 16 * CF && dboff >= 0) a.ws[dboff + (int64_t)blockIdx.x * a.cout + n] = s;
    }
}

typedef void (*WgradPwKernel)(const pvnet_wgrad, const int, const int, const int64_t);

inline WgradPwKernel wgrad_pw_kernel(int cin, int cout) {
    if (cin <= 16) return cout <= 8 ? k_wgrad_pw<1, 1> : k_wgrad_pw<1, 2>;
    return cout <= 8 ? k_wgrad_pw<2, 1> : k_wgrad_pw<2, 2>;
}
