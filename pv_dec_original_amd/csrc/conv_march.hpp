// conv_march.hpp — 3x3x3 convolutions (forward and input gradient) that march through z (gfx950).
//
// A block owns a tile of tx x ty voxels of the x-y plane and 16 wn output channels, and walks a run of
// planes.  The input planes, each with a one-voxel halo and all cin channels, are copied straight from
// memory into LDS (global_load_lds, no registers) one plane ahead of their use, so that the copies run
// under the MFMAs of the plane before.
//   k_conv_ring  any cin whose four plane slots fit: output plane z reads planes z-1, z, z+1 while z+2
//                arrives.  The narrow layers (cin 8, 16, 48): a k-step may span two dz.
//   k_conv_roll  cin % 32 == 0: every k-step lies within one dz, so plane p is read from LDS once for all
//                three output planes p+1 (dz = -1), p and p-1 (dz = +1), whose accumulators roll; two slots.
// The input may come in two parts: channels below `cup` from a tensor of half the size (nearest upsampling), the
// others from x; a copied unit then picks its source, and the upsampled half is never written out.  The output
// may go to two tensors in the same way, so that skips and gradients are dense rows for the layers and poolings
// that read them (a training step on 8 x 96^3: 7.03 -> 5.77 ms, of which the upsampling was 0.30, the poolings
// 0.43 and a skip written into the middle of 96-byte rows 0.22).
// Both run the k-steps of k_conv_fwd in the same order (k = tap * cin + ci, 32 per MFMA), so every output equals that
// kernel's bit for bit.  The weights are the MFMA's A operand and the voxels its B operand: a lane then holds four
// consecutive channels of one voxel and writes them with one 8-byte store.
//
// What bounds them (counters of a training step on 8 x 96^3): in the narrow layers nothing alone.  The matrix cores
// are busy 28 to 31 % of the time, the LDS 40 to 44 % (1 KB of voxels per MFMA when only 16 outputs share it; the
// weights of the ring kernel sit in registers for that reason), and the waves wait 33 to 44 % of theirs.  The deep
// layers, with weights from L2, wait 60 % (matrix cores 18 %): the latency of short runs on few voxels.  Measured
// against the gathering and brick kernels they replace, bf16, us per call (batch x grid, channels): 8 x 96^3 16->16
// 231 -> 124, 48->16 748 -> 389, 16->48 562 -> 355, 8->16 152 -> 99; 8 x 48^3 32->32 83 -> 68, 96->32 452 -> 214;
// 8 x 24^3 64->64 83 -> 57, 224->64 305 -> 132; 8 x 12^3 160->160 96 -> 43; 1 x 24 x 24 x 48 64->64 40 -> 23;
// 3 x 20 x 18 x 28 160->64 96 -> 37.
#pragma once

__device__ uint4 g_march_zero[4];  // source of the units outside the box

// 16 bytes per lane from src to LDS byte address lds + 16 * lane.  Written as one asm statement because the
// compiler would wait for the copy before the next LDS read; march_wait() is the wait, before the barrier
// that hands the slot over.  No register waits for it (m0 is put back); the nop is the hazard between
// writing m0 and its use.
__device__ __forceinline__ void lds_copy16(const void* src, uint32_t lds) {
    uint32_t keep;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep)
                 : "v"(src), "s"(lds)
                 : "memory");
}

__device__ __forceinline__ void march_wait() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
__device__ __forceinline__ void march_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// What a block of either kernel does around its k-loop: its place in the grid, the tables, the plane
// copies, the lanes' voxels and the epilogue.  LDS: NP plane slots, the weights (WL), the k-step table
// (NP rotations of 4 sp entries), the plane offsets.
template <int RT, bool WL, int NP>
struct MarchBlock {
    const pvnet_conv& a;
    const MarchPlan& p;
    const NetParts& q;
    uint4* wl;
    int *tab, *soff;
    int lane, g, c16, wv, nu, n0, nw, x0, y0, z0, z1;  // n0: this wave's 16 channels
    int64_t box;
    uint32_t lds0;
    int vb[RT], vo[RT];      // a voxel's own unit (LDS byte address in slot 0), its index within the plane (-1: none)
    uint32_t woff;           // byte offset of this lane's weight row and chunk
    float bias[4];
    uint2 mk[RT];            // ReLU mask of the plane

    __device__ __forceinline__ MarchBlock(const pvnet_conv& a_, const MarchPlan& p_, const NetParts& q_, uint4* sm, int sp)
        : a(a_), p(p_), q(q_) {
        const int t = threadIdx.x;
        lane = t & 63, g = lane >> 4, c16 = lane & 15;
        wv = __builtin_amdgcn_readfirstlane(t >> 6);
        const int h = a.s.h, w = a.s.w;
        nu = (a.cin >> 3) * p.hp;
        wl = sm + NP * p.su;
        tab = reinterpret_cast<int*>(wl + (WL ? 64 * p.wn * p.nsteps : 0));
        soff = tab + NP * 4 * sp;
        lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint4*)sm;

        int bid = xcd_tile(blockIdx.x, gridDim.x);
        const int nb0 = (bid % p.ng) * 16 * p.wn;
        nw = wv % p.wn;
        n0 = nb0 + nw * 16;
        bid /= p.ng;
        x0 = (bid % p.ntx) * p.tx;
        bid /= p.ntx;
        y0 = (bid % p.nty) * p.ty;
        bid /= p.nty;
        z0 = (bid % p.nzs) * p.zseg, z1 = min(a.s.d, z0 + p.zseg);
        box = bid / p.nzs;

        // element offset of every unit within its plane (-1: outside the box; bit 0: a plane of the half-size
        // tensor).  Two chunks of a voxel lie
        // side by side: a copy then reads 32 contiguous bytes per voxel, and the 16 + 16 lanes that read a
        // fragment's two chunks together cover every bank once, whatever the tap's shift.
        const int hxy = p.hx * (p.ty + 2);
        for (int u = t; u < nu; u += blockDim.x) {
            const int cg = u / (p.g * p.hp), r = u - cg * (p.g * p.hp), v = p.g == 2 ? r >> 1 : r;
            const int ch = cg * p.g + (r - v * p.g);
            const int hy = v / p.hx, x = x0 - 1 + v - hy * p.hx, y = y0 - 1 + hy;
            const bool in = v < hxy && (unsigned)x < (unsigned)w && (unsigned)y < (unsigned)h;
            soff[u] = !in ? -1 : 8 * ch < q.cup ? ((y >> 1) * (w >> 1) + (x >> 1)) * q.ldu + ch * 8 + 1
                                                : (y * w + x) * a.ldx + ch * 8 - q.cup;
        }
        if constexpr (WL) {
            // fragment order: the 64 lanes' operands of (k-step, column tile) are 64 consecutive units
            for (int i = t; i < 64 * p.wn * p.nsteps; i += blockDim.x) {
                const int f = i >> 6, l = i & 63, st = f / p.wn, row = 16 * (f - st * p.wn) + (l & 15);
                wl[i] = *(const uint4*)(a.w + (int64_t)min(nb0 + row, a.cout - 1) * a.kpad + st * BK + (l >> 4) * 8);
            }
        }
#pragma unroll
        for (int i = 0; i < RT; i++) {
            const int s = (wv / p.wn * RT + i) * 16 + c16;
            const int y = s / p.tx, x = s - y * p.tx;
            const bool in = y < p.ty && x0 + x < w && y0 + y < h;
            vb[i] = 16 * p.g * (in ? (y + 1) * p.hx + x + 1 : p.hx + 1);
            vo[i] = in ? (y0 + y) * w + x0 + x : -1;
        }
        // a row beyond cout only feeds outputs beyond cout, which are not written
        woff = ((uint32_t)min(n0 + c16, a.cout - 1) * (uint32_t)a.kpad + (uint32_t)g * 8u) * 2u;
#pragma unroll
        for (int e = 0; e < 4; e++) bias[e] = (a.bias && n0 + 4 * g + e < a.cout) ? a.bias[n0 + 4 * g + e] : 0.f;
    }

    // LDS byte offset, from a voxel's own unit in slot 0, of k-values k .. k + 7 when their plane is in `slot`
    __device__ __forceinline__ int tap_unit(int k, int slot, int dy, int dx) const {
        const int ci = k % a.cin, ch = ci >> 3, cg = ch / p.g;
        return 16 * (slot * p.su + cg * p.g * p.hp + p.g * (dy * p.hx + dx) + ch - cg * p.g);
    }

    // copies plane z into a slot, `first` of `of` waves taking part
    __device__ __forceinline__ void stage_plane(int z, int slot, int first, int of) const {
        const bool zin = (unsigned)z < (unsigned)a.s.d;
        const uint16_t* pb = a.x + (box * a.s.d + (zin ? z : 0)) * ((int64_t)a.s.h * a.s.w) * a.ldx;
        const uint16_t* pu = q.cup ? q.up + (box * (a.s.d >> 1) + (zin ? z >> 1 : 0)) * ((int64_t)(a.s.h >> 1) * (a.s.w >> 1)) * q.ldu - 1
                                   : pb;
        for (int u = 64 * first; u < nu; u += 64 * of) {
            const int ul = u + lane;
            if (ul < nu) {
                const int o = soff[ul];
                const void* src = (zin && o >= 0) ? (const void*)((o & 1 ? pu : pb) + o) : (const void*)g_march_zero;
                lds_copy16(src, __builtin_amdgcn_readfirstlane(lds0 + 16u * (uint32_t)(slot * p.su + u)));
            }
        }
    }

    // this wave's weight fragment of k-step s
    __device__ __forceinline__ uint4 wfrag(int s) const {
        if constexpr (WL) return wl[(s * p.wn + nw) * 64 + lane];
        else return *(const uint4*)((const char*)a.w + (size_t)(s * (2 * BK)) + woff);
    }

    __device__ __forceinline__ void xload(const uint4* sm, int tv, uint4 (&xf)[RT]) const {
#pragma unroll
        for (int i = 0; i < RT; i++) xf[i] = *reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(sm) + vb[i] + tv);
    }

    static __device__ __forceinline__ void mma(f32x4 (&acc)[RT], const uint4& bw, const uint4 (&xf)[RT]) {
#pragma unroll
        for (int i = 0; i < RT; i++)
            acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8*>(&bw),
                                                             *reinterpret_cast<const bf16x8*>(&xf[i]), acc[i], 0, 0, 0);
    }

    static __device__ __forceinline__ void clear(f32x4 (&acc)[RT]) {
#pragma unroll
        for (int i = 0; i < RT; i++) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

    // the ReLU mask of plane z
    __device__ __forceinline__ void load_mask(int z) {
        if (!a.relu_of || n0 + 4 * g >= a.cout) return;
        const int64_t mb = (box * a.s.d + z) * ((int64_t)a.s.h * a.s.w);
#pragma unroll
        for (int i = 0; i < RT; i++)
            if (vo[i] >= 0) mk[i] = *(const uint2*)(a.relu_of + (mb + vo[i]) * a.ldr + n0 + 4 * g);
    }

    __device__ __forceinline__ void store_plane(int z, const f32x4 (&acc)[RT]) const {
        if (n0 + 4 * g >= a.cout) return;
        const bool relu = a.flags & PVNET_RELU, f32out = a.flags & PVNET_F32OUT;
        // whether this lane's channels are in the output's first part: opaque, so that the pointer and row length
        // are not kept in registers through the k-loop
        int n4 = n0 + 4 * g;
        asm volatile("" : "+v"(n4));
        const bool first = n4 < q.c0;
        const uint32_t ld = first ? q.ldy0 : a.ldy;
        const int64_t o0 = (box * a.s.d + z) * ((int64_t)a.s.h * a.s.w) * ld + n4 - (first ? 0 : q.c0);
        char* yb = f32out ? (char*)((float*)a.y + o0) : (char*)((first ? q.y0 : (uint16_t*)a.y) + o0);
#pragma unroll
        for (int i = 0; i < RT; i++) {
            if (vo[i] < 0) continue;
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                v[e] = acc[i][e] + bias[e];
                if (relu) v[e] = v[e] < 0.f ? 0.f : v[e];
                if (a.relu_of && !bf_pos((uint16_t)((e < 2 ? mk[i].x : mk[i].y) >> (16 * (e & 1))))) v[e] = 0.f;
            }
            const uint64_t o = (uint64_t)(uint32_t)vo[i] * ld;
            if (f32out) *(float4*)(yb + 4 * o) = make_float4(v[0], v[1], v[2], v[3]);
            else *(uint2*)(yb + 2 * o) = make_uint2(f2bf_pk(v[0], v[1]), f2bf_pk(v[2], v[3]));
        }
    }
};

// WM: where the weights are during the k-loop: 0 memory (L2), one step ahead; 1 LDS; 2 registers (NSW
// k-steps, fixed at compile time)
template <int RT, int WM, int NSW>
__global__ __launch_bounds__(256) void k_conv_ring(const pvnet_conv a, const MarchPlan p, const NetParts q) {
    extern __shared__ uint4 march_sm[];
    const int sp = WM == 2 ? NSW : p.nsteps;
    MarchBlock<RT, WM == 1, 4> b(a, p, q, march_sm, sp);
    // k-step table per rotation r = z & 3 of the slots: plane z + dz sits in slot (z + dz) & 3
    for (int i = threadIdx.x; i < 4 * 4 * sp; i += 256) {
        const int r = i / (4 * sp), e = i - r * (4 * sp);
        const int k = (e >> 2) * BK + (e & 3) * 8;
        int dz, dy, dx;
        tap_offset(27, k / a.cin, dz, dy, dx);
        b.tab[i] = k < p.K ? b.tap_unit(k, (r + dz) & 3, dy, dx) : 0;
    }
    __syncthreads();
    const bool kbad = (sp - 1) * BK + 8 * b.g >= p.K;  // this lane's last chunk lies beyond K: zero operands
    uint4 wreg[WM == 2 ? NSW : 1];
    if constexpr (WM == 2) {
#pragma unroll
        for (int st = 0; st < NSW; st++) wreg[st] = b.wfrag(st);
    }
    f32x4 acc[RT];
    auto zero_last = [&](uint4 (&xf)[RT]) {
        if (kbad)
#pragma unroll
            for (int i = 0; i < RT; i++) xf[i] = make_uint4(0, 0, 0, 0);
    };
    auto steps = [&](const int* tb) {
        if constexpr (WM == 2) {
            int tv[NSW];
#pragma unroll
            for (int st = 0; st < NSW; st++) tv[st] = tb[4 * st + b.g];
#pragma unroll
            for (int st = 0; st < NSW; st++) {
                uint4 xf[RT];
                b.xload(march_sm, tv[st], xf);
                if (st == NSW - 1) zero_last(xf);
                b.mma(acc, wreg[st], xf);
            }
        } else {
            // the operands of a step are loaded during the MFMAs of the one before
            uint4 bw[2], xf[2][RT];
            auto load = [&](int s, int tv, int c) {
                bw[c] = b.wfrag(s);
                b.xload(march_sm, tv, xf[c]);
            };
            load(0, tb[b.g], 0);
            int tv = sp > 1 ? tb[4 + b.g] : 0;
            int s = 0;
            for (; s + 2 < sp; s += 2) {
                load(s + 1, tv, 1);
                tv = tb[4 * (s + 2) + b.g];
                b.mma(acc, bw[0], xf[0]);
                load(s + 2, tv, 0);
                if (s + 3 < sp) tv = tb[4 * (s + 3) + b.g];
                b.mma(acc, bw[1], xf[1]);
            }
            if (s + 1 < sp) {
                load(s + 1, tv, 1);
                b.mma(acc, bw[0], xf[0]);
                zero_last(xf[1]);
                b.mma(acc, bw[1], xf[1]);
            } else {
                zero_last(xf[0]);
                b.mma(acc, bw[0], xf[0]);
            }
        }
    };
    for (int z = b.z0 - 1; z <= b.z0 + 1; z++) b.stage_plane(z, z & 3, b.wv, 4);
    march_wait();
    march_barrier();
    for (int z = b.z0; z < b.z1; z++) {
        b.clear(acc);
        if (z + 1 < b.z1) b.stage_plane(z + 2, (z + 2) & 3, b.wv, 4);
        b.load_mask(z);
        steps(b.tab + (z & 3) * 4 * sp);
        march_wait();
        b.store_plane(z, acc);
        if (z + 1 < b.z1) march_barrier();
    }
}

// Waves 0 .. wx wn - 1 compute, each RT row tiles x 16 channels of three output planes; the last wave
// only copies planes, so that its copies do not hold up the weight loads of the others (a wave's loads
// return in order).  WL: weights in LDS, else read from memory (L2) two steps ahead.
template <int RT, bool WL>
__global__ __launch_bounds__(512) void k_conv_roll(const pvnet_conv a, const MarchPlan p, const NetParts q) {
    extern __shared__ uint4 march_sm[];
    const int sp = p.nsteps / 3;  // k-steps of one dz: a multiple of 9
    MarchBlock<RT, WL, 2> b(a, p, q, march_sm, sp);
    for (int i = threadIdx.x; i < 2 * 4 * sp; i += blockDim.x) {
        const int r = i / (4 * sp), e = i - r * (4 * sp);
        const int k = (e >> 2) * BK + (e & 3) * 8;
        int dz, dy, dx;
        tap_offset(27, k / a.cin, dz, dy, dx);  // the taps of the first dz
        b.tab[i] = b.tap_unit(k, r, dy, dx);
    }
    __syncthreads();
    const int n = b.z1 - b.z0;  // outputs; plane i = 0 .. n + 1 is z0 - 1 + i
    if (b.wv == p.wx * p.wn) {
        for (int i = 0; i <= n + 1; i++) {
            b.stage_plane(b.z0 - 1 + i, i & 1, 0, 1);
            march_wait();
            __builtin_amdgcn_s_barrier();  // plane i is there, and plane i - 1 is free
        }
        return;
    }

    // weights of k-step s in ring slot s % 3, of the dz in M
    uint4 bw[3][3];
    f32x4 acc[3][RT];
#define MARCH_WLOAD(s, r, M)                                                       \
    _Pragma("unroll") for (int z_ = 0; z_ < 3; z_++) if (((M) >> z_) & 1) bw[r][z_] = b.wfrag(z_ * sp + (s))
    // one plane; M: which dz have an output here (bit 0: dz = -1, starting in acc[0]; 1: dz = 0 in acc[1];
    // 2: dz = +1, ending in acc[2]).  A compile-time set, so that the k-loop has no branch and its loads stay in
    // flight across it.  The last two steps load the first two of the next plane, for every dz.
    auto plane = [&](const int* tb, auto mset) {
        constexpr int M = decltype(mset)::value;
        b.clear(acc[0]);
        uint4 xf[RT];
        b.xload(march_sm, tb[b.g], xf);
        int tv = tb[4 + b.g];
        auto step = [&](int r) {
            uint4 xn[RT];
            b.xload(march_sm, tv, xn);
            if (M & 1) b.mma(acc[0], bw[r][0], xf);
            if (M & 2) b.mma(acc[1], bw[r][1], xf);
            if (M & 4) b.mma(acc[2], bw[r][2], xf);
#pragma unroll
            for (int i = 0; i < RT; i++) xf[i] = xn[i];
            __builtin_amdgcn_sched_barrier(0);  // one step's operands in registers at a time
        };
        const int* tn = tb + 8 + b.g;  // table entry two steps ahead
        for (int s = 0; s < sp - 3; s += 3) {
            MARCH_WLOAD(s + 2, 2, M);
            const int t0 = tn[0];
            step(0);
            tv = t0;
            MARCH_WLOAD(s + 3, 0, M);
            const int t1 = tn[4];
            step(1);
            tv = t1;
            MARCH_WLOAD(s + 4, 1, M);
            const int t2 = tn[8];
            step(2);
            tv = t2;
            tn += 12;
        }
        MARCH_WLOAD(sp - 1, 2, M);
        const int t0 = tn[0];
        step(0);
        tv = t0;
        MARCH_WLOAD(0, 0, 7);
        step(1);
        MARCH_WLOAD(1, 1, 7);
        step(2);  // the operands it loads are not used
    };
    MARCH_WLOAD(0, 0, 7);
    MARCH_WLOAD(1, 1, 7);
    for (int i = 0; i <= n + 1; i++) {
        march_barrier();
        const int* tb = b.tab + (i & 1) * 4 * sp;
        switch ((i < n ? 1 : 0) | (i >= 1 && i <= n ? 2 : 0) | (i >= 2 ? 4 : 0)) {
            case 1: plane(tb, std::integral_constant<int, 1>{}); break;
            case 2: plane(tb, std::integral_constant<int, 2>{}); break;
            case 3: plane(tb, std::integral_constant<int, 3>{}); break;
            case 4: plane(tb, std::integral_constant<int, 4>{}); break;
            case 6: plane(tb, std::integral_constant<int, 6>{}); break;
            default: plane(tb, std::integral_constant<int, 7>{}); break;
        }
        if (i >= 2) {
            b.load_mask(b.z0 + i - 2);
            b.store_plane(b.z0 + i - 2, acc[2]);
        }
#pragma unroll
        for (int q = 0; q < RT; q++) {
            acc[2][q] = acc[1][q];
            acc[1][q] = acc[0][q];
        }
    }
#undef MARCH_WLOAD
}

typedef void (*MarchKernel)(const pvnet_conv, const MarchPlan, const NetParts);

template <int RT>
MarchKernel march_kernel_rt(const MarchPlan& p) {
    if (p.roll) {
        if constexpr (RT <= 5) return p.wm ? k_conv_roll<RT, true> : k_conv_roll<RT, false>;
        return nullptr;
    }
    if constexpr (RT != 5) {
        if (p.wm == 2) {
            if (p.nsteps == 7) return k_conv_ring<RT, 2, 7>;
            if (p.nsteps == 14) return k_conv_ring<RT, 2, 14>;
            if (p.nsteps == 21) return k_conv_ring<RT, 2, 21>;
            if constexpr (RT <= 4) if (p.nsteps == 41) return k_conv_ring<RT, 2, 41>;
            return nullptr;
        }
        return p.wm ? k_conv_ring<RT, 1, 1> : k_conv_ring<RT, 0, 1>;
    }
    return nullptr;
}

inline MarchKernel march_kernel(const MarchPlan& p) {
    switch (p.rt) {
        case 1: return march_kernel_rt<1>(p);
        case 2: return march_kernel_rt<2>(p);
        case 3: return march_kernel_rt<3>(p);
        case 4: return march_kernel_rt<4>(p);
        case 5: return march_kernel_rt<5>(p);
        case 6: return march_kernel_rt<6>(p);
        default: return nullptr;
    }
}

// outputs (and ReLU mask) that can be accessed four channels at a time
inline bool rows_by_four(const pvnet_conv& c) {
    if (c.cout % 4 || c.ldy % 4 || (uintptr_t)c.y % (c.flags & PVNET_F32OUT ? 16 : 8)) return false;
    return !c.relu_of || (c.ldr % 4 == 0 && (uintptr_t)c.relu_of % 8 == 0);
}

// The marching kernels take 3x3x3 convolutions whose outputs (and ReLU mask) can be accessed four channels at a
// time; PVNET_GATHER keeps k_conv_fwd.
inline bool march_ok(const pvnet_conv& c, const NetParts& q) {
    if (c.ntaps != 27 || (c.flags & PVNET_GATHER) || !rows_by_four(c)) return false;
    if ((int64_t)c.s.h * c.s.w * c.ldx >= (int64_t)1 << 31) return false;  // plane offsets are 32-bit
    if ((int64_t)(c.s.h / 2) * (c.s.w / 2) * q.ldu >= (int64_t)1 << 31) return false;
    if (q.c0 && (q.ldy0 % 4 || (uintptr_t)q.y0 % 8)) return false;
    // weight rows and the block count are 32-bit too (a block has at least one voxel of every 16 channels)
    return (int64_t)c.cout * c.kpad * 2 < (int64_t)1 << 32 &&
           (int64_t)c.s.nb * c.s.d * c.s.h * c.s.w * ((c.cout + 15) / 16) < (int64_t)1 << 31;
}
