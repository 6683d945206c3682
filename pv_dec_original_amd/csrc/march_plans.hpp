// march_plans.hpp — how the marching convolutions and weight gradients divide a layer: plans from the sizes alone.
//
// Host code without device parts: what conv_march.hpp and wgrad_march.hpp launch, and what a test can ask for on any
// machine.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstdint>

#include "../../include/pvnet.h"

namespace {

constexpr int BK = 32;  // k-values per MFMA step

// one tile plan; LDS quantities in 16-byte units (8 channels of one voxel)
struct MarchPlan {
    int32_t tx, ty, ntx, nty;  // tile and tiles per plane
    int32_t zseg, nzs;         // output planes per block, runs per box
    int32_t hx, hp;            // halo row pitch, halo units of one channel chunk
    int32_t su;                // units of one plane slot
    int32_t nsteps, ng;        // k-steps, channel groups
    int32_t K;
    int32_t g;                 // channel chunks interleaved per voxel in LDS (2, or 1 for odd cin / 8)
    int32_t roll, rt, wm;      // kernel and template arguments
    int32_t wx, wn;            // compute waves over voxels and over channel tiles (ring: 4, 1)
    int32_t lds;               // bytes
};

// the shape a plan is for
struct MarchKey {
    pvnet_shape s;
    int32_t cin, cout;
    bool operator==(const MarchKey& o) const {
        return s.nb == o.s.nb && s.d == o.s.d && s.h == o.s.h && s.w == o.s.w && cin == o.cin && cout == o.cout;
    }
};

// What a block of the marching kernels costs.  cu: clocks of its CU, the larger part of what it asks of the matrix
// cores, the LDS, the L1 (weights read from memory) and the way to memory plus a share of the others; alone: clocks it
// takes by itself, a chain of k-steps and planes with their latencies.  A CU that holds c blocks needs c cu and one
// alone, of which the longer hides part of the other; blocks beyond what the device holds come in further rounds.
// The constants (clocks, launch in us) were fitted to 53,000 timed plans of 1,550 layers (cin 8-224, cout 8-224, 32 to
// 4 M voxels, whole and ragged, boxes of one voxel to 200 a side): rms error 11 % (ring) and 15 % (roll); over 260
// other layers the plan taken is 3.5 % (mean) and at most 41 % slower than the best one timed.  A plan's price decides
// how long a call takes, never what it computes.
struct MarchPrice {
    double launch;
    double mma, lds, l1, in, out;         // per MFMA, fragment read from LDS, weight fragment from L1, unit in, channel out
    double share, few;                    // of the smaller parts; waves too few to keep the CU busy
    double weights[3];                    // per k-step: weights read at the start (by where they are: memory, LDS, registers)
    double start, step[3], mstep;         // alone: the start, a k-step, its MFMAs
    double plane, unit;                   // a plane and its units
    double hide;                          // of the shorter of the two
};
constexpr double CLOCKS_US = 2400;
constexpr MarchPrice RING_PRICE{2.78, 0.0, 5.31, 26.2, 0.372, 0.188, 0.477, 1.05, {0, 77.7, 79.8}, 784, {20.7, 0, 0}, 0.383, 642, 1.99, 2.2};
constexpr MarchPrice ROLL_PRICE{2.06, 0.715, 2.59, 36.1, 0.173, 0.656, 0.9, 0.0, {0, 133, 0}, 968, {0, 0, 0}, 0.644, 1490, 2.93, 0.68};

// registers of a thread, as the compiler reports them (an old figure here costs time only)
inline int march_vgprs(int roll, int rt, int wm, int steps) {
    static const int ring[] = {0, 44, 60, 78, 100, 0, 138}, held[] = {0, 38, 46, 57, 72, 0, 102}, rolled[] = {0, 116, 149, 182, 218, 256};
    return roll ? std::min(256, rolled[rt] + 15 * wm) : wm == 2 ? held[rt] + 4 * steps : ring[rt];
}

// blocks a CU holds at once: 160 KB of LDS in pieces of 1,280 bytes, 512 registers a SIMD lane
inline int blocks_per_cu(int lds, int vgprs, int waves) {
    constexpr int LDS = 160 * 1024, PIECE = 1280;
    return std::max(1, std::min(LDS / ((lds + PIECE - 1) / PIECE * PIECE), 4 * (512 / ((vgprs + 7) / 8 * 8)) / waves));
}

// time of `blocks` blocks of which a CU holds cc, on 256 CUs, in the unit of cu and alone
inline double rounds_of(double blocks, int cc, double cu, double alone, double hide) {
    const double rounds = std::ceil(blocks / (256.0 * cc)), rest = std::ceil((blocks - (rounds - 1) * 256 * cc) / 256);
    auto one = [&](double c) { return std::max(alone, cu * c) + hide * std::min(alone, cu * c); };
    return (rounds - 1) * one(cc) + one(rest);
}

// The plan of a convolution: every tile, run length, wave split and place of the weights that fits is priced and the
// cheapest is taken; us: its price.
inline bool march_search(const MarchKey& c, MarchPlan& best, double& us) {
    const int steps = (27 * c.cin + BK - 1) / BK, ct = (c.cout + 15) / 16, cch = c.cin / 8;
    const int w = c.s.w, h = c.s.h, d = c.s.d;
    us = 0;
    auto axis = [](int n, const int* cut, int ncut, const int* fix, int nfix, int* out) {
        int k = 0;
        auto add = [&](int v) {
            if (v < 1 || v > n) return;
            for (int i = 0; i < k; i++) if (out[i] == v) return;
            out[k++] = v;
        };
        for (int i = 0; i < ncut; i++) add((n + cut[i] - 1) / cut[i]);
        for (int i = 0; i < nfix; i++) add(fix[i]);
        return k;
    };
    static const int cut[] = {1, 2, 3, 4, 5, 6, 8, 12, 16, 24}, fixx[] = {8, 12, 16, 24}, fixy[] = {4, 6, 8, 12, 16};
    int xs[16], ys[16], zs[16];
    const int nx = axis(w, cut, 8, fixx, 4, xs), ny = axis(h, cut, 8, fixy, 5, ys), nz = axis(d, cut, 10, fixy, 0, zs);
    for (int roll = 0; roll < 2; roll++) {
        if (roll ? c.cin % BK != 0 : c.cin > 128) continue;  // a ring of more channels leaves tiles too small
        const int np = roll ? 2 : 4, sp = roll ? steps / 3 : steps;
        for (int ix = 0; ix < nx; ix++)
            for (int iy = 0; iy < ny; iy++) {
                const int tx = xs[ix], ty = ys[iy], vox = tx * ty;
                if (vox > 384 || (vox < 48 && vox < w * h)) continue;
                const int hp = (tx + 2) * (ty + 2), nu = cch * hp, su = (nu + 63) / 64 * 64;
                if (16 * np * su > 160 * 1024) continue;
                const double tiles = (double)((w + tx - 1) / tx) * ((h + ty - 1) / ty) * c.s.nb;
                for (int wx = roll ? 1 : 4; wx <= (roll ? 4 : 4); wx++) {
                    int rt = (vox + 16 * wx - 1) / (16 * wx);
                    if (rt > (roll ? 5 : 6)) continue;
                    if (!roll && rt == 5) rt = 6;
                    if (vox < 48 ? false : vox < 16 * wx * rt * 0.6) continue;
                    for (int wn = 1; wn <= (roll ? 5 : 1) && wn <= ct; wn++) {
                        const int W = wx * wn;
                        if (roll && (W < 2 || W > 5)) continue;
                        for (int wm = 0; wm < (roll ? 2 : 3); wm++) {
                            if (wm == 2 && steps != 7 && steps != 14 && steps != 21 && !(steps == 41 && rt <= 4)) continue;
                            const int lds = 16 * (np * su + (wm == 1 ? 64 * wn * steps : 0)) + 4 * (np * 4 * sp + nu);
                            if (lds > 160 * 1024) continue;
                            const int cc = std::min(16, blocks_per_cu(lds, march_vgprs(roll, rt, wm, steps), W + roll));
                            const MarchPrice& P = roll ? ROLL_PRICE : RING_PRICE;
                            const double wfill = P.weights[wm] * steps * (wm == 1 ? wn : 1);
                            for (int iz = 0; iz < nz; iz++) {
                                const int nzs = (d + zs[iz] - 1) / zs[iz];
                                const double za = (double)d / nzs, pl = za + 2;
                                const double B = tiles * nzs * ((ct + wn - 1) / wn);
                                if (B * 64 * (W + roll) >= 4294967296.0) continue;  // a launch has fewer than 2^32 threads
                                const double nst = roll ? sp * pl : steps * za, mf = steps * za * rt;
                                const double xr = nst * rt, wr = wm == 2 ? 0 : roll ? sp * (3 * za + 2) : steps * za;
                                const double m = P.mma * mf * W, l = P.lds * (xr + (wm == 1 ? wr : 0)) * W,
                                             l1 = wm == 0 ? P.l1 * wr * W : 0.0, io = P.in * pl * nu + P.out * vox * za * wn * 16;
                                const double top = std::max({m, l, l1, io});
                                const double cu = (top + P.share * (m + l + l1 + io - top)) * (1 + P.few / (cc * W)) + 0.5 * wfill;
                                const double step = P.step[wm] + P.mstep * 16 * mf / nst * std::max(1.0, W / 4.0);
                                const double alone = P.start + wfill + nst * step + pl * (P.plane + P.unit * nu / (roll ? 1 : 4));
                                const double cost = P.launch + rounds_of(B, cc, cu, alone, P.hide) / CLOCKS_US;
                                if (us == 0 || cost < us) {
                                    us = cost;
                                    best = MarchPlan{tx, ty, (w + tx - 1) / tx, (h + ty - 1) / ty, zs[iz], nzs, tx + 2, hp, su, steps,
                                                     (ct + wn - 1) / wn, 27 * c.cin, cch % 2 ? 1 : 2, roll, rt, wm, wx, wn, lds};
                                }
                            }
                        }
                    }
                }
            }
    }
    return us > 0;
}

// The gathering convolution's blocks: 256 voxels for narrow outputs on large grids; 64 channels only when the grid still
// has 2,048 blocks (the K loop is long, so the device needs many blocks in flight).
struct GatherTile {
    int32_t bm, bn;
    int64_t blocks;
};

inline GatherTile gather_tile(int64_t M, int cout) {
    const int64_t mt = (M + 127) / 128;
    if (cout <= 16) return M >= (int64_t)256 * 2048 ? GatherTile{256, 16, (M + 255) / 256} : GatherTile{128, 16, mt};
    if (cout % 64 == 0 && mt * (cout / 64) >= 2048) return {128, 64, mt * (cout / 64)};
    return {128, 32, mt * ((cout + 31) / 32)};
}

// us of a 3x3x3 convolution by gathering, fitted to 5,000 timed layers: rms error 10 % (25 % for 256-voxel blocks, which
// marching beats by a factor)
inline double gather_us(int64_t M, int cin, int cout) {
    struct Price {
        double launch, step, cu, block, hide;  // us: a step of a block alone, of 256 blocks, the blocks' own cost
    };
    const GatherTile t = gather_tile(M, cout);
    const Price P = t.bm == 256  ? Price{8.84, 0.487, 0.0965, 3.49, 1.71}
                    : t.bn == 16 ? Price{9.46, 0.396, 0.140, 1.46, 0.289}
                    : t.bn == 64 ? Price{11.2, 0.657, 0.129, 2.49, 0.866}
                                 : Price{11.5, 0.408, 0.148, 1.07, 0.467};
    const double steps = (27 * cin + BK - 1) / BK, rounds = t.blocks / 256.0;
    const double alone = steps * P.step * std::ceil(rounds / 8), cu = steps * P.cu * rounds;
    return P.launch + std::max(alone, cu) + P.hide * std::min(alone, cu) + P.block * rounds;
}

// the plan of a weight gradient
struct WgradMarch {
    int32_t tx, ty, ntx, nty;   // tile (divides the plane) and tiles per plane
    int32_t zseg, nzs;          // planes per run, runs per box
    int32_t hx, hp, gr;         // halo row pitch and size; 32-voxel groups of a tile
    int32_t su, fu;             // LDS units (16 bytes) of one dy and one x plane
    int32_t cf, ns, nf;         // 16-channel tiles of x per block; blocks over the channels of dy and x
    int32_t units, per, splits; // runs in all, runs per block, blocks over the voxels
    int32_t lds;
};

// The plan of a weight gradient, from the sizes alone (the scratch size a caller asks for and the launch agree on
// any device).  Tiles divide the plane, so that no operand needs masking inside a plane.  Every tile, run length
// and CF that fits is priced as above, with the sum over the splits, and the cheapest is taken; us: its price.  Fitted
// to 41,000 timed plans of 1,550 layers, rms error 10 %; over 260 other layers the plan taken is 1.7 % (mean) and at
// most 13 % slower than the best one timed.
inline bool wgrad_march_search(const pvnet_shape& s, int cin, int cout, WgradMarch& best, double& us) {
    constexpr int WANT = 768;  // blocks: three per CU
    static const int vgprs[] = {75, 113, 139};  // of CF = 1, 2, 3
    us = 0;
    static const int cuts[] = {1, 2, 3, 4, 5, 6, 8, 12, 16, 24, 32, 48};
    const int ft = (cin + 15) / 16, st = (cout + 15) / 16;
    for (int tx = 1; tx <= 256 && tx <= s.w; tx++) {
        if (s.w % tx) continue;
        for (int ty = 1; ty <= 64 && ty <= s.h; ty++) {
            const int vox = tx * ty, gr = (vox + 31) / 32, hp = (tx + 2) * (ty + 2);
            if (s.h % ty || vox > 512 || (vox < 32 && vox < s.w * s.h && tx < s.w)) continue;
            for (int cf = 1; cf <= 3 && cf <= ft; cf++) {
                const int su = (2 * hp + 63) / 64 * 64, fu = (2 * cf * gr * 32 + 63) / 64 * 64;
                const int lds = 16 * (4 * su + 2 * fu) + 4 * (gr * 32 + 2 * hp + 2 * cf * gr * 32);
                if (lds > 160 * 1024) continue;
                const int nf = (ft + cf - 1) / cf;
                const int cc = blocks_per_cu(lds, vgprs[cf - 1], 4);
                for (int cut : cuts) {
                    if (cut > s.d) break;
                    const int zseg = (s.d + cut - 1) / cut, nzs = (s.d + zseg - 1) / zseg;
                    const int64_t units = (int64_t)s.nb * (s.w / tx) * (s.h / ty) * nzs;
                    const int want = (int)std::max<int64_t>(1, std::min<int64_t>(units, WANT / (nf * st)));
                    const int per = (int)((units + want - 1) / want), splits = (int)((units + per - 1) / per);
                    const double B = (double)splits * nf * st, za = (double)s.d / nzs;
                    const double alone = per * (881 + 7.67 * hp + 1260 * (za + 2) + za * gr * (238 + 218.0 * cf));
                    const double cu = per * za * (gr * std::max(118.0 * cf, 26.2 * (7 + cf)) + 0.66 * (hp + cf * gr * 32));
                    // the last: looking for columns that are not finite
                    const double cost = 7.28 + rounds_of(B, cc, cu, alone, 0.41) / CLOCKS_US + splits * (6.72e-5 * cin * cout + 6.7e-4) + 8.4e-5 * cin * cout;
                    if (us == 0 || cost < us) {
                        us = cost;
                        best = WgradMarch{tx, ty, s.w / tx, s.h / ty, zseg, nzs, tx + 2, hp, gr, su, fu, cf, st, nf, (int)units, per, splits, lds};
                    }
                }
            }
        }
    }
    return us > 0;
}

// The tiled weight-gradient kernel: bn output channels by 64 k-values a block, the voxels in nsplit runs of mchunk (LDS
// fills of 128 voxels).  At most 2,048 blocks where there are several splits: two rounds of the four that a CU holds
// (one split more began a third: 27 taps, 8 x 24^3, 64 -> 160 309 us, 274 so; 96 -> 96 287 and 256).
struct TiledWgrad {
    int32_t bn, ktiles, ntiles, nsplit, mchunk;
};

inline TiledWgrad tiled_wgrad(int64_t M, int ntaps, int cin, int cout) {
    const int bn = cout <= 16 ? 16 : (cout <= 32 || cout % 64 != 0) ? 32 : 64;
    const int ktiles = (ntaps * cin + 63) / 64, ntiles = (cout + bn - 1) / bn;
    const int64_t want = 2048 / (ktiles * ntiles), fills = (M + 127) / 128;
    const int64_t ns = std::min<int64_t>(std::max<int64_t>(want, 1), std::max<int64_t>(fills, 1)), per = (fills + ns - 1) / ns;
    return {bn, ktiles, ntiles, (int32_t)((M + per * 128 - 1) / (per * 128)), (int32_t)(per * 128)};
}

// us of a 3x3x3 weight gradient by the tiled kernel and its sum over the splits, fitted to 4,900 timed layers: rms error
// 7 % (16 channels), 13 %, 11 %
inline double tiled_wgrad_us(int64_t M, int cin, int cout) {
    struct Price {
        double launch, start, fill, cu, hide, sum, split;  // us
    };
    const TiledWgrad t = tiled_wgrad(M, 27, cin, cout);
    const Price P = t.bn == 16   ? Price{5.23, 0.797, 0.251, 0.435, 1.08, 2.13e-6, 3.1e-3}
                    : t.bn == 32 ? Price{6.07, 0.013, 0.453, 0.425, 1.07, 2.94e-6, 0}
                                 : Price{9.60, 0.030, 0.775, 0.805, 0.338, 2.07e-6, 0};
    const double fills = t.mchunk / 128;
    return P.launch + rounds_of((double)t.ktiles * t.ntiles * t.nsplit, 4, fills * P.cu, P.start + fills * P.fill, P.hide) +
           t.nsplit * (P.sum * 27 * cin * cout + P.split);
}

// The plan of a shape, a pure function of its key, searched once per thread and kept with the others the thread has
// used.  A key sits in the first free slot from its hash on, so that no shape drives out another; a table that is three
// quarters full starts over.  (A network's training step asks for 41 plans; a search takes 10 to 90 us.)
template <class Plan, class Search>
bool kept_plan(const MarchKey& key, Plan& p, Search search) {
    struct Slot {
        MarchKey key;
        Plan plan;
        int ok;  // 0 empty, 1 plan, 2 no plan
    };
    constexpr int SLOTS = 512, FULL = SLOTS / 4 * 3;
    thread_local Slot slots[SLOTS];
    thread_local int used = 0;
    uint32_t hsh = 2166136261u;
    for (int32_t v : {key.s.nb, key.s.d, key.s.h, key.s.w, key.cin, key.cout}) hsh = (hsh ^ (uint32_t)v) * 16777619u;
    const uint32_t home = (hsh ^ (hsh >> 15)) % SLOTS;
    uint32_t i = home;
    while (slots[i].ok && !(slots[i].key == key)) i = (i + 1) % SLOTS;
    if (!slots[i].ok) {
        if (used == FULL) {
            for (Slot& s : slots) s.ok = 0;
            used = 0;
            i = home;
        }
        slots[i].key = key;
        slots[i].ok = search(key, slots[i].plan) ? 1 : 2;
        used++;
    }
    p = slots[i].plan;
    return slots[i].ok == 1;
}

inline int64_t voxels(const pvnet_shape& s) { return (int64_t)s.nb * s.d * s.h * s.w; }

// The route of a layer: marching where a plan fits and costs no more than the kernel it takes the place of.  That one is
// the cheaper on small or thin planes, where a tile is mostly halo, for deep inputs on few voxels, and for weight
// gradients of few voxels.  Measured, us, marching and the other: convolutions 8 x 52 x 6 x 12 120 -> 56 161 and 62, 64
// x 30 x 3 x 2 112 -> 216 524 and 70, 8 x 48^3 96 -> 32 221 and 442; weight gradients 256 x 2^3 96 -> 32 34 and 12, 8 x 6
// x 2 x 2 160 -> 160 41 and 26, 1 x 88 x 8 x 8 8 -> 16 10.7 and 7.5, 8 x 24^3 64 -> 64 50 and 109.
inline bool march_route(const MarchKey& k, MarchPlan& p) {
    double us;
    return march_search(k, p, us) && us <= gather_us(voxels(k.s), k.cin, k.cout);
}

inline bool wgrad_route(const MarchKey& k, WgradMarch& p) {
    const int64_t M = voxels(k.s);
    double us;
    return M < (int64_t)1 << 31 && wgrad_march_search(k.s, k.cin, k.cout, p, us) && us <= tiled_wgrad_us(M, k.cin, k.cout);
}

inline bool march_plan(const pvnet_shape& s, int cin, int cout, MarchPlan& p) { return kept_plan(MarchKey{s, cin, cout}, p, march_route); }

inline bool wgrad_march_plan(const pvnet_shape& s, int cin, int cout, WgradMarch& p) {
    return kept_plan(MarchKey{s, cin, cout}, p, wgrad_route);
}

}  // namespace
