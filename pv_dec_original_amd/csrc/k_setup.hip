// k_setup.hip — set-up kernels for gfx950: ray-cast voxelisation, boundary detection,
// next-to-wall marking and boundary normals.

#include <hip/hip_runtime.h>

#include "kernels.hpp"
#include "lbm_device.hpp"

namespace pvlbm {

namespace {

// Geometry::isPointInsideTriangle (ComplexGeometry.cpp:620-674), same operation order.
__device__ __forceinline__ bool point_in_triangle(double x, double y, double z, const double* T) {
    double x1 = T[0], y1 = T[1], z1 = T[2];
    double x2 = T[3], y2 = T[4], z2 = T[5];
    double x3 = T[6], y3 = T[7], z3 = T[8];
    double dirX = 0.0, dirY = 0.0, dirZ = 1.0;
    double uX = x2 - x1, uY = y2 - y1, uZ = z2 - z1;
    double vX = x3 - x1, vY = y3 - y1, vZ = z3 - z1;
    double nX = uY * vZ - uZ * vY;
    double nY = uZ * vX - uX * vZ;
    double nZ = uX * vY - uY * vX;
    double nLengthSq = nX * nX + nY * nY + nZ * nZ;
    const double tol = 1e-16;
    if (nLengthSq < tol * tol) return false;
    double w0X = x - x1, w0Y = y - y1, w0Z = z - z1;
    double a = -(nX * w0X + nY * w0Y + nZ * w0Z);
    double b = nX * dirX + nY * dirY + nZ * dirZ;
    if (fabs(b) < tol) return false;
    double pos = a / b;
    double ix = x + pos * dirX;
    double iy = y + pos * dirY;
    double iz = z + pos * dirZ;
    double uu = uX * uX + uY * uY + uZ * uZ;
    double uv = uX * vX + uY * vY + uZ * vZ;
    double vv = vX * vX + vY * vY + vZ * vZ;
    double wX = ix - x1, wY = iy - y1, wZ = iz - z1;
    double wu = wX * uX + wY * uY + wZ * uZ;
    double wv = wX * vX + wY * vY + wZ * vZ;
    double D = uv * uv - uu * vv;
    double s = (uv * wv - vv * wu) / D;
    if (s < 0.0 || s > 1.0) return false;
    double t = (uv * wu - uu * wv) / D;
    if (t < 0.0 || (s + t) > 1.0) return false;
    return true;
}

// One triangle of Geometry::countIntersectinsTriangle (ComplexGeometry.cpp:807-845).
__device__ __forceinline__ bool crosses(const double* T, const double s[3], const double e[3]) {
    const double threshold = 1e-16;
    double px = s[0], py = s[1], pz = s[2];
    double dx = e[0] - s[0], dy = e[1] - s[1], dz = e[2] - s[2];
    double nx = T[9], ny = T[10], nz = T[11];
    double qx = T[0], qy = T[1], qz = T[2];
    double numerator = (qx - px) * nx + (qy - py) * ny + (qz - pz) * nz;
    double denominator = dx * nx + dy * ny + dz * nz;
    if (fabs(denominator) < threshold) return false;
    double t = numerator / denominator;
    if (t >= 0.0 && t <= 1.0) {
        double ix = px + t * dx;
        double iy = py + t * dy;
        double iz = pz + t * dz;
        if (point_in_triangle(ix, iy, iz, T)) return true;
    }
    return false;
}

// Geometry::FindLineTriangleIntersection (ComplexGeometry.cpp:689-730), same operation order:
// plane of the file normal through vertex 1, |denominator| >= 1e-7, 0 <= t <= 1, then the
// point-in-triangle test of the voxeliser.
__device__ __forceinline__ bool line_triangle(const double* T, const double* s, const double* e, double ip[3]) {
    const double threshold = 1e-7;
    double px = s[0], py = s[1], pz = s[2];
    double dx = e[0] - s[0], dy = e[1] - s[1], dz = e[2] - s[2];
    double nx = T[9], ny = T[10], nz = T[11];
    double qx = T[0], qy = T[1], qz = T[2];
    double denom = (dx * nx + dy * ny + dz * nz);
    if (fabs(denom) < threshold) return false;
    double t = ((qx - px) * nx + (qy - py) * ny + (qz - pz) * nz) / denom;
    if (t < 0.0 || t > 1.0) return false;
    double ix = px + t * dx;
    double iy = py + t * dy;
    double iz = pz + t * dz;
    if (point_in_triangle(ix, iy, iz, T)) {
        ip[0] = ix;
        ip[1] = iy;
        ip[2] = iz;
        return true;
    }
    return false;
}

// One wave per (i, j) column; its lanes walk the column's points in z.  The candidate triangles
// of a column are the same for every lane, so their loads are wave-uniform.
__global__ __launch_bounds__(64) void k_voxelize(const VoxParams p) {
    const int64_t col = blockIdx.x;
    const int64_t i = col % p.nx, j = col / p.nx;
    const int64_t c0 = p.col_off[col], c1 = p.col_off[col + 1];
    const double rayOffset = 0.02;
    for (int64_t k = threadIdx.x; k < p.nz; k += 64) {
        // point = min + idx*spacing (ComplexGeometry.cpp:337-340); ray of labelPoints (:989-1003)
        // and adjustLineCoordinates case 0 (:855-884)
        double x = p.ox + (double)i * p.h;
        double y = p.oy + (double)j * p.h;
        double z = p.oz + (double)k * p.h;
        double s[3] = {x, y, z + p.h / 2};
        double rayLength = p.bb[5] - p.bb[4];
        double e[3] = {x, y, z + rayLength + 0.1};
        if (s[0] == p.bb[0]) { s[0] += rayOffset; e[0] += rayOffset; }
        if (s[0] == p.bb[1]) { s[0] -= rayOffset; e[0] -= rayOffset; }
        if (s[1] == p.bb[2]) { s[1] += rayOffset; e[1] += rayOffset; }
        if (s[1] == p.bb[3]) { s[1] -= rayOffset; e[1] -= rayOffset; }
        if (s[2] == p.bb[4]) { s[2] += rayOffset; }
        if (e[2] == p.bb[5]) { e[2] -= rayOffset; }
        int count = 0;
        for (int64_t c = c0; c < c1; c++) {
            const double* T = p.tri + 12 * (int64_t)p.col_tri[c];
            if (crosses(T, s, e)) count++;
        }
        p.fluid[i + (int64_t)p.nx * (j + (int64_t)p.ny * k)] = (count % 2 == 1) ? 1 : 0;
    }
}

// findBoundaryPoints (ComplexGeometry.cpp:1259-1300) over the Q directions: a fluid node is a
// boundary node when a Q neighbour is outside the box or not fluid.
template <int Q>
__global__ __launch_bounds__(256) void k_boundary(const uint8_t* fluid, int64_t nxp, int64_t nyp,
                                                 int64_t nx, int64_t ny, int64_t nz, uint8_t* bflag) {
    const int64_t n = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t total = nxp * nyp * nz;
    if (n >= total) return;
    const int64_t i = n % nxp, j = (n / nxp) % nyp, k = n / (nxp * nyp);
    if (!fluid[n]) {
        bflag[n] = 0;
        return;
    }
    uint32_t m = 0;
#pragma unroll
    for (int d = 0; d < Q; d++) {
        const int64_t a = i + Lat<Q>::cx[d], b = j + Lat<Q>::cy[d], c = k + Lat<Q>::cz[d];
        const bool inside = a >= 0 && a < nx && b >= 0 && b < ny && c >= 0 && c < nz;
        if (!inside || !fluid[a + nxp * (b + nyp * c)]) m |= 1u << d;
    }
    bflag[n] = m != 0;
}

// IdentifyNextToWallLattices (Subdomain.cpp:201-218): interior fluid nodes linked to a wall node.
// Interior nodes have all Q neighbours inside the box.
template <int Q>
__global__ __launch_bounds__(256) void k_ntw(uint8_t* kind, int64_t nxp, int64_t nyp, int64_t nz) {
    const int64_t n = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (n >= nxp * nyp * nz) return;
    if (kind[n] != K_FLUID) return;
    bool near_wall = false;
#pragma unroll
    for (int d = 0; d < Q; d++) {
        const int64_t o = Lat<Q>::cx[d] + nxp * (Lat<Q>::cy[d] + nyp * Lat<Q>::cz[d]);
        near_wall |= kind[n + o] == K_WALL;
    }
    if (near_wall) kind[n] = K_NTW;
}

// Per-triangle quantities of calculateBoundaryNormals (Subdomain.cpp:318-341): unit
// cross-product normal, area, centroid.  prep planes: nx, ny, nz, area, cx, cy, cz.
__global__ __launch_bounds__(256) void k_tri_prep(const double* tri, int64_t ntri, double* prep) {
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= ntri) return;
    const double* T = tri + 12 * t;
    double ux = T[3] - T[0], uy = T[4] - T[1], uz = T[5] - T[2];
    double vx = T[6] - T[0], vy = T[7] - T[1], vz = T[8] - T[2];
    double nx = uy * vz - uz * vy;
    double ny = uz * vx - ux * vz;
    double nz = ux * vy - uy * vx;
    double norm = sqrt(nx * nx + ny * ny + nz * nz);
    if (norm > 0) {
        nx /= norm;
        ny /= norm;
        nz /= norm;
    }
    prep[t] = nx;
    prep[ntri + t] = ny;
    prep[2 * ntri + t] = nz;
    prep[3 * ntri + t] = 0.5 * norm;
    prep[4 * ntri + t] = (T[0] + T[3] + T[6]) / 3.0;
    prep[5 * ntri + t] = (T[1] + T[4] + T[7]) / 3.0;
    prep[6 * ntri + t] = (T[2] + T[5] + T[8]) / 3.0;
}

// Normal of each listed node: sum over all triangles of unit normal * area / distance^2, then normalised
// (Subdomain.cpp:343-368).  The sums run in triangle file order as the reference's do, one chain per node and
// component; what a chain adds, the weight area / distance^2 with its FP64 square root and division, is
// independent of it.  So most threads of a block compute the weights of a chunk of triangles for its NODES nodes
// into LDS while others, one per (component, node), add the chunk before: the reference's roundings, with the
// costly part spread over the chip even when there are few nodes (whole set-up of a subdomain with 16823 such
// nodes and 162664 triangles 31.1 ms with one thread a node, 14.3 this way).  Bound by the FP64
// rate (about 300 clocks a triangle, wave and SIMD) and, with few nodes, by how evenly the blocks fall on the CUs.
constexpr int NRM_CH = 64;  // triangles per chunk, 8 consecutive ones per weight thread

template <int NODES>
constexpr int nrm_threads() { return NODES * NRM_CH / 8 + (3 * NODES + 63) / 64 * 64; }

template <int NODES>
__global__ __launch_bounds__(nrm_threads<NODES>()) void k_normals(const double* __restrict__ prep, int64_t ntri,
                                                                const double* __restrict__ xyz, int64_t n,
                                                                double* __restrict__ nrm) {
    constexpr int WT = NODES * NRM_CH / 8;  // weight threads: whole waves
    constexpr int UNR = NODES == 64 ? 16 : 8;  // 64: hides the LDS reads, 106773 nodes 295 ms (8: 322)
    __shared__ double Wt[2][NRM_CH][NODES];
    const int t = threadIdx.x, node = t % NODES;
    const int64_t w = (int64_t)blockIdx.x * NODES + node;
    const bool act = w < n;
    const int64_t nch = (ntri + NRM_CH - 1) / NRM_CH;
    double a = 0.0;
    if (t < WT) {
        const double x = act ? xyz[w] : 0.0, y = act ? xyz[n + w] : 0.0, z = act ? xyz[2 * n + w] : 0.0;
        // NODES = 64: a wave's triangles are the same for all lanes (scalar loads)
        const int k0 = 8 * (NODES == 64 ? __builtin_amdgcn_readfirstlane(t >> 6) : t / NODES);
        auto weight = [&](int64_t i) {
            const double cX = prep[4 * ntri + i], cY = prep[5 * ntri + i], cZ = prep[6 * ntri + i];
            const double distance = sqrt((x - cX) * (x - cX) + (y - cY) * (y - cY) + (z - cZ) * (z - cZ));
            return prep[3 * ntri + i] / (distance * distance);
        };
        for (int64_t ch = 0; ch <= nch; ch++) {
            const int64_t t0 = ch * NRM_CH + k0;
            if (t0 + 8 <= ntri) {
#pragma unroll
                for (int k = 0; k < 8; k++) Wt[ch & 1][k0 + k][node] = weight(t0 + k);
            } else {
                for (int k = 0; k < 8; k++)
                    if (t0 + k < ntri) Wt[ch & 1][k0 + k][node] = weight(t0 + k);
            }
            __syncthreads();  // chunk ch is there, chunk ch - 1 is consumed
        }
    } else {
        const int c = NODES == 64 ? __builtin_amdgcn_readfirstlane((t - WT) >> 6) : (t - WT) / NODES;
        const double* C = prep + (c < 3 ? c : 2) * ntri;  // threads past the third component repeat it unused
        for (int64_t ch = 0; ch <= nch; ch++) {
            if (ch > 0) {
                const double(*W)[NODES] = Wt[(ch - 1) & 1];
                const int64_t t0 = (ch - 1) * NRM_CH;
                if (t0 + NRM_CH <= ntri) {
#pragma unroll(UNR)
                    for (int k = 0; k < NRM_CH; k++) a += C[t0 + k] * W[k][node];
                } else {
                    for (int64_t i = t0; i < ntri; i++) a += C[i] * W[i - t0][node];
                }
            }
            __syncthreads();
        }
        // the three components of a node sit in three threads: gathered in LDS (free after the last barrier)
        if (c < 3) Wt[0][c][node] = a;
    }
    __syncthreads();
    if (t >= NODES || !act) return;
    double n0 = Wt[0][0][t], n1 = Wt[0][1][t], n2 = Wt[0][2][t];
    const double norm = sqrt(n0 * n0 + n1 * n1 + n2 * n2);
    if (norm > 0) {
        n0 /= norm;
        n1 /= norm;
        n2 /= norm;
    }
    nrm[w] = n0;
    nrm[n + w] = n1;
    nrm[2 * n + w] = n2;
}

}  // namespace

hipError_t launch_voxelize(const VoxParams& p, hipStream_t s) {
    const int64_t cols = (int64_t)p.nx * p.ny;
    if (cols <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_voxelize, dim3((unsigned)cols), dim3(64), 0, s, p);
    return hipGetLastError();
}

hipError_t launch_boundary(int q, const uint8_t* fluid_pad, int64_t nxp, int64_t nyp, int64_t nx,
                           int64_t ny, int64_t nz, uint8_t* bflag, hipStream_t s) {
    const int64_t total = nxp * nyp * nz;
    const unsigned g = (unsigned)((total + 255) / 256);
    if (q == 19) hipLaunchKernelGGL(k_boundary<19>, dim3(g), dim3(256), 0, s, fluid_pad, nxp, nyp, nx, ny, nz, bflag);
    else hipLaunchKernelGGL(k_boundary<27>, dim3(g), dim3(256), 0, s, fluid_pad, nxp, nyp, nx, ny, nz, bflag);
    return hipGetLastError();
}

hipError_t launch_ntw(int q, uint8_t* kind, int64_t nxp, int64_t nyp, int64_t nz, hipStream_t s) {
    const int64_t total = nxp * nyp * nz;
    const unsigned g = (unsigned)((total + 255) / 256);
    if (q == 19) hipLaunchKernelGGL(k_ntw<19>, dim3(g), dim3(256), 0, s, kind, nxp, nyp, nz);
    else hipLaunchKernelGGL(k_ntw<27>, dim3(g), dim3(256), 0, s, kind, nxp, nyp, nz);
    return hipGetLastError();
}

hipError_t launch_tri_prep(const double* tri, int64_t ntri, double* prep, hipStream_t s) {
    if (ntri <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_tri_prep, dim3((unsigned)((ntri + 255) / 256)), dim3(256), 0, s, tri, ntri, prep);
    return hipGetLastError();
}

hipError_t launch_normals(const double* prep, int64_t ntri, const double* xyz, int64_t n, double* nrm,
                          hipStream_t s) {
    if (n <= 0) return hipSuccess;
    // 64 nodes a block read the triangles by scalar loads, which is 10 % less work a pair; 16 divide few nodes
    // more evenly over the chip.  The line is four blocks of 64 nodes a CU, where the unevenness (one block in
    // four at most) has come down to that: 16823 nodes, 162664 triangles 17.8 ms with 64 and 14.3 with 16;
    // 106773 nodes, 850648 triangles 295 with 64 and 330 with 16 (whole set-up of the subdomain).
    if (n >= 4 * 256 * 64)
        hipLaunchKernelGGL(k_normals<64>, dim3((unsigned)((n + 63) / 64)), dim3(nrm_threads<64>()), 0, s, prep,
                           ntri, xyz, n, nrm);
    else
        hipLaunchKernelGGL(k_normals<16>, dim3((unsigned)((n + 15) / 16)), dim3(nrm_threads<16>()), 0, s, prep,
                           ntri, xyz, n, nrm);
    return hipGetLastError();
}

}  // namespace pvlbm

namespace pvlbm {

namespace {

// Streaming copy at the attainable HBM rate, used to calibrate HBM traffic counters against a
// kernel whose bytes are known exactly and as the copy ceiling the benchmark reports: each block
// moves one 16 KiB chunk, each thread four 16-byte vectors 4 KiB apart (four loads in flight,
// then four nontemporal stores); a partial last chunk is copied vector by vector.
typedef double dvec2 __attribute__((ext_vector_type(2)));
__global__ __launch_bounds__(256) void k_copy(const dvec2* __restrict__ src, dvec2* __restrict__ dst, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * 1024 + threadIdx.x;
    if (i + 768 < n) {
        const dvec2 v0 = src[i], v1 = src[i + 256], v2 = src[i + 512], v3 = src[i + 768];
        __builtin_nontemporal_store(v0, dst + i);
        __builtin_nontemporal_store(v1, dst + i + 256);
        __builtin_nontemporal_store(v2, dst + i + 512);
        __builtin_nontemporal_store(v3, dst + i + 768);
    } else {
        for (int k = 0; k < 4; k++)
            if (i + 256 * k < n) dst[i + 256 * k] = src[i + 256 * k];
    }
}

}  // namespace

// link fractions: one thread per segment, candidates from the cells its bounding box touches
__global__ void k_link_q(const double* seg, int64_t npairs, const double* tri, const int32_t* cell_start,
                         const int32_t* cell_tri, double ogx, double ogy, double ogz, double cs, int ncx, int ncy,
                         int ncz, double h, int nearest, double* q) {
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= npairs) return;
    const double* s = seg + 6 * p;
    const double* e = s + 3;
    const double og[3] = {ogx, ogy, ogz};
    const int nc[3] = {ncx, ncy, ncz};
    int c0[3], c1[3];
    for (int a = 0; a < 3; a++) {
        const double lo = fmin(s[a], e[a]) - 1e-9 * cs, hi = fmax(s[a], e[a]) + 1e-9 * cs;
        c0[a] = min(max((int)floor((lo - og[a]) / cs), 0), nc[a] - 1);
        c1[a] = min(max((int)floor((hi - og[a]) / cs), 0), nc[a] - 1);
    }
    // nearest == 0: the triangle of smallest index (the reference's first in file order);
    // nearest == 1: the intersection closest to the start (the wall the link meets first)
    int32_t best = INT32_MAX;
    double bestd = 1e300;
    double ip[3] = {0.0, 0.0, 0.0};
    for (int cz = c0[2]; cz <= c1[2]; cz++)
        for (int cy = c0[1]; cy <= c1[1]; cy++)
            for (int cx = c0[0]; cx <= c1[0]; cx++) {
                const int64_t c = ((int64_t)cz * nc[1] + cy) * nc[0] + cx;
                for (int32_t k = cell_start[c]; k < cell_start[c + 1]; k++) {
                    const int32_t t = cell_tri[k];
                    if (!nearest && t >= best) break;  // ascending within a cell
                    double hit[3];
                    if (line_triangle(tri + 12 * (int64_t)t, s, e, hit)) {
                        const double dd = (hit[0] - s[0]) * (hit[0] - s[0]) + (hit[1] - s[1]) * (hit[1] - s[1]) +
                                          (hit[2] - s[2]) * (hit[2] - s[2]);
                        if (nearest && (dd > bestd || (dd == bestd && t > best))) continue;
                        best = t;
                        bestd = dd;
                        ip[0] = hit[0];
                        ip[1] = hit[1];
                        ip[2] = hit[2];
                        if (!nearest) break;
                    }
                }
            }
    if (best == INT32_MAX) {
        q[p] = -1.0;
        return;
    }
    const double d = sqrt((ip[0] - s[0]) * (ip[0] - s[0]) + (ip[1] - s[1]) * (ip[1] - s[1]) +
                          (ip[2] - s[2]) * (ip[2] - s[2]));
    q[p] = d / h;
}

hipError_t launch_link_q(const double* seg, int64_t npairs, const double* tri, const int32_t* cell_start,
                         const int32_t* cell_tri, const double og[3], double cs, const int32_t nc[3], double h,
                         int nearest, double* q, hipStream_t s) {
    if (npairs <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_link_q, dim3((unsigned)((npairs + 255) / 256)), dim3(256), 0, s, seg, npairs, tri,
                       cell_start, cell_tri, og[0], og[1], og[2], cs, nc[0], nc[1], nc[2], h, nearest, q);
    return hipGetLastError();
}

// coarse-field expansion for starts from a network prediction
__device__ __forceinline__ float coarse_coord(int64_t i, int64_t n, int c, int& i0, int& i1) {
    float x = ((float)i + 0.5f) * (float)c / (float)n - 0.5f;
    x = fminf(fmaxf(x, 0.f), (float)(c - 1));
    i0 = (int)floorf(x);
    i1 = min(i0 + 1, c - 1);
    return x - (float)i0;
}

// The field is expanded at the nodes alone, tile by tile, into the macro planes the handle already holds, and the
// plane fluxes come from a first pass that samples u_x again instead of storing it.  On the 1024 x 512 x 512
// aneurysm (6.45 M nodes of 268 M points, 192 x 96 x 96 coarse) the fluxes take 89 + 21 us and the fields 83 us.
// Filling four FP64 planes of the whole box in a buffer of its own instead took 5.5 ms, and allocating and
// freeing that buffer (9.2 GB) up to 250 ms a call.
// Trilinear sample of the coarse field at box point (x, y, z): rho and u in FP32, false if not finite.
struct CoarseField {
    const float* rho;
    const float* u;
    int cx, cy, cz;
    int64_t nx, ny, nz;
};

template <int C0, int C1>
__device__ __forceinline__ void coarse_sample(const CoarseField& F, int64_t x, int64_t y, int64_t z, float (&v)[4]) {
    int x0, x1, y0, y1, z0, z1;
    const float fx = coarse_coord(x, F.nx, F.cx, x0, x1);
    const float fy = coarse_coord(y, F.ny, F.cy, y0, y1);
    const float fz = coarse_coord(z, F.nz, F.cz, z0, z1);
    const int64_t plane = (int64_t)F.cx * F.cy * F.cz;
#pragma unroll
    for (int c = C0; c < C1; c++) {
        const float* f = c == 0 ? F.rho : F.u + (c - 1) * plane;
        auto at = [&](int zz, int yy, int xx) { return f[((int64_t)zz * F.cy + yy) * F.cx + xx]; };
        const float a = at(z0, y0, x0) * (1.f - fx) + at(z0, y0, x1) * fx;
        const float b = at(z0, y1, x0) * (1.f - fx) + at(z0, y1, x1) * fx;
        const float cc = at(z1, y0, x0) * (1.f - fx) + at(z1, y0, x1) * fx;
        const float d = at(z1, y1, x0) * (1.f - fx) + at(z1, y1, x1) * fx;
        v[c] = (a * (1.f - fy) + b * fy) * (1.f - fz) + (cc * (1.f - fy) + d * fy) * fz;
    }
}

__device__ __forceinline__ bool finite4(const float (&v)[4]) {
    return isfinite(v[0]) && isfinite(v[1]) && isfinite(v[2]) && isfinite(v[3]);
}

// *flag = 1 if a coarse value is not finite or so large that a blend of finite values might not be: only
// then can a sample be non-finite
__global__ void k_coarse_suspect(const float* rho_c, const float* u_c, int64_t n, int* flag) {
    bool bad = false;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < 4 * n; i += (int64_t)gridDim.x * blockDim.x) {
        const float v = i < n ? rho_c[i] : u_c[i - n];
        bad |= !(fabsf(v) < 1e38f);
    }
    if (bad) *flag = 1;
}

// the number of box points whose sample is not finite (none unless the flag is set)
__global__ __launch_bounds__(256) void k_coarse_count(const CoarseField F, const int* flag, unsigned long long* nonfin) {
    if (!*flag) return;
    const int64_t n = F.nx * F.ny * F.nz;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        const int64_t r = i / F.nx;
        float v[4];
        coarse_sample<0, 4>(F, i % F.nx, r % F.ny, r / F.ny, v);
        if (!finite4(v)) atomicAdd(nonfin, 1ull);
    }
}

// Flux of u_x through each plane x over the nodes: a block walks a run of tiles, each wave adding its tiles'
// samples into its own LDS row of XR tile columns (blockIdx.y picks them) in tile order, and writes the sum of
// its waves' rows; k_flux_final adds the blocks.  Fixed order throughout.  Sampling u_x twice (here and in
// k_expand_nodes) costs less than writing and re-reading the field would.
constexpr int FLUX_XR = 16, FLUX_BLOCKS = 512;

__global__ __launch_bounds__(256) void k_flux_nodes(const CoarseField F, int64_t nxp, int64_t nyp, const TileDesc* tdesc,
                                                    int ntiles, double* part) {
    __shared__ double sh[4][FLUX_XR * 64];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    for (int i = threadIdx.x; i < 4 * FLUX_XR * 64; i += 256) (&sh[0][0])[i] = 0.0;
    __syncthreads();
    const int nxt = (int)(nxp / 64), xt0 = blockIdx.y * FLUX_XR;
    const int per = (ntiles + gridDim.x - 1) / gridDim.x, t1 = min(ntiles, ((int)blockIdx.x + 1) * per);
    for (int t = blockIdx.x * per + wv; t < t1; t += 4) {
        const int tile = tdesc[t].tile, row = tile / nxt, xt = tile - row * nxt;
        if (xt < xt0 || xt >= xt0 + FLUX_XR || !((tdesc[t].node >> lane) & 1ull)) continue;
        float v[4];
        coarse_sample<0, 4>(F, 64 * xt + lane, row % (int)nyp, row / (int)nyp, v);
        if (finite4(v)) sh[wv][64 * (xt - xt0) + lane] += (double)v[1];
    }
    __syncthreads();
    for (int i = threadIdx.x; i < FLUX_XR * 64; i += 256) {
        const int64_t x = 64ll * xt0 + i;
        if (x < nxp) part[blockIdx.x * nxp + x] = ((sh[0][i] + sh[1][i]) + sh[2][i]) + sh[3][i];
    }
}

// flux[x] = the blocks' sums: 8 row groups of 32 planes a block, each in ascending order, then the groups
__global__ __launch_bounds__(256) void k_flux_final(const double* part, int nblocks, int64_t nxp, int64_t nx, double* flux) {
    __shared__ double sh[8][32];
    const int c = threadIdx.x & 31, r = threadIdx.x >> 5;
    const int64_t x = (int64_t)blockIdx.x * 32 + c;
    double s = 0.0;
    if (x < nx)
        for (int b = r; b < nblocks; b += 8) s += part[b * nxp + x];
    sh[r][c] = s;
    __syncthreads();
    if (r == 0 && x < nx) {
        for (int k = 1; k < 8; k++) s += sh[k][c];
        flux[x] = s;
    }
}

// The expanded field at the nodes, one wave per tile: the coarse sample (rest where it is not finite), its
// density clipped, the velocity of plane x scaled by target / flux[x] (limited to [1/4, 4]; planes without flux
// keep theirs), drho[x] added to the density, which is clipped again, speeds clipped to umax.  Only the slots of
// nodes are written: nothing reads the others.
__global__ __launch_bounds__(256) void k_expand_nodes(const CoarseField F, int64_t nxp, int64_t nyp, int64_t ns,
                                                      const TileDesc* tdesc, int ntiles, double rlo, double rhi,
                                                      const double* flux, double target, const double* targets,
                                                      const double* drho, double umax, double* out) {
    const int t = blockIdx.x * 4 + (int)(threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (t >= ntiles) return;
    const int tile = tdesc[t].tile, nxt = (int)(nxp / 64), row = tile / nxt;
    if (!((tdesc[t].node >> lane) & 1ull)) return;
    const int64_t n = (int64_t)tile * 64 + lane, x = 64 * (tile - row * nxt) + lane;
    float v[4];
    coarse_sample<0, 4>(F, x, row % (int)nyp, row / (int)nyp, v);
    double r = 1.0, u0 = 0.0, u1 = 0.0, u2 = 0.0;
    if (finite4(v)) {
        r = fmin(fmax((double)v[0], rlo), rhi);
        u0 = v[1];
        u1 = v[2];
        u2 = v[3];
    }
    if (targets) target = targets[x];
    double f = 1.0;
    if (flux && target > 0.0 && flux[x] > 1e-12 * target) f = fmin(fmax(target / flux[x], 0.25), 4.0);
    if (drho) r = fmin(fmax(r + drho[x], rlo), rhi);
    u0 *= f;
    u1 *= f;
    u2 *= f;
    const double sp = sqrt(u0 * u0 + u1 * u1 + u2 * u2);
    if (sp > umax) {
        const double c = umax / sp;
        u0 *= c;
        u1 *= c;
        u2 *= c;
    }
    out[n] = r;
    out[ns + n] = u0;
    out[2 * ns + n] = u1;
    out[3 * ns + n] = u2;
}

int flux_blocks(int ntiles) { return ntiles < 4 * FLUX_BLOCKS ? (ntiles + 3) / 4 : FLUX_BLOCKS; }

int64_t expand_coarse_doubles(int64_t nx, int64_t nxp, int ntiles) { return 3 * nx + 2 + (int64_t)flux_blocks(ntiles) * nxp; }

hipError_t launch_expand_coarse(const float* rho_c, const float* u_c, int cx, int cy, int cz, int64_t nx, int64_t ny,
                                int64_t nz, int64_t nxp, int64_t nyp, int64_t ns, const TileDesc* tdesc, int ntiles,
                                double umax, double rlo, double rhi, double flux_x, const double* targets,
                                const double* drho, double* flux, double* part, int* flag, double* out,
                                unsigned long long* nonfin, hipStream_t s) {
    const CoarseField F{rho_c, u_c, cx, cy, cz, nx, ny, nz};
    const int64_t nc = (int64_t)cx * cy * cz;
    hipLaunchKernelGGL(k_coarse_suspect, dim3((unsigned)(nc / 256 < 1024 ? nc / 256 + 1 : 1024)), dim3(256), 0, s, rho_c, u_c, nc, flag);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_coarse_count, dim3(2048), dim3(256), 0, s, F, flag, nonfin);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (ntiles <= 0) return hipSuccess;
    const bool scale = flux_x > 0.0 || targets;
    if (scale) {
        const int nb = flux_blocks(ntiles);
        hipLaunchKernelGGL(k_flux_nodes, dim3(nb, (unsigned)((nxp / 64 + FLUX_XR - 1) / FLUX_XR)), dim3(256), 0, s, F, nxp, nyp, tdesc, ntiles, part);
        e = hipGetLastError();
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(k_flux_final, dim3((unsigned)((nx + 31) / 32)), dim3(256), 0, s, part, nb, nxp, nx, flux);
        e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(k_expand_nodes, dim3((unsigned)((ntiles + 3) / 4)), dim3(256), 0, s, F, nxp, nyp, ns, tdesc, ntiles,
                       rlo, rhi, scale ? flux : nullptr, flux_x, targets, drho, umax, out);
    return hipGetLastError();
}

// Compact FP32 fields, PT consecutive points of a row per thread (VEC: four, with 16-byte stores).  Bound by the
// output's 16 bytes a point: most points are not nodes and read one kind byte.  1024 x 512 x 512: 1.03 ms
// (4.4 TB/s), 1.30 ms with one point and 64-bit divisions per thread.
template <bool VEC, int PT>
__global__ __launch_bounds__(256) void k_macros_f32(const double* macro, const uint8_t* kind, int64_t nx, uint32_t ny, int64_t nbox,
                                                    uint32_t nq, uint32_t quads, int64_t nxp, int64_t nyp, int64_t ns, float* rho, float* u) {
    const uint32_t q = blockIdx.x * 256 + threadIdx.x;
    if (q >= quads) return;
    const uint32_t row = q / nq;
    const int64_t i = PT * (int64_t)(q - row * nq), r = (int64_t)row;
    const int64_t n = ((int64_t)(row % ny) + nyp * (int64_t)(row / ny)) * nxp + i, b = r * nx + i;
    // rows are padded: four kinds are always within the row
    const uint32_t k4 = PT == 4 ? *reinterpret_cast<const uint32_t*>(kind + n) : kind[n];
    float v[4][PT];
#pragma unroll
    for (int e = 0; e < PT; e++) {
        const bool node = (k4 >> (8 * e)) & 0xffu;
        v[0][e] = node ? (float)macro[n + e] : 1.0f;
#pragma unroll
        for (int c = 1; c < 4; c++) v[c][e] = node ? (float)macro[c * ns + n + e] : 0.0f;
    }
#pragma unroll
    for (int c = 0; c < 4; c++) {
        float* dst = (c == 0 ? rho : u + (c - 1) * nbox) + b;
        if constexpr (VEC) {
            typedef float f4 __attribute__((ext_vector_type(4)));
            __builtin_nontemporal_store(f4{v[c][0], v[c][1], v[c][2], v[c][3]}, reinterpret_cast<f4*>(dst));
        } else {
            for (int e = 0; e < PT; e++)
                if (i + e < nx) dst[e] = v[c][e];
        }
    }
}

hipError_t launch_macros_f32(const double* macro, const uint8_t* kind, int64_t nx, int64_t ny, int64_t nz,
                             int64_t nxp, int64_t nyp, int64_t ns, float* rho, float* u, hipStream_t s) {
    const int64_t nbox = nx * ny * nz;
    if (nbox <= 0) return hipSuccess;
    const bool vec = nx % 4 == 0 && (uintptr_t)rho % 16 == 0 && (uintptr_t)u % 16 == 0;
    // rows that are not whole aligned quads: one point per thread, so that the lanes' 4-byte stores lie side by side
    // (871 x 435 x 435: 0.85 ms; with four points a thread 100 steps and this took 10.17 ms, now 9.75); beyond
    // 32-bit indices four, to stay within a launch
    const bool one = !vec && nbox <= 0xffffff00ll;
    const int64_t nq = one ? nx : (nx + 3) / 4, quads = nq * ny * nz;
    // a thread each, and a launch has fewer than 2^32: boxes of more than 17e9 points, 550 GB of macro planes
    if (quads > 0xffffff00ll) return hipErrorInvalidValue;
    const dim3 g((unsigned)((quads + 255) / 256));
#define PV_MACROS(V, PT) \
    hipLaunchKernelGGL((k_macros_f32<V, PT>), g, dim3(256), 0, s, macro, kind, nx, (uint32_t)ny, nbox, (uint32_t)nq, (uint32_t)quads, nxp, nyp, ns, rho, u)
    if (vec) PV_MACROS(true, 4);
    else if (one) PV_MACROS(false, 1);
    else PV_MACROS(false, 4);
#undef PV_MACROS
    return hipGetLastError();
}

// One wave per tile.  Bound by the four loads of eight bytes a node; what counts is what is not moved: the planes
// are the padded box, most of it without nodes.
__global__ __launch_bounds__(256) void k_macros_nodes(const double* macro, int64_t ns, const TileDesc* tdesc, int32_t t0,
                                                      int32_t nt, double* out) {
    const int32_t t = (int32_t)blockIdx.x * 4 + (int32_t)(threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (t >= nt) return;
    const TileDesc& D = tdesc[t0 + t];
    if (!((D.node >> lane) & 1)) return;
    const int64_t n = (int64_t)D.tile * 64 + lane;
    const int64_t i = (D.first - tdesc[t0].first) + (uint32_t)__popcll(D.node & ((1ull << lane) - 1));
    dvec2* o = reinterpret_cast<dvec2*>(out + 4 * i);
    o[0] = dvec2{macro[n], macro[ns + n]};
    o[1] = dvec2{macro[2 * ns + n], macro[3 * ns + n]};
}

hipError_t launch_macros_nodes(const double* macro, int64_t ns, const TileDesc* tdesc, int32_t t0, int32_t nt,
                               double* out, hipStream_t s) {
    if (nt <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_macros_nodes, dim3((unsigned)((nt + 3) / 4)), dim3(256), 0, s, macro, ns, tdesc, t0, nt, out);
    return hipGetLastError();
}

// one thread per output point of a separable index grid
__global__ void k_sample_kinds(const uint8_t* kind, int64_t nxp, int64_t nyp, const int32_t* ix, int nx,
                               const int32_t* iy, int ny, const int32_t* iz, int nz, uint8_t* out) {
    const int64_t o = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (o >= (int64_t)nx * ny * nz) return;
    const int i = (int)(o % nx);
    const int64_t r = o / nx;
    const int j = (int)(r % ny), k = (int)(r / ny);
    out[o] = kind[ix[i] + nxp * (iy[j] + nyp * (int64_t)iz[k])];
}

hipError_t launch_sample_kinds(const uint8_t* kind, int64_t nxp, int64_t nyp, const int32_t* ix, int nx,
                               const int32_t* iy, int ny, const int32_t* iz, int nz, uint8_t* out, hipStream_t s) {
    const int64_t n = (int64_t)nx * ny * nz;
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_sample_kinds, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, kind, nxp, nyp, ix, nx,
                       iy, ny, iz, nz, out);
    return hipGetLastError();
}

hipError_t launch_copy(const void* src, void* dst, int64_t bytes, hipStream_t s) {
    const int64_t n = bytes / 16;
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_copy, dim3((unsigned)((n + 1023) / 1024)), dim3(256), 0, s, static_cast<const dvec2*>(src),
                       static_cast<dvec2*>(dst), n);
    return hipGetLastError();
}

}  // namespace pvlbm
