// Interpolation from a structured grid with arbitrary vertex positions to scattered points
// (ffdas_create_interpolation_plan / _preprocess / ffdas_interpolation / _destroy).
//
// Plan (once per grid): the vertices as 16-byte vectors, the grid's bounding box and the scale of
// the 128 bins per axis over it (one pass over the vertices, finished on the device).
// Query (once per point set): the points are ordered by bin, and every grid cell tests the points
// in the bins of its quantised bounding box; per point, the lowest tetrahedron id whose FP32
// barycentric test passes (computed without contraction in the reference's operation order) and
// whose own quantised box holds the point's bin, which is the first of the reference's sorted
// list of that bin.  The lookup of a point is that tetrahedron's key and three weights (linear)
// or one vertex id (nearest).
// Evaluation (per call, the per-frame part): x is first copied frame-inner (the frames of a
// chunk, up to 16 for 4-byte data and 8 otherwise, contiguous per vertex; one frame is read as it
// is where the output does not overlap it), so one thread per query point fetches each of its
// vertices' chunk with one vector load; its lookup is read once per chunk; out is packed.
#include <hip/hip_runtime.h>

#include <cstring>   // before rocPRIM, whose iterators use memset

#include <rocprim/rocprim.hpp>

#include <algorithm>
#include <cfloat>
#include <climits>
#include <cmath>
#include <cstdlib>
#include <mutex>
#include <string>
#include <vector>

#include "internal.h"

struct ffdas_interpolation_plan {
    int device = 0;
    int64_t nx = 0, ny = 0, nz = 0;
    int mode = FFDAS_INTERP_LINEAR;
    float4 *verts = nullptr;           // nx * ny * nz, one 16-byte vector per vertex
    unsigned char *flat = nullptr;     // behind them, by base vertex: the cell's flat tetrahedra (bits)
    bool any_flat = false;
    float bmin[3] = {0, 0, 0}, scale[3] = {0, 0, 0};
    int64_t ntet = 0;
    long long list_total = 0;          // entries of the bin lists
    // per-bin lists of tetrahedra, built when the point-by-point location first needs them
    std::mutex list_mutex;
    long long *bin_start = nullptr;    // kBins^3 + 1
    int *bin_list = nullptr;
    // preprocessed query points
    bool pre = false;
    int64_t pre_n = 0;
    int *pre_idx = nullptr;            // n vertex ids (nearest) or tetrahedron keys (linear)
    float *pre_w = nullptr;            // linear: 3 n weights
};

namespace ffdas {
namespace {

constexpr int kBins = 128;
constexpr int64_t kBins3 = (int64_t)kBins * kBins * kBins;

// the six tetrahedra of a cell as corner codes (bit 0: +x, bit 1: +y, bit 2: +z), in the
// reference's order (src/interpolation/spatial_hash_kernels.cuh:183-190): the split fixes
// which vertices a point is interpolated from
constexpr int kTet[6][4] = {{0, 1, 2, 4}, {1, 3, 2, 7}, {1, 2, 4, 7},
                            {2, 4, 6, 7}, {1, 4, 5, 7}, {4, 6, 5, 7}};

constexpr unsigned tet_codes(int t) {
    return kTet[t][0] | kTet[t][1] << 3 | kTet[t][2] << 6 | kTet[t][3] << 9;
}

// the corner codes of tetrahedron t, three bits each, without a table in memory
__device__ __forceinline__ unsigned corner_codes(int t) {
    constexpr uint64_t first = (uint64_t)tet_codes(0) | (uint64_t)tet_codes(1) << 12 |
                               (uint64_t)tet_codes(2) << 24 | (uint64_t)tet_codes(3) << 36 |
                               (uint64_t)tet_codes(4) << 48;
    return t == 5 ? tet_codes(5) : (unsigned)(first >> (12 * t)) & 0xfffu;
}

// Vertex id of corner `code` of the cell at base vertex `base`.
__device__ __forceinline__ int corner(int base, int code, int nx, int ny) {
    return base + (code & 1) + ((code >> 1) & 1) * nx + ((code >> 2) & 1) * ny * nx;
}

// A tetrahedron: key = base vertex * 8 + t, base = cx + cy nx + cz ny nx of its cell.  Keys
// order exactly as the ids cell * 6 + t do (cells in (cz, cy, cx) order, then t), so the lowest
// passing id is the lowest passing key, and the vertices follow from the key without divisions.
__device__ __forceinline__ int cell_base(unsigned cell, int nx, int ny) {
    const unsigned row = cell / (unsigned)(nx - 1), cx = cell - row * (unsigned)(nx - 1);
    const unsigned cz = row / (unsigned)(ny - 1), cy = row - cz * (unsigned)(ny - 1);
    return (int)(cx + (cy + cz * (unsigned)ny) * (unsigned)nx);
}

__device__ __forceinline__ int tet_key(long long tid, int nx, int ny) {
    const unsigned cell = (unsigned)(tid / 6);
    return cell_base(cell, nx, ny) * 8 + (int)(tid - (long long)cell * 6);
}

__device__ __forceinline__ int4 key_vertices(int key, int nx, int ny) {
    const int base = key >> 3;
    const unsigned c = corner_codes(key & 7);
    return int4{corner(base, c & 7, nx, ny), corner(base, (c >> 3) & 7, nx, ny),
                corner(base, (c >> 6) & 7, nx, ny), corner(base, c >> 9, nx, ny)};
}

struct Box {
    float mn[3], sc[3];
};

// round-to-nearest bin of (p - min) * scale with negatives saturated to 0 (NaN counts as
// outside); returns false past the last bin
__device__ __forceinline__ bool quantize(const Box &b, float x, float y, float z, int &ix, int &iy,
                                         int &iz) {
    const float q[3] = {(x - b.mn[0]) * b.sc[0], (y - b.mn[1]) * b.sc[1], (z - b.mn[2]) * b.sc[2]};
    int r[3];
#pragma unroll
    for (int a = 0; a < 3; a++) {
        if (!(q[a] <= (float)(kBins - 1) + 0.5f)) return false;   // beyond the range, or NaN
        const float v = rintf(q[a] > 0.0f ? q[a] : 0.0f);
        if (v > (float)(kBins - 1)) return false;
        r[a] = (int)v;
    }
    ix = r[0];
    iy = r[1];
    iz = r[2];
    return true;
}

// What the plan needs on the host: the box, the number of entries the bin lists would have and whether
// any tetrahedron is flat (flat_tets).
struct PlanHead {
    Box box;
    unsigned long long total;         // below 2^52; and kAnyFlat for each workgroup with flat cells
};
constexpr unsigned long long kAnyFlat = 1ull << 53;      // at most 1024 workgroups

// The vertices into 16-byte vectors, and the minima and maxima of each block's part.
__global__ __launch_bounds__(256) void interp_verts_kernel(const float *__restrict__ v, int64_t n,
                                                           float4 *__restrict__ v4,
                                                           float *__restrict__ part) {
    float mn[3] = {FLT_MAX, FLT_MAX, FLT_MAX}, mx[3] = {-FLT_MAX, -FLT_MAX, -FLT_MAX};
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        const float p[3] = {v[3 * i], v[3 * i + 1], v[3 * i + 2]};
        v4[i] = float4{p[0], p[1], p[2], 0.f};
#pragma unroll
        for (int a = 0; a < 3; a++) {
            mn[a] = fminf(mn[a], p[a]);
            mx[a] = fmaxf(mx[a], p[a]);
        }
    }
    __shared__ float red[6][4];
#pragma unroll
    for (int a = 0; a < 3; a++) {
        for (int o = 32; o > 0; o >>= 1) {
            mn[a] = fminf(mn[a], __shfl_xor(mn[a], o));
            mx[a] = fmaxf(mx[a], __shfl_xor(mx[a], o));
        }
    }
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0) {
#pragma unroll
        for (int a = 0; a < 3; a++) {
            red[a][w] = mn[a];
            red[3 + a][w] = mx[a];
        }
    }
    __syncthreads();
    if (threadIdx.x < 6) {
        const int a = threadIdx.x;
        float r = red[a][0];
        for (int k = 1; k < 4; k++) r = a < 3 ? fminf(r, red[a][k]) : fmaxf(r, red[a][k]);
        part[blockIdx.x * 6 + a] = r;
    }
}

// The box and the bins' scale, in FP32 as the reference (spatial_hash.cu:51-55), from the
// partial minima and maxima; one wave.
__global__ __launch_bounds__(64) void interp_box_kernel(const float *__restrict__ part, int blocks,
                                                        PlanHead *__restrict__ head) {
#pragma clang fp contract(off)
    for (int a = 0; a < 3; a++) {
        float mn = FLT_MAX, mx = -FLT_MAX;
        for (int k = threadIdx.x; k < blocks; k += 64) {
            mn = fminf(mn, part[k * 6 + a]);
            mx = fmaxf(mx, part[k * 6 + 3 + a]);
        }
        for (int o = 32; o > 0; o >>= 1) {
            mn = fminf(mn, __shfl_xor(mn, o));
            mx = fmaxf(mx, __shfl_xor(mx, o));
        }
        if (threadIdx.x == 0) {
            head->box.mn[a] = mn;
            head->box.sc[a] = (float)(kBins - 1) / (mx - mn);
        }
    }
    if (threadIdx.x == 0) head->total = 0;
}

__global__ void interp_zero_kernel(long long *p, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        p[i] = 0;
}

// A vertex lies inside the box: (p - min) * scale is in [0, 127] up to rounding.
__device__ __forceinline__ int vertex_bin(float x, float mn, float sc) {
    return (int)fminf(rintf(fmaxf((x - mn) * sc, 0.0f)), (float)(kBins - 1));
}

// quantised bounding box of tetrahedron tid, clamped to the bins
__device__ __forceinline__ void tet_bins(const Box &b, const float4 *__restrict__ v, int key,
                                         int nx, int ny, int lo[3], int hi[3]) {
    const int4 id = key_vertices(key, nx, ny);
    const int ids[4] = {id.x, id.y, id.z, id.w};
    lo[0] = lo[1] = lo[2] = kBins - 1;
    hi[0] = hi[1] = hi[2] = 0;
#pragma unroll
    for (int c = 0; c < 4; c++) {
        const float4 q = v[ids[c]];
        const float p[3] = {q.x, q.y, q.z};
#pragma unroll
        for (int a = 0; a < 3; a++) {
            const int k = vertex_bin(p[a], b.mn[a], b.sc[a]);
            lo[a] = min(lo[a], k);
            hi[a] = max(hi[a], k);
        }
    }
}

// The tetrahedra of a cell whose FP32 weights may be off by more than a few per cent: |volume| below 1e-4
// of the product of two of its edges and the reach of the bins' points (the cell's diagonal and a bin).
// The numerators and the volume are good to 16 eps = 9.5e-7 of such products, so that a point whose
// weights come out as 0 or more lies within 3 x 9.5e-7 / 1e-4 = 2.9 % of the box of any other tetrahedron.
// The volumes as barycentric() forms them: below 1e-12 no point passes.  The sixth tetrahedron, whose
// four corners are one face of the cell, is flat wherever that face is a plane out of the axes.
__device__ __forceinline__ unsigned flat_tets(const Box &b, const float (&v)[8][3]) {
#pragma clang fp contract(off)
    float reach2 = 0.0f;
#pragma unroll
    for (int a = 0; a < 3; a++) {
        float lo = v[0][a], hi = v[0][a];
#pragma unroll
        for (int k = 1; k < 8; k++) {
            lo = fminf(lo, v[k][a]);
            hi = fmaxf(hi, v[k][a]);
        }
        const float r = hi - lo + 1.0f / b.sc[a];
        reach2 += r * r;
    }
    unsigned flat = 0;
#pragma unroll
    for (int t = 0; t < 6; t++) {
        const float *v0 = v[kTet[t][0]], *v1 = v[kTet[t][1]], *v2 = v[kTet[t][2]], *v3 = v[kTet[t][3]];
        const float a0 = v1[0] - v0[0], a1 = v1[1] - v0[1], a2 = v1[2] - v0[2];
        const float b0 = v2[0] - v0[0], b1 = v2[1] - v0[1], b2 = v2[2] - v0[2];
        const float c0 = v3[0] - v0[0], c1 = v3[1] - v0[1], c2 = v3[2] - v0[2];
        const float bc0 = b1 * c2 - b2 * c1, bc1 = b2 * c0 - b0 * c2, bc2 = b0 * c1 - b1 * c0;
        const float denom = fabsf(a0 * bc0 + a1 * bc1 + a2 * bc2);
        const float na = a0 * a0 + a1 * a1 + a2 * a2, nb = b0 * b0 + b1 * b1 + b2 * b2,
                    nc = c0 * c0 + c1 * c1 + c2 * c2;
        const float pair = sqrtf(fmaxf(na, nb) * fmaxf(fminf(na, nb), nc));
        if (!(denom < 1e-12f) && denom < 1e-4f * pair * sqrtf(reach2)) flat |= 1u << t;
    }
    return flat;
}

// head->total += the bins of every tetrahedron's box; flat = the cells' flat tetrahedra
__global__ __launch_bounds__(256) void interp_total_kernel(const float4 *__restrict__ v,
                                                           int64_t ncell, int nx, int ny,
                                                           PlanHead *__restrict__ head,
                                                           unsigned char *__restrict__ flat) {
    const Box b = head->box;
    unsigned long long sum = 0;
    int any = 0;
    for (int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x; c < ncell; c += (int64_t)gridDim.x * 256) {
        const int base = cell_base((unsigned)c, nx, ny);
        int bin[8][3];
        float p[8][3];
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const float4 q = v[corner(base, k, nx, ny)];
            p[k][0] = q.x;
            p[k][1] = q.y;
            p[k][2] = q.z;
#pragma unroll
            for (int a = 0; a < 3; a++) bin[k][a] = vertex_bin(p[k][a], b.mn[a], b.sc[a]);
        }
#pragma unroll
        for (int t = 0; t < 6; t++) {
            unsigned long long n = 1;
#pragma unroll
            for (int a = 0; a < 3; a++) {
                const int b0 = bin[kTet[t][0]][a], b1 = bin[kTet[t][1]][a],
                          b2 = bin[kTet[t][2]][a], b3 = bin[kTet[t][3]][a];
                n *= (unsigned)(max(max(b0, b1), max(b2, b3)) - min(min(b0, b1), min(b2, b3)) + 1);
            }
            sum += n;
        }
        const unsigned f = flat_tets(b, p);
        flat[base] = (unsigned char)f;
        any |= (int)f;
    }
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
    any = __syncthreads_or(any);
    __shared__ unsigned long long red[4];
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = sum;
    __syncthreads();
    // one write a workgroup: they meet in one line (for the flag an atomic a wave took 50 us, a store 160)
    if (threadIdx.x == 0)
        atomicAdd(&head->total, red[0] + red[1] + red[2] + red[3] + (any ? kAnyFlat : 0));
}

// The per-bin lists of the point-by-point location: every tetrahedron counted into, then
// listed in, each bin of its box.
__global__ __launch_bounds__(256) void interp_count_kernel(Box b, const float4 *__restrict__ v,
                                                           int64_t ntet, int nx, int ny,
                                                           long long *__restrict__ cnt) {
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= ntet) return;
    int lo[3], hi[3];
    tet_bins(b, v, tet_key(t, nx, ny), nx, ny, lo, hi);
    for (int z = lo[2]; z <= hi[2]; z++)
        for (int y = lo[1]; y <= hi[1]; y++)
            for (int x = lo[0]; x <= hi[0]; x++)
                atomicAdd((unsigned long long *)cnt + (x + kBins * (y + kBins * z)), 1ull);
}

__global__ __launch_bounds__(256) void interp_fill_kernel(Box b, const float4 *__restrict__ v,
                                                          int64_t ntet, int nx, int ny,
                                                          const long long *__restrict__ start,
                                                          long long *__restrict__ cursor,
                                                          int *__restrict__ list) {
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= ntet) return;
    const int key = tet_key(t, nx, ny);
    int lo[3], hi[3];
    tet_bins(b, v, key, nx, ny, lo, hi);
    for (int z = lo[2]; z <= hi[2]; z++)
        for (int y = lo[1]; y <= hi[1]; y++)
            for (int x = lo[0]; x <= hi[0]; x++) {
                const int64_t bin = x + kBins * (y + kBins * z);
                const long long k = (long long)atomicAdd((unsigned long long *)cursor + bin, 1ull);
                list[start[bin] + k] = key;
            }
}

// Workgroups are dealt to the 8 XCDs round-robin by linear id.  This bijection hands each
// XCD groups of kXcdGroup consecutive (query block, chunk) tiles instead of single ones, so
// neighbouring query blocks, which share vertices, are served by one L2, while the XCDs
// still take turns over the whole grid (the located points are unevenly spread: whole
// contiguous eighths would leave some XCDs with most of the work).  Tiles past the last
// full round of 8 groups keep their own id.  Returns the tile as (x, y).
constexpr int kXcdGroup = 8;

__device__ __forceinline__ void xcd_tile(int &bx, int &by) {
    const int total = gridDim.x * gridDim.y;
    const int lin = blockIdx.y * gridDim.x + blockIdx.x;
    constexpr int R = 8 * kXcdGroup;
    int L = lin;
    if (lin < total / R * R) {
        const int base = lin / R * R, o = lin - base;   // o = j * 8 + xcd within the round
        L = base + (o % 8) * kXcdGroup + o / 8;
    }
    bx = L % gridDim.x;
    by = L / gridDim.x;
}

// FP32 barycentric coordinates of p in (v0, v1, v2, v3) and whether all are >= 0, in the
// reference's operation order (spatial_hash_kernels.cuh:62-90), with no FMA contraction
__device__ __forceinline__ bool barycentric(const float *p, const float *v0, const float *v1, const float *v2,
                            const float *v3, float w[4]) {
#pragma clang fp contract(off)
    const float a0 = v1[0] - v0[0], a1 = v1[1] - v0[1], a2 = v1[2] - v0[2];
    const float b0 = v2[0] - v0[0], b1 = v2[1] - v0[1], b2 = v2[2] - v0[2];
    const float c0 = v3[0] - v0[0], c1 = v3[1] - v0[1], c2 = v3[2] - v0[2];
    const float q0 = p[0] - v0[0], q1 = p[1] - v0[1], q2 = p[2] - v0[2];
    // cross(b, c), dot(a, .)
    const float bc0 = b1 * c2 - b2 * c1, bc1 = b2 * c0 - b0 * c2, bc2 = b0 * c1 - b1 * c0;
    const float denom = a0 * bc0 + a1 * bc1 + a2 * bc2;
    if (fabsf(denom) < 1e-12f) return false;
    const float qc0 = q1 * c2 - q2 * c1, qc1 = q2 * c0 - q0 * c2, qc2 = q0 * c1 - q1 * c0;
    const float bq0 = b1 * q2 - b2 * q1, bq1 = b2 * q0 - b0 * q2, bq2 = b0 * q1 - b1 * q0;
    const float n1 = q0 * bc0 + q1 * bc1 + q2 * bc2;
    const float n2 = a0 * qc0 + a1 * qc1 + a2 * qc2;
    const float n3 = a0 * bq0 + a1 * bq1 + a2 * bq2;
    // most candidates fail on a sign: a numerator of the other sign than denom with
    // |n| >= 1e-30 |denom| gives a quotient below -1e-30 (never a rounded -0), which the
    // test below rejects, so the divisions are skipped for it
    const float lim = 1e-30f * fabsf(denom);
    const bool neg = denom < 0.0f;
    if (((n1 < 0.0f) != neg && n1 != 0.0f && fabsf(n1) >= lim) ||
        ((n2 < 0.0f) != neg && n2 != 0.0f && fabsf(n2) >= lim) ||
        ((n3 < 0.0f) != neg && n3 != 0.0f && fabsf(n3) >= lim))
        return false;
    w[1] = n1 / denom;
    w[2] = n2 / denom;
    w[3] = n3 / denom;
    w[0] = 1.0f - w[1] - w[2] - w[3];
    return w[0] >= 0.0f && w[1] >= 0.0f && w[2] >= 0.0f && w[3] >= 0.0f;
}

// "no tetrahedron holds the point" in the lookup of point i
__device__ __forceinline__ void write_missing(int64_t i, int *idx) { idx[i] = -1; }

// The lookup of point i in tetrahedron `key` with weights w.  Nearest: the vertex of largest
// weight (the reference's tie order, float4_max_by_key, spatial_hash_kernels.cuh:51-59).
// Linear: the key and weights 1 to 3; weight 0 is 1 - w1 - w2 - w3, formed again in the same order.
__device__ __forceinline__ void write_found(int mode, int64_t i, int key, const float w[4], int nx,
                                            int ny, int *idx, float *wout) {
    if (mode == FFDAS_INTERP_NEAREST) {
        const int4 id = key_vertices(key, nx, ny);
        const int ixy = w[0] > w[1] ? id.x : id.y;
        const float mxy = ixy == id.x ? w[0] : w[1];
        const int izw = w[2] > w[3] ? id.z : id.w;
        const float mzw = izw == id.z ? w[2] : w[3];
        idx[i] = mxy > mzw ? ixy : izw;
    } else {
        idx[i] = key;
        wout[3 * i] = w[1];
        wout[3 * i + 1] = w[2];
        wout[3 * i + 2] = w[3];
    }
}

__device__ __forceinline__ bool test_key(const float p[3], int key, const float4 *__restrict__ v,
                                         int nx, int ny, float w[4]) {
    const int4 id = key_vertices(key, nx, ny);
    const float4 a = v[id.x], b = v[id.y], c = v[id.z], d = v[id.w];
    const float pa[3] = {a.x, a.y, a.z}, pb[3] = {b.x, b.y, b.z}, pc[3] = {c.x, c.y, c.z},
                pd[3] = {d.x, d.y, d.z};
    return barycentric(p, pa, pb, pc, pd, w);
}

// Point by point: every point tests the tetrahedra of its bin's list and keeps the lowest id.
__global__ __launch_bounds__(256) void interp_locate_kernel(
    Box b, const float4 *__restrict__ v, int nx, int ny, int64_t ntet,
    const long long *__restrict__ start, const int *__restrict__ list,
    const float *__restrict__ qp, int64_t n, int mode, int *__restrict__ idx,
    float *__restrict__ wout) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const float p[3] = {qp[3 * i], qp[3 * i + 1], qp[3 * i + 2]};
    int ix, iy, iz;
    int best = INT_MAX;
    float bw[4] = {0, 0, 0, 0};
    if (ntet > 0 && quantize(b, p[0], p[1], p[2], ix, iy, iz)) {
        const int64_t bin = ix + kBins * (iy + kBins * (int64_t)iz);
        for (long long e = start[bin]; e < start[bin + 1]; e++) {
            const int t = list[e];
            float w[4];
            if (t < best && test_key(p, t, v, nx, ny, w)) {
                best = t;
#pragma unroll
                for (int c = 0; c < 4; c++) bw[c] = w[c];
            }
        }
    }
    if (best != INT_MAX)
        write_found(mode, i, best, bw, nx, ny, idx, wout);
    else
        write_missing(i, idx);
}

// ---------------------------------------------------------------------------------------
// Location by cells.  The query points are counted, scanned and ordered by bin, so that the
// points of the bins (x0 .. x1, y, z) are one run, and every cell walks the runs of its quantised
// bounding box (the union of its tetrahedra's boxes: every tetrahedron the reference would list
// in a point's bin is met; what the lanes of a cell do not get through in a few dozen steps is left to a
// second kernel, a wave for each piece).  A point inside the cell's box, widened by 5 % of its extent plus
// 1e-5 of the coordinates' magnitude per axis, is tested against the six tetrahedra in order, any other
// point of the runs near them against the flat ones, whose FP32 weights may err by more than that (flat_tets); one
// that passes, and whose own quantised box holds the point's bin, lowers the point's best key by an
// atomic minimum.  The lookups are written by a last pass over the points.  No lists of
// tetrahedra are built: their atomics met at the apex of a sector, where thousands of small
// cells share a bin (512 x 96 x 96 sector: count 7.9 and fill 8.7 ms of a plan, and 7.7 ms to
// locate 256^3 points in them; now 0.3 ms and 3.6 ms).
// ---------------------------------------------------------------------------------------

__global__ void interp_zero_i32_kernel(int *p, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        p[i] = 0;
}

// cnt[bin] = the points of each bin; a point outside the bins has its lookup written here
__global__ __launch_bounds__(256) void interp_point_bin_kernel(Box b, const float *__restrict__ qp,
                                                               int64_t n, int *__restrict__ cnt,
                                                               int *__restrict__ idx) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    int ix, iy, iz;
    if (quantize(b, qp[3 * i], qp[3 * i + 1], qp[3 * i + 2], ix, iy, iz))
        atomicAdd(cnt + (ix + kBins * (iy + kBins * iz)), 1);
    else
        write_missing(i, idx);
}

// pts[start[bin] ..) = the points of each bin (position, id), counting cnt back down to 0;
// best = none
__global__ __launch_bounds__(256) void interp_point_order_kernel(
    Box b, const float *__restrict__ qp, int64_t n, const int *__restrict__ start,
    int *__restrict__ cnt, float4 *__restrict__ pts, int *__restrict__ best) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const float x = qp[3 * i], y = qp[3 * i + 1], z = qp[3 * i + 2];
    int ix, iy, iz;
    if (!quantize(b, x, y, z, ix, iy, iz)) return;
    const int bin = ix + kBins * (iy + kBins * iz);
    const int e = start[bin] + atomicSub(cnt + bin, 1) - 1;
    pts[e] = float4{x, y, z, __int_as_float((int)i)};
    best[e] = INT_MAX;
}

// Orders the LDS accesses of a wave's lanes among one another: what they wrote before is read after,
// and what they read before is overwritten after.  The hardware keeps them in order; this keeps the
// compiler from moving them.
__device__ __forceinline__ void wave_order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The bounding box of a cell's vertices, widened, and the bins it lies in.
struct CellBox {
    float lo[3], hi[3];
    int b0[3], b1[3];
    __device__ __forceinline__ int rows() const { return (b1[1] - b0[1] + 1) * (b1[2] - b0[2] + 1); }
    // the ordered points of the bins (b0 .. b1, y, z) of row r
    __device__ __forceinline__ int2 run(int r, const int *__restrict__ pstart) const {
        const int ny = b1[1] - b0[1] + 1, dz = r / ny;
        const int row = kBins * (b0[1] + r - dz * ny + kBins * (b0[2] + dz));
        return int2{pstart[row + b0[0]], pstart[row + b1[0] + 1]};
    }
    __device__ __forceinline__ bool holds(const float4 &u) const {
        return u.x >= lo[0] && u.x <= hi[0] && u.y >= lo[1] && u.y <= hi[1] && u.z >= lo[2] && u.z <= hi[2];
    }
};

__device__ __forceinline__ CellBox cell_box(const Box &b, const float4 *__restrict__ v, int base, int nx,
                                            int ny) {
    CellBox c;
#pragma unroll
    for (int a = 0; a < 3; a++) {
        c.lo[a] = 3.4e38f;
        c.hi[a] = -3.4e38f;
        c.b0[a] = kBins - 1;
        c.b1[a] = 0;
    }
#pragma unroll
    for (int k = 0; k < 8; k++) {
        const float4 u = v[corner(base, k, nx, ny)];
        const float p[3] = {u.x, u.y, u.z};
#pragma unroll
        for (int a = 0; a < 3; a++) {
            c.lo[a] = fminf(c.lo[a], p[a]);
            c.hi[a] = fmaxf(c.hi[a], p[a]);
            const int q1 = vertex_bin(p[a], b.mn[a], b.sc[a]);
            c.b0[a] = min(c.b0[a], q1);
            c.b1[a] = max(c.b1[a], q1);
        }
    }
#pragma unroll
    for (int a = 0; a < 3; a++) {
        const float m = 0.05f * (c.hi[a] - c.lo[a]) + 1e-5f * (fabsf(c.lo[a]) + fabsf(c.hi[a])) + 1e-30f;
        c.lo[a] -= m;
        c.hi[a] += m;
    }
    return c;
}

// Where a point outside a cell's box may pass the test of a flat tetrahedron.  Usually the sixth alone
// is flat: its weight n / denom of corner 5 is at most 1, so that |q . (b x c)|, the distance from the
// plane of corners 4, 5 and 7 times an area below `pair`, is at most |denom| < 1e-4 pair reach and the
// rounding of n, 9.5e-7 pair reach (flat_tets).  That leaves few points (one call for a 256 x 64 x 64 sector
// and 128^3 points: 758 us with all of them tested, 548 so, 529 with none).  Points below the box of
// the grid, whose bin is 0 however far they are, are tested always.
struct FlatPlane {
    float n[3] = {0, 0, 0}, d = 0, tol = -1.0f;      // tol < 0: no flat tetrahedron
    __device__ __forceinline__ bool holds(const Box &b, const float4 &u) const {
        if (tol < 0.0f) return false;
        const float r = fabsf(n[0] * u.x + n[1] * u.y + n[2] * u.z - d);
        return !(r > tol) || u.x < b.mn[0] || u.y < b.mn[1] || u.z < b.mn[2];
    }
};

__device__ __forceinline__ FlatPlane flat_plane(const Box &b, const float4 *__restrict__ v, unsigned flat,
                                                const CellBox &c, int base, int nx, int ny) {
    FlatPlane f;
    if (flat == 0) return f;
    f.tol = INFINITY;
    if (flat != 0x20) return f;
    const float4 v4 = v[corner(base, 4, nx, ny)], v5 = v[corner(base, 5, nx, ny)],
                 v6 = v[corner(base, 6, nx, ny)], v7 = v[corner(base, 7, nx, ny)];
    const float ax = v6.x - v4.x, ay = v6.y - v4.y, az = v6.z - v4.z;
    const float bx = v5.x - v4.x, by = v5.y - v4.y, bz = v5.z - v4.z;
    const float cx = v7.x - v4.x, cy = v7.y - v4.y, cz = v7.z - v4.z;
    const float pair = fmaxf(fmaxf(ax * ax + ay * ay + az * az, bx * bx + by * by + bz * bz),
                             cx * cx + cy * cy + cz * cz);      // above any product of two edges
    const float s = 1.0f / pair;
    f.n[0] = (by * cz - bz * cy) * s;
    f.n[1] = (bz * cx - bx * cz) * s;
    f.n[2] = (bx * cy - by * cx) * s;
    f.d = f.n[0] * v4.x + f.n[1] * v4.y + f.n[2] * v4.z;
    float reach = 0.0f, size = 0.0f;
#pragma unroll
    for (int a = 0; a < 3; a++) {
        const float bin = 1.0f / b.sc[a];
        reach += c.hi[a] - c.lo[a] + bin;
        size += fabsf(c.lo[a]) + fabsf(c.hi[a]) + bin;
    }
    f.tol = 1.1e-4f * reach + 1e-6f * size;      // and the rounding of this sum itself
    return f;
}

// The points inside a cell's box are few and come to the lanes at different times, so they are put
// on a queue of the wave, and the tests, most of the work, run with a queued point in every lane
// (one lane testing its own point on the spot: 0.54 ms for the cells of a 256 x 64 x 64 sector and
// 128^3 points, 0.26 ms queued).  FLAT: the points of the bins outside the box are tested against the
// cell's flat tetrahedra.
constexpr int kFlatOnly = 1 << 30;       // base vertices are below 2^28
template <bool FLAT> struct PointQueue {
    Box b;
    const float4 *__restrict__ v;
    const unsigned char *__restrict__ flat;
    int nx, ny;
    const float4 *__restrict__ pts;
    int *__restrict__ best;
    int2 *q;                 // 128 of (base vertex, point)
    int waiting;             // queued points, uniform

    // a queued point against the six tetrahedra of its cell, or the flat ones
    __device__ __forceinline__ void test(int2 c) const {
        const float4 u = pts[c.y];
        const float p[3] = {u.x, u.y, u.z};
        unsigned which = 0x3f;
        if (FLAT && (c.x & kFlatOnly)) {
            c.x &= ~kFlatOnly;
            which = flat[c.x];
        }
        // an outdated best only costs a test: the minimum is taken atomically
        const int known = best[c.y];
#pragma unroll 1
        for (int key = c.x * 8; key < min(c.x * 8 + 6, known); key++) {
            if (FLAT && !(which >> (key & 7) & 1)) continue;
            float w[4];
            if (!test_key(p, key, v, nx, ny, w)) continue;
            int tl[3], th[3], ib[3];
            tet_bins(b, v, key, nx, ny, tl, th);
            (void)quantize(b, p[0], p[1], p[2], ib[0], ib[1], ib[2]);
            if (ib[0] < tl[0] || ib[0] > th[0] || ib[1] < tl[1] || ib[1] > th[1] ||
                ib[2] < tl[2] || ib[2] > th[2])
                continue;
            atomicMin(best + c.y, key);
            break;
        }
    }
    // the lanes with a hit queue theirs (all lanes call); base: with kFlatOnly, for the flat ones
    __device__ __forceinline__ void offer(bool hit, int base, int at) {
        const uint64_t hits = __ballot(hit);
        if (!hits) return;
        if (hit)
            q[waiting + __builtin_amdgcn_mbcnt_hi((unsigned)(hits >> 32),
                                                  __builtin_amdgcn_mbcnt_lo((unsigned)hits, 0))] =
                int2{base, at};
        waiting += __popcll(hits);
        wave_order();
        if (waiting >= 64) {
            waiting -= 64;
            const int2 c = q[waiting + (threadIdx.x & 63)];
            wave_order();
            test(c);
        }
    }
    __device__ __forceinline__ void finish() {
        if ((int)(threadIdx.x & 63) < waiting) test(q[threadIdx.x & 63]);
    }
};

// Work that the lanes of a cell leave to whole waves: runs of points and ranges of rows.  Points in
// a small part of the grid (a zoomed raster) and cells far larger than the rest would otherwise be
// walked by the few lanes that an average cell has.  An entry is (base vertex, first, end, step): rows
// first, first + step, .. before end, at most 64; or, with step 0, the ordered points first .. end.
// The entries are in kLists lists, a cache line for each one's count: 16384 waves that add to one count
// from all XCDs take a millisecond.
constexpr int kLists = 16, kCountStep = 16;        // kCountStep * 8 bytes apart
struct Leftover {
    unsigned long long *count;      // of list l at l * kCountStep
    int4 *work;                     // from l * cap
    int cap, slice;                 // entries of a list, points of one entry
    // room for n entries in this workgroup's list, or none (what was reserved then is empty entries)
    __device__ __forceinline__ int4 *reserve(int n) const {
        const int list = blockIdx.x % kLists;
        unsigned long long *c = count + list * kCountStep;
        int4 *w = work + (int64_t)list * cap;
        if (*(volatile unsigned long long *)c >= (unsigned long long)cap) return nullptr;
        const unsigned long long at = atomicAdd(c, (unsigned long long)n);
        if (at + n <= (unsigned long long)cap) return w + at;
        for (unsigned long long k = at; k < (unsigned long long)cap; k++) w[k] = int4{0, 0, 0, 0};
        return nullptr;
    }
};
// Points and rows a lane walks before it leaves the rest.  256 x 64 x 64 sector, 180^3 points, the two
// kernels: 16 steps 863 us, 24 716, 32 663, 48 608, 96 636; 128^3 points in a quarter of the box along each
// axis 949, 941, 934, 935 (754 us walked by the lanes to the end), in the 64 x 16 x 20 vertices of a box
// 281, 327, 366, 450 and 733 (1708 walked to the end).
constexpr int kLaneSteps = 48;

// The lanes of a wave leave what they have left of their runs (e .. pe) and rows (r .. rows).  Of the
// 2^lgp lanes that share a run and the rows after it the first is nowhere ahead of the others: it
// lists its own rest for all of them.  False where there is no room: they go on.
__device__ __forceinline__ bool leave(const Leftover &rest, int base, int rows, int lgr, int lgp, int e, int pe,
                                      int r) {
    const int lane = threadIdx.x & 63;
    const bool lists = (lane & ((1 << lgp) - 1)) == 0;
    const int slices = lists && e < pe ? (pe - e - 1) / rest.slice + 1 : 0;
    const int ranges = lists && r < rows ? ((rows - 1 - r) >> (lgr + 6)) + 1 : 0;
    int upto = slices + ranges;                  // entries of this lane and those before
    for (int o = 1; o < 64; o <<= 1) {
        const int below = __shfl_up(upto, o);
        if (lane >= o) upto += below;
    }
    const int n = __shfl(upto, 63);
    unsigned long long to = 0;
    if (lane == 0) to = (unsigned long long)rest.reserve(n);
    to = __shfl(to, 0);
    if (to == 0) return false;
    int4 *w = (int4 *)to + (upto - slices - ranges);
    for (int k = 0; k < slices; k++)
        w[k] = int4{base, e + k * rest.slice, e + min(pe - e, (k + 1) * rest.slice), 0};
    for (int k = 0; k < ranges; k++)
        w[slices + k] = int4{base, r + (k << (lgr + 6)), min(rows, r + ((k + 1) << (lgr + 6))), 1 << lgr};
    return true;
}

// 2^(lgr + lgp) lanes per cell: 2^lgr share out the rows of its box, 2^lgp the points of a run.
template <bool FLAT>
__global__ __launch_bounds__(256, FLAT ? 6 : 7) void interp_locate_cells_kernel(
    Box b, const float4 *__restrict__ v, const unsigned char *__restrict__ flat, int64_t ncell, int nx,
    int ny, int lgr, int lgp, const int *__restrict__ pstart, const float4 *__restrict__ pts,
    int *__restrict__ best, Leftover rest) {
    __shared__ int2 queue[4][128];
    PointQueue<FLAT> q{b, v, flat, nx, ny, pts, best, queue[threadIdx.x >> 6], 0};
    const int64_t gid = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t cell = gid >> (lgr + lgp);
    const int psub = (int)gid & ((1 << lgp) - 1), rsub = (int)(gid >> lgp) & ((1 << lgr) - 1);
    const int base = cell < ncell ? cell_base((unsigned)cell, nx, ny) : 0;
    CellBox box{};
    int rows = 0;
    FlatPlane plane;
    if (cell < ncell) {
        box = cell_box(b, v, base, nx, ny);
        rows = box.rows();
        if (FLAT) plane = flat_plane(b, v, flat[base], box, base, nx, ny);
    }
    int r = rsub, e = 0, pe = 0;
    for (bool left = false;;) {
        bool live = true;
        for (int k = left ? INT_MAX : kLaneSteps; k > 0 && live; k--) {
            // a step takes a point of the run, or goes to the next run
            bool hit = false, in = true;
            int at = 0;
            if (e < pe) {
                const float4 u = pts[e];                 // one load
                in = box.holds(u);
                hit = in || (FLAT && plane.holds(b, u));
                at = e;
                e += 1 << lgp;
            } else if (r < rows) {
                const int2 run = box.run(r, pstart);
                e = run.x + psub;
                pe = run.y;
                r += 1 << lgr;
            }
            q.offer(hit, FLAT && !in ? base | kFlatOnly : base, at);
            live = __ballot(e < pe || r < rows) != 0;
        }
        if (!live || leave(rest, base, rows, lgr, lgp, e, pe, r)) break;
        left = true;
    }
    q.finish();
}

// The leftover work, an entry a wave at a time.  All lanes take points: of a range of rows, the rows'
// points one after the other.
template <bool FLAT>
__global__ __launch_bounds__(256) void interp_locate_rest_kernel(
    Box b, const float4 *__restrict__ v, const unsigned char *__restrict__ flat, int nx, int ny,
    const int *__restrict__ pstart, const float4 *__restrict__ pts, int *__restrict__ best, Leftover rest) {
    __shared__ int2 queue[4][128];
    PointQueue<FLAT> q{b, v, flat, nx, ny, pts, best, queue[threadIdx.x >> 6], 0};
    const int lane = threadIdx.x & 63;
    const int wave = blockIdx.x * 4 + (threadIdx.x >> 6), list = wave % kLists;
    const unsigned long long listed = rest.count[list * kCountStep];
    const int count = listed < (unsigned long long)rest.cap ? (int)listed : rest.cap;
    for (int i = wave / kLists; i < count; i += gridDim.x * 4 / kLists) {
        const int4 w = rest.work[(int64_t)list * rest.cap + i];
        const int base = __builtin_amdgcn_readfirstlane(w.x), first = __builtin_amdgcn_readfirstlane(w.y),
                  end = __builtin_amdgcn_readfirstlane(w.z), step = __builtin_amdgcn_readfirstlane(w.w);
        if (first >= end) continue;
        const CellBox box = cell_box(b, v, base, nx, ny);
        FlatPlane plane;
        if (FLAT) plane = flat_plane(b, v, flat[base], box, base, nx, ny);
        const auto offer = [&](bool any, int at) {
            const float4 u = pts[any ? at : 0];
            const bool in = box.holds(u);
            q.offer(any && (in || (FLAT && plane.holds(b, u))), FLAT && !in ? base | kFlatOnly : base, at);
        };
        if (step == 0) {
            for (int e0 = first; e0 < end; e0 += 64) offer(e0 + lane < end, e0 + lane);
            continue;
        }
        const int r = first + lane * step;
        const int2 run = r < end ? box.run(r, pstart) : int2{0, 0};
        int upto = run.y - run.x;                     // points of this lane's row and those before
        for (int o = 1; o < 64; o <<= 1) {
            const int below = __shfl_up(upto, o);
            if (lane >= o) upto += below;
        }
        const int total = __shfl(upto, 63), shift = run.y - upto;
        for (int k0 = 0; k0 < total; k0 += 64) {
            const int k = k0 + lane;
            int row = 0;                              // rows that end at or before point k
#pragma unroll
            for (int o = 32; o > 0; o >>= 1)
                if (__shfl(upto, row + o - 1) <= k) row += o;
            offer(k < total, k + __shfl(shift, row & 63));
        }
    }
    q.finish();
}

// The lookups of the ordered points.
__global__ __launch_bounds__(256) void interp_found_kernel(
    const float4 *__restrict__ v, int nx, int ny, const int *__restrict__ count,
    const float4 *__restrict__ pts, const int *__restrict__ best, int mode, int *__restrict__ idx,
    float *__restrict__ wout) {
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= *count) return;
    const float4 q = pts[e];
    const int key = best[e];
    const int64_t i = __float_as_int(q.w);
    if (key == INT_MAX) {
        write_missing(i, idx);
        return;
    }
    const float p[3] = {q.x, q.y, q.z};
    float w[4];
    (void)test_key(p, key, v, nx, ny, w);
    write_found(mode, i, key, w, nx, ny, idx, wout);
}

// element types: real or complex (two components), FP32 or FP64
template <typename R, int CW>
struct El {
    R c[CW];
};

// Outputs are written once and never read back by the kernel: streamed past the caches (NT) so
// they do not evict the vertex blocks that neighbouring query points gather.
template <bool NT, typename R, int CW>
__device__ __forceinline__ void put_out(El<R, CW> *p, const El<R, CW> &v) {
    if constexpr (NT) {
#pragma unroll
        for (int c = 0; c < CW; c++) __builtin_nontemporal_store(v.c[c], &p->c[c]);
    } else {
        *p = v;
    }
}

constexpr int kFramesPerThread = 8;   // frames per chunk of 8-byte elements, for the extent check

// the frames of one vertex in one chunk, contiguous: one vector load per vertex.  A chunk of one
// frame is x as it is (element-aligned).
template <typename R, int CW, int FPC>
struct alignas(FPC == 1 ? sizeof(R) : (sizeof(R) * CW * FPC < 16 ? sizeof(R) * CW * FPC : 16)) Frames {
    El<R, CW> f[FPC];
};

// x [frame][vertex] -> xfi [chunk][vertex][frame in chunk], zero past the last frame; each
// thread reads its vertex from the chunk's frames (coalesced per frame) and writes the
// vertex's frames as one contiguous block (coalesced across threads)
template <typename R, int CW, int FPC>
__global__ __launch_bounds__(256) void interp_frames_kernel(const El<R, CW> *__restrict__ x,
                                                            Frames<R, CW, FPC> *__restrict__ xfi,
                                                            int64_t npts, int64_t B) {
    const int64_t v = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (v >= npts) return;
    const int64_t b0 = (int64_t)blockIdx.y * FPC;
    Frames<R, CW, FPC> o;
#pragma unroll
    for (int f = 0; f < FPC; f++) {
        if (b0 + f < B) {
            o.f[f] = x[(b0 + f) * npts + v];
        } else {
#pragma unroll
            for (int c = 0; c < CW; c++) o.f[f].c[c] = R(0);
        }
    }
    xfi[blockIdx.y * npts + v] = o;
}

template <typename R, int CW, int FPC>
__global__ __launch_bounds__(256) void interp_nearest_kernel(
    const Frames<R, CW, FPC> *__restrict__ xfi, El<R, CW> *__restrict__ out,
    const int *__restrict__ idx, int64_t n, int64_t npts, int64_t B, El<R, CW> fill) {
    int bx, by;
    xcd_tile(bx, by);
    const int64_t i = (int64_t)bx * 256 + threadIdx.x;
    if (i >= n) return;
    const int k = idx[i];
    const int64_t b0 = (int64_t)by * FPC;
    const int nf = (int)(B - b0 < FPC ? B - b0 : FPC);
    if (k >= 0) {
        const Frames<R, CW, FPC> v = xfi[by * npts + k];
#pragma unroll
        for (int f = 0; f < FPC; f++)
            if (f < nf) put_out<true>(out + (b0 + f) * n + i, v.f[f]);
    } else {
#pragma unroll
        for (int f = 0; f < FPC; f++)
            if (f < nf) put_out<true>(out + (b0 + f) * n + i, fill);
    }
}

// Every output is written once, the frame-inner copy is read about once, and per point a key, and
// three weights where it is located: bound by HBM and by the vector L1, whose accesses are the
// vertex blocks.  Two lanes share a point of a 32-byte block or more, each taking half of its
// vertices' blocks, so that a load instruction touches half as many blocks; a wave covers 64
// consecutive points in two turns, all their loads in flight together.  The stores of an
// instruction are then runs of 32 points (128 bytes of 4-byte elements): streamed where those
// are whole cache lines (NT), through L2, which joins them, where they are not.  16 frames of a
// 512 x 96 x 96 sector to 256^3 points: 0.558 ms with a lane per point and ids and weights of 32
// bytes a point, 0.517 ms with keys and three weights, 0.46 ms with two lanes (four: 0.62, their
// runs are half lines).  To 255^3 points, off the lines, the call takes 0.66 ms through L2 and
// 1.02 ms streamed.
template <typename R, int CW, int FPC, bool NT>
__global__ __launch_bounds__(256) void interp_linear_kernel(
    const Frames<R, CW, FPC> *__restrict__ xfi, El<R, CW> *__restrict__ out,
    const int *__restrict__ idx, const float *__restrict__ wt, int nx, int ny, int64_t n,
    int64_t npts, int64_t B, El<R, CW> fill) {
#pragma clang fp contract(off)
    constexpr int BB = FPC * (int)sizeof(El<R, CW>);          // bytes of a vertex's block
    constexpr int LPP = BB >= 32 ? 2 : 1;
    constexpr int EPL = FPC / LPP;                            // frames of a lane
    using Part = Frames<R, CW, EPL>;
    int bx, by;
    xcd_tile(bx, by);
    const int lane = threadIdx.x & 63, sub = lane % LPP;
    const int64_t i0 = (int64_t)bx * 256 + (threadIdx.x & ~63) + lane / LPP;
    const int64_t b0 = (int64_t)by * FPC + sub * EPL;
    const int nf = (int)(B - b0 < EPL ? B - b0 : EPL);
    const Part *xc = reinterpret_cast<const Part *>(xfi + by * npts) + sub;
    // the lookup is read once per frame chunk: streamed, like the outputs
    int key[LPP];
    bool any = false;
#pragma unroll
    for (int r = 0; r < LPP; r++) {
        const int64_t i = i0 + r * (64 / LPP);
        key[r] = i < n ? __builtin_nontemporal_load(idx + i) : -1;
        any = any || key[r] >= 0;
    }
    if (__ballot(any) == 0) {
#pragma unroll
        for (int r = 0; r < LPP; r++) {
            const int64_t i = i0 + r * (64 / LPP);
#pragma unroll
            for (int f = 0; f < EPL; f++)
                if (i < n && f < nf) put_out<NT>(out + (b0 + f) * n + i, fill);
        }
        return;
    }
    float w[LPP][3];
    Part v[LPP][4];
#pragma unroll
    for (int r = 0; r < LPP; r++) {
        // points outside read vertex 0 and weights that are not used: the loads stay
        // unconditional
        const bool in = key[r] >= 0;
        typedef float F3 __attribute__((ext_vector_type(3), aligned(4)));
        const F3 q = __builtin_nontemporal_load(
            reinterpret_cast<const F3 *>(wt + (in ? 3 * (i0 + r * (64 / LPP)) : 0)));
        w[r][0] = q.x;
        w[r][1] = q.y;
        w[r][2] = q.z;
        const int4 k = in ? key_vertices(key[r], nx, ny) : int4{0, 0, 0, 0};
        v[r][0] = xc[(int64_t)k.x * LPP];
        v[r][1] = xc[(int64_t)k.y * LPP];
        v[r][2] = xc[(int64_t)k.z * LPP];
        v[r][3] = xc[(int64_t)k.w * LPP];
    }
#pragma unroll
    for (int r = 0; r < LPP; r++) {
        const int64_t i = i0 + r * (64 / LPP);
        const float w0 = 1.0f - w[r][0] - w[r][1] - w[r][2];
        // w0 v0 + w1 v1 + w2 v2 + w3 v3, left to right (interpolation_kernels.cuh:110-115)
#pragma unroll
        for (int f = 0; f < EPL; f++) {
            El<R, CW> o;
#pragma unroll
            for (int c = 0; c < CW; c++)
                o.c[c] = key[r] >= 0 ? (R)w0 * v[r][0].f[f].c[c] + (R)w[r][0] * v[r][1].f[f].c[c] +
                                           (R)w[r][1] * v[r][2].f[f].c[c] +
                                           (R)w[r][2] * v[r][3].f[f].c[c]
                                     : fill.c[c];
            if (i < n && f < nf) put_out<NT>(out + (b0 + f) * n + i, o);
        }
    }
}

void free_plan_device(ffdas_interpolation_plan *p) {
    for (void *q : {(void *)p->verts, (void *)p->bin_start, (void *)p->bin_list,
                    (void *)p->pre_idx, (void *)p->pre_w})
        if (q) (void)hipFree(q);
    p->verts = nullptr;
    p->flat = nullptr;
    p->bin_start = nullptr;
    p->bin_list = nullptr;
    p->pre_idx = nullptr;
    p->pre_w = nullptr;
}

Box box_of(const ffdas_interpolation_plan &p) {
    Box b;
    for (int a = 0; a < 3; a++) {
        b.mn[a] = p.bmin[a];
        b.sc[a] = p.scale[a];
    }
    return b;
}

int grid1(int64_t n) { return (int)std::max<int64_t>(1, (n + 255) / 256); }

size_t up256(size_t b) { return (b + 255) & ~(size_t)255; }

// The per-bin lists of the point-by-point location, once per plan.
ffdas_error_t build_lists(ffdas_context &h, ffdas_interpolation_plan &p) {
    std::lock_guard<std::mutex> lock(p.list_mutex);
    if (p.bin_list) return FFDAS_SUCCESS;
    hipStream_t st = h.stream;
    const size_t nb = (size_t)kBins3 + 1;
    long long *start = nullptr, *cnt = nullptr;
    int *list = nullptr;
    void *tmp = nullptr;
    size_t tmp_bytes = 0;
    hipError_t e = rocprim::exclusive_scan(nullptr, tmp_bytes, cnt, start, 0ll, nb,
                                           rocprim::plus<long long>(), st);
    if (e == hipSuccess) e = hipMalloc((void **)&start, nb * sizeof(long long));
    if (e == hipSuccess) e = hipMalloc((void **)&cnt, nb * sizeof(long long));
    if (e == hipSuccess) e = hipMalloc(&tmp, std::max<size_t>(tmp_bytes, 1));
    if (e == hipSuccess)
        e = hipMalloc((void **)&list, (size_t)std::max<long long>(p.list_total, 1) * sizeof(int));
    if (e == hipSuccess) {
        const Box b = box_of(p);
        const int zg = (int)std::min<int64_t>(4096, (kBins3 + 1 + 255) / 256);
        hipLaunchKernelGGL(interp_zero_kernel, dim3(zg), dim3(256), 0, st, cnt, kBins3 + 1);
        if (p.ntet > 0)
            hipLaunchKernelGGL(interp_count_kernel, dim3(grid1(p.ntet)), dim3(256), 0, st, b,
                               p.verts, p.ntet, (int)p.nx, (int)p.ny, cnt);
        // the sentinel count is 0, so start[kBins3] = total
        e = rocprim::exclusive_scan(tmp, tmp_bytes, cnt, start, 0ll, nb,
                                    rocprim::plus<long long>(), st);
        hipLaunchKernelGGL(interp_zero_kernel, dim3(zg), dim3(256), 0, st, cnt, kBins3 + 1);
        if (e == hipSuccess && p.ntet > 0)
            hipLaunchKernelGGL(interp_fill_kernel, dim3(grid1(p.ntet)), dim3(256), 0, st, b,
                               p.verts, p.ntet, (int)p.nx, (int)p.ny, start, cnt, list);
        if (e == hipSuccess) e = hipGetLastError();
        const hipError_t es = hipStreamSynchronize(st);   // cnt and tmp are freed next
        if (e == hipSuccess) e = es;
    }
    if (cnt) (void)hipFree(cnt);
    if (tmp) (void)hipFree(tmp);
    if (e != hipSuccess) {
        if (start) (void)hipFree(start);
        if (list) (void)hipFree(list);
        return e == hipErrorOutOfMemory ? FFDAS_ERROR_ALLOCATION_FAILED : hip_status(e);
    }
    p.bin_start = start;
    p.bin_list = list;
    return FFDAS_SUCCESS;
}

// By cells unless the point ids, and the steps past the last, do not fit an int or
// FFDAS_INTERP_LOCATE is "point".
bool locate_by_cells(int64_t n) {
    const char *how = std::getenv("FFDAS_INTERP_LOCATE");
    return n < INT_MAX - (1 << 20) && !(how && std::string(how) == "point");
}

// Scratch of a location by cells, carved from one block.
struct LocateScratch {
    // the bins' counts, a last 0, and from the next multiple of 128 bytes the lists' counts
    static constexpr int64_t list_counts() { return (kBins3 + 1 + 31) / 32 * 32; }
    static constexpr int64_t counts() { return list_counts() + 2 * kLists * kCountStep; }
    size_t pts = 0, best = 0, cnt = 0, start = 0, scan = 0, scan_bytes = 0, work = 0, total = 0;
    int cap = 0;       // entries of a list of leftover work
    static ffdas_error_t plan(int64_t n, hipStream_t st, LocateScratch &s) {
        const size_t nb = (size_t)kBins3 + 1;
        int *none = nullptr;
        if (rocprim::exclusive_scan(nullptr, s.scan_bytes, none, none, 0, nb, rocprim::plus<int>(),
                                    st) != hipSuccess)
            return FFDAS_ERROR_CUDA_LAUNCH_FAILED;
        s.pts = 0;
        s.best = s.pts + up256((size_t)n * sizeof(float4));
        s.cnt = s.best + up256((size_t)n * sizeof(int));
        s.start = s.cnt + up256(counts() * sizeof(int));
        s.scan = s.start + up256(nb * sizeof(int));
        s.work = s.scan + up256(s.scan_bytes);
        // at most 4096 slices of a run and 256 ranges of a cell's rows fit a list
        s.cap = (int)std::min<int64_t>(std::max<int64_t>(n / 8, 1 << 18), 1 << 21) / kLists;
        s.total = s.work + up256((size_t)s.cap * kLists * sizeof(int4));
        return FFDAS_SUCCESS;
    }
};

// Scratch of one call on the handle's stream: the handle's workspace, which keeps what it grew to, up to
// kKeptScratch (6.7 M points in one call), and beyond that a block of its own that goes back with the
// call: 16.8 M points take 640 MB, which would stay with the handle; allocating and freeing them is 0.4
// of 3.1 ms.  (With 64 MiB kept, 2.1 M points in one call took 0.86 ms instead of 0.51.)
constexpr size_t kKeptScratch = (size_t)256 << 20;
struct CallScratch {
    ffdas_context &h;
    void *own = nullptr;
    explicit CallScratch(ffdas_context &ctx) : h(ctx) {}
    CallScratch(const CallScratch &) = delete;
    ~CallScratch() {
        if (own) (void)hipFreeAsync(own, h.stream);
    }
    ffdas_error_t get(size_t bytes, void **p) {
        hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
        const bool capturing = hipStreamIsCapturing(h.stream, &cs) == hipSuccess &&
                               cs != hipStreamCaptureStatusNone;
        if (bytes <= kKeptScratch || bytes <= h.ws_bytes || capturing) {
            h.xcopy.valid = false;   // the converted-x record of the delay-and-sum calls
            return h.workspace(bytes, p);
        }
        const hipError_t e = hipMallocAsync(&own, bytes, h.stream);
        if (e != hipSuccess) {
            own = nullptr;
            return e == hipErrorOutOfMemory ? FFDAS_ERROR_DEVICE_MEMORY_INSUFFICIENT
                                            : FFDAS_ERROR_ALLOCATION_FAILED;
        }
        *p = own;
        return FFDAS_SUCCESS;
    }
};

// Locate n points into idx (and w): device buffers sized by the caller; `scratch` has the bytes
// of LocateScratch for a location by cells.
ffdas_error_t locate(ffdas_context &h, ffdas_interpolation_plan &p, const float *qp, int64_t n,
                     int *idx, float *w, const LocateScratch &ls, void *scratch) {
    hipStream_t st = h.stream;
    const int nx = (int)p.nx, ny = (int)p.ny;
    if (!scratch) {
        FFDAS_TRY(build_lists(h, p));
        ProfScope ps(st, "interp_locate");
        hipLaunchKernelGGL(interp_locate_kernel, dim3(grid1(n)), dim3(256), 0, st, box_of(p),
                           p.verts, nx, ny, p.ntet, p.bin_start, p.bin_list, qp, n, p.mode, idx, w);
        return hip_status(hipGetLastError(), FFDAS_ERROR_CUDA_LAUNCH_FAILED);
    }
    char *c = static_cast<char *>(scratch);
    float4 *pts = (float4 *)(c + ls.pts);
    int *best = (int *)(c + ls.best), *cnt = (int *)(c + ls.cnt), *start = (int *)(c + ls.start);
    const int64_t ncell = p.ntet / 6;
    // Lanes per cell, from the points in the box of an average tetrahedron (its bins from the
    // list total, the points per bin as if evenly spread): one lane for every six points, those
    // of a run sharing it two points a lane.  Measured by lanes (runs x points): 9 points
    // (256 x 64 x 64 vertices, 128^3 points) 0.59 ms 1 x 1, 0.55 2 x 1, 0.61 2 x 4; 99 points
    // (128 x 32 x 32, 180^3) 2.84 ms 1 x 1, 0.98 4 x 4; 414 points (64 x 16 x 20, 180^3) 12.4 ms
    // 1 x 1, 0.91 8 x 8; 0.2 points (400 x 90 x 90, 40^3) 0.44 ms 1 x 1, 0.53 4 x 1.  A cell may
    // have many waves (2 x 2 x 2 vertices, 128^3 points: 117 ms with 64 lanes a cell, 0.22 so), and what is
    // far from the average is left over (64 x 16 x 20, 128^3 points in a sixteenth of the box along each axis:
    // 52 ms walked by the lanes, 2 so).
    int lgr = 0, lgp = 0;
    if (p.ntet > 0) {
        const double bins = (double)p.list_total / (double)p.ntet, dens = (double)n / (double)kBins3;
        const auto lg = [](double v) { return v > 1.0 ? (int)(std::log2(v) + 0.5) : 0; };
        const int all = lg(bins * dens / 6.0);
        lgp = std::min({all, lg(std::cbrt(bins) * dens / 2.0), 6});      // the lanes of a run in one wave
        lgr = std::min(all - lgp, 14);
        while (lgr + lgp > 0 && ncell > (int64_t)1 << (30 - lgr - lgp)) (lgr > 0 ? lgr : lgp)--;
    }
    const Leftover rest{(unsigned long long *)(cnt + ls.list_counts()), (int4 *)(c + ls.work), ls.cap,
                        (int)std::max<int64_t>(n >> 12, 512)};
    ProfScope ps(st, "interp_locate");
    const Box b = box_of(p);
    hipLaunchKernelGGL(interp_zero_i32_kernel, dim3(1024), dim3(256), 0, st, cnt, ls.counts());
    hipLaunchKernelGGL(interp_point_bin_kernel, dim3(grid1(n)), dim3(256), 0, st, b, qp, n, cnt, idx);
    size_t scan_bytes = ls.scan_bytes;
    if (rocprim::exclusive_scan(c + ls.scan, scan_bytes, cnt, start, 0, (size_t)kBins3 + 1,
                                rocprim::plus<int>(), st) != hipSuccess)
        return FFDAS_ERROR_CUDA_LAUNCH_FAILED;
    hipLaunchKernelGGL(interp_point_order_kernel, dim3(grid1(n)), dim3(256), 0, st, b, qp, n, start,
                       cnt, pts, best);
    if (ncell > 0) {
        auto go = [&](auto cells, auto left) {
            hipLaunchKernelGGL(cells, dim3(grid1(ncell << (lgr + lgp))), dim3(256), 0, st, b, p.verts, p.flat,
                               ncell, nx, ny, lgr, lgp, start, pts, best, rest);
            hipLaunchKernelGGL(left, dim3(1024), dim3(256), 0, st, b, p.verts, p.flat, nx, ny, start, pts,
                               best, rest);
        };
        if (p.any_flat)
            go(interp_locate_cells_kernel<true>, interp_locate_rest_kernel<true>);
        else
            go(interp_locate_cells_kernel<false>, interp_locate_rest_kernel<false>);
    }
    hipLaunchKernelGGL(interp_found_kernel, dim3(grid1(n)), dim3(256), 0, st, p.verts, nx, ny,
                       start + kBins3, pts, best, p.mode, idx, w);
    return hip_status(hipGetLastError(), FFDAS_ERROR_CUDA_LAUNCH_FAILED);
}

size_t lookup_ids(int64_t n) { return up256((size_t)n * sizeof(int)); }
size_t lookup_weights(int mode, int64_t n) {
    return mode == FFDAS_INTERP_NEAREST ? 0 : up256((size_t)n * 3 * sizeof(float));
}

// Frames per chunk: the smallest power of two that holds all, at most 64 bytes of 4-byte
// elements and 8 frames of others (the 64-byte block a vertex load takes whole).
int frames_per_chunk(int64_t B, size_t elem) {
    const int most = elem == 4 ? 16 : 8;
    int f = 1;
    while (f < most && f < B) f *= 2;
    return f;
}

// Bytes of the frame-inner copy.  One frame is read where it is, unless the output overlaps it (a
// call that warps a volume in place): every value of x is read before any output is written.
size_t frames_bytes(int64_t B, int64_t npts, size_t elem, const void *x, const void *out, int64_t n) {
    const int f = frames_per_chunk(B, elem);
    const uintptr_t a = reinterpret_cast<uintptr_t>(x), b = reinterpret_cast<uintptr_t>(out);
    if (f == 1 && (a + (size_t)npts * elem <= b || b + (size_t)n * elem <= a)) return 0;
    return (size_t)((B + f - 1) / f) * f * npts * elem;
}

template <typename R, int CW, int FPC>
ffdas_error_t evaluate_f(ffdas_context &h, const ffdas_interpolation_plan &p, const void *x,
                         void *out, const int *idx, const float *w, int64_t n, int64_t B,
                         const El<R, CW> &f, void *ws) {   // ws: the frame-inner copy, or null
    using E = El<R, CW>;
    using F = Frames<R, CW, FPC>;
    const int64_t npts = p.nx * p.ny * p.nz, chunks = (B + FPC - 1) / FPC;
    const F *xfi = static_cast<const F *>(x);
    if (ws) {
        ProfScope ps(h.stream, "interp_frames");
        hipLaunchKernelGGL((interp_frames_kernel<R, CW, FPC>), dim3(grid1(npts), (unsigned)chunks),
                           dim3(256), 0, h.stream, static_cast<const E *>(x), static_cast<F *>(ws),
                           npts, B);
        xfi = static_cast<const F *>(ws);
    }
    const dim3 grid(grid1(n), (unsigned)chunks);
    ProfScope ps(h.stream, "interp_eval");
    if (p.mode == FFDAS_INTERP_NEAREST)
        hipLaunchKernelGGL((interp_nearest_kernel<R, CW, FPC>), grid, dim3(256), 0, h.stream, xfi,
                           static_cast<E *>(out), idx, n, npts, B, f);
    else
    {
        auto go = [&](auto kern) {
            hipLaunchKernelGGL(kern, grid, dim3(256), 0, h.stream, xfi, static_cast<E *>(out), idx,
                               w, (int)p.nx, (int)p.ny, n, npts, B, f);
        };
        if (reinterpret_cast<uintptr_t>(out) % 128 == 0 && n * sizeof(E) % 128 == 0)
            go(interp_linear_kernel<R, CW, FPC, true>);
        else
            go(interp_linear_kernel<R, CW, FPC, false>);
    }
    return hip_status(hipGetLastError(), FFDAS_ERROR_CUDA_LAUNCH_FAILED);
}

template <typename R, int CW>
ffdas_error_t evaluate(ffdas_context &h, const ffdas_interpolation_plan &p, const void *x, void *out,
                       const int *idx, const float *w, int64_t n, int64_t B, const void *fill,
                       void *ws) {
    El<R, CW> f;
    for (int c = 0; c < CW; c++) f.c[c] = static_cast<const R *>(fill)[c];
    constexpr size_t elem = sizeof(R) * CW;
    switch (frames_per_chunk(B, elem)) {
        case 1: return evaluate_f<R, CW, 1>(h, p, x, out, idx, w, n, B, f, ws);
        case 2: return evaluate_f<R, CW, 2>(h, p, x, out, idx, w, n, B, f, ws);
        case 4: return evaluate_f<R, CW, 4>(h, p, x, out, idx, w, n, B, f, ws);
        case 8: return evaluate_f<R, CW, 8>(h, p, x, out, idx, w, n, B, f, ws);
        default:
            if constexpr (elem == 4) return evaluate_f<R, CW, 16>(h, p, x, out, idx, w, n, B, f, ws);
            return FFDAS_ERROR_INTERNAL;
    }
}

ffdas_error_t build_plan(ffdas_context &h, ffdas_interpolation_plan &p, const float *gridpos) {
    const int64_t npts = p.nx * p.ny * p.nz;
    hipStream_t st = h.stream;
    if (hipMalloc((void **)&p.verts, (size_t)npts * (sizeof(float4) + 1)) != hipSuccess)
        return FFDAS_ERROR_ALLOCATION_FAILED;
    p.flat = reinterpret_cast<unsigned char *>(p.verts + npts);
    const int nblk = (int)std::min<int64_t>(1024, std::max<int64_t>(1, (npts + 255) / 256));
    void *ws = nullptr;
    const size_t head_bytes = up256(sizeof(PlanHead));
    FFDAS_TRY(h.workspace(head_bytes + (size_t)nblk * 6 * sizeof(float), &ws));
    h.xcopy.valid = false;   // the converted-x record of the delay-and-sum calls
    PlanHead *head = static_cast<PlanHead *>(ws);
    float *part = reinterpret_cast<float *>(static_cast<char *>(ws) + head_bytes);
    hipLaunchKernelGGL(interp_verts_kernel, dim3(nblk), dim3(256), 0, st, gridpos, npts, p.verts, part);
    hipLaunchKernelGGL(interp_box_kernel, dim3(1), dim3(64), 0, st, part, nblk, head);
    p.ntet = 6 * (p.nx - 1) * (p.ny - 1) * (p.nz - 1);
    if (p.ntet > 0)
        hipLaunchKernelGGL(interp_total_kernel, dim3(std::min(grid1(p.ntet / 6), 1024)), dim3(256), 0,
                           st, p.verts, p.ntet / 6, (int)p.nx, (int)p.ny, head, p.flat);
    PlanHead hh{};
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipMemcpyAsync(&hh, head, sizeof(hh), hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    FFDAS_TRY(hip_status(e));
    for (int a = 0; a < 3; a++) {
        p.bmin[a] = hh.box.mn[a];
        p.scale[a] = hh.box.sc[a];
    }
    p.any_flat = p.ntet > 0 && hh.total >= kAnyFlat;
    hh.total &= kAnyFlat - 1;
    // entries of a point-by-point location's lists
    if (hh.total > (unsigned long long)INT_MAX || p.ntet > INT_MAX) return FFDAS_ERROR_DIMS_TOO_LARGE;
    p.list_total = (long long)hh.total;
    return FFDAS_SUCCESS;
}

}  // namespace
}  // namespace ffdas

using namespace ffdas;

static ffdas_error_t create_interpolation_plan_call(ffdas_handle_t handle,
                                                         ffdas_interpolation_plan_t *plan,
                                                         int64_t nx, int64_t ny, int64_t nz,
                                                         const float *gridpos,
                                                         ffdas_interp_mode_t mode) {
    if (!handle) return FFDAS_ERROR_INVALID_HANDLE;
    if (!plan || !gridpos) return FFDAS_ERROR_NULL_POINTER;
    *plan = nullptr;
    if (nx <= 0 || ny <= 0 || nz <= 0) return FFDAS_ERROR_INVALID_DIMS;
    if (mode != FFDAS_INTERP_NEAREST && mode != FFDAS_INTERP_LINEAR)
        return FFDAS_ERROR_INVALID_ARGUMENT;
    // vertex ids are 32-bit in the lookup arrays; the bin lists hold vertex * 8 + t
    if (nx > INT_MAX / 8 / ny / nz || 6 * (nx - 1) * (ny - 1) * (nz - 1) > INT_MAX)
        return FFDAS_ERROR_DIMS_TOO_LARGE;
    FFDAS_TRY(handle->check_device());
    auto *p = new (std::nothrow) ffdas_interpolation_plan;
    if (!p) return FFDAS_ERROR_HOST_MEMORY_INSUFFICIENT;
    p->device = handle->device_id;
    p->nx = nx;
    p->ny = ny;
    p->nz = nz;
    p->mode = mode;
    const ffdas_error_t err = build_plan(*handle, *p, gridpos);
    if (err != FFDAS_SUCCESS) {
        (void)hipStreamSynchronize(handle->stream);
        free_plan_device(p);
        delete p;
        return err;
    }
    *plan = p;
    return FFDAS_SUCCESS;
}

extern "C" ffdas_error_t ffdas_create_interpolation_plan(ffdas_handle_t handle,
                                                         ffdas_interpolation_plan_t *plan,
                                                         int64_t nx, int64_t ny, int64_t nz,
                                                         const float *gridpos,
                                                         ffdas_interp_mode_t mode) {
    ffdas::CallScope cs(handle, "ffdas_create_interpolation_plan");
    return cs.done(create_interpolation_plan_call(handle, plan, nx, ny, nz, gridpos, mode));
}

static ffdas_error_t interpolation_preprocess_call(ffdas_handle_t handle,
                                                        ffdas_interpolation_plan_t plan,
                                                        int64_t num_querypos,
                                                        const float *querypos) {
    if (!handle) return FFDAS_ERROR_INVALID_HANDLE;
    if (!plan || !querypos) return FFDAS_ERROR_NULL_POINTER;
    if (num_querypos <= 0) return FFDAS_ERROR_INVALID_DIMS;
    FFDAS_TRY(handle->check_device());
    // drop an earlier preprocessed set (the stream may still read it)
    if (plan->pre_idx || plan->pre_w) {
        FFDAS_TRY(hip_status(hipStreamSynchronize(handle->stream), FFDAS_ERROR_CUDA_SYNC_FAILED));
        if (plan->pre_idx) (void)hipFree(plan->pre_idx);
        if (plan->pre_w) (void)hipFree(plan->pre_w);
        plan->pre_idx = nullptr;
        plan->pre_w = nullptr;
    }
    plan->pre = false;
    plan->pre_n = 0;
    LocateScratch ls;
    CallScratch call(*handle);
    void *scratch = nullptr;
    if (locate_by_cells(num_querypos)) {
        FFDAS_TRY(LocateScratch::plan(num_querypos, handle->stream, ls));
        FFDAS_TRY(call.get(ls.total, &scratch));
    }
    const size_t wb = lookup_weights(plan->mode, num_querypos);
    if (hipMalloc((void **)&plan->pre_idx, lookup_ids(num_querypos)) != hipSuccess)
        return FFDAS_ERROR_ALLOCATION_FAILED;
    if (wb && hipMalloc((void **)&plan->pre_w, wb) != hipSuccess) return FFDAS_ERROR_ALLOCATION_FAILED;
    FFDAS_TRY(locate(*handle, *plan, querypos, num_querypos, plan->pre_idx, plan->pre_w, ls, scratch));
    plan->pre = true;
    plan->pre_n = num_querypos;
    return FFDAS_SUCCESS;
}

extern "C" ffdas_error_t ffdas_interpolation_preprocess(ffdas_handle_t handle,
                                                        ffdas_interpolation_plan_t plan,
                                                        int64_t num_querypos,
                                                        const float *querypos) {
    ffdas::CallScope cs(handle, "ffdas_interpolation_preprocess");
    return cs.done(interpolation_preprocess_call(handle, plan, num_querypos, querypos));
}

static ffdas_error_t interpolation_call(ffdas_handle_t handle, ffdas_interpolation_plan_t plan,
                                             int64_t num_querypos, const float *querypos,
                                             ffdas_tensor_desc_t x_desc, const void *x, void *out,
                                             const void *fill_value) {
    if (!handle) return FFDAS_ERROR_INVALID_HANDLE;
    if (!plan || !x_desc || !x || !out || !fill_value) return FFDAS_ERROR_NULL_POINTER;
    const bool use_pre = plan->pre && plan->pre_n == num_querypos;
    if (!querypos && !use_pre) return FFDAS_ERROR_INVALID_ARGUMENT;
    if (num_querypos <= 0) return FFDAS_ERROR_INVALID_DIMS;
    const ffdas_tensor_desc &xd = *x_desc;
    const size_t nd = xd.dims.size();
    if (nd != 3 && nd != 4) return FFDAS_ERROR_INVALID_DIMS;
    const size_t o = nd - 3;
    if (xd.dims[o] != plan->nz || xd.dims[o + 1] != plan->ny || xd.dims[o + 2] != plan->nx)
        return FFDAS_ERROR_INVALID_DIMS;
    // packed layout: the kernels index x as [frame][vertex]
    int64_t expect = 1;
    for (size_t k = nd; k-- > 0;) {
        if (xd.dims[k] > 1 && xd.strides[k] != expect) return FFDAS_ERROR_NON_CONTIGUOUS;
        expect *= xd.dims[k];
    }
    const int64_t B = nd == 4 ? xd.dims[0] : 1;
    if (B <= 0) return FFDAS_ERROR_INVALID_DIMS;
    const int64_t bs = plan->nz * plan->ny * plan->nx;
    if ((B + kFramesPerThread - 1) / kFramesPerThread > 65535) return FFDAS_ERROR_DIMS_TOO_LARGE;
    FFDAS_TRY(handle->check_device());

    size_t elem;
    switch (xd.dtype) {
        case FFDAS_R_32F: elem = 4; break;
        case FFDAS_C_32F: case FFDAS_R_64F: elem = 8; break;
        case FFDAS_C_64F: elem = 16; break;
        default: return FFDAS_ERROR_UNSUPPORTED_TYPE;
    }
    if (!use_pre) {
        // a location is not captured into a graph (preprocess first)
        hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(handle->stream, &cs) == hipSuccess && cs != hipStreamCaptureStatusNone)
            return FFDAS_ERROR_ALLOCATION_FAILED;
    }
    // The one-shot lookup, then the location's scratch or, after it, the frame-inner copy of x (a copy
    // alone is kept in the workspace, as of preprocessed points).
    const bool cells = !use_pre && locate_by_cells(num_querypos);
    LocateScratch ls;
    if (cells) FFDAS_TRY(LocateScratch::plan(num_querypos, handle->stream, ls));
    const size_t ib = use_pre ? 0 : lookup_ids(num_querypos);
    const size_t wb = use_pre ? 0 : lookup_weights(plan->mode, num_querypos);
    const size_t fb = frames_bytes(B, bs, elem, x, out, num_querypos);
    CallScratch call(*handle);
    const int *idx = plan->pre_idx;
    const float *w = plan->pre_w;
    void *frames = nullptr;
    if (!use_pre) {
        void *ws = nullptr;
        FFDAS_TRY(call.get(ib + wb + std::max(ls.total, fb), &ws));
        char *c = static_cast<char *>(ws), *rest = c + ib + wb;
        int *tidx = reinterpret_cast<int *>(c);
        float *tw = wb ? reinterpret_cast<float *>(c + ib) : nullptr;
        FFDAS_TRY(locate(*handle, *plan, querypos, num_querypos, tidx, tw, ls, cells ? rest : nullptr));
        idx = tidx;
        w = tw;
        if (fb) frames = rest;
    } else {
        handle->xcopy.valid = false;
        FFDAS_TRY(handle->workspace(fb, &frames));
    }
    ffdas_error_t err;
    switch (xd.dtype) {
        case FFDAS_R_32F: err = evaluate<float, 1>(*handle, *plan, x, out, idx, w, num_querypos, B, fill_value, frames); break;
        case FFDAS_C_32F: err = evaluate<float, 2>(*handle, *plan, x, out, idx, w, num_querypos, B, fill_value, frames); break;
        case FFDAS_R_64F: err = evaluate<double, 1>(*handle, *plan, x, out, idx, w, num_querypos, B, fill_value, frames); break;
        default: err = evaluate<double, 2>(*handle, *plan, x, out, idx, w, num_querypos, B, fill_value, frames); break;
    }
    return err;
}

extern "C" ffdas_error_t ffdas_interpolation(ffdas_handle_t handle, ffdas_interpolation_plan_t plan,
                                             int64_t num_querypos, const float *querypos,
                                             ffdas_tensor_desc_t x_desc, const void *x, void *out,
                                             const void *fill_value) {
    ffdas::CallScope cs(handle, "ffdas_interpolation");
    return cs.done(interpolation_call(handle, plan, num_querypos, querypos, x_desc, x, out,
                                      fill_value));
}

extern "C" ffdas_error_t ffdas_destroy_interpolation_plan(ffdas_handle_t handle,
                                                          ffdas_interpolation_plan_t plan) {
    if (!plan) return FFDAS_SUCCESS;
    if (handle) (void)hipStreamSynchronize(handle->stream);
    free_plan_device(plan);
    delete plan;
    return FFDAS_SUCCESS;
}
