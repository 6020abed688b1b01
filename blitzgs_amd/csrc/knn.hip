// distCUDA2 for gfx950: mean squared distance to the three nearest neighbours.
//
// Reference: BlitzGS submodule/simple-knn/spatial.cu:15-26 and
// simple_knn.cu:30-221 (bbox reduce, 10-bit Morton codes, radix sort, boxes of
// 1024 sorted points, box-pruned exact 3-NN, output (d0+d1+d2)/3).  The
// reference's pruning is conservative, so its output is the exact 3-NN
// statistic; it scans every box for every point (O(P^2/1024) box tests).
//
// Here: a uniform grid of about 4.5 points per cell is built with a counting
// sort (bbox reduce, cell histogram, device-wide scan, scatter), and every
// point searches the cell shells around its own cell until the third-best
// squared distance is below the distance to the unsearched region (computed
// in double with a relative safety margin).  Queries run in cell order so a
// wave's lanes walk neighbouring cells.  Distances use
// (dx*dx + dy*dy) + dz*dz with dx = other - self and no fused multiply-add,
// and the output is ((b0 + b1) + b2) / 3 -- the reference's expressions -- so
// the result is the same exact value the CPU oracle computes.
#include <float.h>

#include <algorithm>
#include <cmath>
#include <mutex>

#include "gs_device.h"
#include "gs_host.h"
#include "../../include/blitzgs_amd.h"

namespace {

constexpr int RED_BLOCKS = 1024;
constexpr int SCAN_BLOCK = 1024;
constexpr int QT = 64;         // queries per block: one wave, whose LDS is free as soon as it ends

constexpr size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

struct KnnLayout {
    size_t partial, cell_of, rank, count, start, blocksum, sorted, total;
};

// upper bound on the grid's cell count (the host grid rule enlarges the cell
// size until it holds, e.g. for flat or degenerate point sets)
constexpr size_t max_cells(int P) { return 2 * (size_t)P + 1024; }

constexpr KnnLayout knn_layout(int P)
{
    KnnLayout l{};
    const size_t NCmax = max_cells(P);
    size_t o = 0;
    l.partial = o; o = align256(o + sizeof(float) * 6 * RED_BLOCKS);
    l.cell_of = o; o = align256(o + sizeof(uint32_t) * (size_t)P);
    l.rank = o; o = align256(o + sizeof(uint32_t) * (size_t)P);
    l.count = o; o = align256(o + sizeof(uint32_t) * (NCmax + 1));
    l.start = o; o = align256(o + sizeof(uint32_t) * (NCmax + 1));
    l.blocksum = o; o = align256(o + sizeof(uint32_t) * ((NCmax + 1) / SCAN_BLOCK + 2));
    l.sorted = o; o = align256(o + sizeof(float4) * (size_t)P);
    l.total = o;
    return l;
}

template <typename T>
T* at(void* base, size_t off) { return reinterpret_cast<T*>(static_cast<char*>(base) + off); }

__global__ __launch_bounds__(256) void bbox_partial_kernel(int P, const float* __restrict__ pts, float* __restrict__ partial)
{
    float mn[3] = {FLT_MAX, FLT_MAX, FLT_MAX}, mx[3] = {-FLT_MAX, -FLT_MAX, -FLT_MAX};
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < P; i += gridDim.x * blockDim.x) {
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const float v = pts[3 * (size_t)i + k];
            mn[k] = fminf(mn[k], v);
            mx[k] = fmaxf(mx[k], v);
        }
    }
    __shared__ float s[6][256];
#pragma unroll
    for (int k = 0; k < 3; k++) { s[k][threadIdx.x] = mn[k]; s[3 + k][threadIdx.x] = mx[k]; }
    __syncthreads();
    for (int off = 128; off > 0; off >>= 1) {
        if ((int)threadIdx.x < off) {
#pragma unroll
            for (int k = 0; k < 3; k++) {
                s[k][threadIdx.x] = fminf(s[k][threadIdx.x], s[k][threadIdx.x + off]);
                s[3 + k][threadIdx.x] = fmaxf(s[3 + k][threadIdx.x], s[3 + k][threadIdx.x + off]);
            }
        }
        __syncthreads();
    }
    if (threadIdx.x < 6) partial[6 * blockIdx.x + threadIdx.x] = s[threadIdx.x][0];
}

struct Grid {
    double mn[3], hk[3];
    double slack[3];   // bounds the rounding of cell coordinates and cell faces
    int n[3];
};

__device__ __forceinline__ int cell_coord(float v, double mn, double hk, int n)
{
    int c = (int)floor(((double)v - mn) / hk);
    return c < 0 ? 0 : (c >= n ? n - 1 : c);
}

__global__ __launch_bounds__(256) void zero_u32_kernel(size_t n, uint32_t* __restrict__ p)
{
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = 0;
}

__global__ __launch_bounds__(256) void cell_hist_kernel(int P, const float* __restrict__ pts, Grid g,
                                                        uint32_t* __restrict__ cell_of, uint32_t* __restrict__ rank,
                                                        uint32_t* __restrict__ count)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= P) return;
    const int cx = cell_coord(pts[3 * (size_t)i], g.mn[0], g.hk[0], g.n[0]);
    const int cy = cell_coord(pts[3 * (size_t)i + 1], g.mn[1], g.hk[1], g.n[1]);
    const int cz = cell_coord(pts[3 * (size_t)i + 2], g.mn[2], g.hk[2], g.n[2]);
    const uint32_t c = (uint32_t)((cz * g.n[1] + cy) * g.n[0] + cx);
    cell_of[i] = c;
    rank[i] = atomicAdd(&count[c], 1u);
}

// device-wide exclusive scan, three kernels: block scan + block sums, scan of
// the block sums, add
__device__ __forceinline__ uint32_t block_scan_excl(uint32_t v, uint32_t* s_wave, uint32_t* total)
{
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    uint32_t x = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t y = __shfl_up(x, off, 64);
        if (lane >= off) x += y;
    }
    if (lane == 63) s_wave[wid] = x;
    __syncthreads();
    if (wid == 0) {
        uint32_t w = lane < 16 ? s_wave[lane] : 0;
#pragma unroll
        for (int off = 1; off < 16; off <<= 1) {
            const uint32_t y = __shfl_up(w, off, 64);
            if (lane >= off) w += y;
        }
        if (lane < 16) s_wave[16 + lane] = w;
    }
    __syncthreads();
    const uint32_t wbase = wid == 0 ? 0 : s_wave[16 + wid - 1];
    *total = s_wave[31];
    __syncthreads();
    return wbase + x - v;
}

__global__ __launch_bounds__(SCAN_BLOCK) void scan_blocks_kernel(size_t n, const uint32_t* __restrict__ in,
                                                                 uint32_t* __restrict__ out, uint32_t* __restrict__ bsum)
{
    __shared__ uint32_t s_wave[32];
    const size_t i = blockIdx.x * (size_t)SCAN_BLOCK + threadIdx.x;
    const uint32_t v = i < n ? in[i] : 0u;
    uint32_t tot;
    const uint32_t pre = block_scan_excl(v, s_wave, &tot);
    if (i < n) out[i] = pre;
    if (threadIdx.x == 0) bsum[blockIdx.x] = tot;
}

__global__ __launch_bounds__(SCAN_BLOCK) void scan_sums_kernel(int nb, uint32_t* __restrict__ bsum)
{
    __shared__ uint32_t s_wave[32];
    uint32_t base = 0;
    for (int b0 = 0; b0 < nb; b0 += SCAN_BLOCK) {
        const int b = b0 + threadIdx.x;
        const uint32_t v = b < nb ? bsum[b] : 0u;
        uint32_t tot;
        const uint32_t pre = block_scan_excl(v, s_wave, &tot);
        if (b < nb) bsum[b] = base + pre;
        base += tot;
    }
}

__global__ __launch_bounds__(256) void scan_add_kernel(size_t n, uint32_t* __restrict__ out, const uint32_t* __restrict__ bsum)
{
    const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    if (i < n) out[i] += bsum[i / SCAN_BLOCK];
}

__global__ __launch_bounds__(256) void cell_scatter_kernel(int P, const float* __restrict__ pts,
                                                           const uint32_t* __restrict__ cell_of,
                                                           const uint32_t* __restrict__ rank,
                                                           const uint32_t* __restrict__ start,
                                                           float4* __restrict__ sorted)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= P) return;
    const uint32_t pos = start[cell_of[i]] + rank[i];
    sorted[pos] = make_float4(pts[3 * (size_t)i], pts[3 * (size_t)i + 1], pts[3 * (size_t)i + 2], __uint_as_float((uint32_t)i));
}

// insertion of d into the ascending triple b0 <= b1 <= b2 (updateKBest,
// simple_knn.cu:132-146): min / median-of-three are exact, so
//   b0' = min(b0, d), b1' = med3(b0, b1, d), b2' = med3(b1, b2, d)
// is the same triple the reference's swap chain produces (inputs are finite or +inf)
__device__ __forceinline__ void upd3(float& b0, float& b1, float& b2, float d)
{
    const float n2 = __builtin_amdgcn_fmed3f(b1, b2, d);
    const float n1 = __builtin_amdgcn_fmed3f(b0, b1, d);
    b0 = __builtin_fminf(b0, d);
    b1 = n1;
    b2 = n2;
}

// candidates sorted[k, k + 4) against the query, four loads in flight.  TAIL:
// those from hi on are masked (and their loads clamped); OWN: so is the query
// itself, at sorted position `self`, which only its own run of cells holds.
// The masks are half of a candidate's VALU instructions, which bind where the
// runs are long (points with a few far outliers, whose bulk shares a few cells):
// 100k points, three of them far away, 45.8 ms with both masks on every
// candidate, 35.4 ms so; without outliers 0-8 % faster.
template <bool TAIL, bool OWN>
__device__ __forceinline__ void scan_four(uint32_t k, uint32_t hi, const float4* __restrict__ sorted, float4 q,
                                          uint32_t self, float& b0, float& b1, float& b2)
{
    float4 o[4];
#pragma unroll
    for (uint32_t u = 0; u < 4; u++) o[u] = sorted[TAIL ? min(k + u, hi - 1) : k + u];
#pragma unroll
    for (uint32_t u = 0; u < 4; u++) {
        const float dx = o[u].x - q.x, dy = o[u].y - q.y, dz = o[u].z - q.z;
        const float d = (dx * dx + dy * dy) + dz * dz;
        upd3(b0, b1, b2, (TAIL && k + u >= hi) || (OWN && k + u == self) ? __builtin_huge_valf() : d);
    }
}

// candidates sorted[lo, hi)
template <bool OWN>
__device__ __forceinline__ void scan_segment(uint32_t lo, uint32_t hi, const float4* __restrict__ sorted, float4 q,
                                             uint32_t self, float& b0, float& b1, float& b2)
{
    uint32_t k = lo;
    for (; k + 4 <= hi; k += 4) scan_four<false, OWN>(k, hi, sorted, q, self, b0, b1, b2);
    if (k < hi) scan_four<true, OWN>(k, hi, sorted, q, self, b0, b1, b2);
}

// What a point `gap` cells beyond the neighbouring cell keeps from the query
// along one axis, squared: `near` is the query's distance to that neighbour's
// face.  The slack covers the double rounding of the cell coordinates and of the
// faces, the relative margin the fp32 rounding of the distances it is compared
// with (below 4e-7) and of this value.
__device__ __forceinline__ float axis_gap2(double near, double h, int gap, double slack)
{
    const double d = fmax(near + (double)gap * h - slack, 0.0);
    return (float)(d * d * (1.0 - 2e-6));
}

// distance from the query to the outside of the cell box c +- r (grid borders
// excluded); DBL_MAX when the box covers the whole grid
__device__ __forceinline__ double box_bound(const Grid& g, const int (&c)[3], const float (&qv)[3], int r)
{
    double bound = DBL_MAX;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const double lo = g.mn[k] + (double)(c[k] - r) * g.hk[k];
        const double hi = g.mn[k] + (double)(c[k] + r + 1) * g.hk[k];
        if (c[k] - r > 0) bound = fmin(bound, (double)qv[k] - lo - g.slack[k]);
        if (c[k] + r + 1 < g.n[k]) bound = fmin(bound, hi - (double)qv[k] - g.slack[k]);
    }
    return bound;
}

// true when the third-best squared distance is provably below every point
// outside the box (the bound is padded by a relative margin)
__device__ __forceinline__ bool box_done(double bound, float b2)
{
    if (bound == DBL_MAX) return true;
    if (bound < 0) bound = 0;
    return (double)b2 < bound * bound * (1.0 - 1e-6);
}

// Queries run in cell order (one thread per sorted point), so a wave's
// queries sit in neighbouring cells.  The 3x3x3 cells around the query are 9
// runs of x-consecutive cells, i.e. 9 contiguous ranges of the cell-sorted
// points.  The query's own run is scanned first; of the other eight a lane
// keeps, in an LDS list, only the cells whose nearest face is not beyond its
// third-best distance, and walks its list candidate by candidate.  Where the
// points are denser than the grid's average that leaves about a quarter of the
// candidates, and one flat loop over them costs a wave its longest lane's
// total, not the sum over the runs of the longest lane in each.  Only if the
// third-best distance is not yet provably final are further shells visited,
// again without the rows that lie beyond it.  Bound by the latency of the
// gathered candidates and by the longest lane of a wave; by VALU issue where a
// cell holds hundreds of points.  10M points of a ground plane with dense
// clusters, whole call at 3 points per cell: 6.1 ms with every run scanned in
// turn, 4.3 ms so.
__global__ __launch_bounds__(QT) void knn_query_kernel(int P, Grid g, const uint32_t* __restrict__ start,
                                                       const float4* __restrict__ sorted, float* __restrict__ out)
{
    __shared__ uint32_t s_lo[8][QT], s_hi[8][QT];
    __shared__ float s_gap[8][QT];
    const int t = threadIdx.x;
    const int s = blockIdx.x * QT + t;
    if (s >= P) return;
    const float4 q = sorted[s];
    const uint32_t self = (uint32_t)s;   // the query's own position in the sorted points
    const float qv[3] = {q.x, q.y, q.z};
    int c[3];
    double dlo[3], dhi[3];               // distances to the faces of the query's cell
#pragma unroll
    for (int k = 0; k < 3; k++) {
        c[k] = cell_coord(qv[k], g.mn[k], g.hk[k], g.n[k]);
        dlo[k] = (double)qv[k] - (g.mn[k] + (double)c[k] * g.hk[k]);
        dhi[k] = (g.mn[k] + (double)(c[k] + 1) * g.hk[k]) - (double)qv[k];
    }
    float b0 = FLT_MAX, b1 = FLT_MAX, b2 = FLT_MAX;

    // r <= 1
    {
        const int x0 = max(0, c[0] - 1), x1 = min(g.n[0] - 1, c[0] + 1);
        const uint32_t own = (uint32_t)((c[2] * g.n[1] + c[1]) * g.n[0]);
        scan_segment<true>(start[own + (uint32_t)x0], start[own + (uint32_t)x1 + 1], sorted, q, self, b0, b1, b2);
        float lo2[3], hi2[3];
#pragma unroll
        for (int k = 0; k < 3; k++) {
            lo2[k] = axis_gap2(dlo[k], g.hk[k], 0, g.slack[k]);
            hi2[k] = axis_gap2(dhi[k], g.hk[k], 0, g.slack[k]);
        }
        // the four runs that share a face with the query's own come first
        constexpr int DY[8] = {-1, 1, 0, 0, -1, 1, -1, 1}, DZ[8] = {0, 0, -1, 1, -1, -1, 1, 1};
        uint32_t lo[8], hi[8];
        float gap[8];
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int z = c[2] + DZ[j], y = c[1] + DY[j];
            gap[j] = (DY[j] < 0 ? lo2[1] : DY[j] > 0 ? hi2[1] : 0.f) + (DZ[j] < 0 ? lo2[2] : DZ[j] > 0 ? hi2[2] : 0.f);
            lo[j] = hi[j] = 0;
            if (z >= 0 && z < g.n[2] && y >= 0 && y < g.n[1] && !(b2 < gap[j])) {
                const uint32_t row = (uint32_t)((z * g.n[1] + y) * g.n[0]);
                const int xa = b2 < gap[j] + lo2[0] ? c[0] : x0, xb = b2 < gap[j] + hi2[0] ? c[0] : x1;
                lo[j] = start[row + (uint32_t)xa];
                hi[j] = start[row + (uint32_t)xb + 1];
            }
        }
        int n = 0;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            if (lo[j] < hi[j]) {
                s_lo[n][t] = lo[j];
                s_hi[n][t] = hi[j];
                s_gap[n][t] = gap[j];
                n++;
            }
        }
        // a lane reads only what it wrote itself: no barrier
        uint32_t k = 0, e = 0;
        for (int i = 0;;) {
            while (k >= e && i < n) {
                k = s_lo[i][t];
                e = b2 < s_gap[i][t] ? k : s_hi[i][t];
                i++;
            }
            if (k >= e) break;
            if (gs::ballot(k + 4 > e) == 0)   // no lane at its segment's end
                scan_four<false, false>(k, e, sorted, q, self, b0, b1, b2);
            else
                scan_four<true, false>(k, e, sorted, q, self, b0, b1, b2);
            k += 4;
        }
    }
    const int rmax = max(g.n[0], max(g.n[1], g.n[2]));
    if (!box_done(box_bound(g, c, qv, 1), b2)) {
        for (int r = 2; r <= rmax; r++) {
            const int z0 = max(0, c[2] - r), z1 = min(g.n[2] - 1, c[2] + r);
            const int y0 = max(0, c[1] - r), y1 = min(g.n[1] - 1, c[1] + r);
            const int xa = max(0, c[0] - r), xb = min(g.n[0] - 1, c[0] + r);
            const float xlo2 = axis_gap2(dlo[0], g.hk[0], r - 1, g.slack[0]);
            const float xhi2 = axis_gap2(dhi[0], g.hk[0], r - 1, g.slack[0]);
            for (int z = z0; z <= z1; z++) {
                const float gz = z < c[2] ? axis_gap2(dlo[2], g.hk[2], c[2] - z - 1, g.slack[2])
                               : z > c[2] ? axis_gap2(dhi[2], g.hk[2], z - c[2] - 1, g.slack[2]) : 0.f;
                if (b2 < gz) continue;
                for (int y = y0; y <= y1; y++) {
                    const float gy = gz + (y < c[1] ? axis_gap2(dlo[1], g.hk[1], c[1] - y - 1, g.slack[1])
                                         : y > c[1] ? axis_gap2(dhi[1], g.hk[1], y - c[1] - 1, g.slack[1]) : 0.f);
                    if (b2 < gy) continue;
                    const uint32_t row = (uint32_t)((z * g.n[1] + y) * g.n[0]);
                    const bool shell_zy = (z == c[2] - r || z == c[2] + r || y == c[1] - r || y == c[1] + r);
                    if (shell_zy) {
                        // the whole x run of this shell row is new: one segment
                        scan_segment<false>(start[row + (uint32_t)xa], start[row + (uint32_t)xb + 1], sorted, q, self,
                                            b0, b1, b2);
                    } else {
                        // interior rows: only the two x ends are new
                        if (c[0] - r >= 0 && !(b2 < gy + xlo2)) {
                            const uint32_t cc = row + (uint32_t)(c[0] - r);
                            scan_segment<false>(start[cc], start[cc + 1], sorted, q, self, b0, b1, b2);
                        }
                        if (c[0] + r < g.n[0] && !(b2 < gy + xhi2)) {
                            const uint32_t cc = row + (uint32_t)(c[0] + r);
                            scan_segment<false>(start[cc], start[cc + 1], sorted, q, self, b0, b1, b2);
                        }
                    }
                }
            }
            if (box_done(box_bound(g, c, qv, r), b2)) break;
        }
    }
    out[__float_as_uint(q.w)] = ((b0 + b1) + b2) / 3.0f;
}

}  // namespace

extern "C" size_t gs_knn_workspace_bytes(int P) { return knn_layout(P < 0 ? 0 : P).total; }

namespace {

// grid build + query over the caller's (or the scratch) workspace of
// knn_layout(P).total bytes; every workspace array is written before it is
// read (the cell counters by a fill kernel), so its previous contents do not
// matter
int knn_impl(int P, const float* points, float* out, void* workspace, hipStream_t stream)
{
    const KnnLayout L = knn_layout(P);
    float* partial = at<float>(workspace, L.partial);
    uint32_t* cell_of = at<uint32_t>(workspace, L.cell_of);
    uint32_t* count = at<uint32_t>(workspace, L.count);
    uint32_t* start = at<uint32_t>(workspace, L.start);
    uint32_t* bsum = at<uint32_t>(workspace, L.blocksum);
    float4* sorted = at<float4>(workspace, L.sorted);
    uint32_t* rank = at<uint32_t>(workspace, L.rank);   // a point's place in its cell

    const int nred = (int)std::min<size_t>(RED_BLOCKS, gs_div_up((size_t)P, 256));
    GS_TIMED("knn_bbox_kernel", stream,
             hipLaunchKernelGGL(bbox_partial_kernel, dim3(nred), dim3(256), 0, stream, P, points, partial));
    GS_LAUNCH_CHECK("bbox_partial_kernel");
    float hp[6 * RED_BLOCKS];
    GS_HIP(hipMemcpyAsync(hp, partial, sizeof(float) * 6 * nred, hipMemcpyDeviceToHost, stream));
    GS_HIP(hipStreamSynchronize(stream));
    double mn[3], mx[3];
    for (int k = 0; k < 3; k++) { mn[k] = hp[k]; mx[k] = hp[3 + k]; }
    for (int b = 1; b < nred; b++)
        for (int k = 0; k < 3; k++) {
            if (hp[6 * b + k] < mn[k]) mn[k] = hp[6 * b + k];
            if (hp[6 * b + 3 + k] > mx[k]) mx[k] = hp[6 * b + 3 + k];
        }
    Grid g;
    double ext[3], vol = 1.0;
    for (int k = 0; k < 3; k++) {
        GS_REQUIRE(std::isfinite(mn[k]) && std::isfinite(mx[k]), "points must be finite");
        ext[k] = mx[k] - mn[k];
        if (ext[k] < 1e-12) ext[k] = 1e-12;
        vol *= ext[k];
    }
    // about 4.5 points per cell: coarser cells spare the points in the sparse parts
    // their shells, and the query skips what they add elsewhere (measured, whole
    // call, at 2 / 3 / 4.5 per cell: 10M points of a ground plane with dense clusters
    // 5.15 / 4.30 / 3.82 ms, 5M in clusters 2.13 / 1.70 / 1.50 ms, 1M uniform
    // 205 / 198 / 197 us, 2M on a sphere 0.54 / 0.61 / 0.70 ms; at 6 and 8 the 10M
    // take 0 and 5 % longer).  Points with a few far outliers take 24 to 33 ms per 100k
    // at any of them, by where the cell faces fall in their bulk,
    // at most 1024 cells per axis and max_cells(P) in total
    double h = cbrt(vol / ((double)P / 4.5 + 1.0));
    size_t NC = 0;
    for (int iter = 0; iter < 200; iter++) {
        NC = 1;
        for (int k = 0; k < 3; k++) {
            double c = ceil(ext[k] / h);
            if (c < 1) c = 1;
            if (c > 1024) c = 1024;
            g.n[k] = (int)c;
            NC *= (size_t)g.n[k];
        }
        if (NC <= max_cells(P)) break;
        h *= 1.25;
    }
    GS_REQUIRE(NC <= max_cells(P), "internal: grid of %zu cells exceeds the workspace bound", NC);
    for (int k = 0; k < 3; k++) {
        g.mn[k] = mn[k];
        g.hk[k] = ext[k] / g.n[k];
        g.slack[k] = 4e-15 * (std::fabs(mn[k]) + ext[k]);
    }
    GS_TIMED("knn_zero_kernel", stream,
             hipLaunchKernelGGL(zero_u32_kernel, dim3(1024), dim3(256), 0, stream, NC + 1, count));
    GS_LAUNCH_CHECK("zero_u32_kernel");
    GS_TIMED("knn_hist_kernel", stream,
             hipLaunchKernelGGL(cell_hist_kernel, dim3(gs_div_up((size_t)P, 256)), dim3(256), 0, stream, P, points, g,
                                cell_of, rank, count));
    GS_LAUNCH_CHECK("cell_hist_kernel");
    const size_t n = NC + 1;
    const unsigned nb = gs_div_up(n, SCAN_BLOCK);
    GS_TIMED("knn_scan_kernel", stream,
             hipLaunchKernelGGL(scan_blocks_kernel, dim3(nb), dim3(SCAN_BLOCK), 0, stream, n, count, start, bsum));
    GS_LAUNCH_CHECK("scan_blocks_kernel");
    GS_TIMED("knn_scan_sums_kernel", stream,
             hipLaunchKernelGGL(scan_sums_kernel, dim3(1), dim3(SCAN_BLOCK), 0, stream, (int)nb, bsum));
    GS_LAUNCH_CHECK("scan_sums_kernel");
    GS_TIMED("knn_scan_add_kernel", stream,
             hipLaunchKernelGGL(scan_add_kernel, dim3(gs_div_up(n, 256)), dim3(256), 0, stream, n, start, bsum));
    GS_LAUNCH_CHECK("scan_add_kernel");
    GS_TIMED("knn_scatter_kernel", stream,
             hipLaunchKernelGGL(cell_scatter_kernel, dim3(gs_div_up((size_t)P, 256)), dim3(256), 0, stream, P, points,
                                cell_of, rank, start, sorted));
    GS_LAUNCH_CHECK("cell_scatter_kernel");
    GS_TIMED("knn_query_kernel", stream,
             hipLaunchKernelGGL(knn_query_kernel, dim3(gs_div_up((size_t)P, QT)), dim3(QT), 0, stream, P, g, start,
                                sorted, out));
    GS_LAUNCH_CHECK("knn_query_kernel");
    GS_HIP(hipStreamSynchronize(stream));
    return GS_OK;
}

}  // namespace

extern "C" int gs_knn_meandist3(int P, const float* points, float* out, void* workspace, hipStream_t stream)
{
    gs::clear_error();
    GS_REQUIRE(P >= 0, "P must be >= 0");
    if (P == 0) return GS_OK;
    GS_REQUIRE(workspace != nullptr, "workspace must be non-null (gs_knn_workspace_bytes)");
    return knn_impl(P, points, out, workspace, stream);
}

// ---------------------------------------------------------- allocation-free
//
// gs_knn_meandist3_noalloc: the same computation with its workspace in a
// file-scope device array instead of caller memory, for callers that cannot
// allocate (serving loops, harnesses that forbid hipMalloc).  It cannot be
// captured into a HIP graph: like gs_knn_meandist3 it reads the bounding box
// back to the host mid-call and synchronises the stream.  Each GPU the library
// runs on holds its own copy of the array (KNN_SCRATCH_BYTES, about 42 MB)
// until the process ends.  In host code `scratch` names a host-side stand-in,
// never the device memory: the per-device address comes from
// hipGetSymbolAddress on the first call on each device and only that address
// is passed to kernels and copies.  A per-device lock is held for the whole
// call, which ends with a synchronisation of its stream, so calls from several
// host threads on one GPU run one after another instead of sharing the array.

constexpr int KNN_NOALLOC_MAX_P = 1 << 20;
constexpr size_t KNN_SCRATCH_BYTES = knn_layout(KNN_NOALLOC_MAX_P).total;
static_assert(KNN_SCRATCH_BYTES % 256 == 0, "scratch size");

static __device__ __align__(256) unsigned char scratch[KNN_SCRATCH_BYTES];

namespace {
constexpr int KNN_MAX_DEVICES = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[KNN_MAX_DEVICES] = {};
std::mutex g_call_mu[KNN_MAX_DEVICES];   // one call at a time per device's scratch

// the current device's copy of `scratch` (looked up once per device)
int scratch_of_current_device(void** out)
{
    int dev = -1;
    GS_HIP(hipGetDevice(&dev));
    GS_REQUIRE(dev >= 0 && dev < KNN_MAX_DEVICES, "device %d out of range", dev);
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (g_scratch_ptr[dev] == nullptr) {
        void* p = nullptr;
        GS_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        GS_REQUIRE(p != nullptr, "no device address for the scratch array on device %d", dev);
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return GS_OK;
}
}  // namespace

extern "C" int gs_knn_meandist3_noalloc(int P, const float* points, float* out, hipStream_t stream)
{
    gs::clear_error();
    GS_REQUIRE(P >= 0, "P must be >= 0");
    GS_REQUIRE(P <= KNN_NOALLOC_MAX_P, "P = %d exceeds the allocation-free limit of %d points", P,
               KNN_NOALLOC_MAX_P);
    if (P == 0) return GS_OK;
    if (stream != nullptr) {
        int cur = -1, sdev = -1;
        GS_HIP(hipGetDevice(&cur));
        GS_HIP(hipStreamGetDevice(stream, &sdev));
        GS_REQUIRE(sdev == cur, "stream belongs to device %d, the current device is %d", sdev, cur);
    }
    void* ws = nullptr;
    if (int rc = scratch_of_current_device(&ws); rc != GS_OK) return rc;
    int dev = -1;
    GS_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lk(g_call_mu[dev]);
    return knn_impl(P, points, out, ws, stream);
}
