// Exact k-nearest neighbours on a uniform cell grid.
//
// The reference builds a left-balanced kd-tree with log2(N) thrust sorts and
// walks it per query (KNN_GWN.cu:42-66, builder_thrust.h:486-724).  Here the
// points are bucketed once into a dense cell grid (counting sort: one
// histogram, one scan, one scatter).  Many queries are answered tile by tile
// from points staged in LDS; the ones that leaves open, and small query sets,
// walk the grid's occupancy pyramid.  Candidates are kept as 64-bit keys
// (float bits of d² << 32 | index) in registers, so results are the exact k
// smallest (d², index) pairs — identical to a brute-force scan with the same
// float d² formula, ties to the lower index.
#include <algorithm>
#include <cmath>

#include "knn.h"
#include "scan.h"

dwg_knn_index::~dwg_knn_index() {
    for (auto& L : lvl) {
        dwg::dev_free(L.cell_start);
        dwg::dev_free(L.pts);
        dwg::dev_free(L.empty);
        dwg::dev_free(L.pyr);
        dwg::dev_free(L.pyr_dim);
        dwg::dev_free(L.pyr_off);
        dwg::dev_free(L.pbox);
    }
}

namespace dwg {

__device__ __forceinline__ int cell_coord(float v, float lo, float inv_cell, int dim) {
    int c = int(floorf((v - lo) * inv_cell));
    return min(max(c, 0), dim - 1);
}

__device__ __forceinline__ int cell_of_point(const KnnGridArgs& G, const float* __restrict__ p, int64_t i) {
    const int cx = cell_coord(p[3 * i], G.lo[0], G.inv_cell, G.dim[0]);
    const int cy = cell_coord(p[3 * i + 1], G.lo[1], G.inv_cell, G.dim[1]);
    const int cz = cell_coord(p[3 * i + 2], G.lo[2], G.inv_cell, G.dim[2]);
    return int(cx + int64_t(G.dim[0]) * (cy + int64_t(G.dim[1]) * cz));
}

// place (nullable): (cell, place in it) of every point
__global__ void knn_count_kernel(const float* __restrict__ p, int64_t n, KnnGridArgs G,
                                 unsigned long long* __restrict__ counts, int2* __restrict__ place) {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    const int c = i < n ? cell_of_point(G, p, i) : -1;  // every lane takes part in the run detection
    if (place) {
        const int at = take_place(c, counts);
        if (i < n) place[i] = make_int2(c, at);
        return;
    }
    const int lane = threadIdx.x & 63;
    const uint64_t starts = run_starts(c);
    if (c >= 0 && ((starts >> lane) & 1ull)) atomicAdd(&counts[c], (unsigned long long)run_length(starts, lane));
}

__global__ void knn_scatter_kernel(const float* __restrict__ p, int64_t n, const int2* __restrict__ place,
                                   const int64_t* __restrict__ cell_start, float4* __restrict__ out) {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int2 c = place[i];
    out[cell_start[c.x] + c.y] = make_float4(p[3 * i], p[3 * i + 1], p[3 * i + 2], __int_as_float(int(i)));
}

__global__ __launch_bounds__(256) void bounds_kernel(const float* __restrict__ p, int64_t n, float* __restrict__ partial) {
    __shared__ float lds[6][256];
    float mn[3] = {INFINITY, INFINITY, INFINITY}, mx[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < n; i += int64_t(gridDim.x) * 256)
        for (int d = 0; d < 3; ++d) {
            mn[d] = fminf(mn[d], p[3 * i + d]);
            mx[d] = fmaxf(mx[d], p[3 * i + d]);
        }
    for (int d = 0; d < 3; ++d) {
        lds[d][threadIdx.x] = mn[d];
        lds[3 + d][threadIdx.x] = mx[d];
    }
    __syncthreads();
    for (int off = 128; off > 0; off >>= 1) {
        if (threadIdx.x < off)
            for (int d = 0; d < 3; ++d) {
                lds[d][threadIdx.x] = fminf(lds[d][threadIdx.x], lds[d][threadIdx.x + off]);
                lds[3 + d][threadIdx.x] = fmaxf(lds[3 + d][threadIdx.x], lds[3 + d][threadIdx.x + off]);
            }
        __syncthreads();
    }
    if (threadIdx.x < 6) partial[6 * blockIdx.x + threadIdx.x] = lds[threadIdx.x][0];
}

void bounds(dwg_ctx* ctx, const float* p, int64_t n, float* lo, float* hi) {
    DWG_REQUIRE(n > 0, "bounds of an empty point set");
    const int blocks = 256;
    float* partial = static_cast<float*>(ctx->buf("bounds_partial", sizeof(float) * 6 * blocks));
    hipLaunchKernelGGL(bounds_kernel, dim3(blocks), dim3(256), 0, ctx->stream, p, n, partial);
    check_launch();
    std::vector<float> h(6 * blocks);
    DWG_HIP_CHECK(hipMemcpyAsync(h.data(), partial, sizeof(float) * 6 * blocks, hipMemcpyDeviceToHost, ctx->stream));
    DWG_HIP_CHECK(hipStreamSynchronize(ctx->stream));
    for (int d = 0; d < 3; ++d) {
        lo[d] = INFINITY;
        hi[d] = -INFINITY;
    }
    for (int b = 0; b < blocks; ++b)
        for (int d = 0; d < 3; ++d) {
            lo[d] = std::min(lo[d], h[6 * b + d]);
            hi[d] = std::max(hi[d], h[6 * b + 3 + d]);
        }
}

__global__ void count_occupied_kernel(const int64_t* __restrict__ counts, int64_t nc,
                                      unsigned long long* __restrict__ out) {
    __shared__ int lds[256];
    int c = 0;
    for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < nc; i += int64_t(gridDim.x) * 256) c += counts[i] != 0;
    lds[threadIdx.x] = c;
    __syncthreads();
    for (int off = 128; off > 0; off >>= 1) {
        if (threadIdx.x < off) lds[threadIdx.x] += lds[threadIdx.x + off];
        __syncthreads();
    }
    if (threadIdx.x == 0) atomicAdd(out, (unsigned long long)lds[0]);
}

static KnnGridArgs grid_args(const float* lo, const float* hi, double cell) {
    KnnGridArgs G{};
    G.cell = float(cell);
    G.inv_cell = float(1.0 / cell);
    for (int d = 0; d < 3; ++d) {
        G.lo[d] = lo[d];
        G.dim[d] = std::max(1, int(std::floor((hi[d] - lo[d]) / cell)) + 1);
    }
    return G;
}

static double cells_of(const float* lo, const float* hi, double cell) {
    double nc = 1;
    for (int d = 0; d < 3; ++d) nc *= std::floor((hi[d] - lo[d]) / cell) + 1;
    return nc;
}

// histogram + scan + scatter of the points into level L; without `scatter`
// only the histogram
static void bucket(dwg_ctx* ctx, const float* p, int64_t n, dwg_knn_index::Level& L, bool scatter) {
    L.ncells = int64_t(L.G.dim[0]) * L.G.dim[1] * L.G.dim[2];
    dwg::dev_free(L.cell_start);
    L.cell_start = nullptr;
    L.cell_start = static_cast<decltype(L.cell_start)>(dev_malloc(sizeof(int64_t) * (L.ncells + 1)));
    int2* place = scatter ? static_cast<int2*>(ctx->buf("knn_place", sizeof(int2) * n)) : nullptr;
    fill_u32(ctx, L.cell_start, 0, 2 * (L.ncells + 1));
    hipLaunchKernelGGL(knn_count_kernel, dim3(grid_for(n, 256)), dim3(256), 0, ctx->stream, p, n, L.G,
                       reinterpret_cast<unsigned long long*>(L.cell_start), place);
    check_launch();
    if (!scatter) return;
    exclusive_scan<int64_t>(ctx, L.cell_start, L.ncells);
    L.pts = static_cast<decltype(L.pts)>(dev_malloc(sizeof(float4) * n));
    hipLaunchKernelGGL(knn_scatter_kernel, dim3(grid_for(n, 256)), dim3(256), 0, ctx->stream, p, n, place, L.cell_start,
                       L.pts);
    check_launch();
}

// Chebyshev distance (in cells) from every cell to the nearest occupied one,
// as three separable passes: along x the distance to the nearest occupied
// cell of the row, then d(y) = min_y' max(|y − y'|, d_prev(y')) along y and z.
__global__ void empty_dist_x_kernel(const int64_t* __restrict__ cell_start, int dx, int dy, int dz,
                                    int* __restrict__ out) {
    const int64_t c = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (c >= int64_t(dx) * dy * dz) return;
    const int x = int(c % dx);
    const int64_t row = c - x;
    int best = 1 << 28;
    for (int x2 = 0; x2 < dx; ++x2)
        if (cell_start[row + x2 + 1] > cell_start[row + x2]) best = min(best, abs(x2 - x));
    out[c] = best;
}

__global__ void empty_dist_pass_kernel(const int* __restrict__ in, int dx, int dy, int dz, int axis,
                                       int* __restrict__ out) {
    const int64_t c = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (c >= int64_t(dx) * dy * dz) return;
    const int x = int(c % dx), y = int((c / dx) % dy), z = int(c / (int64_t(dx) * dy));
    const int len = axis == 1 ? dy : dz, pos = axis == 1 ? y : z;
    const int64_t stride = axis == 1 ? int64_t(dx) : int64_t(dx) * dy;
    const int64_t base = c - int64_t(pos) * stride;
    int best = 1 << 28;
    for (int t = 0; t < len; ++t) best = min(best, max(abs(t - pos), in[base + int64_t(t) * stride]));
    out[c] = best;
    (void)x;
}

static void empty_distance(dwg_ctx* ctx, dwg_knn_index::Level& L) {
    const int dx = L.G.dim[0], dy = L.G.dim[1], dz = L.G.dim[2];
    L.empty = static_cast<decltype(L.empty)>(dev_malloc(sizeof(int) * L.ncells));
    int* tmp = static_cast<int*>(ctx->buf("knn_empty_tmp", sizeof(int) * L.ncells));
    const unsigned g = grid_for(L.ncells, 256);
    hipLaunchKernelGGL(empty_dist_x_kernel, dim3(g), dim3(256), 0, ctx->stream, L.cell_start, dx, dy, dz, L.empty);
    check_launch();
    hipLaunchKernelGGL(empty_dist_pass_kernel, dim3(g), dim3(256), 0, ctx->stream, L.empty, dx, dy, dz, 1, tmp);
    check_launch();
    hipLaunchKernelGGL(empty_dist_pass_kernel, dim3(g), dim3(256), 0, ctx->stream, tmp, dx, dy, dz, 2, L.empty);
    check_launch();
}

// Occupancy pyramid of a level: byte b of level l ≥ 1 has bit c set when
// child c (x + 2y + 4z) of block b, at level l − 1, holds a point.
__global__ void pyr_first_kernel(const int64_t* __restrict__ cell_start, int dx, int dy, int dz, int ux, int uy, int uz,
                                 uint8_t* __restrict__ out) {
    const int64_t b = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (b >= int64_t(ux) * uy * uz) return;
    const int x = int(b % ux), y = int((b / ux) % uy), z = int(b / (int64_t(ux) * uy));
    uint32_t m = 0;
    for (int c = 0; c < 8; ++c) {
        const int X = 2 * x + (c & 1), Y = 2 * y + ((c >> 1) & 1), Z = 2 * z + (c >> 2);
        if (X < dx && Y < dy && Z < dz) {
            const int64_t cell = X + int64_t(dx) * (Y + int64_t(dy) * Z);
            if (cell_start[cell + 1] > cell_start[cell]) m |= 1u << c;
        }
    }
    out[b] = uint8_t(m);
}

__global__ void pyr_up_kernel(const uint8_t* __restrict__ lower, int dx, int dy, int dz, int ux, int uy, int uz,
                              uint8_t* __restrict__ out) {
    const int64_t b = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (b >= int64_t(ux) * uy * uz) return;
    const int x = int(b % ux), y = int((b / ux) % uy), z = int(b / (int64_t(ux) * uy));
    uint32_t m = 0;
    for (int c = 0; c < 8; ++c) {
        const int X = 2 * x + (c & 1), Y = 2 * y + ((c >> 1) & 1), Z = 2 * z + (c >> 2);
        if (X < dx && Y < dy && Z < dz && lower[X + int64_t(dx) * (Y + int64_t(dy) * Z)]) m |= 1u << c;
    }
    out[b] = uint8_t(m);
}

// Bounding boxes of the points themselves, per cell and per pyramid block:
// a query far from the cloud is as close to a box of a surface patch as to
// the patch, where the cell's own box can be a cell width nearer.  Exact
// bounds of float points need no rounding allowance: the box distance,
// computed like a point's d², never exceeds the d² of a point inside.
__global__ void cell_box_kernel(const int64_t* __restrict__ cell_start, const float4* __restrict__ pts, int64_t ncells,
                                float4* __restrict__ box) {
    const int64_t c = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (c >= ncells) return;
    float4 lo = make_float4(INFINITY, INFINITY, INFINITY, 0.f), hi = make_float4(-INFINITY, -INFINITY, -INFINITY, 0.f);
    for (int64_t s = cell_start[c], e = cell_start[c + 1]; s < e; ++s) {
        const float4 p = pts[s];
        lo.x = fminf(lo.x, p.x);
        lo.y = fminf(lo.y, p.y);
        lo.z = fminf(lo.z, p.z);
        hi.x = fmaxf(hi.x, p.x);
        hi.y = fmaxf(hi.y, p.y);
        hi.z = fmaxf(hi.z, p.z);
    }
    box[2 * c] = lo;
    box[2 * c + 1] = hi;
}

__global__ void box_up_kernel(const float4* __restrict__ lower, int dx, int dy, int dz, int ux, int uy, int uz,
                              float4* __restrict__ out) {
    const int64_t b = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (b >= int64_t(ux) * uy * uz) return;
    const int x = int(b % ux), y = int((b / ux) % uy), z = int(b / (int64_t(ux) * uy));
    float4 lo = make_float4(INFINITY, INFINITY, INFINITY, 0.f), hi = make_float4(-INFINITY, -INFINITY, -INFINITY, 0.f);
    for (int c = 0; c < 8; ++c) {
        const int X = 2 * x + (c & 1), Y = 2 * y + ((c >> 1) & 1), Z = 2 * z + (c >> 2);
        if (X < dx && Y < dy && Z < dz) {
            const int64_t i = X + int64_t(dx) * (Y + int64_t(dy) * Z);
            const float4 a = lower[2 * i], h = lower[2 * i + 1];
            lo.x = fminf(lo.x, a.x);
            lo.y = fminf(lo.y, a.y);
            lo.z = fminf(lo.z, a.z);
            hi.x = fmaxf(hi.x, h.x);
            hi.y = fmaxf(hi.y, h.y);
            hi.z = fmaxf(hi.z, h.z);
        }
    }
    out[2 * b] = lo;
    out[2 * b + 1] = hi;
}

// the points' bounding boxes of every cell and pyramid block, built the first
// time a walk needs them (only the wave-shared walk does).  One caller builds
// them, and waits until they are there: searches on other streams take them as
// soon as they see them
static const float4* ensure_boxes(dwg_ctx* ctx, dwg_knn_index::Level& L) {
    std::lock_guard<std::mutex> lock(L.building);
    if (const float4* there = L.pbox) return there;
    const int levels = L.pyr_levels;
    const int4* dims = L.pyr_dim_h;
    const int64_t* off = L.pyr_off_h;
    int64_t total = 0;
    for (int l = 1; l < levels; ++l) total += int64_t(dims[l].x) * dims[l].y * dims[l].z;
    DevBuf mem;
    float4* box = static_cast<float4*>(mem.ensure(sizeof(float4) * 2 * size_t(L.ncells + total)));
    hipLaunchKernelGGL(cell_box_kernel, dim3(grid_for(L.ncells, 256)), dim3(256), 0, ctx->stream, L.cell_start, L.pts,
                       L.ncells, box);
    check_launch();
    for (int l = 1; l < levels; ++l) {
        const int4 lo = dims[l - 1], up = dims[l];
        const int64_t nb = int64_t(up.x) * up.y * up.z;
        const float4* lower = box + 2 * (l == 1 ? 0 : L.ncells + off[l - 1]);
        hipLaunchKernelGGL(box_up_kernel, dim3(grid_for(nb, 256)), dim3(256), 0, ctx->stream, lower, lo.x, lo.y, lo.z,
                           up.x, up.y, up.z, box + 2 * (L.ncells + off[l]));
        check_launch();
    }
    DWG_HIP_CHECK(hipStreamSynchronize(ctx->stream));
    mem.ptr = nullptr;  // the index's from here on
    L.pbox = box;
    return box;
}

// cell boundaries are computed as lo + b·w in float and points are
// assigned by floor((v − lo)/cell): both are within a few ulp of the exact
// boundary, so a box of cells is shrunk by 16 ulp of the largest coordinate
// plus 1e-5 cell before it may exclude a point
static float cell_margin(const KnnGridArgs& G) {
    float ext = 0.f;
    for (int a = 0; a < 3; ++a)
        ext = std::max({ext, std::fabs(G.lo[a]), std::fabs(G.lo[a] + G.cell * float(G.dim[a]))});
    return 16.f * 1.1920929e-7f * ext + 1e-5f * G.cell;
}

// the first pyramid level counting only points that `skip` keeps
__global__ void pyr_first_masked_kernel(const int64_t* __restrict__ cell_start, const float4* __restrict__ pts,
                                        const uint8_t* __restrict__ skip, int dx, int dy, int dz, int ux, int uy,
                                        int uz, uint8_t* __restrict__ out) {
    const int64_t b = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (b >= int64_t(ux) * uy * uz) return;
    const int x = int(b % ux), y = int((b / ux) % uy), z = int(b / (int64_t(ux) * uy));
    uint32_t m = 0;
    for (int c = 0; c < 8; ++c) {
        const int X = 2 * x + (c & 1), Y = 2 * y + ((c >> 1) & 1), Z = 2 * z + (c >> 2);
        if (X < dx && Y < dy && Z < dz) {
            const int64_t cell = X + int64_t(dx) * (Y + int64_t(dy) * Z);
            for (int64_t s = cell_start[cell], e = cell_start[cell + 1]; s < e; ++s)
                if (!skip[__float_as_int(pts[s].w)]) {
                    m |= 1u << c;
                    break;
                }
        }
    }
    out[b] = uint8_t(m);
}

// An occupancy pyramid of the fine level that ignores the points `skip`
// drops (same layout as Level::pyr, in a context buffer): a walk with that
// skip mask then never opens a block of skipped points only
static const uint8_t* masked_pyramid(dwg_ctx* ctx, const dwg_knn_index::Level& L, const uint8_t* skip) {
    const int levels = L.pyr_levels;
    const int4* dims = L.pyr_dim_h;
    const int64_t* off = L.pyr_off_h;
    int64_t total = 0;
    for (int l = 1; l < levels; ++l) total += int64_t(dims[l].x) * dims[l].y * dims[l].z;
    uint8_t* pyr = static_cast<uint8_t*>(ctx->buf("knn_pyr_masked", size_t(total) + 64));
    for (int l = 1; l < levels; ++l) {
        const int4 lo = dims[l - 1], up = dims[l];
        const int64_t nb = int64_t(up.x) * up.y * up.z;
        if (l == 1)
            hipLaunchKernelGGL(pyr_first_masked_kernel, dim3(grid_for(nb, 256)), dim3(256), 0, ctx->stream,
                               L.cell_start, L.pts, skip, lo.x, lo.y, lo.z, up.x, up.y, up.z, pyr + off[1]);
        else
            hipLaunchKernelGGL(pyr_up_kernel, dim3(grid_for(nb, 256)), dim3(256), 0, ctx->stream, pyr + off[l - 1],
                               lo.x, lo.y, lo.z, up.x, up.y, up.z, pyr + off[l]);
        check_launch();
    }
    return pyr;
}

static void pyramid(dwg_ctx* ctx, dwg_knn_index::Level& L) {
    int4* dims = L.pyr_dim_h;
    int64_t* off = L.pyr_off_h;
    int d[3] = {L.G.dim[0], L.G.dim[1], L.G.dim[2]};
    dims[0] = make_int4(d[0], d[1], d[2], 0);
    off[0] = 0;
    int levels = 1;
    int64_t total = 0;
    while (d[0] > 1 || d[1] > 1 || d[2] > 1) {
        if (levels == kMaxPyr) return;  // no pyramid: queries take the shell search
        for (int a = 0; a < 3; ++a) d[a] = (d[a] + 1) / 2;
        dims[levels] = make_int4(d[0], d[1], d[2], 0);
        off[levels] = total;
        total += int64_t(d[0]) * d[1] * d[2];
        ++levels;
    }
    if (levels == 1) return;  // one cell: the shell search is already optimal
    L.pyr = static_cast<decltype(L.pyr)>(dev_malloc(size_t(total)));
    L.pyr_dim = static_cast<decltype(L.pyr_dim)>(dev_malloc(sizeof(int4) * kMaxPyr));
    L.pyr_off = static_cast<decltype(L.pyr_off)>(dev_malloc(sizeof(int64_t) * kMaxPyr));
    DWG_HIP_CHECK(hipMemcpyAsync(L.pyr_dim, dims, sizeof(int4) * levels, hipMemcpyHostToDevice, ctx->stream));
    DWG_HIP_CHECK(hipMemcpyAsync(L.pyr_off, off, sizeof(int64_t) * levels, hipMemcpyHostToDevice, ctx->stream));
    for (int l = 1; l < levels; ++l) {
        const int4 lo = dims[l - 1], up = dims[l];
        const int64_t nb = int64_t(up.x) * up.y * up.z;
        if (l == 1)
            hipLaunchKernelGGL(pyr_first_kernel, dim3(grid_for(nb, 256)), dim3(256), 0, ctx->stream, L.cell_start, lo.x,
                               lo.y, lo.z, up.x, up.y, up.z, L.pyr + off[1]);
        else
            hipLaunchKernelGGL(pyr_up_kernel, dim3(grid_for(nb, 256)), dim3(256), 0, ctx->stream, L.pyr + off[l - 1],
                               lo.x, lo.y, lo.z, up.x, up.y, up.z, L.pyr + off[l]);
        check_launch();
    }
    L.pyr_margin = cell_margin(L.G);
    L.pyr_levels = levels;
}

dwg_knn_index* knn_build(dwg_ctx* ctx, const float* p, int64_t n, int k_hint) {
    DWG_REQUIRE(n > 0 && n < (int64_t(1) << 31) - 1, "kNN index needs 1 ≤ n < 2^31 points");
    float lo[3], hi[3];
    bounds(ctx, p, n, lo, hi);
    auto* I = new dwg_knn_index();
    try {
        I->n = n;
        ProfileScope ps(ctx, "knn_build");
        const double ext = std::max({double(hi[0] - lo[0]), double(hi[1] - lo[1]), double(hi[2] - lo[2]), 1e-6});
        const double max_cells = double(1 << 27);
        // about `target` points per occupied cell puts ~k points in the 3×3×3
        // block around a query on a surface-like cloud
        const double target = std::max(2.0, 0.3 * double(std::max(k_hint, 1)));
        double cell = ext / std::max(1.0, std::sqrt(double(n) / target));
        while (cells_of(lo, hi, cell) > max_cells) cell *= 1.25;
        // measure the occupancy at this cell size and rescale (occupancy of a
        // surface-like cloud grows with cell²)
        dwg_knn_index::Level probe;
        probe.G = grid_args(lo, hi, cell);
        bucket(ctx, p, n, probe, false);
        unsigned long long* occ = static_cast<unsigned long long*>(ctx->buf("knn_occ", sizeof(uint64_t)));
        fill_u32(ctx, occ, 0, 2);
        hipLaunchKernelGGL(count_occupied_kernel, dim3(512), dim3(256), 0, ctx->stream, probe.cell_start, probe.ncells,
                           occ);
        check_launch();
        const double occupied = double(std::max<unsigned long long>(1, read_scalar<unsigned long long>(ctx, occ)));
        dev_free(probe.cell_start);
        probe.cell_start = nullptr;
        const double o = double(n) / occupied;
        double scale = std::sqrt(target / o);
        scale = std::min(16.0, std::max(0.25, scale));
        cell *= scale;
        while (cells_of(lo, hi, cell) > max_cells) cell *= 1.25;
        I->lvl[0].G = grid_args(lo, hi, cell);
        bucket(ctx, p, n, I->lvl[0], true);
        pyramid(ctx, I->lvl[0]);
        if (I->lvl[0].pyr_levels < 2) {  // its queries take the coarse level's shells
            I->lvl[1].G = grid_args(lo, hi, cell * 8.0);
            bucket(ctx, p, n, I->lvl[1], true);
            empty_distance(ctx, I->lvl[1]);
        }
    } catch (...) {
        delete I;
        throw;
    }
    return I;
}

// The k best keys of a query live in registers as a descending list:
// best[0] is the k-th smallest key so far (the insertion threshold), the
// slots k..K−1 hold 0 and never move (every key is ≥ 0).  Every access uses
// a constant index, so the list is never demoted to scratch memory.
// An empty slot: above every key with a d² up to ∞ (the high word of a key is the
// float bits of its d²) and below those of a d² that is no number, so that a point
// or a query with a NaN has no neighbours and is none
constexpr uint64_t kNoKey = 0x7F800000FFFFFFFFull;

template <int K>
__device__ __forceinline__ void knn_reset(uint64_t (&best)[K], int k) {
#pragma unroll
    for (int j = 0; j < K; ++j) best[j] = j < k ? kNoKey : 0ull;
}

// The key takes its place in the list and the largest key leaves it (the key
// itself, if it is not below that).  Every key (and kNoKey, and the 0 of an
// unused slot) read as a double is a non-negative number, never NaN, and
// non-negative doubles order as their bit patterns do (the kernels keep FP64
// denormals): slot i takes max(min(key, slot i), slot i + 1), one FP64 min and
// one max which return one of their operands bit for bit.  Both in place, so
// no slot waits for another and no register is copied; written as the
// instructions themselves, as the compiler would first quiet possible
// signalling NaNs of the operands, which these keys never are.
template <int K>
__device__ __forceinline__ void knn_insert(uint64_t (&best)[K], uint64_t key) {
#pragma unroll
    for (int i = 0; i + 1 < K; ++i)
        asm("v_min_f64 %0, %1, %0\n\tv_max_f64 %0, %0, %2" : "+&v"(best[i]) : "v"(key), "v"(best[i + 1]));
    asm("v_min_f64 %0, %1, %0" : "+v"(best[K - 1]) : "v"(key));
}

// writes the k keys in ascending order (index −1 / d² ∞ where fewer were found)
template <int K>
__device__ __forceinline__ void knn_store(const uint64_t (&best)[K], int k, int64_t row, int32_t* __restrict__ out_idx,
                                          float* __restrict__ out_d2) {
#pragma unroll
    for (int j = 0; j < K; ++j) {
        if (j < k) {
            const uint64_t b = best[j];
            const int64_t o = row * k + (k - 1 - j);
            out_idx[o] = b == kNoKey ? -1 : int32_t(uint32_t(b));
            if (out_d2) out_d2[o] = b == kNoKey ? INFINITY : __uint_as_float(uint32_t(b >> 32));
        }
    }
}

// ---------------------------------------------------------------------------
// Tiled queries.  Queries are bucketed by tile (kTile³ fine cells); one
// workgroup per non-empty tile stages the points of the tile plus a kHalo
// ring of cells in LDS and every lane (one query each) scans the same
// candidates in lockstep, so LDS reads are broadcasts and no lane diverges.
// A query is final when its k-th key is closer than every face of the
// staged box that is not on the grid boundary; the rest (sparse or clustered
// regions) walk the pyramid.  All paths keep the k smallest (d², index) keys,
// so the result does not depend on the path.
// ---------------------------------------------------------------------------
constexpr double kScatterFix = 1099511627776.0;  // 2^40
constexpr int kTile = 4;
constexpr int kStage = 512;
constexpr int kTileThreads = 256;
// The candidates are tested kBatch at a time: half of the batches hold nothing
// for any lane of a wave, which one compare then tells.  Of 300 candidates a
// wave takes in about 100, as the union of its lanes' neighbours alone has 75:
// these insertions and the distances bound the pass (3M centroids over 1M
// points, 15 neighbours: 1.29 → 1.13 ms; 300,000 points, 17: 0.151 → 0.120).
// Sorting a batch to join it at once spills (1.38 ms); boxes around the
// batches, also with the nearest first, cost what they save.
constexpr int kBatch = 16;
static_assert(kStage % kBatch == 0 && kTileThreads >= kBatch, "whole batches, filled up by one thread a place");
// most queries close within 2 cells of their tile.  Wider passes for the
// others (5 and 9 cells) cost more than walking the pyramid at once: 200,000
// queries over 1M points, half of them off the surface, 5.6 → 3.4 ms
constexpr int kHalo = 2;
// the tiled passes bucket their queries by 2×2×2-cell eighth of the tile
// (8 buckets per tile), so that the 64 queries of a wave sit close together
// (first pass 2.07 → 1.97 ms, and the far walk that takes its open queries
// in this order 1.89 → 1.81 ms)
constexpr int kSubTiled = 8;

// exclusive sum over the block's threads (NT threads, a multiple of 64);
// every thread calls it; wsum holds NT / 64 ints of LDS
template <int NT>
__device__ __forceinline__ int block_exclusive_sum(int v, int* wsum) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int incl = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int y = __shfl_up(incl, off, 64);
        if (lane >= off) incl += y;
    }
    if (lane == 63) wsum[w] = incl;
    __syncthreads();
    int before = 0;
#pragma unroll
    for (int i = 0; i < NT / 64; ++i) before += i < w ? wsum[i] : 0;
    return before + incl - v;
}

struct TileArgs {
    int tdim[3];  // tiles per axis
};

// bucket of a point: its tile, times 8, plus the eighth of the tile it lies in
__device__ __forceinline__ int bucket_of_point(const KnnGridArgs& G, const TileArgs& T, float x, float y, float z) {
    const int cx = cell_coord(x, G.lo[0], G.inv_cell, G.dim[0]);
    const int cy = cell_coord(y, G.lo[1], G.inv_cell, G.dim[1]);
    const int cz = cell_coord(z, G.lo[2], G.inv_cell, G.dim[2]);
    const int tile = cx / kTile + T.tdim[0] * (cy / kTile + T.tdim[1] * (cz / kTile));
    constexpr int h = kTile / 2;
    return tile * kSubTiled + int(cx % kTile >= h) + 2 * int(cy % kTile >= h) + 4 * int(cz % kTile >= h);
}

// masked queries are left out
__global__ void tile_count_kernel(const float* __restrict__ q, int64_t nq, const uint8_t* __restrict__ qmask, KnnGridArgs G, TileArgs T,
                                  int2* __restrict__ place, unsigned long long* __restrict__ count) {
    const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    int tl = -1;  // every lane takes part in the run detection
    if (t < nq && (!qmask || qmask[t])) tl = bucket_of_point(G, T, q[3 * t], q[3 * t + 1], q[3 * t + 2]);
    const int at = take_place(tl, count);
    if (t < nq) place[t] = make_int2(tl, at);
}

__global__ void tile_scatter_kernel(const int2* __restrict__ place, int64_t nq, const int64_t* __restrict__ start,
                                    int* __restrict__ order) {
    const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= nq) return;
    const int2 b = place[t];
    if (b.x >= 0) order[start[b.x] + b.y] = int(t);
}

// The blocks that the tiles' queries take, `chunk` each, listed by (tile,
// chunk): a block's tiles take their places with one atomic add, so the list
// is in order but for the order of the blocks, on which no result depends.
constexpr int kListThreads = 1024;
__global__ __launch_bounds__(kListThreads) void tile_list_kernel(const int64_t* __restrict__ start, int64_t ntiles,
                                                                 int chunk, int2* __restrict__ list,
                                                                 unsigned long long* __restrict__ nlist) {
    __shared__ int s_wsum[kListThreads / 64];
    __shared__ int s_first;
    const int64_t t = int64_t(blockIdx.x) * kListThreads + threadIdx.x;
    const int64_t len = t < ntiles ? start[kSubTiled * (t + 1)] - start[kSubTiled * t] : 0;
    const int blocks = int((len + chunk - 1) / chunk);
    const int before = block_exclusive_sum<kListThreads>(blocks, s_wsum);
    if (threadIdx.x == kListThreads - 1)
        s_first = before + blocks > 0 ? int(atomicAdd(nlist, (unsigned long long)(before + blocks))) : 0;
    __syncthreads();
    for (int c = 0; c < blocks; ++c) list[s_first + before + c] = make_int2(int(t), c);
}

// Staged candidates are ordered by ring: the rows of cells that cross the
// tile first, then the halo rings outwards, so a query meets its nearest
// points early and its k-th key (the insertion threshold) tightens fast.
// SCATTER: besides its neighbours, every closed query adds its value
// (3 floats) in 2^-40 fixed point into acc[neighbour] — the normal scatter
// of the diffusion (TurboDWG.cu:179-204).  The tile gathers these sums in an
// LDS hash table keyed by point index and flushes each key once with 64-bit
// global atomics; integer sums are associative, so the result equals
// per-pair atomics bit for bit.
template <int K, bool SCATTER>
__global__ __launch_bounds__(kTileThreads, K <= 17 ? 4 : 2) void knn_tile_kernel(
    KnnGridArgs G, TileArgs T, const int64_t* __restrict__ cell_start, const float4* __restrict__ pts,
    const int2* __restrict__ tiles, int chunk, const int64_t* __restrict__ tile_start, const int* __restrict__ order,
    const float* __restrict__ q, int k, const uint8_t* __restrict__ skip, int32_t* __restrict__ out_idx,
    float* __restrict__ out_d2, int* __restrict__ redo, float* __restrict__ redo_kth,
    unsigned long long* __restrict__ nredo, int64_t* __restrict__ tile_open, const int64_t* __restrict__ ntiles,
    KnnScatter sc) {
    if (ntiles && int64_t(blockIdx.x) >= *ntiles) {  // launched for the most tiles there can be
        if (tile_open && threadIdx.x == 0) tile_open[blockIdx.x] = 0;
        return;
    }
    constexpr int kRegion = kTile + 2 * kHalo;
    // each row is split into the tile's own cells and the halo cells at x
    // distance 1 and 2 on either side, so that the staging order (by
    // Chebyshev ring from the tile) starts with the tile's own cells
    constexpr int kParts = 5;
    constexpr int kRows = kRegion * kRegion * kParts;
    constexpr int kHash = SCATTER ? 256 : 1;
    __shared__ int s_hkey[kHash];
    __shared__ unsigned long long s_hacc[kHash][3];
    if (SCATTER) {
        for (int h = threadIdx.x; h < kHash; h += kTileThreads) {
            s_hkey[h] = -1;
            s_hacc[h][0] = s_hacc[h][1] = s_hacc[h][2] = 0ull;
        }
    }
    __shared__ float4 s_pts[kStage];
    __shared__ int s_rb[kRows];
    __shared__ int s_pref[kRows + 1];  // the rows' point counts, then their exclusive prefix
    __shared__ int s_wsum[kTileThreads / 64];
    __shared__ int s_ring[kHalo + 2];
    __shared__ int s_open;
    if (threadIdx.x == 0) s_open = 0;
    const int tile = tiles[blockIdx.x].x;
    const int tx = tile % T.tdim[0], ty = (tile / T.tdim[0]) % T.tdim[1], tz = tile / (T.tdim[0] * T.tdim[1]);
    const int x0 = max(tx * kTile - kHalo, 0), x1 = min(tx * kTile + kTile - 1 + kHalo, G.dim[0] - 1);
    const int y0 = max(ty * kTile - kHalo, 0), y1 = min(ty * kTile + kTile - 1 + kHalo, G.dim[1] - 1);
    const int z0 = max(tz * kTile - kHalo, 0), z1 = min(tz * kTile + kTile - 1 + kHalo, G.dim[2] - 1);
    const int ny = y1 - y0 + 1, nrows = ny * (z1 - z0 + 1) * kParts;
    if (threadIdx.x < kHalo + 2) s_ring[threadIdx.x] = 0;
    __syncthreads();
    // each (y, z) row of cells x0..x1 (or each of its parts) is one
    // contiguous range of points; a thread takes rows threadIdx.x +
    // h · kTileThreads, h < kRowIters
    constexpr int kRowIters = (kRows + kTileThreads - 1) / kTileThreads;
    int ring[kRowIters], rank[kRowIters], rc[kRowIters];
    int rb[kRowIters];
#pragma unroll
    for (int h = 0; h < kRowIters; ++h) {
        ring[h] = rank[h] = rc[h] = 0;
        rb[h] = 0;
        const int r = threadIdx.x + h * kTileThreads;
        if (r < nrows) {
            const int row = r / kParts, part = r % kParts;
            const int y = y0 + row % ny, z = z0 + row / ny;
            // the part's cells xa..xb and their x distance from the tile
            int xa, xb, dx = 0;
            const int t0 = tx * kTile, t1 = tx * kTile + kTile - 1;
            if (part == 0) { xa = t0; xb = t1; }
            else if (part <= 2) { xa = xb = t0 - part; dx = part; }
            else { xa = xb = t1 + (part - 2); dx = part - 2; }
            xa = max(xa, x0);
            xb = min(xb, x1);
            const int64_t c = xa + int64_t(G.dim[0]) * (y + int64_t(G.dim[1]) * z);
            rb[h] = int(cell_start[c]);  // an index holds fewer than 2^31 points
            rc[h] = xb >= xa ? int(cell_start[c + (xb - xa) + 1]) - rb[h] : 0;
            const int dy = max(max(ty * kTile - y, y - (ty * kTile + kTile - 1)), 0);
            const int dz = max(max(tz * kTile - z, z - (tz * kTile + kTile - 1)), 0);
            ring[h] = max(max(dy, dz), dx);
            rank[h] = atomicAdd(&s_ring[ring[h] + 1], 1);
        }
    }
    __syncthreads();
    if (threadIdx.x == 0)
        for (int r = 1; r <= kHalo + 1; ++r) s_ring[r] += s_ring[r - 1];
    __syncthreads();
#pragma unroll
    for (int h = 0; h < kRowIters; ++h) {
        if (threadIdx.x + h * kTileThreads < nrows) {
            const int pos = s_ring[ring[h]] + rank[h];
            s_rb[pos] = rb[h];
            s_pref[pos] = rc[h];
        }
    }
    __syncthreads();
    {
        // s_pref: exclusive prefix of the rows' point counts, thread t
        // owning rows kRowIters·t .. kRowIters·t + kRowIters − 1
        int loc[kRowIters], sum = 0;
#pragma unroll
        for (int i = 0; i < kRowIters; ++i) {
            const int r = threadIdx.x * kRowIters + i;
            loc[i] = r < nrows ? s_pref[r] : 0;
            sum += loc[i];
        }
        int run = block_exclusive_sum<kTileThreads>(sum, s_wsum);
#pragma unroll
        for (int i = 0; i < kRowIters; ++i) {
            const int r = threadIdx.x * kRowIters + i;
            if (r <= nrows) s_pref[r] = run;
            run += loc[i];
        }
        if (threadIdx.x == kTileThreads - 1) s_pref[nrows] = run;  // the total, also when nrows fills every slot
    }
    __syncthreads();
    const int total = s_pref[nrows];
    // faces of the staged box that are not on the grid boundary
    const float flx = x0 > 0 ? G.lo[0] + float(x0) * G.cell : -INFINITY;
    const float fhx = x1 + 1 < G.dim[0] ? G.lo[0] + float(x1 + 1) * G.cell : INFINITY;
    const float fly = y0 > 0 ? G.lo[1] + float(y0) * G.cell : -INFINITY;
    const float fhy = y1 + 1 < G.dim[1] ? G.lo[1] + float(y1 + 1) * G.cell : INFINITY;
    const float flz = z0 > 0 ? G.lo[2] + float(z0) * G.cell : -INFINITY;
    const float fhz = z1 + 1 < G.dim[2] ? G.lo[2] + float(z1 + 1) * G.cell : INFINITY;
    const int64_t qs = tile_start[int64_t(tile) * kSubTiled] + int64_t(tiles[blockIdx.x].y) * chunk;
    const int64_t qe = min(tile_start[int64_t(tile + 1) * kSubTiled], qs + chunk);
    // one staging serves all queries: the waves left over leave after it (a
    // barrier waits for the waves that are there).  Half of them are, with 105
    // queries a tile, and held the places of others (1.13 → 1.07 ms for 3M
    // centroids)
    const bool once = total <= kStage && qe - qs <= kTileThreads;
    const int stay = once ? int(qe - qs + 63) / 64 * 64 : kTileThreads;
    for (int64_t qb = qs; qb < qe; qb += kTileThreads) {
        const int64_t t = qb + threadIdx.x;
        const bool active = t < qe;
        const int qi = active ? order[t] : 0;
        // (a lane without a query is at no distance from anything)
        const float qx = active ? q[3 * int64_t(qi)] : NAN, qy = active ? q[3 * int64_t(qi) + 1] : NAN,
                    qz = active ? q[3 * int64_t(qi) + 2] : NAN;
        uint64_t best[K];
        const uint64_t has = __builtin_amdgcn_ballot_w64(active);
        knn_reset<K>(best, k);
        auto kth = [&]() { return __uint_as_float(uint32_t(best[0] >> 32)); };  // the k-th d², or ∞
        for (int cb = 0; cb < total; cb += kStage) {
            const int cnt = min(kStage, total - cb);
            __syncthreads();
            for (int j = threadIdx.x; j < cnt; j += kTileThreads) {
                const int g = cb + j;
                int lo = 0, hi = nrows - 1;  // last row with s_pref[row] <= g
                while (lo < hi) {
                    const int mid = (lo + hi + 1) >> 1;
                    if (s_pref[mid] <= g) lo = mid;
                    else hi = mid - 1;
                }
                float4 p = pts[s_rb[lo] + (g - s_pref[lo])];
                if (skip && skip[__float_as_int(p.w)]) p.x = NAN;  // at no distance
                s_pts[j] = p;
            }
            const int padded = (cnt + kBatch - 1) / kBatch * kBatch;
            if (threadIdx.x < padded - cnt) s_pts[cnt + threadIdx.x] = make_float4(NAN, 0.f, 0.f, 0.f);
            __syncthreads();
            // a wave without queries is done where nothing is staged after this
            if (!has && once) return;
            for (int j = 0; j < (has ? padded : 0); j += kBatch) {
                float d2[kBatch], least = NAN;  // no number for a lane without a query
#pragma unroll
                for (int u = 0; u < kBatch; ++u) {
                    const float4 p = s_pts[j + u];
                    d2[u] = dist2(qx - p.x, qy - p.y, qz - p.z);
                    least = fminf(least, d2[u]);
                }
                if (!__builtin_amdgcn_ballot_w64(least <= kth())) continue;
#pragma unroll
                for (int u = 0; u < kBatch; ++u) {
                    const bool near = d2[u] <= kth();
                    if (!__builtin_amdgcn_ballot_w64(near)) continue;
                    knn_insert<K>(best, near ? (uint64_t(__float_as_uint(d2[u])) << 32) | __float_as_uint(s_pts[j + u].w)
                                             : kNoKey);
                }
            }
        }
        if (!active) continue;
        const float dmin = fminf(fminf(fminf(qx - flx, fhx - qx), fminf(qy - fly, fhy - qy)), fminf(qz - flz, fhz - qz));
        bool exact = dmin == INFINITY;
        if (!exact && best[0] != kNoKey) {
            const float safe = dmin * (1.0f - 1e-5f) - 1e-6f * G.cell;
            exact = safe > 0.f && kth() < safe * safe;
        }
        if (!exact) {
            // a wave lists its open queries side by side: with the tile's
            // others at the start of its range of places (tile_open), or after
            // those of any tile; the k candidates a query has bound its k-th
            // distance
            const uint64_t open = __builtin_amdgcn_ballot_w64(true);
            const int lane = threadIdx.x & 63, head = __builtin_ctzll(open);
            int at = 0;
            if (lane == head)
                at = tile_open ? int(qs) + atomicAdd(&s_open, __builtin_popcountll(open))
                               : int(atomicAdd(nredo, (unsigned long long)__builtin_popcountll(open)));
            at = __shfl(at, head, 64) + __builtin_popcountll(open & ((1ull << lane) - 1ull));
            redo[at] = qi;
            redo_kth[at] = kth();
            continue;
        }
        knn_store<K>(best, k, qi, out_idx, out_d2);
        if (SCATTER) {
            long long v[3];
#pragma unroll
            for (int d = 0; d < 3; ++d) v[d] = __double2ll_rn(double(sc.val[3 * int64_t(qi) + d]) * kScatterFix);
#pragma unroll
            for (int j = 0; j < K; ++j) {
                if (j >= k || best[j] == kNoKey) continue;
                const int idx = int(uint32_t(best[j]));
                int h = int((uint32_t(idx) * 0x9E3779B1u) >> 24);  // 8 bits
                bool done = false;
                for (int probe = 0; probe < 8 && !done; ++probe) {
                    const int prev = atomicCAS(&s_hkey[h], -1, idx);
                    if (prev == -1 || prev == idx) {
#pragma unroll
                        for (int d = 0; d < 3; ++d) atomicAdd(&s_hacc[h][d], (unsigned long long)v[d]);
                        done = true;
                    }
                    h = (h + 1) & (kHash - 1);
                }
                if (!done)
#pragma unroll
                    for (int d = 0; d < 3; ++d) atomicAdd(&sc.acc[3 * int64_t(idx) + d], (unsigned long long)v[d]);
            }
        }
    }
    if (SCATTER || tile_open) __syncthreads();
    if (tile_open && threadIdx.x == 0) tile_open[blockIdx.x] = s_open;
    if (SCATTER) {
        for (int h = threadIdx.x; h < kHash; h += stay) {
            const int key = s_hkey[h];
            if (key >= 0)
#pragma unroll
                for (int d = 0; d < 3; ++d) atomicAdd(&sc.acc[3 * int64_t(key) + d], s_hacc[h][d]);
        }
    }
}

// The open queries of the tiles, each tile's at the start of its range of
// places, one after the other in the list's order (pos: the scan of tile_open)
__global__ __launch_bounds__(64) void tile_open_kernel(const int2* __restrict__ tiles, int chunk,
                                                       const int64_t* __restrict__ tile_start,
                                                       const int64_t* __restrict__ pos, const int* __restrict__ tmp_q,
                                                       const float* __restrict__ tmp_kth, int* __restrict__ redo,
                                                       float* __restrict__ redo_kth) {
    const int64_t b = pos[blockIdx.x], n = pos[blockIdx.x + 1] - b;
    if (n == 0) return;
    const int2 e = tiles[blockIdx.x];
    const int64_t qs = tile_start[int64_t(e.x) * kSubTiled] + int64_t(e.y) * chunk;
    for (int64_t j = threadIdx.x; j < n; j += 64) {
        redo[b + j] = tmp_q[qs + j];
        redo_kth[b + j] = tmp_kth[qs + j];
    }
}

// acc[neighbour] += value of the query, for every query
__global__ void scatter_pairs_kernel(const int32_t* __restrict__ knn, int k, int64_t nq, KnnScatter sc) {
    const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= nq * k) return;
    const int64_t qi = t / k;
    const int32_t s = knn[qi * k + t % k];
    if (s < 0) return;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const long long v = __double2ll_rn(double(sc.val[3 * qi + d]) * kScatterFix);
        atomicAdd(&sc.acc[3 * int64_t(s) + d], (unsigned long long)v);
    }
}

// The same for 256 consecutive queries of qlist per block (qlist is in tile
// order, so they are neighbours and share most of their neighbours): the
// pairs are summed in an LDS hash keyed by point index and each key is
// flushed once with 64-bit global atomics (integer sums: bit for bit the
// per-pair result).
__global__ __launch_bounds__(256) void scatter_pairs_hashed_kernel(const int32_t* __restrict__ knn, int k,
                                                                   const int* __restrict__ qlist,
                                                                   const int64_t* __restrict__ count, KnnScatter sc) {
    const int64_t nq = *count;  // launched for every query
    if (int64_t(blockIdx.x) * 256 >= nq) return;
    constexpr int kHash = 1024;
    __shared__ int s_hkey[kHash];
    __shared__ unsigned long long s_hacc[kHash][3];
    for (int h = threadIdx.x; h < kHash; h += 256) {
        s_hkey[h] = -1;
        s_hacc[h][0] = s_hacc[h][1] = s_hacc[h][2] = 0ull;
    }
    __syncthreads();
    const int64_t t = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (t < nq) {
        const int64_t qi = qlist[t];
        long long v[3];
#pragma unroll
        for (int d = 0; d < 3; ++d) v[d] = __double2ll_rn(double(sc.val[3 * qi + d]) * kScatterFix);
        for (int j = 0; j < k; ++j) {
            const int32_t idx = knn[qi * k + j];
            if (idx < 0) continue;
            int h = int((uint32_t(idx) * 0x9E3779B1u) >> 22);  // 10 bits
            bool done = false;
            for (int probe = 0; probe < 8 && !done; ++probe) {
                const int prev = atomicCAS(&s_hkey[h], -1, idx);
                if (prev == -1 || prev == idx) {
#pragma unroll
                    for (int d = 0; d < 3; ++d) atomicAdd(&s_hacc[h][d], (unsigned long long)v[d]);
                    done = true;
                }
                h = (h + 1) & (kHash - 1);
            }
            if (!done)
#pragma unroll
                for (int d = 0; d < 3; ++d) atomicAdd(&sc.acc[3 * int64_t(idx) + d], (unsigned long long)v[d]);
        }
    }
    __syncthreads();
    for (int h = threadIdx.x; h < kHash; h += 256) {
        const int key = s_hkey[h];
        if (key >= 0)
#pragma unroll
            for (int d = 0; d < 3; ++d) atomicAdd(&sc.acc[3 * int64_t(key) + d], s_hacc[h][d]);
    }
}

__device__ __forceinline__ uint64_t shfl64(uint64_t v, int src) {
    const uint32_t lo = uint32_t(__shfl(int(uint32_t(v)), src, 64));
    const uint32_t hi = uint32_t(__shfl(int(uint32_t(v >> 32)), src, 64));
    return (uint64_t(hi) << 32) | lo;
}

__device__ __forceinline__ uint64_t wave_min_u64(uint64_t v) {
    for (int off = 32; off > 0; off >>= 1) {
        const uint64_t o = shfl64(v, (threadIdx.x & 63) ^ off);
        v = o < v ? o : v;
    }
    return v;
}

// One wave per query, for indices without a pyramid (a single cell, or a grid
// too elongated for one).  On the coarse level the cells of each Chebyshev shell are read 64 at a time, their
// points flattened and scanned 64 per step (one candidate per lane), each
// lane keeping its own k best keys.  The smallest lane-local k-th key bounds
// the wave's k-th key from above, so the search stops once it is closer than
// every cell not yet visited; k rounds of wave minima then merge the lists
// into the exact k smallest (d², index) keys.
// Cell offset of entry id of the Chebyshev shell of radius r, which has
// 24r² + 2 cells (one for r = 0): the two z faces, then the two y faces
// without their z rims, then the two x faces without either rim.
__device__ __forceinline__ int3 shell_cell(int id, int r) {
    if (r == 0) return make_int3(0, 0, 0);
    const int s = 2 * r + 1, t = 2 * r - 1, nz = s * s, ny = s * t;
    if (id < 2 * nz) {
        const int f = id / nz, rem = id - f * nz;
        return make_int3(rem % s - r, rem / s - r, f ? r : -r);
    }
    id -= 2 * nz;
    if (id < 2 * ny) {
        const int f = id / ny, rem = id - f * ny;
        return make_int3(rem % s - r, f ? r : -r, rem / s - (r - 1));
    }
    id -= 2 * ny;
    const int tt = t * t, f = id / tt, rem = id - f * tt;
    return make_int3(f ? r : -r, rem % t - (r - 1), rem / t - (r - 1));
}

template <int K>
__global__ __launch_bounds__(256) void knn_wave_kernel(KnnGridArgs G, const int64_t* __restrict__ cell_start,
                                                       const float4* __restrict__ pts, const int* __restrict__ empty,
                                                       const float* __restrict__ q, int64_t nq,
                                                       const int64_t* __restrict__ count,
                                                       const int* __restrict__ qlist, int k,
                                                       const uint8_t* __restrict__ skip,
                                                       const uint8_t* __restrict__ qmask, int32_t* __restrict__ out_idx,
                                                       float* __restrict__ out_d2) {
    const int lane = threadIdx.x & 63;
    const int64_t t = int64_t(blockIdx.x) * (blockDim.x >> 6) + (threadIdx.x >> 6);
    if (t >= (count ? *count : nq)) return;  // uniform per wave
    const int64_t i = qlist ? int64_t(qlist[t]) : t;
    if (qmask && !qmask[i]) return;
    const float qx = q[3 * i], qy = q[3 * i + 1], qz = q[3 * i + 2];
    uint64_t best[K];
    knn_reset<K>(best, k);
    const int c0x = cell_coord(qx, G.lo[0], G.inv_cell, G.dim[0]);
    const int c0y = cell_coord(qy, G.lo[1], G.inv_cell, G.dim[1]);
    const int c0z = cell_coord(qz, G.lo[2], G.inv_cell, G.dim[2]);
    const int maxr = max(G.dim[0], max(G.dim[1], G.dim[2]));
    int r = empty[c0x + int64_t(G.dim[0]) * (c0y + int64_t(G.dim[1]) * c0z)];
    for (; r <= maxr; ++r) {
        // only the shell's own cells: O(r²) per shell
        const int shell = r == 0 ? 1 : 24 * r * r + 2;
        for (int base = 0; base < shell; base += 64) {
            const int id = base + lane;
            int64_t b = 0;
            int cnt = 0;
            if (id < shell) {
                const int3 o = shell_cell(id, r);
                const int x = c0x + o.x, y = c0y + o.y, z = c0z + o.z;
                if (x >= 0 && y >= 0 && z >= 0 && x < G.dim[0] && y < G.dim[1] && z < G.dim[2]) {
                    const int64_t c = x + int64_t(G.dim[0]) * (y + int64_t(G.dim[1]) * z);
                    b = cell_start[c];
                    cnt = int(cell_start[c + 1] - b);
                }
            }
            // inclusive scan of the 64 cell sizes
            int incl = cnt;
            for (int off = 1; off < 64; off <<= 1) {
                const int v = __shfl_up(incl, off, 64);
                if (lane >= off) incl += v;
            }
            const int total = __shfl(incl, 63, 64);
            for (int cb = 0; cb < total; cb += 64) {
                const int j = cb + lane;
                // owner lane: the number of lanes whose inclusive count is ≤ j
                // (six uniform steps, every lane active for the shuffles)
                int lo = 0;
                for (int step = 32; step > 0; step >>= 1)
                    if (__shfl(incl, lo + step - 1, 64) <= j) lo += step;
                lo = min(lo, 63);
                const int64_t ob = shfl64(uint64_t(b), lo);
                const int oexcl = __shfl(incl - cnt, lo, 64);
                if (j < total) {
                    const float4 p = pts[ob + (j - oexcl)];
                    const int idx = __float_as_int(p.w);
                    if (!(skip && skip[idx])) {
                        const float d2 = dist2(qx - p.x, qy - p.y, qz - p.z);
                        const uint64_t key = (uint64_t(__float_as_uint(d2)) << 32) | uint32_t(idx);
                        if (key < best[0]) knn_insert<K>(best, key);
                    }
                }
            }
        }
        // no unvisited point is closer than the nearest face of the searched
        // block that is not on the grid boundary
        float dmin = INFINITY;
        if (c0x - r > 0) dmin = fminf(dmin, qx - (G.lo[0] + float(c0x - r) * G.cell));
        if (c0x + r + 1 < G.dim[0]) dmin = fminf(dmin, (G.lo[0] + float(c0x + r + 1) * G.cell) - qx);
        if (c0y - r > 0) dmin = fminf(dmin, qy - (G.lo[1] + float(c0y - r) * G.cell));
        if (c0y + r + 1 < G.dim[1]) dmin = fminf(dmin, (G.lo[1] + float(c0y + r + 1) * G.cell) - qy);
        if (c0z - r > 0) dmin = fminf(dmin, qz - (G.lo[2] + float(c0z - r) * G.cell));
        if (c0z + r + 1 < G.dim[2]) dmin = fminf(dmin, (G.lo[2] + float(c0z + r + 1) * G.cell) - qz);
        if (dmin == INFINITY) break;
        const uint64_t bound = wave_min_u64(best[0]);
        if (bound != kNoKey) {
            const float kd2 = __uint_as_float(uint32_t(bound >> 32));
            const float safe = dmin * (1.0f - 1e-5f) - 1e-6f * G.cell;
            if (safe > 0.f && kd2 < safe * safe) break;
        }
    }
    // merge: reverse each list to ascending order, drop the K−k zero slots
    // from its front, then the j-th smallest key is the wave minimum of the
    // lanes' heads (keys are distinct: one lane pops)
    uint64_t asc[K];
#pragma unroll
    for (int j = 0; j < K; ++j) asc[j] = best[K - 1 - j];
    for (int s = 0; s < K - k; ++s) {
#pragma unroll
        for (int c = 0; c < K - 1; ++c) asc[c] = asc[c + 1];
        asc[K - 1] = kNoKey;
    }
    for (int j = 0; j < k; ++j) {
        const uint64_t m = wave_min_u64(asc[0]);
        const uint64_t win = __ballot(asc[0] == m && m != kNoKey);
        if (win && lane == __ffsll((unsigned long long)win) - 1) {
#pragma unroll
            for (int c = 0; c < K - 1; ++c) asc[c] = asc[c + 1];
            asc[K - 1] = kNoKey;
        }
        if (lane == 0) {
            out_idx[i * k + j] = m == kNoKey ? -1 : int32_t(uint32_t(m));
            if (out_d2) out_d2[i * k + j] = m == kNoKey ? INFINITY : __uint_as_float(uint32_t(m >> 32));
        }
    }
}

// The occupancy pyramid of the fine level, as a walk reads it
struct PyrArgs {
    const uint8_t* mask;
    const int4* dim;
    const int64_t* off;
    int levels;
    float margin;
    const float4* box;  // the points' bounding boxes (dwg_knn_index::Level::pbox)
    int64_t ncells;
};

// squared distance from q to a box (lo, hi), computed like a point's d²
// (dist2): every step is monotone, so it never exceeds the d² of a point
// inside the box
__device__ __forceinline__ float tight_box_d2(const float4 lo, const float4 hi, float qx, float qy, float qz) {
    const float gx = fmaxf(fmaxf(lo.x - qx, qx - hi.x), 0.f);
    const float gy = fmaxf(fmaxf(lo.y - qy, qy - hi.y), 0.f);
    const float gz = fmaxf(fmaxf(lo.z - qz, qz - hi.z), 0.f);
    return dist2(gx, gy, gz);
}

// squared distance from q to the box of cells [b·2^l, (b+1)·2^l) along each
// axis, each axis gap shrunk by the rounding margin of the cells and, as the
// differences to the box's side and to a point on the wrong side of it by less
// than that margin may round apart by a unit in their last place (far larger
// than the margin for a far query), by four units of its own
__device__ __forceinline__ float pyr_box_d2(const KnnGridArgs& G, float w, float margin, float qx, float qy, float qz,
                                            int x, int y, int z) {
    auto gap = [&](float v, float lo, int b) {
        const float a = __builtin_fmaf(float(b), w, lo);
        return fmaxf(__builtin_fmaf(fmaxf(a - v, v - (a + w)), 1.f - 0x1p-22f, -margin), 0.f);
    };
    const float gx = gap(qx, G.lo[0], x), gy = gap(qy, G.lo[1], y), gz = gap(qz, G.lo[2], z);
    return __builtin_fmaf(gz, gz, __builtin_fmaf(gy, gy, gx * gx));
}

// One wave per query over the occupancy pyramid, for queries that are few or
// whose search is long: the lanes test the 8 children of up to 8 blocks in
// one step, and scan 64 points in one.  The k best keys lie in ascending
// order in lanes 0 .. k − 1 of one register pair, so the wave's exact k-th
// key bounds every step, with no list per lane to fill first, and few
// registers leave room for many waves.  Blocks wait on a stack in LDS with
// their box distance; until k points are known one block is opened a step,
// its nearest child on top, then 8.  Bound by the latency of a step (a child
// load, then a point load) where queries are few (1,500 over 100,000 points:
// 0.12 ms), by instructions where they fill the card.
// The stack never overflows: opening a block leaves at most 7 entries more
// than it took, a step takes several only while that leaves kDescReserve
// entries free, and a single depth-first descent needs no more than these.
constexpr int kDescWaves = 4;
constexpr int kDescStack = 320;
constexpr int kDescReserve = 7 * kMaxPyr + 8;
constexpr int kDescGreedy = 64;  // steps of one block at most while no k points are known
constexpr int kDescPoints = 8;   // points a cell hands out a round

template <int CTRL, int ROWS = 0xF>
__device__ __forceinline__ int dpp_or_zero(int v) {
    return __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xF, false);
}

// inclusive prefix sum over the wave
__device__ __forceinline__ int wave_scan_add(int v) {
    v += dpp_or_zero<0x111>(v);  // row_shr 1, 2, 4, 8: within rows of 16 lanes
    v += dpp_or_zero<0x112>(v);
    v += dpp_or_zero<0x114>(v);
    v += dpp_or_zero<0x118>(v);
    v += dpp_or_zero<0x142, 0xA>(v);  // row_bcast 15: rows 1 and 3 take the row before
    v += dpp_or_zero<0x143, 0xC>(v);  // row_bcast 31: the upper half takes lane 31
    return v;
}

// maximum over the wave
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
    v = max(v, uint32_t(dpp_or_zero<0x111>(int(v))));
    v = max(v, uint32_t(dpp_or_zero<0x112>(int(v))));
    v = max(v, uint32_t(dpp_or_zero<0x114>(int(v))));
    v = max(v, uint32_t(dpp_or_zero<0x118>(int(v))));
    v = max(v, uint32_t(dpp_or_zero<0x142, 0xA>(int(v))));
    v = max(v, uint32_t(dpp_or_zero<0x143, 0xC>(int(v))));
    return uint32_t(__builtin_amdgcn_readlane(int(v), 63));
}

__device__ __forceinline__ uint32_t read_lane(uint32_t v, int l) {
    return uint32_t(__builtin_amdgcn_readlane(int(v), l));
}
__device__ __forceinline__ uint64_t read_lane64(uint64_t v, int l) {
    return (uint64_t(read_lane(uint32_t(v >> 32), l)) << 32) | read_lane(uint32_t(v), l);
}

// The keys `key` of the lanes `cand` (all < kth) join the wave's best keys,
// ascending in the lanes 0 .. k − 1 of `list` (kNoKey where there is none), of
// which the least k stay; kth is the k-th then.  Up to kDescOneByOne keys enter
// one after the other, each shifting the list.  Where there are more, a
// bisection finds a bound with k keys below it, in the bits of the squared
// distance and, if several points lie at the k-th distance, of the index: two
// compares and some scalar work a step, whatever the number of keys; the keys
// that stay are then placed by the number of smaller ones.  A cell's first
// points are 20 to 60 keys, and one by one they were half of the kernel's work;
// a long walk's later cells add a few each, which the bisection's serial steps
// only delay (1,500 queries over 100,000 points: all by bisection 188 µs, all
// one by one 173, mixed 2 % below that; a reconstruction of 30,000 points on a
// 128³ grid with 50,000 far centroids an iteration 7.27 → 7.04 ms).
constexpr int kDescOneByOne = 12;

__device__ __forceinline__ void desc_take(uint64_t& list, uint64_t& kth, uint64_t key, uint64_t cand, int k,
                                          uint64_t* sel) {
    const int lane = threadIdx.x & 63;
    const int many = __builtin_popcountll(cand);
    if (many <= kDescOneByOne) {
        for (; cand; cand &= cand - 1) {
            const uint64_t c = read_lane64(key, __builtin_ctzll(cand));
            if (!(c < kth)) continue;
            // c enters at p: the lanes from p on take their lower neighbour's key
            const int p = __builtin_popcountll(__builtin_amdgcn_ballot_w64(list < c));
            const uint32_t plo = uint32_t(dpp_or_zero<0x138>(int(uint32_t(list))));  // wave_shr 1
            const uint32_t phi = uint32_t(dpp_or_zero<0x138>(int(uint32_t(list >> 32))));
            const uint64_t prev = (uint64_t(phi) << 32) | plo;
            list = lane == p ? c : (lane > p ? prev : list);
            list = lane < k ? list : kNoKey;
            kth = read_lane64(list, k - 1);
        }
        return;
    }
    const bool is = (cand >> lane) & 1ull;
    key = is ? key : ~0ull;
    const uint32_t ld = uint32_t(list >> 32), kd = uint32_t(key >> 32);
    const int total = __builtin_popcountll(__builtin_amdgcn_ballot_w64(list < kNoKey)) + many;
    uint64_t limit = kNoKey;  // the keys below it stay
    if (total > k) {
        // count(d < lo) < k < count(d < hi) in the distance's bits
        uint32_t lo = 0, hi = uint32_t(kth >> 32) + 1u;
        if (kth == kNoKey) hi = wave_max_u32(max(is ? kd : 0u, list < kNoKey ? ld : 0u)) + 1u;
        // first a quarter of the largest squared distance: on a surface a
        // quarter of the points
        uint32_t mid = hi > (2u << 24) ? hi - (2u << 23) : hi >> 1;
        bool found = false;
        while (hi - lo > 1) {
            const int c = __builtin_popcountll(__builtin_amdgcn_ballot_w64(ld < mid)) +
                          __builtin_popcountll(__builtin_amdgcn_ballot_w64(kd < mid));
            if (c == k) {
                found = true;
                break;
            }
            (c > k ? hi : lo) = mid;
            mid = lo + ((hi - lo) >> 1);
        }
        limit = uint64_t(mid) << 32;
        if (!found) {  // some of the points at distance lo stay
            uint64_t l = uint64_t(lo) << 32, h = l + (1ull << 32);
            for (;;) {  // keys differ, so some bound has k keys below it
                limit = l + ((h - l) >> 1);
                const int c = __builtin_popcountll(__builtin_amdgcn_ballot_w64(list < limit)) +
                              __builtin_popcountll(__builtin_amdgcn_ballot_w64(key < limit));
                if (c == k || h - l <= 1) break;
                (c > k ? h : l) = limit;
            }
        }
    }
    // the new keys that stay, then the old ones
    const uint64_t below = (1ull << lane) - 1ull;
    const uint64_t in = __builtin_amdgcn_ballot_w64(key < limit), old = __builtin_amdgcn_ballot_w64(list < limit);
    const int nin = __builtin_popcountll(in), n = min(total, k);
    if ((in >> lane) & 1ull) sel[__builtin_popcountll(in & below)] = key;
    if ((old >> lane) & 1ull) sel[nin + __builtin_popcountll(old & below)] = list;
    __builtin_amdgcn_wave_barrier();
    const uint64_t mine = lane < n ? sel[lane] : kNoKey;
    __builtin_amdgcn_wave_barrier();
    int place = lane < n ? 0 : lane;
    for (int j = 0; j < n; ++j) place += lane < n && read_lane64(mine, j) < mine ? 1 : 0;
    sel[place] = mine;
    __builtin_amdgcn_wave_barrier();
    list = sel[lane];
    __builtin_amdgcn_wave_barrier();
    kth = read_lane64(list, k - 1);
}

// far queries below which none share a walk (see shared_walk_budget)
constexpr int64_t kShareMin = 65536;

// The queries of a search: `list` (nullable) holds them, `count` (nullable)
// their number on the device (else nq), kth[t] (nullable) bounds the k-th d² of
// entry t.  From kShareMin queries on, what the shared walks left of them takes
// their place, if there is a `rest`.
struct DescQueries {
    int64_t nq;
    const int64_t* count;
    const int* list;
    const float* kth;
    const int64_t* rest;
    const int* rest_list;
    const float* rest_kth;
};

template <bool BOXES>
__global__ __launch_bounds__(kDescWaves * 64) void knn_descent_kernel(
    KnnGridArgs G, PyrArgs Y, const int64_t* __restrict__ cell_start, const float4* __restrict__ pts,
    const float* __restrict__ q, DescQueries S, int k, const uint8_t* __restrict__ skip,
    const uint8_t* __restrict__ qmask, int32_t* __restrict__ out_idx, float* __restrict__ out_d2) {
    __shared__ uint64_t s_ent[kDescWaves][kDescStack];  // x | y << 16 | z << 32 | occupancy << 48 | level << 56
    __shared__ float s_ed2[kDescWaves][kDescStack];     // box distance
    __shared__ int s_pt[kDescWaves][64 * kDescPoints];
    __shared__ uint64_t s_sel[kDescWaves][64];
    __shared__ int4 s_dim[kMaxPyr];
    __shared__ int64_t s_off[kMaxPyr];
    if (threadIdx.x < Y.levels) {
        s_dim[threadIdx.x] = Y.dim[threadIdx.x];
        s_off[threadIdx.x] = Y.off[threadIdx.x];
    }
    __syncthreads();
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const uint64_t below = (1ull << lane) - 1ull;
    uint64_t* ent = s_ent[wave];
    float* ed2 = s_ed2[wave];
    int* pt = s_pt[wave];
    uint64_t* sel = s_sel[wave];
    int64_t n = S.count ? int64_t(uniform64(uint64_t(*S.count))) : S.nq;
    const bool rest = S.rest && n >= kShareMin;
    if (rest) n = int64_t(uniform64(uint64_t(*S.rest)));
    const int* qlist = rest ? S.rest_list : S.list;
    const float* init_kth = rest ? S.rest_kth : S.kth;
    const int top = Y.levels - 1;
    const uint64_t root = (uint64_t(uint32_t(uniform(int(Y.mask[s_off[top]])))) << 48) | (uint64_t(uint32_t(top)) << 56);
    for (int64_t t = int64_t(blockIdx.x) * kDescWaves + wave; t < n; t += int64_t(gridDim.x) * kDescWaves) {
        const int64_t i = qlist ? int64_t(uniform(qlist[t])) : t;
        if (qmask && !uniform(int(qmask[i]))) continue;
        const float qx = q[3 * i], qy = q[3 * i + 1], qz = q[3 * i + 2];
        const float cap = init_kth ? init_kth[t] : INFINITY;
        uint64_t list = kNoKey, kth = kNoKey;
        float bound = qx == qx && qy == qy && qz == qz ? cap : -1.f;  // below every distance for no number
        int sp = 1, steps = 0;
        ent[0] = root;
        ed2[0] = 0.f;
        __builtin_amdgcn_wave_barrier();
        while (sp > 0) {
            int nb = 1;
            if (bound < INFINITY || steps >= kDescGreedy)
                nb = min(8, max(1, (kDescStack - kDescReserve - sp) / 7));
            nb = min(nb, sp);
            ++steps;
            // lane 8g + c: child c of the g-th entry from the top
            const int g = lane >> 3, c = lane & 7;
            uint64_t e = 0;
            bool on = g < nb;
            if (on) {
                e = ent[sp - 1 - g];
                on = ed2[sp - 1 - g] <= bound && ((e >> (48 + c)) & 1ull);
            }
            sp -= nb;
            const int l = int(e >> 56) & 0xF;
            const int x = 2 * int(e & 0xFFFF) + (c & 1), y = 2 * int((e >> 16) & 0xFFFF) + ((c >> 1) & 1),
                      z = 2 * int((e >> 32) & 0xFFFF) + (c >> 2);
            uint32_t ci = 0;  // an index has at most 2^27 cells
            float d = INFINITY;
            if (on) {
                const int4 cd = s_dim[l - 1];
                ci = uint32_t(x) + uint32_t(cd.x) * (uint32_t(y) + uint32_t(cd.y) * uint32_t(z));
                if (BOXES) {
                    const int64_t bi = 2 * ((l == 1 ? 0 : Y.ncells + s_off[l - 1]) + ci);
                    d = tight_box_d2(Y.box[bi], Y.box[bi + 1], qx, qy, qz);
                } else {
                    d = pyr_box_d2(G, G.cell * float(1 << (l - 1)), Y.margin, qx, qy, qz, x, y, z);
                }
                on = d <= bound;
            }
            const bool push = on && l > 1, cell = on && l == 1;
            __builtin_amdgcn_wave_barrier();
            const uint64_t pm = __builtin_amdgcn_ballot_w64(push);
            if (pm) {
                const int occ = push ? int(Y.mask[s_off[l - 1] + ci]) : 0;
                int at = sp + __builtin_popcountll(pm & below);
                sp = uniform(sp + __builtin_popcountll(pm));
                // the nearest child of the top entry that pushes goes on top
                // (of the wave's first 8 lanes where these push any)
                const uint32_t db = push && g == 0 ? __float_as_uint(d) : 0xFFFFFFFFu;
                uint32_t mn = min(db, uint32_t(dpp_or_zero<0xB1>(int(db))));     // quad_perm: lane ^ 1
                mn = min(mn, uint32_t(dpp_or_zero<0x4E>(int(mn))));              // lane ^ 2
                mn = min(mn, uint32_t(dpp_or_zero<0x141>(int(mn))));             // row_half_mirror: the other quad
                const uint64_t lead = __builtin_amdgcn_ballot_w64(push && g == 0 && db == mn);
                if (lead) {
                    const int ll = __builtin_ctzll(lead);
                    const int was = __builtin_amdgcn_readlane(at, ll);
                    at = lane == ll ? sp - 1 : (at == sp - 1 ? was : at);
                }
                if (push) {
                    ent[at] = uint64_t(uint32_t(x)) | (uint64_t(uint32_t(y)) << 16) | (uint64_t(uint32_t(z)) << 32) |
                              (uint64_t(uint32_t(occ)) << 48) | (uint64_t(uint32_t(l - 1)) << 56);
                    ed2[at] = d;
                }
            }
            if (__builtin_amdgcn_ballot_w64(cell)) {
                int64_t b = 0, be = 0;
                if (cell) {
                    b = cell_start[ci];
                    be = cell_start[ci + 1];
                }
                // the cells' points, up to kDescPoints of each a round, laid
                // out one after the other and scanned 64 a step
                while (__builtin_amdgcn_ballot_w64(b < be)) {
                    const int m = int(min(be - b, int64_t(kDescPoints)));
                    const int incl = wave_scan_add(m);
                    const int total = __builtin_amdgcn_readlane(incl, 63);
                    for (int j = 0; j < m; ++j) pt[incl - m + j] = int(b + j);
                    b += m;
                    __builtin_amdgcn_wave_barrier();
                    for (int cb = 0; cb < total; cb += 64) {
                        uint64_t key = ~0ull;
                        if (cb + lane < total) {
                            const float4 p = pts[pt[cb + lane]];
                            const int idx = __float_as_int(p.w);
                            key = (uint64_t(__float_as_uint(dist2(qx - p.x, qy - p.y, qz - p.z))) << 32) | uint32_t(idx);
                            // the skip byte only for a point that would enter the list
                            if (key < kth && skip && skip[idx]) key = ~0ull;
                        }
                        if (const uint64_t cand = __builtin_amdgcn_ballot_w64(key < kth))
                            desc_take(list, kth, key, cand, k, sel);
                    }
                    __builtin_amdgcn_wave_barrier();
                }
                bound = fminf(cap, __uint_as_float(uint32_t(kth >> 32)));  // (∞ while there are fewer)
            }
            __builtin_amdgcn_wave_barrier();
        }
        if (lane < k) {
            out_idx[i * k + lane] = list == kNoKey ? -1 : int32_t(uint32_t(list));
            if (out_d2) out_d2[i * k + lane] = list == kNoKey ? INFINITY : __uint_as_float(uint32_t(list >> 32));
        }
    }
}

// The same pyramid walk shared by a wave: 64 neighbouring queries (the far
// queries arrive tile by tile) walk the union of their searches with one
// wave-uniform stack of (block, lanes that need it) in LDS, the way the
// Barnes-Hut walk shares its tree.  Every block and every point is then one
// load for the wave instead of 64 scattered ones, and the lanes stay in
// step.  Children are taken nearest-first for the wave's first active lane;
// each lane still prunes with its own k-th key, so its result is exactly
// its own k nearest points.  A child's distance is that of the bounding box
// of its points, not of its cells: a far query over a surface patch then
// opens the few cells near its foot point instead of every cell whose box
// comes within a cell width of its k-th distance.
//
// The walk is a chain of dependent loads, so each step issues its loads
// together: opening a block fetches its 8 children's boxes and their own
// occupancy bytes (or, for cells, their point ranges) in one vector load
// over a few lanes; a stack entry carries its block's occupancy byte; a
// cell's points come in one vector load (64 at a time) staged in LDS.
constexpr int kPwWaves = 2;  // small blocks free their slots sooner: the walks end at very different times
constexpr int kPwStack = 128;  // ≥ 7 · kMaxPyr + 1 entries
// A walk's length varies tenfold and more, and the launch lasts as long as
// its longest walks, on an otherwise idle chip: a wave stops after this many
// pops and hands its open queries, with the bounds they have, to a search of
// their own (knn_descent_kernel).  Sharing pays while the waves fill the
// chip, so the more queries, the more pops, and walks are longer in a larger
// cloud: 120,000 far of 30,000 points 880 µs with 470 pops, 644 with 117;
// 270,000 of 300,000 3.3 ms with 1,024, 2.35 with 527, 2.12 with 264; 180,000 of
// 1M 5.3 ms with 1,024, 3.78 with 350, 4.18 with 88.  Below kShareMin queries
// none share (53,000 of 30,000 points: 0.41 ms with 100 pops, 0.35 alone).
__device__ __forceinline__ int shared_walk_budget(int64_t nq, int64_t points) {
    return int(min(max(nq / 1024 + points / 6144, int64_t(64)), int64_t(1024)));
}

template <int K>
__global__ __launch_bounds__(kPwWaves * 64) void knn_pyramid_wave_kernel(KnnGridArgs G, PyrArgs Y,
                                                                        const int64_t* __restrict__ cell_start,
                                                                        const float4* __restrict__ pts,
                                                                        const float* __restrict__ q,
                                                                        const int64_t* __restrict__ count,
                                                                        const int* __restrict__ qlist, int k,
                                                                        const uint8_t* __restrict__ skip,
                                                                        const float* __restrict__ init_kth,
                                                                        int32_t* __restrict__ out_idx,
                                                                        float* __restrict__ out_d2, int64_t points,
                                                                        int* __restrict__ open_q,
                                                                        float* __restrict__ open_kth,
                                                                        unsigned long long* __restrict__ n_open) {
    const int64_t nq = *count;  // launched for every query
    if (nq < kShareMin || int64_t(blockIdx.x) * kPwWaves * 64 >= nq) return;
    const int budget = shared_walk_budget(nq, points);
    // stack entry: (x | y << 16, z | level << 16 | occupancy << 20, lanes lo, lanes hi)
    __shared__ int4 s_stk[kPwWaves][kPwStack];
    __shared__ float4 s_box[kPwWaves][16];    // box of child c: lo at 2c, hi at 2c + 1
    __shared__ int64_t s_rng[kPwWaves][16];   // level 1: point range of child cell c at 2c, 2c + 1
    __shared__ int s_cocc[kPwWaves][16];      // level ≥ 2: occupancy byte of child c at 2c
    __shared__ float4 s_pts[kPwWaves][64];    // points of the cell being scanned
    __shared__ int4 s_dim[kMaxPyr];
    __shared__ int64_t s_off[kMaxPyr];
    if (threadIdx.x < Y.levels) {
        s_dim[threadIdx.x] = Y.dim[threadIdx.x];
        s_off[threadIdx.x] = Y.off[threadIdx.x];
    }
    __syncthreads();
    // waves take the 64-query chunks alternately from the front and the back
    // of the list (wave w: chunk w/2 if w is even, else the (w/2)-th from
    // the end).  The longest walks are not known before they run and come
    // in runs along the list; started from both ends, fewer of them start
    // late and end after everything else (far walk 1.65 → 1.54 ms per
    // learned iteration)
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int64_t nchunks = (nq + 63) / 64, w = int64_t(blockIdx.x) * kPwWaves + wave;
    const int64_t chunk = (w & 1) ? nchunks - 1 - (w >> 1) : (w >> 1);
    const int64_t t = chunk * 64 + lane;
    const bool valid = w < nchunks && t < nq;
    const int64_t i = valid ? (qlist ? int64_t(qlist[t]) : t) : 0;
    const float qx = valid ? q[3 * i] : 0.f, qy = valid ? q[3 * i + 1] : 0.f, qz = valid ? q[3 * i + 2] : 0.f;
    uint64_t best[K];
    knn_reset<K>(best, k);
    const float cap = (valid && init_kth) ? init_kth[t] : INFINITY;
    const uint64_t all = __builtin_amdgcn_ballot_w64(valid);
    if (all == 0) return;
    auto kth_of = [&]() { return best[0] == kNoKey ? cap : fminf(cap, __uint_as_float(uint32_t(best[0] >> 32))); };
    int4* stk = s_stk[wave];
    float4* box = s_box[wave];
    const int top = Y.levels - 1;
    const int occ_top = uniform(int(Y.mask[s_off[top]]));
    // every lane writes the same entries (no divergent branch: the stack
    // pointer stays in a scalar register)
    stk[0] = make_int4(0, (top << 16) | (occ_top << 20), int(uint32_t(all)), int(uint32_t(all >> 32)));
    __builtin_amdgcn_wave_barrier();
    int sp = 1;
    for (int pops = 0; sp > 0 && pops < budget; ++pops) {
        --sp;
        const int4 e = stk[sp];
        const uint32_t e0 = uint32_t(uniform(e.x)), e1 = uint32_t(uniform(e.y));
        const int bx = int(e0 & 0xFFFFu), by = int(e0 >> 16), bz = int(e1 & 0xFFFFu), l = int((e1 >> 16) & 0xFu);
        const uint32_t occ = e1 >> 20;
        const uint64_t mask = (uint64_t(uint32_t(uniform(e.w))) << 32) | uint32_t(uniform(e.z));
        const bool act = __builtin_amdgcn_inverse_ballot_w64(mask);
        // the children's loads, together: lanes 2c and 2c + 1 fetch child
        // c's box (lo, hi); lanes 16 + 2c and 17 + 2c its point range (a
        // cell) or lane 16 + 2c its occupancy byte (a block)
        {
            const int c = (lane >> 1) & 7;
            if ((occ >> c) & 1u) {
                const int4 cdm = s_dim[l - 1];
                const int x = 2 * bx + (c & 1), y = 2 * by + ((c >> 1) & 1), z = 2 * bz + (c >> 2);
                const int64_t ci = x + int64_t(cdm.x) * (y + int64_t(cdm.y) * z);
                if (lane < 16) {
                    box[lane] = Y.box[2 * ((l == 1 ? 0 : Y.ncells + s_off[l - 1]) + ci) + (lane & 1)];
                } else if (lane < 32) {
                    if (l == 1) s_rng[wave][lane - 16] = cell_start[ci + (lane & 1)];
                    else if (!(lane & 1)) s_cocc[wave][lane - 16] = int(Y.mask[s_off[l - 1] + ci]);
                }
            }
        }
        __builtin_amdgcn_wave_barrier();
        const float kth = kth_of();
        // the children that some lane still needs, keyed by the first active
        // lane's box distance (float bits, positive) with the child number in
        // the low 3 bits, sorted on the scalar unit
        const int ref = __builtin_ctzll(mask);
        uint32_t key[8];
        uint64_t need[8];
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            need[c] = 0;
            key[c] = 0xFFFFFFFFu;
            if ((occ >> c) & 1u) {
                const float d = tight_box_d2(box[2 * c], box[2 * c + 1], qx, qy, qz);
                need[c] = __builtin_amdgcn_ballot_w64(act && d <= kth);
                if (need[c]) {
                    const uint32_t dr = uint32_t(__builtin_amdgcn_readlane(int(__float_as_uint(d)), ref));
                    key[c] = (dr & ~7u) | uint32_t(c);
                }
            }
        }
        // sorting network on 8 scalar keys (19 compare-exchanges)
        auto cx = [&](int a, int b) {
            const uint32_t lo = min(key[a], key[b]), hi = max(key[a], key[b]);
            key[a] = lo;
            key[b] = hi;
        };
        cx(0, 1); cx(2, 3); cx(4, 5); cx(6, 7);
        cx(0, 2); cx(1, 3); cx(4, 6); cx(5, 7);
        cx(1, 2); cx(5, 6); cx(0, 4); cx(3, 7);
        cx(1, 5); cx(2, 6);
        cx(1, 4); cx(3, 6);
        cx(2, 4); cx(3, 5);
        cx(3, 4);
        if (l == 1) {  // children are cells: scan their points, nearest first
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                if (key[j] == 0xFFFFFFFFu) break;
                const int c = int(key[j] & 7u);
                // the lanes that still need this cell with their k-th key now
                const float d = tight_box_d2(box[2 * c], box[2 * c + 1], qx, qy, qz);
                const bool use = act && d <= kth_of();
                if (!__builtin_amdgcn_ballot_w64(use)) continue;
                const int64_t cb = uniform64(uint64_t(s_rng[wave][2 * c])), ce = uniform64(uint64_t(s_rng[wave][2 * c + 1]));
                for (int64_t s0 = cb; s0 < ce; s0 += 64) {
                    const int cnt = int(min(ce - s0, int64_t(64)));
                    if (lane < cnt) {
                        float4 p = pts[s0 + lane];
                        if (skip && skip[__float_as_int(p.w)]) p.w = __int_as_float(-1);
                        s_pts[wave][lane] = p;
                    }
                    __builtin_amdgcn_wave_barrier();
                    for (int jj = 0; jj < cnt; ++jj) {
                        const float4 p = s_pts[wave][jj];
                        const int idx = __float_as_int(p.w);
                        if (idx < 0) continue;
                        const float d2 = dist2(qx - p.x, qy - p.y, qz - p.z);
                        const uint64_t kk = (uint64_t(__float_as_uint(d2)) << 32) | uint32_t(idx);
                        if (use && kk < best[0]) knn_insert<K>(best, kk);
                    }
                    __builtin_amdgcn_wave_barrier();
                }
            }
        } else {  // push the needed children, farthest first so the nearest pops first
#pragma unroll
            for (int j = 7; j >= 0; --j) {
                if (key[j] == 0xFFFFFFFFu) continue;
                const int c = int(key[j] & 7u);
                uint64_t m = 0;
                int co = 0;
#pragma unroll
                for (int cc = 0; cc < 8; ++cc) {
                    m = cc == c ? need[cc] : m;
                }
                co = uniform(s_cocc[wave][2 * c]);
                const int x = 2 * bx + (c & 1), y = 2 * by + ((c >> 1) & 1), z = 2 * bz + (c >> 2);
                stk[sp] = make_int4(x | (y << 16), z | ((l - 1) << 16) | (co << 20), int(uint32_t(m)),
                                    int(uint32_t(m >> 32)));
                ++sp;
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
    // out of pops: the lanes that blocks on the stack still wait for are
    // listed with the bound they have, for a search of their own
    uint64_t open = 0;
    for (int j = 0; j < sp; ++j)
        open |= (uint64_t(uint32_t(uniform(stk[j].w))) << 32) | uint32_t(uniform(stk[j].z));
    if (open) {
        unsigned int base = 0;
        if (lane == 0) base = (unsigned int)(atomicAdd(n_open, (unsigned long long)__builtin_popcountll(open)));
        base = uint32_t(uniform(int(base)));
        if ((open >> lane) & 1ull) {
            const unsigned int slot = base + unsigned(__builtin_popcountll(open & ((1ull << lane) - 1ull)));
            open_q[slot] = int(i);
            open_kth[slot] = kth_of();
        }
    }
    if (valid && !((open >> lane) & 1ull)) knn_store<K>(best, k, i, out_idx, out_d2);
}

// Query sets answered by one search per query from the start: below
// kDescAlways the tiles' bucketing costs more than it saves also for queries
// on the surface (10,000 queries over as many points: 137 → 67 µs); up to
// kDescFew where they are fewer than the points, as then few share a tile
// (20,000 over 30,000: 286 → 198 µs; at 90,000 self queries the tiles win,
// 190 against 328 µs); up to kDescSparse where they are under one per 8
// points (30,000 over 1M: 3.3 ms by coarse-cell shells, 1.2 ms)
constexpr int64_t kDescAlways = 16384, kDescFew = 32768, kDescSparse = 65536;

// (box: null for the boxes of the cells)
static PyrArgs pyr_args(const dwg_knn_index::Level& L, const uint8_t* mask, const float4* box) {
    return PyrArgs{mask ? mask : L.pyr, L.pyr_dim, L.pyr_off, L.pyr_levels, L.pyr_margin, box, L.ncells};
}

// nq queries (of which *count, when given), one wave each
static void launch_wave(dwg_ctx* ctx, const dwg_knn_index* I, const float* q, int64_t nq, const int64_t* count,
                        const int* qlist, int k, const uint8_t* skip, const uint8_t* qmask, int32_t* out_idx,
                        float* out_d2) {
    dim3 grid(grid_for(nq, 4)), block(256);
    const auto& L = I->lvl[1];
#define DWG_KNNW(KK)                                                                                               \
    hipLaunchKernelGGL(knn_wave_kernel<KK>, grid, block, 0, ctx->stream, L.G, L.cell_start, L.pts, L.empty, q, nq, \
                       count, qlist, k, skip, qmask, out_idx, out_d2)
    if (k <= 10) DWG_KNNW(10);
    else if (k <= 17) DWG_KNNW(17);
    else DWG_KNNW(32);
#undef DWG_KNNW
    check_launch();
}

static void launch_descent(dwg_ctx* ctx, const dwg_knn_index* I, const float* q, const DescQueries& S, int k,
                           const uint8_t* skip, const uint8_t* qmask,
                           int32_t* out_idx, float* out_d2, const uint8_t* pyr_mask = nullptr) {
    const auto& L = I->lvl[0];
    if (L.pyr_levels < 2) {
        launch_wave(ctx, I, q, S.nq, S.count, S.list, k, skip, qmask, out_idx, out_d2);
        return;
    }
    const PyrArgs Y = pyr_args(L, pyr_mask, L.pbox);
    // enough blocks to fill the chip; the waves take further queries in turn.
    // Far queries' walks differ most in length and get two waves where others
    // have one (75,000 left of 180,000 far ones: 3.88 ms the diffusion with 4096
    // blocks, 3.72 with 8192, 3.76 with 16384; 60,000 queries among 1M points
    // 1.41, 1.43 and 1.53)
    const int64_t blocks = S.count ? 8192 : 4096;
    dim3 grid(unsigned(std::min<int64_t>(grid_for(S.nq, kDescWaves), blocks))), block(kDescWaves * 64);
    if (Y.box)
        hipLaunchKernelGGL(knn_descent_kernel<true>, grid, block, 0, ctx->stream, L.G, Y, L.cell_start, L.pts, q, S, k,
                           skip, qmask, out_idx, out_d2);
    else
        hipLaunchKernelGGL(knn_descent_kernel<false>, grid, block, 0, ctx->stream, L.G, Y, L.cell_start, L.pts, q, S, k,
                           skip, qmask, out_idx, out_d2);
    check_launch();
}

// the queries qlist[0..*count) that the tiled pass left open (of nq) with
// their bounds; `shared`: 64 neighbours share a walk first, counting in *n_open
// (0) what they leave
static void launch_far(dwg_ctx* ctx, const dwg_knn_index* I, const float* q, int64_t nq, const int64_t* count,
                       const int* qlist, int k, const uint8_t* skip, int32_t* out_idx, float* out_d2,
                       const float* init_kth, bool shared, unsigned long long* n_open, const uint8_t* pyr_mask) {
    const auto& L = I->lvl[0];
    // an index without boxes (its first such query) builds them, a dozen
    // launches and 70 µs for 30,000 points, only if there are enough far
    // queries that these gain as much at once: 48,000 of a cloud of 30,000
    // points 445 µs by cell boxes, 345 by the points' boxes
    constexpr int64_t kBoxMin = 32768;
    if (shared && L.pyr_levels >= 2 && !L.pbox && read_scalar<int64_t>(ctx, count) < kBoxMin) shared = false;
    DescQueries S{nq, count, qlist, init_kth, nullptr, nullptr, nullptr};
    if (!shared || L.pyr_levels < 2) {
        launch_descent(ctx, I, q, S, k, skip, nullptr, out_idx, out_d2, pyr_mask);
        return;
    }
    // the boxes are a cache of the index's own points: building them
    // leaves the index unchanged
    const PyrArgs Y = pyr_args(L, pyr_mask, ensure_boxes(ctx, const_cast<dwg_knn_index::Level&>(L)));
    DWG_REQUIRE(L.pyr_levels <= kMaxPyr && 7 * L.pyr_levels + 1 <= kPwStack, "pyramid deeper than the wave stack");
    int* open_q = static_cast<int*>(ctx->buf("knn_open_q", sizeof(int) * nq));
    float* open_kth = static_cast<float*>(ctx->buf("knn_open_kth", sizeof(float) * nq));
    dim3 grid(grid_for(nq, kPwWaves * 64)), block(kPwWaves * 64);
#define DWG_KNNPW(KK)                                                                                           \
    hipLaunchKernelGGL(knn_pyramid_wave_kernel<KK>, grid, block, 0, ctx->stream, L.G, Y, L.cell_start, L.pts, q, \
                       count, qlist, k, skip, init_kth, out_idx, out_d2, I->n, open_q, open_kth, n_open)
    if (k <= 8) DWG_KNNPW(8);
    else if (k <= 10) DWG_KNNPW(10);
    else if (k == 15) DWG_KNNPW(15);  // the diffusion's 15 neighbours: no spare slot to sink through
    else if (k <= 16) DWG_KNNPW(16);
    else if (k <= 17) DWG_KNNPW(17);  // the learned start's 16-point patches with the point itself
    else DWG_KNNPW(32);
#undef DWG_KNNPW
    check_launch();
    S.rest = reinterpret_cast<const int64_t*>(n_open);
    S.rest_list = open_q;
    S.rest_kth = open_kth;
    launch_descent(ctx, I, q, S, k, skip, nullptr, out_idx, out_d2, pyr_mask);
}

// The queries 0..nq−1 (masked by qmask) bucketed by tile of kTile³ fine cells
// and eighth of it: order[start[sub·t]..start[sub·(t+1))) are tile t's
// queries, list[0..*nlist) the tiles that have any, once for each `chunk` of
// them (tile, chunk); *nopen and the number after it are 0
constexpr int64_t kTileBlocks = 4096;
struct TileBuckets {
    TileArgs T;
    int64_t ntiles = 0, max_list = 0;
    int chunk = 0;
    int64_t* nlist = nullptr;
    int64_t* nopen = nullptr;
    int64_t* start = nullptr;
    int* order = nullptr;
    int2* list = nullptr;
};

static TileBuckets tile_buckets(dwg_ctx* ctx, const dwg_knn_index* I, const float* q, int64_t nq,
                                const uint8_t* qmask) {
    const KnnGridArgs& G = I->lvl[0].G;
    TileBuckets B;
    constexpr int sub = kSubTiled;
    TileArgs& T = B.T;
    for (int d = 0; d < 3; ++d) T.tdim[d] = (G.dim[d] + kTile - 1) / kTile;
    const int64_t ntiles = int64_t(T.tdim[0]) * T.tdim[1] * T.tdim[2], nb = ntiles * sub;
    DWG_REQUIRE(nb < (int64_t(1) << 31), "too many query buckets");
    B.ntiles = ntiles;
    int2* place = static_cast<int2*>(ctx->buf("knnt_place", sizeof(int2) * nq));
    // the buckets' starts, then the counts
    int64_t* start = static_cast<int64_t*>(ctx->buf("knnt_start", sizeof(int64_t) * (nb + 4)));
    B.nlist = start + nb + 1;
    B.nopen = start + nb + 2;
    int* order = static_cast<int*>(ctx->buf("knnt_order", sizeof(int) * nq));
    // a tile's queries are split over blocks so that there are a few thousand:
    // 230,000 centroids over 3,375 points fill 300 tiles, each a thousand
    // queries long (tiled pass 1.3 → 0.2 ms)
    B.chunk = kTileThreads * int(std::max<int64_t>(1, nq / (kTileBlocks * kTileThreads)));
    B.max_list = std::min(ntiles, nq) + nq / B.chunk;
    int2* list = static_cast<int2*>(ctx->buf("knnt_list", sizeof(int2) * size_t(B.max_list)));
    fill_u32(ctx, start, 0, 2 * (nb + 4));
    hipLaunchKernelGGL(tile_count_kernel, dim3(grid_for(nq, 256)), dim3(256), 0, ctx->stream, q, nq, qmask, G, T,
                       place, reinterpret_cast<unsigned long long*>(start));
    check_launch();
    exclusive_scan<int64_t>(ctx, start, nb);
    hipLaunchKernelGGL(tile_scatter_kernel, dim3(grid_for(nq, 256)), dim3(256), 0, ctx->stream, place, nq, start,
                       order);
    check_launch();
    B.start = start;
    B.order = order;
    hipLaunchKernelGGL(tile_list_kernel, dim3(grid_for(ntiles, kListThreads)), dim3(kListThreads), 0, ctx->stream, start,
                       ntiles, B.chunk, list, reinterpret_cast<unsigned long long*>(B.nlist));
    check_launch();
    B.list = list;
    return B;
}

// up to this many tile blocks are launched without reading how many have
// queries: the surplus blocks return at once, for less than the read costs
constexpr int64_t kTileBlind = 16384;

// From this many queries the open ones are brought into the order of their
// tiles (three launches): there may then be enough of them to share walks,
// which need 64 neighbours.  180,000 of 3M centroids without it: walks and
// their left-over searches 1.80 → 2.43 ms
constexpr int64_t kOpenOrder = 262144;

// The tiled pass over the queries 0..nq−1 (masked by qmask); the queries it
// cannot close are listed in redo with their k-th bound in redo_kth, tile by
// tile.  Returns the device address of their count; *left is that of a 0.
static const int64_t* tiled_pass(dwg_ctx* ctx, const dwg_knn_index* I, const float* q, int64_t nq, const uint8_t* qmask,
                                 int k, const uint8_t* skip, int32_t* out_idx, float* out_d2, int* redo,
                                 float* redo_kth, const std::string& name, const KnnScatter* sc,
                                 unsigned long long** left) {
    const KnnGridArgs& G = I->lvl[0].G;
    const TileBuckets B = tile_buckets(ctx, I, q, nq, qmask);
    const TileArgs& T = B.T;
    if (ctx->profile) ctx->count(name + ":queries", read_scalar<int64_t>(ctx, B.start + B.ntiles * kSubTiled));
    auto* nopen = reinterpret_cast<unsigned long long*>(B.nopen);
    *left = nopen + 1;
    int* open_q = redo;
    float* open_kth = redo_kth;
    int64_t* tile_open = nullptr;
    int64_t blocks = B.max_list;
    const int64_t* exact = B.nlist;
    if (blocks > kTileBlind) {
        blocks = read_scalar<int64_t>(ctx, B.nlist);
        exact = nullptr;
    }
    if (nq >= kOpenOrder) {
        open_q = static_cast<int*>(ctx->buf("knnt_rtmp", sizeof(int) * nq));
        open_kth = static_cast<float*>(ctx->buf("knnt_rkth", sizeof(float) * nq));
        tile_open = static_cast<int64_t*>(ctx->buf("knnt_topen", sizeof(int64_t) * (blocks + 1)));
    }
    if (blocks > 0) {
        ProfileScope pt(ctx, name.c_str());
        const KnnScatter scv = sc ? *sc : KnnScatter{nullptr, nullptr};
#define DWG_KNNT(KK)                                                                                                \
    do {                                                                                                            \
        if (sc)                                                                                                     \
            hipLaunchKernelGGL((knn_tile_kernel<KK, true>), dim3(unsigned(blocks)), dim3(kTileThreads), 0,          \
                               ctx->stream, G, T, I->lvl[0].cell_start, I->lvl[0].pts, B.list, B.chunk, B.start, B.order, \
                               q, k, skip, out_idx, out_d2, open_q, open_kth, nopen, tile_open, exact, scv);              \
        else                                                                                                        \
            hipLaunchKernelGGL((knn_tile_kernel<KK, false>), dim3(unsigned(blocks)), dim3(kTileThreads), 0,         \
                               ctx->stream, G, T, I->lvl[0].cell_start, I->lvl[0].pts, B.list, B.chunk, B.start, B.order, \
                               q, k, skip, out_idx, out_d2, open_q, open_kth, nopen, tile_open, exact, scv);              \
    } while (0)
        if (k <= 8) DWG_KNNT(8);
        else if (k <= 10) DWG_KNNT(10);
        else if (k == 15) DWG_KNNT(15);  // the diffusion's 15 neighbours: no spare slot to sink through
        else if (k <= 16) DWG_KNNT(16);
        else if (k <= 17) DWG_KNNT(17);  // the learned start's 16-point patches with the point itself
        else DWG_KNNT(32);
#undef DWG_KNNT
        check_launch();
    }
    if (!tile_open) return B.nopen;
    exclusive_scan<int64_t>(ctx, tile_open, blocks);
    if (blocks > 0) {
        hipLaunchKernelGGL(tile_open_kernel, dim3(unsigned(blocks)), dim3(64), 0, ctx->stream, B.list, B.chunk, B.start,
                           tile_open, open_q, open_kth, redo, redo_kth);
        check_launch();
    }
    return tile_open + blocks;
}

void knn_query(dwg_ctx* ctx, const dwg_knn_index* I, const float* q, int64_t nq, int k, const uint8_t* skip,
               const uint8_t* qmask, int32_t* out_idx, float* out_d2, const char* tag, const KnnScatter* sc) {
    DWG_REQUIRE(I, "null kNN index");
    DWG_REQUIRE(k >= 1 && k <= 32, "k must be in [1, 32]");
    DWG_REQUIRE(nq >= 0, "negative query count");
    DWG_REQUIRE(nq < (int64_t(1) << 31) - 1, "too many queries");
    DWG_REQUIRE(!sc || !qmask, "a scattering query covers every point");
    if (nq == 0) return;
    ProfileScope ps(ctx, tag ? tag : "knn_query");
    const std::string base = tag ? tag : "knn_query";
    const bool sparse = nq * 8 < I->n;
    if (nq < kDescAlways || (nq < kDescFew && nq < I->n) || (nq < kDescSparse && sparse)) {
        ctx->count(base + (sparse ? ":sparse" : ":tiles3:redo"), nq);
        launch_descent(ctx, I, q, DescQueries{nq}, k, skip, qmask, out_idx, out_d2);
        if (sc) {
            hipLaunchKernelGGL(scatter_pairs_kernel, dim3(grid_for(nq * k, 256)), dim3(256), 0, ctx->stream, out_idx, k,
                               nq, *sc);
            check_launch();
        }
        return;
    }
    int* redo = static_cast<int*>(ctx->buf("knnt_redo", sizeof(int) * nq + 64));
    float* kth = static_cast<float*>(ctx->buf("knnt_kth", sizeof(float) * nq + 64));
    // at least as many queries as indexed points (triangle centroids): the
    // far ones come in dense patches (spurious surface pieces) and in tile
    // order, so a wave's 64 share most of their search and take the
    // wave-shared walk; sparser far queries are spread apart and search alone
    const bool shared = nq >= I->n;
    unsigned long long* left = nullptr;
    const int64_t* nfar = tiled_pass(ctx, I, q, nq, qmask, k, skip, out_idx, out_d2, redo, kth, base + ":tiles", sc, &left);
    if (ctx->profile) {  // the queries that no tiled pass closes
        const int64_t n = read_scalar<int64_t>(ctx, nfar);
        ctx->count(base + ":tiles:redo", n);
        ctx->count(base + (shared ? ":far_shared" : ":tiles3:redo"), n);
    }
    {
        const std::string name = base + ":redo";
        ProfileScope pr(ctx, name.c_str());
        const uint8_t* pm = (skip && I->lvl[0].pyr_levels >= 2) ? masked_pyramid(ctx, I->lvl[0], skip) : nullptr;
        launch_far(ctx, I, q, nq, nfar, redo, k, skip, out_idx, out_d2, kth, shared, left, pm);
    }
    if (sc) {
        const std::string name = base + ":scatter";
        ProfileScope pr(ctx, name.c_str());
        hipLaunchKernelGGL(scatter_pairs_hashed_kernel, dim3(grid_for(nq, 256)), dim3(256), 0, ctx->stream, out_idx, k,
                           redo, nfar, *sc);
        check_launch();
    }
}

}  // namespace dwg
