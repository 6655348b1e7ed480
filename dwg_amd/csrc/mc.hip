// Marching cubes with wavefront prefix-sum compaction.
//
// The reference launches one 12-thread block per cube and appends triangles
// through a global atomic counter into a buffer of max(R³/2, 1e6) triangles
// (TurboMC.cu:383-478, 572-638), so only 12 of 64 lanes work and the output
// order is unordered.  Here a first pass reads the field once, in runs of 64
// samples along x, keeps one bit a sample and finds the cubes the surface
// crosses with a few operations for 16 of them; it counts the triangles of
// every brick of 8 × 8 × 16 cubes.  A scan turns the counts into offsets, and
// an emit pass takes one block per brick with triangles, one lane a triangle,
// and writes them in brick order, cube order inside a brick.  The result is
// exact-size and deterministic.  Corner convention, edge interpolation, table
// and the negated face normal follow TurboMC.cu:399-470.
#include "mc.h"
#include "mc_table.h"
#include "scan.h"

namespace dwg {

__constant__ uint64_t c_mc_rows[256];
static bool g_mc_table_ready[64] = {false};

static void ensure_table(dwg_ctx* ctx) {
    if (ctx->device >= 0 && ctx->device < 64 && g_mc_table_ready[ctx->device]) return;
    static const dwg_mc::PackedTable tab = dwg_mc::make_packed_table();
    DWG_HIP_CHECK(hipMemcpyToSymbol(HIP_SYMBOL(c_mc_rows), tab.row, sizeof(tab.row)));
    if (ctx->device >= 0 && ctx->device < 64) g_mc_table_ready[ctx->device] = true;
}

constexpr int kMcThreads = 256;

struct McArgs {
    const float* f;
    int rx, ry, rz;
    float ox, oy, oz, h, iso;
};

// the 4 corners of face z of the cubes in column (x, y): face corner j is
// at (corner_dx(j), corner_dy(j)); a cube's corners 0-3 lie on its face
// z + 1, corners 4-7 on its face z
__device__ __forceinline__ void load_face(const McArgs& A, int x, int y, int z, float (&f)[4]) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
        f[j] = A.f[int64_t(x + dwg_mc::corner_dx(j)) +
                   int64_t(A.rx) * (int64_t(y + dwg_mc::corner_dy(j)) + int64_t(A.ry) * z)];
}

__device__ __forceinline__ int cube_case(const McArgs& A, const float (&lo)[4], const float (&hi)[4]) {
    int c = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) c |= (hi[j] > A.iso ? 1 << j : 0) | (lo[j] > A.iso ? 16 << j : 0);
    return c;
}

// A block takes a brick of 8 × 8 × 16 cubes, each thread a column of 4
// cubes along z whose shared faces it loads once.  Bricks are numbered x,
// y, z fastest first and dealt to the XCDs in contiguous runs
// (xcd_block), so the rows two neighbouring bricks share come from one L2.
// (Bricks of whole 64-cube rows read the grid in longer runs but leave a
// wave few lanes with triangles to write: the emit pass doubles.)
constexpr int kBx = 8, kBy = 8, kZPer = 4, kBz = 4 * kZPer;
static_assert(kBx * kBy * (kBz / kZPer) == kMcThreads, "one column of kZPer cubes per thread");

struct McBricks {
    int nbx, nby, nbz;
};

__device__ __forceinline__ int64_t brick_of_block() { return xcd_block(blockIdx.x, gridDim.x); }

__device__ __forceinline__ void column_of(const McBricks& B, int64_t b, int thread, int& x, int& y, int& z0) {
    x = int(b % B.nbx) * kBx + (thread & (kBx - 1));
    y = int((b / B.nbx) % B.nby) * kBy + ((thread / kBx) & (kBy - 1));
    z0 = int(b / (int64_t(B.nbx) * B.nby)) * kBz + (thread / (kBx * kBy)) * kZPer;
}

// the cases of a thread's column; 0 past the grid
__device__ __forceinline__ void column_cases(const McArgs& A, int x, int y, int z0, int (&cases)[kZPer]) {
    float lo[4] = {0.f, 0.f, 0.f, 0.f};
    const bool col = x < A.rx - 1 && y < A.ry - 1;
    if (col && z0 < A.rz - 1) load_face(A, x, y, z0, lo);
#pragma unroll
    for (int j = 0; j < kZPer; ++j) {
        cases[j] = 0;
        if (col && z0 + j < A.rz - 1) {
            float hi[4];
            load_face(A, x, y, z0 + j + 1, hi);
            cases[j] = cube_case(A, lo, hi);
#pragma unroll
            for (int k = 0; k < 4; ++k) lo[k] = hi[k];
        }
    }
}

__device__ __forceinline__ int wave_inclusive_sum(int v) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int y = __shfl_up(v, off, 64);
        if (lane >= off) v += y;
    }
    return v;
}

// exclusive prefix of v over the block and the block total
__device__ int block_exclusive_sum(int v, int& total) {
    __shared__ int wsum[kMcThreads / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int incl = wave_inclusive_sum(v);
    if (lane == 63) wsum[wave] = incl;
    __syncthreads();
    int before = 0;
    total = 0;
#pragma unroll
    for (int w = 0; w < kMcThreads / 64; ++w) {
        before += w < wave ? wsum[w] : 0;
        total += wsum[w];
    }
    return before + incl - v;
}

// sample at corner i of the cube (x, y, z)
__device__ __forceinline__ float corner_value(const McArgs& A, int x, int y, int z, int i) {
    return A.f[int64_t(x + dwg_mc::corner_dx(i)) +
               int64_t(A.rx) * (int64_t(y + dwg_mc::corner_dy(i)) + int64_t(A.ry) * (z + dwg_mc::corner_dz(i)))];
}

// triangle t of table row `row` of the cube (x, y, z), written to slot o
__device__ __forceinline__ void emit_triangle(const McArgs& A, int x, int y, int z, uint64_t row, int t, int64_t o,
                                              float* __restrict__ tris, float* __restrict__ cent,
                                              float* __restrict__ nrm) {
    float P[3][3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const int e = int((row >> (4 * (3 * t + k))) & 0xF);
        const int a = dwg_mc::edge_a(e), b = dwg_mc::edge_b(e);
        const float va = corner_value(A, x, y, z, a), vb = corner_value(A, x, y, z, b);
        const float pa[3] = {__builtin_fmaf(float(x + dwg_mc::corner_dx(a)), A.h, A.ox),
                             __builtin_fmaf(float(y + dwg_mc::corner_dy(a)), A.h, A.oy),
                             __builtin_fmaf(float(z + dwg_mc::corner_dz(a)), A.h, A.oz)};
        const float pb[3] = {__builtin_fmaf(float(x + dwg_mc::corner_dx(b)), A.h, A.ox),
                             __builtin_fmaf(float(y + dwg_mc::corner_dy(b)), A.h, A.oy),
                             __builtin_fmaf(float(z + dwg_mc::corner_dz(b)), A.h, A.oz)};
        // P = P1 − ell (P2 − P1), ell = (a1 − iso)/(a2 − a1 + 1e-10)
        const float ell = (va - A.iso) / (vb - va + 1e-10f);
#pragma unroll
        for (int d = 0; d < 3; ++d) P[k][d] = pa[d] - ell * (pb[d] - pa[d]);
    }
    if (tris) {
#pragma unroll
        for (int k = 0; k < 3; ++k)
#pragma unroll
            for (int d = 0; d < 3; ++d) tris[9 * o + 3 * k + d] = P[k][d];
    }
    if (cent) {
#pragma unroll
        for (int d = 0; d < 3; ++d) cent[3 * o + d] = (P[0][d] + P[1][d] + P[2][d]) / 3.0f;
    }
    if (nrm) {
        const float u[3] = {P[1][0] - P[0][0], P[1][1] - P[0][1], P[1][2] - P[0][2]};
        const float w[3] = {P[2][0] - P[0][0], P[2][1] - P[0][1], P[2][2] - P[0][2]};
        const float c[3] = {u[1] * w[2] - u[2] * w[1], u[2] * w[0] - u[0] * w[2], u[0] * w[1] - u[1] * w[0]};
        const float s = -1.0f / (sqrtf(c[0] * c[0] + c[1] * c[1] + c[2] * c[2]) + 1e-8f);
#pragma unroll
        for (int d = 0; d < 3; ++d) nrm[3 * o + d] = c[d] * s;
    }
}

// The first pass over the field: a run of 64 cubes along x, kBy along y and
// kBz along z.  A row of 64 samples is one 256-byte load; of its values only
// the bit v > iso is kept, lane x holding the kBz + 1 bits along z of each of
// its rows, so 16 cubes of a column are tested at once.  A wave takes ROWS of
// the run's kBy rows of cubes (with the samples at x + 64 that its last lane's
// cubes need, one row a lane).  Reading the field once in whole lines bounds
// it: 480×512×451, 206 µs with four loads a cube face, 96 µs so (4.6 TB/s).
constexpr int kRunX = 64, kRunWaves = 4, kFacesZ = kBz + 1;
static_assert(kRunX % kBx == 0 && kFacesZ <= 32 && kBy % kRunWaves == 0, "bits of a column in a word, whole bricks");

// Rows of cubes a wave takes: all kBy, a run a wave, or kBy / kRunWaves, a run
// a block, which loads the rows between two waves twice but has four times the
// waves.  Fewer than kRunFew runs leave the card short of loads in flight when
// a wave takes all rows: a counted and emitted mesh 98 µs against 77 at 128³
// (256 runs), 129 against 115 at 256³, 179 against 172 at 350³ (5808 runs),
// but 315 against 320 at 480×512×451 (14848); the any-order pass at 128³ 91
// against 40.
constexpr int kRowsAll = kBy, kRowsFew = kBy / kRunWaves;
constexpr int64_t kRunFew = 8192;
// The any-order pass writes a wave's triangles too, and of a field that crosses its
// level in most cubes these are all the work: grids of fewer runs than these give a
// wave 8 or 4 cubes along z instead of 16, reading the faces between two waves
// twice.  A sphere and a noise field in µs by 16, 8 and 4: 64³ (32 runs) 44, 38, 34
// and 180, 106, 72; 97³ (144) 49, 41, 44 and 201, 152, 128; 128³ (256) 47, 46, 56 and
// 229, 182, 170; 192³ (864) 74, 69, 87 and 465, 429, 429; 256³ (2048) 82, 94, 138 and
// 927, 906, 898
constexpr int64_t kRunTiny = 256, kRunSmall = 2048;

// a wave's part of a run, NZ cubes along z of ROWS rows, and the bits of the cubes
// that exist in a lane's columns (0 past the grid along x)
struct Run {
    int x0, y0, z0, ny;
    uint32_t cubes;
};

template <int ROWS, int NZ>
__device__ __forceinline__ bool run_of_wave(const McArgs& A, const McBricks& B, Run& R) {
    constexpr int W = kBy / ROWS * (kBz / NZ);  // waves of a run
    const int nrx = (B.nbx * kBx + kRunX - 1) / kRunX;
    const int64_t wave = brick_of_block() * kRunWaves + (threadIdx.x >> 6), id = wave / W;
    if (id >= int64_t(nrx) * B.nby * B.nbz) return false;
    const int w = int(wave % W);
    R.x0 = int(id % nrx) * kRunX;
    R.y0 = int(id / nrx % B.nby) * kBy + w % (kBy / ROWS) * ROWS;
    R.z0 = int(id / (int64_t(nrx) * B.nby)) * kBz + w / (kBy / ROWS) * NZ;
    R.ny = R.z0 < A.rz - 1 ? min(ROWS, A.ry - 1 - R.y0) : 0;  // none or less: a wave past the grid
    R.cubes = R.x0 + int(threadIdx.x & 63) < A.rx - 1 ? (1u << min(NZ, max(A.rz - 1 - R.z0, 0))) - 1u : 0u;
    return true;
}

// a wave's samples as bits along z, one word a sample column
template <int ROWS>
using RunBits = uint32_t[ROWS + 1][kRunX + 1];

template <int ROWS, int NZ>
__device__ __forceinline__ void run_bits(const McArgs& A, const Run& R, RunBits<ROWS>& bits) {
    const int lane = threadIdx.x & 63;
    // samples past the grid repeat its last one (no cube uses them)
    const int x = min(R.x0 + lane, A.rx - 1), xe = min(R.x0 + kRunX, A.rx - 1);
    const int64_t plane = int64_t(A.rx) * A.ry;
    const float *col[ROWS + 1], *end = A.f + xe + int64_t(A.rx) * min(R.y0 + min(lane, ROWS), A.ry - 1);
#pragma unroll
    for (int r = 0; r <= ROWS; ++r) col[r] = A.f + x + int64_t(A.rx) * min(R.y0 + r, A.ry - 1);
    uint32_t w[ROWS + 1] = {}, we = 0;
#pragma unroll 4
    for (int s = 0; s <= NZ; ++s) {
        const int64_t z = plane * min(R.z0 + s, A.rz - 1);
        float v[ROWS + 1];
#pragma unroll
        for (int r = 0; r <= ROWS; ++r) v[r] = col[r][z];
        const float e = end[z];
#pragma unroll
        for (int r = 0; r <= ROWS; ++r) w[r] |= (v[r] > A.iso ? 1u : 0u) << s;
        we |= (e > A.iso ? 1u : 0u) << s;
    }
#pragma unroll
    for (int r = 0; r <= ROWS; ++r) bits[r][lane] = w[r];
    if (lane <= ROWS) bits[lane][kRunX] = we;
    __builtin_amdgcn_wave_barrier();
}

// row r of a lane's column: bits along z at its four samples (x, y), (x + 1, y),
// (x, y + 1) and (x + 1, y + 1), and the cubes that the surface crosses
struct RunColumn {
    uint32_t a, a1, b, b1, crossed;
};

template <int ROWS>
__device__ __forceinline__ RunColumn run_column(const RunBits<ROWS>& bits, int r, uint32_t cubes) {
    const int lane = threadIdx.x & 63;
    RunColumn C{bits[r][lane], bits[r][lane + 1], bits[r + 1][lane], bits[r + 1][lane + 1], 0};
    const uint32_t any = C.a | C.a1 | C.b | C.b1, all = C.a & C.a1 & C.b & C.b1;
    C.crossed = (any | (any >> 1)) & ~(all & (all >> 1)) & cubes;
    return C;
}

// the case of cube z of the column: corners 0-3 on its face z + 1, 4-7 on z
__device__ __forceinline__ uint32_t run_case(const RunColumn& C, int z) {
    const uint32_t a = C.a >> z, a1 = C.a1 >> z, b = C.b >> z, b1 = C.b1 >> z;
    return ((a >> 1) & 1u) | (a1 & 2u) | ((b1 & 2u) << 1) | ((b & 2u) << 2) | ((a & 1u) << 4) | ((a1 & 1u) << 5) |
           ((b1 & 1u) << 6) | ((b & 1u) << 7);
}

template <int ROWS>
__global__ __launch_bounds__(kRunWaves * 64) void mc_count_kernel(McArgs A, McBricks B, int64_t* __restrict__ tile_counts,
                                                                   int* __restrict__ list,
                                                                   unsigned long long* __restrict__ nlist) {
    __shared__ uint8_t s_ntri[256];  // triangles of each case, read per lane from LDS
    __shared__ RunBits<ROWS> s_bits[kRunWaves];
    __shared__ int s_cnt[kRunWaves][kRunX / kBx];
    static_assert(kRunWaves * 64 == 256, "one table entry per thread");
    s_ntri[threadIdx.x] = uint8_t(c_mc_rows[threadIdx.x] >> 60);
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    Run R;
    const bool have = run_of_wave<ROWS, kBz>(A, B, R);
    int cnt = 0;
    if (have && R.ny > 0) {
        run_bits<ROWS, kBz>(A, R, s_bits[wave]);
#pragma unroll 1
        for (int r = 0; r < R.ny; ++r) {
            const RunColumn C = run_column<ROWS>(s_bits[wave], r, R.cubes);
            for (uint32_t m = C.crossed; m; m &= m - 1u) cnt += s_ntri[run_case(C, __builtin_ctz(m))];
        }
        // the sum over a brick's 8 columns along x
#pragma unroll
        for (int off = 1; off < kBx; off <<= 1) cnt += __shfl_xor(cnt, off, 64);
    }
    if constexpr (ROWS < kBy) {  // the block is one run: the sum over its waves
        static_assert(kBy / ROWS == kRunWaves, "a run a block");
        if (lane % kBx == 0) s_cnt[wave][lane / kBx] = cnt;
        __syncthreads();
        if (wave > 0) return;
        cnt = 0;
#pragma unroll
        for (int w = 0; w < kRunWaves; ++w) cnt += s_cnt[w][lane / kBx];
    }
    const int bx = R.x0 / kBx + lane / kBx;
    if (have && lane % kBx == 0 && bx < B.nbx) {
        const int64_t b = bx + int64_t(B.nbx) * (R.y0 / kBy + int64_t(B.nby) * (R.z0 / kBz));
        tile_counts[b] = cnt;
        // the bricks with triangles, in any order: the emit pass takes one
        // block each (its output place comes from the scan of the counts)
        if (cnt > 0) list[atomicAdd(nlist, 1ull)] = int(b);
    }
}

// The emit pass: each thread finds the cases of a column of kZPer cubes, then
// the block lists its triangles in order and takes one a lane, so that all
// lanes write, side by side (the threads whose columns the surface crosses
// wrote theirs alone: 111 → 44 µs for 480×512×451).
constexpr int kEmitList = 2048;

__global__ __launch_bounds__(kMcThreads) void mc_emit_kernel(McArgs A, McBricks B, const int64_t* __restrict__ tile_offsets,
                                                             const int* __restrict__ list, float* __restrict__ tris,
                                                             float* __restrict__ cent, float* __restrict__ nrm) {
    __shared__ uint32_t s_tri[kEmitList];  // thread | cube << 8 | case << 12 | triangle << 20
    const int64_t b = list[blockIdx.x];  // a brick with triangles
    int x, y, z0;
    column_of(B, b, threadIdx.x, x, y, z0);
    int cases[kZPer];
    column_cases(A, x, y, z0, cases);
    int cnt = 0;
#pragma unroll
    for (int j = 0; j < kZPer; ++j) cnt += int(c_mc_rows[cases[j]] >> 60);
    int total;
    const int first = block_exclusive_sum(cnt, total);
    const int64_t o = tile_offsets[b];
    for (int w0 = 0; w0 < total; w0 += kEmitList) {
        __syncthreads();
        if (cnt > 0 && first < w0 + kEmitList && first + cnt > w0) {
            int k = first - w0;
#pragma unroll
            for (int j = 0; j < kZPer; ++j) {  // the column's cubes in z order, each in table order
                const int nt = int(c_mc_rows[cases[j]] >> 60);
                for (int t = 0; t < nt; ++t, ++k)
                    if (k >= 0 && k < kEmitList)
                        s_tri[k] = threadIdx.x | (uint32_t(j) << 8) | (uint32_t(cases[j]) << 12) | (uint32_t(t) << 20);
            }
        }
        __syncthreads();
        for (int k = threadIdx.x; k < min(kEmitList, total - w0); k += kMcThreads) {
            const uint32_t e = s_tri[k];
            int tx, ty, tz;
            column_of(B, b, int(e & 255u), tx, ty, tz);
            emit_triangle(A, tx, ty, tz + int((e >> 8) & 15u), c_mc_rows[(e >> 12) & 255u], int(e >> 20), o + w0 + k,
                          tris, cent, nrm);
        }
    }
}

// One pass for callers that take the triangles in any order (the
// diffusion's centroids and face normals, whose sums do not depend on it): the
// first pass's wave lists the cubes that the surface crosses and, whenever
// enough are listed, takes an output range with one atomic add and writes
// their triangles, one a lane.  The values are those of the ordered
// passes.  A list writes only when its whole range fits in capacity; the count
// is complete either way.  The field's read bounds it where the surface is a
// small part of the grid: 512³ 0.42 → 0.256 ms, 128³ 93 → 40 µs (from one
// thread a column of 4 cubes, writing that column's triangles).
constexpr int kFusedList = 256;  // cubes listed before their triangles are written

template <int ROWS, int NZ>
__global__ __launch_bounds__(kRunWaves * 64) void mc_fused_kernel(McArgs A, McBricks B,
                                                                   unsigned long long* __restrict__ ntri,
                                                                   int64_t capacity, float* __restrict__ cent,
                                                                   float* __restrict__ nrm) {
    constexpr int kMaxTri = 5;  // triangles of a cube
    __shared__ uint8_t s_ntri[256];
    __shared__ RunBits<ROWS> s_bits[kRunWaves];
    __shared__ uint32_t s_cube[kRunWaves][kFusedList];      // lane | row << 6 | z << 9 | case << 13
    __shared__ uint32_t s_tri[kRunWaves][64 * kMaxTri];     // the cube, triangle << 21
    s_ntri[threadIdx.x] = uint8_t(c_mc_rows[threadIdx.x] >> 60);
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    Run R;
    if (!run_of_wave<ROWS, NZ>(A, B, R) || R.ny <= 0) return;
    uint32_t *cubes = s_cube[wave], *tri = s_tri[wave];
    run_bits<ROWS, NZ>(A, R, s_bits[wave]);
    int listed = 0, r = 0;
    RunColumn C = run_column<ROWS>(s_bits[wave], 0, R.cubes);
    uint32_t m = C.crossed;
    for (bool more = true; more;) {
        // list cubes, one a lane, until the list is full or the rows are done
        while (listed + 64 <= kFusedList) {
            const uint64_t act = __builtin_amdgcn_ballot_w64(m != 0);
            if (!act) {
                if (++r >= R.ny) {
                    more = false;
                    break;
                }
                C = run_column<ROWS>(s_bits[wave], r, R.cubes);
                m = C.crossed;
                continue;
            }
            if (m) {
                const int z = __builtin_ctz(m);
                m &= m - 1u;
                cubes[listed + __builtin_popcountll(act & ((1ull << lane) - 1ull))] =
                    uint32_t(lane) | (uint32_t(r) << 6) | (uint32_t(z) << 9) | (run_case(C, z) << 13);
            }
            listed += __builtin_popcountll(act);
        }
        __builtin_amdgcn_wave_barrier();
        int cnt = 0;
        for (int k = lane; k < listed; k += 64) cnt += s_ntri[cubes[k] >> 13];
        const int total = __builtin_amdgcn_readlane(wave_inclusive_sum(cnt), 63);
        unsigned long long at = 0;
        if (lane == 0 && total > 0) at = atomicAdd(ntri, (unsigned long long)total);
        int64_t o = int64_t((uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(int(uint32_t(at >> 32))))) << 32) |
                            uint32_t(__builtin_amdgcn_readfirstlane(int(uint32_t(at)))));
        if ((cent || nrm) && o + total <= capacity) {
            for (int k0 = 0; k0 < listed; k0 += 64) {
                const uint32_t e = k0 + lane < listed ? cubes[k0 + lane] : 0u;
                const int nt = k0 + lane < listed ? int(s_ntri[e >> 13]) : 0;
                const int incl = wave_inclusive_sum(nt), n = __builtin_amdgcn_readlane(incl, 63);
                for (int t = 0; t < nt; ++t) tri[incl - nt + t] = e | (uint32_t(t) << 21);
                __builtin_amdgcn_wave_barrier();
                for (int k = lane; k < n; k += 64) {
                    const uint32_t c = tri[k];
                    emit_triangle(A, R.x0 + int(c & 63u), R.y0 + int((c >> 6) & 7u), R.z0 + int((c >> 9) & 15u),
                                  c_mc_rows[(c >> 13) & 255u], int(c >> 21), o + k, nullptr, cent, nrm);
                }
                __builtin_amdgcn_wave_barrier();
                o += n;
            }
        }
        listed = 0;
    }
}

static McArgs mc_args(const float* field, const dwg_grid* g, float iso, McBricks& B, int64_t& tiles) {
    DWG_REQUIRE(g && g->res[0] >= 2 && g->res[1] >= 2 && g->res[2] >= 2, "grid needs at least 2 samples per axis");
    const McArgs A{field, g->res[0], g->res[1], g->res[2], g->origin[0], g->origin[1], g->origin[2], g->h, iso};
    B = McBricks{(A.rx - 1 + kBx - 1) / kBx, (A.ry - 1 + kBy - 1) / kBy, (A.rz - 1 + kBz - 1) / kBz};
    tiles = int64_t(B.nbx) * B.nby * B.nbz;
    DWG_REQUIRE(tiles < (int64_t(1) << 31), "grid too large for the marching-cubes launch");
    return A;
}

static int64_t mc_runs(const McBricks& B) {
    return (int64_t(B.nbx) * kBx + kRunX - 1) / kRunX * B.nby * B.nbz;
}

int64_t marching_cubes_any_order(dwg_ctx* ctx, const float* field, const dwg_grid* g, float iso, int64_t capacity,
                                 float* cent, float* nrm) {
    DWG_REQUIRE(capacity >= 0, "negative capacity");
    McBricks B;
    int64_t tiles;
    const McArgs A = mc_args(field, g, iso, B, tiles);
    ensure_table(ctx);
    auto* n = static_cast<unsigned long long*>(ctx->buf("mc_fused_count", 64));
    fill_u32(ctx, n, 0u, 2);
    {
        ProfileScope ps(ctx, "mc_fused");
        const int64_t runs = mc_runs(B);
        // LAUNCH(rows, cubes along z) of a wave
#define DWG_MC_FUSED(R, Z)                                                                                          \
    hipLaunchKernelGGL((mc_fused_kernel<R, Z>), dim3(grid_for(runs * (kBy / (R)) * (kBz / (Z)), kRunWaves)),        \
                       dim3(kRunWaves * 64), 0, ctx->stream, A, B, n, capacity, cent, nrm)
        if (runs < kRunTiny) DWG_MC_FUSED(kRowsFew, kBz / 4);
        else if (runs < kRunSmall) DWG_MC_FUSED(kRowsFew, kBz / 2);
        else if (runs < kRunFew) DWG_MC_FUSED(kRowsFew, kBz);
        else DWG_MC_FUSED(kRowsAll, kBz);
#undef DWG_MC_FUSED
        check_launch();
    }
    const int64_t total = int64_t(read_scalar<unsigned long long>(ctx, n));
    if (total > capacity) throw Error(DWG_ERR_CAPACITY, "marching cubes output exceeds capacity", total);
    return total;
}

// 480×512×451 into exact-size buffers 300 µs with a call to count and one to
// count and emit, 176 so
int64_t marching_cubes_alloc(dwg_ctx* ctx, const float* field, const dwg_grid* g, float iso, dwg_mc_alloc alloc,
                             void* user) {
    McBricks B;
    int64_t tiles;
    const McArgs A = mc_args(field, g, iso, B, tiles);
    ensure_table(ctx);
    // brick counts (scanned in place: offsets, the total at [tiles]) and, at
    // [tiles + 1], the number of bricks with triangles
    int64_t* offs = static_cast<int64_t*>(ctx->buf("mc_tiles", sizeof(int64_t) * (tiles + 2)));
    int* list = static_cast<int*>(ctx->buf("mc_list", sizeof(int) * tiles));
    auto* nlist = reinterpret_cast<unsigned long long*>(offs + tiles + 1);
    fill_u32(ctx, nlist, 0u, 2);
    {
        ProfileScope ps(ctx, "mc_count");
        const int64_t runs = mc_runs(B);
        if (runs < kRunFew)
            hipLaunchKernelGGL(mc_count_kernel<kRowsFew>, dim3(unsigned(runs)), dim3(kRunWaves * 64), 0, ctx->stream,
                               A, B, offs, list, nlist);
        else
            hipLaunchKernelGGL(mc_count_kernel<kRowsAll>, dim3(grid_for(runs, kRunWaves)), dim3(kRunWaves * 64), 0,
                               ctx->stream, A, B, offs, list, nlist);
        check_launch();
        exclusive_scan<int64_t>(ctx, offs, tiles);
    }
    struct Totals {
        int64_t tris, bricks;
    };
    const Totals tot = read_scalar<Totals>(ctx, reinterpret_cast<const Totals*>(offs + tiles));
    const int64_t total = tot.tris;
    float *tris = nullptr, *cent = nullptr, *nrm = nullptr;
    DWG_REQUIRE(alloc(user, total, &tris, &cent, &nrm) == 0, "marching cubes buffers refused");
    if (total > 0 && (tris || cent || nrm)) {
        ProfileScope ps(ctx, "mc_emit");
        hipLaunchKernelGGL(mc_emit_kernel, dim3(unsigned(tot.bricks)), dim3(kMcThreads), 0, ctx->stream, A, B, offs,
                           list, tris, cent, nrm);
        check_launch();
    }
    return total;
}

int64_t marching_cubes(dwg_ctx* ctx, const float* field, const dwg_grid* g, float iso, int64_t capacity, float* tris,
                       float* cent, float* nrm) {
    struct Buffers {
        int64_t capacity;
        float *tris, *cent, *nrm;
    } b{capacity, tris, cent, nrm};
    const int64_t total = marching_cubes_alloc(
        ctx, field, g, iso,
        [](void* user, int64_t count, float** t, float** c, float** n) {
            auto* u = static_cast<Buffers*>(user);
            if (count <= u->capacity) {
                *t = u->tris;
                *c = u->cent;
                *n = u->nrm;
            }
            return 0;
        },
        &b);
    if (total > capacity) throw Error(DWG_ERR_CAPACITY, "marching cubes output exceeds capacity", total);
    return total;
}

}  // namespace dwg
