// svdag_voxelize.hip -- device fragment producer: a triangle soup -> unsorted
// Morton keys with duplicates, the input contract of the DAG build.
//
// The reference produces its fragments with an OpenGL conservative rasteriser
// (src/Voxelizer.cpp:254-369, Shaders/FragmentShader.glsl:19-32, 208-209).
// Here the triangles are voxelised by the thin surface rule of the
// triangle-surface workload generator (after Schwarz & Seidel 2010): one voxel
// per column along the dominant normal axis, kept when the voxel centre passes
// the three projected edge tests dilated by half the larger edge-normal
// component.  Every floating-point step is the generator's, in the same order
// and without fused multiply-adds, so both emit the same voxels.
//
// Work is spread by columns, not triangles (sizes are heavy-tailed):
//   k_tri_setup     per triangle: normal, dominant axis, edge functions and
//                   the column rectangle; its row count (rows run along w)
//   (scan)          row offsets per triangle
//   k_row_setup     per row: the columns whose centres can pass the dominant
//                   projection's edge tests (a conservative superset, so the
//                   exact per-column test below decides; about a fifth of the
//                   rectangle for the triangle workload), cut into units of at
//                   most 8 columns
//   (scan)          unit offsets per row
//   k_vox_count     one thread per unit: its columns' tests, two result bits
//                   per column, keys per tile of 256 units
//   (scan)          key offsets per tile
//   k_vox_write     the columns with a bit set again, now only for their keys,
//                   staged in LDS and written in runs (no room for the bits: all
//                   tests again)
// A unit never leaves its row, so a thread keeps its triangle's edge functions
// in registers and the wave has no row changes to diverge on.  Threads that
// walked 8 columns across rows reloaded them at nearly every column (some lane
// of the wave always changed rows) and held their keys in scratch memory: 1307
// us for 47.9M voxels of 20k triangles in a 2048^3 grid, and 172 us more to move
// the keys out of per-tile staging areas; now 350 + 246 us.  Bound by the float64
// divisions and edge tests and by the row lookups.
#pragma clang fp contract(off)

#include "svdag_device.hpp"
#include "svdag_internal.hpp"

namespace svdag {

namespace {

constexpr int kVoxThreads = 256;
constexpr int kVoxIpt = 8;  // rows per thread and tile in the row kernels
constexpr uint64_t kVoxTile = uint64_t(kVoxThreads) * kVoxIpt;
static_assert(kVoxTile == kVoxTileItems, "tile size shared with the planner");
constexpr int kUnitCols = 8;  // columns per unit of work
static_assert(kVoxThreads == kVoxUnitTile && 2 * kUnitCols <= 16, "one unit per thread, two result bits per column");

__device__ __forceinline__ double pick3(const double (&v)[3], int i) { return i == 0 ? v[0] : (i == 1 ? v[1] : v[2]); }

__device__ __forceinline__ uint64_t split_by_3(uint32_t a)
{
    uint64_t x = a & 0x1fffff;
    x = (x | x << 32) & 0x1f00000000ffffull;
    x = (x | x << 16) & 0x1f0000ff0000ffull;
    x = (x | x << 8) & 0x100f00f00f00f00full;
    x = (x | x << 4) & 0x10c30c30c30c30c3ull;
    x = (x | x << 2) & 0x1249249249249249ull;
    return x;
}


// A triangle with a non-finite coordinate gets no rows and sets kErrKeyRange
// in *err.
__global__ __launch_bounds__(kVoxThreads) void k_tri_setup(const double* __restrict__ tris, uint64_t n_tris,
                                                           int64_t side, TriSetup* __restrict__ setup,
                                                           uint32_t* __restrict__ rows,
                                                           unsigned long long* __restrict__ rect_columns,
                                                           unsigned long long* __restrict__ err)
{
    __shared__ uint64_t s_red[kVoxThreads / kWave];
    const uint64_t t = uint64_t(blockIdx.x) * kVoxThreads + threadIdx.x;
    uint64_t rect = 0;  // columns of the triangle's rectangle (bounds the row ranges)
    if (t < n_tris) {
        double vs[3][3];
        bool finite = true;
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                vs[c][k] = tris[9 * t + 3 * c + k];
                finite &= isfinite(vs[c][k]);
            }
        if (!finite) atomicOr(err, (unsigned long long)kErrKeyRange);
        // n = (v1 - v0) x (v2 - v0)
        const double e1x = vs[1][0] - vs[0][0], e1y = vs[1][1] - vs[0][1], e1z = vs[1][2] - vs[0][2];
        const double e2x = vs[2][0] - vs[0][0], e2y = vs[2][1] - vs[0][1], e2z = vs[2][2] - vs[0][2];
        TriSetup S{};
        S.n[0] = e1y * e2z - e1z * e2y;
        S.n[1] = e1z * e2x - e1x * e2z;
        S.n[2] = e1x * e2y - e1y * e2x;
        const double an0 = fabs(S.n[0]), an1 = fabs(S.n[1]), an2 = fabs(S.n[2]);
        const int a = an0 >= an1 && an0 >= an2 ? 0 : (an1 >= an2 ? 1 : 2);
        const double ana = a == 0 ? an0 : (a == 1 ? an1 : an2);
        uint64_t nu = 0;
        if (finite && ana != 0.0) {  // else degenerate (or rejected): no rows
            const int u = (a + 1) % 3, w = (a + 2) % 3;
            S.a = a;
            S.u = u;
            S.w = w;
            // Projected edge functions for the three axis planes (xy, yz, zx).
            for (int p = 0; p < 3; ++p) {
                const int i0 = p, i1 = (p + 1) % 3;
                const double sgn = pick3(S.n, (p + 2) % 3) >= 0 ? 1.0 : -1.0;
                if (pick3(S.n, (p + 2) % 3) != 0.0) S.planes |= 1 << p;
                for (int e = 0; e < 3; ++e) {
                    const int b = (e + 1) % 3;
                    const double ex = vs[b][i0] - vs[e][i0], ey = vs[b][i1] - vs[e][i1];
                    const double nx = -ey * sgn, ny = ex * sgn;
                    S.ex[p][e] = nx;
                    S.ey[p][e] = ny;
                    S.ed[p][e] = -(nx * vs[e][i0] + ny * vs[e][i1]) + 0.5 * fmax(fabs(nx), fabs(ny));
                }
            }
            const double lo_u = fmin(fmin(vs[0][u], vs[1][u]), vs[2][u]),
                         hi_u = fmax(fmax(vs[0][u], vs[1][u]), vs[2][u]);
            const double lo_w = fmin(fmin(vs[0][w], vs[1][w]), vs[2][w]),
                         hi_w = fmax(fmax(vs[0][w], vs[1][w]), vs[2][w]);
            const int64_t u0 = max(int64_t(0), int64_t(floor(lo_u)) - 1), u1 = min(side - 1, int64_t(floor(hi_u)) + 1);
            const int64_t w0 = max(int64_t(0), int64_t(floor(lo_w)) - 1), w1 = min(side - 1, int64_t(floor(hi_w)) + 1);
            S.nd = S.n[0] * vs[0][0] + S.n[1] * vs[0][1] + S.n[2] * vs[0][2];
            S.u0 = u0;
            S.w0 = w0;
            S.nw = w1 >= w0 ? uint32_t(w1 - w0 + 1) : 0u;
            nu = u1 >= u0 && S.nw ? uint64_t(u1 - u0 + 1) : 0u;
        }
        setup[t] = S;
        rows[t] = uint32_t(nu);  // at most the grid side, 2^21
        rect = nu * S.nw;
    }
    const uint64_t sum = block_reduce_sum<kVoxThreads>(rect, s_red);
    if (threadIdx.x == 0 && sum) atomicAdd(rect_columns, (unsigned long long)sum);
}

// Owner of global item g: the last i in [lo, hi) with off[i] <= g.
__device__ __forceinline__ uint64_t owner_of(const uint64_t* __restrict__ off, uint64_t lo, uint64_t hi, uint64_t g)
{
    while (hi - lo > 1) {
        const uint64_t mid = (lo + hi) / 2;
        if (off[mid] <= g) lo = mid;
        else hi = mid;
    }
    return lo;
}

// Row r of the triangles' rectangles (row u = u0 + j of triangle t, j = r -
// row_off[t]): the columns [lo, hi] of the rectangle whose centres can pass
// the edge tests of the dominant projection (the plane of u and w).  Edge e
// passes where (nx * cu + ny * cw) + d >= 0; for ny != 0 that bounds cw on
// one side at c* = -(nx * cu + d) / ny.  The bound is widened by the rounding
// error of the test and of c* (far below 2^-46 of their magnitudes) plus one
// column, so it never drops a column the test keeps.
// Rows are handled in tiles of kVoxTile; each tile's unit total goes to
// tile_units for the scan that k_row_offsets finishes (a column total of 2^32 or
// more sets kErrInternal in *err).
__global__ __launch_bounds__(kVoxThreads) void k_row_setup(const TriSetup* __restrict__ setup,
                                                           const uint64_t* __restrict__ row_off,
                                                           const uint64_t* __restrict__ n_tris_ptr,
                                                           const uint64_t* __restrict__ n_rows_ptr,
                                                           uint32_t* __restrict__ row_tri, uint32_t* __restrict__ row_u,
                                                           uint32_t* __restrict__ row_w0,
                                                           uint32_t* __restrict__ row_cols,
                                                           uint32_t* __restrict__ tile_units,
                                                           unsigned long long* __restrict__ err)
{
    __shared__ uint64_t s_red[kVoxThreads / kWave];
    const uint64_t n_tris = *n_tris_ptr, n_rows = *n_rows_ptr;
    const uint64_t ntiles = (n_rows + kVoxTile - 1) / kVoxTile;
    for (uint64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        uint64_t tile_sum = 0, unit_sum = 0;
        const uint64_t end = min(n_rows, (tile + 1) * kVoxTile);
        for (uint64_t r = tile * kVoxTile + threadIdx.x; r < end; r += kVoxThreads) {
            const uint64_t t = owner_of(row_off, 0, n_tris, r);
            const TriSetup& S = setup[t];
            const int64_t iu = S.u0 + int64_t(r - row_off[t]);
            const double cu = double(iu) + 0.5;
            int64_t lo = S.w0, hi = S.w0 + int64_t(S.nw) - 1;
            const double cw_far = double(hi) + 0.5;
            const int p = S.u;
            for (int e = 0; e < 3; ++e) {
                const double nx = S.ex[p][e], ny = S.ey[p][e], d = S.ed[p][e];
                const double g = nx * cu + d;
                if (ny == 0.0) {
                    // The test is g >= 0 for every column (adding ny * cw =
                    // +-0 changes no sign).
                    if (g < 0) hi = lo - 1;
                    continue;
                }
                const double cstar = -g / ny;
                const double mag = fabs(nx * cu) + fabs(ny) * cw_far + fabs(d);
                const double slack = mag * 0x1p-46 / fabs(ny) + fabs(cstar) * 0x1p-46 + 1.0;
                if (!(fabs(cstar) < 0x1p40) || !(slack < 0x1p30)) continue;  // no usable bound
                if (ny > 0) lo = max(lo, int64_t(floor(cstar - 0.5 - slack)));
                else hi = min(hi, int64_t(ceil(cstar - 0.5 + slack)));
            }
            const uint32_t cols = hi >= lo ? uint32_t(hi - lo + 1) : 0u;
            row_tri[r] = uint32_t(t);
            row_u[r] = uint32_t(iu);
            row_w0[r] = uint32_t(lo);
            row_cols[r] = cols;
            tile_sum += cols;
            unit_sum += (cols + kUnitCols - 1) / kUnitCols;
        }
        const uint64_t sum = block_reduce_sum<kVoxThreads>(tile_sum, s_red);
        const uint64_t units = block_reduce_sum<kVoxThreads>(unit_sum, s_red);
        if (threadIdx.x == 0) {
            tile_units[tile] = uint32_t(units);
            if (sum > 0xFFFFFFFFull) atomicOr(err, (unsigned long long)kErrInternal);
        }
    }
}

// unit_off[r] = tile_off[tile] + the units of the tile's rows before r.
__global__ __launch_bounds__(kVoxThreads) void k_row_offsets(const uint32_t* __restrict__ row_cols,
                                                             const uint64_t* __restrict__ tile_off,
                                                             const uint64_t* __restrict__ n_rows_ptr,
                                                             uint64_t* __restrict__ unit_off)
{
    __shared__ uint32_t s_scan[kVoxThreads / kWave];
    const uint64_t n_rows = *n_rows_ptr;
    const uint64_t ntiles = (n_rows + kVoxTile - 1) / kVoxTile;
    for (uint64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const uint64_t r0 = tile * kVoxTile + uint64_t(threadIdx.x) * kVoxIpt;
        uint32_t c[kVoxIpt];
        uint32_t mine = 0;
#pragma unroll
        for (int i = 0; i < kVoxIpt; ++i) {
            c[i] = r0 + i < n_rows ? (row_cols[r0 + i] + kUnitCols - 1) / kUnitCols : 0u;
            mine += c[i];
        }
        uint32_t unused;
        uint64_t o = tile_off[tile] + block_exclusive_scan<kVoxThreads>(mine, s_scan, unused);
#pragma unroll
        for (int i = 0; i < kVoxIpt; ++i) {
            if (r0 + i < n_rows) unit_off[r0 + i] = o;
            o += c[i];
        }
    }
}

// The voxels [lo, hi] along the dominant axis whose centres are within one of
// column crossing `ac` (at most two; lo > hi: none).
__device__ __forceinline__ void column_range(double ac, int64_t side, int32_t& lo, int32_t& hi)
{
    if (fabs(ac) < 0x1p30) {
        lo = max(int32_t(floor(ac - 1.0)), 0);
        hi = min(int32_t(floor(ac)), int32_t(side - 1));
    } else {  // far outside the grid, or not a number
        const int64_t k0 = max(int64_t(floor(ac - 1.0)), int64_t(0)), k1 = min(int64_t(floor(ac)), side - 1);
        lo = k0 <= k1 ? int32_t(k0) : 1;
        hi = k0 <= k1 ? int32_t(k1) : 0;
    }
}

// The unit rows: unit_off is the exclusive scan of the rows' unit counts.
struct RowTable {
    const uint32_t* tri;
    const uint32_t* u;
    const uint32_t* w0;
    const uint32_t* cols;
    const uint64_t* unit_off;
};

// Rows of unit tile t lie in [tile_row[t], tile_row[t + 1] + 1) (tile_row[t] =
// row of the tile's first unit, one entry past the last tile), found by one
// thread per tile.
__global__ __launch_bounds__(kVoxThreads) void k_tile_rows(const uint64_t* __restrict__ unit_off,
                                                           const uint64_t* __restrict__ n_rows_ptr,
                                                           const uint64_t* __restrict__ total_ptr,
                                                           uint64_t* __restrict__ tile_row)
{
    const uint64_t n_rows = *n_rows_ptr, total = *total_ptr;
    const uint64_t ntiles = (total + kVoxThreads - 1) / kVoxThreads;
    for (uint64_t t = uint64_t(blockIdx.x) * kVoxThreads + threadIdx.x; t <= ntiles;
         t += uint64_t(gridDim.x) * kVoxThreads)
        tile_row[t] = t < ntiles ? owner_of(unit_off, 0, n_rows, t * kVoxThreads) : n_rows - 1;
}

// The thread's unit of tile `tile`: its triangle, row, first column and columns.
struct Unit {
    uint32_t tri, u, w0;
    int cols;  // 0: past the last unit
};
__device__ __forceinline__ Unit unit_of(const RowTable& R, const uint64_t* __restrict__ tile_row, uint64_t total,
                                        uint64_t tile)
{
    const uint64_t g = tile * kVoxThreads + threadIdx.x;
    if (g >= total) return Unit{0, 0, 0, 0};
    const uint64_t r = owner_of(R.unit_off, tile_row[tile], tile_row[tile + 1] + 1, g);
    const uint32_t first = uint32_t(g - R.unit_off[r]) * kUnitCols;
    return Unit{R.tri[r], R.u[r], R.w0[r] + first, int(min(uint32_t(kUnitCols), R.cols[r] - first))};
}

// Unit U's voxels: bit 2i + j says that voxel lo + j of its column i is in (lo:
// column_range).
__device__ __forceinline__ uint32_t unit_bits(const TriSetup& S, const Unit& U, int64_t side)
{
    uint32_t found = 0;
    const int a = S.a, u = S.u, w = S.w, planes = S.planes;
    const double cu = double(int64_t(U.u)) + 0.5;
    // Edge functions of the planes (u, w), (a, u) and (w, a), with the
    // terms that the row fixes multiplied out.
    double uu[3], uw[3], ud[3], aa[3], au[3], ad[3], ww[3], wa[3], wd[3];
#pragma unroll
    for (int e = 0; e < 3; ++e) {
        uu[e] = S.ex[u][e] * cu;
        uw[e] = S.ey[u][e];
        ud[e] = S.ed[u][e];
        aa[e] = S.ex[a][e];
        au[e] = S.ey[a][e] * cu;
        ad[e] = S.ed[a][e];
        ww[e] = S.ex[w][e];
        wa[e] = S.ey[w][e];
        wd[e] = S.ed[w][e];
    }
    const double q = S.nd - pick3(S.n, u) * cu, nw = pick3(S.n, w), na = pick3(S.n, a);
    const bool plane_a = (planes >> a) & 1, plane_w = (planes >> w) & 1;  // else edge-on there
#pragma unroll 1
    for (int i = 0; i < U.cols; ++i) {
        const double cw = double(int64_t(U.w0) + i) + 0.5;
        // The dominant projection sees only the column.
        bool in = true;
#pragma unroll
        for (int e = 0; e < 3; ++e) in &= !(uu[e] + uw[e] * cw + ud[e] < 0);
        if (!in) continue;
        const double ac = (q - nw * cw) / na;
        int32_t lo, hi;
        column_range(ac, side, lo, hi);
        double wx[3];
#pragma unroll
        for (int e = 0; e < 3; ++e) wx[e] = ww[e] * cw;
        for (int32_t kk = lo; kk <= hi; ++kk) {
            const double ck = double(kk) + 0.5;
            bool ok = !(fabs(ck - ac) > 0.5);
#pragma unroll
            for (int e = 0; e < 3; ++e) {
                ok &= !(plane_a && aa[e] * ck + au[e] + ad[e] < 0);
                ok &= !(plane_w && wx[e] + wa[e] * ck + wd[e] < 0);
            }
            found |= uint32_t(ok) << (2 * i + (kk - lo));
        }
    }
    return found;
}

// counts[tile] = the tile's voxels; with bits, also the units' bits.
__global__ __launch_bounds__(kVoxThreads) void k_vox_count(const TriSetup* __restrict__ setup, RowTable R,
                                                           const uint64_t* __restrict__ tile_row,
                                                           const uint64_t* __restrict__ total_ptr, int64_t side,
                                                           uint16_t* __restrict__ bits, uint32_t* __restrict__ counts)
{
    __shared__ uint64_t s_red[kVoxThreads / kWave];
    const uint64_t total = *total_ptr;
    const uint64_t ntiles = (total + kVoxThreads - 1) / kVoxThreads;
    for (uint64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const Unit U = unit_of(R, tile_row, total, tile);
        uint32_t found = 0;
        if (U.cols) {
            found = unit_bits(setup[U.tri], U, side);
            if (bits) bits[tile * kVoxThreads + threadIdx.x] = uint16_t(found);
        }
        const uint64_t sum = block_reduce_sum<kVoxThreads>(uint64_t(__popc(found)), s_red);
        if (threadIdx.x == 0) counts[tile] = uint32_t(sum);
    }
}

// The keys of the voxels whose bit is set, in unit, column and voxel order.
// Without STORED bits (no memory was left for them) the tests are made again.
template <bool STORED>
__global__ __launch_bounds__(kVoxThreads) void k_vox_write(const TriSetup* __restrict__ setup, RowTable R,
                                                           const uint64_t* __restrict__ tile_row,
                                                           const uint64_t* __restrict__ total_ptr, int64_t side,
                                                           const uint16_t* __restrict__ bits,
                                                           const uint64_t* __restrict__ tile_offsets,
                                                           uint64_t* __restrict__ keys)
{
    constexpr uint64_t kThirds = 0x1249249249249249ull;
    __shared__ uint32_t s_scan[kVoxThreads / kWave];
    __shared__ uint64_t s_keys[kVoxThreads * 2 * kUnitCols];
    const uint64_t total = *total_ptr;
    const uint64_t ntiles = (total + kVoxThreads - 1) / kVoxThreads;
    for (uint64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const uint64_t g = tile * kVoxThreads + threadIdx.x;
        uint32_t left = 0;
        if constexpr (STORED) {
            if (g < total) left = bits[g];
        } else {
            const Unit U = unit_of(R, tile_row, total, tile);
            if (U.cols) left = unit_bits(setup[U.tri], U, side);
        }
        uint32_t tile_keys;
        uint32_t o = block_exclusive_scan<kVoxThreads>(uint32_t(__popc(left)), s_scan, tile_keys);
        if (left) {
            const Unit U = unit_of(R, tile_row, total, tile);
            const TriSetup& S = setup[U.tri];
            const int a = S.a, u = S.u, w = S.w;
            const double cu = double(int64_t(U.u)) + 0.5;
            const double q = S.nd - pick3(S.n, u) * cu, nw = pick3(S.n, w), na = pick3(S.n, a);
            const uint64_t row = split_by_3(U.u) << (2 - u);
            uint64_t col = split_by_3(U.w0);
#pragma unroll 1
            for (uint32_t i = 0; left; ++i, left >>= 2, col = ((col | ~kThirds) + 1) & kThirds) {
                if (!(left & 3u)) continue;
                const double cw = double(int64_t(U.w0) + i) + 0.5;
                int32_t lo, hi;
                column_range((q - nw * cw) / na, side, lo, hi);
                const uint64_t rc = row | col << (2 - w);
                if (left & 1u) s_keys[o++] = rc | split_by_3(uint32_t(lo)) << (2 - a);
                if (left & 2u) s_keys[o++] = rc | split_by_3(uint32_t(lo) + 1) << (2 - a);
            }
        }
        __syncthreads();
        uint64_t* const dst = keys + tile_offsets[tile];
        for (uint32_t j = threadIdx.x; j < tile_keys; j += kVoxThreads) dst[j] = s_keys[j];
        __syncthreads();  // s_keys is rewritten by the next tile
    }
}

}  // namespace

void launch_tri_setup(hipStream_t s, const double* tris, uint64_t n_tris, int depth, TriSetup* setup, uint32_t* rows,
                      uint64_t* rect_columns, unsigned long long* err)
{
    if (n_tris == 0) return;
    TimedLaunch t(kKVoxSetup, s);
    hipLaunchKernelGGL(k_tri_setup, dim3(uint32_t((n_tris + kVoxThreads - 1) / kVoxThreads)), dim3(kVoxThreads), 0, s,
                       tris, n_tris, int64_t(1) << depth, setup, rows,
                       reinterpret_cast<unsigned long long*>(rect_columns), err);
}

void launch_row_setup(hipStream_t s, const TriSetup* setup, const uint64_t* row_off, const uint64_t* n_tris_dev,
                      const uint64_t* n_rows_dev, uint64_t n_rows, const VoxRows& rows, uint32_t* tile_units,
                      uint64_t* tile_off, uint64_t* total_units_dev, unsigned long long* err)
{
    if (n_rows == 0) return;
    const uint32_t grid = uint32_t(std::min<uint64_t>((n_rows + kVoxTile - 1) / kVoxTile, device_cu_count() * 8ull));
    {
        TimedLaunch t(kKVoxSetup, s);
        hipLaunchKernelGGL(k_row_setup, dim3(grid), dim3(kVoxThreads), 0, s, setup, row_off, n_tris_dev, n_rows_dev,
                           rows.tri, rows.u, rows.w0, rows.cols, tile_units, err);
    }
    launch_scan_counts(s, tile_units, tile_off, n_rows_dev, kVoxTile, total_units_dev);
    TimedLaunch t(kKVoxSetup, s);
    hipLaunchKernelGGL(k_row_offsets, dim3(grid), dim3(kVoxThreads), 0, s, rows.cols, tile_off, n_rows_dev,
                       rows.unit_off);
}

void launch_vox_count(hipStream_t s, const TriSetup* setup, const VoxRows& rows, const uint64_t* n_rows_dev,
                      const uint64_t* total_units_dev, uint64_t total_units, int depth, uint64_t* tile_row,
                      uint16_t* bits, uint32_t* tile_counts)
{
    TimedLaunch t(kKVoxCount, s);
    const uint64_t tiles = (total_units + kVoxThreads - 1) / kVoxThreads;
    hipLaunchKernelGGL(k_tile_rows, dim3(uint32_t((tiles + kVoxThreads) / kVoxThreads)), dim3(kVoxThreads), 0, s,
                       rows.unit_off, n_rows_dev, total_units_dev, tile_row);
    const RowTable R{rows.tri, rows.u, rows.w0, rows.cols, rows.unit_off};
    hipLaunchKernelGGL(k_vox_count, dim3(resident_grid(k_vox_count, kVoxThreads, tiles)), dim3(kVoxThreads), 0, s, setup,
                       R, tile_row, total_units_dev, int64_t(1) << depth, bits, tile_counts);
}

void launch_vox_write(hipStream_t s, const TriSetup* setup, const VoxRows& rows, const uint64_t* tile_row,
                      const uint64_t* total_units_dev, uint64_t total_units, int depth, const uint16_t* bits,
                      const uint64_t* tile_offsets, uint64_t* keys)
{
    TimedLaunch t(kKVoxWrite, s);
    const uint64_t tiles = (total_units + kVoxThreads - 1) / kVoxThreads;
    const RowTable R{rows.tri, rows.u, rows.w0, rows.cols, rows.unit_off};
    auto run = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(resident_grid(kernel, kVoxThreads, tiles)), dim3(kVoxThreads), 0, s, setup, R,
                           tile_row, total_units_dev, int64_t(1) << depth, bits, tile_offsets, keys);
    };
    if (bits) run(k_vox_write<true>);
    else run(k_vox_write<false>);
}

}  // namespace svdag
