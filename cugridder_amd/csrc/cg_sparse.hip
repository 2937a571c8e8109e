// W-stacking gridding of sparse uv coverage: F[p][y][x] = sum_j c_j psi(x - gx_j)
// psi(y - gy_j) psi(p - gz_j) (src/fourier/conv.cu:522-627), every cell written
// once, in registers.
//
// A wave owns an 8 x 8 block of grid cells of 16 planes and accumulates it as
// FP64 matrix products over the points that reach it,
//   D[plane][cell] = sum_k (v_k psi_z,k(plane)) (psi_x,k psi_y,k)(cell),
// four points per v_mfma_f64_16x16x4f64 (A[i][k] from lane i + 16 k, B[k][j]
// from lane j + 16 k, D[4 v + l / 16][l % 16] in lane l, register v), four
// 16-cell products (two rows of the block each) for the real and four for
// the imaginary part.  The points of the bins whose footprints can reach the
// block are read as one list, 64 at a time; those that reach the block and
// its planes are compacted into an LDS queue (ballot + prefix count: the
// order and the sums are reproducible).  Each lane then evaluates two kernel
// values per four points (one along x or y, one along z), the others arrive
// by lane shuffles.  Kernel values and products with them are in the
// caller's precision, the sums in FP64.
//
// Bound by writing the planes where points are few: 10^6 rows at eps 1e-12
// over 4096 x 4096 x 194 complex128 cells take 12.5 ms, 52 GB at 4.2 TB/s (one
// thread per point adding its 13^3 taps to an LDS tile with atomics: 274 ms,
// the 34 points of a tile on 512 threads); 2500 x 3000 x 10 complex64 cells
// with 196608 points 0.18 ms (0.52 ms).  Around crowded blocks by the chain of
// one wave: 0.14 us per point, 0.55 us per four (their 512 cycles of matrix
// instructions, and the latency of evaluating their kernel values); where k_grid is
// faster such regions are left to it.
#include <type_traits>

#include "cg_kernel.hpp"

namespace cg {

constexpr int kWin = 16;     // planes per window
constexpr int kSpWaves = 4;  // independent waves per workgroup
// bins that reach a block: along an axis at most ceil((kBlk + kw - 2) / tile)
// + 1 of tiles of at least two cells, kw <= 16
constexpr int kSpBins = 13 * 13;
constexpr int kSpQueue = 68;  // queued points: < 4 carried + 64 new

typedef double v4d __attribute__((ext_vector_type(4)));

template <typename T>
struct SparseQueue {
    T gx[kSpQueue], gy[kSpQueue], gz[kSpQueue];  // offset of the first tap from the point
    T vr[kSpQueue], vi[kSpQueue];
    int xs[kSpQueue], ys[kSpQueue], zs[kSpQueue];  // first tap relative to the block / window, in [0, n)
    int pre[kSpBins], beg[kSpBins];                // list position and first point of each bin
    int nbins;
    unsigned short ox[kSpBins], oy[kSpBins];       // bin origin relative to the block, in [0, n)
};

// the bins b0, b0 + 1, ... (nb of them, cyclic in nt bins of t cells over an
// axis of n) holding the start cells lo .. lo + len - 1 (lo may be negative)
struct AxisBins {
    int b0, nb;
};
__device__ __forceinline__ AxisBins axis_bins(int lo, int len, int n, int t, int nt)
{
    if (len >= n) return AxisBins{0, nt};
    const int l = lo < 0 ? lo + n : lo;
    const int h = lo + len - 1;  // < n by construction
    const int bl = l / t, bh = h / t;
    if (l <= h) return AxisBins{bl, bh - bl + 1};
    // wraps past the end of the axis
    return bl <= bh ? AxisBins{0, nt} : AxisBins{bl, bh + nt - bl + 1};
}

// Work items (block, window), window fastest, one per wave.  kSpRun rounds of
// a workgroup in a row are contiguous on one XCD: adjacent blocks' bins and
// the two halves of a 128-byte line meet in one L2, and crowded regions of the
// uv plane still spread over all eight (one contiguous eighth of the grid per
// XCD, with complex64 stores non-temporal besides: 0.46 ms where this takes
// 0.18 ms).
constexpr int kSpRun = 16;

// NQ row pairs of the block at a time: all four, or (NQ = 1) each on its own
// wave
template <typename T, int NQ>
__device__ __forceinline__ void grid_blocks(SparseQueue<T> &Q, const geo_t<T> *__restrict__ geo,
                                            const cx_t<T> *__restrict__ val,
                                            const int32_t *__restrict__ tile_start,
                                            cx_t<T> *__restrict__ fw, const GridArgs &g, int kw, int nbx,
                                            int64_t nitem, int nwin)
{
    constexpr int ROWS = 2 * NQ, PARTS = kBlk / ROWS;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int k = lane >> 4, r = lane & 15;
    const KernelEval<T> ker(g, kw);
    const int zn = slab_planes(g);
    struct Item {
        int x0, y0, p0, np;
    };
    auto item_at = [&](int64_t it) {
        const int64_t bw = it / PARTS;
        const int bi = (int)(bw / nwin), win = (int)(bw - (int64_t)bi * nwin);
        const int block = __builtin_amdgcn_readfirstlane(g.tile_list ? g.tile_list[1 + bi] : bi);
        const int by = block / nbx, bx = block - by * nbx, p0 = g.zb + win * kWin;
        return Item{bx * kBlk, by * kBlk + ROWS * (int)(it % PARTS), p0, min(kWin, g.zb + zn - p0)};
    };
    // the bins that reach the block, as one list of points: returns its length
    auto list_points = [&](const Item &I) -> int {
        const AxisBins X = axis_bins(I.x0 - (kw - 1), min(kBlk, g.nf1 - I.x0) + kw - 1, g.nf1, g.tx, g.ntx);
        const AxisBins Y = axis_bins(I.y0 - (kw - 1), min(ROWS, g.nf2 - I.y0) + kw - 1, g.nf2, g.ty, g.nty);
        const int nbins = X.nb * Y.nb;
        int total = 0;
        for (int c0 = 0; c0 < nbins; c0 += 64) {
            const int b = c0 + lane;
            int n = 0;
            if (b < nbins) {
                const int jy = b / X.nb, jx = b - jy * X.nb;
                int tby = Y.b0 + jy, tbx = X.b0 + jx;
                if (tby >= g.nty) tby -= g.nty;
                if (tbx >= g.ntx) tbx -= g.ntx;
                const int tile = tby * g.ntx + tbx;
                const int beg = tile_start[tile];
                n = tile_start[tile + 1] - beg;
                // dense bins are added afterwards by k_grid_dense2
                if (g.dense_min > 0 && n >= g.dense_min) n = 0;
                int ox = tbx * g.tx - I.x0, oy = tby * g.ty - I.y0;
                if (ox < 0) ox += g.nf1;
                if (oy < 0) oy += g.nf2;
                Q.beg[b] = beg;
                Q.ox[b] = (unsigned short)ox;
                Q.oy[b] = (unsigned short)oy;
            }
            int s = n;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const int t = __shfl_up(s, d);
                if (lane >= d) s += t;
            }
            if (b < nbins) Q.pre[b] = total + s - n;
            total += __builtin_amdgcn_readfirstlane(__shfl(s, 63));
        }
        if (lane == 0) Q.nbins = nbins;
        wave_lds_sync();
        return total;
    };

    v4d cre[NQ], cim[NQ];
    // one product over queued points e0 .. e0 + 3: the lane's kernel values ...
    struct Operand {
        T e1;           // along x (r < 8) or y
        double ar, ai;  // along z, times the strength
    };
    auto operand = [&](int e0) {
        const int e = e0 + k;
        const bool isx = r < 8;
        // tap index of the lane's position: position minus start, cyclic
        int t1 = (r & 7) - (isx ? Q.xs[e] : Q.ys[e]);
        if (t1 < 0) t1 += isx ? g.nf1 : g.nf2;
        int t2 = r - Q.zs[e];
        if (t2 < 0) t2 += g.nf3;
        const T o1 = isx ? Q.gx[e] : Q.gy[e], oz = Q.gz[e];
        Operand A;
        A.e1 = t1 < kw ? ker(o1, t1) : (T)0;
        const T e2 = t2 < kw ? ker(oz, t2) : (T)0;
        A.ar = (double)(Q.vr[e] * e2);
        A.ai = (double)(Q.vi[e] * e2);
        return A;
    };
    // ... and the eight matrix instructions
    auto multiply = [&](const Operand &A) {
        const T ex = __shfl(A.e1, 16 * k + (r & 7));
#pragma unroll
        for (int q = 0; q < NQ; q++) {
            const T ey = __shfl(A.e1, 16 * k + 8 + 2 * q + (r >> 3));
            const double w = (double)(ex * ey);
            cre[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(A.ar, w, cre[q], 0, 0, 0);
            cim[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(A.ai, w, cim[q], 0, 0, 0);
        }
    };
    // the products of the listed points
    auto accumulate = [&](const Item &I, int total) {
#pragma unroll
        for (int q = 0; q < NQ; q++) cre[q] = cim[q] = v4d{0.0, 0.0, 0.0, 0.0};
        const int nbins = Q.nbins;
        int queued = 0;  // wave-uniform, < 4 between chunks
        for (int base = 0; base < total; base += 64) {
            const int i = base + lane;
            bool touch = false;
            int rx = 0, ry = 0, rz = 0;
            geo_t<T> G{};
            cx_t<T> v{};
            if (i < total) {
                // last bin b with pre[b] <= i (empty bins before it share its position)
                int lo = 0, hi = nbins;
                while (hi - lo > 1) {
                    const int mid = (lo + hi) >> 1;
                    if (Q.pre[mid] <= i) lo = mid;
                    else hi = mid;
                }
                const int idx = Q.beg[lo] + i - Q.pre[lo];
                G = geo[idx];
                v = val[idx];
                const uint32_t pk = geo_bits(G.w);
                rx = Q.ox[lo] + (int)(pk & 0xffu);
                if (rx >= g.nf1) rx -= g.nf1;
                ry = Q.oy[lo] + (int)((pk >> 8) & 0xffu);
                if (ry >= g.nf2) ry -= g.nf2;
                rz = (int)(pk >> 16) - I.p0;
                if (rz < 0) rz += g.nf3;
                touch = (rx < kBlk || rx + kw > g.nf1) && (ry < ROWS || ry + kw > g.nf2) &&
                        (rz < I.np || rz + kw > g.nf3);
            }
            const uint64_t mask = __ballot(touch);
            if (!mask) continue;
            if (touch) {
                const int pos = queued + (int)__popcll(mask & ((1ull << lane) - 1ull));
                Q.xs[pos] = rx;
                Q.ys[pos] = ry;
                Q.zs[pos] = rz;
                Q.gx[pos] = G.x;
                Q.gy[pos] = G.y;
                Q.gz[pos] = G.z;
                Q.vr[pos] = v.x;
                Q.vi[pos] = v.y;
            }
            wave_lds_sync();
            queued += (int)__popcll(mask);
            const int full = queued & ~3;
            int e0 = 0;
            // complex64 has the registers for two products in flight
            if constexpr (sizeof(T) == 4)
                for (; e0 + 8 <= full; e0 += 8) {
                    const Operand A = operand(e0), B = operand(e0 + 4);
                    multiply(A);
                    multiply(B);
                }
            for (; e0 < full; e0 += 4) multiply(operand(e0));
            const int rest = queued - full;
            if (rest && full && lane < rest) {
                // carry the last (< 4) queued points to the front (source
                // entries >= 4, destinations < 3: the ranges are disjoint)
                const int src = full + lane;
                Q.xs[lane] = Q.xs[src];
                Q.ys[lane] = Q.ys[src];
                Q.zs[lane] = Q.zs[src];
                Q.gx[lane] = Q.gx[src];
                Q.gy[lane] = Q.gy[src];
                Q.gz[lane] = Q.gz[src];
                Q.vr[lane] = Q.vr[src];
                Q.vi[lane] = Q.vi[src];
            }
            queued = rest;
            wave_lds_sync();
        }
        if (queued) {
            // pad the last step with points of no strength
            if (lane >= queued && lane < 4) {
                Q.xs[lane] = Q.ys[lane] = Q.zs[lane] = 0;
                Q.gx[lane] = Q.gy[lane] = Q.gz[lane] = (T)0;
                Q.vr[lane] = Q.vi[lane] = (T)0;
            }
            wave_lds_sync();
            multiply(operand(0));
        }
        wave_lds_sync();  // the tables are rebuilt for the next item
    };
    const int xcd = blockIdx.x & 7;
    for (int64_t j = blockIdx.x >> 3;; j += gridDim.x >> 3) {
        const int64_t it = ((j / kSpRun * 8 + xcd) * kSpRun + j % kSpRun) * kSpWaves + wave;
        if (it >= nitem * PARTS) break;  // it grows with j; the waves share no barrier
        const Item I = item_at(it);
        if (I.y0 >= g.nf2) continue;
        accumulate(I, list_points(I));
        // lane l holds planes 4 v + l / 16 of cell l % 16 of each row pair
        const int x = I.x0 + (r & 7);
        if (x >= g.nf1) continue;
#pragma unroll
        for (int q = 0; q < NQ; q++) {
            const int y = I.y0 + 2 * q + (r >> 3);
            if (y >= g.nf2) continue;
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int p = 4 * v + k;
                if (p >= I.np) continue;
                cx_t<T> *dst = fw + ((size_t)(I.p0 - g.zb + p) * g.nf2 + y) * g.nf1 + x;
                // whole 128-byte lines only in complex128
                if constexpr (sizeof(T) == 8) store_nt(dst, mkc(cre[q][v], cim[q][v]));
                else *dst = mkc((T)cre[q][v], (T)cim[q][v]);
            }
        }
    }
}

// With at most kSpSplit blocks a block's four row pairs are separate work: the
// time is then that of the most crowded block on one wave (a 2000-row snapshot
// on 192 x 256 x 12 cells: 27.4 us whole, 14.2 us split).
constexpr int kSpSplit = 2048;

template <typename T>
__global__ __launch_bounds__(64 * kSpWaves, 3) void k_grid_sparse(const geo_t<T> *__restrict__ geo,
                                                                 const cx_t<T> *__restrict__ val,
                                                                 const int32_t *__restrict__ tile_start,
                                                                 cx_t<T> *__restrict__ fw, GridArgs g,
                                                                 int kw, int nbx, int nblocks, int nwin)
{
    __shared__ SparseQueue<T> Qs[kSpWaves];
    SparseQueue<T> &Q = Qs[__builtin_amdgcn_readfirstlane(threadIdx.x >> 6)];
    const int64_t nitem = (int64_t)(g.tile_list ? g.tile_list[0] : nblocks) * nwin;
    if (nitem <= kSpSplit) grid_blocks<T, 1>(Q, geo, val, tile_start, fw, g, kw, nbx, nitem, nwin);
    else grid_blocks<T, 4>(Q, geo, val, tile_start, fw, g, kw, nbx, nitem, nwin);
}

// list[0] = number of 8 x 8 blocks with a masked-in row and a masked-in
// column (all without masks), list[1..] = those blocks (any order; each is
// gridded independently).  With crowd_min > 0 the blocks of a crowded region go
// to crowd_list as its sort tiles instead.  A region is a block, or the sort tile
// if that is larger (edges along an axis divide one another), and the points of
// all bins that can reach it count, those of the dense path aside.
__global__ __launch_bounds__(256) void k_need_blocks(const int32_t *__restrict__ tile_start, int nbx,
                                                     int nblocks, GridArgs g, int kw,
                                                     int32_t *__restrict__ list)
{
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= nblocks) return;
    const int by = t / nbx, bx = t - by * nbx;
    const int x0 = bx * kBlk, x1 = min(x0 + kBlk, g.nf1), y0 = by * kBlk, y1 = min(y0 + kBlk, g.nf2);
    auto wanted = [&](int xa, int xb, int ya, int yb) -> bool {
        bool row = !g.rowmask, col = !g.rowmask;
        for (int y = ya; y < yb && !row; y++) row = g.rowmask[y] != 0;
        for (int x = xa; x < xb && !col; x++) col = g.colmask[x] != 0;
        return row && col;
    };
    if (g.crowd_min > 0) {
        const int ex = max(kBlk, g.tx), ey = max(kBlk, g.ty), rx = x0 / ex * ex, ry = y0 / ey * ey;
        const int nx = min(ex, g.nf1 - rx), ny = min(ey, g.nf2 - ry);
        if (!wanted(rx, rx + nx, ry, ry + ny)) return;
        const AxisBins X = axis_bins(rx - (kw - 1), nx + kw - 1, g.nf1, g.tx, g.ntx);
        const AxisBins Y = axis_bins(ry - (kw - 1), ny + kw - 1, g.nf2, g.ty, g.nty);
        int64_t n = 0;
        for (int j = 0; j < Y.nb; j++)
            for (int i = 0; i < X.nb; i++) {
                int ty = Y.b0 + j, tx = X.b0 + i;
                if (ty >= g.nty) ty -= g.nty;
                if (tx >= g.ntx) tx -= g.ntx;
                const int bin = ty * g.ntx + tx, c = tile_start[bin + 1] - tile_start[bin];
                if (g.dense_min <= 0 || c < g.dense_min) n += c;
            }
        if (n >= g.crowd_min) {
            // the tiles that begin in this block
            for (int ty = (y0 + g.ty - 1) / g.ty; ty * g.ty < y1; ty++)
                for (int tx = (x0 + g.tx - 1) / g.tx; tx * g.tx < x1; tx++)
                    g.crowd_list[1 + atomicAdd(g.crowd_list, 1)] = ty * g.ntx + tx;
            return;
        }
    }
    if (wanted(x0, x1, y0, y1)) list[1 + atomicAdd(list, 1)] = t;
}

int64_t sparse_blocks(int nf1, int nf2)
{
    return ceil_div(nf1, kBlk) * ceil_div(nf2, kBlk);
}

// the blocks and the sort tiles of a crowded region cover the same cells
bool sparse_crowdable(const GridArgs &g)
{
    auto fits = [](int t) { return t % kBlk == 0 || kBlk % t == 0; };
    return fits(g.tx) && fits(g.ty);
}

template <typename T>
int launch_grid_sparse(const geo_t<T> *geo, const cx_t<T> *val, const int32_t *ts, cx_t<T> *fw,
                       const GridArgs &g, int kw, hipStream_t s)
{
    if (kw < 2 || kw > kMaxKW || g.nf1 < 2 * kw || g.nf2 < 2 * kw || g.nf3 < 2 * kw || g.tx < 2 ||
        g.ty < 2 || g.nf1 > 65536 || g.nf2 > 65536)
        return CG_ERR_ARG;
    const int nbx = (int)ceil_div(g.nf1, kBlk);
    const int64_t nblocks = sparse_blocks(g.nf1, g.nf2);
    const int nwin = (int)ceil_div(slab_planes(g), kWin);
    if (g.crowd_min > 0 && (!g.tile_list || !g.crowd_list || !sparse_crowdable(g))) return CG_ERR_ARG;
    if (g.tile_list && g.zb == 0) {
        hipLaunchKernelGGL(k_need_blocks, dim3((unsigned)ceil_div(nblocks, 256)), dim3(256), 0, s, ts, nbx,
                           (int)nblocks, g, kw, g.tile_list);
        CG_HIP(hipGetLastError());
    }
    // (a short list, split by row pairs, has four times as many items)
    const int64_t wgs = ceil_div(nblocks * nwin * 4, kSpWaves);
    const unsigned grid = (unsigned)std::min<int64_t>(ceil_div(wgs, 8) * 8, 256 * 8);
    hipLaunchKernelGGL(k_grid_sparse<T>, dim3(grid), dim3(64 * kSpWaves), 0, s, geo, val, ts, fw, g,
                       kw, nbx, (int)nblocks, nwin);
    CG_HIP(hipGetLastError());
    return CG_OK;
}

// ------------------------------------------------------------ degridding
//
// Tiles with few points: each point is interpolated straight from the planes
// in HBM / L2, G lanes (8 or 16) per point, lane t holding tap t along the
// fast axis, so a row of the footprint is one contiguous read of the group;
// the KW rows of a plane are in flight together.  Staging such a tile in LDS
// would read its whole halo, and one thread per point leaves most of a
// workgroup idle.  A wave takes one unit (k_tile_units) at a time; units are
// short, so that the last ones do not leave the GPU waiting.  Bound by the
// plane reads where points are few: 10^6 rows at eps 1e-12 over 4096 x 4096 x
// 194 complex128 cells (15 points per 16 x 16 tile) take 8 ms, staged 124 ms.
constexpr int kDirWaves = 4;

constexpr int direct_lanes(int kw) { return kw <= 8 ? 8 : 16; }
constexpr int kDirSteps = 2;  // steps (64 / G points each) per unit
int degrid_direct_unit(int kw) { return kDirSteps * (64 / direct_lanes(kw)); }

template <typename T, int KW>
__global__ __launch_bounds__(64 * kDirWaves) void k_degrid_direct(const geo_t<T> *__restrict__ geo,
                                                                  const cx_t<T> *__restrict__ fac,
                                                                  const int32_t *__restrict__ perm,
                                                                  const int32_t *__restrict__ tile_start,
                                                                  const cx_t<T> *__restrict__ fw,
                                                                  cx_t<T> *__restrict__ out, GridArgs g,
                                                                  const int32_t *__restrict__ list)
{
    constexpr int G = direct_lanes(KW), PW = 64 / G, UNIT = kDirSteps * PW;
    // planes in flight: all of a narrow complex64 footprint
    constexpr int UZ = sizeof(T) == 4 && KW <= 8 ? KW : 1;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int gl = lane & (G - 1);
    const KernelEval<T> ker(g, KW);
    const int zn = slab_planes(g);
    const size_t plane = (size_t)g.nf1 * g.nf2;
    const int xcd = blockIdx.x & 7, nunit = list[0];
    // units dealt to the XCDs in contiguous runs, as in k_grid_sparse
    for (int64_t j = blockIdx.x >> 3;; j += gridDim.x >> 3) {
        const int64_t e = ((j / kSpRun * 8 + xcd) * kSpRun + j % kSpRun) * kDirWaves + wave;
        if (e >= nunit) break;  // e grows with j; the waves share no barrier
        const int tile = list[2 + 2 * e];
        const int beg = tile_start[tile] + list[3 + 2 * e], end = min(tile_start[tile + 1], beg + UNIT);
        const int by = tile / g.ntx, bx = tile - by * g.ntx;
        for (int i0 = beg; i0 < end; i0 += PW) {
            const int i = i0 + lane / G;
            const bool ok = i < end;
            const geo_t<T> R = geo[ok ? i : i0];
            const uint32_t pk = geo_bits(R.w);
            const T kx = gl < KW ? ker(R.x, gl) : (T)0;
            const T kyl = gl < KW ? ker(R.y, gl) : (T)0;
            const T kzl = gl < KW ? ker(R.z, gl) : (T)0;
            int x = bx * g.tx + (int)(pk & 0xffu) + gl;
            if (x >= g.nf1) x -= g.nf1;
            const int y0 = by * g.ty + (int)((pk >> 8) & 0xffu);
            T ky[KW];
            int off[KW];
#pragma unroll
            for (int t = 0; t < KW; t++) {
                ky[t] = __shfl(kyl, t, G);
                int y = y0 + t;
                if (y >= g.nf2) y -= g.nf2;
                off[t] = y * g.nf1 + x;
            }
            const bool rd = ok && gl < KW;
            T ar = 0, ai = 0;
            int p = (int)(pk >> 16) - g.zb;  // plane in the buffer
#pragma unroll UZ
            for (int tz = 0; tz < KW; tz++, p++) {
                if (p + g.zb >= g.nf3) p -= g.nf3;
                const T kz = __shfl(kzl, tz, G);
                T sr = 0, si = 0;
                if (rd && p >= 0 && p < zn) {
                    const cx_t<T> *src = fw + (size_t)p * plane;
                    cx_t<T> f[KW];
#pragma unroll
                    for (int t = 0; t < KW; t++) f[t] = src[off[t]];
#pragma unroll
                    for (int t = 0; t < KW; t++) {
                        sr += f[t].x * ky[t];
                        si += f[t].y * ky[t];
                    }
                }
                ar += sr * kz;
                ai += si * kz;
            }
            ar *= kx;
            ai *= kx;
#pragma unroll
            for (int d = 1; d < G; d <<= 1) {
                ar += __shfl_xor(ar, d);
                ai += __shfl_xor(ai, d);
            }
            if (ok && gl == 0) {
                const cx_t<T> f = fac[i];
                const int dst = perm[i];
                if (dst >= 0 && dst < g.m) {  // a valid permutation always passes
                    cx_t<T> v = mkc(ar * f.x - ai * f.y, ar * f.y + ai * f.x);
                    if (g.accumulate) {
                        const cx_t<T> prev = out[dst];
                        v.x += prev.x;
                        v.y += prev.y;
                    }
                    out[dst] = v;
                }
            }
        }
    }
}

template <typename T>
int launch_degrid_direct(const geo_t<T> *geo, const cx_t<T> *fac, const int32_t *perm,
                         const int32_t *ts, const cx_t<T> *fw, cx_t<T> *out, const GridArgs &g, int kw,
                         const DegridLists &L, hipStream_t s)
{
    if (g.nf1 < 2 * kw || g.nf2 < 2 * kw || g.nf3 < 2 * kw) return CG_ERR_ARG;
    const int64_t wgs = ceil_div(L.max_direct, kDirWaves);
    const unsigned grid = (unsigned)std::min<int64_t>(ceil_div(wgs, 8) * 8, 256 * 8);
    switch (kw) {
#define CG_CASE(K)                                                                                   \
    case K:                                                                                          \
        hipLaunchKernelGGL((k_degrid_direct<T, K>), dim3(grid), dim3(64 * kDirWaves), 0, s, geo, fac, \
                           perm, ts, fw, out, g, L.direct);                                         \
        break;
        CG_CASE(2) CG_CASE(3) CG_CASE(4) CG_CASE(5) CG_CASE(6) CG_CASE(7) CG_CASE(8) CG_CASE(9)
        CG_CASE(10) CG_CASE(11) CG_CASE(12) CG_CASE(13) CG_CASE(14) CG_CASE(15) CG_CASE(16)
#undef CG_CASE
    default: return CG_ERR_ARG;
    }
    CG_HIP(hipGetLastError());
    return CG_OK;
}

template int launch_degrid_direct<float>(const float4 *, const float2 *, const int32_t *, const int32_t *, const float2 *, float2 *, const GridArgs &, int, const DegridLists &, hipStream_t);
template int launch_degrid_direct<double>(const double4 *, const double2 *, const int32_t *, const int32_t *, const double2 *, double2 *, const GridArgs &, int, const DegridLists &, hipStream_t);
template int launch_grid_sparse<float>(const float4 *, const float2 *, const int32_t *, float2 *, const GridArgs &, int, hipStream_t);
template int launch_grid_sparse<double>(const double4 *, const double2 *, const int32_t *, double2 *, const GridArgs &, int, hipStream_t);

}  // namespace cg
