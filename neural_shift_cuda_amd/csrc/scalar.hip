// scalar.hip -- accumulate_uz_scalar (GASD scalar-per-transform weights).
//
// Semantics (reference csrc/shift_ops_cuda.cu:806-980, ops.py:350-390):
//   U[b,c,p]  = sum_s w[s,b,c] x[b,c,(p+s) mod]        Z[b,c,p] = sum_s w[s,b,c]
//   gx[q]     = sum_s w[s,b,c] gU[(q-s) mod]
//   gw[s,b,c] = sum_{p} gU[p] x[(p+s) mod] + gZ[p]
// The weights are tiny (S*B*C) and x, gU are re-read S times, so the op is
// bound by the vector ALU (one FMA per pixel and shift and pass) and, if
// every FMA takes its own LDS read, by LDS.  One workgroup (four waves) owns
// a 64 x 32 tile of one (b, c) plane; the tile of x (or gU) with a kRmax halo
// sits in LDS, a lane owns one column and a wave reads 64 consecutive words
// of a row, free of bank conflicts.
//
// Tables are mostly dense windows, so the rows near enough for the LDS tile
// are laid out as a grid of (dy, dx) over their bounding box (SGrid) and a
// lane walks the grid column by column: P + 3 values of its column serve four
// neighbouring dx of its P pixels (11 LDS reads for 32 FMAs; 35 for 128 in
// gw), instead of one LDS read and a share of the row's decoding per FMA.
// Tables that repeat a row or fill less than half of their box (a walk of the
// whole box would then read more than the row-by-row loop) take the
// row-by-row loop, as do rows beyond the halo (from global memory).  16 x 3 x
// 256^2, 121 rows, fp32, row by row -> grid: forward 64 -> 31 us, gx 62 -> 30
// us, gw 79 -> 28 us (0.76 GFLOP a pass: 10 us at the vector ALU's rate; the
// rest is mostly the tile's prologue, one round of workgroups).
//
// gw is a deterministic two-level reduction: a wave forms, for its share of
// the shifts, the sum over the tile's pixels of gU[p] x[p+s] + gZ[p] (lane
// sums over 32 rows, then a wave64 DPP reduction) into a caller workspace of
// S*B*C*ntiles partials, and a second kernel adds the tiles of each
// (s, b, c) in index order.
#include <initializer_list>
#include <type_traits>

#include "nsh_common.hpp"
#include "scatter.hpp"

namespace nsh {

constexpr int kScTW = 64;   // tile columns: one per lane of a wave
constexpr int kScTH = 32;   // tile rows
constexpr int kScWaves = 4;
constexpr int kScThreads = 64 * kScWaves;
constexpr int kScP = kScTH / kScWaves;  // rows per lane of the forward and gx
constexpr int kScPitch = kScTW + 2 * kRmax;
constexpr int kScLH = kScTH + 2 * kRmax;
constexpr int kScChunk = 4;  // neighbouring dx taken from one set of column values
// rows a chunk's column values may reach past the halo (never used there)
constexpr int kScPad = kScChunk - 1;
constexpr int kScTile = (kScLH + kScPad) * kScPitch;
constexpr int kScBatch = 4;  // rows in flight where the table is no grid

// The table's near rows (|dx|, |dy| <= kRmax) as a grid over their bounding
// box: cell (dyi, dxi) holds the table row of displacement (dx0 + dxi,
// dy0 + dyi).  SGN = -1 grids the negated displacements (gx reads q - s).
constexpr int kScBox = 2 * kRmax + 1;
constexpr int kScChunks = (kScBox + kScChunk - 1) / kScChunk;
constexpr int kScRow = kScChunks * kScChunk;  // cells of a grid row, whole chunks
struct SGrid {
    int dx0, n, dy0, m;  // first displacement and extent in dx and dy
    bool dense;          // every near row has its own cell, at least half of them taken
    int single, far;     // near rows outside the grid (all of them or none), rows beyond the halo
};

// Builds the grid in `cell` (m rows of kScRow; -1: empty) from the staged
// table, and the table's far and near rows in order as lists: far row k at
// list[k], near row k at list[S - 1 - k]; ends with a barrier.  A table of a
// few rows is not worth a grid (one row, 16 x 3 x 256^2 fp64: the forward took
// 20 us with it, 15 without).
constexpr int kScGridRows = 5;

template <int SGN>
__device__ __forceinline__ SGrid stage_grid(const int4* shl, int S, int* cell, int* list) {
    const int lane = threadIdx.x & 63;
    if (S >= kScGridRows)
        for (int i = threadIdx.x; i < kScBox * kScRow; i += blockDim.x) cell[i] = -1;
    // extent and number of the near rows, by every wave for itself
    int lox = kRmax, hix = -kRmax, loy = kRmax, hiy = -kRmax, near = 0, nlist = 0, flist = 0;
    for (int s0 = 0; s0 < S; s0 += 64) {
        const int s = s0 + lane;
        const bool row = s < S;
        const int dx = row ? SGN * shl[s].x : 0, dy = row ? SGN * shl[s].y : 0;
        const bool in = row && dx >= -kRmax && dx <= kRmax && dy >= -kRmax && dy <= kRmax;
        const uint64_t nm = __ballot(in), fm = __ballot(row && !in);
        if (threadIdx.x < 64 && row) {
            const uint64_t before = (uint64_t(1) << lane) - 1;
            if (in)
                list[S - 1 - nlist - __popcll(nm & before)] = s;
            else
                list[flist + __popcll(fm & before)] = s;
        }
        nlist += __popcll(nm);
        flist += __popcll(fm);
        if (!in) continue;
        lox = min(lox, dx);
        hix = max(hix, dx);
        loy = min(loy, dy);
        hiy = max(hiy, dy);
        ++near;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        lox = min(lox, __shfl_xor(lox, o, 64));
        hix = max(hix, __shfl_xor(hix, o, 64));
        loy = min(loy, __shfl_xor(loy, o, 64));
        hiy = max(hiy, __shfl_xor(hiy, o, 64));
        near += __shfl_xor(near, o, 64);
    }
    SGrid g;
    g.dx0 = __builtin_amdgcn_readfirstlane(lox);
    g.dy0 = __builtin_amdgcn_readfirstlane(loy);
    g.n = __builtin_amdgcn_readfirstlane(hix) - g.dx0 + 1;
    g.m = __builtin_amdgcn_readfirstlane(hiy) - g.dy0 + 1;
    const int count = __builtin_amdgcn_readfirstlane(near);
    g.dense = S >= kScGridRows && count > 0 && 2 * count >= g.n * g.m;
    g.far = S - count;
    __syncthreads();
    if (g.dense) {
        for (int s = threadIdx.x; s < S; s += blockDim.x) {
            const int dx = SGN * shl[s].x, dy = SGN * shl[s].y;
            if (dx < -kRmax || dx > kRmax || dy < -kRmax || dy > kRmax) continue;
            atomicMax(&cell[(dy - g.dy0) * kScRow + dx - g.dx0], s);
        }
        __syncthreads();
        int taken = 0;  // a repeated row: fewer cells taken than rows
        for (int i = lane; i < g.m * kScRow; i += 64) taken += cell[i] >= 0;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) taken += __shfl_xor(taken, o, 64);
        g.dense = __builtin_amdgcn_readfirstlane(taken) == count;
    }
    g.single = g.dense ? 0 : count;
    return g;
}

// The tile of a plane with its kRmax halo, every load of a lane before its
// first write (15 of them in flight).
template <typename T, typename A>
__device__ __forceinline__ void stage_scalar_tile(A* st, const T* __restrict__ plane, int H, int W,
                                                  int h0, int w0) {
    constexpr int N = kScLH * kScPitch / kScThreads;
    static_assert(N * kScThreads == kScLH * kScPitch, "whole rounds");
    const bool cheap = H >= kScLH && W >= kScPitch;
    T v[N];
#pragma unroll
    for (int i = 0; i < N; ++i)
        v[i] = plane[halo_offset(threadIdx.x + i * kScThreads, kScPitch, h0, w0, H, W, cheap)];
#pragma unroll
    for (int i = 0; i < N; ++i) st[threadIdx.x + i * kScThreads] = to_acc(v[i]);
}

// The weights of the grid's cells (0 in an empty one) and, per chunk of four
// neighbouring dx, which of them are taken.
template <typename A>
__device__ __forceinline__ void stage_grid_weights(const SGrid& g, const int* cell, const A* wl,
                                                   A* kw, int* mask) {
    for (int i = threadIdx.x; i < g.m * kScRow; i += blockDim.x)
        kw[i] = cell[i] >= 0 ? wl[cell[i]] : A(0);
    for (int i = threadIdx.x; i < g.m * kScChunks; i += blockDim.x) {
        int m = 0;
#pragma unroll
        for (int j = 0; j < kScChunk; ++j) m |= cell[i * kScChunk + j] >= 0 ? 1 << j : 0;
        mask[i] = m;
    }
    __syncthreads();
}

// Sum over the 64 lanes of a wave, returned uniform (in every lane).
// fp32: DPP adds (row_shr 1, 2, 4, 8 leave each 16-lane row's sum in its
// lane 15; row_bcast 15 and 31 fold the rows into lane 63), all VALU work;
// fp64: xor butterfly.  The order of additions is fixed.
template <int CTRL, int ROWMASK>
__device__ __forceinline__ float dpp_add(float v) {
    const int moved = __builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, ROWMASK, 0xf, true);
    return v + __int_as_float(moved);
}
__device__ __forceinline__ float wave_sum(float v) {
    v = dpp_add<0x111, 0xf>(v);  // row_shr:1
    v = dpp_add<0x112, 0xf>(v);  // row_shr:2
    v = dpp_add<0x114, 0xf>(v);  // row_shr:4
    v = dpp_add<0x118, 0xf>(v);  // row_shr:8
    v = dpp_add<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
    v = dpp_add<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// MODE 0: forward (src = x, writes U and Z);  MODE 1: gx (src = gU).
template <typename T, int MODE>
__global__ __launch_bounds__(kScThreads, sizeof(acc_t<T>) == 4 ? 8 : 4) void scalar_tile_kernel(
    const void* __restrict__ src_v, const T* __restrict__ w, const int64_t* __restrict__ shifts,
    int cols, int S, int B, int C, int H, int W, int ntw, int nth, void* __restrict__ out0,
    acc_t<T>* __restrict__ out1) {
    using A = acc_t<T>;
    using Src = std::conditional_t<MODE == 0, T, A>;
    constexpr int SGN = MODE == 0 ? 1 : -1;
    constexpr int P = kScP, CH = kScChunk;
    extern __shared__ __align__(16) unsigned char smem[];
    int4* shl = reinterpret_cast<int4*>(smem);
    A* kw = reinterpret_cast<A*>(smem + shift_lds_bytes(S));
    A* st = kw + kScBox * kScRow;
    A* wl = st + kScTile;
    int* cell = reinterpret_cast<int*>(wl + S);
    int* mask = cell + kScBox * kScRow;
    int* list = mask + kScBox * kScChunks;

    const TileIdx ti = tile_of(xcd_tile(blockIdx.x, gridDim.x), ntw, nth, kScTH, kScTW);
    const int64_t HW = static_cast<int64_t>(H) * W;
    const int64_t BC = static_cast<int64_t>(B) * C;
    const Src* src = static_cast<const Src*>(src_v) + ti.bc * HW;
    for (int s = threadIdx.x; s < S; s += blockDim.x) wl[s] = to_acc(w[s * BC + ti.bc]);
    stage_scalar_tile<Src, A>(st, src, H, W, ti.h0, ti.w0);
    stage_shifts(shl, shifts, S, cols, H, W, 0);  // ends with a barrier
    const SGrid g = stage_grid<SGN>(shl, S, cell, list);

    const int col = threadIdx.x & 63;
    const int r0 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) * P;
    const A* own = st + (r0 + kRmax) * kScPitch + col + kRmax;  // pixel i at own + i * pitch
    A u[P];
#pragma unroll
    for (int i = 0; i < P; ++i) u[i] = A(0);
    A z = A(0);  // lane sums of the weights, then the wave's
    if (MODE == 0) {
        for (int s = col; s < S; s += 64) z += wl[s];
        z = wave_sum(z);
    }

    if (g.dense) {
        stage_grid_weights<A>(g, cell, wl, kw, mask);
        const int nch = (g.n + CH - 1) / CH;
        // the next chunk's mask and weights are read one chunk ahead
        int mn = mask[0];
        A wn[CH];
        load_out<A, CH>(kw, wn);
        for (int dyi = 0; dyi < g.m; ++dyi) {
            const A* cv = own + g.dx0 * kScPitch + g.dy0 + dyi;
            for (int c = 0; c < nch; ++c, cv += CH * kScPitch) {
                const int m = __builtin_amdgcn_readfirstlane(mn);
                A v[P + CH - 1], ws[CH];
#pragma unroll
                for (int i = 0; i < P + CH - 1; ++i) v[i] = cv[i * kScPitch];
#pragma unroll
                for (int j = 0; j < CH; ++j) ws[j] = wn[j];
                const int next = c + 1 < nch ? dyi * kScChunks + c + 1
                                             : min(dyi + 1, g.m - 1) * kScChunks;
                mn = mask[next];
                load_out<A, CH>(kw + next * CH, wn);
                // an empty cell is skipped, not weighted by 0 (0 x inf)
                if (m == (1 << CH) - 1) {
#pragma unroll
                    for (int j = 0; j < CH; ++j)
#pragma unroll
                        for (int i = 0; i < P; ++i) u[i] = fma_acc(ws[j], v[i + j], u[i]);
                } else {
#pragma unroll
                    for (int j = 0; j < CH; ++j)
                        if (m & (1 << j))
#pragma unroll
                            for (int i = 0; i < P; ++i) u[i] = fma_acc(ws[j], v[i + j], u[i]);
                }
            }
        }
    }
    // Near rows without a grid, kScBatch at a time: the column values of all of
    // them in flight, the next batch's records read before this one's FMAs.
    if (g.single > 0) {
        int offs[kScBatch];
        A wsn[kScBatch];
        auto rows = [&](int k0) {
#pragma unroll
            for (int j = 0; j < kScBatch; ++j) {
                const int s = list[S - 1 - min(k0 + j, g.single - 1)];
                const int4 r = shl[s];
                offs[j] = __builtin_amdgcn_readfirstlane(SGN * (r.x * kScPitch + r.y));
                wsn[j] = wl[s];
            }
        };
        rows(0);
        for (int k0 = 0; k0 < g.single; k0 += kScBatch) {
            A v[kScBatch][P], ws[kScBatch];
#pragma unroll
            for (int j = 0; j < kScBatch; ++j) {
                ws[j] = wsn[j];
#pragma unroll
                for (int i = 0; i < P; ++i) v[j][i] = own[offs[j] + i * kScPitch];
            }
            rows(k0 + kScBatch);
#pragma unroll
            for (int j = 0; j < kScBatch; ++j)
                if (k0 + j < g.single)
#pragma unroll
                    for (int i = 0; i < P; ++i) u[i] = fma_acc(ws[j], v[j][i], u[i]);
        }
    }
    // Rows beyond the halo, from global memory, kScBatch at a time.  A pixel
    // outside the image reads some pixel's value and stores nothing.
    const int w_px = ti.w0 + col;
    const bool wact = w_px < W;
    for (int k0 = 0; k0 < g.far; k0 += kScBatch) {
        A v[kScBatch][P], ws[kScBatch];
#pragma unroll
        for (int j = 0; j < kScBatch; ++j) {
            const int s = __builtin_amdgcn_readfirstlane(list[min(k0 + j, g.far - 1)]);
            const ShiftRec r = read_shift(shl, s);
            ws[j] = wl[s];
            // (p - s) mod = (p + (H - dx mod H)) mod
            const int dxm = MODE == 0 ? r.dxm : (r.dxm ? H - r.dxm : 0);
            const int dym = MODE == 0 ? r.dym : (r.dym ? W - r.dym : 0);
            const uint32_t ww = wrap1(min(w_px, W - 1) + dym, W);
            int hh = wrap1(min(ti.h0 + r0, H - 1) + dxm, H);
#pragma unroll
            for (int i = 0; i < P; ++i) {
                v[j][i] = to_acc(src[static_cast<uint32_t>(hh) * static_cast<uint32_t>(W) + ww]);
                hh = hh + 1 == H ? 0 : hh + 1;
            }
        }
#pragma unroll
        for (int j = 0; j < kScBatch; ++j)
            if (k0 + j < g.far)
#pragma unroll
                for (int i = 0; i < P; ++i) u[i] = fma_acc(ws[j], v[j][i], u[i]);
    }
    if (!wact) return;
#pragma unroll
    for (int i = 0; i < P; ++i) {
        const int h = ti.h0 + r0 + i;
        if (h >= H) continue;
        const int64_t o = ti.bc * HW + static_cast<uint32_t>(h) * static_cast<uint32_t>(W) + w_px;
        if (MODE == 0) {
            static_cast<A*>(out0)[o] = u[i];
            out1[o] = z;
        } else {
            static_cast<T*>(out0)[o] = from_acc<T>(u[i]);
        }
    }
}

// The wave sums of four values at once, lane 15 + 16 j of the result holding
// that of v[j]: the halves of two values, then the 16-lane rows of two such
// pairs, trade places in one instruction each (permlane32_swap,
// permlane16_swap), so four sums take ten instructions instead of 28.
__device__ __forceinline__ void swap_add(float& a, float b, bool rows16) {
    const auto r = rows16 ? __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b),
                                                             false, false)
                          : __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b),
                                                             false, false);
    a = __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float wave_sum4(float (&v)[4]) {
    swap_add(v[0], v[2], false);
    swap_add(v[1], v[3], false);
    swap_add(v[0], v[1], true);
    float t = dpp_add<0x111, 0xf>(v[0]);
    t = dpp_add<0x112, 0xf>(t);
    t = dpp_add<0x114, 0xf>(t);
    return dpp_add<0x118, 0xf>(t);
}
__device__ __forceinline__ double wave_sum4(double (&v)[4]) {
    const int row = (threadIdx.x & 63) >> 4;
    double t = 0.0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const double w = wave_sum(v[j]);
        t = row == j ? w : t;
    }
    return t;
}

// sum over i < 16 of gu[i0 + i] value(i), as two chains of eight products: one
// chain over a column's 32 rows made the weight gradient's error against 64
// bits 4 to 12% larger than sums of four pixels over eight waves; with the
// chains and their tree it is smaller.
template <typename A, typename F>
__device__ __forceinline__ A gu_sum(const A (&gu)[kScTH], int i0, F&& value) {
    A a = A(0), b = A(0);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        a = fma_acc(gu[i0 + i], value(i), a);
        b = fma_acc(gu[i0 + 8 + i], value(8 + i), b);
    }
    return a + b;
}

// gw partials of one tile: part[(s*BC + bc)*ntp + tile] =
//   sum_{p in tile} gU[p] x[(p+s) mod] + gZ[p]
// Every wave holds the whole tile's gU (a lane its column, 32 rows) and takes
// its share of the shifts: chunks of four neighbouring dx of the grid, or
// single rows.  A chunk reads the column values of 16 rows at a time.
template <typename T>
__global__ __launch_bounds__(kScThreads) void scalar_gw_tile_kernel(
    const T* __restrict__ x, const acc_t<T>* __restrict__ gU, const acc_t<T>* __restrict__ gZ,
    const int64_t* __restrict__ shifts, int cols, int S, int B, int C, int H, int W, int ntw,
    int nth, acc_t<T>* __restrict__ part) {
    using A = acc_t<T>;
    constexpr int CH = kScChunk, TH = kScTH, SUB = 16;
    extern __shared__ __align__(16) unsigned char smem[];
    int4* shl = reinterpret_cast<int4*>(smem);
    A* xt = reinterpret_cast<A*>(smem + shift_lds_bytes(S));
    A* gzw = xt + kScTile;  // the waves' shares of the tile's gZ
    int* cell = reinterpret_cast<int*>(gzw + kScWaves);
    int* list = cell + kScBox * kScRow;

    // plain tile order: the partial index is the tile's position in its plane
    const int64_t ntp = static_cast<int64_t>(ntw) * nth;
    const TileIdx ti = tile_of(blockIdx.x, ntw, nth, kScTH, kScTW);
    const int64_t tile = blockIdx.x - ti.bc * ntp;
    const int64_t HW = static_cast<int64_t>(H) * W;
    const int64_t BC = static_cast<int64_t>(B) * C;
    const T* xp = x + ti.bc * HW;
    const int col = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int w_px = ti.w0 + col;
    const bool wact = w_px < W;

    constexpr int ZR = TH / kScWaves;  // rows of gZ a wave adds up
    A gu[TH];
    A gz = A(0);
#pragma unroll
    for (int i = 0; i < TH; ++i) {
        const bool act = wact && ti.h0 + i < H;
        const int64_t o = ti.bc * HW + (act ? static_cast<uint32_t>(ti.h0 + i) *
                                                      static_cast<uint32_t>(W) + w_px
                                            : 0u);
        gu[i] = act ? gU[o] : A(0);
    }
#pragma unroll
    for (int i = 0; i < ZR; ++i) {
        const int h = ti.h0 + wave * ZR + i;
        const bool act = wact && h < H;
        const int64_t o = ti.bc * HW + (act ? static_cast<uint32_t>(h) *
                                                      static_cast<uint32_t>(W) + w_px
                                            : 0u);
        gz += act ? gZ[o] : A(0);
    }
    gz = wave_sum(gz);
    if (col == 0) gzw[wave] = gz;
    stage_scalar_tile<T, A>(xt, xp, H, W, ti.h0, ti.w0);
    stage_shifts(shl, shifts, S, cols, H, W, 0);  // ends with a barrier
    const SGrid g = stage_grid<1>(shl, S, cell, list);
    A gz_tile = A(0);  // the sum of gZ over the tile, part of every shift's sum
#pragma unroll
    for (int i = 0; i < kScWaves; ++i) gz_tile += gzw[i];
    const A* own = xt + kRmax * kScPitch + col + kRmax;

    if (g.dense) {
        const int nch = (g.n + CH - 1) / CH;
        for (int job = wave; job < g.m * nch; job += kScWaves) {
            const int dyi = job / nch, dxi = (job - dyi * nch) * CH;
            const A* cv = own + (g.dx0 + dxi) * kScPitch + g.dy0 + dyi;
            A acc[CH];
#pragma unroll
            for (int i0 = 0; i0 < TH; i0 += SUB) {
                A v[SUB + CH - 1];
#pragma unroll
                for (int i = 0; i < SUB + CH - 1; ++i) v[i] = cv[(i0 + i) * kScPitch];
#pragma unroll
                for (int j = 0; j < CH; ++j) {
                    const A t = gu_sum<A>(gu, i0, [&](int i) { return v[i + j]; });
                    acc[j] = i0 == 0 ? t : acc[j] + t;
                }
            }
            static_assert(CH == 4, "one value per 16-lane row");
            const int s = cell[dyi * kScRow + dxi + (col >> 4)];  // -1 beyond the box
            const A t = wave_sum4(acc) + gz_tile;
            if ((col & 15) == 15 && s >= 0)
                part[(static_cast<int64_t>(s) * BC + ti.bc) * ntp + tile] = t;
        }
    }
    for (int k = wave; k < g.single; k += kScWaves) {
        const int s = __builtin_amdgcn_readfirstlane(list[S - 1 - k]);
        const ShiftRec r = read_shift(shl, s);
        const A* sr = own + r.dx * kScPitch + r.dy;
        A acc = A(0);
#pragma unroll
        for (int i0 = 0; i0 < TH; i0 += SUB) {
            A v[SUB];
#pragma unroll
            for (int i = 0; i < SUB; ++i) v[i] = sr[(i0 + i) * kScPitch];
            acc += gu_sum<A>(gu, i0, [&](int i) { return v[i]; });
        }
        const A t = wave_sum(acc) + gz_tile;
        if (col == 0) part[(static_cast<int64_t>(s) * BC + ti.bc) * ntp + tile] = t;
    }
    // Rows beyond the halo, from global memory.  A pixel outside the image
    // reads some pixel's value and takes 0 (gU is 0 there, but the value may
    // be infinite).
    for (int k = wave; k < g.far; k += kScWaves) {
        const int s = __builtin_amdgcn_readfirstlane(list[k]);
        const ShiftRec r = read_shift(shl, s);
        const uint32_t ww = wrap1(min(w_px, W - 1) + r.dym, W);
        int hh = wrap1(ti.h0 + r.dxm, H);
        int rows = wact ? H - ti.h0 : 0;  // the lane's pixels
        asm volatile("" : "+v"(rows));    // 32 comparisons a row, not 32 masks kept over all rows
        A acc = A(0);
#pragma unroll
        for (int i0 = 0; i0 < TH; i0 += SUB) {
            A v[SUB];
#pragma unroll
            for (int i = 0; i < SUB; ++i) {
                v[i] = to_acc(xp[static_cast<uint32_t>(hh) * static_cast<uint32_t>(W) + ww]);
                hh = hh + 1 == H ? 0 : hh + 1;
            }
            acc += gu_sum<A>(gu, i0, [&](int i) {
                return i0 + i < rows ? v[i] : A(0);
            });
        }
        const A t = wave_sum(acc) + gz_tile;
        if (col == 0) part[(static_cast<int64_t>(s) * BC + ti.bc) * ntp + tile] = t;
    }
}

template <typename T>
__global__ __launch_bounds__(256) void scalar_gw_final_kernel(const acc_t<T>* __restrict__ partial,
                                                              int64_t n, int nsplit,
                                                              T* __restrict__ gw) {
    using A = acc_t<T>;
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (i >= n) return;
    A t = A(0);
    for (int k = 0; k < nsplit; ++k) t += partial[i * nsplit + k];
    gw[i] = from_acc<T>(t);
}

static void sc_tiles(int H, int W, int* ntw, int* nth) {
    *ntw = static_cast<int>(nsh_host::ceil_div(W, kScTW));
    *nth = static_cast<int>(nsh_host::ceil_div(H, kScTH));
}

template <typename T, int MODE>
static int s_tile(const void* src, const void* w, const int64_t* sh, int cols, int S, int B, int C,
                  int H, int W, void* out0, void* out1, hipStream_t st) {
    using A = acc_t<T>;
    int ntw, nth;
    sc_tiles(H, W, &ntw, &nth);
    const int64_t tiles = static_cast<int64_t>(B) * C * ntw * nth;
    const size_t lds = shift_lds_bytes(S) +
                       (kScBox * kScRow + static_cast<size_t>(kScTile) + S) * sizeof(A) +
                       (kScBox * (kScRow + kScChunks) + S) * sizeof(int);
    hipLaunchKernelGGL((scalar_tile_kernel<T, MODE>), dim3(static_cast<unsigned>(tiles)),
                       dim3(kScThreads), lds, st, src, static_cast<const T*>(w), sh, cols, S, B, C,
                       H, W, ntw, nth, out0, static_cast<A*>(out1));
    return nsh_host::check_launch(MODE == 0 ? "accumulate_uz_scalar_forward"
                                            : "accumulate_uz_scalar_backward");
}

// Partials per (s, b, c): the tiles of one plane.
static int scalar_splits(int64_t H, int64_t W) {
    int ntw, nth;
    sc_tiles(static_cast<int>(H), static_cast<int>(W), &ntw, &nth);
    return ntw * nth;
}

template <typename T>
static int s_gw(const void* x, const void* gU, const void* gZ, const int64_t* sh, int cols, int S,
                int B, int C, int H, int W, void* gw, void* partial, hipStream_t st) {
    using A = acc_t<T>;
    int ntw, nth;
    sc_tiles(H, W, &ntw, &nth);
    const int nsplit = ntw * nth;
    const int64_t tiles = static_cast<int64_t>(B) * C * nsplit;
    const size_t lds = shift_lds_bytes(S) + (kScTile + kScWaves) * sizeof(A) +
                       (kScBox * kScRow + S) * sizeof(int);
    hipLaunchKernelGGL((scalar_gw_tile_kernel<T>), dim3(static_cast<unsigned>(tiles)),
                       dim3(kScThreads), lds, st, static_cast<const T*>(x),
                       static_cast<const A*>(gU), static_cast<const A*>(gZ), sh, cols, S, B, C, H,
                       W, ntw, nth, static_cast<A*>(partial));
    if (int rc = nsh_host::check_launch("accumulate_uz_scalar_backward (gw partial)")) return rc;
    const int64_t n = static_cast<int64_t>(S) * B * C;
    hipLaunchKernelGGL((scalar_gw_final_kernel<T>),
                       dim3(static_cast<unsigned>(nsh_host::ceil_div(n, 256))), dim3(256), 0, st,
                       static_cast<const A*>(partial), n, nsplit, static_cast<T*>(gw));
    return nsh_host::check_launch("accumulate_uz_scalar_backward (gw final)");
}

}  // namespace nsh

using nsh_host::fail;

static int s_check(const char* op, int64_t S, int64_t cols, int64_t B, int64_t C, int64_t H,
                   int64_t W, int dtype) {
    if (S < 1 || S > 1024) return fail(NSH_ERR_INVALID, "%s: tree reduction requires 1 <= S <= 1024", op);
    if (cols != 2 && cols != 3) return fail(NSH_ERR_INVALID, "%s: shifts must have 2 or 3 columns", op);
    if (B < 1 || C < 1 || H < 1 || W < 1) return fail(NSH_ERR_INVALID, "%s: empty tensor", op);
    if (dtype < NSH_DTYPE_FLOAT16 || dtype > NSH_DTYPE_FLOAT64)
        return fail(NSH_ERR_INVALID, "%s: unsupported dtype code %d", op, dtype);
    const int64_t es = dtype == NSH_DTYPE_FLOAT64 ? 8 : 4;
    if (H * W * es >= (int64_t(1) << 31))
        return fail(NSH_ERR_INVALID, "%s: one (b, c) plane must stay below 2^31 bytes", op);
    if (B * C > (int64_t(1) << 24)) return fail(NSH_ERR_INVALID, "%s: B*C too large", op);
    return NSH_OK;
}

extern "C" int nsh_scalar_backward_splits(int64_t H, int64_t W) { return nsh::scalar_splits(H, W); }

extern "C" int nsh_accumulate_uz_scalar_forward(const void* x, const void* weights,
                                                const int64_t* shifts, int64_t S,
                                                int64_t shift_cols, int64_t B, int64_t C, int64_t H,
                                                int64_t W, int dtype, void* U, void* Z,
                                                void* stream) {
    if (int rc = s_check("accumulate_uz_scalar", S, shift_cols, B, C, H, W, dtype)) return rc;
    if (!x || !weights || !shifts || !U || !Z)
        return fail(NSH_ERR_INVALID, "accumulate_uz_scalar: null pointer argument");
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int s = (int)S, c = (int)shift_cols, b = (int)B, ch = (int)C, h = (int)H, w = (int)W;
    switch (dtype) {
        case NSH_DTYPE_FLOAT16: return nsh::s_tile<nsh::f16, 0>(x, weights, shifts, c, s, b, ch, h, w, U, Z, st);
        case NSH_DTYPE_BFLOAT16: return nsh::s_tile<nsh::bf16, 0>(x, weights, shifts, c, s, b, ch, h, w, U, Z, st);
        case NSH_DTYPE_FLOAT32: return nsh::s_tile<float, 0>(x, weights, shifts, c, s, b, ch, h, w, U, Z, st);
        default: return nsh::s_tile<double, 0>(x, weights, shifts, c, s, b, ch, h, w, U, Z, st);
    }
}

extern "C" int nsh_accumulate_uz_scalar_backward(const void* x, const void* weights,
                                                 const void* grad_U, const void* grad_Z,
                                                 const int64_t* shifts, int64_t S,
                                                 int64_t shift_cols, int64_t B, int64_t C,
                                                 int64_t H, int64_t W, int dtype, void* grad_x,
                                                 void* grad_w, void* grad_w_partial, void* stream) {
    if (int rc = s_check("accumulate_uz_scalar_backward", S, shift_cols, B, C, H, W, dtype)) return rc;
    if (!x || !weights || !grad_U || !grad_Z || !shifts || !grad_x || !grad_w || !grad_w_partial)
        return fail(NSH_ERR_INVALID, "accumulate_uz_scalar_backward: null pointer argument");
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int s = (int)S, c = (int)shift_cols, b = (int)B, ch = (int)C, h = (int)H, w = (int)W;
    int rc = NSH_OK;
    switch (dtype) {
        case NSH_DTYPE_FLOAT16:
            rc = nsh::s_tile<nsh::f16, 1>(grad_U, weights, shifts, c, s, b, ch, h, w, grad_x, nullptr, st);
            return rc ? rc : nsh::s_gw<nsh::f16>(x, grad_U, grad_Z, shifts, c, s, b, ch, h, w, grad_w, grad_w_partial, st);
        case NSH_DTYPE_BFLOAT16:
            rc = nsh::s_tile<nsh::bf16, 1>(grad_U, weights, shifts, c, s, b, ch, h, w, grad_x, nullptr, st);
            return rc ? rc : nsh::s_gw<nsh::bf16>(x, grad_U, grad_Z, shifts, c, s, b, ch, h, w, grad_w, grad_w_partial, st);
        case NSH_DTYPE_FLOAT32:
            rc = nsh::s_tile<float, 1>(grad_U, weights, shifts, c, s, b, ch, h, w, grad_x, nullptr, st);
            return rc ? rc : nsh::s_gw<float>(x, grad_U, grad_Z, shifts, c, s, b, ch, h, w, grad_w, grad_w_partial, st);
        default:
            rc = nsh::s_tile<double, 1>(grad_U, weights, shifts, c, s, b, ch, h, w, grad_x, nullptr, st);
            return rc ? rc : nsh::s_gw<double>(x, grad_U, grad_Z, shifts, c, s, b, ch, h, w, grad_w, grad_w_partial, st);
    }
}
