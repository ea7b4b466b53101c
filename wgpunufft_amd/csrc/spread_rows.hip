// Plain (FP32 / FP64) type-1 spreading of 3D row tiles (kernel widths 2..8
// in FP32, 2..16 in FP64) and of 2D row tiles (widths 2..8), for one plan or
// for the plans of a batch.
//
// Same contract as the reference's output-stationary spreader
// (src/gpu_nd_spread.rs:1-36, 1583-1667): every cell of an 8 x 8 x 8 tile
// (x, y, z) is owned by one wavefront, which adds the records whose support
// reaches the tile in a fixed order (reach row by reach row, slot order
// inside a row) and writes the cell once; tiles with too many records are
// split into parts whose partial sums are added in part order.  No atomics,
// so results are bitwise repeatable.
//
// Mapping: bins are one cell along y and z, so the records of one reach row
// share their y and z support.  The sum over a tile's records j is a matrix
// product in the plan's own precision, G[(y, z), (x, re|im)] +=
// sum_j (Ky_j[y] Kz_j[z]) (Kx_j[x] c_j): four 16-row blocks (8 y by 2 z) of
// 16 columns (8 x cells, re and im), four records per
// v_mfma_{f32,f64}_16x16x4 (FP32 or FP64 products and sums, as the vector
// FMAs).  Records are staged 64 at a time (their global loads issued one
// chunk ahead), compacted to those whose x support touches the tile, with
// their weights laid out over the tile's own cells (zero off the support).
// Records come in z order, so a group of four touches few z cells: row
// blocks that none of the four reaches are skipped (at width 7 2.3 of the 4
// blocks are left).
//
// What bounds it: the vector ALU (staging: search, weights, LDS stores; the
// operand products) at about half of its issue rate, the matrix cores a
// quarter, with 2 (FP64) to 4 (FP32) waves per SIMD to hide the LDS and
// record latency.  The vector form before it (a lane owned a row of cells,
// 16 FMAs, 5 LDS reads and a product per record, weights by sqrt and exp in
// every tile visited) against this one: 3D FP32 width 7, 2e6 points on
// 240 x 200 x 150 cells 629 -> 365 us; 3D FP64 width 10, 1e6 points on 128^3
// 1465 -> 725 us; 2D FP32 width 7, 5e7 points on 2048^2 3.64 -> 1.68 ms, 1e5
// points on 256^2 95 -> 41 us.  Accumulators stay in VGPRs (at least two
// waves per SIMD asked for): in AGPRs the compiler copied them back after
// every instruction (2D: 1.98 ms).
#include <hip/hip_runtime.h>

#include "mfma_ops.hpp"
#include "spread.hpp"
#include "spread_device.hpp"
#include "tile_stage.hpp"

namespace mnufft {

namespace {

constexpr int kRowsTX = 8, kRowsTY = 8, kRowsTZ = 8;

// A staged record: its weights over the tile's cells of each axis (zero off
// the support; z cells ordered by parity, then z / 2, so that a lane reads
// its cells of the four row blocks as one vector) and its strength.  Records
// lie an odd multiple of four LDS banks apart, so 64 lanes writing their own
// records spread over all banks.
template <typename T>
struct alignas(16) Row3Rec {
    T kx[kRowsTX];
    T ky[kRowsTY];
    T kz[kRowsTZ];
    T c[2];
};
template <typename T>
struct Rows3Stage {
    Row3Rec<T> rec[64];
    uint32_t blocks[64];  // row blocks each record touches
};
static_assert(sizeof(Row3Rec<float>) % 32 == 16 && sizeof(Row3Rec<double>) % 32 == 16,
              "records an odd multiple of 16 bytes apart");

// Weights of a record over the N cells of a tile axis from `rel` (the
// support start relative to the tile origin) and its offset; cell i goes to
// dst[place(i)].
template <typename T, int W, int N, typename Place>
__device__ __forceinline__ void tile_weights(T *dst, int rel, T off, T beta, UniformPtr<T> panels,
                                             Place place)
{
#pragma unroll
    for (int i = 0; i < N; ++i) dst[i] = (T)0;
    es_axis_weights<T, W>(off, beta, panels, [&](int t, T w) {
        const unsigned i = (unsigned)(rel + t);
        if (i < (unsigned)N) dst[place(i)] = w;
    });
}

// Clears the staged weights: a group of four may read up to three records
// past the staged ones (seven for two groups), whose strengths are then zero.
template <typename T, typename Stage>
__device__ inline void clear_stage(Stage &st, int lane)
{
    uint32_t *p = (uint32_t *)&st;
    for (int i = lane; i < (int)(sizeof(Stage) / 4); i += 64) p[i] = 0;
    wave_sync();
}

// Bit s of the ballot: staged record s touches block b.
__device__ inline uint64_t touch_ballot(uint32_t blocks, int b)
{
    return __ballot((blocks >> b) & 1u);
}

// Sums the records [klo, khi) of the reach of the tile at (x0, y0, z0) into
// acc: row block b holds the cells z = 2b, 2b + 1.  `offsets` are the bin
// offsets of the tile's own grid; slots index the records and strengths `cv`
// directly.
template <typename T, int W, int NROWS>
__device__ __forceinline__ void rows3_accumulate(Rows3Stage<T> &st, TileRows<NROWS> &rows, int lane,
                                                 const GridParams &g, int64_t x0, int64_t y0,
                                                 int64_t z0, int64_t klo, int64_t khi,
                                                 const uint32_t *__restrict__ offsets,
                                                 const T *__restrict__ rec_off,
                                                 const T *__restrict__ cv,
                                                 typename mfma::ExactMma<T>::Acc (&acc)[4])
{
    using Mma = mfma::ExactMma<T>;
    using V4 = typename Vec4Of<T>::V4;
    constexpr int TX = kRowsTX, TY = kRowsTY, TZ = kRowsTZ;
    constexpr int NRY = TY + W - 1;
    const T beta = (T)g.beta;
    const UniformPtr<T> panels = panel_coefficients<T>(g);
    const int64_t n0 = g.ax[0].n;
    const AxisReach rx = axis_reach(x0, TX, W, g.ax[0]);
    int64_t xs = x0 - (W - 1);
    if (xs < 0) xs += n0;

    stage_tile_rows<3, TY, TZ, W, NROWS>(rows, lane, y0, z0, rx, g, offsets);
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[b] = typename Mma::Acc{(T)0, (T)0, (T)0, (T)0};
    const int lk = lane >> 4, ly = lane & 7, lz = 4 * ((lane >> 3) & 1);
    const int lx = (lane & 15) >> 1, lc = lane & 1;
    // records in chunks of 64, the next chunk's loads in flight while the
    // current one is added
    Fetched<T> nx = fetch_record<T, NROWS>(rows, klo + lane, khi, rec_off, cv);
    for (int64_t k0 = klo; k0 < khi; k0 += 64) {
        const Fetched<T> cur = nx;
        nx = fetch_record<T, NROWS>(rows, k0 + 64 + lane, khi, rec_off, cv);
        bool take = false;
        int ee = 0;
        if (cur.valid) {
            int64_t e64 = (int64_t)cur.sx0 - xs;
            if (e64 < 0) e64 += n0;
            take = e64 < TX + W - 1 && on_support<T>(cur.off.x);
            ee = (int)e64;
        }
        const uint64_t mask = __ballot(take);
        const int pos = __popcll(mask & ((1ull << lane) - 1ull));
        const int nst = __popcll(mask);
        if (take) {
            const auto same = [](unsigned i) { return i; };
            const auto by_block = [](unsigned i) { return 4 * (i & 1) + (i >> 1); };
            const int rz = cur.q / NRY - (W - 1);
            Row3Rec<T> &R = st.rec[pos];
            tile_weights<T, W, TX>(R.kx, ee - (W - 1), (T)cur.off.x, beta, panels, same);
            tile_weights<T, W, TY>(R.ky, cur.q % NRY - (W - 1), (T)cur.off.y, beta, panels, same);
            tile_weights<T, W, TZ>(R.kz, rz, (T)cur.off.z, beta, panels, by_block);
            R.c[0] = cur.c[0].x;
            R.c[1] = cur.c[0].y;
            const int lo = rz > 0 ? rz >> 1 : 0, hi = rz + W - 1 < TZ ? (rz + W - 1) >> 1 : 3;
            st.blocks[pos] = (2u << hi) - (1u << lo);
        }
        if (lane < 7 && nst + lane < 64) st.rec[nst + lane].c[0] = st.rec[nst + lane].c[1] = (T)0;
        wave_sync();
        const uint32_t blocks = lane < nst ? st.blocks[lane] : 0;
        uint64_t touch[4];
#pragma unroll
        for (int b = 0; b < 4; ++b) touch[b] = touch_ballot(blocks, b);
        // two groups of four at a time, their LDS reads in flight together
        for (int s = 0; s < nst; s += 8) {
            T ky[2], kxc[2];
            V4 kz[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const Row3Rec<T> &R = st.rec[s + 4 * h + lk];
                ky[h] = R.ky[ly];
                kz[h] = *(const V4 *)&R.kz[lz];
                kxc[h] = R.kx[lx] * R.c[lc];
            }
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int at = s + 4 * h;
                if ((touch[0] >> at) & 15) acc[0] = Mma::mma(ky[h] * kz[h].x, kxc[h], acc[0]);
                if ((touch[1] >> at) & 15) acc[1] = Mma::mma(ky[h] * kz[h].y, kxc[h], acc[1]);
                if ((touch[2] >> at) & 15) acc[2] = Mma::mma(ky[h] * kz[h].z, kxc[h], acc[2]);
                if ((touch[3] >> at) & 15) acc[3] = Mma::mma(ky[h] * kz[h].w, kxc[h], acc[3]);
            }
        }
        wave_sync();
    }
}

// The tile's cells: into the grid `gv` (one vector) when the tile is one
// part, else into the part's partial-sum slot `slot` (8 x 8 x 8).  Sixteen
// lanes write the 8 cells of an x row.
template <typename T>
__device__ __forceinline__ void rows3_store(int lane, const GridParams &g, int64_t x0, int64_t y0,
                                            int64_t z0, bool whole, T *__restrict__ gv,
                                            T *__restrict__ slot,
                                            const typename mfma::ExactMma<T>::Acc (&acc)[4])
{
    const int col = lane & 15;
    const int64_t n0 = g.ax[0].n, n1 = g.ax[1].n, n2 = g.ax[2].n;
    const bool in_x = x0 + (col >> 1) < n0;
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = mfma::ExactMma<T>::row(lane, r);
            const int y = i & 7, z = 2 * b + (i >> 3);
            if (whole) {
                if (in_x && y0 + y < n1 && z0 + z < n2)
                    gv[2 * (x0 + n0 * (y0 + y + n1 * (z0 + z))) + col] = acc[b][r];
            } else {
                slot[partial_index<kRowsTX, kRowsTY, kRowsTZ>(0, 1, 0, 0, y, z) + col] = acc[b][r];
            }
        }
}

template <typename T, int W>
__global__ __launch_bounds__(64, sizeof(T) == 4 ? 4 : 2) void k_spread_rows(
    GridParams g, SpreadParams sp, const uint32_t *__restrict__ offsets,
    const T *__restrict__ rec_off,
    const T *__restrict__ c_sorted, int64_t M, const uint32_t *__restrict__ totals,
    const uint32_t *__restrict__ parts, const uint32_t *__restrict__ item_off,
    const uint32_t *__restrict__ heavy_base, const uint32_t *__restrict__ ctrl,
    T *__restrict__ grid, T *__restrict__ partial)
{
    static_assert(W <= kMaxRowsWidth, "widths beyond the row tiles");
    constexpr int TX = kRowsTX, TY = kRowsTY, TZ = kRowsTZ;
    constexpr int NROWS = (TY + W - 1) * (TZ + W - 1);
    __shared__ Rows3Stage<T> st;
    __shared__ TileRows<NROWS> rows;

    const int lane = threadIdx.x;
    clear_stage<T>(st, lane);
    const int64_t v = blockIdx.y;
    const int64_t n_items = ctrl[0];
    const uint32_t part_len_cap = ctrl[3];
    const T *cv = c_sorted + 2 * v * M;

    for (int64_t item = blockIdx.x; item < n_items; item += gridDim.x) {
        const TileItem ti = tile_item(item, sp.block_count, item_off, parts, totals, part_len_cap,
                                      n_items);
        const int64_t b = ti.b;
        const int64_t x0 = (b % sp.nblocks[0]) * TX;
        const int64_t y0 = ((b / sp.nblocks[0]) % sp.nblocks[1]) * TY;
        const int64_t z0 = (b / (sp.nblocks[0] * sp.nblocks[1])) * TZ;
        typename mfma::ExactMma<T>::Acc acc[4];
        rows3_accumulate<T, W, NROWS>(st, rows, lane, g, x0, y0, z0, ti.rlo, ti.rhi, offsets,
                                      rec_off, cv, acc);
        const bool whole = ti.np == 1;
        T *slot = whole ? nullptr
                        : partial + partial_index<TX, TY, TZ>((int64_t)heavy_base[b] + ti.p,
                                                              gridDim.y, v, 0, 0, 0);
        rows3_store<T>(lane, g, x0, y0, z0, whole, grid + 2 * v * g.fine_total, slot, acc);
    }
}

// The 3D row tiles of every problem of a batch class (one vector each, one
// kernel width), as k_spread_rows2_many does for 2D.
template <typename T, int W>
__global__ __launch_bounds__(64, sizeof(T) == 4 ? 4 : 2) void k_spread_rows3_many(
    const BatchProblem *__restrict__ probs, const SpreadProblem *__restrict__ sprobs, int nprob,
    const uint32_t *__restrict__ offsets, const T *__restrict__ rec_off, const T *__restrict__ c_sorted,
    const uint32_t *__restrict__ totals, const uint32_t *__restrict__ parts,
    const uint32_t *__restrict__ item_off, const uint32_t *__restrict__ heavy_base,
    const uint32_t *__restrict__ pctrl, const int64_t *__restrict__ pbase,
    T *__restrict__ partial)
{
    static_assert(W <= kMaxRowsWidth, "widths beyond the row tiles");
    constexpr int TX = kRowsTX, TY = kRowsTY, TZ = kRowsTZ;
    constexpr int NROWS = (TY + W - 1) * (TZ + W - 1);
    __shared__ Rows3Stage<T> st;
    __shared__ TileRows<NROWS> rows;

    const int lane = threadIdx.x;
    clear_stage<T>(st, lane);
    const int64_t n_items = pbase[4 * nprob];
    for (int64_t item = blockIdx.x; item < n_items; item += gridDim.x) {
        const int q = batch_problem_of(pbase, nprob, 0, item);
        const BatchProblem &pb = probs[q];
        const SpreadProblem &spb = sprobs[q];
        const int64_t bb = spb.block_base;
        const TileItem ti = tile_item(item - pbase[4 * q], spb.sp.block_count, item_off + bb,
                                      parts + bb, totals + bb, pctrl[8 * q + 3], pctrl[8 * q]);
        const int64_t b = ti.b;
        const int64_t nb0 = spb.sp.nblocks[0], nb1 = spb.sp.nblocks[1];
        const int64_t x0 = (b % nb0) * TX, y0 = ((b / nb0) % nb1) * TY, z0 = (b / (nb0 * nb1)) * TZ;
        typename mfma::ExactMma<T>::Acc acc[4];
        rows3_accumulate<T, W, NROWS>(st, rows, lane, pb.g, x0, y0, z0, ti.rlo, ti.rhi,
                                      offsets + pb.bin_base, rec_off, c_sorted, acc);
        const bool whole = ti.np == 1;
        T *slot = whole ? nullptr
                        : partial + partial_index<TX, TY, TZ>(
                                        pbase[4 * q + 1] + (int64_t)heavy_base[bb + b] + ti.p, 1,
                                        0, 0, 0, 0);
        rows3_store<T>(lane, pb.g, x0, y0, z0, whole, (T *)pb.grid, slot, acc);
    }
}

// 2D row tiles of 16 x 16 cells: G[y, (x, re|im)] += sum_j Ky_j[y] (Kx_j[x]
// c_j), one 16-row block (y) by two column blocks (x cells 0..7 and 8..15),
// four records per v_mfma_{f32,f64}_16x16x4; a column block that none of the
// four records reaches is skipped.  Bins are one cell along y, so the records
// of a reach row share their y support.  Same order, parts and partial-sum
// layout as the 3D tiles.
constexpr int kRows2T = 16;

template <typename T>
struct alignas(16) Row2Rec {
    T kx[kRows2T];
    T ky[kRows2T];
    T c[2];
};
template <typename T>
struct Rows2Stage {
    Row2Rec<T> rec[64];
    uint32_t blocks[64];  // column blocks each record touches
};
static_assert(sizeof(Row2Rec<float>) % 32 == 16 && sizeof(Row2Rec<double>) % 32 == 16,
              "records an odd multiple of 16 bytes apart");

// Sums the records [klo, khi) of the reach of the tile at (x0, y0) into acc:
// column block b holds the x cells 8b .. 8b + 7.  `offsets` are the bin
// offsets of the tile's own grid; slots index the records and strengths `cv`
// directly.
template <typename T, int W, int NROWS>
__device__ __forceinline__ void rows2_accumulate(Rows2Stage<T> &st, TileRows<NROWS> &rows, int lane,
                                                 const GridParams &g, int64_t x0, int64_t y0,
                                                 int64_t klo, int64_t khi,
                                                 const uint32_t *__restrict__ offsets,
                                                 const T *__restrict__ rec_off,
                                                 const T *__restrict__ cv,
                                                 typename mfma::ExactMma<T>::Acc (&acc)[2])
{
    using Mma = mfma::ExactMma<T>;
    constexpr int TX = kRows2T, TY = kRows2T;
    const T beta = (T)g.beta;
    const UniformPtr<T> panels = panel_coefficients<T>(g);
    const int64_t n0 = g.ax[0].n;
    const AxisReach rx = axis_reach(x0, TX, W, g.ax[0]);
    int64_t xs = x0 - (W - 1);
    if (xs < 0) xs += n0;

    stage_tile_rows<2, TY, 1, W, NROWS>(rows, lane, y0, 0, rx, g, offsets);
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[b] = typename Mma::Acc{(T)0, (T)0, (T)0, (T)0};
    const int lk = lane >> 4, ly = lane & 15, lx = (lane & 15) >> 1, lc = lane & 1;
    Fetched<T> nx = fetch_record<T, NROWS>(rows, klo + lane, khi, rec_off, cv);
    for (int64_t k0 = klo; k0 < khi; k0 += 64) {
        const Fetched<T> cur = nx;
        nx = fetch_record<T, NROWS>(rows, k0 + 64 + lane, khi, rec_off, cv);
        bool take = false;
        int ee = 0;
        if (cur.valid) {
            int64_t e64 = (int64_t)cur.sx0 - xs;
            if (e64 < 0) e64 += n0;
            take = e64 < TX + W - 1 && on_support<T>(cur.off.x);
            ee = (int)e64;
        }
        const uint64_t mask = __ballot(take);
        const int pos = __popcll(mask & ((1ull << lane) - 1ull));
        const int nst = __popcll(mask);
        if (take) {
            const auto same = [](unsigned i) { return i; };
            const int rel = ee - (W - 1);
            Row2Rec<T> &R = st.rec[pos];
            tile_weights<T, W, TX>(R.kx, rel, (T)cur.off.x, beta, panels, same);
            tile_weights<T, W, TY>(R.ky, cur.q - (W - 1), (T)cur.off.y, beta, panels, same);
            R.c[0] = cur.c[0].x;
            R.c[1] = cur.c[0].y;
            st.blocks[pos] = (rel < 8 ? 1u : 0u) | (rel + W > 8 ? 2u : 0u);
        }
        if (lane < 7 && nst + lane < 64) st.rec[nst + lane].c[0] = st.rec[nst + lane].c[1] = (T)0;
        wave_sync();
        const uint32_t blocks = lane < nst ? st.blocks[lane] : 0;
        const uint64_t t0 = touch_ballot(blocks, 0), t1 = touch_ballot(blocks, 1);
        for (int s = 0; s < nst; s += 8) {
            T ky[2], kl[2], kr[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const Row2Rec<T> &R = st.rec[s + 4 * h + lk];
                const T c = R.c[lc];
                ky[h] = R.ky[ly];
                kl[h] = R.kx[lx] * c;
                kr[h] = R.kx[8 + lx] * c;
            }
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int at = s + 4 * h;
                if ((t0 >> at) & 15) acc[0] = Mma::mma(ky[h], kl[h], acc[0]);
                if ((t1 >> at) & 15) acc[1] = Mma::mma(ky[h], kr[h], acc[1]);
            }
        }
        wave_sync();
    }
}

// The tile's cells: into the grid `gv` (one vector) when the tile is one
// part, else into the part's 16 x 16 partial-sum slot `slot`.
template <typename T>
__device__ __forceinline__ void rows2_store(int lane, const GridParams &g, int64_t x0, int64_t y0,
                                            bool whole, T *__restrict__ gv, T *__restrict__ slot,
                                            const typename mfma::ExactMma<T>::Acc (&acc)[2])
{
    const int col = lane & 15;
    const int64_t n0 = g.ax[0].n, n1 = g.ax[1].n;
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        const int x = 8 * b + (col >> 1);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int y = mfma::ExactMma<T>::row(lane, r);
            if (whole) {
                if (x0 + x < n0 && y0 + y < n1)
                    gv[2 * (x0 + 8 * b + n0 * (y0 + y)) + col] = acc[b][r];
            } else {
                slot[2 * (y * kRows2T + 8 * b) + col] = acc[b][r];
            }
        }
    }
}

template <typename T, int W>
__global__ __launch_bounds__(64, sizeof(T) == 4 ? 4 : 2) void k_spread_rows2(
    GridParams g, SpreadParams sp, const uint32_t *__restrict__ offsets,
    const T *__restrict__ rec_off,
    const T *__restrict__ c_sorted, int64_t M, const uint32_t *__restrict__ totals,
    const uint32_t *__restrict__ parts, const uint32_t *__restrict__ item_off,
    const uint32_t *__restrict__ heavy_base, const uint32_t *__restrict__ ctrl,
    T *__restrict__ grid, T *__restrict__ partial)
{
    static_assert(W <= 8, "widths beyond the 2D row tiles");
    constexpr int NROWS = kRows2T + W - 1;
    __shared__ Rows2Stage<T> st;
    __shared__ TileRows<NROWS> rows;

    const int lane = threadIdx.x;
    clear_stage<T>(st, lane);
    const int64_t v = blockIdx.y;
    const int64_t n_items = ctrl[0];
    const uint32_t part_len_cap = ctrl[3];
    const T *cv = c_sorted + 2 * v * M;

    for (int64_t item = blockIdx.x; item < n_items; item += gridDim.x) {
        const TileItem ti = tile_item(item, sp.block_count, item_off, parts, totals, part_len_cap,
                                      n_items);
        const int64_t b = ti.b;
        const int64_t x0 = (b % sp.nblocks[0]) * kRows2T, y0 = (b / sp.nblocks[0]) * kRows2T;
        typename mfma::ExactMma<T>::Acc acc[2];
        rows2_accumulate<T, W, NROWS>(st, rows, lane, g, x0, y0, ti.rlo, ti.rhi, offsets,
                                      rec_off, cv, acc);
        const bool whole = ti.np == 1;
        T *slot = whole ? nullptr
                        : partial + partial_index<kRows2T, kRows2T, 1>(
                                        (int64_t)heavy_base[b] + ti.p, gridDim.y, v, 0, 0, 0);
        rows2_store<T>(lane, g, x0, y0, whole, grid + 2 * v * g.fine_total, slot, acc);
    }
}

// The 2D row tiles of every problem of a batch class (one vector each, one
// kernel width): item -> problem (item bases) -> the problem's tile and
// part, summed as the problem's own spread sums it.
template <typename T, int W>
__global__ __launch_bounds__(64, sizeof(T) == 4 ? 4 : 2) void k_spread_rows2_many(
    const BatchProblem *__restrict__ probs, const SpreadProblem *__restrict__ sprobs, int nprob,
    const uint32_t *__restrict__ offsets, const T *__restrict__ rec_off, const T *__restrict__ c_sorted,
    const uint32_t *__restrict__ totals, const uint32_t *__restrict__ parts,
    const uint32_t *__restrict__ item_off, const uint32_t *__restrict__ heavy_base,
    const uint32_t *__restrict__ pctrl, const int64_t *__restrict__ pbase,
    T *__restrict__ partial)
{
    static_assert(W <= 8, "widths beyond the 2D row tiles");
    constexpr int NROWS = kRows2T + W - 1;
    __shared__ Rows2Stage<T> st;
    __shared__ TileRows<NROWS> rows;

    const int lane = threadIdx.x;
    clear_stage<T>(st, lane);
    const int64_t n_items = pbase[4 * nprob];
    for (int64_t item = blockIdx.x; item < n_items; item += gridDim.x) {
        const int q = batch_problem_of(pbase, nprob, 0, item);
        const BatchProblem &pb = probs[q];
        const SpreadProblem &spb = sprobs[q];
        const int64_t bb = spb.block_base;
        const TileItem ti = tile_item(item - pbase[4 * q], spb.sp.block_count, item_off + bb,
                                      parts + bb, totals + bb, pctrl[8 * q + 3], pctrl[8 * q]);
        const int64_t b = ti.b;
        const int64_t x0 = (b % spb.sp.nblocks[0]) * kRows2T;
        const int64_t y0 = (b / spb.sp.nblocks[0]) * kRows2T;
        typename mfma::ExactMma<T>::Acc acc[2];
        rows2_accumulate<T, W, NROWS>(st, rows, lane, pb.g, x0, y0, ti.rlo, ti.rhi,
                                      offsets + pb.bin_base, rec_off, c_sorted, acc);
        const bool whole = ti.np == 1;
        T *slot = whole ? nullptr
                        : partial + partial_index<kRows2T, kRows2T, 1>(
                                        pbase[4 * q + 1] + (int64_t)heavy_base[bb + b] + ti.p, 1,
                                        0, 0, 0, 0);
        rows2_store<T>(lane, pb.g, x0, y0, whole, (T *)pb.grid, slot, acc);
    }
}

template <typename T, int W>
bool launch_rows_width(int tx, dim3 grid3, const GridParams &g, const SpreadParams &sp,
                       const uint32_t *offsets, const T *rec_off,
                       const T *c_sorted, int64_t M, const TileWork &w, T *grid, T *partial,
                       hipStream_t stream)
{
    if (tx != kRowsTX) return false;
    k_spread_rows<T, W><<<grid3, 64, 0, stream>>>(
        g, sp, offsets, rec_off, c_sorted, M, w.totals, w.parts, w.item_off,
        w.heavy_base, w.ctrl, grid, partial);
    return true;
}

}  // namespace

template <typename T>
bool launch_rows2_tiles(const GridParams &g, const SpreadParams &sp, const uint32_t *offsets,
                        const T *rec_off, const T *c_sorted, int64_t M,
                        int64_t vectors, const TileWork &w, T *grid, T *partial,
                        hipStream_t stream)
{
    const dim3 grid3(w.items_grid, (unsigned)vectors);
    if (sp.block[0] != kRows2T || sp.block[1] != kRows2T) {
        set_error("plain 2D row tiles are 16 x 16 cells");
        return false;
    }
#define MNUFFT_ROWS2(W)                                                                             \
    case W:                                                                                         \
        k_spread_rows2<T, W><<<grid3, 64, 0, stream>>>(g, sp, offsets, rec_off,          \
                                                       c_sorted, M, w.totals, w.parts, w.item_off,  \
                                                       w.heavy_base, w.ctrl, grid, partial);        \
        break;
    switch (g.width) {
        MNUFFT_ROWS2(2)
        MNUFFT_ROWS2(3)
        MNUFFT_ROWS2(4)
        MNUFFT_ROWS2(5)
        MNUFFT_ROWS2(6)
        MNUFFT_ROWS2(7)
        MNUFFT_ROWS2(8)
    default:
        set_error("plain 2D row tiles need a width of 2..8");
        return false;
    }
#undef MNUFFT_ROWS2
    return hip_ok(hipGetLastError(), "2D row-tile spread launch");
}

template <typename T>
bool launch_rows2_many(int width, const BatchProblem *probs, const SpreadProblem *sprobs,
                       int nprob, unsigned items_grid, const uint32_t *offsets,
                       const T *rec_off, const T *c_sorted,
                       const uint32_t *totals, const uint32_t *parts, const uint32_t *item_off,
                       const uint32_t *heavy_base, const uint32_t *pctrl, const int64_t *pbase,
                       T *partial, hipStream_t stream)
{
#define MNUFFT_ROWS2_MANY(W)                                                                        \
    case W:                                                                                         \
        k_spread_rows2_many<T, W><<<items_grid, 64, 0, stream>>>(                                   \
            probs, sprobs, nprob, offsets, rec_off, c_sorted, totals, parts, item_off,   \
            heavy_base, pctrl, pbase, partial);                                                     \
        break;
    switch (width) {
        MNUFFT_ROWS2_MANY(2)
        MNUFFT_ROWS2_MANY(3)
        MNUFFT_ROWS2_MANY(4)
        MNUFFT_ROWS2_MANY(5)
        MNUFFT_ROWS2_MANY(6)
        MNUFFT_ROWS2_MANY(7)
        MNUFFT_ROWS2_MANY(8)
    default:
        set_error("batched 2D row tiles need a width of 2..8");
        return false;
    }
#undef MNUFFT_ROWS2_MANY
    return hip_ok(hipGetLastError(), "batched 2D row-tile spread launch");
}

template bool launch_rows2_many<float>(int, const BatchProblem *, const SpreadProblem *, int,
                                       unsigned, const uint32_t *, const float *,
                                       const float *, const uint32_t *, const uint32_t *,
                                       const uint32_t *, const uint32_t *, const uint32_t *,
                                       const int64_t *, float *, hipStream_t);
template bool launch_rows2_many<double>(int, const BatchProblem *, const SpreadProblem *, int,
                                        unsigned, const uint32_t *, const double *,
                                        const double *, const uint32_t *, const uint32_t *,
                                        const uint32_t *, const uint32_t *, const uint32_t *,
                                        const int64_t *, double *, hipStream_t);

template <typename T>
bool launch_rows3_many(int width, const BatchProblem *probs, const SpreadProblem *sprobs,
                       int nprob, unsigned items_grid, const uint32_t *offsets,
                       const T *rec_off, const T *c_sorted,
                       const uint32_t *totals, const uint32_t *parts, const uint32_t *item_off,
                       const uint32_t *heavy_base, const uint32_t *pctrl, const int64_t *pbase,
                       T *partial, hipStream_t stream)
{
    bool ok = true;
#define MNUFFT_ROWS3_MANY(W)                                                                        \
    case W:                                                                                         \
        k_spread_rows3_many<T, W><<<items_grid, 64, 0, stream>>>(                                   \
            probs, sprobs, nprob, offsets, rec_off, c_sorted, totals, parts, item_off,   \
            heavy_base, pctrl, pbase, partial);                                                     \
        break;
    switch (width) {
        MNUFFT_ROWS3_MANY(2)
        MNUFFT_ROWS3_MANY(3)
        MNUFFT_ROWS3_MANY(4)
        MNUFFT_ROWS3_MANY(5)
        MNUFFT_ROWS3_MANY(6)
        MNUFFT_ROWS3_MANY(7)
        MNUFFT_ROWS3_MANY(8)
    default:
        ok = false;
        if constexpr (sizeof(T) == 8) {
            ok = true;
            switch (width) {
                MNUFFT_ROWS3_MANY(9)
                MNUFFT_ROWS3_MANY(10)
                MNUFFT_ROWS3_MANY(11)
                MNUFFT_ROWS3_MANY(12)
                MNUFFT_ROWS3_MANY(13)
                MNUFFT_ROWS3_MANY(14)
                MNUFFT_ROWS3_MANY(15)
                MNUFFT_ROWS3_MANY(16)
            default: ok = false; break;
            }
        }
        break;
    }
#undef MNUFFT_ROWS3_MANY
    if (!ok) {
        set_error("batched 3D row tiles need a width of 2..8 (FP32) or 2..16 (FP64)");
        return false;
    }
    return hip_ok(hipGetLastError(), "batched 3D row-tile spread launch");
}

template bool launch_rows3_many<float>(int, const BatchProblem *, const SpreadProblem *, int,
                                       unsigned, const uint32_t *, const float *,
                                       const float *, const uint32_t *, const uint32_t *,
                                       const uint32_t *, const uint32_t *, const uint32_t *,
                                       const int64_t *, float *, hipStream_t);
template bool launch_rows3_many<double>(int, const BatchProblem *, const SpreadProblem *, int,
                                        unsigned, const uint32_t *, const double *,
                                        const double *, const uint32_t *, const uint32_t *,
                                        const uint32_t *, const uint32_t *, const uint32_t *,
                                        const int64_t *, double *, hipStream_t);

template <typename T>
bool launch_rows_tiles(const GridParams &g, const SpreadParams &sp, const uint32_t *offsets,
                       const T *rec_off, const T *c_sorted, int64_t M,
                       int64_t vectors, const TileWork &w, T *grid, T *partial, hipStream_t stream)
{
    if (g.dims == 2)
        return launch_rows2_tiles<T>(g, sp, offsets, rec_off, c_sorted, M, vectors, w,
                                     grid, partial, stream);
    const dim3 grid3(w.items_grid, (unsigned)vectors);
    const int tx = (int)sp.block[0];
    if (sp.block[1] != kRowsTY || sp.block[2] != kRowsTZ) {
        set_error("plain row tiles are 8 x 8 x 8 cells");
        return false;
    }
    bool ok = false;
    switch (g.width) {
    case 2: ok = launch_rows_width<T, 2>(tx, grid3, g, sp, offsets, rec_off, c_sorted, M, w, grid, partial, stream); break;
    case 3: ok = launch_rows_width<T, 3>(tx, grid3, g, sp, offsets, rec_off, c_sorted, M, w, grid, partial, stream); break;
    case 4: ok = launch_rows_width<T, 4>(tx, grid3, g, sp, offsets, rec_off, c_sorted, M, w, grid, partial, stream); break;
    case 5: ok = launch_rows_width<T, 5>(tx, grid3, g, sp, offsets, rec_off, c_sorted, M, w, grid, partial, stream); break;
    case 6: ok = launch_rows_width<T, 6>(tx, grid3, g, sp, offsets, rec_off, c_sorted, M, w, grid, partial, stream); break;
    case 7: ok = launch_rows_width<T, 7>(tx, grid3, g, sp, offsets, rec_off, c_sorted, M, w, grid, partial, stream); break;
    case 8: ok = launch_rows_width<T, 8>(tx, grid3, g, sp, offsets, rec_off, c_sorted, M, w, grid, partial, stream); break;
    default:
        if constexpr (sizeof(T) == 8) {
            switch (g.width) {
            case 9: ok = launch_rows_width<T, 9>(tx, grid3, g, sp, offsets, rec_off, c_sorted, M, w, grid, partial, stream); break;
            case 10: ok = launch_rows_width<T, 10>(tx, grid3, g, sp, offsets, rec_off, c_sorted, M, w, grid, partial, stream); break;
            case 11: ok = launch_rows_width<T, 11>(tx, grid3, g, sp, offsets, rec_off, c_sorted, M, w, grid, partial, stream); break;
            case 12: ok = launch_rows_width<T, 12>(tx, grid3, g, sp, offsets, rec_off, c_sorted, M, w, grid, partial, stream); break;
            case 13: ok = launch_rows_width<T, 13>(tx, grid3, g, sp, offsets, rec_off, c_sorted, M, w, grid, partial, stream); break;
            case 14: ok = launch_rows_width<T, 14>(tx, grid3, g, sp, offsets, rec_off, c_sorted, M, w, grid, partial, stream); break;
            case 15: ok = launch_rows_width<T, 15>(tx, grid3, g, sp, offsets, rec_off, c_sorted, M, w, grid, partial, stream); break;
            case 16: ok = launch_rows_width<T, 16>(tx, grid3, g, sp, offsets, rec_off, c_sorted, M, w, grid, partial, stream); break;
            default: break;
            }
        }
        break;
    }
    if (!ok) {
        set_error("plain row tiles need a 3D plan, a width of 2..8 (FP32) or 2..16 (FP64) and "
                  "8 x 8 x 8 tiles");
        return false;
    }
    return hip_ok(hipGetLastError(), "row-tile spread launch");
}

template bool launch_rows_tiles<float>(const GridParams &, const SpreadParams &, const uint32_t *,
                                       const float *, const float *, int64_t,
                                       int64_t, const TileWork &, float *, float *, hipStream_t);
template bool launch_rows_tiles<double>(const GridParams &, const SpreadParams &,
                                        const uint32_t *, const double *,
                                        const double *, int64_t, int64_t, const TileWork &,
                                        double *, double *, hipStream_t);

}  // namespace mnufft
