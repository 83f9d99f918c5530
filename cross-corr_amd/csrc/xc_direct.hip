// Host side of the wave64 direct kernel (see xc_direct_kernel.hpp): the tile catalog, the
// plan of a launch (tile, block shape, work distribution) and the launchers; the float
// instances of the kernel.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <vector>

#include "xc_direct_kernel.hpp"

namespace xc {

const void* direct_kernel_f32(const direct_tile& t) {
#define XC_PICK(A, B, C, D) \
    if (t.ty == A && t.rm == B && t.lm == C && t.jb == D) return reinterpret_cast<const void*>(&direct_kernel<float, A, B, C, D>);
    XC_DIRECT_TILES(XC_PICK)
#undef XC_PICK
    return nullptr;
}

namespace {

constexpr direct_tile kCatalog[] = {
#define XC_ENTRY(A, B, C, D) {A, B, C, D},
    XC_DIRECT_TILES(XC_ENTRY)
#undef XC_ENTRY
};

// The largest catalog tile that is nowhere above the request: most FMAs per staged value
// (TY*RM*LM*JB), then more right matrices, left matrices, shifts.
direct_tile round_to_catalog(const direct_tile& req) {
    direct_tile best{1, 1, 1, 1};
    long best_score = -1;
    for (const auto& c : kCatalog) {
        if (c.ty > req.ty || c.rm > req.rm || c.lm > req.lm || c.jb > req.jb) continue;
        const long score = (long)c.ty * c.rm * c.lm * c.jb * 4096 + c.rm * 256 + c.lm * 16 + c.ty;
        if (score > best_score) {
            best_score = score;
            best = c;
        }
    }
    return best;
}

int pow2_floor(uint32_t v, int cap) {
    int p = 1;
    while (p * 2 <= (int)v && p * 2 <= cap) p *= 2;
    return p;
}

template <typename T>
const void* kernel_of(const direct_tile& t) {
    return sizeof(T) == 4 ? direct_kernel_f32(t) : direct_kernel_f64(t);
}

struct direct_plan {
    direct_tile t;
    uint32_t nwx, nwy, tiles_x, tiles_y, chunks, rows_per_chunk, groups_l, groups_r;
    int len;
    uint32_t lds;
};

template <typename T>
direct_plan plan_direct(const family_args& a, const xc_options& opt) {
    const bool n_to_m = a.family == XC_N_TO_M;
    uint32_t per_left = a.m;  // right matrices that share one left
    if (a.family == XC_N_TO_MN) per_left = a.m / a.n;
    if (a.family == XC_ONE_TO_ONE) per_left = 1;

    // Requested tile, or the default of the family.
    direct_tile t{};
    t.ty = opt.shifts_per_thread ? pow2_floor(opt.shifts_per_thread, 16) : 0;
    t.rm = opt.right_mats_per_thread ? pow2_floor(opt.right_mats_per_thread, 8) : 0;
    t.lm = opt.left_mats_per_thread ? pow2_floor(opt.left_mats_per_thread, 4) : 0;
    t.jb = opt.rows_per_step ? pow2_floor(opt.rows_per_step, 4) : 0;
    // Defaults measured on MI355X (one_to_one 128^2, one_to_many 64 x 256^2, n_to_m 16 x 64 of
    // 64^2): one right matrix: 4 shifts x 4 rows per step; several right matrices per left:
    // 4 shifts x 2 matrices x 2 rows; n_to_m: 2 shifts x 4 right x 2 left matrices x 2 rows.
    const bool many_left = n_to_m && a.n >= 2;
    if (!t.rm) t.rm = many_left ? 4 : (per_left >= 2 ? 2 : 1);
    if (!t.lm) t.lm = many_left ? 2 : 1;
    if (!t.ty) t.ty = many_left ? 2 : 4;
    if (!t.jb) t.jb = t.rm * t.lm == 1 ? 4 : 2;
    // Matrices that do not exist are not tiled.
    t.rm = std::min<int>(t.rm, pow2_floor(per_left, 8));
    t.lm = n_to_m ? std::min<int>(t.lm, pow2_floor(a.n, 4)) : 1;
    t = round_to_catalog(t);
    direct_plan d{};
    d.t = t;
    const uint32_t SX = 2 * a.cols - 1, SY = 2 * a.rows - 1;
    // 8 waves where one block row spans 256 dx or more and there are enough groups, else 4.
    uint32_t waves = opt.waves_per_block ? (uint32_t)pow2_floor(opt.waves_per_block, 8)
                                         : (SX >= 256 && a.pairs >= 8 ? 8 : 4);
    const uint32_t need_x = (SX + 63) / 64;
    d.nwx = 1;
    while (d.nwx * 2 <= waves && d.nwx < need_x) d.nwx *= 2;
    d.nwy = waves / d.nwx;
    d.tiles_x = (SX + 64 * d.nwx - 1) / (64 * d.nwx);
    d.tiles_y = (SY + t.ty * d.nwy - 1) / (t.ty * d.nwy);
    if (n_to_m) {
        d.groups_l = (a.n + t.lm - 1) / t.lm;
        d.groups_r = (a.m + t.rm - 1) / t.rm;
    } else if (a.family == XC_N_TO_MN) {
        d.groups_l = 1;
        d.groups_r = a.n * ((per_left + t.rm - 1) / t.rm);
    } else {
        d.groups_l = 1;
        d.groups_r = (a.m + t.rm - 1) / t.rm;
    }
    // Work distribution over the right rows of each tile.
    if (opt.split && opt.rows_per_block)
        fail(XC_ERR_INVALID_ARGUMENT, "give either split (rectangle) or rows_per_block (triangle), not both");
    d.chunks = 1;
    d.rows_per_chunk = 0;
    const uint64_t base = (uint64_t)d.tiles_x * d.tiles_y * d.groups_r * d.groups_l;
    if (opt.rows_per_block) {
        d.rows_per_chunk = std::max<uint32_t>(opt.rows_per_block, (uint32_t)t.jb);
        d.chunks = (a.rows + d.rows_per_chunk - 1) / d.rows_per_chunk;
    } else if (opt.split) {
        d.chunks = std::min(opt.split, a.rows);
    } else {
        // Enough blocks to fill 256 CUs several times over: triangle chunks.
        uint32_t c = 1;
        while (base * c < 2048 && c * 2 <= a.rows / 8 + 1) c *= 2;
        if (c > 1) {
            d.rows_per_chunk = (a.rows + c - 1) / c;
            d.rows_per_chunk = std::max<uint32_t>(d.rows_per_chunk, (uint32_t)t.jb);
            d.chunks = (a.rows + d.rows_per_chunk - 1) / d.rows_per_chunk;
        }
    }
    const uint32_t cw = 4;
    d.len = (int)(((a.cols + 64 * d.nwx + cw + 8) + 3) & ~3u);
    d.lds = 2u * (uint32_t)(t.jb * t.rm) * (uint32_t)d.len * (uint32_t)sizeof(T);
    return d;
}

dk_args args_of(const family_args& a, const direct_plan& d) {
    dk_args k{};
    k.family = a.family;
    k.H = (int)a.rows;
    k.W = (int)a.cols;
    k.n = a.family == XC_ONE_TO_ONE || a.family == XC_ONE_TO_MANY ? 1 : a.n;
    k.m = a.family == XC_ONE_TO_ONE ? 1 : a.m;
    k.mpl = a.family == XC_N_TO_MN ? a.m / a.n : 0;
    k.tiles_x = d.tiles_x;
    k.tiles_y = d.tiles_y;
    k.chunks = d.chunks;
    k.rows_per_chunk = d.rows_per_chunk;
    k.groups_l = d.groups_l;
    k.groups_r = d.groups_r;
    k.nwx = d.nwx;
    k.nwy = d.nwy;
    k.len = d.len;
    k.atomic = d.chunks > 1 ? 1 : 0;
    return k;
}

// ---------------------------------------------------------------- lanes over pairs
// Definition-based FP32 kernel for batches with many rights per left (one_to_many, n_to_m,
// n_to_mn).  A wave takes one left and 64 of its rights (the pairs (left, right), one per
// lane; a left's last wave may be partial) and a tile of TY consecutive dy x 4 consecutive
// dx, so every lane
// runs the same loops: no lane spends FMAs on another lane's zero padding (the register-tile
// kernel's lanes take 64 consecutive dx and share the union of their column ranges), and
// the left values are wave-uniform scalar loads.  Per right row j and chunk of 4 columns
// c0 .. c0+3 a lane loads one quad of its right row and does TY*4*4 FMAs
//   out(dy0+y, dx0+x) += L[j+dy0+y][c0+t] * R[j][c0+t-dx0-x],   y < TY, x, t < 4,
// the right values R[j][c0-dx0-3 .. c0-dx0+4] being a window of two quads that slides by one
// quad per chunk.  The inputs come from padded copies: the rights as quads interleaved over
// slots (quad position p of row j of slot i at ((j * Q4 + p) * count + i) * 4, column q at
// position q + PL, PL = 8 + (-W mod 4), so every window starts on a quad and reads zeros
// outside [0, W)), the slots ordered so that a wave's 64 rights are consecutive (n_to_mn:
// left l's rights l, l+n, l+2n, ... at slots l*MP .. l*MP+MP-1, MP their count rounded up to
// 64; zero past the last); the lefts row-major with TY-1 zero rows above and below and rows
// padded with zeros to a multiple of 4.  Products are summed in FP32 partials of 64 that are added into
// FP64 totals.  Tiles run nearest-the-centre first (the largest overlaps start first).
struct dp_args {
    int family, H, W;
    uint32_t n, m, pairs, groups;     // groups: waves of 64 rights of one left, all lefts
    uint32_t mpl, wpl;                // rights per left, waves per left
    uint32_t tiles_y, tiles_x, nbx;   // nbx: blocks of 4 x-tiles (one per wave)
    uint32_t r_count;                 // matrices in the right copy
    int Q4, PL, Hl, Wl;               // right copy: quads per row, column offset; left copy: rows, row length
    int by_unit;                      // block order (see the kernel)
    uint32_t mp;                      // slots of the right copy per left (n_to_mn) or in all: mpl rounded up
    uint32_t gpl;                     // direct_matrix_kernel: groups of 16 rights per left
};

// Four consecutive elements of a row: 16 bytes (float) or 32 bytes (double).
template <typename T>
struct quad_of;
template <>
struct quad_of<float> {
    using type = float4;
    // the lane's quad of a right-copy quad position (base wave-uniform)
    __device__ static float4 load(const float* base, uint32_t lane_bytes) { return buffer_quad(base, lane_bytes, 0); }
};
template <>
struct quad_of<double> {
    using type = double4;
    __device__ static double4 load(const double* base, uint32_t lane_bytes) {
        const float* b = reinterpret_cast<const float*>(base);
        const double2 lo = __builtin_bit_cast(double2, buffer_quad(b, lane_bytes, 0));
        const double2 hi = __builtin_bit_cast(double2, buffer_quad(b, lane_bytes, 16));
        return make_double4(lo.x, lo.y, hi.x, hi.y);
    }
};

template <typename T, int TY>
__global__ __launch_bounds__(256) void direct_pairs_kernel(const T* __restrict__ Lc, const T* __restrict__ Rq,
                                                           T* __restrict__ O, dp_args a,
                                                           const uint32_t* __restrict__ only_if) {
    using Q = typename quad_of<T>::type;
    constexpr int TX = 4, FLUSHC = 16;  // FLUSHC chunks of 4 columns per partial sum
    if (only_if && *only_if == 0) return;  // direct_matrix_kernel has done the batch
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    // Blocks go round-robin to the 8 XCDs; tiles run nearest the centre (largest overlap)
    // first.  Right copies larger than an XCD's L2 (by_unit): a unit (one x-block of 4
    // tiles, one group of 64 pairs) keeps all its dy bands on one XCD; those waves have the
    // same column range, so they take about the same time per right row and read each row
    // while it is in that XCD's L2.  Units are dealt to the XCDs in snake order.  Smaller
    // copies: a band of TY dy (all its x-blocks and groups) per XCD, bands dealt in turn
    // (measured faster where the copy fits the L2).
    uint32_t u, band;
    if (!block_order(blockIdx.x, a.groups * a.nbx, a.tiles_y, a.by_unit, u, band)) return;
    const uint32_t g = u % a.groups;
    const int ty = center_first((int)band, (int)a.tiles_y);
    const int tx = center_first((int)(u / a.groups), (int)a.nbx) * 4 + wave;
    if (tx >= (int)a.tiles_x) return;
    const int H = a.H, W = a.W;
    const int dy0 = -(H - 1) + TY * ty, dx0 = -(W - 1) + TX * tx;
    // the wave's left and its lanes' rights (t: index among the left's rights; lanes past the
    // last right read a zero slot and store nothing)
    const uint32_t li = g / a.wpl, t = (g % a.wpl) * 64 + (uint32_t)lane;
    const bool valid = t < a.mpl;
    const uint32_t slot = (a.family == XC_N_TO_MN ? li * a.mp : 0) + min(t, a.mp - 1);
    const uint32_t pk = a.family == XC_N_TO_M ? li * a.m + t : (a.family == XC_N_TO_MN ? li + a.n * t : t);
    // right rows: those that meet a dy of the tile; columns: the union over the tile's dx,
    // from a multiple of 4
    const int jlo = max(0, -(dy0 + TY - 1)), jhi = min(H, H - dy0);
    const int clo = max(0, dx0) & ~3;
    const int nch = (min(W, W + dx0 + TX - 1) - clo + 3) >> 2;
    const uint32_t lane_bytes = slot * 4u * (uint32_t)sizeof(T);
    const int64_t rq = (int64_t)a.r_count * 4;  // elements between quad positions of one row
    const T* __restrict__ lt = Lc + ((int64_t)li * a.Hl + dy0 + TY - 1) * a.Wl + clo;  // + j * Wl: row j + dy0
    const T* __restrict__ rt = Rq + (int64_t)((clo - dx0 - 3 + a.PL) >> 2) * rq;       // + j * Q4 * rq: row j
    T acc[TY][TX];
    double tot[TY][TX];
#pragma unroll
    for (int y = 0; y < TY; ++y)
#pragma unroll
        for (int x = 0; x < TX; ++x) acc[y][x] = T(0), tot[y][x] = 0.0;
    int cnt = 0;
    auto flush = [&]() {
#pragma unroll
        for (int y = 0; y < TY; ++y)
#pragma unroll
            for (int x = 0; x < TX; ++x) {
                tot[y][x] += (double)acc[y][x];
                acc[y][x] = T(0);
            }
    };
    for (int j = jlo; j < jhi; ++j) {
        const T* __restrict__ lr = lt + (int64_t)j * a.Wl;
        const T* __restrict__ rr = rt + (int64_t)j * a.Q4 * rq;
        Q w0 = quad_of<T>::load(rr, lane_bytes), w1 = quad_of<T>::load(rr + rq, lane_bytes);
        Q lv[TY];
#pragma unroll
        for (int y = 0; y < TY; ++y) lv[y] = *reinterpret_cast<const Q*>(lr + (int64_t)y * a.Wl);
        for (int ch = 0; ch < nch; ++ch) {
            // the next chunk's values in flight during this one (the copies hold a quad past
            // the last window, the left copy a chunk past the last one)
            const Q w2 = quad_of<T>::load(rr + (ch + 2) * rq, lane_bytes);
            Q ln[TY];
#pragma unroll
            for (int y = 0; y < TY; ++y) ln[y] = *reinterpret_cast<const Q*>(lr + (int64_t)y * a.Wl + 4 * ch + 4);
            const T w[8] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w};
#pragma unroll
            for (int y = 0; y < TY; ++y) {
                const T l[4] = {lv[y].x, lv[y].y, lv[y].z, lv[y].w};
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int x = 0; x < TX; ++x) acc[y][x] = fma(l[t], w[t + 3 - x], acc[y][x]);
            }
            w0 = w1;
            w1 = w2;
#pragma unroll
            for (int y = 0; y < TY; ++y) lv[y] = ln[y];
            if (++cnt == FLUSHC) {
                flush();
                cnt = 0;
            }
        }
    }
    flush();
    if (!valid) return;
    T* __restrict__ op = O + (size_t)pk * (2 * W - 1) * (2 * H - 1);
#pragma unroll
    for (int y = 0; y < TY; ++y) {
        const int dy = dy0 + y;
        if (dy > H - 1) break;
#pragma unroll
        for (int x = 0; x < TX; ++x)
            if (dx0 + x <= W - 1) op[(size_t)(dy + H - 1) * (2 * W - 1) + (dx0 + x + W - 1)] = (T)tot[y][x];
    }
}

// Left copy: count matrices of H x W into rows of Wl (zero outside the matrix) with pad zero rows
// above and below: element (r, c) of matrix i at (i * Hl + r + pad) * Wl + c + padc.  Clears
// *flag when one is given.
template <typename T>
__global__ __launch_bounds__(256) void pairs_copy_left_kernel(const T* __restrict__ X, T* __restrict__ Xc,
                                                              uint32_t count, int H, int W, int Hl, int Wl, int pad,
                                                              int padc, uint32_t* __restrict__ flag) {
    if (flag && blockIdx.x == 0 && threadIdx.x == 0) *flag = 0;
    const uint64_t total = (uint64_t)count * Hl * Wl;
    for (uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += (uint64_t)gridDim.x * blockDim.x) {
        const int c = (int)(e % (uint64_t)Wl) - padc;
        const uint64_t rest = e / (uint64_t)Wl;
        const int r = (int)(rest % (uint64_t)Hl) - pad;
        const uint64_t i = rest / (uint64_t)Hl;
        Xc[e] = (r >= 0 && r < H && c >= 0 && c < W) ? X[(i * H + r) * W + c] : T(0);
    }
}

// Right copy: quad position p of row j of slot i at ((j * Q4 + p) * count + i) * 4, holding
// columns 4p - PL .. 4p - PL + 3 (zero outside [0, W)) of the slot's matrix: with ln = 0 slot
// i is matrix i (zero for i >= nmat); with ln lefts (n_to_mn), slot l*MP + t is matrix
// l + ln*t (zero for t >= mpl).  Thread e writes quad e.  With a flag given, *flag is set if a
// value here, or one of the lsize values of the left copy Lc, is an infinity or a NaN.
template <typename T>
__global__ __launch_bounds__(256) void pairs_copy_right_kernel(const T* __restrict__ X, T* __restrict__ Xq,
                                                               uint32_t count, uint32_t nmat, uint32_t ln,
                                                               uint32_t mp, uint32_t mpl, int H, int W, int Q4, int PL,
                                                               const T* __restrict__ Lc, uint64_t lsize,
                                                               uint32_t* __restrict__ flag) {
    const uint64_t total = (uint64_t)count * H * Q4;
    bool bad = false;
    if (flag)
        for (uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; e < lsize; e += (uint64_t)gridDim.x * blockDim.x)
            bad |= !isfinite(Lc[e]);
    for (uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t i = e % count, rest = e / count;
        const int p = (int)(rest % (uint64_t)Q4), j = (int)(rest / (uint64_t)Q4);
        uint64_t mat = i;
        bool ok = i < nmat;
        if (ln) {
            const uint64_t l = i / mp, t = i % mp;
            mat = l + (uint64_t)ln * t;
            ok = t < mpl;
        }
        const T* __restrict__ row = X + ((ok ? mat : 0) * H + j) * W;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int q = 4 * p + t - PL;
            const T v = (ok && q >= 0 && q < W) ? row[q] : T(0);
            bad |= !isfinite(v);
            Xq[e * 4 + t] = v;
        }
    }
    if (flag && bad) *flag = 1;  // every writer stores the same value
}

// The same sums on the FP32 matrix instructions (v_mfma_f32_16x16x4_f32: FP32 products and FP32
// sums at 256 FLOPs per CU and clock, twice the rate of FP32 FMAs that are not packed).  For one
// left, rights x shifts is a matrix product over the pixels: A = 16 rights x 4 pixels, B = 4 pixels
// of the left x 16 consecutive dx.  A block takes 16 rights of one left and a tile of 4 dy x 16 dx; its four waves split the tile's (right row, 16 columns) steps evenly, each wave with its own
// FP32 partial sums of 32 products and FP64 totals, which are added through LDS in a fixed
// order.  The order of the 16 pixels of a step is free as long as A and B agree: lane group k = lane /
// 16 takes columns q + 4k .. q + 4k + 3, so that a lane's four A values are one quad of the
// lanes-over-pairs kernel's right copy, and its four B values four neighbours in the left copy.  Five
// 16-byte loads, one step ahead, feed 16 instructions of 32 cycles: no LDS, no barriers.  Bound: the
// matrix instructions, 4.0 ms at 2.4 GHz of the 4.57 that 64 of 256^2 take (lanes over pairs 9.12; 120
// TFLOP/s of the definition); partial sums of 64 took 4.36, of 32 bring the error of signed
// data from 1.43e-7 to 1.04e-7 (lanes over pairs 1.45e-7); two groups of rights per wave took 4.57 too,
// with 149 registers, and twice as long where the second was idle.  16 x 64 of 64^2 700 -> 465 us.
// Columns are the union over 16 dx, rounded up to 16 (about 16 more than a single dx has), rows
// the union over 4 dy.  A zero of the copies' padding must not meet an infinity or a NaN: a batch
// that holds one (*nonfinite) is left to the kernel behind this one (launch_direct_pairs).
constexpr int kMatrixPadC = 20;  // zero columns of the left copy before column 0
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void direct_matrix_kernel(
    const float* __restrict__ Lc, const float* __restrict__ Rq, float* __restrict__ O, dp_args a,
    const uint32_t* __restrict__ nonfinite) {
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    constexpr int TY = 4;
    __shared__ double part[4][2 * 4 * 64];  // a wave's totals of two of the tile's dy
    if (*nonfinite) return;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63, l16 = lane & 15, kg = lane >> 4;
    const uint32_t groups = a.n * a.gpl;
    uint32_t u, band;
    if (!block_order(blockIdx.x, groups * a.tiles_x, a.tiles_y, a.by_unit, u, band)) return;
    const uint32_t g = u % groups, li = g / a.gpl, t0 = (g % a.gpl) * 16;
    const int H = a.H, W = a.W;
    const int dy0 = -(H - 1) + TY * center_first((int)band, (int)a.tiles_y);
    const int dx0 = -(W - 1) + 16 * center_first((int)(u / groups), (int)a.tiles_x);
    // right rows and columns that meet the tile, the first column on a quad of the right copy
    const int jlo = max(0, -(dy0 + TY - 1)), jhi = min(H, H - dy0);
    const int qmin = max(0, -(dx0 + 15)), qlo = qmin - ((qmin + a.PL) & 3);
    const int nch = (min(W, W - dx0) - qlo + 15) >> 4;
    const int steps = (jhi - jlo) * nch;
    const int s0 = (int)((int64_t)steps * wave >> 2), s1 = (int)((int64_t)steps * (wave + 1) >> 2);
    const int64_t rq = (int64_t)a.r_count * 4;  // elements between quad positions of one row
    const uint32_t slot = (a.family == XC_N_TO_MN ? li * a.mp : 0) + t0 + (uint32_t)l16;
    const uint32_t a_off = (uint32_t)kg * (uint32_t)(rq * 4) + slot * 16u;
    const uint32_t b_off = (uint32_t)(4 * kg + l16) * 4u;
    const float* __restrict__ at = Rq + (int64_t)((qlo + a.PL) >> 2) * rq;
    const float* __restrict__ bt = Lc + ((int64_t)li * a.Hl + dy0 + TY - 1) * a.Wl + kMatrixPadC + qlo + dx0;
    f32x4 acc[TY];
    double tot[TY][4];
#pragma unroll
    for (int y = 0; y < TY; ++y)
#pragma unroll
        for (int r = 0; r < 4; ++r) tot[y][r] = 0.0;
    auto load = [&](int j, int ch, float4& av, float4 (&bv)[TY]) {
        const float* bp = bt + (int64_t)j * a.Wl + 16 * ch;
        av = buffer_quad(at + ((int64_t)j * a.Q4 + 4 * ch) * rq, a_off, 0);
#pragma unroll
        for (int y = 0; y < TY; ++y) bv[y] = buffer_quad(bp + (int64_t)y * a.Wl, b_off, 0);
    };
    if (s0 < s1) {
        int j = jlo + s0 / nch, ch = s0 % nch;
        float4 a0, b0[TY], a1, b1[TY];
        auto next = [&](int s, float4& av, float4 (&bv)[TY]) {
            if (s + 1 < s1 && ++ch == nch) {  // the last step loads itself again
                ch = 0;
                ++j;
            }
            load(j, ch, av, bv);
            __builtin_amdgcn_sched_barrier(0);  // in flight before this step's products, not behind them
        };
        auto products = [&](const float4& av, const float4 (&bv)[TY], auto first) {
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int y = 0; y < TY; ++y) {
                    const f32x4 c = decltype(first)::value && t == 0 ? f32x4{0, 0, 0, 0} : acc[y];
                    acc[y] = __builtin_amdgcn_mfma_f32_16x16x4f32((&av.x)[t], (&bv[y].x)[t], c, 0, 0, 0);
                }
        };
        load(j, ch, a0, b0);
        for (int s = s0; s < s1; s += 2) {
            next(s, a1, b1);
            products(a0, b0, std::true_type{});
            if (s + 1 < s1) {
                next(s + 1, a0, b0);
                products(a1, b1, std::false_type{});
            }
#pragma unroll
            for (int y = 0; y < TY; ++y)
#pragma unroll
                for (int r = 0; r < 4; ++r) tot[y][r] += (double)acc[y][r];
        }
    }
    // the waves' totals, two dy at a time; lane `el` of a tile holds dx el % 16 of rights 4 (el / 16) + r
    const int SX = 2 * W - 1, SY = 2 * H - 1;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        if (h) __syncthreads();
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
            for (int r = 0; r < 4; ++r) part[wave][(4 * y + r) * 64 + lane] = tot[2 * h + y][r];
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int e = (int)threadIdx.x + 256 * q;
            const double v = ((part[0][e] + part[1][e]) + part[2][e]) + part[3][e];
            const int el = e & 63, r = (e >> 6) & 3, y = e >> 8;
            const int oy = dy0 + 2 * h + y + H - 1, ox = dx0 + (el & 15) + W - 1;
            const uint32_t t = t0 + (uint32_t)(4 * (el >> 4) + r);
            const uint32_t pk = a.family == XC_N_TO_M ? li * a.m + t : (a.family == XC_N_TO_MN ? li + a.n * t : t);
            if (t < a.mpl && oy < SY && ox < SX) O[((size_t)pk * SY + oy) * SX + ox] = (float)v;
        }
    }
}

constexpr int kPairsTY = 4;

// Rights per left of a family (0: one_to_one, which the kernel does not serve).
uint32_t rights_per_left(const family_args& a) {
    switch (a.family) {
    case XC_ONE_TO_MANY: return a.m;
    case XC_N_TO_M: return a.m;
    case XC_N_TO_MN: return a.m / a.n;
    default: return 0;
    }
}

// Waves of the lanes-over-pairs kernel.
uint64_t pairs_kernel_waves(const family_args& a) {
    const uint32_t nl = a.family == XC_ONE_TO_MANY ? 1 : a.n;
    return (uint64_t)nl * ((rights_per_left(a) + 63) / 64) * ((2 * a.rows - 1 + kPairsTY - 1) / kPairsTY) *
           ((2 * a.cols - 1 + 3) / 4);
}

bool one_row_by_pairs(const family_args& a) {
    return a.rows == 1 && a.cols > 32 && a.cols <= 256 && a.family != XC_N_TO_M;
}

// Whether the lanes-over-pairs kernel serves this batch by default: at least 48 rights per left
// (a wave's lanes at least 3/4 busy below 64), its copy of the rights (the other kernels need
// none) at most 16 GiB, and enough waves.  Double data: 2048 waves (against the register tiles
// 0.45-0.9x at 128-1024 waves, 1.14x at 2048, 1.6-2.2x from 4096).  Float data competes with the matrix
// kernel, whose 16 dx and 16 columns are mostly padding in narrow matrices, and with the 16 x 16 shifts,
// whose 16 dx are; a wave's time does not shrink with its pairs, so the lines lie at waves * (busy
// lanes)^3, by columns.  Up to 4 all of 2048 waves (us, pairs / the faster of the two: 20 x 186 of 142x1
// 80 / 365, 24 x 107 of 305x1 208 / 1064, 28 x 78 of 397x3 743 / 1500, 4 x 218 of 205x3 103 / 191); 5 columns
// 2000 (51 x 73 of 365x5 1914 / 2260, 323 of 380x5 242 / 221); 6 to 12 4000 (17 x 49 of 283x7 304 / 413, 3 x 78 of
// 247x8 171 / 98, 113 calls past 4500 0.87 of the time, 2 x 271 of 247x8 285 / 163); 13 to 15 columns none (54 calls
// 1.4 times).  One row, whose few steps the matrix kernel's four waves share: 33 to 256 columns, rights of
// one left only and 6000 waves (20253 of 1x37 25 / 31, 39512 of 1x63 68 / 95, 12316 of 1x87 34 / 42, 12400 of
// 1x38 51 / 24, 3 x 5345 of 1x300 283 / 263, n_to_m 17 x 1056 of 1x98 208 / 59).  The last rule is for batches
// whose copies are too large for the matrix kernel: against the 16 x 16 shifts 100 of 128^2 1563 / 1287, 4 x 50
// of 100^2 950 / 1283, 56 of 200^2 3805 / 4499, 80 of 256^2 16620 / 15070.
bool pairs_kernel_applies(const family_args& a, bool float_data) {
    const uint32_t mpl = rights_per_left(a);
    if (mpl < 48) return false;
    const uint64_t lefts = a.family == XC_ONE_TO_MANY ? 1 : a.n;
    const uint64_t slots = (a.family == XC_N_TO_MN ? lefts : 1) * ((mpl + 63) / 64 * 64);
    const uint64_t copy = slots * a.rows * (a.cols + 24) * sizeof(float);
    if (copy > (16ull << 30)) return false;
    const double busy = (double)mpl / (double)((mpl + 63) / 64 * 64), waves = (double)pairs_kernel_waves(a);
    if (!float_data || a.cols <= 4) return waves >= 2048;
    const double full = waves * busy * busy * busy;
    if (a.cols <= 12) return full >= (a.cols == 5 ? 2000 : 4000);
    if (one_row_by_pairs(a)) return waves >= 6000;
    return busy == 1.0 ? waves >= 2048 : busy >= 0.7 && full >= 4500;
}

bool matrix_copies_fit(const family_args& a) {
    const uint32_t mpl = rights_per_left(a);
    if (mpl == 0) return false;
    const double lefts = a.family == XC_ONE_TO_MANY ? 1 : a.n, H = a.rows, W = a.cols;
    const double slots = (a.family == XC_N_TO_MN ? lefts : 1) * ((mpl + 15) / 16 * 16);
    const double copies = slots * H * (W + 27) + lefts * (H + 6) * (W + 55);
    return copies * sizeof(float) <= (double)(16ull << 30) && slots * 64 < (double)(1u << 31);
}

// Whether direct_matrix_kernel serves this float batch by default: its copies of both sides at most 16
// GiB, and a shorter estimated time than the 16 x 16 shifts kernel's.  Both estimates are products
// issued (the padding of tiles and of groups of 16 rights among them) over a rate, plus the launches;
// the matrix kernel's also six steps per wave for its start and end, and 0.6 of its longest wave,
// which small grids wait for.  Measured us, matrix / shifts: 8 of 128^2 127 / 115, 10 of 128^2 127 / 143,
// 48 of 128^2 298 / 590, 64 of 128^2 380 / 800 (lanes over pairs 898), 16 of 64^2 34 / 27, 32 of 64^2 37 / 47,
// 20 x 10 of 64^2 149 / 190, 64 of 32^2 18 / 14, 256 of 32^2 28 / 33, 8 of 256^2 1228 / 1552.  Up to
// 12 columns, and for single rows, the lanes-over-pairs kernel is asked first (200 x 64 of 10^2 59 / 86 us).
bool matrix_kernel_applies(const family_args& a) {
    const uint32_t mpl = rights_per_left(a);
    if (!matrix_copies_fit(a)) return false;
    const double lefts = a.family == XC_ONE_TO_MANY ? 1 : a.n, groups = lefts * ((mpl + 15) / 16);
    const double H = a.rows, W = a.cols;
    if ((a.cols <= 12 || one_row_by_pairs(a)) && pairs_kernel_applies(a, true)) return false;
    const double SX = (2 * a.cols - 1 + 15) / 16 * 16, SY = (2 * a.rows - 1 + 3) / 4 * 4;
    const double SYs = (2 * a.rows - 1 + 15) / 16 * 16;
    const double step = 512 / 2.4e3, waves = groups * (SX / 16) * (SY / 4) * 4;  // us of a step; waves
    const double matrix = 12 + groups * 16 * SX * SY * (H / 2 + 2) * (W / 2 + 16.5) / 68e6 +
                          waves * 6 * step / 1024 + 0.6 * step * (H / 4) * std::ceil((W + 15) / 16);
    const double shifts = 10 + lefts * mpl * SX * SYs * (H / 2 + 8) * (W / 2 + 8) / 25e6;
    return matrix < shifts;
}

// The register tiles behind direct_matrix_kernel, in one chunk (no atomics, which would need a zeroed
// output): the plan, and its kernel if it is one of the defaults for several rights per left.
const void* tiles_behind(const family_args& a, direct_plan& d) {
    xc_options o{};
    o.split = 1;
    d = plan_direct<float>(a, o);
    const uint64_t nblocks = (uint64_t)d.tiles_x * d.tiles_y * d.groups_r * d.groups_l;
    if (d.lds > 160 * 1024 || !fits_one_launch(nblocks, 64 * d.nwx * d.nwy)) return nullptr;
    if (d.t.ty == 4 && d.t.rm == 2 && d.t.lm == 1 && d.t.jb == 2)
        return reinterpret_cast<const void*>(&direct_kernel<float, 4, 2, 1, 2, true>);
    if (d.t.ty == 2 && d.t.rm == 4 && d.t.lm == 2 && d.t.jb == 2)
        return reinterpret_cast<const void*>(&direct_kernel<float, 2, 4, 2, 2, true>);
    return nullptr;
}

void launch_tiles_behind(const family_args& a, const float* L, const float* R, float* O, const direct_plan& d,
                         const void* fn, const uint32_t* flag, hipStream_t s) {
    dk_args k = args_of(a, d);
    k.only_if = flag;
    if (d.lds > 65536) allow_dynamic_lds(fn, d.lds);
    void* args[] = {(void*)&L, (void*)&R, (void*)&O, (void*)&k};
    XC_HIP(hipLaunchKernel(fn, dim3(d.tiles_x * d.tiles_y * d.groups_r * d.groups_l), dim3(64 * d.nwx * d.nwy), args,
                           d.lds, s));
}

// matrix: by direct_matrix_kernel, with another kernel behind it for data that is not finite: up to 39
// rights per left the register tiles, from 40 on direct_pairs_kernel, whose lanes are then 5/8 busy.
// us with a NaN, tiles / pairs behind (the tiles by themselves): 16 of 128^2 569 / 1167 (391), 32 of 200^2
// 3170 / 3700 (3090), 16 x 12 of 64^2 484 / 640 (288).
// False (nothing launched) if there is no memory for the copies, unless the kernel is `asked` for by
// the caller (then an error), or if a grid does not fit one launch.
template <typename T>
bool launch_direct_pairs(const family_args& a, const T* L, const T* R, T* O, hipStream_t s, bool matrix, bool asked) {
    constexpr int TY = kPairsTY;
    const int H = (int)a.rows, W = (int)a.cols;
    const uint32_t nl = a.family == XC_ONE_TO_MANY ? 1 : a.n;
    dp_args k{};
    k.family = a.family;
    k.H = H;
    k.W = W;
    k.n = nl;
    k.m = a.m;
    k.pairs = a.pairs;
    k.mpl = rights_per_left(a);
    k.wpl = (k.mpl + 63) / 64;
    k.groups = nl * k.wpl;
    // right slots: the rights in order, padded to a multiple of 64 (16 for the matrix kernel);
    // n_to_mn: per left, its rights, padded to such a multiple each
    k.mp = matrix ? (k.mpl + 15) / 16 * 16 : k.wpl * 64;
    const uint32_t nr = a.family == XC_N_TO_MN ? nl * k.mp : k.mp;
    k.tiles_y = (uint32_t)(2 * H - 1 + TY - 1) / TY;
    k.tiles_x = (uint32_t)(2 * W - 1 + 3) / 4;
    k.nbx = (k.tiles_x + 3) / 4;
    k.r_count = nr;
    k.PL = 8 + (4 - W % 4) % 4;
    k.Q4 = (k.PL + W + (matrix ? 16 : 12) + 3) / 4;  // a quad past the last window; a step of 16 columns
    k.Hl = H + 2 * (TY - 1);
    // a chunk past the last one (prefetch); 16 columns and 16 dx past the last column
    const int padc = matrix ? kMatrixPadC : 0;
    k.Wl = matrix ? (padc + W + 32 + 3) / 4 * 4 : (W + 3) / 4 * 4 + 4;
    if ((uint64_t)nr * 4 * sizeof(T) + 16 >= (1ull << 31)) fail(XC_ERR_UNSUPPORTED, "direct kernel: too many right matrices");
    const uint64_t lsize = (uint64_t)nl * k.Hl * k.Wl, rsize = (uint64_t)nr * H * k.Q4 * 4;
    const size_t bytes = sizeof(T) * (lsize + rsize) + sizeof(uint32_t);
    k.by_unit = rsize * sizeof(T) > (4u << 20);  // larger than one XCD's L2
    const uint64_t punits = (uint64_t)k.groups * k.nbx;
    const uint64_t nblocks = blocks_for_order((uint32_t)punits, k.tiles_y, k.by_unit);
    dp_args mk = k;  // of the matrix kernel
    mk.gpl = k.mp / 16;
    mk.tiles_x = (uint32_t)(2 * W - 1 + 15) / 16;
    const uint64_t units = (uint64_t)nl * mk.gpl * mk.tiles_x;
    // a unit's bands on one XCD (16 of 128^2 127 us; bands dealt to the XCDs in turn 179: each CU's
    // blocks are then the same units of several bands), unless that leaves XCDs idle
    mk.by_unit = (units + 7) / 8 * 8 * 10 <= units * 11;
    const uint64_t mblocks = blocks_for_order((uint32_t)units, k.tiles_y, mk.by_unit);
    direct_plan behind{};
    const void* tiles = matrix && k.mpl < 40 ? tiles_behind(a, behind) : nullptr;
    if ((!tiles && !fits_one_launch(std::max(punits, nblocks), 256)) ||
        (matrix && !fits_one_launch(std::max(units, mblocks), 256)))
        return false;
    T* Lc = static_cast<T*>(asked ? workspace(WS_DIRECT, bytes, s) : workspace_if_free(WS_DIRECT, bytes, s));
    if (!Lc) return false;
    T* Rq = Lc + lsize;
    uint32_t* flag = matrix ? reinterpret_cast<uint32_t*>(Rq + rsize) : nullptr;
    auto blocks_for = [](uint64_t n) { return (uint32_t)std::min<uint64_t>((n + 255) / 256, 16384); };
    hipLaunchKernelGGL(pairs_copy_left_kernel<T>, dim3(blocks_for(lsize)), dim3(256), 0, s, L, Lc, nl, H, W, k.Hl,
                       k.Wl, TY - 1, padc, flag);
    XC_HIP(hipGetLastError());
    // with a flag it reads the lefts too, of which there may be far more than rights (62544 pairs of 5212
    // lefts of 1x2 1999 us with blocks for 12 rights only, the tiles 58)
    const uint64_t copied = std::max(rsize / 4, flag ? lsize / 4 : 0);
    hipLaunchKernelGGL(pairs_copy_right_kernel<T>, dim3(blocks_for(copied)), dim3(256), 0, s, R, Rq, nr, a.m,
                       a.family == XC_N_TO_MN ? nl : 0u, k.mp, k.mpl, H, W, k.Q4, k.PL, Lc, lsize, flag);
    XC_HIP(hipGetLastError());
    if constexpr (std::is_same<T, float>::value) {
        if (matrix) {
            const dim3 grid((uint32_t)mblocks), block(256);
            record_launch("direct_pairs_kernel<f32> matrix instructions", grid, block, 0, a.rows, a.cols, a.pairs, 1);
            timed td("direct_kernel", s);
            hipLaunchKernelGGL(direct_matrix_kernel, grid, block, 0, s, Lc, Rq, O, mk, flag);
            XC_HIP(hipGetLastError());
        }
        if (tiles) {
            launch_tiles_behind(a, L, R, O, behind, tiles, flag, s);
            return true;
        }
    }
    dim3 grid((uint32_t)nblocks), block(256);
    if (!matrix)
        record_launch(sizeof(T) == 4 ? "direct_pairs_kernel<f32> ty4 tx4" : "direct_pairs_kernel<f64> ty4 tx4", grid,
                      block, 0, a.rows, a.cols, a.pairs, 1);
    timed td("direct_kernel", s, !matrix);
    hipLaunchKernelGGL((direct_pairs_kernel<T, TY>), grid, block, 0, s, Lc + padc, Rq, O, k,
                       static_cast<const uint32_t*>(flag));
    XC_HIP(hipGetLastError());
    return true;
}

// ---------------------------------------------------------------- lanes over shifts and rows
// Definition-based FP32 kernel for batches with few rights per left.  A block takes one pair and
// a tile of 16 dy x 16 dx; its NW waves have four groups of 16 lanes each, and each of the 4 NW
// groups sums its share of the tile's right rows.  A lane holds 4 x 4 outputs (lane gx + 4 gy of
// a group: dx0 + 4 gx .., dy0 + 4 gy ..).  The inputs go through the wave's own LDS in panels of
// 8 right rows x 16 columns (zeros outside the matrices), the next panel's values loaded into
// registers meanwhile; per right row and 4 columns a lane does 64 FMAs from three 16-byte LDS
// reads (two quads of the right row: the 7 values of its window; one quad of the left row that
// enters, the other three rows stay in registers):
//   out(dy0+y, dx0+x) += L[j+dy0+y][c0+t] * R[j][c0+t-dx0-x].
// No barriers until the groups' FP64 totals are added through LDS at the end, in a fixed order.
//
// Bound: FP32 FMAs (LDS a fifth of the FMAs' time): 22.8 T products/s at 40 pairs of 256^2, where
// the register tiles run 17.8; n_to_m 2 x 6 of 100x120 349 -> 137 us, 1 pair of 512^2 9.5 -> 3.4 ms.
// All lanes of a tile share one column range and one row range, the unions over 16 shifts: (W/2 +
// 8)(H/2 + 8) products issued per W/2 * H/2, where the register tiles' 64-dx waves issue W/2 + 32
// columns and take 32 4-byte LDS reads per 128 FMAs.  A value that is not finite reaches only the
// shifts whose overlap holds it: its products are added after the panels (direct_shifts_nonfinite).
struct ds_args {
    int family, H, W;
    uint32_t n, m, pairs, tiles_x, tiles_y;
};

struct ds_panel {
    static constexpr int JP = 8, CP = 16;            // right rows x columns
    static constexpr int NLR = JP + 15;              // left rows
    static constexpr int RQ = 68, LQ = 129, LS = 5;  // quads: right part, left part of a group, left row stride (bank spread)
    static constexpr int WQ = 4 * (RQ + LQ);         // quads of a wave
};
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) f32x4 lds_quad;
typedef __attribute__((address_space(3))) float lds_float;
typedef __attribute__((address_space(3))) double lds_double;

__device__ __forceinline__ void wave_lds_sync() {  // the wave's own LDS: ordering its accesses is enough
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// The products of the first JN right rows of a panel in LDS (rq, lq: a group's right and left part).  An
// FP32 sum takes 8 columns of the panel's rows, at most 64 products; `narrow` (matrices of one panel's
// columns) 4, since the register tiles' sums of such matrices ended with each step's rows: 100x12, signed
// data, relative error in the 2-norm 9.6e-8 with 8 columns, 7.8e-8 with 4, the
// tiles 9.0e-8.
template <int JN, typename Quad>
__device__ __forceinline__ void sum_panel(const Quad* rq, const Quad* lq, int gx, int gy, bool narrow,
                                          float (&acc)[4][4], double (&tot)[4][4]) {
#pragma unroll 1
    for (int q = 0; q < ds_panel::CP / 4; ++q) {
        const Quad* rrow = rq + (q - gx + 3);
        const Quad* lrow = lq + 4 * gy * ds_panel::LS + q;
        float l[4][4];
#pragma unroll
        for (int y = 0; y < 3; ++y) {
            const auto v = lrow[y * ds_panel::LS];
            l[y + 1][0] = v.x, l[y + 1][1] = v.y, l[y + 1][2] = v.z, l[y + 1][3] = v.w;
        }
#pragma unroll
        for (int j = 0; j < JN; ++j) {
#pragma unroll
            for (int y = 0; y < 3; ++y)
#pragma unroll
                for (int t = 0; t < 4; ++t) l[y][t] = l[y + 1][t];
            const auto v = lrow[(j + 3) * ds_panel::LS];
            l[3][0] = v.x, l[3][1] = v.y, l[3][2] = v.z, l[3][3] = v.w;
            const auto w0 = rrow[j * 8], w1 = rrow[j * 8 + 1];
            float w[8] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w};
            asm volatile("" : "+v"(w[0]));  // not used: keeps the quad one 16-byte read
#pragma unroll
            for (int y = 0; y < 4; ++y)
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int x = 0; x < 4; ++x) acc[y][x] = fmaf(l[y][t], w[t - x + 4], acc[y][x]);
        }
        if ((q & 1) || narrow) {
#pragma unroll
            for (int y = 0; y < 4; ++y)
#pragma unroll
                for (int x = 0; x < 4; ++x) tot[y][x] += (double)acc[y][x], acc[y][x] = 0.f;
        }
    }
}

// The sums of a wave that met a value that is not finite, again: the same sums with zeros in place of
// these values, and then what they bring to the shifts whose overlap holds them.  A NaN makes NaN of
// such a shift whatever its factor: bit masks of a row's NaNs against each shift's columns.  An infinity
// meets its factors one by one.  Leaves the totals in the wave's LDS as the kernel does.  A call of its
// own, so that the kernel keeps its registers.  Data with one NaN per right or left, with 1% of NaNs, and
// finite data, us (the register tiles take as long either way): 2 x 6 of 100x120 215, 468, 140 (341); 4 x
// 4 of 300^2 11730, 15240, 6100 (19900); 8 x 4 of 64^2 110, 192, 48 (90); 1 x 4 of 10^2 20, 21, 7 (13.6).
__device__ __attribute__((noinline)) void direct_shifts_again(const float* Lp, const float* Rp, lds_quad* wave_lds, int H,
                                                              int W, int dx0, int dy0, int js, int je, int clo,
                                                              int cpanels, int panels) {
    using P = ds_panel;
    const int lane = threadIdx.x & 63, g = lane >> 4, l16 = lane & 15, gx = lane & 3, gy = (lane >> 2) & 3;
    lds_quad* const rq = wave_lds + g * P::RQ;
    lds_quad* const lq = wave_lds + 4 * P::RQ + g * P::LQ;
    lds_float* const rp = reinterpret_cast<lds_float*>(rq);
    lds_float* const lp = reinterpret_cast<lds_float*>(lq);
    // This lane's values of panel p.
    float pr[2 * P::JP], pl[P::NLR];
    auto load = [&](int p) {
        const int j0 = js + p / cpanels * P::JP, c = clo + p % cpanels * P::CP + l16, q0 = c - dx0 - 16;
#pragma unroll
        for (int k = 0; k < 2 * P::JP; ++k) {
            const int j = j0 + (k >> 1), q = q0 + 16 * (k & 1);
            pr[k] = j < je && q >= 0 && q < W ? Rp[(size_t)j * W + q] : 0.f;
        }
#pragma unroll
        for (int k = 0; k < P::NLR; ++k) {
            const int r = j0 + dy0 + k;
            pl[k] = r >= 0 && r < H && c < W ? Lp[(size_t)r * W + c] : 0.f;
        }
    };
    auto store = [&] {
#pragma unroll
        for (int k = 0; k < 2 * P::JP; ++k) rp[l16 + k * 16] = pr[k];
#pragma unroll
        for (int k = 0; k < P::NLR; ++k) lp[l16 + k * 4 * P::LS] = pl[k];
        wave_lds_sync();
    };
    double tot[4][4];
    int p0 = panels, p1 = -1;  // the panels with such values
    {
        float acc[4][4];
#pragma unroll
        for (int y = 0; y < 4; ++y)
#pragma unroll
            for (int x = 0; x < 4; ++x) acc[y][x] = 0.f, tot[y][x] = 0.0;
        for (int p = 0; p < panels; ++p) {
            load(p);
            bool finite = true;
#pragma unroll
            for (int k = 0; k < 2 * P::JP; ++k) {
                finite = finite & __builtin_isfinite(pr[k]);
                pr[k] = __builtin_isfinite(pr[k]) ? pr[k] : 0.f;
            }
#pragma unroll
            for (int k = 0; k < P::NLR; ++k) {
                finite = finite & __builtin_isfinite(pl[k]);
                pl[k] = __builtin_isfinite(pl[k]) ? pl[k] : 0.f;
            }
            if (!__all(finite)) p0 = min(p0, p), p1 = p;
            store();
            sum_panel<P::JP>(rq, lq, gx, gy, W <= P::CP, acc, tot);
            wave_lds_sync();  // the next panel overwrites this one
        }
    }
    uint32_t nan = 0;  // bit 4 y + x: shift (y, x) is NaN, or beyond the result's edges
#pragma unroll
    for (int y = 0; y < 4; ++y)
#pragma unroll
        for (int x = 0; x < 4; ++x)
            nan |= dx0 + 4 * gx + x >= W || dy0 + 4 * gy + y >= H ? 1u << (4 * y + x) : 0u;
    auto spread = [](uint32_t y) { return (y & 1) | (y & 2) << 3 | (y & 4) << 6 | (y & 8) << 9; };
    for (int p = p0; p <= p1 && __any(nan != 0xffffu && js < je); ++p) {
        const int j0 = js + p / cpanels * P::JP, c0 = clo + p % cpanels * P::CP, q0 = c0 - dx0 - 16;
        const int jn = min(P::JP, je - j0), cn = min(P::CP, W - c0);
        load(p);
        store();
        // per shift x: the panel's left columns whose right column lies in the matrix, and the right
        // columns of all its left columns; left rows in the matrix
        uint32_t cm[4], qm[4], rm = 0;
#pragma unroll
        for (int x = 0; x < 4; ++x) {
            const int d = 16 - 4 * gx - x;  // right column of the window = left column of the panel + d
            cm[x] = 0;
#pragma unroll
            for (int c = 0; c < P::CP; ++c) cm[x] |= c < cn && (uint32_t)(q0 + c + d) < (uint32_t)W ? 1u << c : 0u;
            qm[x] = ((1u << cn) - 1) << d;
        }
#pragma unroll
        for (int k = 0; k < P::NLR; ++k) rm |= (uint32_t)(j0 + dy0 + k) < (uint32_t)H ? 1u << k : 0u;
#pragma unroll 1
        for (int j = 0; j < P::JP; ++j) {
            const float v0 = rp[l16 + j * 32], v1 = rp[l16 + j * 32 + 16];
            if (__all(__builtin_isfinite(v0) && __builtin_isfinite(v1))) continue;
            const uint32_t ym = j < jn ? rm >> (j + 4 * gy) & 15u : 0u;
            const uint32_t nans = ((uint32_t)(__ballot(v0 != v0) >> (16 * g)) & 0xffffu) |
                                  (uint32_t)(__ballot(v1 != v1) >> (16 * g)) << 16;
#pragma unroll
            for (int x = 0; x < 4; ++x) nan |= nans & qm[x] ? spread(ym) << x : 0u;
            uint32_t infs = ((uint32_t)(__ballot(__builtin_isinf(v0)) >> (16 * g)) & 0xffffu) |
                            (uint32_t)(__ballot(__builtin_isinf(v1)) >> (16 * g)) << 16;
            for (; __any(infs != 0); infs &= infs - 1) {
                const int q = infs ? __builtin_ctz(infs) : 16;
                const float v = infs ? (float)rp[j * 32 + q] : 0.f;
#pragma unroll
                for (int x = 0; x < 4; ++x) {
                    const int c = q - 16 + 4 * gx + x;
#pragma unroll
                    for (int y = 0; y < 4; ++y)
                        if (infs && (uint32_t)c < (uint32_t)cn && (ym >> y & 1))
                            tot[y][x] += (double)(v * lp[c + (j + 4 * gy + y) * 4 * P::LS]);
                }
            }
        }
#pragma unroll 1
        for (int k = 0; k < P::NLR; ++k) {
            const float v0 = lp[l16 + k * 4 * P::LS];
            if (__all(__builtin_isfinite(v0))) continue;
            uint32_t ym = 0;
#pragma unroll
            for (int y = 0; y < 4; ++y) ym |= (uint32_t)(k - 4 * gy - y) < (uint32_t)max(jn, 0) ? 1u << y : 0u;
            const uint32_t nans = (uint32_t)(__ballot(v0 != v0) >> (16 * g)) & 0xffffu;
#pragma unroll
            for (int x = 0; x < 4; ++x) nan |= nans & cm[x] ? spread(ym) << x : 0u;
            uint32_t infs = (uint32_t)(__ballot(__builtin_isinf(v0)) >> (16 * g)) & 0xffffu;
            for (; __any(infs != 0); infs &= infs - 1) {
                const int c = infs ? __builtin_ctz(infs) : 0;
                const float v = infs ? (float)lp[c + k * 4 * P::LS] : 0.f;
#pragma unroll
                for (int x = 0; x < 4; ++x)
#pragma unroll
                    for (int y = 0; y < 4; ++y)
                        if (infs && (cm[x] >> c & 1) && (ym >> y & 1)) {
                            const float w = rp[(k - 4 * gy - y) * 32 + c + 16 - 4 * gx - x];
                            if (!__builtin_isinf(w)) tot[y][x] += (double)(v * w);  // else it has met this one
                        }
            }
        }
#pragma unroll
        for (int y = 0; y < 4; ++y)
#pragma unroll
            for (int x = 0; x < 4; ++x) nan |= tot[y][x] != tot[y][x] ? 1u << (4 * y + x) : 0u;
        wave_lds_sync();  // the next panel, or the totals, overwrite this one
    }
    auto* const td = reinterpret_cast<lds_double*>(wave_lds) + g * 256;
#pragma unroll
    for (int y = 0; y < 4; ++y)
#pragma unroll
        for (int x = 0; x < 4; ++x)
            td[(4 * gy + y) * 16 + 4 * gx + x] = nan >> (4 * y + x) & 1 ? __builtin_nan("") : tot[y][x];
}

template <int NW>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(3))) void direct_shifts_kernel(const float* __restrict__ L,
                                                                const float* __restrict__ R, float* __restrict__ O,
                                                                ds_args a) {
    constexpr int JP = ds_panel::JP, CP = ds_panel::CP, NLR = ds_panel::NLR;
    constexpr int RQ = ds_panel::RQ, LQ = ds_panel::LQ, LS = ds_panel::LS, WQ = ds_panel::WQ;
    __shared__ float4 smem[NW * WQ];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int g = lane >> 4, l16 = lane & 15, gx = lane & 3, gy = (lane >> 2) & 3;
    // tiles nearest the centre (the longest sums) first, all pairs of a tile together
    uint32_t bid = xcd_remap(blockIdx.x, gridDim.x);
    const uint32_t pair = bid % a.pairs;
    bid /= a.pairs;
    const int tx = center_first((int)(bid % a.tiles_x), (int)a.tiles_x);
    const int ty = center_first((int)(bid / a.tiles_x), (int)a.tiles_y);
    const int H = a.H, W = a.W, dx0 = -(W - 1) + 16 * tx, dy0 = -(H - 1) + 16 * ty;
    uint32_t li, ri;
    pair_of(a.family, a.n, a.m, pair, li, ri);
    const float* __restrict__ Lp = L + (size_t)li * H * W;
    const float* __restrict__ Rp = R + (size_t)ri * H * W;
    const int jlo = max(0, -(dy0 + 15)), cnt = min(H, H - dy0) - jlo;
    const int clo = max(0, dx0), chi = min(W, W + dx0 + 15);
    const int split = wave * 4 + g;
    const int js = jlo + cnt * split / (4 * NW), je = jlo + cnt * (split + 1) / (4 * NW);
    const int jpanels = (cnt + 4 * NW * JP - 1) / (4 * NW * JP), cpanels = (chi - clo + CP - 1) / CP;

    float4* const rq = smem + wave * WQ + g * RQ;
    float4* const lq = smem + wave * WQ + 4 * RQ + g * LQ;
    float* const rw = reinterpret_cast<float*>(rq) + l16;
    float* const lw = reinterpret_cast<float*>(lq) + l16;
    float pr[2 * JP], pl[NLR];
    // This lane's share of the panel at right row j0, column c0: right columns c0 - dx0 - 16 + l16
    // and the 16 after, left column c0 + l16.  Bounds-checked buffer loads: rows outside a matrix
    // fall outside its bytes, columns outside it get an offset that does (kOut; the launcher keeps
    // matrices below 2^31 bytes), and both read zero without a select after the load, which
    // would have to wait for it.
    constexpr uint32_t kOut = 0x80000000u;
    const uint32_t bytes = (uint32_t)H * (uint32_t)W * 4u, pitch = (uint32_t)W * 4u;
    const __amdgpu_buffer_rsrc_t rl = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(Lp), 0, bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rr = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(Rp), 0, bytes, 0x00020000);
    auto load = [](const __amdgpu_buffer_rsrc_t rsrc, uint32_t offset) {
        return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)offset, 0, 0));
    };
    auto fetch = [&](int j0, int c0) {
        const int q0 = c0 - dx0 - 16 + l16, q1 = q0 + 16, c = c0 + l16;
        const uint32_t row = (uint32_t)j0 * pitch;
        const uint32_t o0 = q0 >= 0 && q0 < W ? row + (uint32_t)q0 * 4u : kOut;
        const uint32_t o1 = q1 >= 0 && q1 < W ? row + (uint32_t)q1 * 4u : kOut;
        const uint32_t ol = c < W ? (uint32_t)(j0 + dy0) * pitch + (uint32_t)c * 4u : kOut;
#pragma unroll
        for (int k = 0; k < JP; ++k) {
            const bool in = j0 + k < je;  // the group's share of the rows ends here
            pr[2 * k] = load(rr, in ? o0 + k * pitch : kOut);
            pr[2 * k + 1] = load(rr, in ? o1 + k * pitch : kOut);
        }
#pragma unroll
        for (int k = 0; k < NLR; ++k) pl[k] = load(rl, ol + k * pitch);
    };
    float acc[4][4];
    double tot[4][4];
#pragma unroll
    for (int y = 0; y < 4; ++y)
#pragma unroll
        for (int x = 0; x < 4; ++x) acc[y][x] = 0.f, tot[y][x] = 0.0;

    const int panels = jpanels * cpanels, share = (cnt + 4 * NW - 1) / (4 * NW);
    fetch(js, clo);
    int jp = 0, cp = 0;
    for (int p = 0; p < panels; ++p) {
#pragma unroll
        for (int k = 0; k < 2 * JP; ++k) rw[k * 16] = pr[k];
#pragma unroll
        for (int k = 0; k < NLR; ++k) lw[k * 4 * LS] = pl[k];
        const int rows_left = share - jp * JP;  // of the longest group
        if (++cp == cpanels) cp = 0, ++jp;
        if (p + 1 < panels) fetch(js + jp * JP, clo + cp * CP);
        wave_lds_sync();
        if (rows_left > JP / 2)
            sum_panel<JP>(rq, lq, gx, gy, W <= CP, acc, tot);
        else
            sum_panel<JP / 2>(rq, lq, gx, gy, W <= CP, acc, tot);
        wave_lds_sync();  // the next panel overwrites this one
    }
    bool finite = true;
#pragma unroll
    for (int y = 0; y < 4; ++y)
#pragma unroll
        for (int x = 0; x < 4; ++x) finite = finite & __builtin_isfinite(tot[y][x]);
    // The groups' totals, added in order.  A value that is not finite makes a total of every lane that
    // met it so, overlap or not (0 * inf): such a wave sums again.
    if (__all(finite)) {
        double* const td = reinterpret_cast<double*>(smem + wave * WQ) + g * 256;
#pragma unroll
        for (int y = 0; y < 4; ++y)
#pragma unroll
            for (int x = 0; x < 4; ++x) td[(4 * gy + y) * 16 + 4 * gx + x] = tot[y][x];
    } else {
        direct_shifts_again(Lp, Rp, (lds_quad*)(float4*)(smem + wave * WQ), H, W, dx0, dy0, js, je, clo, cpanels, panels);
    }
    __syncthreads();
    const int SX = 2 * W - 1, SY = 2 * H - 1;
    float* __restrict__ Op = O + (size_t)pair * SX * SY;
    for (int o = threadIdx.x; o < 256; o += 64 * NW) {
        double v = 0.0;
        for (int w = 0; w < NW; ++w)
#pragma unroll
            for (int k = 0; k < 4; ++k) v += reinterpret_cast<const double*>(smem + w * WQ)[k * 256 + o];
        const int oy = 16 * ty + (o >> 4), ox = 16 * tx + (o & 15);
        if (oy < SY && ox < SX) Op[(size_t)oy * SX + ox] = (float)v;
    }
}

// Waves per block, each with four of the tile's 4 NW shares of right rows: more waves while the
// shares keep about 4 rows and the tiles are too few to balance the 256 CUs (the longer the sums,
// the more of them it takes), and where even four waves a tile leave places on the chip, until a share has
// the 4 rows of a half panel.  Measured us with 1 / 2 / 4 waves: 1 pair of 64^2 43 / 24 / 18, 8 of 128^2
// 194 / 150 / 114, 64 of 64^2 72 / 70 / 90, 40 of 32^2 14 / 13 / 18, 40 of 256^2 7630 / 7880 / 8110, 64
// of 50x80 87 / 92 / 107; 2 / 4 waves: 1 pair of 39x344 118 / 76, of 33x321 112 / 72.
int direct_shifts_waves(uint64_t tiles, uint32_t rows) {
    int nw = 1;
    while (nw < 4 && rows >= 20u * nw && tiles * nw < 72ull * rows) nw *= 2;
    if (tiles <= 768)
        while (nw < 4 && rows > 16u * nw) nw *= 2;
    return nw;
}

// Whether the register tiles take less time than the 16 x 16 shifts for batches of one right per left,
// where neither fills the chip and a wave's own chain of steps counts.  Both are estimated, in us: the
// shifts from a tile's panels (a half one for a last share of up to 4 rows) and the products issued, the
// tiles from a block's steps (rows of its chunk, in turns of 4) times columns, longer the more waves
// share the chip; more than it holds at once, 4096, take a second round, which the estimate does not
// know.  1358 shapes of 6 to 512 rows and columns, 1 to 12 pairs, were measured with both: the estimates
// are off by 7% and 9%.  The shifts by themselves are more than 3% slower than the tiles at 271 shapes, by
// up to 1.9 times; the choice at 28, by up to 1.15 times, and it is 1.29 times as fast on average.  us,
// shifts / tiles: 129x37 28.3 / 20.0, 26x335 72 / 53, 65x124 45 / 34, 64x128 30.1 / 25.5, 128^2 45.4 /
// 44.1, 54x61 16.6 / 27.9, 130^2 79 / 121, 256x64 45 / 55.  Up to 5 rows (7 to 18 us; the tiles up to a
// fifth less) the shifts stay.
bool register_tiles_faster(const family_args& a) {
    if (rights_per_left(a) > 1 || (a.family == XC_N_TO_M && a.n > 1) || a.rows <= 5) return false;
    const direct_plan d = plan_direct<float>(a, xc_options{});
    const double waves = (double)d.tiles_x * d.tiles_y * d.chunks * d.groups_r * d.groups_l * d.nwx * d.nwy;
    if (waves > 4096) return false;
    const double W = a.cols, tx = (2 * a.cols - 1 + 15) / 16, ty = (2 * a.rows - 1 + 15) / 16;
    const int nw = direct_shifts_waves((uint64_t)a.pairs * (uint64_t)(tx * ty), a.rows);
    const uint32_t share = (a.rows + 4 * nw - 1) / (4 * nw), rest = share % 8;
    const double panel = 5.07 * (share / 8 + (rest > 4)) + (rest > 0 && rest <= 4 ? 3.18 : 0.0);
    const double chain = 3.4 + std::ceil(W / 16) * panel;
    const double issue = a.pairs * tx * ty * 256 * (a.rows / 2.0 + 8) * (W / 2 + 8) / 19.8e6;
    const double shifts = std::pow(std::pow(chain, 1.84) + std::pow(issue, 1.84), 1 / 1.84);
    const uint32_t rows = d.rows_per_chunk ? d.rows_per_chunk : a.rows, steps = (rows + d.t.jb - 1) / d.t.jb;
    const double tiles = 3.6 + (d.chunks > 1 ? 2.0 : 0.0) +
                         steps * (W + 24) * (0.0575 + 0.0775 * std::pow(waves / 4096, 1.13));
    return tiles < 1.02 * shifts;
}

// The kernel for float batches of several results of up to 12 rows, where the 16 dy of the shifts and the 4
// waves of the matrix kernel are partly padding and a call may take little more than its launches: all
// three times are estimated, in us (the tiles and shifts as above, with the tiles' products per step and the
// shifts' cost per tile; the matrix kernel from its products and waves), over 1650 shapes of 1 to 32 rows,
// 1 to 400 columns and up to 300000 results with an error of 16, 8 and 11%.  The choice takes 1.025 times the
// fastest kernel's time there; without it 1.08, up to 3 times as long as the tiles (us, tiles): 1792 x 3 of
// 4x53 257 (73), 848 x 5 of 5x75 371 (174), 1549 pairs of 10x97 433 (216), 4092 of 2x22 51 (30), 1098 x 6 of 4x19
// 80 (39), 21 x 10 of 1x44 15.4 (7.4), 6 x 793 of 3x7 17.6 (13.7), 14 x 499 of 4x74 61 by the matrix kernel
// (153).  With several rights per left the shifts, the more exact ones, keep what they are 10% slower at.
enum class few_rows { none, tiles, shifts, matrix };
few_rows few_rows_choice(const family_args& a) {
    if (a.rows > 12 || a.pairs < 2) return few_rows::none;
    if ((a.cols <= 12 || one_row_by_pairs(a)) && pairs_kernel_applies(a, true)) return few_rows::none;
    const direct_plan d = plan_direct<float>(a, xc_options{});
    const double H = a.rows, W = a.cols, tx = (2 * a.cols - 1 + 15) / 16, ty = (2 * a.rows - 1 + 15) / 16;
    const double turns = std::ceil(W / 16);
    const double tile_waves = (double)d.tiles_x * d.tiles_y * d.chunks * d.groups_r * d.groups_l * d.nwx * d.nwy;
    const uint32_t rows = d.rows_per_chunk ? d.rows_per_chunk : a.rows, steps = (rows + d.t.jb - 1) / d.t.jb;
    const double tiles = 5.4 + (d.chunks > 1 ? 1.8 : 0.0) + steps * (W + 24) * (d.t.ty * d.t.rm * d.t.lm * d.t.jb / 16.0) *
                                                                (0.041 + 0.077 * std::pow(tile_waves / 4096, 1.1));
    const double shift_tiles = a.pairs * tx * ty;
    const int nw = direct_shifts_waves((uint64_t)shift_tiles, a.rows);
    const uint32_t share = (a.rows + 4 * nw - 1) / (4 * nw), rest = share % 8;
    const double panel = 3.2 * (share / 8 + (rest > 4)) + (rest > 0 && rest <= 4 ? 2.5 : 0.0);
    const double shifts = 4.1 + turns * panel + shift_tiles * (0.37e-3 + 1.3e-6 * (H + 60) * (W + 16.5));
    double matrix = HUGE_VAL;
    if (matrix_copies_fit(a)) {
        const double groups = (a.family == XC_ONE_TO_MANY ? 1.0 : a.n) * ((rights_per_left(a) + 15) / 16);
        const double bands = (2 * a.rows - 1 + 3) / 4, waves = groups * tx * bands * 4;
        matrix = 13.8 + waves * (256 * (H / 2 + 0.21) * (W / 2 + 8.2) * 2.36e-8 + 0.66e-3) +
                 0.098 * (H / 4) * std::ceil((W + 15) / 16);
    }
    if (tiles < (rights_per_left(a) > 1 ? 0.9 : 1.0) * shifts && tiles < matrix) return few_rows::tiles;
    return shifts < matrix ? few_rows::shifts : few_rows::matrix;
}

// False (nothing launched) where the grid does not fit one launch.
bool launch_direct_shifts(const family_args& a, const float* L, const float* R, float* O, hipStream_t s) {
    ds_args k{};
    k.family = a.family;
    k.H = (int)a.rows;
    k.W = (int)a.cols;
    k.n = a.family == XC_ONE_TO_ONE || a.family == XC_ONE_TO_MANY ? 1 : a.n;
    k.m = a.m;
    k.pairs = a.pairs;
    k.tiles_x = (2 * a.cols - 1 + 15) / 16;
    k.tiles_y = (2 * a.rows - 1 + 15) / 16;
    const uint64_t tiles = (uint64_t)a.pairs * k.tiles_x * k.tiles_y;
    const int nw = direct_shifts_waves(tiles, a.rows);
    if (!fits_one_launch(tiles, 64 * nw)) return false;
    const dim3 grid((uint32_t)tiles), block(64 * nw);
    record_launch("direct_kernel<f32> 16x16 shifts, rows over lanes", grid, block, 0, a.rows, a.cols, a.pairs, 1);
    timed td("direct_kernel", s);
    if (nw == 1)
        hipLaunchKernelGGL(direct_shifts_kernel<1>, grid, block, 0, s, L, R, O, k);
    else if (nw == 2)
        hipLaunchKernelGGL(direct_shifts_kernel<2>, grid, block, 0, s, L, R, O, k);
    else
        hipLaunchKernelGGL(direct_shifts_kernel<4>, grid, block, 0, s, L, R, O, k);
    XC_HIP(hipGetLastError());
    return true;
}

template <typename T>
void launch_direct(const family_args& a, const T* L, const T* R, T* O, const xc_options& opt, hipStream_t s) {
    if (a.cols > (uint32_t)kMaxCols) fail(XC_ERR_UNSUPPORTED, "direct kernel: cols above 32768");
    // tile 0, with no register tile or work distribution requested: float data of few rows by
    // few_rows_choice, other by the matrix kernel where it applies, then the lanes-over-pairs kernel where it
    // applies, else (float data) the 16 x 16 shifts kernel where the tiles are not faster; 1: the
    // register-tile kernel; 2: the lanes-over-pairs kernel (float and double data alike)
    if (opt.tile > 2)
        fail(XC_ERR_INVALID_ARGUMENT, "direct-method tile must be 0 (default), 1 (register tiles) or 2 (lanes over pairs)");
    const bool keys = opt.shifts_per_thread || opt.right_mats_per_thread || opt.left_mats_per_thread ||
                      opt.rows_per_step || opt.waves_per_block || opt.split || opt.rows_per_block;
    if (opt.tile == 2 && rights_per_left(a) == 0)
        fail(XC_ERR_UNSUPPORTED, "direct-method tile 2 (lanes over pairs) does not serve one_to_one");
    const bool free_choice = opt.tile == 0 && !keys;
    const few_rows few = std::is_same<T, float>::value && free_choice ? few_rows_choice(a) : few_rows::none;
    if (std::is_same<T, float>::value && free_choice &&
        (few == few_rows::none ? matrix_kernel_applies(a) : few == few_rows::matrix) &&
        launch_direct_pairs<T>(a, L, R, O, s, true, false))
        return;
    if ((opt.tile == 2 || (free_choice && few == few_rows::none && pairs_kernel_applies(a, sizeof(T) == 4))) &&
        launch_direct_pairs<T>(a, L, R, O, s, false, opt.tile == 2))
        return;
    if (opt.tile == 2) fail(XC_ERR_INVALID_ARGUMENT, "problem too large for one launch");
    if constexpr (std::is_same<T, float>::value) {
        // Few rights per left: 16 x 16 shifts per wave or block, unless the matrices are so flat
        // that a tile's 16 dy are mostly padding (16 rows < cols).  Measured, 16 pairs, us, against
        // the register tiles: 20x100 29 / 41, 20x300 110 / 109, 20x1000 833 / 676, 40x1000 1970 /
        // 1850, 64x1000 2950 / 4960, 1000x20 640 / 1150; its buffer offsets need matrices below
        // 2^31 bytes.
        const bool apt = few == few_rows::shifts ||
                         (few != few_rows::tiles && 16ull * a.rows >= a.cols && !register_tiles_faster(a));
        if (free_choice && apt && (uint64_t)a.rows * a.cols < (1u << 29) && launch_direct_shifts(a, L, R, O, s))
            return;
    }
    direct_plan d = plan_direct<T>(a, opt);
    if (d.lds > 160 * 1024) {
        if (opt.rows_per_step || opt.right_mats_per_thread)
            fail(XC_ERR_UNSUPPORTED, "direct kernel: the staged rows of this tile exceed the LDS");
        xc_options o = opt;
        o.rows_per_step = 1;
        o.right_mats_per_thread = 1;
        d = plan_direct<T>(a, o);
        if (d.lds > 160 * 1024) fail(XC_ERR_UNSUPPORTED, "matrix too wide for the direct kernel's LDS row buffer");
    }
    const uint64_t nblocks = (uint64_t)d.tiles_x * d.tiles_y * d.chunks * d.groups_r * d.groups_l;
    if (nblocks == 0 || !fits_one_launch(nblocks, 64 * d.nwx * d.nwy))
        fail(XC_ERR_INVALID_ARGUMENT, "problem too large for one launch");
    dk_args k = args_of(a, d);
    if (k.atomic) {
        const uint64_t count = (uint64_t)a.pairs * (2 * a.cols - 1) * (2 * a.rows - 1);
        uint32_t zb = (uint32_t)std::min<uint64_t>((count + 255) / 256, 8192);
        timed tz("zero_kernel", s);
        hipLaunchKernelGGL(zero_kernel<T>, dim3(zb), dim3(256), 0, s, O, count);
    }
    const void* fn = kernel_of<T>(d.t);
    if (!fn) fail(XC_ERR_UNSUPPORTED, "direct kernel: tile not in the catalog");
    if (d.lds > 65536) allow_dynamic_lds(fn, d.lds);
    dim3 grid((uint32_t)nblocks), block(64 * d.nwx * d.nwy);
    char name[96];
    std::snprintf(name, sizeof(name), "direct_kernel<%s> ty%d rm%d lm%d jb%d", sizeof(T) == 4 ? "f32" : "f64", d.t.ty,
                  d.t.rm, d.t.lm, d.t.jb);
    record_launch(name, grid, block, d.lds, a.rows, a.cols, a.pairs, d.chunks);
    timed td("direct_kernel", s);
    void* args[] = {(void*)&L, (void*)&R, (void*)&O, (void*)&k};
    XC_HIP(hipLaunchKernel(fn, grid, block, args, d.lds, s));
}

}  // namespace

void launch_direct_f32(const family_args& a, const float* L, const float* R, float* O, const xc_options& opt,
                       hipStream_t s) {
    launch_direct<float>(a, L, R, O, opt, s);
}

void launch_direct_f64(const family_args& a, const double* L, const double* R, double* O, const xc_options& opt,
                       hipStream_t s) {
    launch_direct<double>(a, L, R, O, opt, s);
}

void launch_zero_f32(float* p, uint64_t count, hipStream_t s) {
    uint32_t zb = (uint32_t)std::min<uint64_t>((count + 255) / 256, 8192);
    if (zb) hipLaunchKernelGGL(zero_kernel<float>, dim3(zb), dim3(256), 0, s, p, count);
}

void launch_zero_f64(double* p, uint64_t count, hipStream_t s) {
    uint32_t zb = (uint32_t)std::min<uint64_t>((count + 255) / 256, 8192);
    if (zb) hipLaunchKernelGGL(zero_kernel<double>, dim3(zb), dim3(256), 0, s, p, count);
}

}  // namespace xc
