// FFT method on this library's own FP64 FFT kernels (no rocFFT): three fused passes over HBM.
//
// The reference's FFT algorithm (src/one_to_many.hpp:679-745, src/n_to_m.hpp:700-736):
// zero-pad both matrices to 2H x 2W, R2C, multiply the left spectrum by the conjugate of
// each right spectrum (hadamard_original, src/hadamard.cu:33-58), C2R, then normalise on the host
// (src/fft_helpers.hpp:193-261: divide by the padded area, swap quadrants, crop).  Here the
// padded sizes are Pr x Pc, the powers of two >= 2H-1 and >= 2W-1 (any size >= 2N-1 makes
// the circular correlation equal the linear one), and the work is three kernels:
//
//   rows_fwd : two real input rows per complex FFT of length Pc (zero padding implicit),
//              split into the two half spectra, written transposed as S[mat][k][r]
//              (k = 0..Pc/2, only the H nonzero rows r);
//   cols     : per (pair, column k): X = FFT of length Pr of S[right][k][0..H-1] (zero
//              padded), then a second FFT of conj(Lhat) * X: the conjugate of
//              Pr * IFFT(Lhat * conj(X)) (Lhat = the left's 2D spectrum, made by the same
//              kernel in "left" mode, or inside the block where few pairs share a left:
//              cols_group), of which only the 2H-1 circular rows of the result are kept:
//              Z[pair][k][z_row(rho)];
//   rows_inv : per pair, two output rows per complex FFT of length Pc: the Hermitian half
//              rows of Z are extended, inverse transformed, scaled by 1/(Pr*Pc) and written
//              straight into the cropped (2H-1) x (2W-1) result (quadrant swap by index).
//
// All arithmetic is FP64, in radix-8/4/2 Stockham passes.  Transforms of up to 2048 points
// live in registers (a wave owns each up to 512 points, 2 or 4 waves of a block at 1024 and
// 2048; LDS only for the exchanges between passes); 4096-point transforms are done by a block
// in an LDS slab (padded LDS index against bank conflicts).  Twiddles come from a 4096-entry
// table, read once per kernel into registers; every HBM load of a kernel is issued before its
// first use.  Uneven batches run jobs whose matrices share the padded lengths but keep their
// own sizes (a per-matrix size table).
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <cmath>
#include <mutex>
#include <tuple>
#include <type_traits>
#include <vector>

#include "xc_fftk_core.hpp"
#include "xc_methods.hpp"

namespace xc {
namespace {

constexpr int kFT = 256;  // threads per block: slab kernels, block-owned column FFTs

// Slab (values per block) of a transform length: 2^11 values, or one transform of 4096.
// Lengths of up to 2048 points are transformed in registers (fft_regs), 4096 in a slab.
template <int LOGP>
struct slab_of {
    static constexpr int LOGS = LOGP <= 11 ? 11 : LOGP;
};

// First radix of a length-2^LOGP transform (8, 2 or 4 as LOGP mod 3 is 0, 1, 2; it takes no
// twiddles) and the number of twiddled radix-8 passes after it.
template <int LOGP>
struct radix_plan {
    static constexpr int REM = LOGP % 3;
    static constexpr int LOGR0 = REM == 0 ? 3 : REM;
    static constexpr int NTW = (LOGP - LOGR0) / 3;
};

// Pass roots of the slab transforms of length 2^LOGP (1024..4096): w[j][q] is the root of the
// j-th twiddled radix-8 pass (p = 2^(LOGR0 + 3j)) for this thread's q-th butterfly, b =
// threadIdx + kFT q.  Kernels load them once, before their first transform: a table read
// inside a pass would wait on memory after every barrier.
template <int LOGP>
struct slab_roots {
    static constexpr int NB8 = (1 << slab_of<LOGP>::LOGS) / 8 / kFT;  // radix-8 butterflies per thread
    double2 w[radix_plan<LOGP>::NTW][NB8];
};
template <int LOGP>
__device__ __forceinline__ slab_roots<LOGP> load_slab_roots(const double2* __restrict__ tw) {
    slab_roots<LOGP> sr;
#pragma unroll
    for (int j = 0; j < radix_plan<LOGP>::NTW; ++j) {
        const int logpp = radix_plan<LOGP>::LOGR0 + 3 * j;
#pragma unroll
        for (int q = 0; q < slab_roots<LOGP>::NB8; ++q) {
            const int i = ((int)threadIdx.x + kFT * q) & ((1 << (LOGP - 3)) - 1);
            sr.w[j][q] = tw[(i & ((1 << logpp) - 1)) << (kLogMaxP - logpp - 3)];
        }
    }
    return sr;
}

// One Stockham radix-R pass over T transforms of length P = 2^LOGP in buf (slots `at`),
// T * P <= 2^LOGS; 2^LOGPP is the product of the radices already applied.  Butterfly i of a
// transform reads elements i + r*P/R and writes (i - k)*R + k + r*p, k = i mod p, after
// multiplying input r by exp(-2 pi i r k / (p R)).  Butterflies go to threads block-strided.
template <int R, int LOGR, int LOGP, int LOGPP>
__device__ __forceinline__ void fft_pass(double2* buf, int T, const slab_roots<LOGP>& sr) {
    constexpr int MAXB = (1 << slab_of<LOGP>::LOGS) / R / kFT;
    static_assert(MAXB >= 1, "slab too small for the radix");
    constexpr int LOGPR = LOGP - LOGR;
    const int nb = T << LOGPR;
    double2 u[MAXB][R];
#pragma unroll
    for (int q = 0; q < MAXB; ++q) {
        const int b = (int)threadIdx.x + kFT * q;
        if (b < nb) {
            const int t = b >> LOGPR, i = b & ((1 << LOGPR) - 1);
#pragma unroll
            for (int r = 0; r < R; ++r) u[q][r] = buf[at<LOGP>(t, i + (r << LOGPR))];
        }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < MAXB; ++q) {
        const int b = (int)threadIdx.x + kFT * q;
        if (b < nb) {
            const int t = b >> LOGPR, i = b & ((1 << LOGPR) - 1);
            const int k = i & ((1 << LOGPP) - 1);
            if constexpr (LOGPP > 0) {
                static_assert(R == 8, "only the first pass has another radix");
                const double2 w1 = sr.w[(LOGPP - radix_plan<LOGP>::LOGR0) / 3][q];
                double2 w = w1;
#pragma unroll
                for (int r = 1; r < R; ++r) {
                    u[q][r] = cmul(u[q][r], w);
                    if (r + 1 < R) w = cmul(w, w1);
                }
            }
            dft<R>(u[q]);
            const int j = ((i - k) << LOGR) + k;
#pragma unroll
            for (int r = 0; r < R; ++r) buf[at<LOGP>(t, j + (r << LOGPP))] = u[q][r];
        }
    }
    __syncthreads();
}

template <int LOGP, int LOGPP>
__device__ __forceinline__ void radix8_passes(double2* buf, int T, const slab_roots<LOGP>& sr) {
    if constexpr (LOGPP < LOGP) {
        fft_pass<8, 3, LOGP, LOGPP>(buf, T, sr);
        radix8_passes<LOGP, LOGPP + 3>(buf, T, sr);
    }
}

// Forward FFT of T transforms of length 2^LOGP (1024..4096) in buf; natural order.  The caller
// has synchronised the block before; the block is synchronised on return.
template <int LOGP>
__device__ __forceinline__ void fft_slab(double2* buf, int T, const slab_roots<LOGP>& sr) {
    static_assert(LOGP >= 10, "shorter transforms run in registers");
    constexpr int LOGR0 = radix_plan<LOGP>::LOGR0;
    fft_pass<1 << LOGR0, LOGR0, LOGP, 0>(buf, T, sr);
    radix8_passes<LOGP, LOGR0>(buf, T, sr);
}

// Threads per block of the row kernels (INV: rows_inv): 256, or more for register transforms
// of 1024 and 2048 points so that a block holds four transforms (8 rows: a column's piece of
// S or Z is a whole 128-byte line) -- except rows_inv at 2048 points, where two transforms per
// block (two blocks per CU instead of one) measured faster.  LOGS is the block's slab.
constexpr int rows_threads(int logP, bool inv) {
    return logP == 10 ? 512 : (logP == 11 ? (inv ? 512 : 1024) : 256);
}
template <int LOGP, bool INV>
struct rows_block {
    static constexpr int NT = rows_threads(LOGP, INV);
    static constexpr int LOGS = regs_of<LOGP>::ON ? (NT == 256 ? 11 : (NT == 512 ? 12 : 13)) : slab_of<LOGP>::LOGS;
};

// The block's T transformed row pairs (spectra in natural order in LDS) -> the half spectra
// of rows r0 .. r0 + 2T - 1 (those below Hm), written column-major into Sm (column stride Hs):
// with z = FFT(a + i b), A[k] = (z[k] + conj(z[P-k]))/2 and B[k] = (z[k] - conj(z[P-k]))/(2i).
template <int LOGPC, int NT>
__device__ __forceinline__ void split_rows(const double2* buf, double2* __restrict__ Sm, uint32_t r0, uint32_t Hm,
                                           uint32_t Hs, int logT) {
    constexpr int Pc = 1 << LOGPC;
    constexpr uint32_t Kc = Pc / 2 + 1;
    const int rows2 = 2 << logT;
    for (int idx = threadIdx.x; idx < (int)Kc * rows2; idx += NT) {
        const int k = idx >> (logT + 1), rr = idx & (rows2 - 1);
        const uint32_t r = r0 + rr;
        if (r >= Hm) continue;
        const int t = rr >> 1;
        const double2 zk = buf[at<LOGPC>(t, k)];
        const double2 zn = cconj(buf[at<LOGPC>(t, (Pc - k) & (Pc - 1))]);
        double2 v;
        if ((rr & 1) == 0) {
            v = make_double2(0.5 * (zk.x + zn.x), 0.5 * (zk.y + zn.y));
        } else {
            const double2 d = mul_mi(csub(zk, zn));
            v = make_double2(0.5 * d.x, 0.5 * d.y);
        }
        Sm[(size_t)k * Hs + r] = v;
    }
}

// rows_fwd for register transforms (up to 2048 points; 65 matrices of 256^2 in 17.9 us, 4.8 TB/s;
// 20.2 with index arithmetic per split value): a persistent grid of the blocks that
// fit at once, each taking row groups (items: matrix, group of 2T rows) in turn and loading
// the next item's rows into registers while it transforms and stores the current one, so
// that HBM latency is paid once per block rather than once per item.  Items are dealt so
// that each XCD (blocks b with b mod 8 = x) walks one contiguous eighth of the item range:
// the partial lines of S that neighbouring groups write meet in its L2.  Matrices, offsets
// and sizes as in rows_fwd_slab_kernel below.
template <typename Tin, int LOGPC, int NT = rows_block<LOGPC, false>::NT>
__global__ __launch_bounds__(NT) void rows_fwd_regs_kernel(const Tin* __restrict__ XL, const Tin* __restrict__ XR,
                                                           const uint64_t* __restrict__ moff,
                                                           const uint2* __restrict__ mdims, uint32_t nl, uint32_t H,
                                                           uint32_t Hs, uint32_t W, uint32_t groups, uint32_t items,
                                                           double2* __restrict__ SL, double2* __restrict__ SR,
                                                           const double2* __restrict__ tw) {
    static_assert(regs_of<LOGPC>::ON, "register transforms only");
    constexpr int Pc = 1 << LOGPC, Q = Pc / 8, T = 8 * NT / Pc, LOGT = rows_block<LOGPC, false>::LOGS - LOGPC;
    constexpr uint32_t Kc = Pc / 2 + 1;
    static_assert(T == 1 << LOGT, "transforms per block");
    extern __shared__ double2 buf[];
    const regs_pos<LOGPC> ps((int)threadIdx.x);
    const int t0 = ps.t0, t = ps.t, i = ps.i;
    const auto rr = load_roots<LOGPC, exact_roots<Tin>>(i, tw);
    // this block's items: x * per + k + j * bpx, j = 0, 1, ... below min((x + 1) * per, items)
    const uint32_t nx = gridDim.x >= 8 ? 8 : 1;
    const uint32_t x = blockIdx.x % nx, kb = blockIdx.x / nx, bpx = gridDim.x / nx;
    const uint32_t per = (items + nx - 1) / nx;
    const uint32_t end = min((x + 1) * per, items);
    // the matrix of item `it`, its size and the first row of its group
    struct where {
        uint32_t matg, r0, Hm, Wm;
    };
    auto locate = [&](uint32_t it) {
        where w;
        w.matg = it / groups;
        w.r0 = (it - w.matg * groups) << (LOGT + 1);
        w.Hm = H;
        w.Wm = W;
        if (mdims) {
            const uint2 d = mdims[w.matg];
            w.Hm = d.x;
            w.Wm = d.y;
        }
        return w;
    };
    // Rows r0 + 2t and the next; rows and columns outside the matrix read zero (W <= Pc / 2: the
    // upper half of a row is padding).
    auto fetch = [&](const where& w, Tin (&va)[4], Tin (&vb)[4]) {
        const uint32_t mat = w.matg < nl ? w.matg : w.matg - nl;
        const Tin* Xm = (w.matg < nl ? XL : XR) + (moff ? moff[w.matg] : (size_t)mat * H * W);
        const __amdgpu_buffer_rsrc_t rx = buf_of(Xm, w.Hm * w.Wm * (uint32_t)sizeof(Tin));
        const uint32_t row = ((w.r0 + 2 * (uint32_t)t) * w.Wm + (uint32_t)i) * (uint32_t)sizeof(Tin);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint32_t off = (uint32_t)(i + Q * r) < w.Wm ? row + (uint32_t)(Q * r * sizeof(Tin)) : kOut;
            va[r] = buf_load_real<Tin>(rx, off, 0);
            vb[r] = buf_load_real<Tin>(rx, off + w.Wm * (uint32_t)sizeof(Tin), 0);
        }
    };
    uint32_t it = x * per + kb;
    if (it >= end) return;
    where cur = locate(it);
    Tin va[4], vb[4];
    fetch(cur, va, vb);
    while (true) {
        const uint32_t nxt = it + bpx;
        const bool more = nxt < end;
        double2 u[8];
#pragma unroll
        for (int r = 0; r < 4; ++r) u[r] = make_double2((double)va[r], (double)vb[r]);
        where nw{};
        if (more) {  // the next item's rows are in flight during this item's transform and stores
            nw = locate(nxt);
            fetch(nw, va, vb);
        }
        if (cur.r0 < cur.Hm) {  // block-uniform: a row group beyond a smaller matrix is skipped
            fft_regs<LOGPC, true>(u, buf + at<LOGPC>(t0, 0), rr, t - t0, i);
#pragma unroll
            for (int r = 0; r < 8; ++r)
                buf[Q % 8 == 0 ? at<LOGPC>(t, i) + r * (Q + Q / 8) : at<LOGPC>(t, i + Q * r)] = u[r];
            __syncthreads();
            // Split into the rows' half spectra, column-major into S: with z = FFT(a + i b), A[k] =
            // (z[k] + conj(z[P-k]))/2 and B[k] = (z[k] - conj(z[P-k]))/(2i).  A thread takes row rw
            // of the group (an A or a B) at columns k0 + (Q/2) q; the component of z that the sum
            // takes is the real one for A and the imaginary one for B, the other goes into the
            // difference, so both read as 8-byte values at a lane's own offset.
            const int rw = (int)threadIdx.x & (2 * T - 1), tq = rw >> 1, odd = rw & 1;
            const int k0 = (int)threadIdx.x >> (LOGT + 1);
            constexpr int KS = Q / 2;
            const double hs = odd ? -0.5 : 0.5;
            const double* zs = reinterpret_cast<const double*>(buf) + odd;      // the sum's component
            const double* zd = reinterpret_cast<const double*>(buf) + 1 - odd;  // the difference's
            const bool left = cur.matg < nl;
            const size_t mat = left ? cur.matg : cur.matg - nl;
            const __amdgpu_buffer_rsrc_t rs = buf_of((left ? SL : SR) + mat * Kc * Hs, Kc * Hs * 16u);
            const uint32_t row = cur.r0 + (uint32_t)rw, step = KS * Hs * 16u;
            const uint32_t off = row < cur.Hm ? ((uint32_t)k0 * Hs + row) * 16u : kOut;
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const int a = KS % 8 == 0 ? at<LOGPC>(tq, k0) + q * (KS + KS / 8) : at<LOGPC>(tq, k0 + KS * q);
                const int b = q == 0        ? at<LOGPC>(tq, (Pc - k0) & (Pc - 1))
                              : KS % 8 == 0 ? at<LOGPC>(tq, Pc - k0) - q * (KS + KS / 8)
                                            : at<LOGPC>(tq, Pc - k0 - KS * q);
                buf_store(make_double2(0.5 * (zs[2 * a] + zs[2 * b]), hs * (zd[2 * a] - zd[2 * b])), rs, off, q * step);
            }
            if (k0 == 0)  // column Pc / 2
                buf_store(make_double2(zs[2 * at<LOGPC>(tq, Pc / 2)], 0.0), rs, off, 8 * step);
            __syncthreads();  // the next item's transform reuses the slab
        }
        if (!more) break;
        it = nxt;
        cur = nw;
    }
}

// rows_fwd for 4096-point transforms (the LDS slab): block (matrix, group of 2T rows);
// matrices 0..nl-1 are the left ones (into SL), the rest the right ones (into SR).  Matrix i
// starts at element moff[i] of its input when the offset table is given (uneven batches),
// else at i * H * W.  With mdims (uneven batches), matrix i is mdims[i].x x mdims[i].y, at
// most H x W (the padded lengths are those of H x W); S keeps a column stride of Hs.
template <typename Tin, int LOGPC, int NT = rows_block<LOGPC, false>::NT>
__global__ __launch_bounds__(NT) void rows_fwd_slab_kernel(const Tin* __restrict__ XL, const Tin* __restrict__ XR,
                                                           const uint64_t* __restrict__ moff,
                                                           const uint2* __restrict__ mdims, uint32_t nl, uint32_t H,
                                                           uint32_t Hs, uint32_t W, int logT, uint32_t groups,
                                                           double2* __restrict__ SL, double2* __restrict__ SR,
                                                           const double2* __restrict__ tw) {
    static_assert(!regs_of<LOGPC>::ON && NT == kFT, "slab transforms");
    constexpr int logPc = LOGPC;
    extern __shared__ double2 buf[];
    // XCD-aware order: the row groups of one matrix run on one XCD, so the partial lines of S
    // that neighbouring groups write (2T rows of a column) merge in that XCD's L2.
    const uint32_t bid = xcd_remap(blockIdx.x, gridDim.x);
    const uint32_t matg = bid / groups, g = bid - matg * groups;
    const bool left = matg < nl;
    const uint32_t mat = left ? matg : matg - nl;
    const int Pc = 1 << logPc, T = 1 << logT;
    const uint32_t r0 = g << (logT + 1);
    uint32_t Hm = H, Wm = W;
    if (mdims) {
        const uint2 d = mdims[matg];
        Hm = d.x;
        Wm = d.y;
    }
    if (r0 >= Hm) return;  // the whole block: a row group beyond a smaller matrix of the job
    const Tin* Xm = (left ? XL : XR) + (moff ? moff[matg] : (size_t)mat * H * W);
    double2* S = left ? SL : SR;
    // T = 2^LOGS / Pc transforms at most; element idx of the slab is column c of transform t.
    // Branch-free clamped loads first, then the LDS writes.
    constexpr int NI = (1 << slab_of<LOGPC>::LOGS) / kFT;
    const slab_roots<LOGPC> sr = load_slab_roots<LOGPC>(tw);
    const int n_el = T << logPc;
    Tin va[NI], vb[NI];
#pragma unroll
    for (int q = 0; q < NI; ++q) {
        const int idx = threadIdx.x + kFT * q;
        const uint32_t t = idx >> logPc, c = idx & (Pc - 1);
        const uint32_t a = r0 + 2 * t, b = a + 1;
        const size_t cc = c < Wm ? c : Wm - 1;
        va[q] = Xm[(size_t)(a < Hm ? a : Hm - 1) * Wm + cc];
        vb[q] = Xm[(size_t)(b < Hm ? b : Hm - 1) * Wm + cc];
    }
#pragma unroll
    for (int q = 0; q < NI; ++q) {
        const int idx = threadIdx.x + kFT * q;
        if (idx >= n_el) continue;
        const uint32_t t = idx >> logPc, c = idx & (Pc - 1);
        const uint32_t a = r0 + 2 * t, b = a + 1;
        const bool in = c < Wm;
        buf[at<LOGPC>(t, c)] = make_double2(a < Hm && in ? (double)va[q] : 0.0, b < Hm && in ? (double)vb[q] : 0.0);
    }
    __syncthreads();
    fft_slab<LOGPC>(buf, T, sr);
    split_rows<LOGPC, NT>(buf, S + (size_t)mat * (Pc / 2 + 1) * Hs, r0, Hm, Hs, logT);
}

// S and Z are column-major with column strides Hs and Ys = 2 Hs, Hs = the job's row count H
// rounded up to 8: every column starts on a 128-byte line, and so does each group of 8 rows that
// the row kernels move (off the lines, at 299 rows, fftk_rows_inv took 131 us where 304 rows took
// 115: 64 pairs of 512 columns).
//
// Row of Z that keeps circular row rho of a pair with H rows: the result's shifts dy = rho
// (rho < H) stay in place, dy = rho - Pr (rho > Pr - H) move down by Pr - Ys to the rows below
// Ys, so that both halves keep the transform's alignment (and for Pr = Ys nothing moves); -1 for
// the rows in between.
__device__ __forceinline__ int z_row(uint32_t rho, uint32_t H, uint32_t Ys, uint32_t Pr) {
    if (rho < H) return (int)rho;
    if (rho > Pr - H && rho < Pr) return (int)(rho - (Pr - Ys));
    return -1;
}

// Output row (dy + H - 1) of row z of Z (z_row's inverse), -1 for the rows in between.
__device__ __forceinline__ int out_row_of_z(uint32_t z, uint32_t H, uint32_t Ys) {
    if (z < H) return (int)(z + H - 1);
    if (z > Ys - H && z < Ys) return (int)(z + H - 1 - Ys);
    return -1;
}
// Whether none of the `rows` rows from z0 on is a row of a result.
__device__ __forceinline__ bool z_gap(uint32_t z0, uint32_t rows, uint32_t H, uint32_t Ys) {
    return z0 >= Ys || (z0 >= H && z0 + rows <= Ys - H + 1);
}

// Threads per block of the column kernel: one wave for wave-owned register transforms (up to
// 512 points; C = 512 / Pr columns per block, so that a pair's last column group wastes at
// most a wave), 256 for the block-owned and slab transforms.
// Rows of each half of a column of Z that are stored: whole 128-byte lines, with outputs of the transform that
// nothing reads past the result's.  Partly written lines are read back first where Z does not stay in the
// Infinity Cache (8 x 67 of 100x200: cols 143 -> 131 us, rows_inv 157 -> 142; of 100x420 322 -> 283, 280 -> 267; whole
// 64-byte sectors only 316 and 278).  From 64 rows; of few rows the lines' rest is most of them (72 x 13 of 2x150
// 37.5 -> 42.8).
__device__ __forceinline__ uint32_t z_lines(uint32_t rows, uint32_t Ys) {
    return rows < 64 ? rows : min((rows + 7) & ~7u, Ys / 2);
}
// The first row rho of the second half that is stored.
__device__ __forceinline__ uint32_t z_second(uint32_t rows, uint32_t whole, uint32_t P) {
    return rows < 64 ? P - rows + 1 : P - whole;
}

constexpr int cols_threads(int logP) { return logP <= 9 ? 64 : kFT; }

// cols: block (item, group of C columns k).  mode 0: item = left matrix l, writes its full
// column spectra Lhat[l][k][rho] (the FFT along rho of SL[l][k][0..H), zero padded).  With
// mdims (uneven batches) a matrix has mdims[i].x rows of its own (i = l, or nl + r for the
// right of a pair); S keeps a column stride of Hs.
// mode 1: item = pair q0 + item (left l, right r from the family's order, or from the pair
// table of an uneven batch): X = the same FFT of SR[r][k], then a second FFT of
// conj(Lhat) * X: the conjugate of Pr * IFFT_rho(Lhat * conj(X)), whose circular row rho goes to
// Z[item][k][z_row(rho)] (column stride Ys; the rows between the result's two halves are
// dropped, but for those of a line that has result rows: z_lines).
// Blocks are ordered column-group major through the XCD remap, so the pairs that read the
// same Lhat columns run on one XCD and find them in its L2.
// cols_group: block (group of C columns k, G consecutive pairs from q0 + item G): the columns of
// the pairs' left matrix are transformed here and kept in registers while the left stays the
// same, so the left spectra are neither written to Lhat nor read back, and one launch is saved;
// the rest as cols mode 1 below.  Against that path a left's columns are transformed once per
// block instead of once per call, and the registers of the left stay occupied during the second
// transform of a pair (118 instead of 96 at 512 points: 4 waves per SIMD for 5).  So it is taken for
// at most 4 pairs per left (64 pairs of n_to_mn at 256^2: one per left 189 -> 131 us, two 151 ->
// 108, four 110 -> 101; eight 100 -> 100, sixteen 94 -> 95; the uneven batch of 128 x 4 pairs 796 ->
// 720) and where the pairs' columns are at most 6144 waves, so that the launch counts (one pair of
// 128^2 15.9 -> 13.6 us, of 512^2 32.2 -> 28.6, 1 x 16 of 256^2 40.0 -> 37.4; 1 x 24 46.6 -> 46.0, 1 x
// 32 55.2 -> 56.1).  G = 2 above 4608 waves (the batch 772 -> 740 in one run), G = 1 below (1 x 4 of
// 256^2 20.7 against 22.1, 64 x 64 of 128^2 37.7 against 39.7).
// X: regs_roots (the batch's data are double).
template <int LOGPR, bool X>
__global__ __launch_bounds__(cols_threads(LOGPR)) void cols_group_kernel(
    const double2* __restrict__ SL, const double2* __restrict__ SR, double2* __restrict__ Z,
    const uint2* __restrict__ ptab, const uint2* __restrict__ mdims, uint32_t nl, int family, uint32_t n, uint32_t m,
    uint32_t q0, uint32_t pairs, uint32_t G, uint32_t items, uint32_t H, uint32_t Hs, uint32_t Kc, uint32_t Ys,
    const double2* __restrict__ tw) {
    extern __shared__ double2 buf[];
    constexpr int Q = 1 << (LOGPR - 3), P = 1 << LOGPR;
    constexpr uint32_t C = 8 * cols_threads(LOGPR) / P;
    const uint32_t bid = xcd_remap(blockIdx.x, gridDim.x);
    const uint32_t cg = bid / items, first = (bid - cg * items) * G, last = min(first + G, pairs);
    const regs_pos<LOGPR> ps((int)threadIdx.x);
    const uint32_t k = cg * C + ps.t;
    const bool ok = k < Kc;
    double2* wb = buf + at<LOGPR>(ps.t0, 0);
    const auto rr = load_roots<LOGPR, X>(ps.i, tw);
    auto column = [&](const double2* S, uint32_t mat, uint32_t rows, int i, double2 (&u)[8]) {
        const __amdgpu_buffer_rsrc_t rs = buf_of(S + (size_t)mat * Kc * Hs, Kc * Hs * 16u);
        const uint32_t so = (k * Hs + (uint32_t)i) * 16u;
#pragma unroll
        for (int r = 0; r < 4; ++r)  // rows <= Pr / 2: the upper half of a column is padding
            u[r] = buf_load(rs, (uint32_t)(i + Q * r) < rows ? so + 16u * Q * r : kOut, 0);
    };
    double2 lh[8];
    uint32_t have = ~0u;
    for (uint32_t p = first; p < last; ++p) {
        uint32_t l, r;
        if (ptab) {
            l = ptab[q0 + p].x;
            r = ptab[q0 + p].y;
        } else {
            pair_of(family, n, m, q0 + p, l, r);
        }
        const uint32_t Hq = mdims ? mdims[nl + r].x : H, rows = ok ? Hq : 0;
        // opaque copies of the position: no transform keeps another one's LDS addresses live
        int tl = ps.t - ps.t0, i = ps.i;
        double2 u[8];
        if (l != have) {  // block-uniform
            asm volatile("" : "+v"(tl), "+v"(i));
            column(SL, l, rows, i, lh);
            column(SR, r, rows, i, u);
            fft_regs<LOGPR, true>(lh, wb, rr, tl, i);
            have = l;
        } else {
            asm volatile("" : "+v"(tl), "+v"(i));
            column(SR, r, rows, i, u);
        }
        asm volatile("" : "+v"(tl), "+v"(i));
        fft_regs<LOGPR, true>(u, wb, rr, tl, i);
#pragma unroll
        for (int s = 0; s < 8; ++s) u[s] = cmul(cconj(lh[s]), u[s]);
        asm volatile("" : "+v"(tl), "+v"(i));
        fft_regs<LOGPR>(u, wb, rr, tl, i);
        // z_row: rows below Hq (s < 4: Hq <= Pr / 2) in place, rows above Pr - Hq (s >= 4) down by
        // Pr - Ys
        const uint32_t whole = z_lines(rows, Ys), second = z_second(rows, whole, P);
        const __amdgpu_buffer_rsrc_t rz = buf_of(Z + (size_t)p * Kc * Ys, Kc * Ys * 16u);
        const uint32_t zlo = (k * Ys + (uint32_t)i) * 16u, zhi = zlo - ((uint32_t)P - Ys) * 16u;
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            const uint32_t rho = (uint32_t)(i + Q * s);
            const bool in = s < 4 ? rho < whole : rho >= second;
            buf_store(u[s], rz, in ? (s < 4 ? zlo : zhi) + 16u * Q * s : kOut, 0);
        }
    }
}

template <int LOGPR, int MODE, bool X>
__global__ __launch_bounds__(cols_threads(LOGPR)) void cols_kernel(const double2* __restrict__ S, double2* __restrict__ Lhat,
                                                   double2* __restrict__ Z, const uint2* __restrict__ ptab,
                                                   const uint2* __restrict__ mdims, uint32_t nl, int family,
                                                   uint32_t n, uint32_t m, uint32_t q0, uint32_t items, uint32_t H, uint32_t Hs,
                                                   uint32_t Kc, uint32_t Ys, int logC,
                                                   const double2* __restrict__ tw) {
    constexpr int logPr = LOGPR;
    extern __shared__ double2 buf[];
    const uint32_t bid = xcd_remap(blockIdx.x, gridDim.x);
    const uint32_t cg = bid / items, item = bid - cg * items;
    const int Pr = 1 << logPr, C = 1 << logC;
    const uint32_t k0 = cg << logC;
    uint32_t l = item, r = item;
    if constexpr (MODE == 1) {
        if (ptab) {
            l = ptab[q0 + item].x;
            r = ptab[q0 + item].y;
        } else {
            pair_of(family, n, m, q0 + item, l, r);
        }
    }
    const uint32_t Hq = mdims ? mdims[MODE == 1 ? nl + r : l].x : H;  // rows of this item's matrices
    const double2* Sm = S + (size_t)r * Kc * Hs;
    double2* Ll = Lhat + (size_t)l * Kc * Pr;
    if constexpr (regs_of<LOGPR>::ON) {
        // C = 8 * threads / Pr: the columns go from HBM to HBM through fft_regs; the product with
        // conj(Lhat) happens in registers between the two FFTs.
        constexpr int Q = 1 << (LOGPR - 3), P = 1 << LOGPR;
        const regs_pos<LOGPR> ps((int)threadIdx.x);
        const int t0 = ps.t0, i = ps.i;
        const uint32_t k = k0 + ps.t;
        const bool ok = k < Kc;
        double2* wb = buf + at<LOGPR>(t0, 0);
        const auto rr = load_roots<LOGPR, X>(i, tw);
        const __amdgpu_buffer_rsrc_t rs = buf_of(Sm, Kc * Hs * 16u), rl = buf_of(Ll, Kc * (uint32_t)P * 16u);
        const uint32_t so = (k * Hs + (uint32_t)i) * 16u, lo = ok ? (k * (uint32_t)P + (uint32_t)i) * 16u : kOut;
        const uint32_t rows = ok ? Hq : 0;
        double2 u[8], lh[8];
#pragma unroll
        for (int r = 0; r < 4; ++r)  // Hq <= Pr / 2: the upper half of a column is padding
            u[r] = buf_load(rs, (uint32_t)(i + Q * r) < rows ? so + 16u * Q * r : kOut, 0);
        // The left spectrum is loaded together with the column (its latency overlaps the
        // first transform's).
        if constexpr (MODE == 1) {
#pragma unroll
            for (int r = 0; r < 8; ++r) lh[r] = buf_load(rl, lo, 16u * Q * r);
        }
        fft_regs<LOGPR, true>(u, wb, rr, ps.t - t0, i);
        if constexpr (MODE == 0) {
#pragma unroll
            for (int r = 0; r < 8; ++r) buf_store(u[r], rl, lo, 16u * Q * r);
            return;
        }
#pragma unroll
        for (int r = 0; r < 8; ++r) u[r] = cmul(cconj(lh[r]), u[r]);
        // An opaque copy of the position: the second transform recomputes its LDS addresses
        // instead of keeping the first one's live across the product (fewer VGPRs).
        int tl2 = ps.t - t0, i2 = i;
        asm volatile("" : "+v"(tl2), "+v"(i2));
        fft_regs<LOGPR>(u, wb, rr, tl2, i2);
        // z_row: rows below Hq (r < 4: Hq <= Pr / 2) in place, rows above Pr - Hq (r >= 4) down by
        // Pr - Ys; indices from the opaque i2, so that those of the loads are not kept live.
        const uint32_t whole = z_lines(rows, Ys), second = z_second(rows, whole, P);
        const __amdgpu_buffer_rsrc_t rz = buf_of(Z + (size_t)item * Kc * Ys, Kc * Ys * 16u);
        const uint32_t zlo = (k * Ys + (uint32_t)i2) * 16u, zhi = zlo - ((uint32_t)P - Ys) * 16u;
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            const uint32_t rho = (uint32_t)(i2 + Q * r);
            const bool in = r < 4 ? rho < whole : rho >= second;
            buf_store(u[r], rz, in ? (r < 4 ? zlo : zhi) + 16u * Q * r : kOut, 0);
        }
        return;
    } else {
    // Slab: C = 2^LOGS / Pr columns; element idx of the slab is row rho of column k0 + t.
    // All loads (the column and, for pairs, the left spectrum) are issued before the first
    // transform, from clamped in-bounds addresses.
    constexpr int NI = (1 << slab_of<LOGPR>::LOGS) / kFT;
    const slab_roots<LOGPR> sr = load_slab_roots<LOGPR>(tw);
    double2 xs[NI], lh[NI];
#pragma unroll
    for (int q = 0; q < NI; ++q) {
        const int idx = threadIdx.x + kFT * q;
        const uint32_t k = k0 + (idx >> logPr), rho = idx & (Pr - 1);
        const uint32_t kk = k < Kc ? k : Kc - 1;
        xs[q] = Sm[(size_t)kk * Hs + (rho < Hq ? rho : Hq - 1)];
        lh[q] = MODE == 1 ? Ll[(size_t)kk * Pr + rho] : make_double2(0.0, 0.0);
    }
#pragma unroll
    for (int q = 0; q < NI; ++q) {
        const int idx = threadIdx.x + kFT * q;
        const uint32_t k = k0 + (idx >> logPr), rho = idx & (Pr - 1);
        buf[at<LOGPR>(idx >> logPr, rho)] = (k < Kc && rho < Hq) ? xs[q] : make_double2(0.0, 0.0);
    }
    __syncthreads();
    fft_slab<LOGPR>(buf, C, sr);
    if constexpr (MODE == 0) {
#pragma unroll
        for (int q = 0; q < NI; ++q) {
            const int idx = threadIdx.x + kFT * q;
            const uint32_t k = k0 + (idx >> logPr);
            if (k < Kc) Ll[(size_t)k * Pr + (idx & (Pr - 1))] = buf[at<LOGPR>(idx >> logPr, idx & (Pr - 1))];
        }
        return;
    }
    // conj(Lhat * conj(X)) = conj(Lhat) * X; its forward FFT, conjugated, is Pr * IFFT.
#pragma unroll
    for (int q = 0; q < NI; ++q) {
        const int idx = threadIdx.x + kFT * q;
        double2& v = buf[at<LOGPR>(idx >> logPr, idx & (Pr - 1))];
        v = k0 + (idx >> logPr) < Kc ? cmul(cconj(lh[q]), v) : make_double2(0.0, 0.0);
    }
    __syncthreads();
    fft_slab<LOGPR>(buf, C, sr);
    double2* Zq = Z + (size_t)item * Kc * Ys;
#pragma unroll
    for (int q = 0; q < NI; ++q) {
        const int idx = threadIdx.x + kFT * q;
        const uint32_t k = k0 + (idx >> logPr);
        const int y = z_row((uint32_t)(idx & (Pr - 1)), Hq, Ys, (uint32_t)Pr);
        if (k < Kc && y >= 0) Zq[(size_t)k * Ys + y] = buf[at<LOGPR>(idx >> logPr, idx & (Pr - 1))];
    }
    }
}

// rows_inv: block (pair item, group of 2T consecutive rows z0 = 2T*g ... of Z, column stride
// Ys), so that each thread's two rows are adjacent in Z and a group's rows are one aligned
// run.  With mdims (uneven batches) the pair's size is that of its right matrix
// nl + ptab[q].y.  Row z goes to output row out_row_of_z(z) (row H of Z, which holds nothing,
// is read as zero); output column ox = dx + W - 1 takes circular column dx mod Pc.  Pair q's
// result starts at ooff[q] when the table is given, else at q times the result size.
template <typename Tout, int LOGPC, int NT = rows_block<LOGPC, true>::NT>
__global__ __launch_bounds__(NT) void rows_inv_slab_kernel(const double2* __restrict__ Z, Tout* __restrict__ O,
                                                       const uint64_t* __restrict__ ooff,
                                                       const uint2* __restrict__ ptab, const uint2* __restrict__ mdims,
                                                       uint32_t nl, uint32_t q0, uint32_t H, uint32_t W, uint32_t Ys,
                                                       int logT, uint32_t groups, double scale,
                                                       const double2* __restrict__ tw) {
    constexpr int logPc = LOGPC;
    extern __shared__ double2 buf[];
    // XCD-aware order: the row groups of one pair run on one XCD, so the lines of Z that
    // neighbouring groups read in pieces (2T rows of a column) are fetched into its L2 once.
    const uint32_t bid = xcd_remap(blockIdx.x, gridDim.x);
    const uint32_t item = bid / groups, g = bid - item * groups;
    const int Pc = 1 << logPc, T = 1 << logT;
    const int half = Pc / 2;
    const uint32_t Kc = (uint32_t)half + 1;
    if (mdims) {  // uneven batch: this pair's own size (at most H x W)
        const uint2 d = mdims[nl + ptab[q0 + item].y];
        H = d.x;
        W = d.y;
    }
    const uint32_t SX = 2 * W - 1;
    const uint32_t z0 = g << (logT + 1);
    const int rows2 = 2 << logT;
    if (z_gap(z0, (uint32_t)rows2, H, Ys)) return;  // between the two halves of the result
    const double2* Zq = Z + (size_t)item * Kc * Ys;
    static_assert(!regs_of<LOGPC>::ON && NT == kFT, "slab transforms");
    const slab_roots<LOGPC> sr = load_slab_roots<LOGPC>(tw);
    // One thread per (column kk, transform t) loads the two rows' values A[kk], B[kk] (32
    // adjacent bytes, conjugated) and writes both slots kk and Pc-kk of conj(Y), Y[k] = A[k] +
    // i B[k] extended by A[Pc-k] = conj(A[k]), B[Pc-k] = conj(B[k]).
    {
        // At most TMAX = 2^LOGS / Pc transforms, so (Kc << logT) <= (Pc/2 + 1) * TMAX items: all
        // loads first, then the writes.
        constexpr int TMAX = (1 << rows_block<LOGPC, true>::LOGS) >> LOGPC;
        constexpr int NQ = (((1 << (LOGPC - 1)) + 1) * TMAX + NT - 1) / NT;
        const int items = (int)Kc << logT;
        double2 A[NQ], B[NQ];
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const int idx = threadIdx.x + NT * q;
            const int kk = idx >> logT, t = idx & (T - 1);
            const uint32_t za = z0 + 2 * t;
            const double2* zc = Zq + (size_t)kk * Ys + za;
            A[q] = make_double2(0.0, 0.0);
            B[q] = make_double2(0.0, 0.0);
            if (idx < items && out_row_of_z(za, H, Ys) >= 0) A[q] = zc[0];
            if (idx < items && out_row_of_z(za + 1, H, Ys) >= 0) B[q] = zc[1];
        }
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const int idx = threadIdx.x + NT * q;
            if (idx >= items) continue;
            const int kk = idx >> logT, t = idx & (T - 1);
            buf[at<LOGPC>(t, kk)] = cadd(A[q], mul_mi(B[q]));
            if (kk > 0 && kk < half) buf[at<LOGPC>(t, Pc - kk)] = cadd(cconj(A[q]), mul_mi(cconj(B[q])));
        }
    }
    __syncthreads();
    Tout* Oq = O + (ooff ? ooff[q0 + item] : (size_t)(q0 + item) * (2 * H - 1) * SX);
    fft_slab<LOGPC>(buf, T, sr);
    // IFFT(Y) = conj(FFT(conj(Y))) / Pc: row A is the real part, row B minus the imaginary.
    for (int rr = threadIdx.x >> 6; rr < rows2; rr += NT / 64) {
        const int oy = out_row_of_z(z0 + rr, H, Ys);
        if (oy < 0) continue;
        Tout* orow = Oq + (size_t)oy * SX;
        const int t = rr >> 1;
        for (int ox = threadIdx.x & 63; ox < (int)SX; ox += 64) {
            const int c = (ox - (int)(W - 1)) & (Pc - 1);
            const double2 f = buf[at<LOGPC>(t, c)];
            orow[ox] = (Tout)(((rr & 1) ? -f.y : f.x) * scale);
        }
    }
}

// rows_inv for register transforms (up to 2048 points), T row pairs per block.  A thread's columns
// kk0 + Q q and its LDS slots are a constant apart (Q = Pc / 8 threads per row pair), and rows and
// columns outside the result are dropped by their buffer offsets, so that little but the FP64 work
// is left: 422 VALU instructions at 512 points for 294 of FP64, where branches and index
// arithmetic had made them 700 for 316 (64 pairs of 256^2 35.8 -> 33.1 us, 32 of 1024^2 430 -> 368).
template <typename Tout, int LOGPC, int NT = rows_block<LOGPC, true>::NT>
__global__ __launch_bounds__(NT) void rows_inv_regs_kernel(const double2* __restrict__ Z, Tout* __restrict__ O,
                                                           const uint64_t* __restrict__ ooff,
                                                           const uint2* __restrict__ ptab,
                                                           const uint2* __restrict__ mdims, uint32_t nl, uint32_t q0,
                                                           uint32_t H, uint32_t W, uint32_t Ys, uint32_t groups,
                                                           double scale, const double2* __restrict__ tw) {
    static_assert(regs_of<LOGPC>::ON, "register transforms only");
    constexpr int Pc = 1 << LOGPC, half = Pc / 2, Q = Pc / 8;
    constexpr uint32_t Kc = half + 1;
    constexpr int T = 8 * NT / Pc, LOGT = rows_block<LOGPC, true>::LOGS - LOGPC;
    static_assert(T == 1 << LOGT, "transforms per block");
    extern __shared__ double2 buf[];
    // XCD-aware order: the row groups of one pair run on one XCD, so the lines of Z that
    // neighbouring groups read in pieces (2T rows of a column) are fetched into its L2 once.
    const uint32_t bid = xcd_remap(blockIdx.x, gridDim.x);
    const uint32_t item = bid / groups, g = bid - item * groups;
    if (mdims) {  // uneven batch: this pair's own size (at most H x W)
        const uint2 d = mdims[nl + ptab[q0 + item].y];
        H = d.x;
        W = d.y;
    }
    const uint32_t z0 = g << (LOGT + 1);
    if (z_gap(z0, 2 * T, H, Ys)) return;  // between the two halves of the result
    const regs_pos<LOGPC> ps((int)threadIdx.x);
    const auto rr = load_roots<LOGPC, exact_roots<Tout>>(ps.i, tw);
    // Columns kk0 + Q q of row pair tq: A, B (conjugated) -> slots kk and Pc - kk of conj(Y), Y[k] =
    // A[k] + i B[k] extended by A[Pc-k] = conj(A[k]), B[Pc-k] = conj(B[k]).
    {
        const int tq = (int)threadIdx.x & (T - 1), kk0 = (int)threadIdx.x >> LOGT;
        const uint32_t za = z0 + 2 * tq;
        const bool oka = out_row_of_z(za, H, Ys) >= 0, okb = out_row_of_z(za + 1, H, Ys) >= 0;
        const __amdgpu_buffer_rsrc_t rz = buf_of(Z + (size_t)item * Kc * Ys, Kc * Ys * 16u);
        const uint32_t voff = ((uint32_t)kk0 * Ys + za) * 16u, va = oka ? voff : kOut, vb = okb ? voff + 16u : kOut;
        const uint32_t step = Q * Ys * 16u;
        double2 A[4], B[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            A[q] = buf_load(rz, va, q * step);
            B[q] = buf_load(rz, vb, q * step);
        }
        if (kk0 == 0) {  // column Pc / 2
            const double2 a = buf_load(rz, va, 4 * step), b = buf_load(rz, vb, 4 * step);
            buf[at<LOGPC>(tq, half)] = cadd(a, mul_mi(b));
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const double2 a = A[q], b = B[q];
            // at(t, kk0 + Q q) = at(t, kk0) + q (Q + Q/8) when 8 divides Q, at(t, Pc - kk) likewise;
            // slot Pc, for column 0, is the pad slot behind transform t
            const int s0 = Q % 8 == 0 ? at<LOGPC>(tq, kk0) + q * (Q + Q / 8) : at<LOGPC>(tq, kk0 + Q * q);
            const int s1 = Q % 8 == 0 ? at<LOGPC>(tq, Pc - kk0) - q * (Q + Q / 8) : at<LOGPC>(tq, Pc - kk0 - Q * q);
            buf[s0] = make_double2(a.x + b.y, a.y - b.x);
            buf[s1] = make_double2(a.x - b.y, -a.y - b.x);
        }
    }
    __syncthreads();
    const int t = ps.t, i = ps.i;
    double2 u[8];
#pragma unroll
    for (int r = 0; r < 8; ++r)
        u[r] = buf[Q % 8 == 0 ? at<LOGPC>(t, i) + r * (Q + Q / 8) : at<LOGPC>(t, i + Q * r)];
    // a block-owned transform's first pass overwrites slots other waves still read
    if constexpr (regs_of<LOGPC>::BLOCK) __syncthreads();
    fft_regs<LOGPC>(u, buf + at<LOGPC>(ps.t0, 0), rr, t - ps.t0, i);
    // IFFT(Y) = conj(FFT(conj(Y))) / Pc: row A is the real part, row B minus the imaginary; circular
    // column c = i + Q r is shift c for r < 4 and c - Pc above (W <= Pc / 2).
    const int SX = 2 * (int)W - 1;
    Tout* Oq = O + (ooff ? ooff[q0 + item] : (size_t)(q0 + item) * (2 * H - 1) * SX);
    const __amdgpu_buffer_rsrc_t ro = buf_of(Oq, (2 * H - 1) * (uint32_t)SX * (uint32_t)sizeof(Tout));
    const int oa = out_row_of_z(z0 + 2 * t, H, Ys), ob = out_row_of_z(z0 + 2 * t + 1, H, Ys);
    const uint32_t va = oa >= 0 ? (uint32_t)(oa * SX + i) * (uint32_t)sizeof(Tout) : kOut;
    const uint32_t vb = ob >= 0 ? (uint32_t)(ob * SX + i) * (uint32_t)sizeof(Tout) : kOut;
#pragma unroll
    for (int r = 0; r < 8; ++r) {
        const bool in = r < 4 ? i + Q * r < (int)W : i + Q * r > Pc - (int)W;
        const uint32_t off = (uint32_t)(Q * r + (r < 4 ? (int)W - 1 : (int)W - 1 - Pc)) * (uint32_t)sizeof(Tout);
        buf_store((Tout)(u[r].x * scale), ro, in && oa >= 0 ? va + off : kOut, 0);
        buf_store((Tout)(-u[r].y * scale), ro, in && ob >= 0 ? vb + off : kOut, 0);
    }
}

// Row transforms of P = 3N points (N = 2^LOGN, 16..512), for widths where 3N >= 2W - 1 is
// shorter than the power of two.  A transform (row pair) is three of N points through
// fft_regs<LOGN> (3T wave-owned transforms per block, sub-transform 3t + m) and one radix-3 step,
// with w = exp(-2 pi i / P) and W_3 = w^N:
//   forward (decimation in time): F_m = FFT of x[3n + m]; the split into the two rows' spectra is
//     done on the F_m, a_m[k] = (F_m[k] + conj(F_m[N-k])) / 2 and b_m[k] = (F_m[k] -
//     conj(F_m[N-k])) / 2i, and row A's bins are A[k + N j] = sum_m w^(km) W_3^(jm) a_m[k] for
//     k = 0..N/2 (bin k + 2N is the conjugate of bin N - k), so the spectrum of the pair never
//     goes through LDS;
//   inverse (decimation in frequency): from the conjugated bins k, N + k, N - k of rows A and B,
//     ah_m = w^(km) sum_j W_3^(jm) conj(A[k + N j]) and bh_m, the sub-sequences of the extended
//     row are y_m[k] = ah_m - i bh_m and y_m[N - k] = conj(ah_m) - i conj(bh_m); their transforms
//     give X[3q + m], which go through LDS as real output values so that rows are stored whole.
// HBM-bound.  Splitting the sub-transforms' spectra instead of the whole one saves a write and a
// read of all values through LDS with a barrier in both directions, and bounds-checked loads and
// stores a branch per element: at 65 matrices of 350^2 rows_fwd3 54 -> 43 us (3.9 TB/s), rows_inv3
// 125 -> 111 us (3.6 TB/s); the whole call 291 -> 254 us, 640^2 1124 -> 977, 190^2 69.7 -> 63.8.
// A block holds T transforms (3T N / 8 threads, a multiple of 64): 2 at 1536 points (two
// blocks per CU measured faster than one), 4 from 384 to 768, more below (192 threads).
constexpr int rows3_t(int logN) { return logN >= 9 ? 2 : (logN >= 7 ? 4 : 512 >> logN); }
template <int LOGN>
struct rows3 {
    static constexpr int N = 1 << LOGN, P = 3 * N, Q = N / 8;
    static constexpr int T = rows3_t(LOGN);                 // transforms (row pairs) per block
    static constexpr int NT = 3 * T * N / 8;
    static constexpr int LOGT = T == 2 ? 1 : (T == 4 ? 2 : (T == 8 ? 3 : (T == 16 ? 4 : 5)));
    static constexpr int SLOTS = 3 * T * (N + N / 8 + 1);
    static constexpr int FS = NT / (2 * T), IS = NT / T;    // k steps of the split and of the extension
    static constexpr int FQ = 3, IQ = 2;                    // and their number: k = 0..N/2
    static_assert(NT % 64 == 0 && NT <= 1024 && (1 << LOGT) == T && 8 * NT == T * P, "rows3 geometry");
    static_assert(FS * FQ > N / 2 && IS * IQ > N / 2, "rows3 steps");
    static_assert(NT < P || (NT % P == 0 && 2 * T % (NT / P) == 0), "rows3 output rows");
};

// tw3[j] = exp(-2 pi i j / 12288): the P-th roots for P = 3 * 2^n <= 12288, one table per
// device, kept for the process.
constexpr int kTw3 = 3 * kSlab;
const double2* twiddles3();

// 3-point DFT: x0 = a + b + c, x1 and x2 its other bins.
__device__ __forceinline__ void dft3(const double2 a, const double2 b, const double2 c, double2& x0, double2& x1,
                                     double2& x2) {
    constexpr double h = 0.86602540378443864676;  // sqrt(3) / 2
    const double2 sm = cadd(b, c), df = csub(b, c);
    const double2 t1 = make_double2(a.x - 0.5 * sm.x, a.y - 0.5 * sm.y);
    x0 = cadd(a, sm);
    x1 = make_double2(fma(h, df.y, t1.x), fma(-h, df.x, t1.y));
    x2 = make_double2(fma(-h, df.y, t1.x), fma(h, df.x, t1.y));
}

// rows_fwd for P = 3N: a persistent grid as rows_fwd_regs_kernel (items: matrix, group of 2T
// rows; each XCD walks one contiguous eighth of the items; the next item's rows are loaded
// into registers while the current one is transformed and stored), matrices, offsets, sizes
// and output S as rows_fwd_slab_kernel.
template <typename Tin, int LOGN>
__global__ __launch_bounds__(rows3<LOGN>::NT) void rows_fwd3_kernel(
    const Tin* __restrict__ XL, const Tin* __restrict__ XR, const uint64_t* __restrict__ moff,
    const uint2* __restrict__ mdims, uint32_t nl, uint32_t H, uint32_t Hs, uint32_t W, uint32_t groups,
    uint32_t items, double2* __restrict__ SL, double2* __restrict__ SR, const double2* __restrict__ tw,
    const double2* __restrict__ tw3) {
    using G = rows3<LOGN>;
    constexpr int N = G::N, P = G::P, Q = G::Q, T = G::T, FS = G::FS;
    constexpr uint32_t Kc = P / 2 + 1;
    extern __shared__ double2 buf[];
    const regs_pos<LOGN> ps((int)threadIdx.x);
    const int sub = ps.t, tt = sub / 3, m = sub - 3 * tt, i = ps.i;
    const auto rr = load_roots<LOGN, exact_roots<Tin>>(i, tw);
    // the split: row rw of the group (an A or a B of row pair tq) at k = k0 + FS q
    const int rw = (int)threadIdx.x & (2 * T - 1), tq = rw >> 1, odd = rw & 1;
    const int k0 = (int)threadIdx.x >> (G::LOGT + 1);
    double2 w1[G::FQ], w2[G::FQ];
#pragma unroll
    for (int q = 0; q < G::FQ; ++q) {
        w1[q] = tw3[(k0 + FS * q) * (kTw3 / P)];
        if constexpr (exact_roots<Tin>) w2[q] = tw3[2 * (k0 + FS * q) * (kTw3 / P)];
    }
    const uint32_t nx = gridDim.x >= 8 ? 8 : 1;
    const uint32_t x = blockIdx.x % nx, kb = blockIdx.x / nx, bpx = gridDim.x / nx;
    const uint32_t per = (items + nx - 1) / nx;
    const uint32_t end = min((x + 1) * per, items);
    struct where {
        uint32_t matg, r0, Hm, Wm;
    };
    auto locate = [&](uint32_t it) {
        where w;
        w.matg = it / groups;
        w.r0 = (it - w.matg * groups) * (2 * T);
        w.Hm = H;
        w.Wm = W;
        if (mdims) {
            const uint2 d = mdims[w.matg];
            w.Hm = d.x;
            w.Wm = d.y;
        }
        return w;
    };
    // element n = i + Q r of sub-sequence m is column 3n + m; rows and columns outside the matrix
    // read zero (W <= P / 2: the upper half of a sub-sequence is padding)
    auto fetch = [&](const where& w, Tin (&va)[4], Tin (&vb)[4]) {
        const uint32_t mat = w.matg < nl ? w.matg : w.matg - nl;
        const Tin* Xm = (w.matg < nl ? XL : XR) + (moff ? moff[w.matg] : (size_t)mat * H * W);
        const __amdgpu_buffer_rsrc_t rx = buf_of(Xm, w.Hm * w.Wm * (uint32_t)sizeof(Tin));
        const uint32_t c0 = 3u * (uint32_t)i + (uint32_t)m;
        const uint32_t row = ((w.r0 + 2 * (uint32_t)tt) * w.Wm + c0) * (uint32_t)sizeof(Tin);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint32_t off = c0 + 3u * Q * r < w.Wm ? row + (uint32_t)(3 * Q * r * sizeof(Tin)) : kOut;
            va[r] = buf_load_real<Tin>(rx, off, 0);
            vb[r] = buf_load_real<Tin>(rx, off + w.Wm * (uint32_t)sizeof(Tin), 0);
        }
    };
    uint32_t it = x * per + kb;
    if (it >= end) return;
    where cur = locate(it);
    Tin va[4], vb[4];
    fetch(cur, va, vb);
    while (true) {
        const uint32_t nxt = it + bpx;
        const bool more = nxt < end;
        double2 u[8];
#pragma unroll
        for (int r = 0; r < 4; ++r) u[r] = make_double2((double)va[r], (double)vb[r]);
        where nw{};
        if (more) {
            nw = locate(nxt);
            fetch(nw, va, vb);
        }
        if (cur.r0 < cur.Hm) {  // block-uniform: a row group beyond a smaller matrix is skipped
            fft_regs<LOGN, true>(u, buf + at<LOGN>(ps.t0, 0), rr, sub - ps.t0, i);
#pragma unroll
            for (int r = 0; r < 8; ++r)
                buf[Q % 8 == 0 ? at<LOGN>(sub, i) + r * (Q + Q / 8) : at<LOGN>(sub, i + Q * r)] = u[r];
            __syncthreads();
            // the components of F_m that row rw takes, as in rows_fwd_regs_kernel
            const double hs = odd ? -0.5 : 0.5;
            const double* zs = reinterpret_cast<const double*>(buf) + odd;
            const double* zd = reinterpret_cast<const double*>(buf) + 1 - odd;
            const bool left = cur.matg < nl;
            const size_t mat = left ? cur.matg : cur.matg - nl;
            const __amdgpu_buffer_rsrc_t rs = buf_of((left ? SL : SR) + mat * Kc * Hs, Kc * Hs * 16u);
            const uint32_t row = cur.r0 + (uint32_t)rw;
#pragma unroll
            for (int q = 0; q < G::FQ; ++q) {
                const int k = k0 + FS * q;
                if (k > N / 2) continue;
                double2 f[3];
#pragma unroll
                for (int mm = 0; mm < 3; ++mm) {
                    const int a = at<LOGN>(3 * tq + mm, k), b = at<LOGN>(3 * tq + mm, (N - k) & (N - 1));
                    f[mm] = make_double2(0.5 * (zs[2 * a] + zs[2 * b]), hs * (zd[2 * a] - zd[2 * b]));
                }
                double2 x0, x1, x2;
                dft3(f[0], cmul(w1[q], f[1]), cmul(exact_roots<Tin> ? w2[q] : csqr(w1[q]), f[2]), x0, x1, x2);
                const uint32_t off = row < cur.Hm ? ((uint32_t)k * Hs + row) * 16u : kOut;
                buf_store(x0, rs, off, 0);
                buf_store(x1, rs, off, N * Hs * 16u);
                // bin N - k; k = 0 and N/2 have it already
                const bool third = k != 0 && k != N / 2 && row < cur.Hm;
                buf_store(cconj(x2), rs, third ? ((uint32_t)(N - k) * Hs + row) * 16u : kOut, 0);
            }
            __syncthreads();  // the next item's transform reuses the slab
        }
        if (!more) break;
        it = nxt;
        cur = nw;
    }
}

// rows_inv for P = 3N: block (pair item, group of 2T rows z0 = 2T g ... of Z), otherwise as
// rows_inv_regs_kernel (Z rows by z_row, output rows out_row_of_z, crop and quadrant swap by index).
template <typename Tout, int LOGN>
__global__ __launch_bounds__(rows3<LOGN>::NT) void rows_inv3_kernel(
    const double2* __restrict__ Z, Tout* __restrict__ O, const uint64_t* __restrict__ ooff,
    const uint2* __restrict__ ptab, const uint2* __restrict__ mdims, uint32_t nl, uint32_t q0, uint32_t H, uint32_t W,
    uint32_t Ys, uint32_t groups, double scale, const double2* __restrict__ tw, const double2* __restrict__ tw3) {
    using G = rows3<LOGN>;
    constexpr int N = G::N, P = G::P, Q = G::Q, T = G::T, IS = G::IS;
    constexpr uint32_t Kc = P / 2 + 1;
    extern __shared__ double2 buf[];
    const uint32_t bid = xcd_remap(blockIdx.x, gridDim.x);
    const uint32_t item = bid / groups, g = bid - item * groups;
    if (mdims) {
        const uint2 d = mdims[nl + ptab[q0 + item].y];
        H = d.x;
        W = d.y;
    }
    const uint32_t z0 = g * (2 * T);
    if (z_gap(z0, 2 * T, H, Ys)) return;
    const regs_pos<LOGN> ps((int)threadIdx.x);
    const int sub = ps.t, tt = sub / 3, m = sub - 3 * tt, i = ps.i;
    const auto rr = load_roots<LOGN, exact_roots<Tout>>(i, tw);
    // The extension: row pair tq at k = k0 + IS q, the bins k, N + k and N - k of both rows (Z holds
    // them conjugated).
    {
        const int tq = (int)threadIdx.x & (T - 1), k0 = (int)threadIdx.x >> G::LOGT;
        const uint32_t za = z0 + 2 * tq;
        const bool oka = out_row_of_z(za, H, Ys) >= 0, okb = out_row_of_z(za + 1, H, Ys) >= 0;
        const __amdgpu_buffer_rsrc_t rz = buf_of(Z + (size_t)item * Kc * Ys, Kc * Ys * 16u);
        double2 A[G::IQ][3], B[G::IQ][3], w1[G::IQ], wx[G::IQ];
#pragma unroll
        for (int q = 0; q < G::IQ; ++q) {
            const int k = k0 + IS * q;
            const uint32_t lo = ((uint32_t)k * Ys + za) * 16u, hi = ((uint32_t)(N - k) * Ys + za) * 16u;
            const bool ka = oka && k <= N / 2, kb = okb && k <= N / 2;
            w1[q] = tw3[(k <= N / 2 ? k : 0) * (kTw3 / P)];
            if constexpr (exact_roots<Tout>) wx[q] = tw3[2 * (k <= N / 2 ? k : 0) * (kTw3 / P)];
            A[q][0] = buf_load(rz, ka ? lo : kOut, 0);
            B[q][0] = buf_load(rz, kb ? lo + 16u : kOut, 0);
            A[q][1] = buf_load(rz, ka ? lo : kOut, N * Ys * 16u);
            B[q][1] = buf_load(rz, kb ? lo + 16u : kOut, N * Ys * 16u);
            A[q][2] = buf_load(rz, ka ? hi : kOut, 0);
            B[q][2] = buf_load(rz, kb ? hi + 16u : kOut, 0);
        }
#pragma unroll
        for (int q = 0; q < G::IQ; ++q) {
            const int k = k0 + IS * q;
            if (k > N / 2) continue;
            const double2 w2 = exact_roots<Tout> ? wx[q] : csqr(w1[q]);
            double2 a[3], b[3];
            dft3(A[q][0], A[q][1], cconj(A[q][2]), a[0], a[1], a[2]);
            dft3(B[q][0], B[q][1], cconj(B[q][2]), b[0], b[1], b[2]);
            a[1] = cmul(w1[q], a[1]);
            b[1] = cmul(w1[q], b[1]);
            a[2] = cmul(w2, a[2]);
            b[2] = cmul(w2, b[2]);
#pragma unroll
            for (int mm = 0; mm < 3; ++mm) {  // slot N, for k = 0, is the pad slot behind the sub-transform
                buf[at<LOGN>(3 * tq + mm, k)] = make_double2(a[mm].x + b[mm].y, a[mm].y - b[mm].x);
                buf[at<LOGN>(3 * tq + mm, N - k)] = make_double2(a[mm].x - b[mm].y, -a[mm].y - b[mm].x);
            }
        }
    }
    __syncthreads();
    double2 u[8];
#pragma unroll
    for (int r = 0; r < 8; ++r)
        u[r] = buf[Q % 8 == 0 ? at<LOGN>(sub, i) + r * (Q + Q / 8) : at<LOGN>(sub, i + Q * r)];
    wave_sync();
    fft_regs<LOGN>(u, buf + at<LOGN>(ps.t0, 0), rr, sub - ps.t0, i);
    __syncthreads();  // the output rows overlap the sub-transforms' slots
    // IFFT(Y) = conj(FFT(conj(Y))) / P: row A is the real part, row B minus the imaginary; element
    // q = i + Q r of sub-transform m is circular column 3q + m
    Tout* rows = reinterpret_cast<Tout*>(buf);
#pragma unroll
    for (int r = 0; r < 8; ++r) {
        const int c = 3 * (i + Q * r) + m;
        rows[(2 * tt) * P + c] = (Tout)(u[r].x * scale);
        rows[(2 * tt + 1) * P + c] = (Tout)(-u[r].y * scale);
    }
    __syncthreads();
    const int SX = 2 * (int)W - 1;
    Tout* Oq = O + (ooff ? ooff[q0 + item] : (size_t)(q0 + item) * (2 * H - 1) * SX);
    // The block's threads take as many rows at once as they hold P columns: at 48 and 96 points one row
    // each time leaves most of them idle (527 pairs of 230x18 48 us; 25 before rows went through LDS).
    constexpr int RP = G::NT >= P ? G::NT / P : 1, TR = G::NT >= P ? P : G::NT;  // rows; threads of each
    const int zr = (int)threadIdx.x / TR, x0 = (int)threadIdx.x - zr * TR;
#pragma unroll
    for (int z1 = 0; z1 < 2 * T; z1 += RP) {
        const int z = z1 + zr, oy = out_row_of_z(z0 + z, H, Ys);
        if (oy < 0) continue;
        for (int ox = x0; ox < SX; ox += TR) {
            const int c = ox - ((int)W - 1);
            Oq[(size_t)oy * SX + ox] = rows[z * P + (c < 0 ? c + P : c)];
        }
    }
}

int ilog2_ceil(uint32_t x) {
    int e = 0;
    while ((1u << e) < x) ++e;
    return e;
}

// Twiddle tables in device memory of the code object (no allocation): tw[j] =
// exp(-2 pi i j / 4096), tw[4096 + N + j] = exp(-2 pi i j / N) for N = 2, 4 .. 2048 and j < N (the same
// values side by side: packed_roots), and tw3[j] = exp(-2 pi i j / 12288).  The host computes them, in long
// double (the angle rounded to double is up to 4e-16 off), and copies them in once per device.
__device__ double2 g_tw[2 * kSlab];
__device__ double2 g_tw3[kTw3];

std::vector<double2> twiddle_values() {
    std::vector<double2> h(2 * kSlab);
    const long double two_pi = 6.283185307179586476925286766559005768L;
    for (int j = 0; j < kSlab; ++j) {
        // exact at the eighths of the circle, where cos/sin of the rounded argument are not
        const int oct = j % (kSlab / 8);
        if (oct == 0) {
            static const double c8[8][2] = {{1, 0},
                                            {0.70710678118654752440, -0.70710678118654752440},
                                            {0, -1},
                                            {-0.70710678118654752440, -0.70710678118654752440},
                                            {-1, 0},
                                            {-0.70710678118654752440, 0.70710678118654752440},
                                            {0, 1},
                                            {0.70710678118654752440, 0.70710678118654752440}};
            h[j] = make_double2(c8[j / (kSlab / 8)][0], c8[j / (kSlab / 8)][1]);
        } else {
            const long double a = two_pi * j / kSlab;
            h[j] = make_double2((double)std::cos(a), (double)-std::sin(a));
        }
    }
    for (int n = 2; n < kSlab; n *= 2)
        for (int j = 0; j < n; ++j) h[packed_roots(n) + j] = h[j * (kSlab / n)];
    return h;
}

std::vector<double2> twiddle3_values() {
    std::vector<double2> h(kTw3);
    const long double two_pi = 6.283185307179586476925286766559005768L;
    for (int j = 0; j < kTw3; ++j) {
        const long double a = two_pi * j / kTw3;
        h[j] = make_double2((double)std::cos(a), (double)-std::sin(a));
    }
    // exact at the twelfths of the circle (the radix-3 and radix-4 points)
    const double s3 = 0.86602540378443864676;
    const double c12[12][2] = {{1, 0},   {s3, -0.5}, {0.5, -s3}, {0, -1},  {-0.5, -s3}, {-s3, -0.5},
                               {-1, 0},  {-s3, 0.5}, {-0.5, s3}, {0, 1},   {0.5, s3},   {s3, 0.5}};
    for (int q = 0; q < 12; ++q) h[q * (kTw3 / 12)] = make_double2(c12[q][0], c12[q][1]);
    return h;
}

struct device_tables {
    bool ready = false;
    double2* tw = nullptr;
    double2* tw3 = nullptr;
};

// The current device's twiddle tables: on its first use the symbols' addresses are looked up
// and the values copied in (synchronously, before any kernel reads them).
const device_tables& tables_of_device() {
    static std::mutex mu;
    static std::vector<device_tables> per_dev;
    int dev = 0;
    XC_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lock(mu);
    if ((int)per_dev.size() <= dev) per_dev.resize(dev + 1);
    device_tables& t = per_dev[dev];
    if (!t.ready) {
        XC_HIP(hipGetSymbolAddress(reinterpret_cast<void**>(&t.tw), HIP_SYMBOL(g_tw)));
        XC_HIP(hipGetSymbolAddress(reinterpret_cast<void**>(&t.tw3), HIP_SYMBOL(g_tw3)));
        const std::vector<double2> h = twiddle_values(), h3 = twiddle3_values();
        XC_HIP(hipMemcpy(t.tw, h.data(), sizeof(double2) * h.size(), hipMemcpyHostToDevice));
        XC_HIP(hipMemcpy(t.tw3, h3.data(), sizeof(double2) * kTw3, hipMemcpyHostToDevice));
        t.ready = true;
    }
    return t;
}

const double2* twiddles() { return tables_of_device().tw; }
const double2* twiddles3() { return tables_of_device().tw3; }

struct slab_shape {
    int logS;      // log2 of the slab (values per block)
    bool regs;     // register transforms (regs_of)
    int logT;      // log2 of the transforms per block
    uint32_t lds;  // dynamic LDS bytes
};

// The slab of slab_of<LOGP> and the transforms per block: as many as `want` asks for, within
// the slab.  Register transforms (up to 2048 points) always fill it: 8 values per thread, so a
// block of `threads` holds 8 threads / P of them.
slab_shape shape_for(int logP, uint32_t want, int threads = 256) {
    slab_shape v{};
    v.regs = logP <= 11;  // as regs_of<LOGP>::ON
    // as rows_block<LOGP>::LOGS for the row kernels (threads), slab_of<LOGP>::LOGS otherwise
    v.logS = v.regs ? ilog2_ceil((uint32_t)threads) + 3 : std::max(11, logP);
    int lt = v.regs ? v.logS - logP : 0;
    while (lt + logP < v.logS && (1u << lt) < want) ++lt;
    v.logT = lt;
    v.lds = (uint32_t)(((1u << lt) * ((1u << logP) + (1u << logP) / 8 + 1)) * sizeof(double2));
    return v;
}

// Calls f(std::integral_constant<int, LOGP>) for the run-time transform length 2^logP.
template <typename F>
void with_logp(int logP, F&& f) {
    switch (logP) {
    case 4: f(std::integral_constant<int, 4>{}); break;
    case 5: f(std::integral_constant<int, 5>{}); break;
    case 6: f(std::integral_constant<int, 6>{}); break;
    case 7: f(std::integral_constant<int, 7>{}); break;
    case 8: f(std::integral_constant<int, 8>{}); break;
    case 9: f(std::integral_constant<int, 9>{}); break;
    case 10: f(std::integral_constant<int, 10>{}); break;
    case 11: f(std::integral_constant<int, 11>{}); break;
    case 12: f(std::integral_constant<int, 12>{}); break;
    default: fail(XC_ERR_UNSUPPORTED, "own-FFT method: transform length out of range");
    }
}

template <typename K>
void allow_lds(K kernel, uint32_t bytes) {
    if (bytes > 65536) allow_dynamic_lds(reinterpret_cast<const void*>(kernel), bytes);
}

struct fftk_geom {
    int logPr, logPc;  // logPc: of a power-of-two row length
    bool f3;           // row length Pc = 3 * 2^logN (rows3 kernels)
    int logN;
    uint32_t Pr, Pc, Kc;
    slab_shape v1, vc, v3;
    uint32_t g1, cg, g3;
    // A pair's half spectrum fits one block (xc_fftk_small.hip): lengths 2^logPrs x 2^logPcs; the
    // right spectra take S's place (column spectra of Pr values), Z and the left S are not used.
    bool small;
    int logPrs, logPcs;
    uint32_t Hs, Ys;  // column strides of S and Z (z_row)
    size_t s_bytes, sl_bytes, col_bytes, z_bytes;  // S per right and per left, Lhat per left, Z per pair
};

// Whether the one-block kernels serve H x W.  Not 129 to 192 columns, up to 16 rows: rows of 384 points, which
// they don't have, let the three passes take half the time (one pair of 2x180 24 / 11.5 us, 72 x 13 of 2x150
// 84 / 38; of 32x512 points at 16x150 25 / 14).  Nor 65 to 96 columns, up to 8 rows, padded to 32x256 instead of
// 16x192 points (926 of 1x73 45 / 26, 446 of 3x71 35 / 22, one of 5x90 14.5 / 13.2, 20 x 50 of 8x96 33 / 33; with
// more rows pairs that share their matrices lose: 16 x 64 of 20x80 42.5 / 47.5, 30 x 60 of 32x96 78 / 90).
bool small_serves(uint32_t H, uint32_t W) {
    const int lr = std::max(5, ilog2_ceil(2 * H - 1)), lc = std::max(5, ilog2_ceil(2 * W - 1));
    if (lc == 9 && 2 * W - 1 <= 384) return false;
    if (lc == 8 && 2 * W - 1 <= 192 && H <= 8) return false;
    return fftk_small_fits(lr, lc);
}

// plain: the layout that takes the least memory per matrix (no one-block kernels, no rounding of
// the column strides).
fftk_geom geom_of(uint32_t H, uint32_t W, bool pow2_rows = false, bool plain = false) {
    if (H == 0 || W == 0 || 2 * H - 1 > (uint32_t)kSlab || 2 * W - 1 > (uint32_t)kSlab)
        fail(XC_ERR_UNSUPPORTED, "own-FFT method: rows and cols must be 1..2048");
    fftk_geom g{};
    g.logPr = std::max(4, ilog2_ceil(2 * H - 1));
    g.Pr = 1u << g.logPr;
    g.Pc = pow2_rows ? fftk_col_len(W) : fftk_row_len(W);
    g.f3 = (g.Pc & (g.Pc - 1)) != 0;
    g.logN = g.f3 ? ilog2_ceil(g.Pc / 3) : 0;
    g.logPc = g.f3 ? 0 : ilog2_ceil(g.Pc);
    g.Kc = g.Pc / 2 + 1;
    // Slab shape per kernel (see shape_for): rows_fwd 2T input rows per block, cols C columns,
    // rows_inv 2T output rows.
    g.vc = shape_for(g.logPr, g.Kc, cols_threads(g.logPr));
    if (g.f3) {  // rows3<logN>: T = 8 NT / P transforms per block of NT threads
        const uint32_t n = g.Pc / 3, t = (uint32_t)rows3_t(g.logN), slots = 3 * t * (n + n / 8 + 1);
        g.v1 = slab_shape{0, true, ilog2_ceil(t), slots * (uint32_t)sizeof(double2)};
        g.v3 = g.v1;
    } else {
        g.v1 = shape_for(g.logPc, (H + 1) / 2, rows_threads(g.logPc, false));
        g.v3 = shape_for(g.logPc, H, rows_threads(g.logPc, true));
    }
    g.g1 = (H + (2u << g.v1.logT) - 1) >> (g.v1.logT + 1);
    g.cg = (g.Kc + (1u << g.vc.logT) - 1) >> g.vc.logT;
    g.Hs = plain ? H : (H + 7) & ~7u;
    g.Ys = 2 * g.Hs;
    g.g3 = (g.Ys + (2u << g.v3.logT) - 1) >> (g.v3.logT + 1);  // a block may be taller
    g.s_bytes = sizeof(double2) * (size_t)g.Kc * g.Hs;
    g.col_bytes = sizeof(double2) * (size_t)g.Kc * g.Pr;
    g.z_bytes = sizeof(double2) * (size_t)g.Kc * g.Ys;
    g.sl_bytes = g.s_bytes;
    g.logPrs = std::max(5, g.logPr);
    g.logPcs = std::max(5, ilog2_ceil(2 * W - 1));
    g.small = !plain && small_serves(H, W);
    if (g.small) {
        g.col_bytes = sizeof(double2) * (size_t)((1u << g.logPcs) / 2 + 1) << g.logPrs;
        g.s_bytes = g.col_bytes;
        g.sl_bytes = g.z_bytes = 0;
    }
    return g;
}

// Blocks of `kernel` (threads, dynamic LDS bytes) that the device holds at once, for a
// persistent grid over `items` work items: at most `items`, a multiple of the 8 XCDs when
// there are at least 8.  The occupancy is queried once per kernel and size.
uint32_t resident_grid(const void* kernel, int threads, uint32_t lds, uint32_t items) {
    static std::mutex mu;
    static std::vector<std::tuple<const void*, int, uint32_t, int, uint32_t>> known;  // kernel, threads, lds, dev, blocks
    int dev = 0;
    XC_HIP(hipGetDevice(&dev));
    uint32_t resident = 0;
    {
        std::lock_guard<std::mutex> lock(mu);
        for (const auto& e : known)
            if (std::get<0>(e) == kernel && std::get<1>(e) == threads && std::get<2>(e) == lds && std::get<3>(e) == dev)
                resident = std::get<4>(e);
        if (resident == 0) {
            int per_cu = 0, cus = 0;
            XC_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, threads, lds));
            XC_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
            resident = (uint32_t)cus * (uint32_t)std::max(per_cu, 1);
            known.emplace_back(kernel, threads, lds, dev, resident);
        }
    }
    uint32_t g = std::min<uint32_t>(items, resident);
    if (g >= 8) g -= g % 8;
    return std::max<uint32_t>(g, 1);
}

template <typename Tio>
void launch_job(const fftk_job& j, const Tio* L, const Tio* R, Tio* O, const fftk_ws& ws, hipStream_t s,
                bool timing) {
    const uint32_t H = j.H, W = j.W;
    const fftk_geom g = geom_of(H, W, j.pow2_rows, j.plain);
    if (g.small) {
        if constexpr (std::is_same<Tio, float>::value)
            fftk_small_f32(j, g.logPrs, g.logPcs, L, R, O, ws, s, timing);
        else
            fftk_small_f64(j, g.logPrs, g.logPcs, L, R, O, ws, s, timing);
        return;
    }
    const double2* tw = twiddles();
    double2* SR = static_cast<double2*>(ws.sr);
    double2* SL = static_cast<double2*>(ws.sl);
    double2* LH = static_cast<double2*>(ws.lh);
    double2* Zw = static_cast<double2*>(ws.z);
    const uint32_t chunk = std::max<uint32_t>(1, std::min<uint32_t>(j.pairs, ws.zchunk));
    const uint2* ptab = reinterpret_cast<const uint2*>(j.ptab);
    const uint2* mdims = reinterpret_cast<const uint2*>(j.mdims);
    const double2* tw3 = g.f3 ? twiddles3() : nullptr;
    if (g.f3) {
        with_logp(g.logN, [&](auto LN) {
            constexpr int LOGN = decltype(LN)::value;
            if constexpr (LOGN <= 9) {
                using G3 = rows3<LOGN>;
                if (G3::SLOTS * sizeof(double2) != g.v1.lds || G3::P != (int)g.Pc)
                    fail(XC_ERR_UNSUPPORTED, "own-FFT method: inconsistent 3N-point row geometry");
                auto k = rows_fwd3_kernel<Tio, LOGN>;
                allow_lds(k, g.v1.lds);
                const uint32_t items = (j.nl + j.nr) * g.g1;
                const uint32_t grid = resident_grid(reinterpret_cast<const void*>(k), G3::NT, g.v1.lds, items);
                launch_timed("fftk_rows_fwd", timing, k, dim3(grid), dim3(G3::NT), g.v1.lds, s, L, R, j.moff, mdims,
                             j.nl, H, g.Hs, W, g.g1, items, SL, SR, tw, tw3);
            }
        });
    } else
    with_logp(g.logPc, [&](auto LP) {
        constexpr int LOGPC = decltype(LP)::value;
        const uint32_t items = (j.nl + j.nr) * g.g1;
        if constexpr (regs_of<LOGPC>::ON) {
            auto k = rows_fwd_regs_kernel<Tio, LOGPC>;
            allow_lds(k, g.v1.lds);
            const uint32_t grid = resident_grid(reinterpret_cast<const void*>(k), rows_threads(LOGPC, false),
                                                g.v1.lds, items);
            launch_timed("fftk_rows_fwd", timing, k, dim3(grid), dim3(rows_threads(LOGPC, false)), g.v1.lds, s, L, R,
                         j.moff, mdims, j.nl, H, g.Hs, W, g.g1, items, SL, SR, tw);
        } else {
            auto k = rows_fwd_slab_kernel<Tio, LOGPC>;
            allow_lds(k, g.v1.lds);
            launch_timed("fftk_rows_fwd", timing, k, dim3(items), dim3(kFT), g.v1.lds, s, L, R, j.moff, mdims, j.nl, H,
                         g.Hs, W, g.v1.logT, g.g1, SL, SR, tw);
        }
    });
    auto cols = [&](const char* name, const double2* S, double2* Zout, auto MODE, uint32_t items,
                    uint32_t q0) {
        with_logp(g.logPr, [&](auto LP) {
            auto k = cols_kernel<decltype(LP)::value, decltype(MODE)::value, exact_roots<Tio>>;
            allow_lds(k, g.vc.lds);
            launch_timed(name, timing, k, dim3(items * g.cg), dim3(cols_threads(g.logPr)), g.vc.lds, s, S, LH, Zout,
                         ptab, mdims, j.nl, j.family, j.n, j.m, q0, items, H, g.Hs, g.Kc, g.Ys, g.vc.logT, tw);
        });
    };
    // Column kernel of a chunk: grouped (cols_group_kernel has the reasons for both lines) or from Lhat.
    const uint32_t waves = std::min(chunk, j.pairs) * g.cg * (uint32_t)cols_threads(g.logPr) / 64;
    const bool grouped = g.logPr <= 11 && (j.pairs <= 4 * j.nl || waves <= 6144);
    const uint32_t G = waves > 4608 && j.pairs > j.nl ? 2 : 1;
    auto cols_group = [&](uint32_t nq, uint32_t q0) {
        with_logp(g.logPr, [&](auto LP) {
            constexpr int LOGPR = decltype(LP)::value;
            if constexpr (regs_of<LOGPR>::ON) {
                auto k = cols_group_kernel<LOGPR, exact_roots<Tio>>;
                allow_lds(k, g.vc.lds);
                const uint32_t items = (nq + G - 1) / G;
                launch_timed("fftk_cols", timing, k, dim3(items * g.cg), dim3(cols_threads(g.logPr)), g.vc.lds, s,
                             (const double2*)SL, (const double2*)SR, Zw, ptab, mdims, j.nl, j.family, j.n, j.m, q0, nq,
                             G, items, H, g.Hs, g.Kc, g.Ys, tw);
            }
        });
    };
    if (!grouped) cols("fftk_cols_left", SL, nullptr, std::integral_constant<int, 0>{}, j.nl, 0);
    const double scale = 1.0 / ((double)g.Pr * (double)g.Pc);
    for (uint32_t q0 = 0; q0 < j.pairs; q0 += chunk) {
        const uint32_t nq = std::min(chunk, j.pairs - q0);
        if (grouped)
            cols_group(nq, q0);
        else
            cols("fftk_cols", SR, Zw, std::integral_constant<int, 1>{}, nq, q0);
        if (g.f3) {
            with_logp(g.logN, [&](auto LN) {
                constexpr int LOGN = decltype(LN)::value;
                if constexpr (LOGN <= 9) {
                    using G3 = rows3<LOGN>;
                    auto k = rows_inv3_kernel<Tio, LOGN>;
                    allow_lds(k, g.v3.lds);
                    launch_timed("fftk_rows_inv", timing, k, dim3(nq * g.g3), dim3(G3::NT), g.v3.lds, s,
                                 (const double2*)Zw, O, j.ooff, ptab, mdims, j.nl, q0, H, W, g.Ys, g.g3, scale, tw,
                                 tw3);
                }
            });
            continue;
        }
        with_logp(g.logPc, [&](auto LP) {
            constexpr int LOGPC = decltype(LP)::value;
            const dim3 grid(nq * g.g3), block(rows_threads(LOGPC, true));
            if constexpr (regs_of<LOGPC>::ON) {
                auto k = rows_inv_regs_kernel<Tio, LOGPC>;
                allow_lds(k, g.v3.lds);
                launch_timed("fftk_rows_inv", timing, k, grid, block, g.v3.lds, s, (const double2*)Zw, O, j.ooff, ptab,
                             mdims, j.nl, q0, H, W, g.Ys, g.g3, scale, tw);
            } else {
                auto k = rows_inv_slab_kernel<Tio, LOGPC>;
                allow_lds(k, g.v3.lds);
                launch_timed("fftk_rows_inv", timing, k, grid, block, g.v3.lds, s, (const double2*)Zw, O, j.ooff, ptab,
                             mdims, j.nl, q0, H, W, g.Ys, g.v3.logT, g.g3, scale, tw);
            }
        });
    }
    XC_HIP(hipGetLastError());
    record_launch("fftk_rows_inv", dim3(g.g3),
                  dim3(g.f3 ? 3u * (uint32_t)rows3_t(g.logN) * (g.Pc / 3) / 8 : (uint32_t)rows_threads(g.logPc, true)),
                  g.v3.lds, H, W, j.pairs, 1);
}

size_t bytes_of(const fftk_ws_sizes& z) { return z.sr + z.sl + z.lh + z.z; }

template <typename Tio>
void run_fftk(const family_args& a, const Tio* L, const Tio* R, Tio* O, uint32_t max_chunk, bool pow2_rows,
              hipStream_t s) {
    fftk_job j{};
    j.max_chunk = max_chunk;
    j.pow2_rows = pow2_rows;
    j.H = a.rows;
    j.W = a.cols;
    j.nl = a.family == XC_ONE_TO_ONE || a.family == XC_ONE_TO_MANY ? 1 : a.n;
    j.nr = a.family == XC_ONE_TO_ONE ? 1 : a.m;
    j.pairs = a.pairs;
    j.family = a.family;
    j.n = a.n;
    j.m = a.m;
    // The faster layout where kFftkExtra lets it and its memory is there, the right spectra (the
    // bulk of it) last; else the plain one.
    const fftk_ws_sizes fast = fftk_sizes(j);
    j.plain = true;
    const fftk_ws_sizes plain = fftk_sizes(j);
    fftk_ws ws{};
    if (bytes_of(fast) <= bytes_of(plain) + kFftkExtra) {
        ws.z = workspace_if_free(WS_FK_Z, fast.z, s);
        ws.lh = ws.z ? workspace_if_free(WS_FK_LHAT, fast.lh, s) : nullptr;
        ws.sl = ws.lh ? workspace_if_free(WS_FK_SL, fast.sl, s) : nullptr;
        ws.sr = ws.sl ? workspace_if_free(WS_FK_SR, fast.sr, s) : nullptr;
        ws.zchunk = fast.chunk;
        j.plain = !ws.sr;
    }
    if (j.plain) {
        ws.sr = workspace(WS_FK_SR, plain.sr, s);
        ws.sl = workspace(WS_FK_SL, plain.sl, s);
        ws.lh = workspace(WS_FK_LHAT, plain.lh, s);
        ws.z = workspace(WS_FK_Z, plain.z, s);
        ws.zchunk = plain.chunk;
    }
    launch_job<Tio>(j, L, R, O, ws, s, true);
}

// ---- allocation-free entry point ---------------------------------------------------------
// The row spectra S, the left spectra Lhat and the column-pass results Z of
// xc_cross_corr_noalloc_f32 live in this array of the code object instead of allocated
// workspaces.  Every device that runs the library holds one copy for the process; calls on
// one device share it, so calls that overlap on one device race (each call overwrites what it
// reads before reading it, so nothing needs clearing between calls).
constexpr size_t kScratchBytes = size_t(256) << 20;
__device__ __attribute__((aligned(256))) char scratch[kScratchBytes];

// The current device's address of `scratch`, looked up on the first call on that device.
char* scratch_of_device() {
    static std::mutex mu;
    static std::vector<char*> ptrs;
    int dev = 0;
    XC_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lock(mu);
    if ((int)ptrs.size() <= dev) ptrs.resize(dev + 1, nullptr);
    if (!ptrs[dev]) {
        char* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(reinterpret_cast<void**>(&p), HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            fail(XC_ERR_HIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
        ptrs[dev] = p;
    }
    return ptrs[dev];
}

size_t align256(size_t x) { return (x + 255) & ~size_t(255); }

// One launch sequence of the allocation-free path: a regular family over a slice of the
// call's matrices (element offsets of its first left, right and result).
struct noalloc_part {
    int family;
    uint32_t n, m, pairs;  // lefts, rights, results of the part
    size_t loff, roff, ooff;
    uint32_t chunk;        // pairs per launch of the column / inverse-row kernels
};

// Scratch bytes of a part with nl left and nr right spectra and `chunk` pairs of Z.
size_t part_bytes(const fftk_geom& g, uint32_t nl, uint32_t nr, uint32_t chunk) {
    return align256(g.s_bytes * nr) + align256(g.sl_bytes * nl) + align256(g.col_bytes * nl) +
           align256(g.z_bytes * chunk);
}

// Splits a call into parts whose spectra fit the scratch array: the whole call if it fits,
// else groups of right matrices (one_to_many, n_to_mn: whole groups of n), of left matrices
// against every right (n_to_m), or of right matrices per left (n_to_m when the rights alone do
// not fit).  Each part's results are contiguous in the output.
std::vector<noalloc_part> plan_noalloc(const family_args& a, const fftk_geom& g) {
    const size_t B = kScratchBytes, hw = (size_t)a.rows * a.cols;
    const size_t out_elems = (size_t)(2 * a.rows - 1) * (2 * a.cols - 1);
    const size_t one_pair = part_bytes(g, 1, 1, 1);
    if (one_pair > B)
        fail(XC_ERR_UNSUPPORTED, "allocation-free entry point: one pair of " + std::to_string(a.rows) + " x " +
                                     std::to_string(a.cols) + " needs " + std::to_string(one_pair >> 20) +
                                     " MiB of scratch, above its " + std::to_string(kScratchBytes >> 20) + " MiB");
    std::vector<noalloc_part> parts;
    // Right matrices of `rights` consecutive results, with `nl` lefts, chunk = all pairs.
    auto fit_rights = [&](uint32_t nl, uint32_t unit, uint32_t most) -> uint32_t {
        uint32_t g_best = 0;
        for (uint32_t c = unit; c <= most; c += unit) {
            if (part_bytes(g, nl, c, c) > B) break;
            g_best = c;
        }
        return g_best;
    };
    switch (a.family) {
    case XC_ONE_TO_ONE:
        parts.push_back({XC_ONE_TO_ONE, 1, 1, 1, 0, 0, 0, 1});
        break;
    case XC_ONE_TO_MANY: {
        const uint32_t gr = fit_rights(1, 1, a.m);
        for (uint32_t r0 = 0; r0 < a.m; r0 += gr) {
            const uint32_t c = std::min(gr, a.m - r0);
            parts.push_back({XC_ONE_TO_MANY, 1, c, c, 0, r0 * hw, r0 * out_elems, c});
        }
        break;
    }
    case XC_N_TO_MN: {
        const uint32_t gr = fit_rights(a.n, a.n, a.m);
        if (gr == 0)
            fail(XC_ERR_UNSUPPORTED, "allocation-free entry point: the spectra of " + std::to_string(a.n) +
                                         " left matrices do not fit its scratch array");
        for (uint32_t r0 = 0; r0 < a.m; r0 += gr) {
            const uint32_t c = std::min(gr, a.m - r0);  // a multiple of n, as m is
            parts.push_back({XC_N_TO_MN, a.n, c, c, 0, r0 * hw, r0 * out_elems, c});
        }
        break;
    }
    default: {  // n_to_m
        uint32_t gl = 0;
        for (uint32_t c = 1; c <= a.n; ++c) {
            if (part_bytes(g, c, a.m, a.m) > B) break;
            gl = c;
        }
        if (gl > 0) {
            for (uint32_t l0 = 0; l0 < a.n; l0 += gl) {
                const uint32_t c = std::min(gl, a.n - l0);
                // as many pairs per launch as the rest of the array holds (at least m: gl fits them)
                const size_t rest = B - part_bytes(g, c, a.m, 0);
                uint32_t chunk = (uint32_t)std::min<size_t>((size_t)c * a.m, rest / g.z_bytes);
                while (chunk > a.m && part_bytes(g, c, a.m, chunk) > B) --chunk;
                parts.push_back({XC_N_TO_M, c, a.m, c * a.m, l0 * hw, 0, (size_t)l0 * a.m * out_elems, chunk});
            }
        } else {
            const uint32_t gr = fit_rights(1, 1, a.m);
            for (uint32_t l = 0; l < a.n; ++l)
                for (uint32_t r0 = 0; r0 < a.m; r0 += gr) {
                    const uint32_t c = std::min(gr, a.m - r0);
                    parts.push_back({XC_ONE_TO_MANY, 1, c, c, l * hw, r0 * hw, ((size_t)l * a.m + r0) * out_elems, c});
                }
        }
    }
    }
    return parts;
}

}  // namespace

void run_fftk_noalloc_f32(const family_args& a, const float* L, const float* R, float* O, hipStream_t s) {
    char* base = scratch_of_device();
    (void)tables_of_device();
    // The plain layout decides what fits and how a call is split; a call that fits whole in the
    // faster layout of the allocating calls takes that one.
    fftk_geom g = geom_of(a.rows, a.cols, false, true);
    std::vector<noalloc_part> parts = plan_noalloc(a, g);
    const bool one = a.family == XC_ONE_TO_ONE || a.family == XC_ONE_TO_MANY;
    const fftk_geom fast = geom_of(a.rows, a.cols);
    const bool whole = part_bytes(fast, one ? 1 : a.n, a.family == XC_ONE_TO_ONE ? 1 : a.m, a.pairs) <= kScratchBytes;
    if (whole) {
        g = fast;
        parts = {{a.family, one ? 1 : a.n, a.family == XC_ONE_TO_ONE ? 1 : a.m, a.pairs, 0, 0, 0, a.pairs}};
    }
    for (const noalloc_part& p : parts) {
        fftk_job j{};
        j.H = a.rows;
        j.W = a.cols;
        j.family = p.family;
        j.n = p.n;
        j.m = p.m;
        j.nl = p.family == XC_ONE_TO_ONE || p.family == XC_ONE_TO_MANY ? 1 : p.n;
        j.nr = p.m;
        j.pairs = p.pairs;
        j.plain = !whole;
        fftk_ws ws{};
        char* q = base;
        ws.sr = q;
        q += align256(g.s_bytes * j.nr);
        ws.sl = q;
        q += align256(g.sl_bytes * j.nl);
        ws.lh = q;
        q += align256(g.col_bytes * j.nl);
        ws.z = q;
        ws.zchunk = p.chunk;
        if ((size_t)(q - base) + align256(g.z_bytes * p.chunk) > kScratchBytes)
            fail(XC_ERR_INVALID_ARGUMENT, "allocation-free entry point: internal scratch plan out of bounds");
        launch_job<float>(j, L + p.loff, R + p.roff, O + p.ooff, ws, s, false);
    }
}

const double2* fftk_twiddles() { return twiddles(); }

uint32_t fftk_col_len(uint32_t rows) {
    uint32_t p = 16;
    while (p < 2 * rows - 1) p <<= 1;
    return p;
}

uint32_t fftk_row_len(uint32_t cols) {
    const uint32_t p = fftk_col_len(cols);
    for (uint32_t n = 16; n <= 512; n <<= 1)
        if (3 * n >= 2 * cols - 1) return 3 * n < p ? 3 * n : p;
    return p;
}

std::pair<uint32_t, uint32_t> fftk_class(uint32_t rows, uint32_t cols) {
    if (small_serves(rows, cols))
        return {1u << std::max(5, ilog2_ceil(2 * rows - 1)), 1u << std::max(5, ilog2_ceil(2 * cols - 1))};
    return {fftk_col_len(rows), fftk_row_len(cols)};
}

fftk_ws_sizes fftk_sizes(const fftk_job& j) {
    const fftk_geom g = geom_of(j.H, j.W, j.pow2_rows, j.plain);
    fftk_ws_sizes z{};
    // Z is processed in chunks of pairs of at most ~2 GiB.
    z.chunk = (uint32_t)std::max<size_t>(1, std::min<size_t>(j.pairs, (size_t(2) << 30) / std::max<size_t>(g.z_bytes, 1)));
    if (j.max_chunk) z.chunk = std::min(z.chunk, j.max_chunk);
    z.sr = std::max<size_t>(g.s_bytes * j.nr, 16);
    z.sl = std::max<size_t>(g.sl_bytes * j.nl, 16);
    z.lh = std::max<size_t>(g.col_bytes * j.nl, 16);
    z.z = std::max<size_t>(g.z_bytes * z.chunk, 16);
    return z;
}

void fftk_prepare() {
    (void)twiddles();
    (void)twiddles3();
}

void fftk_launch_f32(const fftk_job& j, const float* L, const float* R, float* O, const fftk_ws& ws, hipStream_t s) {
    launch_job<float>(j, L, R, O, ws, s, false);
}

void run_fftk_f32(const family_args& a, const float* L, const float* R, float* O, uint32_t max_chunk, bool pow2_rows,
                  hipStream_t s) {
    run_fftk<float>(a, L, R, O, max_chunk, pow2_rows, s);
}

void run_fftk_f64(const family_args& a, const double* L, const double* R, double* O, uint32_t max_chunk,
                  bool pow2_rows, hipStream_t s) {
    run_fftk<double>(a, L, R, O, max_chunk, pow2_rows, s);
}

}  // namespace xc
