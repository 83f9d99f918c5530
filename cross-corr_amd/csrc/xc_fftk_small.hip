// Own-FFT method for small matrices: a pair's whole padded half spectrum in one block's LDS.
//
// The three-pass kernels (xc_fftk.hip) move the row spectra S and the column results Z of every
// pair through memory, in four launches, and transform a right's columns once per pair.  Where
// Pr * Pc <= 16384 (64 x 64 matrices and smaller, or longer and narrower ones) both exchanges
// between row and column transforms fit the 160 KB LDS of a CU, so two launches do the work:
//
//   small_spec  : one block per matrix: row FFTs, split and column FFTs in LDS; the 2D half
//                 spectrum F[mat][k][rho] (k = 0..Pc/2) is all that is written;
//   small_pairs : one block per pair: conj(F_left) * F_right, column FFTs, row FFTs, the cropped
//                 result straight from registers.
//
// A pair (or matrix) takes Pr * Pc / 16 threads of 8 values each: Pc/2 column transforms of
// Pr/8 threads, then Pr/2 row transforms (two result rows each) of Pc/8 threads.  Columns 0 and
// Pc/2 of the product have Hermitian spectra (their inverses are real), so they share one
// transform and the Pc/2 + 1 columns fill the block exactly.  The two rows of a row transform
// are rho and rho + Pr/2: a column thread holds both after its FFT (elements i + Q r and
// i + Q (r + 4)), so the Hermitian extension needs no exchange between lanes.
//
// Bound: FP64 VALU and LDS inside the block, then the spectra from L2.  Against the three passes
// (one call, float): n_to_m 16 x 64 of 64^2 77.9 -> 42.5 us, of 32^2 36 -> 16, 1 x 64 of 10^2 20.3 ->
// 13.9, 1 x 256 of 40^2 38.4 -> 32.0 (there with 96-point rows).
//
// small_pairs with one column per thread loads, transforms and stores in turn: at 128 x 128 points
// its 1024-thread block fills the CU's LDS, and nothing runs while it waits for the spectra.  With
// two columns per thread (the second column's transform after the first, in the same scratch) and
// the rows in two passes through half the slots, a pair takes half the threads and LDS, and the
// blocks that share a CU overlap each other's phases.  It is taken for more pairs than the chip
// holds at once in the other form: 16 x 64 of 64^2 53.8 -> 42.5 us, 32 x 128 201 -> 136; of 60 x 30
// 28.8 -> 26.3 and 78 -> 65.5; of 30^2 17.4 -> 16.4 and 39.8 -> 34.3.  Fewer pairs, where a pair's
// own latency counts, are 0.5 us faster to 2 us slower that way (one pair of 60 x 30 12.1 -> 14.0).
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "xc_fftk_core.hpp"
#include "xc_methods.hpp"

namespace xc {
namespace {

// Geometry of a padded size Pr x Pc = 2^LR x 2^LC.
template <int LR, int LC>
struct small_geom {
    static constexpr int Pr = 1 << LR, Pc = 1 << LC, Qr = Pr / 8, Qc = Pc / 8;
    static constexpr int NC = Pc / 2, NR = Pr / 2;  // column and row transforms
    static constexpr int NT = Pr * Pc / 16;         // threads: a wave at least
    static constexpr int SR = Pr + Pr / 8 + 1, SC = Pc + Pc / 8 + 1;  // strides of `at`
    static constexpr int SLOTS = NC * SR > NR * SC ? NC * SR : NR * SC;
    static constexpr uint32_t LDS = (uint32_t)(SLOTS * (int)sizeof(double2));
    static_assert(NT >= 64 && NT <= 1024 && LR >= 5 && LC >= 5 && LR <= 9 && LC <= 9, "one block per pair");
};

// small_pairs with PS columns per thread and PS passes of rows: threads and LDS of a block.
template <int LR, int LC, int PS>
struct pairs_geom : small_geom<LR, LC> {
    using G = small_geom<LR, LC>;
    static constexpr int NT = G::NT / PS;
    static constexpr uint32_t LDS = G::LDS / PS;
};

// Matrices 0..nl-1 are the left ones (XL into FL), the rest the right ones (XR into FR); moff and
// mdims as in rows_fwd_regs_kernel.
template <typename Tin, int LR, int LC>
__global__ __launch_bounds__((small_geom<LR, LC>::NT)) void small_spec_kernel(
    const Tin* __restrict__ XL, const Tin* __restrict__ XR, const uint64_t* __restrict__ moff,
    const uint2* __restrict__ mdims, uint32_t nl, uint32_t H, uint32_t W, double2* __restrict__ FL,
    double2* __restrict__ FR, const double2* __restrict__ tw) {
    using G = small_geom<LR, LC>;
    extern __shared__ double2 buf[];
    const int tp = (int)threadIdx.x;
    const uint32_t matg = blockIdx.x;
    const bool left = matg < nl;
    const uint32_t mat = left ? matg : matg - nl;
    const Tin* X = (left ? XL : XR) + (moff ? moff[matg] : (size_t)mat * H * W);
    if (mdims) {
        const uint2 d = mdims[matg];
        H = d.x;
        W = d.y;
    }
    const regs_pos<LR> pc(tp);
    const auto rrc = load_roots<LR, exact_roots<Tin>>(pc.i, tw);
    // Rows rho and rho + Pr/4 in one transform (H <= Pr/2): Pr/4 of them, on half the threads.
    if (G::NT < 128 || tp < G::NT / 2) {
        const regs_pos<LC> pr(tp);
        const auto rr = load_roots<LC, exact_roots<Tin>>(pr.i, tw);
        const uint32_t a = pr.t, b = a + G::Pr / 4;
        const bool oka = a < H && pr.t < G::Pr / 4, okb = b < H && pr.t < G::Pr / 4;
        const Tin* xa = X + (oka ? (size_t)a * W : 0);
        const Tin* xb = X + (okb ? (size_t)b * W : 0);
        double2 u[8];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint32_t c = pr.i + G::Qc * r, cc = c < W ? c : W - 1;
            const Tin va = xa[cc], vb = xb[cc];
            u[r] = make_double2(oka && c < W ? (double)va : 0.0, okb && c < W ? (double)vb : 0.0);
        }
        fft_regs<LC, true>(u, buf + at<LC>(pr.t0, 0), rr, pr.t - pr.t0, pr.i);
#pragma unroll
        for (int r = 0; r < 8; ++r) buf[at<LC>(pr.t, pr.i + G::Qc * r)] = u[r];
    }
    __syncthreads();
    // Column k = t: rows i, i + Qr from the A parts, the rows Pr/4 above from the B parts of the
    // split; k = 0 takes column 0 + i * column Pc/2 (both real).
    const int k = pc.t, i = pc.i;
    double2 u[8];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        const int rho = i + G::Qr * s;
        const double2 zk = buf[at<LC>(rho, k)];
        const double2 zp = buf[at<LC>(rho, k == 0 ? G::Pc / 2 : G::Pc - k)];
        const double2 zn = cconj(zp), d = mul_mi(csub(zk, zn));
        u[s] = k == 0 ? make_double2(zk.x, zp.x) : make_double2(0.5 * (zk.x + zn.x), 0.5 * (zk.y + zn.y));
        u[s + 2] = k == 0 ? make_double2(zk.y, zp.y) : make_double2(0.5 * d.x, 0.5 * d.y);
    }
    __syncthreads();  // the column transforms use the rows' slots
    fft_regs<LR, true>(u, buf + at<LR>(pc.t0, 0), rrc, pc.t - pc.t0, i);
    double2* F = (left ? FL : FR) + ((size_t)mat * (G::NC + 1) + k) * G::Pr + i;
    if (tp < 64) {  // the wave of column 0: X0 = (Y + conj(Y-)) / 2, X_Pc/2 = (Y - conj(Y-)) / 2i
#pragma unroll
        for (int r = 0; r < 8; ++r) buf[at<LR>(pc.t, i + G::Qr * r)] = u[r];
        wave_sync();
        if (k == 0) {
#pragma unroll
            for (int r = 0; r < 8; ++r) {
                const double2 y = cconj(buf[at<LR>(pc.t, (G::Pr - (i + G::Qr * r)) & (G::Pr - 1))]);
                const double2 d = mul_mi(csub(u[r], y));
                F[(size_t)G::NC * G::Pr + G::Qr * r] = make_double2(0.5 * d.x, 0.5 * d.y);
                u[r] = make_double2(0.5 * (u[r].x + y.x), 0.5 * (u[r].y + y.y));
            }
        }
    }
#pragma unroll
    for (int r = 0; r < 8; ++r) F[G::Qr * r] = u[r];
}

// Pairs q0 .. q0 + gridDim.x - 1 of the job in this order: the pairs of one right are consecutive
// for n_to_m (an XCD's share of the pairs then reads few rights with all lefts, which its L2
// holds), else the family's own order.
template <typename Tout, int LR, int LC, int PS>
__global__ __launch_bounds__((pairs_geom<LR, LC, PS>::NT), 4) void small_pairs_kernel(
    const double2* __restrict__ FL, const double2* __restrict__ FR, Tout* __restrict__ O,
    const uint64_t* __restrict__ ooff, const uint2* __restrict__ ptab, const uint2* __restrict__ mdims, uint32_t nl,
    int family, uint32_t n, uint32_t m, uint32_t q0, uint32_t H, uint32_t W, double scale,
    const double2* __restrict__ tw) {
    using G = pairs_geom<LR, LC, PS>;
    extern __shared__ double2 buf[];
    const int tp = (int)threadIdx.x;
    uint32_t q = q0 + xcd_remap(blockIdx.x, gridDim.x), l, r;
    if (ptab) {
        l = ptab[q].x;
        r = ptab[q].y;
    } else if (family == XC_N_TO_M) {
        r = q / n;
        l = q - r * n;
        q = l * m + r;
    } else {
        pair_of(family, n, m, q, l, r);
    }
    if (mdims) {
        const uint2 d = mdims[nl + r];
        H = d.x;
        W = d.y;
    }
    // Columns pc.t + h NC/PS: the products' transforms, combined to the row transforms' inputs.
    const regs_pos<LR> pc(tp);
    const int i = pc.i;
    const bool wave0 = tp < 64;  // holds column 0 (selects in every wave cost 60 instructions)
    double2 u[PS][8];
    {
        const auto rr = load_roots<LR, exact_roots<Tout>>(i, tw);
        const size_t nyq = (size_t)G::NC * G::Pr;
#pragma unroll
        for (int h = 0; h < PS; ++h) {
            const int k = pc.t + h * (G::NC / PS);
            const size_t col = (size_t)k * G::Pr + i;
            const double2* Lf = FL + (size_t)l * (G::NC + 1) * G::Pr + col;
            const double2* Rf = FR + (size_t)r * (G::NC + 1) * G::Pr + col;
            double2 v[8];
#pragma unroll
            for (int s = 0; s < 8; ++s) {
                u[h][s] = Rf[G::Qr * s];
                v[s] = Lf[G::Qr * s];
            }
#pragma unroll
            for (int s = 0; s < 8; ++s) u[h][s] = cmul(cconj(v[s]), u[h][s]);
            if (h == 0 && wave0 && k == 0) {
#pragma unroll
                for (int s = 0; s < 8; ++s) {
                    const double2 g = cmul(cconj(Lf[nyq + G::Qr * s]), Rf[nyq + G::Qr * s]);
                    u[h][s] = make_double2(u[h][s].x - g.y, u[h][s].y + g.x);
                }
            }
            fft_regs<LR>(u[h], buf + at<LR>(pc.t0, 0), rr, pc.t - pc.t0, i);
            // conj(Y) of row transform rho: with a, b the conjugated column results at rho and
            // rho + Pr/2, a - i b at k and conj(a) - i conj(b) at Pc - k; column 0 carries the two
            // real columns 0 and Pc/2.
            if (h == 0 && wave0 && pc.t == 0) {
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    const double2 a = u[h][s], b = u[h][s + 4];
                    u[h][s] = make_double2(a.x, -b.x);
                    u[h][s + 4] = make_double2(a.y, -b.y);
                }
            } else {
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    const double2 a = u[h][s], b = u[h][s + 4];
                    u[h][s] = make_double2(a.x + b.y, a.y - b.x);
                    u[h][s + 4] = make_double2(a.x - b.y, -a.y - b.x);
                }
            }
        }
    }
    const regs_pos<LC> pr(tp);
    const auto rr = load_roots<LC, exact_roots<Tout>>(pr.i, tw);
    const int SX = 2 * (int)W - 1;
    Tout* Oq = O + (ooff ? ooff[q] : (size_t)q * (2 * H - 1) * SX);
    const int wlo = (int)W - 1, whi = -(G::Pc - (int)W + 1);
    // Row transforms rho = pass NR/PS + pr.t.
#pragma unroll
    for (int pass = 0; pass < PS; ++pass) {
        __syncthreads();  // the rows' slots overlap the columns' scratch, or the last pass's rows
#pragma unroll
        for (int h = 0; h < PS; ++h) {
            const int k = pc.t + h * (G::NC / PS);
            double2* y0 = buf + at<LC>(i, k);
            double2* y1 = buf + at<LC>(i, h == 0 && wave0 && k == 0 ? G::Pc / 2 : G::Pc - k);
#pragma unroll
            for (int s = 0; s < 4 / PS; ++s) {
                y0[s * G::Qr * G::SC] = u[h][pass * (4 / PS) + s];
                y1[s * G::Qr * G::SC] = u[h][pass * (4 / PS) + s + 4];
            }
        }
        __syncthreads();
        double2 w[8];
#pragma unroll
        for (int s = 0; s < 8; ++s) w[s] = buf[at<LC>(pr.t, pr.i + G::Qc * s)];
        wave_sync();
        fft_regs<LC>(w, buf + at<LC>(pr.t0, 0), rr, pr.t - pr.t0, pr.i);
        // Circular row rho (shifts 0..H-1) and rho + Pr/2 (shifts -(H-1)..-1 are rows > Pr - H);
        // circular columns i + Qc s likewise, s < 4 and s >= 4 (H <= Pr/2, W <= Pc/2).
        const int rho = pr.t + pass * (G::NR / PS);
        const bool oka = rho < (int)H, okb = rho + G::Pr / 2 > G::Pr - (int)H;
        Tout* oa = Oq + (rho + (int)H - 1) * SX + pr.i;
        Tout* ob = Oq + (rho - (G::Pr / 2 - (int)H + 1)) * SX + pr.i;
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            const int c = pr.i + G::Qc * s, off = G::Qc * s + (s < 4 ? wlo : whi);
            const bool in = s < 4 ? c < (int)W : c > G::Pc - (int)W;
            if (in && oka) oa[off] = (Tout)(w[s].x * scale);
            if (in && okb) ob[off] = (Tout)(-w[s].y * scale);
        }
    }
}

// Calls f(LR, LC) with the padded lengths as integral constants.
template <typename F>
void with_small(int lr, int lc, F&& f) {
    auto outer = [&](auto LR) {
        auto inner = [&](auto LC) {
            if constexpr (decltype(LR)::value + decltype(LC)::value <= kSmallLog) f(LR, LC);
        };
        switch (lc) {
        case 5: inner(std::integral_constant<int, 5>{}); break;
        case 6: inner(std::integral_constant<int, 6>{}); break;
        case 7: inner(std::integral_constant<int, 7>{}); break;
        case 8: inner(std::integral_constant<int, 8>{}); break;
        case 9: inner(std::integral_constant<int, 9>{}); break;
        }
    };
    switch (lr) {
    case 5: outer(std::integral_constant<int, 5>{}); break;
    case 6: outer(std::integral_constant<int, 6>{}); break;
    case 7: outer(std::integral_constant<int, 7>{}); break;
    case 8: outer(std::integral_constant<int, 8>{}); break;
    case 9: outer(std::integral_constant<int, 9>{}); break;
    }
}

template <typename K>
void allow_lds(K kernel, uint32_t bytes) {
    if (bytes > 65536) allow_dynamic_lds(reinterpret_cast<const void*>(kernel), bytes);
}

template <typename Tio>
void launch_small(const fftk_job& j, int lr, int lc, const Tio* L, const Tio* R, Tio* O, const fftk_ws& ws,
                  hipStream_t s, bool timing) {
    if (!fftk_small_fits(lr, lc)) fail(XC_ERR_UNSUPPORTED, "own-FFT method: inconsistent small geometry");
    const double2* tw = fftk_twiddles();
    double2* FL = static_cast<double2*>(ws.lh);
    double2* FR = static_cast<double2*>(ws.sr);
    const uint2* ptab = reinterpret_cast<const uint2*>(j.ptab);
    const uint2* mdims = reinterpret_cast<const uint2*>(j.mdims);
    with_small(lr, lc, [&](auto LR, auto LC) {
        using G = small_geom<decltype(LR)::value, decltype(LC)::value>;
        auto ks = small_spec_kernel<Tio, decltype(LR)::value, decltype(LC)::value>;
        allow_lds(ks, G::LDS);
        launch_timed("fftk_small_spec", timing, ks, dim3(j.nl + j.nr), dim3(G::NT), G::LDS, s, L, R, j.moff, mdims,
                     j.nl, j.H, j.W, FL, FR, tw);
        auto pairs = [&](auto PS) {
            using P = pairs_geom<decltype(LR)::value, decltype(LC)::value, decltype(PS)::value>;
            auto kp = small_pairs_kernel<Tio, decltype(LR)::value, decltype(LC)::value, decltype(PS)::value>;
            allow_lds(kp, P::LDS);
            // one launch holds fewer than 2^32 threads (67 M pairs of up to 16 x 16)
            constexpr uint32_t kMost = 0xffffffffu / P::NT;
            for (uint32_t q0 = 0; q0 < j.pairs; q0 += std::min(kMost, j.pairs - q0))
                launch_timed("fftk_small_pairs", timing, kp, dim3(std::min(kMost, j.pairs - q0)), dim3(P::NT), P::LDS,
                             s, (const double2*)FL, (const double2*)FR, O, j.ooff, ptab, mdims, j.nl, j.family, j.n,
                             j.m, q0, j.H, j.W, 1.0 / ((double)G::Pr * (double)G::Pc), tw);
            record_launch("fftk_small_pairs", dim3(std::min(kMost, j.pairs)), dim3(P::NT), P::LDS, j.H, j.W, j.pairs,
                          1);
        };
        if constexpr (G::NT >= 128) {
            // More pairs than the 256 CUs hold at once with one column per thread (1024 threads each).
            if (j.pairs > 256 * 1024 / G::NT)
                pairs(std::integral_constant<int, 2>{});
            else
                pairs(std::integral_constant<int, 1>{});
        } else {
            pairs(std::integral_constant<int, 1>{});
        }
        XC_HIP(hipGetLastError());
    });
}

}  // namespace

bool fftk_small_fits(int lr, int lc) { return lr >= 5 && lc >= 5 && lr <= 9 && lc <= 9 && lr + lc <= kSmallLog; }

void fftk_small_f32(const fftk_job& j, int lr, int lc, const float* L, const float* R, float* O, const fftk_ws& ws,
                    hipStream_t s, bool timing) {
    launch_small<float>(j, lr, lc, L, R, O, ws, s, timing);
}
void fftk_small_f64(const fftk_job& j, int lr, int lc, const double* L, const double* R, double* O, const fftk_ws& ws,
                    hipStream_t s, bool timing) {
    launch_small<double>(j, lr, lc, L, R, O, ws, s, timing);
}

}  // namespace xc
