// Register FFTs of the own-FFT method (FP64, 16..2048 points) and their LDS layout, shared by
// the three-pass kernels (xc_fftk.hip) and the one-block kernels (xc_fftk_small.hip).
#pragma once

#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include "xc_internal.hpp"

namespace xc {

// The current device's table of exp(-2 pi i j / 4096), j = 0..4095, and packed_roots (xc_fftk.hip).
const double2* fftk_twiddles();

namespace {

constexpr int kLogMaxP = 12;          // longest transform: 4096 (the twiddle table's length)
constexpr int kSlab = 1 << kLogMaxP;  // twiddle table entries
// Where the roots of length n = 2, 4 .. 2048 lie side by side behind the table.
constexpr int packed_roots(int n) { return kSlab + n; }

// LDS slot of element j of transform t (length P = 2^LOGP): one pad slot per 8 values, and a
// transform stride of 9P/8 + 1 slots, so that lanes touching the same j of consecutive
// transforms, or j = 8i, hit different banks.  With P a compile-time constant the pad and
// stride arithmetic folds into immediate LDS offsets.
template <int LOGP>
__device__ __forceinline__ int at(int t, int j) {
    constexpr int S = (1 << LOGP) + (1 << LOGP) / 8 + 1;
    return t * S + j + (j >> 3);
}

__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
    return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ double2 cconj(double2 a) { return make_double2(a.x, -a.y); }
__device__ __forceinline__ double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ double2 mul_mi(double2 a) { return make_double2(a.y, -a.x); }  // (-i) * a

// Bounds-checked buffer accesses relative to a wave-uniform base: `voff` bytes per lane plus a
// uniform `soff`; with `voff` past `bytes` (below 2^31: kOut always is) loads give zero and stores do
// nothing, so a condition costs one select of the offset instead of a branch and a cleared
// register.  Only `voff` may be what leaves the buffer: `soff` stays inside it by construction.
constexpr uint32_t kOut = 0x80000000u;
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_of(const void* base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, bytes, 0x00020000);
}
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ double2 buf_load(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
    const i32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)voff, (int)soff, 0);
    return __builtin_bit_cast(double2, v);
}
template <typename T>
__device__ __forceinline__ T buf_load_real(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
    if constexpr (sizeof(T) == 4)
        return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(r, (int)voff, (int)soff, 0));
    else
        return __builtin_bit_cast(T, (i32x2)__builtin_amdgcn_raw_buffer_load_b64(r, (int)voff, (int)soff, 0));
}
__device__ __forceinline__ void buf_store(double2 v, __amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(i32x4, v), r, (int)voff, (int)soff, 0);
}
__device__ __forceinline__ void buf_store(float v, __amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, v), r, (int)voff, (int)soff, 0);
}
__device__ __forceinline__ void buf_store(double v, __amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(i32x2, v), r, (int)voff, (int)soff, 0);
}

// In-register forward DFT of R points: X[k] = sum_j u[j] exp(-2 pi i jk / R).
__device__ __forceinline__ void dft2(double2& a, double2& b) {
    const double2 t = a;
    a = cadd(t, b);
    b = csub(t, b);
}
__device__ __forceinline__ void dft4(double2& u0, double2& u1, double2& u2, double2& u3) {
    const double2 t0 = cadd(u0, u2), t1 = csub(u0, u2), t2 = cadd(u1, u3), t3 = mul_mi(csub(u1, u3));
    u0 = cadd(t0, t2);
    u2 = csub(t0, t2);
    u1 = cadd(t1, t3);
    u3 = csub(t1, t3);
}
// The last two levels of an 8-point DFT from its first: t0, t1 = x0 +- x4, t2, t3 = x2 +- x6,
// s0, s1 = x1 +- x5, s2, s3 = x3 +- x7.  The rotations by odd eighths, c (p, q), go into the sums
// as FMAs: 36 instructions where rotating first took 40.
__device__ __forceinline__ void dft8_last(double2 t0, double2 t1, double2 t2, double2 t3, double2 s0, double2 s1,
                                          double2 s2, double2 s3, double2 (&u)[8]) {
    constexpr double c = 0.70710678118654752440;  // sqrt(1/2)
    const double2 e0 = cadd(t0, t2), e2 = csub(t0, t2), o0 = cadd(s0, s2), o2 = csub(s0, s2);
    const double2 e1 = make_double2(t1.x + t3.y, t1.y - t3.x), e3 = make_double2(t1.x - t3.y, t1.y + t3.x);
    const double2 o1 = make_double2(s1.x + s3.y, s1.y - s3.x), o3 = make_double2(s1.x - s3.y, s1.y + s3.x);
    u[0] = cadd(e0, o0);
    u[4] = csub(e0, o0);
    u[2] = make_double2(e2.x + o2.y, e2.y - o2.x);
    u[6] = make_double2(e2.x - o2.y, e2.y + o2.x);
    const double p1 = o1.x + o1.y, q1 = o1.y - o1.x, p3 = o3.y - o3.x, q3 = o3.x + o3.y;
    u[1] = make_double2(fma(c, p1, e1.x), fma(c, q1, e1.y));
    u[5] = make_double2(fma(-c, p1, e1.x), fma(-c, q1, e1.y));
    u[3] = make_double2(fma(c, p3, e3.x), fma(-c, q3, e3.y));
    u[7] = make_double2(fma(-c, p3, e3.x), fma(c, q3, e3.y));
}
// s = a + w b, d = a - w b = 2 a - s: 6 FMAs where product, sum and difference (X) take 8
// instructions; d has the rounding of s too.
template <bool X>
__device__ __forceinline__ void bfly(double2 a, double2 w, double2 b, double2& s, double2& d) {
    if constexpr (X) {
        const double2 p = cmul(w, b);
        d = csub(a, p);
        s = cadd(a, p);
        return;
    }
    s.x = fma(w.x, b.x, fma(-w.y, b.y, a.x));
    s.y = fma(w.x, b.y, fma(w.y, b.x, a.y));
    d.x = fma(2.0, a.x, -s.x);
    d.y = fma(2.0, a.y, -s.y);
}
template <int R>
__device__ __forceinline__ void dft(double2 (&u)[R]) {
    if constexpr (R == 2) {
        dft2(u[0], u[1]);
    } else if constexpr (R == 4) {
        dft4(u[0], u[1], u[2], u[3]);
    } else {
        static_assert(R == 8, "radix");
        const double2 t0 = cadd(u[0], u[4]), t1 = csub(u[0], u[4]), t2 = cadd(u[2], u[6]), t3 = csub(u[2], u[6]);
        const double2 s0 = cadd(u[1], u[5]), s1 = csub(u[1], u[5]), s2 = cadd(u[3], u[7]), s3 = csub(u[3], u[7]);
        dft8_last(t0, t1, t2, t3, s0, s1, s2, s3, u);
    }
}

// Barrier between the LDS phases of a wave-owned transform: every value a lane reads was
// written by its own wave, so ordering the wave's LDS accesses is enough.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// Transforms of up to 2048 points run in registers: P/8 threads hold one transform, 8 values
// each.  Up to 512 points a transform lives in one wave (BLOCK false: the wave holds 512/P of
// them); 1024 and 2048 points span two and four waves of the block.
template <int LOGP>
struct regs_of {
    static constexpr bool ON = LOGP <= 11;
    static constexpr bool BLOCK = LOGP > 9;
};
template <bool BLOCK>
__device__ __forceinline__ void regs_sync() {
    if constexpr (BLOCK)
        __syncthreads();
    else
        wave_sync();
}

// Passes of fft_regs: radix 8 (no twiddles), twiddled radix-8 passes, and for log2 P mod 3 = 1
// or 2 a last twiddled pass of radix 2 or 4.  The short radix stands last and not first because
// a twiddled radix-2 or 4 pass multiplies 4 or 6 of a thread's 8 values where a radix-8 pass
// multiplies 7 and forms 6 powers: per 8 points 92 FP64 instructions against 124 at 16 points,
// 196 against 232 at 128, 312 against 340 at 1024 (234 against 248 at 256).
//
// X (double data): more roots of a pass are the table's own.  Powers and rotations of a single root
// carry its rounding and their own: results of unsigned values of 64^2 were 4.0e-16 off in the 2-norm
// with one root per pass and are 2.0e-16 off with these (2.3e-16 with a short radix first and powers one
// by one); n_to_m 16 x 64 of 64^2 50 -> 60 us.  Float results round at 6e-8, where neither shows.
template <int LOGP, bool X = false>
struct regs_roots {
    static constexpr int REM = LOGP % 3;
    static constexpr int N8 = LOGP / 3 - 1;  // twiddled radix-8 passes
    static constexpr int N = N8 + (REM ? 1 : 0);
    double2 w[N];
    const double2* tw;  // X: the table
};
// A pass's further roots with X.  Radix 8: powers 2 to 4 of the root w; radix 2: the root at i + P/8 (w2);
// radix 4: that and w^2 (w3).  Read where the pass before ends, so that they are in flight during the
// exchange, whose registers are free: kept from the start of the kernel they spill, and w read here too
// is waited for (64 of 128^2 36.5 -> 39.7 us).  From the tables where a length's roots lie side by side: at the
// strides of the 4096-point table every lane's root is in a line of its own (50 x 27 of 191x61 609 us, 546 so).
struct pass_roots {
    double2 w2, w3, w4;
};
template <int LOGP, int LOGPP>
__device__ __forceinline__ pass_roots load_pass_roots(int i, const double2* __restrict__ tw) {
    asm volatile("" : "+v"(i));  // here, not hoisted
    pass_roots x;
    constexpr int PP = 1 << LOGPP, P = 1 << LOGP;
    if constexpr (LOGP - LOGPP >= 3) {
        const int e = i & (PP - 1);
        x.w2 = tw[packed_roots(4 * PP) + e];
        x.w4 = tw[packed_roots(2 * PP) + e];
        x.w3 = tw[packed_roots(8 * PP) + 3 * e];
    } else {
        x.w2 = tw[packed_roots(P) + P / 8 + i];
        if constexpr (LOGP - LOGPP == 2) x.w3 = tw[packed_roots(P / 2) + i];
    }
    return x;
}
// Whether kernels on data of type T take the roots X.
template <typename T>
constexpr bool exact_roots = sizeof(T) == 8;

// Pass roots at lane position i: w[j] = exp(-2 pi i k / (8p)), k = i mod p, p = 8^(j+1) for the
// twiddled radix-8 passes, exp(-2 pi i i / P) for a last radix-2 or 4 pass.  Kernels load them
// once, before their first transform: a table read inside a pass would wait on memory after
// every LDS exchange.
template <int LOGP, bool X = false>
__device__ __forceinline__ regs_roots<LOGP, X> load_roots(int i, const double2* __restrict__ tw) {
    using RR = regs_roots<LOGP, X>;
    RR rr;
#pragma unroll
    for (int j = 0; j < RR::N8; ++j) {
        const int logpp = 3 + 3 * j;
        rr.w[j] = tw[(i & ((1 << logpp) - 1)) << (kLogMaxP - logpp - 3)];
    }
    if constexpr (RR::REM != 0) rr.w[RR::N8] = tw[i << (kLogMaxP - LOGP)];
    if constexpr (X) rr.tw = tw;
    return rr;
}

__device__ __forceinline__ double2 csqr(double2 a) {
    return make_double2(a.x * a.x - a.y * a.y, (a.x + a.x) * a.y);
}
// a * exp(-2 pi i m / 8), m = 1, 2, 3
template <int M>
__device__ __forceinline__ double2 rot8(double2 a) {
    constexpr double c = 0.70710678118654752440;  // sqrt(1/2)
    if constexpr (M == 0) return a;
    else if constexpr (M == 1) return make_double2(c * (a.x + a.y), c * (a.y - a.x));
    else if constexpr (M == 2) return mul_mi(a);
    else return make_double2(c * (a.y - a.x), -c * (a.x + a.y));
}

// The first pass's DFT of 8 values whose upper four are zero (a zero-padded input): 36 FP64
// instructions against 52.
__device__ __forceinline__ void dft8_half(double2 (&u)[8]) {
    dft8_last(u[0], u[0], u[2], u[2], u[1], u[1], u[3], u[3], u);
}

// Swap of one register index bit with bit 5 (4) of the lane: a holds index 0, b index 1.
// v_permlane32_swap exchanges a's lanes 32..63 with b's lanes 0..31, v_permlane16_swap the odd
// rows of 16 lanes of a with the even rows of b.
template <int BIT>
__device__ __forceinline__ void lane_swap(double& a, double& b) {
    typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
    const u32x2 x = __builtin_bit_cast(u32x2, a), y = __builtin_bit_cast(u32x2, b);
    u32x2 p, q;
    if constexpr (BIT == 5) {
        const auto lo = __builtin_amdgcn_permlane32_swap(x[0], y[0], false, false);
        const auto hi = __builtin_amdgcn_permlane32_swap(x[1], y[1], false, false);
        p = u32x2{lo[0], hi[0]};
        q = u32x2{lo[1], hi[1]};
    } else {
        const auto lo = __builtin_amdgcn_permlane16_swap(x[0], y[0], false, false);
        const auto hi = __builtin_amdgcn_permlane16_swap(x[1], y[1], false, false);
        p = u32x2{lo[0], hi[0]};
        q = u32x2{lo[1], hi[1]};
    }
    a = __builtin_bit_cast(double, p);
    b = __builtin_bit_cast(double, q);
}
template <int BIT>
__device__ __forceinline__ void lane_swap(double2& a, double2& b) {
    lane_swap<BIT>(a.x, b.x);
    lane_swap<BIT>(a.y, b.y);
}

// The exchange before a short last pass (radix 2^REM, p = P / 2^REM): the pass before it leaves
// element (itop, r, k) -- itop the top REM bits of the lane position i, which lie in lane bits 5
// (and 4) (regs_pos) -- and the last pass wants the top three element bits in the register
// index: the low REM bits of r change places with itop.  16 (32) swap instructions instead of 8
// LDS writes and 8 reads of 16 bytes per lane, and no synchronisation.
template <int REM>
__device__ __forceinline__ void lane_exchange(double2 (&u)[8]) {
    double2 v[8];
    if constexpr (REM == 1) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            lane_swap<5>(u[2 * q], u[2 * q + 1]);
            v[q] = u[2 * q];
            v[q + 4] = u[2 * q + 1];
        }
    } else {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            lane_swap<5>(u[4 * h], u[4 * h + 2]);
            lane_swap<5>(u[4 * h + 1], u[4 * h + 3]);
            lane_swap<4>(u[4 * h], u[4 * h + 1]);
            lane_swap<4>(u[4 * h + 2], u[4 * h + 3]);
#pragma unroll
            for (int x = 0; x < 4; ++x) v[2 * x + h] = u[4 * h + x];
        }
    }
#pragma unroll
    for (int r = 0; r < 8; ++r) u[r] = v[r];
}

template <int LOGP, int LOGPP, bool X>
__device__ __forceinline__ void fft_regs_next(double2 (&u)[8], double2* wb, int tl, int i,
                                              const regs_roots<LOGP, X>& rr);

// Twiddled passes of fft_regs from p = 2^LOGPP on (u[r] = element i + Q r); the last one leaves
// its outputs i + (P/8) r in registers.
template <int LOGP, int LOGPP, bool X>
__device__ __forceinline__ void fft_regs_passes(double2 (&u)[8], double2* wb, int tl, int i,
                                                const regs_roots<LOGP, X>& rr, const pass_roots& x) {
    // The root passes through an empty asm so that its powers are formed here, in this pass:
    // otherwise the compiler hoists the power chains of every pass (and keeps them for a second
    // transform with the same roots), which costs tens of VGPRs.
    double2 w1 = rr.w[LOGPP / 3 - 1];
    asm volatile("" : "+v"(w1.x), "+v"(w1.y));
    if constexpr (LOGP - LOGPP == 1) {  // radix 2: butterfly i + Q m takes u[m], u[m + 4]
        const double2 wr = X ? x.w2 : rot8<1>(w1);
        bfly<X>(u[0], w1, u[4], u[0], u[4]);
        bfly<X>(u[1], wr, u[5], u[1], u[5]);
        bfly<X>(u[2], mul_mi(w1), u[6], u[2], u[6]);
        bfly<X>(u[3], X ? mul_mi(x.w2) : rot8<3>(w1), u[7], u[3], u[7]);
    } else if constexpr (LOGP - LOGPP == 2) {  // radix 4: butterfly i + Q m takes u[m + 2 r]
#pragma unroll
        for (int m = 0; m < 2; ++m) {
            const double2 wm = m ? (X ? x.w2 : rot8<1>(w1)) : w1;
            const double2 w2 = X ? (m ? mul_mi(x.w3) : x.w3) : csqr(wm);
            double2 t0, t1, t2, t3;
            bfly<X>(u[m], w2, u[m + 4], t0, t1);
            bfly<X>(cmul(u[m + 2], wm), cmul(w2, wm), u[m + 6], t2, t3);
            u[m] = cadd(t0, t2);
            u[m + 4] = csub(t0, t2);
            u[m + 2] = make_double2(t1.x + t3.y, t1.y - t3.x);
            u[m + 6] = make_double2(t1.x - t3.y, t1.y + t3.x);
        }
    } else {
        // The powers as a tree (squares take 3 instructions and the chain is 3 long, not 6); the
        // products of the upper four inputs go into the first level's sums (bfly): 93 FP64
        // instructions against 105.
        const double2 w2 = X ? x.w2 : csqr(w1), w3 = X ? x.w3 : cmul(w2, w1), w4 = X ? x.w4 : csqr(w2);
        double2 t0, t1, t2, t3, s0, s1, s2, s3;
        bfly<X>(u[0], w4, u[4], t0, t1);
        bfly<X>(cmul(u[1], w1), cmul(w4, w1), u[5], s0, s1);
        bfly<X>(cmul(u[2], w2), X ? cmul(w4, w2) : csqr(w3), u[6], t2, t3);
        bfly<X>(cmul(u[3], w3), cmul(w4, w3), u[7], s2, s3);
        dft8_last(t0, t1, t2, t3, s0, s1, s2, s3, u);
        regs_sync<regs_of<LOGP>::BLOCK>();
        if constexpr (LOGPP + 3 < LOGP) fft_regs_next<LOGP, LOGPP + 3>(u, wb, tl, i, rr);
    }
}

// From the outputs of the radix-8 pass before p = 2^LOGPP (element ((i - k) << 3) + k + r p/8 in
// u[r], k = i mod p/8) to the pass at p: a short last pass takes them by lane swaps, a radix-8
// one through LDS.
template <int LOGP, int LOGPP, bool X>
__device__ __forceinline__ void fft_regs_next(double2 (&u)[8], double2* wb, int tl, int i,
                                              const regs_roots<LOGP, X>& rr) {
    constexpr int Q = 1 << (LOGP - 3);
    pass_roots x;
    if constexpr (X) x = load_pass_roots<LOGP, LOGPP>(i, rr.tw);
    if constexpr (LOGP - LOGPP < 3) {
        lane_exchange<LOGP - LOGPP>(u);
    } else {
        constexpr int LOGK = LOGPP - 3;
        const int k = i & ((1 << LOGK) - 1);
#pragma unroll
        for (int r = 0; r < 8; ++r) wb[at<LOGP>(tl, ((i - k) << 3) + k + (r << LOGK))] = u[r];
        regs_sync<regs_of<LOGP>::BLOCK>();
        if constexpr (Q >= 8) {
            // at(tl, i + Q r) = at(tl, i) + r (Q + Q/8) when 8 divides Q: one address register
            // and constant offsets (the compiler does not split the shift of the sum by itself,
            // and keeps eight addresses live through both transforms otherwise).
            const int a = at<LOGP>(tl, i);
#pragma unroll
            for (int r = 0; r < 8; ++r) u[r] = wb[a + r * (Q + (Q >> 3))];
        } else {
#pragma unroll
            for (int r = 0; r < 8; ++r) u[r] = wb[at<LOGP>(tl, i + Q * r)];
        }
    }
    fft_regs_passes<LOGP, LOGPP>(u, wb, tl, i, rr, x);
}

// FFTs entered and left in registers, for P = 2^LOGP of 16..2048 points (regs_of).  Thread
// (tl, i) of the owning wave (up to 512 points) or block (1024, 2048) -- tl = id / Q,
// i = id mod Q, Q = P/8 -- holds elements i + Q s (s = 0..7) of its transform tl on entry, and
// the transform's outputs at the same positions on return.  The first pass (radix 8, butterfly
// i, no twiddles) reads registers only and the last pass writes registers only, so a kernel
// that moves those positions to and from HBM needs LDS only for the exchanges between passes
// of radix 8 (none for 16 and 32 points, one for 64..256, two for 512..2048).  HALF: the upper half of the
// input is zero (u[4..7] are not read), as in every zero-padded forward transform.  wb is the
// owner's first transform slot; transform tl lives at wb + at<LOGP>(tl, .).  rr holds the pass
// roots of this thread (load_roots<LOGP>(i, table)).  A block-owned transform synchronises the
// block: every thread of it must call.  (tl, i) are passed in (regs_pos) so that a kernel
// calling twice can keep the compiler from holding the first call's LDS addresses in registers
// for the second.
template <int LOGP, bool HALF = false, bool X>
__device__ __forceinline__ void fft_regs(double2 (&u)[8], double2* wb, const regs_roots<LOGP, X>& rr, int tl,
                                         int i) {
    static_assert(LOGP >= 4 && regs_of<LOGP>::ON, "register FFTs take 16..2048 points");
    if constexpr (HALF)
        dft8_half(u);
    else
        dft<8>(u);
    fft_regs_next<LOGP, 3>(u, wb, tl, i, rr);
}

// Position in the register FFTs of 2^LOGP points of thread `id` of a block: transform t, the
// first transform t0 of the owning wave (0 for block-owned transforms), and i within the
// transform.  The top log2 P mod 3 bits of i lie in the wave's lane bits 5 (and 4), for
// lane_exchange; the bits below run over neighbouring lanes, 8 at least from 64 points on, so
// that loads and stores of consecutive elements move whole 128-byte lines.
template <int LOGP>
struct regs_pos {
    int t0, t, i;
    __device__ __forceinline__ explicit regs_pos(int id) {
        constexpr int REM = LOGP % 3;
        const int lane = id & 63, itop = lane >> (6 - REM);
        if constexpr (regs_of<LOGP>::BLOCK) {
            constexpr int LL = 6 - REM;  // lane bits below itop; the wave's bits follow
            t0 = 0;
            t = id >> (LOGP - 3);
            const int wave = (id >> 6) & ((1 << (LOGP - 9)) - 1);
            i = (itop << (LOGP - 3 - REM)) | (wave << LL) | (lane & ((1 << LL) - 1));
        } else {
            constexpr int LL = LOGP - 3 - REM;  // low bits of i; the transform's bits follow
            t0 = (id >> 6) << (9 - LOGP);
            t = t0 + ((lane >> LL) & ((1 << (9 - LOGP)) - 1));
            i = (itop << LL) | (lane & ((1 << LL) - 1));
        }
    }
};

// Launch, with the kernel's own start and end recorded under `name` while kernel timing is on.
template <typename K, typename... Args>
void launch_timed(const char* name, bool timing, K kernel, dim3 grid, dim3 block, uint32_t lds, hipStream_t s,
                  Args... args) {
    if (timing && timing_enabled()) {
        hipEvent_t a = nullptr, b = nullptr;
        timing_launch_events(name, &a, &b);
        hipExtLaunchKernelGGL(kernel, grid, block, lds, s, a, b, 0, args...);
    } else {
        hipLaunchKernelGGL(kernel, grid, block, lds, s, args...);
    }
}

}  // namespace
}  // namespace xc
