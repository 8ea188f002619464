// Batched LongRange1d in matrix form by fast Fourier transforms: the product
// part[r] = K (un[r] - ub[r]) of fq_longrange.hpp with the circulant K, as one
// real cyclic convolution per replica, one workgroup each, in LDS. A product
// of an N-chain costs ~10 N log2 N operations instead of 2 N^2.
//
// The real sequence of length M is transformed as L = M / 2 complex points
// z_n = x_2n + i x_2n+1. M = N if N is a power of two (K is then the cyclic
// convolution itself), else the smallest power of two >= 2 N - 1 (K embedded
// in a larger circulant, x padded with zeros). The kernel is even, so its
// spectrum H is real and the product in the frequency domain only mixes the
// points k and L - k:
//   E = (Z_k + conj Z_L-k) / 2, O = (Z_k - conj Z_L-k) / 2i, w = exp(-2 pi i k / M)
//   Z'_k = (s E + d w O) + i (s O + d conj(w) E), s, d = (H_k +- H_L-k) / 2
// (the halves of X_k = E + w O, X_k+L = E - w O scaled by H_k, H_L-k).
//
// Forward: radix-8 passes (a last one of radix 2 or 4) from blocks of L down,
// in place, natural to digit-reversed order; the inverse runs the same passes
// backwards, so no reordering pass is needed. The first pass reads the slips
// from memory, the last forward one, the frequency product and the first
// inverse one stay in registers (a thread then holds 8 consecutive points,
// and reads their partners from LDS), the last one writes the result. 2 log8 L
// exchanges through LDS, padded by one point in 8 against bank conflicts.
//
// Measured: 256 x 8192 in 24.8 us (k_lr_gemm 506 us), bound by the latency of
// its eight exchanges and the twiddle reads, one workgroup per CU. Error of
// the forces against extended precision, root mean square over that of the
// forces (k_lr_gemm in parentheses): slips of N = 1000 / 3001 / 8192 scattered
// by 2: 8.7e-16 (9.2e-16) / 7.3e-16 (8.6e-16) / 2.9e-15 (2.9e-15); random
// walks: 1.3e-14 (1.7e-14) / 5.0e-14 (5.9e-14) / 1.2e-13 (1.3e-13).
#pragma once

#include "fq_resident.hpp"

namespace fq {

struct LrFft {
    const double* tw; // [L][2] exp(-2 pi i k / L)
    const double* sd; // [L][3] s, d Re w, d Im w of point k, divided by L
};

struct cplx {
    double re, im;
};

FQ_HD cplx operator+(cplx a, cplx b)
{
    return {a.re + b.re, a.im + b.im};
}

FQ_HD cplx operator-(cplx a, cplx b)
{
    return {a.re - b.re, a.im - b.im};
}

FQ_HD cplx cmul(cplx a, cplx b)
{
    return {__builtin_fma(-a.im, b.im, a.re * b.re), __builtin_fma(a.im, b.re, a.re * b.im)};
}

// multiplication by -i (forward) or i (inverse)
template <bool INV>
FQ_HD cplx rot(cplx a)
{
    return INV ? cplx{-a.im, a.re} : cplx{a.im, -a.re};
}

// DFTs of 2, 4 and 8 points in registers, natural order in and out
template <bool INV>
__device__ __forceinline__ void dft4(cplx& a, cplx& b, cplx& c, cplx& d)
{
    const cplx s0 = a + c, s1 = a - c, s2 = b + d, s3 = rot<INV>(b - d);
    a = s0 + s2;
    b = s1 + s3;
    c = s0 - s2;
    d = s1 - s3;
}

template <bool INV>
__device__ __forceinline__ void dft8(cplx (&x)[8])
{
    constexpr double h = 0.70710678118654752440;
    cplx a0 = x[0] + x[4], a1 = x[1] + x[5], a2 = x[2] + x[6], a3 = x[3] + x[7];
    cplx b0 = x[0] - x[4], b1 = x[1] - x[5], b2 = x[2] - x[6], b3 = x[3] - x[7];
    // b1 exp(-+ i pi / 4), b2 (-+ i), b3 exp(-+ 3 i pi / 4)
    const cplx r1 = rot<INV>(b1), r3 = rot<INV>(b3);
    b1 = {h * (b1.re + r1.re), h * (b1.im + r1.im)};
    b2 = rot<INV>(b2);
    b3 = {h * (r3.re - b3.re), h * (r3.im - b3.im)};
    dft4<INV>(a0, a1, a2, a3);
    dft4<INV>(b0, b1, b2, b3);
    x[0] = a0;
    x[1] = b0;
    x[2] = a1;
    x[3] = b1;
    x[4] = a2;
    x[5] = b2;
    x[6] = a3;
    x[7] = b3;
}

template <int LOGL>
struct LrFftPlan {
    static constexpr int L = 1 << LOGL;
    static constexpr int T = L / 8;           // threads: 8 points each
    static constexpr int P8 = LOGL / 3;       // passes of radix 8
    static constexpr int LAST = LOGL - 3 * P8; // log2 of the last pass's radix (0: none)
    static constexpr int LDS = L + L / 8;     // points with padding

    static FQ_HD int pad(int i)
    {
        return i + (i >> 3);
    }

    // frequency held at position q after the forward passes, and back
    static FQ_HD int freq(int q)
    {
        int k = 0;
#pragma unroll
        for (int p = 0; p < P8; ++p) {
            k |= ((q >> (LOGL - 3 * (p + 1))) & 7) << (3 * p);
        }
        return k | ((q & ((1 << LAST) - 1)) << (3 * P8));
    }
    static FQ_HD int pos(int k)
    {
        int q = 0;
#pragma unroll
        for (int p = 0; p < P8; ++p) {
            q |= ((k >> (3 * p)) & 7) << (LOGL - 3 * (p + 1));
        }
        return q | (k >> (3 * P8));
    }
};

template <int LOGL>
__global__ void __launch_bounds__(LrFftPlan<LOGL>::T) k_lr_fft(LrBuffers lb, LrFft f)
{
    using F = LrFftPlan<LOGL>;
    constexpr int L = F::L, T = F::T, P8 = F::P8, LAST = F::LAST;
    extern __shared__ double s_dyn[];
    cplx* const buf = (cplx*)s_dyn;
    const cplx* const tw = (const cplx*)f.tw;
    const int t = threadIdx.x;
    const int N = (int)lb.N;
    const double* const x = lb.un + (int64_t)blockIdx.x * N;
    double* const out = lb.part + (int64_t)blockIdx.x * N;
    const double ub = x[0];

    cplx z[8];
    // pass p works on blocks of B = L >> 3p, elements j + m B / 8 of the block
    auto place = [&](int p, int m) -> int {
        const int s = LOGL - 3 * (p + 1); // log2 of B / 8
        const int j = t & ((1 << s) - 1), blk = t >> s;
        return (blk << (s + 3)) + (m << s) + j;
    };
    auto twiddle = [&](int p, bool inv) {
        const int s = LOGL - 3 * (p + 1);
        const int j = t & ((1 << s) - 1);
#pragma unroll
        for (int m = 1; m < 8; ++m) {
            cplx w = tw[(j * m) << (3 * p)];
            if (inv) {
                w.im = -w.im;
            }
            z[m] = cmul(z[m], w);
        }
    };
    // the last pass (radix 2 or 4) on 8 consecutive points
    auto tail = [&](auto inv) {
        constexpr bool INV = decltype(inv)::value;
        if constexpr (LAST == 1) {
#pragma unroll
            for (int m = 0; m < 8; m += 2) {
                const cplx a = z[m] + z[m + 1], b = z[m] - z[m + 1];
                z[m] = a;
                z[m + 1] = b;
            }
        }
        else if constexpr (LAST == 2) {
            dft4<INV>(z[0], z[1], z[2], z[3]);
            dft4<INV>(z[4], z[5], z[6], z[7]);
        }
    };
    // without a last pass of its own the radix-8 passes end on consecutive points
    constexpr int REG = LAST == 0 ? P8 - 1 : P8; // first pass done on consecutive points

#pragma unroll
    for (int m = 0; m < 8; ++m) {
        const int n = 2 * (t + m * T);
        z[m].re = n < N ? x[n] - ub : 0.0;
        z[m].im = n + 1 < N ? x[n + 1] - ub : 0.0;
    }
    for (int p = 0; p < REG; ++p) {
        if (p > 0) {
            __syncthreads();
#pragma unroll
            for (int m = 0; m < 8; ++m) {
                z[m] = buf[F::pad(place(p, m))];
            }
        }
        dft8<false>(z);
        twiddle(p, false);
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            buf[F::pad(place(p, m))] = z[m];
        }
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < 8; ++m) {
        z[m] = buf[F::pad(8 * t + m)];
    }
    if constexpr (LAST == 0) {
        dft8<false>(z);
    }
    else {
        tail(std::false_type{});
    }
#pragma unroll
    for (int m = 0; m < 8; ++m) {
        buf[F::pad(8 * t + m)] = z[m];
    }
    __syncthreads();
    // frequency product
#pragma unroll
    for (int m = 0; m < 8; ++m) {
        const int k = F::freq(8 * t + m);
        const cplx c = buf[F::pad(F::pos((L - k) & (L - 1)))];
        const cplx E = {0.5 * (z[m].re + c.re), 0.5 * (z[m].im - c.im)};
        const cplx O = {0.5 * (z[m].im + c.im), 0.5 * (c.re - z[m].re)};
        const double s = f.sd[3 * k];
        const cplx dw = {f.sd[3 * k + 1], f.sd[3 * k + 2]};
        const cplx a = cmul(dw, O), b = cmul({dw.re, -dw.im}, E);
        const cplx Ey = {__builtin_fma(s, E.re, a.re), __builtin_fma(s, E.im, a.im)};
        const cplx Oy = {__builtin_fma(s, O.re, b.re), __builtin_fma(s, O.im, b.im)};
        z[m] = {Ey.re - Oy.im, Ey.im + Oy.re};
    }
    if constexpr (LAST == 0) {
        dft8<true>(z);
    }
    else {
        tail(std::true_type{});
    }
    __syncthreads(); // every partner was read
#pragma unroll
    for (int m = 0; m < 8; ++m) {
        buf[F::pad(8 * t + m)] = z[m];
    }
    for (int p = REG - 1; p >= 0; --p) {
        __syncthreads();
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            z[m] = buf[F::pad(place(p, m))];
        }
        twiddle(p, true);
        dft8<true>(z);
        if (p > 0) {
#pragma unroll
            for (int m = 0; m < 8; ++m) {
                buf[F::pad(place(p, m))] = z[m];
            }
        }
    }
#pragma unroll
    for (int m = 0; m < 8; ++m) {
        const int n = 2 * (t + m * T);
        if (n < N) {
            out[n] = z[m].re;
        }
        if (n + 1 < N) {
            out[n + 1] = z[m].im;
        }
    }
}

} // namespace fq
