// Device-side building blocks of the gfx950 FFT kernels: complex arithmetic, compile-time DFT
// constants, radix-R butterflies, fast integer division, and the LDS-resident Stockham engine that
// every transform kernel is built from.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>
#include <utility>

namespace kfr_amd
{

template <typename T>
struct alignas(2 * sizeof(T)) cx
{
    T re, im;
};

template <typename T>
__device__ __forceinline__ cx<T> cadd(cx<T> a, cx<T> b)
{
    return { a.re + b.re, a.im + b.im };
}
template <typename T>
__device__ __forceinline__ cx<T> csub(cx<T> a, cx<T> b)
{
    return { a.re - b.re, a.im - b.im };
}
template <typename T>
__device__ __forceinline__ cx<T> cmul(cx<T> a, cx<T> b)
{
    return { a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re };
}
// a * conj(b)
template <typename T>
__device__ __forceinline__ cx<T> cmulc(cx<T> a, cx<T> b)
{
    return { a.re * b.re + a.im * b.im, a.im * b.re - a.re * b.im };
}
// multiply by a forward twiddle (INV = false) or by its conjugate (INV = true)
template <bool INV, typename T>
__device__ __forceinline__ cx<T> ctw(cx<T> a, cx<T> w)
{
    if constexpr (INV)
        return cmulc(a, w);
    else
        return cmul(a, w);
}
template <typename T>
__device__ __forceinline__ cx<T> cscale(cx<T> a, T s)
{
    return { a.re * s, a.im * s };
}
template <typename T>
__device__ __forceinline__ cx<T> cconj(cx<T> a)
{
    return { a.re, -a.im };
}
// multiply by -i (forward) or +i (inverse)
template <bool INV, typename T>
__device__ __forceinline__ cx<T> cmul_mi(cx<T> a)
{
    if constexpr (INV)
        return { -a.im, a.re };
    else
        return { a.im, -a.re };
}

// ---------------------------------------------------------------------------------------------
// Compile-time cos/sin of 2*pi*k/n for the constant twiddles inside butterflies, rounded from a sum of two
// doubles: the angle is reduced to the first eighth of a turn in whole numbers, pi and the Taylor series
// carry about 100 bits (two_sum, two_product and their quotient, Dekker 1971). Plain double series are off by up
// to 4 units in the last place, which a 9-point butterfly's error shows (FP64, 9 points: 2.2e-16 against
// 1.6e-16 with rounded constants).
struct two_double
{
    double hi, lo;
};
constexpr two_double two_sum(double a, double b)
{
    const double s = a + b, t = s - a;
    return { s, (a - (s - t)) + (b - t) };
}
constexpr two_double two_product(double a, double b)
{
    constexpr double split = 134217729.0; // 2^27 + 1
    const double p = a * b, ca = split * a, cb = split * b;
    const double ah = ca - (ca - a), al = a - ah, bh = cb - (cb - b), bl = b - bh;
    return { p, ((ah * bh - p) + ah * bl + al * bh) + al * bl };
}
constexpr two_double dd_add(two_double a, two_double b)
{
    const two_double s = two_sum(a.hi, b.hi);
    return two_sum(s.hi, s.lo + (a.lo + b.lo));
}
constexpr two_double dd_mul(two_double a, two_double b)
{
    const two_double p = two_product(a.hi, b.hi);
    return two_sum(p.hi, p.lo + (a.hi * b.lo + a.lo * b.hi));
}
constexpr two_double dd_div(two_double a, double b)
{
    const double q = a.hi / b;
    const two_double p = two_product(q, b);
    return two_sum(q, (((a.hi - p.hi) - p.lo) + a.lo) / b);
}
// sin (odd = true) or cos of 2*pi*k/n, 0 <= 8k <= n
constexpr double taylor_2pi(long k, long n, bool odd)
{
    constexpr two_double pi = { 3.141592653589793116, 1.2246467991473532e-16 };
    const two_double x  = dd_div(dd_mul(pi, { double(2 * k), 0.0 }), double(n));
    const two_double x2 = dd_mul(x, x);
    two_double term     = odd ? x : two_double{ 1.0, 0.0 };
    two_double sum      = term;
    for (int i = odd ? 2 : 1; i < 28; i += 2)
    {
        term = dd_div(dd_mul(term, { -x2.hi, -x2.lo }), double(i * (i + 1)));
        sum  = dd_add(sum, term);
    }
    return sum.hi;
}
// cos(2*pi*k/n)
constexpr double ccos2pi(long k, long n)
{
    k %= n;
    if (k < 0)
        k += n;
    if (2 * k > n)
        k = n - k; // cos is even
    // quarter and eighth turns in units of 1/4n and 1/8n: every reduction is exact
    if (4 * k > n)
        return 8 * k > 3 * n ? -taylor_2pi(n - 2 * k, 2 * n, false) : -taylor_2pi(4 * k - n, 4 * n, true);
    return 8 * k > n ? taylor_2pi(n - 4 * k, 4 * n, true) : taylor_2pi(k, n, false);
}
// sin(2*pi*k/n) = cos(2*pi*(4k - n)/4n)
constexpr double csin2pi(long k, long n) { return ccos2pi(4 * (k % n) - n, 4 * n); }

// ---------------------------------------------------------------------------------------------
// Butterflies: in-place DFT of R points, X[k] = sum_n x[n] exp(-+2*pi*i*n*k/R)
// (minus sign for the forward transform, plus for the inverse). No scaling.

template <bool INV, typename T>
__device__ __forceinline__ void bfly2(cx<T>& a, cx<T>& b)
{
    cx<T> t = a;
    a       = cadd(t, b);
    b       = csub(t, b);
}

template <bool INV, typename T>
__device__ __forceinline__ void bfly4(cx<T>& a0, cx<T>& a1, cx<T>& a2, cx<T>& a3)
{
    cx<T> t0 = cadd(a0, a2), t1 = csub(a0, a2);
    cx<T> t2 = cadd(a1, a3), t3 = cmul_mi<INV>(csub(a1, a3));
    a0       = cadd(t0, t2);
    a2       = csub(t0, t2);
    a1       = cadd(t1, t3);
    a3       = csub(t1, t3);
}

// multiply by exp(-+2*pi*i*k/n) with compile-time k, n
template <bool INV, long K, long N, typename T>
__device__ __forceinline__ cx<T> twc(cx<T> a)
{
    constexpr long k = ((K % N) + N) % N;
    if constexpr (k == 0)
        return a;
    else if constexpr (4 * k == N)
        return cmul_mi<INV>(a);
    else if constexpr (2 * k == N)
        return { -a.re, -a.im };
    else if constexpr (4 * k == 3 * N)
        return cmul_mi<!INV>(a);
    else
    {
        constexpr T c = T(ccos2pi(k, N));
        constexpr T s = INV ? T(csin2pi(k, N)) : T(-csin2pi(k, N));
        return { a.re * c - a.im * s, a.re * s + a.im * c };
    }
}

template <bool INV, typename T>
__device__ __forceinline__ void bfly8(cx<T>* v)
{
    // radix-2 x radix-4: 4-point DFTs over even/odd, combined with W8 twiddles
    bfly4<INV>(v[0], v[2], v[4], v[6]);
    bfly4<INV>(v[1], v[3], v[5], v[7]);
    v[3] = twc<INV, 1, 8>(v[3]);
    v[5] = twc<INV, 2, 8>(v[5]);
    v[7] = twc<INV, 3, 8>(v[7]);
    bfly2<INV>(v[0], v[1]);
    bfly2<INV>(v[2], v[3]);
    bfly2<INV>(v[4], v[5]);
    bfly2<INV>(v[6], v[7]);
    // outputs now at: X0=v0, X4=v1, X1=v2, X5=v3, X2=v4, X6=v5, X3=v6, X7=v7
    cx<T> x[8] = { v[0], v[2], v[4], v[6], v[1], v[3], v[5], v[7] };
#pragma unroll
    for (int i = 0; i < 8; ++i)
        v[i] = x[i];
}

template <bool INV, typename T>
__device__ __forceinline__ void bfly16(cx<T>* v)
{
    // 4 x 4: column DFTs over n = n1 + 4*n2 (stride-4 groups), twiddle W16^(n1*k2), row DFTs
#pragma unroll
    for (int n1 = 0; n1 < 4; ++n1)
        bfly4<INV>(v[n1], v[n1 + 4], v[n1 + 8], v[n1 + 12]);
    // element (n1, k2) sits at v[n1 + 4*k2]
    v[5]  = twc<INV, 1, 16>(v[5]);
    v[6]  = twc<INV, 2, 16>(v[6]);
    v[7]  = twc<INV, 3, 16>(v[7]);
    v[9]  = twc<INV, 2, 16>(v[9]);
    v[10] = twc<INV, 4, 16>(v[10]);
    v[11] = twc<INV, 6, 16>(v[11]);
    v[13] = twc<INV, 3, 16>(v[13]);
    v[14] = twc<INV, 6, 16>(v[14]);
    v[15] = twc<INV, 9, 16>(v[15]);
#pragma unroll
    for (int k2 = 0; k2 < 4; ++k2)
        bfly4<INV>(v[4 * k2], v[4 * k2 + 1], v[4 * k2 + 2], v[4 * k2 + 3]);
    // (k2, k1) at v[4*k2 + k1] holds X[k2 + 4*k1]
    cx<T> x[16];
#pragma unroll
    for (int k2 = 0; k2 < 4; ++k2)
#pragma unroll
        for (int k1 = 0; k1 < 4; ++k1)
            x[k2 + 4 * k1] = v[4 * k2 + k1];
#pragma unroll
    for (int i = 0; i < 16; ++i)
        v[i] = x[i];
}

// An opaque copy of v (an empty asm statement that the compiler must assume rewrites the register).
// Indices derived from the copy are not merged with those derived from v, so a kernel recomputes its
// cheap per-slot offsets in each phase instead of keeping dozens of them live (and spilled) across
// the phases in between.
__device__ __forceinline__ int fresh(int v)
{
    asm volatile("" : "+v"(v));
    return v;
}

// Makes a value exist in registers at this point: the arithmetic that forms it cannot sink below,
// so the (more numerous) operands it was formed from die here.
template <typename T>
__device__ __forceinline__ void settle(cx<T>& a)
{
    asm volatile("" : "+v"(a.re), "+v"(a.im));
}

// f(std::integral_constant<int, I>) for I = 0 .. N-1, unrolled at compile time
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f)
{
    [&]<int... I>(std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>{}), ...); }(
        std::make_integer_sequence<int, N>{});
}

// Odd prime R: conjugate-pair form. X[0] = sum; for k>0 X[k] = x0 + sum_{n=1}^{h}
// (x_n + x_{R-n}) cos(2 pi n k/R) -+ i (x_n - x_{R-n}) sin(2 pi n k/R).
template <int R, bool INV, typename T>
__device__ __forceinline__ void bfly_odd(cx<T>* v)
{
    constexpr int h = (R - 1) / 2;
    cx<T> s[h], d[h];
    cx<T> x0 = v[0], sum = v[0];
#pragma unroll
    for (int n = 1; n <= h; ++n)
    {
        s[n - 1] = cadd(v[n], v[R - n]);
        d[n - 1] = csub(v[n], v[R - n]);
        sum      = cadd(sum, s[n - 1]);
    }
    v[0] = sum;
    // the cosines and sines are template constants: evaluated by the compiler, never at run time
    static_for<h>([&](auto km1)
    {
        constexpr int k = decltype(km1)::value + 1;
        cx<T> a = x0, b = { T(0), T(0) };
        static_for<h>([&](auto nm1)
        {
            constexpr int n  = decltype(nm1)::value + 1;
            constexpr T c    = T(ccos2pi(long(n) * k, R));
            constexpr T sn   = T(csin2pi(long(n) * k, R));
            a.re += s[n - 1].re * c;
            a.im += s[n - 1].im * c;
            b.re += d[n - 1].re * sn;
            b.im += d[n - 1].im * sn;
        });
        // forward: X[k] = a - i b, X[R-k] = a + i b ; inverse: swapped signs
        cx<T> ib = { -b.im, b.re };
        if constexpr (INV)
        {
            v[k]     = cadd(a, ib);
            v[R - k] = csub(a, ib);
        }
        else
        {
            v[k]     = csub(a, ib);
            v[R - k] = cadd(a, ib);
        }
    });
}

template <int R, bool INV, typename T>
__device__ __forceinline__ void butterfly(cx<T>* v);

// inverse of a modulo m (coprime)
constexpr int mod_inverse(int a, int m)
{
    for (int x = 1; x < m; ++x)
        if (a * x % m == 1)
            return x;
    return 1;
}

// N1*N2 points with coprime N1 and N2 (Good and Thomas's prime factor map): input N2*n1 + N1*n2 and
// output N2*(N2^-1 mod N1)*k1 + N1*(N1^-1 mod N2)*k2, both mod N1*N2, make it an N1 x N2 DFT without
// twiddles between the two.
template <int N1, int N2, bool INV, typename T>
__device__ __forceinline__ void bfly_pfa(cx<T>* v)
{
    constexpr int N = N1 * N2;
    cx<T> a[N1][N2];
    static_for<N2>([&](auto i2)
    {
        constexpr int n2 = decltype(i2)::value;
        cx<T> u[N1];
        static_for<N1>([&](auto i1)
        {
            constexpr int n1 = decltype(i1)::value;
            u[n1]            = v[(N2 * n1 + N1 * n2) % N];
        });
        butterfly<N1, INV>(u);
        static_for<N1>([&](auto i1) { a[decltype(i1)::value][n2] = u[decltype(i1)::value]; });
    });
    static_for<N1>([&](auto i1)
    {
        constexpr int k1 = decltype(i1)::value;
        butterfly<N2, INV>(a[k1]);
        static_for<N2>([&](auto i2)
        {
            constexpr int k2 = decltype(i2)::value;
            constexpr int k  = (N2 * mod_inverse(N2 % N1, N1) * k1 + N1 * mod_inverse(N1 % N2, N2) * k2) % N;
            v[k]             = a[k1][k2];
        });
    });
}

template <bool INV, typename T>
__device__ __forceinline__ void bfly9(cx<T>* v)
{
    // 3 x 3: column DFTs over n = 3*n1 + n2, twiddle W9^(n2*k1), row DFTs; X[k1 + 3*k2]
    cx<T> a[3][3];
    static_for<3>([&](auto i2)
    {
        constexpr int n2 = decltype(i2)::value;
        cx<T> u[3]       = { v[n2], v[3 + n2], v[6 + n2] };
        bfly_odd<3, INV>(u);
        a[0][n2] = u[0];
        a[1][n2] = twc<INV, n2, 9>(u[1]);
        a[2][n2] = twc<INV, 2 * n2, 9>(u[2]);
    });
    static_for<3>([&](auto i1)
    {
        constexpr int k1 = decltype(i1)::value;
        bfly_odd<3, INV>(a[k1]);
        v[k1]     = a[k1][0];
        v[k1 + 3] = a[k1][1];
        v[k1 + 6] = a[k1][2];
    });
}

template <int R, bool INV, typename T>
__device__ __forceinline__ void butterfly(cx<T>* v)
{
    if constexpr (R == 2)
        bfly2<INV>(v[0], v[1]);
    else if constexpr (R == 4)
        bfly4<INV>(v[0], v[1], v[2], v[3]);
    else if constexpr (R == 8)
        bfly8<INV>(v);
    else if constexpr (R == 16)
        bfly16<INV>(v);
    else if constexpr (R == 9)
        bfly9<INV>(v);
    else if constexpr (R == 6)
        bfly_pfa<2, 3, INV>(v);
    else if constexpr (R == 10)
        bfly_pfa<2, 5, INV>(v);
    else if constexpr (R == 12)
        bfly_pfa<4, 3, INV>(v);
    else if constexpr (R == 14)
        bfly_pfa<2, 7, INV>(v);
    else if constexpr (R == 15)
        bfly_pfa<3, 5, INV>(v);
    else
        bfly_odd<R, INV>(v);
}

// ---------------------------------------------------------------------------------------------
// Division by a runtime-invariant divisor d < 2^31 for dividends n < 2^31:
// q = (umulhi(n, m) + n) >> s with s = ceil(log2 d), m = floor(2^32 (2^s - d) / d) + 1.
struct fastdiv
{
    uint32_t d = 1, m = 1, s = 0;
};

__host__ inline fastdiv make_fastdiv(uint32_t d)
{
    fastdiv f;
    f.d      = d;
    uint32_t s = 0;
    while ((uint64_t(1) << s) < d)
        ++s;
    f.s = s;
    f.m = (uint32_t)(((uint64_t(1) << 32) * ((uint64_t(1) << s) - d)) / d + 1);
    return f;
}

__device__ __forceinline__ uint32_t fdiv(uint32_t n, const fastdiv& f)
{
    return (uint32_t)(((uint64_t)__umulhi(n, f.m) + n) >> f.s);
}

// ---------------------------------------------------------------------------------------------
// LDS Stockham engine.
//
// A transform of length n is computed by passes p = 0..np-1 of radix R_p. With Ns the product of the
// radices before pass p, butterfly j (0 <= j < n/R) reads x[j + r*n/R] (r = 0..R-1), multiplies
// element r by W_{Ns*R}^{r*(j mod Ns)}, runs the R-point DFT and writes element r to
// (j - j mod Ns)*R + j mod Ns + r*Ns. The last pass has Ns*R = n and writes j + r*n/R, so the
// result is in natural order without a reorder pass. Where data are plain, the first pass reads
// its operands straight from HBM (consecutive threads, consecutive addresses) and the last pass
// writes straight to HBM, so a transform of np passes crosses LDS np - 1 times; a load or store
// phase with element operations stages through LDS instead. What bounded these kernels was instructions
// and LDS trips: staging both ends and radices of at most 7 for odd factors, 960 points made five trips
// and took 173 us for 16384 f32 transforms; as 15 x 8 x 8 with two trips they take 54 us (a copy of the same
// bytes 49 us). f64 30240 x 256 (four-step, 168 x 180) 228 -> 114 us, the uneven batch of 20,000 transforms
// 429 -> 338 us.

constexpr int max_passes = 20;
// Complex values a thread holds per pass: about 16 complex f32 or 8 complex f64 (bflies). Kernels come
// in two register classes: power-of-two radices only, with up to 1024 threads per block (128 VGPRs
// each), and mixed radices, with up to 512 threads (256 VGPRs each).
// The f64 value is a build option so that the CPU emulation of these kernels (tests/cpu_emu) can check
// the 16-points-per-thread geometry for f64 too; the library is built with 8.
#ifndef KFR_AMD_PMAX_F64
#define KFR_AMD_PMAX_F64 8
#endif
template <typename T>
inline constexpr int pmax_of = sizeof(T) == 4 ? 16 : KFR_AMD_PMAX_F64;
constexpr int max_block_pow2  = 1024;
constexpr int max_block_mixed = 512;
__host__ __device__ constexpr int max_block_of(bool mixed) { return mixed ? max_block_mixed : max_block_pow2; }

enum pass_kind : int
{
    pass_radix   = 0, // specialised butterfly (lds_radix)
    pass_generic = 1  // direct R-point DFT (R prime, 11..127) from a W_{Ns*R} table
};

struct pass_desc
{
    int radix;
    int ns;
    int nb; // butterflies, n / radix
    int tw; // offset of this pass's twiddles in the plan's table (complex elements)
    int kind;
    fastdiv ns_div;
};

struct lds_geom
{
    int n;       // transform length
    int np;      // number of passes
    int tpt;     // threads per transform
    int tpb;     // transforms per block
    int mapping; // 0: transform = tid / tpt ; 1: transform = tid % tpb
    int ls;      // LDS element stride
    int ld;      // LDS distance between transforms
    int padshift; // LDS padding: one slot per 2^padshift elements (padded kernels)
    fastdiv tpt_div;
    pass_desc pass[max_passes];
};

// Radices with a butterfly, and butterflies per thread of a radix-R pass: as many as a thread's pm
// values hold, rounded up for the small radices so that every length up to 512*pm runs on at most 512
// threads; one of radix 12, 14 and 15, whose tables and temporaries are the largest.
__host__ __device__ constexpr bool lds_radix(int r)
{
    return (r >= 2 && r <= 10) || r == 12 || r == 14 || r == 15 || r == 16;
}
__host__ __device__ constexpr int bflies(int r, int pm) { return r >= 12 ? (pm >= r ? pm / r : 1) : (pm + r - 1) / r; }
template <typename T, int R>
inline constexpr int bflies_of = bflies(R, pmax_of<T>);

// Padded LDS layout (PAD): logical element x lives at x + (x >> padshift), one padding slot per 16
// (or 32) elements, so that the power-of-two strides of the Stockham passes spread over the banks
// instead of hitting one. Mixed schedules run unpadded, one addition per address instead of three
// operations: most start with an odd radix, whose strided writes spread by themselves, and those of even radices
// only (a quarter of the 7-smooth lengths, 192 = 16 * 12, 768 = 16 * 8 * 6) gain as much from the other changes of
// these kernels (768 x 10922 f32 81 -> 31 us, f64 960 = 12 * 10 * 8 x 8738 76 -> 46); padded they were not measured.
template <bool PAD>
__device__ __forceinline__ int lds_pad(int x, int s)
{
    if constexpr (PAD)
        return x + (x >> s);
    else
        return x;
}
__host__ __device__ inline size_t lds_padded_elems(size_t logical) { return logical + logical / 16 + 1; }

template <typename T, bool PAD>
struct fft_ctx
{
    cx<T>* lds;  // the block's LDS
    int base;    // this transform's logical LDS offset (tb * ld)
    int ls;      // logical element stride
    int ps;      // padding shift
    int t;       // thread index within the transform
    int tb;      // transform index within the block
    bool valid;  // transform exists (batch tail)
    long long g; // global transform index
    // slot at logical offset x
    __device__ __forceinline__ cx<T>& slot(int x) const { return lds[lds_pad<PAD>(x, ps)]; }
    // element i of this transform
    __device__ __forceinline__ cx<T>& at(int i) const { return slot(base + i * ls); }
};

// Where a pass reads and writes its values: LDS, or (first and last pass) strided global memory.
struct via_lds
{
    static constexpr bool global = false;
};
// first pass: element i at p[i * stride]; conj reads conjugates; threads of missing transforms read
// zeros
template <typename T, bool CONJ = false>
struct from_global
{
    static constexpr bool global = true;
    const cx<T>* p;
    long long stride;
    bool valid;
    bool conj = false;
    __device__ __forceinline__ cx<T> get(const cx<T>* q) const
    {
        cx<T> v = valid ? *q : cx<T>{ T(0), T(0) };
        if constexpr (CONJ)
            v.im = conj ? -v.im : v.im;
        return v;
    }
};
// last pass: element i to p[i * stride]; NT: nontemporal stores
template <typename T, bool CONJ = false, bool NT = false>
struct to_global
{
    static constexpr bool global  = true;
    static constexpr bool twiddle = false;
    cx<T>* p;
    long long stride;
    bool valid;
    bool conj = false;
    __device__ __forceinline__ void put(cx<T>* q, cx<T> v) const
    {
        if constexpr (CONJ)
            v.im = conj ? -v.im : v.im;
        if constexpr (NT)
        {
            using V2 = T __attribute__((ext_vector_type(2)));
            __builtin_nontemporal_store(V2{ v.re, v.im }, reinterpret_cast<V2*>(q));
        }
        else
            *q = v;
    }
};
// last pass of a four-step column: element i times W_n^(col*i) (ta[h] = W_n^(h*2^lbits), tb[l] = W_n^l;
// none if ta is null) to p[i * stride]
template <typename T>
struct to_column : to_global<T>
{
    static constexpr bool twiddle = true;
    const cx<T>*ta, *tb;
    int lbits;
    unsigned col;
    __device__ __forceinline__ cx<T> table(unsigned long long m) const
    {
        return cmul(ta[m >> lbits], tb[m & ((1ull << lbits) - 1)]);
    }
};

__host__ __device__ constexpr int ceil_log2(int v)
{
    int l = 0;
    while ((1 << l) < v)
        ++l;
    return l;
}

// workgroup barrier for LDS exchanges: the fences cover the local address space only, so it does not
// wait for outstanding global memory operations
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// one radix pass from src to dst; FIRST: pass 0 (Ns = 1, no twiddles). When dst is LDS, it ends with a
// barrier.
template <typename T, int R, bool INV, bool FIRST, bool PAD, typename Src, typename Dst>
__device__ __forceinline__ void radix_pass(const lds_geom& G, const pass_desc& P, const cx<T>* __restrict__ tw,
                                           const fft_ctx<T, PAD>& c, const Src& src, const Dst& dst)
{
    constexpr int M = bflies_of<T, R>;
    const int nb    = P.nb;
    cx<T> v[M][R];
#pragma unroll
    for (int m = 0; m < M; ++m)
    {
        const int j = c.t + m * G.tpt;
        if (j < nb)
        {
            if constexpr (Src::global)
            {
                const cx<T>* q = src.p + (long long)j * src.stride;
                const long long step = (long long)nb * src.stride;
#pragma unroll
                for (int r = 0; r < R; ++r)
                    v[m][r] = src.get(q + r * step);
            }
            else
            {
                const int x = c.base + j * c.ls, step = nb * c.ls;
#pragma unroll
                for (int r = 0; r < R; ++r)
                    v[m][r] = c.slot(x + r * step);
            }
        }
    }
    if constexpr (!Src::global && !Dst::global)
        lds_barrier(); // every value of the previous pass is read before this pass overwrites it
    [[maybe_unused]] cx<T> B[R];
    if constexpr (Dst::global)
        if constexpr (Dst::twiddle)
        {
            // output j + r*Ns of a column takes W^(col*j) times W^(col*Ns*r), the latter built from the
            // table values at r = 2^b with one product per value
            if (dst.ta)
            {
#pragma unroll
                for (int b = 0; (1 << b) < R; ++b)
                    B[1 << b] = dst.table((unsigned long long)dst.col * ((unsigned)P.ns << b));
#pragma unroll
                for (int r = 3; r < R; ++r)
                    if ((r & (r - 1)) != 0)
                        B[r] = cmul(B[r - (1 << (ceil_log2(r + 1) - 1))], B[1 << (ceil_log2(r + 1) - 1)]);
            }
        }
#pragma unroll
    for (int m = 0; m < M; ++m)
    {
        const int j = c.t + m * G.tpt;
        if (j < nb)
        {
            int k = 0;
            if constexpr (!FIRST)
            {
                if (P.ns > 1)
                {
                    // the table's row of k: W_{Ns*R}^(r*k) at k*(R-1) + r-1 (one base address, wide loads)
                    k              = Dst::global ? j : (int)(j - fdiv(j, P.ns_div) * P.ns);
                    const cx<T>* w = tw + P.tw + k * (R - 1);
#pragma unroll
                    for (int r = 1; r < R; ++r)
                        v[m][r] = ctw<INV>(v[m][r], w[r - 1]);
                }
            }
            butterfly<R, INV>(v[m]);
            if constexpr (Dst::global)
            {
                // last pass: j < Ns, output r of butterfly j is element j + r*Ns
                if constexpr (Dst::twiddle)
                {
                    if (dst.ta)
                    {
                        const cx<T> A = dst.table((unsigned long long)dst.col * (unsigned)j);
#pragma unroll
                        for (int r = 0; r < R; ++r)
                            v[m][r] = ctw<INV>(v[m][r], r == 0 ? A : cmul(A, B[r]));
                    }
                }
                if (dst.valid)
                {
                    cx<T>* q             = dst.p + (long long)j * dst.stride;
                    const long long step = (long long)P.ns * dst.stride;
#pragma unroll
                    for (int r = 0; r < R; ++r)
                        dst.put(q + r * step, v[m][r]);
                }
            }
            else
            {
                const int x = c.base + ((j - k) * R + k) * c.ls, step = P.ns * c.ls;
#pragma unroll
                for (int r = 0; r < R; ++r)
                    c.slot(x + r * step) = v[m][r];
            }
        }
    }
    if constexpr (!Dst::global)
        lds_barrier();
}

// direct DFT pass for a prime radix without a specialised butterfly, LDS -> LDS.
// Output o = q*Ns*R + k2*Ns + k is sum_r x[j + r*n/R] W_{Ns*R}^{r*(k + k2*Ns)} with j = q*Ns + k;
// the pass's table holds W_{Ns*R}^m for m in [0, Ns*R).
template <typename T, bool INV, bool PAD>
__device__ __forceinline__ void generic_pass(const lds_geom& G, const pass_desc& P, const cx<T>* __restrict__ tw,
                                             const fft_ctx<T, PAD>& c)
{
    const int R  = P.radix;
    const int nb = G.n / R;
    const int M  = P.ns * R; // table length
    const cx<T>* w = tw + P.tw;
    cx<T> out[pmax_of<T>];
#pragma unroll
    for (int m = 0; m < pmax_of<T>; ++m)
    {
        const int o = c.t + m * G.tpt;
        out[m]      = { T(0), T(0) };
        if (o < G.n)
        {
            const int q    = o / M;
            const int rem  = o - q * M;
            const int k2   = rem / P.ns;
            const int k    = rem - k2 * P.ns;
            const int j    = q * P.ns + k;
            const int step = k + k2 * P.ns;
            int idx        = 0;
            cx<T> acc      = { T(0), T(0) };
            for (int r = 0; r < R; ++r)
            {
                acc = cadd(acc, ctw<INV>(c.at(j + r * nb), w[idx]));
                idx += step;
                if (idx >= M)
                    idx -= M;
            }
            out[m] = acc;
        }
    }
    lds_barrier();
#pragma unroll
    for (int m = 0; m < pmax_of<T>; ++m)
    {
        const int o = c.t + m * G.tpt;
        if (o < G.n)
            c.at(o) = out[m];
    }
    lds_barrier();
}

// f(std::integral_constant<int, R>) for the radix r of a pass (MIXED = false: only the power-of-two
// butterflies; radix 16 only where a thread holds 16 values: check_pass_radices rejects it elsewhere)
template <typename T, bool MIXED, typename F>
__device__ __forceinline__ void with_radix(int r, F&& f)
{
    auto call = [&](auto R)
    {
        if constexpr ((decltype(R)::value & (decltype(R)::value - 1)) == 0
                          ? decltype(R)::value <= 8 || pmax_of<T> >= 16
                          : MIXED)
            f(R);
    };
    switch (r)
    {
    case 2: call(std::integral_constant<int, 2>{}); break;
    case 3: call(std::integral_constant<int, 3>{}); break;
    case 4: call(std::integral_constant<int, 4>{}); break;
    case 5: call(std::integral_constant<int, 5>{}); break;
    case 6: call(std::integral_constant<int, 6>{}); break;
    case 7: call(std::integral_constant<int, 7>{}); break;
    case 8: call(std::integral_constant<int, 8>{}); break;
    case 9: call(std::integral_constant<int, 9>{}); break;
    case 10: call(std::integral_constant<int, 10>{}); break;
    case 12: call(std::integral_constant<int, 12>{}); break;
    case 14: call(std::integral_constant<int, 14>{}); break;
    case 15: call(std::integral_constant<int, 15>{}); break;
    case 16: call(std::integral_constant<int, 16>{}); break;
    default: break;
    }
}

// passes [first, last) of the transform held in LDS; GEN: direct passes among them (MIXED builds)
template <typename T, bool INV, bool MIXED, bool GEN, bool PAD>
__device__ __forceinline__ void fft_passes(const lds_geom& G, const cx<T>* tw, const fft_ctx<T, PAD>& c, int first,
                                           int last)
{
    for (int p = first; p < last; ++p)
    {
        const pass_desc& P = G.pass[p];
        if constexpr (MIXED && GEN)
        {
            if (P.kind == pass_generic)
            {
                generic_pass<T, INV>(G, P, tw, c);
                continue;
            }
        }
        with_radix<T, MIXED>(P.radix, [&](auto R) {
            radix_pass<T, decltype(R)::value, INV, false>(G, P, tw, c, via_lds{}, via_lds{});
        });
    }
}
// all passes (natural order in, natural order out)
template <typename T, bool INV, bool MIXED, bool PAD>
__device__ __forceinline__ void fft_passes(const lds_geom& G, const cx<T>* tw, const fft_ctx<T, PAD>& c)
{
    fft_passes<T, INV, MIXED, true>(G, tw, c, 0, G.np);
}
// pass 0 from src to LDS
template <typename T, bool INV, bool MIXED, bool PAD, typename Src>
__device__ __forceinline__ void first_pass(const lds_geom& G, const cx<T>* tw, const fft_ctx<T, PAD>& c, const Src& src)
{
    with_radix<T, MIXED>(G.pass[0].radix, [&](auto R) {
        radix_pass<T, decltype(R)::value, INV, true>(G, G.pass[0], tw, c, src, via_lds{});
    });
}
// the last of two or more passes from LDS to dst
template <typename T, bool INV, bool MIXED, bool PAD, typename Dst>
__device__ __forceinline__ void last_pass(const lds_geom& G, const cx<T>* tw, const fft_ctx<T, PAD>& c, const Dst& dst)
{
    const pass_desc& P = G.pass[G.np - 1];
    with_radix<T, MIXED>(P.radix, [&](auto R) {
        radix_pass<T, decltype(R)::value, INV, false>(G, P, tw, c, via_lds{}, dst);
    });
}

template <bool PAD, typename T>
__device__ __forceinline__ fft_ctx<T, PAD> make_ctx(const lds_geom& G, cx<T>* lds, long long first_g, long long batch)
{
    fft_ctx<T, PAD> c;
    const int tid = threadIdx.x;
    if (G.mapping == 0)
    {
        c.tb = (int)fdiv((uint32_t)tid, G.tpt_div);
        c.t  = tid - c.tb * G.tpt;
    }
    else
    {
        c.t  = tid / G.tpb;
        c.tb = tid - c.t * G.tpb;
    }
    c.g     = first_g + c.tb;
    c.valid = c.g < batch;
    c.lds   = lds;
    c.base  = c.tb * G.ld;
    c.ls    = G.ls;
    c.ps    = G.padshift;
    return c;
}

} // namespace kfr_amd
