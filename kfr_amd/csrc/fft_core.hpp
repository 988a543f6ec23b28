// Core GPU transform machinery shared by all plans: FP64 table generation, the LDS Stockham kernels
// with fused element operations, the four-step two-pass transform for lengths beyond one workgroup,
// and the schedule (radix choice and launch geometry) for every length.
//
// Element operations connect a transform to its data: the load phase calls ld.load(b, e) for element
// e of batch item b, and the store phase calls st.store(b, e, v). Bluestein chirps, DCT mirroring,
// real-spectrum repacking and pointwise spectrum products are element operations, so none of them
// costs an extra trip through HBM. They are selected at run time (a kernel-uniform switch), which
// keeps the number of compiled kernels small.
#pragma once

#include "fft_device.hpp"
#include "fft_engine.hpp"
#include "fft_mixed.hpp"
#include "fft_pow2.hpp"
#include "fft_timing.hpp"

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

namespace kfr_amd
{

inline unsigned nblocks(long long count, int bs) { return (unsigned)((count + bs - 1) / bs); }

// kernels that use more than 64 KiB of dynamic LDS (up to the CU's 160 KiB) must say so first
template <typename K>
inline void allow_lds(K kernel, size_t bytes)
{
    if (bytes > 65536)
        hip_check(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes),
                  "dynamic LDS attribute");
}

// ------------------------------------------------------------------------------------------------
// element operations

enum ld_mode : int
{
    ld_plain    = 0, // p[b*pdist + e]
    ld_real_pad = 1, // real pairs p[2e], p[2e+1] of a zero-padded (optionally reversed) real signal
    ld_dct2     = 2, // (x[mirror(e)], 0)
    ld_dct3     = 3, // x[e] * W_{4n}^e (x[0] halved)
    ld_cpad     = 4, // zero-padded (optionally reversed) complex signal
    ld_mul      = 5  // p[b*pdist + e] * q[e] (flag: conj(q[e]))
};

enum st_mode : int
{
    st_plain      = 0, // p[b*pdist + e] = v
    st_real_trunc = 1, // real pairs, truncated to n reals, scaled
    st_dct2       = 2, // y[e] = Re(v * W_{4n}^e)
    st_dct3       = 3, // y[mirror(e)] = Re(v)
    st_ctrunc     = 4  // complex, truncated to n, scaled; flag = keep imaginary part
};

__device__ __forceinline__ long long dct_mirror(long long e, long long n)
{
    return e < (n + 1) / 2 ? 2 * e : 2 * (n - 1 - e) + 1;
}

template <typename T>
struct xload
{
    int mode      = ld_plain;
    int flag      = 0; // real_pad/cpad: reversed; half spectra: pack format (1 CCs, 0 Perm); mul: conjugate q
    int src       = 0; // half spectra (spec): 0 p, 1 p*q*scale, 2 p*conj(q)*scale
    int mconj     = 0; // conjugate the post-multiplier
    const void* p = nullptr;
    long long pdist  = 0;
    const cx<T>* q   = nullptr;
    long long qdist  = 0;
    const cx<T>* r   = nullptr; // half spectra: from_fmt twiddles
    long long n      = 0;
    T scale          = T(1);
    long long b0     = 0;
    const cx<T>* mtab = nullptr; // post-multiplier table (Bluestein chirp)
    long long lim    = LLONG_MAX; // elements at or beyond lim are zero

    // value k of half spectrum b (k_real_inv, k_real_unpack)
    __device__ cx<T> spec(long long b, long long k) const
    {
        const cx<T> a = static_cast<const cx<T>*>(p)[b * pdist + k];
        if (src == 0)
            return a;
        const cx<T> c = q[b * qdist + k];
        return cscale(src == 1 ? cmul(a, c) : cmulc(a, c), scale);
    }

    __device__ cx<T> base(long long b, long long e) const
    {
        switch (mode)
        {
        case ld_plain:
        default:
            return static_cast<const cx<T>*>(p)[b * pdist + e];
        case ld_real_pad:
        {
            const T* x         = static_cast<const T*>(p) + b * pdist;
            const long long i0 = 2 * e, i1 = 2 * e + 1;
            T a = T(0), c = T(0);
            if (i0 < n)
                a = flag ? x[n - 1 - i0] : x[i0];
            if (i1 < n)
                c = flag ? x[n - 1 - i1] : x[i1];
            return { a, c };
        }
        case ld_dct2:
            return { static_cast<const T*>(p)[b * n + dct_mirror(e, n)], T(0) };
        case ld_dct3:
        {
            const T v = static_cast<const T*>(p)[b * n + e] * (e == 0 ? T(0.5) : T(1));
            return { v * q[e].re, v * q[e].im };
        }
        case ld_cpad:
        {
            if (e >= n)
                return { T(0), T(0) };
            return static_cast<const cx<T>*>(p)[b * pdist + (flag ? n - 1 - e : e)];
        }
        case ld_mul:
        {
            const cx<T> a = static_cast<const cx<T>*>(p)[b * pdist + e];
            return flag ? cmulc(a, q[e]) : cmul(a, q[e]);
        }
        }
    }

    __device__ __forceinline__ cx<T> load(long long b, long long e) const
    {
        if (e >= lim)
            return { T(0), T(0) };
        cx<T> v = base(b + b0, e);
        if (mtab)
            v = mconj ? cmulc(v, mtab[e]) : cmul(v, mtab[e]);
        return v;
    }
};

template <typename T>
struct xstore
{
    int mode       = st_plain;
    int flag       = 0;
    int mconj      = 0;
    void* p        = nullptr;
    long long pdist = 0;
    const cx<T>* q = nullptr; // dct table
    long long n    = 0;
    T scale        = T(1);
    long long b0   = 0;
    const cx<T>* mtab = nullptr; // pre-multiplier (Bluestein chirp)
    long long lim  = LLONG_MAX;  // elements at or beyond lim are dropped

    __device__ void base(long long b, long long e, cx<T> v) const
    {
        switch (mode)
        {
        case st_plain:
        default:
            static_cast<cx<T>*>(p)[b * pdist + e] = v;
            break;
        case st_real_trunc:
        {
            T* y               = static_cast<T*>(p) + b * pdist;
            const long long i0 = 2 * e;
            if (i0 < n)
                y[i0] = v.re * scale;
            if (i0 + 1 < n)
                y[i0 + 1] = v.im * scale;
            break;
        }
        case st_dct2:
        {
            const cx<T> w = q[e];
            static_cast<T*>(p)[b * n + e] = v.re * w.re - v.im * w.im;
            break;
        }
        case st_dct3:
            static_cast<T*>(p)[b * n + dct_mirror(e, n)] = v.re;
            break;
        case st_ctrunc:
            if (e < n)
                static_cast<cx<T>*>(p)[b * pdist + e] = { v.re * scale, flag ? v.im * scale : T(0) };
            break;
        }
    }

    __device__ __forceinline__ void store(long long b, long long e, cx<T> v) const
    {
        if (e >= lim)
            return;
        if (mtab)
            v = mconj ? cmulc(v, mtab[e]) : cmul(v, mtab[e]);
        base(b + b0, e, v);
    }
};

template <typename T>
inline xload<T> load_plain(const void* p, long long dist)
{
    xload<T> l;
    l.p     = p;
    l.pdist = dist;
    return l;
}
template <typename T>
inline xstore<T> store_plain(void* p, long long dist)
{
    xstore<T> s;
    s.p     = p;
    s.pdist = dist;
    return s;
}

// ------------------------------------------------------------------------------------------------
// FP64 table generation: out[i] = exp(-2*pi*i*a_i/M), a_i reduced exactly in integers, evaluated
// with FP64 sincospi and rounded once to T.

enum twiddle_mode : int
{
    tw_linear = 0, // a = (i*mult + add) mod M
    tw_radix  = 1, // radix-pass table: i = k*(R-1) + (r-1), a = r*k; M = Ns*R
    tw_square = 2, // a = i^2 mod M (Bluestein chirp, M = 2N)
    tw_radix_full = 3, // radix-pass table with r = 0 included: i = k*R + r, a = r*k; M = Ns*R
    tw_powers = 4 // power-of-two pass table: i = b*Ns + k, a = k << b (b < log2 R); M = Ns*R
};

template <typename T>
__global__ void k_twiddles(cx<T>* out, long long count, long long M, long long mult, long long add, int mode,
                           int R)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count)
        return;
    unsigned long long a;
    if (mode == tw_powers)
    {
        const long long ns = M / R;
        const long long b  = i / ns;
        a                  = (unsigned long long)(((i - b * ns) << b) % M);
    }
    else if (mode == tw_radix_full)
    {
        const long long k = i / R;
        const long long r = i - k * R;
        a                 = (unsigned long long)((r * k) % M);
    }
    else if (mode == tw_radix)
    {
        const long long k = i / (R - 1);
        const long long r = i - k * (R - 1) + 1;
        a                 = (unsigned long long)((r * k) % M);
    }
    else if (mode == tw_square)
    {
        const unsigned long long ii = (unsigned long long)i % (unsigned long long)M;
        a = (unsigned long long)(((unsigned __int128)ii * ii) % (unsigned long long)M);
    }
    else
    {
        a = (unsigned long long)(((__int128)i * mult + add) % M);
    }
    long long as = (long long)a; // symmetric range keeps the FP64 argument small
    if (2 * as > M)
        as -= M;
    const double x = 2.0 * (double)as / (double)M;
    double s, c;
    sincospi(x, &s, &c);
    out[i] = { (T)c, (T)(-s) };
}

template <typename T>
void gen_twiddles(cx<T>* out, long long count, long long M, long long mult, long long add, int mode, int R,
                  hipStream_t s)
{
    if (count <= 0)
        return;
    timing::span ts([] { return timing::kernel_name("k_twiddles", timing::type_name<T>()); },
                    (long long)sizeof(cx<T>) * count, s);
    hipLaunchKernelGGL(k_twiddles<T>, dim3(nblocks(count, 256)), dim3(256), 0, s, out, count, M, mult, add, mode,
                       R);
    hip_check(hipGetLastError(), "twiddle generation launch");
}

// ------------------------------------------------------------------------------------------------
// Stockham schedule (host): GPU radix choice, twiddle layout and launch geometry for one length.

struct stockham
{
    int n = 0;
    std::vector<int> radix, kind, ns;
    std::vector<long long> tw_off;
    long long tw_count = 0;
    int tpt            = 0;
};

// Pass geometry of an explicit radix list (product n): strides, twiddle offsets, threads per transform
inline bool stockham_from_radices(long long nn, const std::vector<int>& radices, stockham& S, int pm)
{
    S = stockham{};
    if (nn < 1 || nn > (1 << 28) || (int)radices.size() > max_passes)
        return false;
    const int n = (int)nn;
    S.n         = n;
    S.radix     = radices;
    long long ns = 1, off = 0;
    int tpt      = 1;
    for (int r : S.radix)
    {
        const bool g = !lds_radix(r);
        S.kind.push_back(g ? pass_generic : pass_radix);
        S.ns.push_back((int)ns);
        S.tw_off.push_back(off);
        if (g)
        {
            off += ns * r;
            tpt = std::max(tpt, (n + pm - 1) / pm);
        }
        else
        {
            if (ns > 1)
                off += ns * (r - 1);
            const int M  = bflies(r, pm);
            const int nb = n / r;
            tpt          = std::max(tpt, (nb + M - 1) / M);
        }
        ns *= r;
    }
    if (ns != nn)
        return false;
    S.tw_count = off;
    S.tpt      = tpt;
    return true;
}

// prime factors of m other than 2 (7, 5, 3 first, then 11..127 ascending); false if another remains
inline bool odd_factors(long long& m, std::vector<int>& odd)
{
    for (int p : { 7, 5, 3 })
        while (m % p == 0)
        {
            odd.push_back(p);
            m /= p;
        }
    for (int p = 11; m > 1 && p <= 127; p += 2)
        while (m % p == 0)
        {
            odd.push_back(p);
            m /= p;
        }
    return m == 1;
}

// Factors of n: its power-of-two part in the largest butterflies that fit a thread's pm values (16 for
// f32, 8 for f64) and the remainder 8/4/2; then 7, 5, 3; then any other prime factor up to 127 (a direct
// DFT pass). False if another prime remains. This is the schedule of the power-of-two lengths, and its
// thread count is the capacity rule of one workgroup for every length (workgroup_threads).
inline bool factor_radices(long long nn, std::vector<int>& radix, int pm)
{
    radix.clear();
    if (nn < 1 || nn > (1 << 28))
        return false;
    long long m = nn;
    int a       = 0;
    while (m % 2 == 0)
    {
        m /= 2;
        ++a;
    }
    const int rbits = pm >= 16 ? 4 : 3;
    while (a >= rbits)
    {
        radix.push_back(1 << rbits);
        a -= rbits;
    }
    if (a > 0)
        radix.push_back(1 << a);
    return odd_factors(m, radix);
}

// Threads that one transform counts for in the capacity rule (which lengths one workgroup takes): at
// most pm values per thread in every pass of factor_radices, or with `wide` one butterfly more. The
// planned schedule of a length within the rule never needs more threads than the workgroup limit.
inline int workgroup_threads(long long nn, int pm, bool wide)
{
    std::vector<int> radix;
    if (!factor_radices(nn, radix, pm))
        return INT_MAX;
    long long t = 1;
    for (int r : radix)
    {
        const bool g      = !(r <= 5 || r == 7 || r == 8 || r == 16);
        const long long M = g ? 1 : wide ? (pm + r - 1) / r : std::max(1, pm / r);
        t                 = std::max(t, g ? (nn + pm - 1) / pm : (nn / r + M - 1) / M);
    }
    return (int)std::min<long long>(t, INT_MAX);
}

// Schedule of a length with odd factors: the product of butterfly radices (2..10, 12, 14, 15, 16) with
// the least modelled work per point. A pass costs its butterfly's arithmetic, its twiddles and one
// exchange through LDS, times the lanes that its butterflies leave idle at the schedule's thread count,
// so few passes of large radices with equal thread counts win: 960 points run as 15 x 8 x 8 on 64
// threads. The largest odd radix goes first (its strided LDS writes meet no bank twice), direct passes
// of larger primes last.
inline bool plan_mixed(long long nn, stockham& S, int pm, int max_threads)
{
    std::vector<int> base;
    if (!factor_radices(nn, base, pm))
        return false;
    std::vector<int> direct;
    long long m = nn;
    for (int r : base)
        if (r > 7 && r % 2 != 0)
        {
            direct.push_back(r);
            m /= r;
        }
    struct choice
    {
        int r;
        double cost; // vector instructions per point of the butterfly
    };
    static constexpr choice menu[] = { { 16, 10.5 }, { 15, 13 }, { 14, 16 }, { 12, 9 }, { 10, 10 }, { 9, 11 }, { 8, 7 },
                                       { 7, 14 },    { 6, 7 },   { 5, 8 },   { 4, 4 },  { 3, 5 },   { 2, 2 } };
    constexpr int choices = (int)(sizeof(menu) / sizeof(menu[0]));
    std::vector<int> cur, best;
    double best_cost = 1e300;
    auto search = [&](auto&& self, long long rest, int from) -> void
    {
        if (rest == 1)
        {
            // threads per transform as stockham_from_radices finds them
            long long tpt = direct.empty() ? 1 : (nn + pm - 1) / pm;
            for (int r : cur)
                tpt = std::max(tpt, (nn / r + bflies(r, pm) - 1) / bflies(r, pm));
            if ((cur.empty() && direct.empty()) || tpt > max_threads)
                return;
            double cost = 0;
            for (int r : cur)
                for (const choice& c : menu)
                    if (c.r == r)
                        cost += (c.cost + 4 + 13) * ((double)tpt * bflies(r, pm) * r / (double)nn);
            if (cost < best_cost)
            {
                best_cost = cost;
                best      = cur;
            }
            return;
        }
        if ((int)cur.size() + (int)direct.size() >= max_passes)
            return;
        for (int i = from; i < choices; ++i)
        {
            const int r = menu[i].r;
            // no 16-point butterfly in the f64 builds (check_pass_radices); with 12, 14 and 15 points f64
            // 30240 x 277 (180 x 168 = 15*12 x 14*12) takes 112 us, 173 with at most 10 points
            if (rest % r != 0 || (pm < 16 && r == 16))
                continue;
            cur.push_back(r);
            self(self, rest / r, i);
            cur.pop_back();
        }
    };
    search(search, m, 0);
    if (best_cost == 1e300)
        return false;
    auto odd = std::find_if(best.begin(), best.end(), [](int r) { return r % 2 != 0; }); // the largest
    if (odd != best.end())
        std::rotate(best.begin(), odd, odd + 1);
    best.insert(best.end(), direct.begin(), direct.end());
    return stockham_from_radices(nn, best, S, pm);
}

// Factor n into GPU passes: the fixed schedule for powers of two, the planned one for the others. Planned
// pass lists are kept per process (lengths of one workgroup, so at most some ten thousand short lists):
// the four-step planner asks for those of every divisor.
inline bool make_stockham(long long nn, stockham& S, int pm)
{
    std::vector<int> radix;
    if (!factor_radices(nn, radix, pm))
        return false;
    if ((nn & (nn - 1)) == 0)
        return stockham_from_radices(nn, radix, S, pm);
    static std::mutex mu;
    static std::map<std::pair<long long, int>, std::vector<int>> planned;
    const std::pair<long long, int> key{ nn, pm };
    {
        std::lock_guard<std::mutex> lock(mu);
        auto f = planned.find(key);
        if (f != planned.end())
            return stockham_from_radices(nn, f->second, S, pm);
    }
    if (!plan_mixed(nn, S, pm, max_block_mixed))
        return stockham_from_radices(nn, radix, S, pm);
    if (nn <= 1 << 14)
    {
        std::lock_guard<std::mutex> lock(mu);
        planned[key] = S.radix;
    }
    return true;
}

// A finer schedule of the same transform for progressive execution, about `want` passes: every odd
// prime factor its own pass, the power-of-two part split into near-equal passes (at most 2^4 points
// for f32, 2^3 for f64, at least 2) so that the pass count approaches `want`.
inline bool make_stockham_progressive(long long nn, int want, stockham& S, int pm)
{
    long long m = nn;
    int a       = 0;
    while (m % 2 == 0)
    {
        m /= 2;
        ++a;
    }
    std::vector<int> odd;
    if (!odd_factors(m, odd))
        return false;
    const int rbits = pm >= 16 ? 4 : 3;
    int np2         = 0;
    if (a > 0)
        np2 = std::min(a, std::max((a + rbits - 1) / rbits, want - (int)odd.size()));
    std::vector<int> radix;
    for (int q = 0; q < np2; ++q)
    {
        const int bits = a / np2 + (q < a % np2 ? 1 : 0);
        radix.push_back(1 << bits);
    }
    radix.insert(radix.end(), odd.begin(), odd.end());
    return stockham_from_radices(nn, radix, S, pm);
}

template <typename T>
void gen_stockham_twiddles(const stockham& S, cx<T>* tw, hipStream_t s)
{
    for (size_t p = 0; p < S.radix.size(); ++p)
    {
        const int r  = S.radix[p];
        const int ns = S.ns[p];
        if (S.kind[p] == pass_generic)
            gen_twiddles(tw + S.tw_off[p], (long long)ns * r, (long long)ns * r, 1, 0, tw_linear, r, s);
        else if (ns > 1)
            gen_twiddles(tw + S.tw_off[p], (long long)ns * (r - 1), (long long)ns * r, 0, 0, tw_radix, r, s);
    }
}

inline lds_geom make_geom(const stockham& S, int tpb, int mapping, int ls, int ld)
{
    lds_geom G{};
    G.n       = S.n;
    G.np      = (int)S.radix.size();
    G.tpt     = S.tpt;
    G.tpt_div = make_fastdiv((uint32_t)S.tpt);
    G.tpb     = tpb;
    G.mapping = mapping;
    G.ls      = ls;
    G.ld      = ld;
    static const int padshift = []
    {
        const char* e = std::getenv("KFR_AMD_LDS_PADSHIFT");
        // the tiles are sized for one padding slot per 16 values (lds_padded_elems): sparser only
        return e ? std::max(4, std::min(30, atoi(e))) : 4;
    }();
    G.padshift = padshift;
    for (int p = 0; p < G.np; ++p)
    {
        G.pass[p].radix  = S.radix[p];
        G.pass[p].ns     = S.ns[p];
        G.pass[p].nb     = S.n / S.radix[p];
        G.pass[p].tw     = (int)S.tw_off[p];
        G.pass[p].kind   = S.kind[p];
        G.pass[p].ns_div = make_fastdiv((uint32_t)S.ns[p]);
    }
    return G;
}

// ------------------------------------------------------------------------------------------------
// Kernels

enum kernel_role : int
{
    role_direct = 0, // transform g is batch item g; contiguous block load and store
    role_col    = 1, // four-step pass A: column transforms, twiddled, into the intermediate
    role_row    = 2, // four-step pass B: row transforms of the intermediate, transposed store
    role_pass   = 3, // one HBM pass of a multi-pass Stockham transform: W consecutive butterflies of
                     // radix 2^L, twiddled inputs, outputs at the autosort positions
    role_conv   = 4, // a transform inside another kernel (one per workgroup, whole-length LDS)
    role_block  = 5  // a transform inside another kernel whose LDS only the passes use
};

template <typename T>
struct fourstep_args
{
    cx<T>* scratch = nullptr;
    const cx<T>* ta = nullptr; // W_n^(h*2^lbits)
    const cx<T>* tb = nullptr; // W_n^l, l < 2^lbits
    fastdiv n1div, n2div, ndiv;
    int n1 = 1, n2 = 1, lbits = 0;
    long long n = 1;
};

// Load and store phases. A thread stages up to stage_values elements at a time in registers, so that
// all of their global loads (or stores) are in flight together. In the power-of-two builds (PAD) one
// round holds them all.
template <typename T>
inline constexpr int stage_values = pmax_of<T>;

template <typename T>
__host__ __device__ __forceinline__ bool plain(const xload<T>& ld)
{
    return ld.mode == ld_plain && ld.mtab == nullptr && ld.lim == LLONG_MAX;
}
template <typename T>
__host__ __device__ __forceinline__ bool plain(const xstore<T>& st)
{
    return st.mode == st_plain && st.mtab == nullptr && st.lim == LLONG_MAX;
}

// the block's transforms, element index fastest (e = tb*n + i); LDS layout lds[e] (ld = n, ls = 1)
template <bool PAD, typename T>
__device__ __forceinline__ void block_load(const lds_geom& G, cx<T>* lds, long long first, long long batch,
                                           const xload<T>& ld, const fastdiv& ndiv)
{
    const int total     = G.tpb * G.n;
    const int bs        = blockDim.x;
    const long long rem = (batch - first) * (long long)G.n;
    const int lim       = rem < total ? (int)rem : total;
    int e0 = threadIdx.x;
    do
    {
        cx<T> v[stage_values<T>];
        if (plain(ld) && ld.pdist == G.n)
        {
            const cx<T>* src = static_cast<const cx<T>*>(ld.p) + (first + ld.b0) * (long long)G.n;
#pragma unroll
            for (int k = 0; k < stage_values<T>; ++k)
            {
                const int e = e0 + k * bs;
                v[k]        = e < lim ? src[e] : cx<T>{ T(0), T(0) };
            }
        }
        else
        {
#pragma unroll
            for (int k = 0; k < stage_values<T>; ++k)
            {
                const int e = e0 + k * bs;
                v[k]        = { T(0), T(0) };
                if (e < lim)
                {
                    const int tb = (int)fdiv((uint32_t)e, ndiv);
                    v[k]         = ld.load(first + tb, e - tb * G.n);
                }
            }
        }
#pragma unroll
        for (int k = 0; k < stage_values<T>; ++k)
        {
            const int e = e0 + k * bs;
            if (e < total)
                lds[lds_pad<PAD>(e, G.padshift)] = v[k];
        }
        e0 += stage_values<T> * bs;
    } while (!PAD && e0 < total);
}
template <bool PAD, typename T>
__device__ __forceinline__ void block_store(const lds_geom& G, const cx<T>* lds, long long first, long long batch,
                                            const xstore<T>& st, const fastdiv& ndiv)
{
    const int total     = G.tpb * G.n;
    const int bs        = blockDim.x;
    const long long rem = (batch - first) * (long long)G.n;
    const int lim       = rem < total ? (int)rem : total;
    int e0 = threadIdx.x;
    do
    {
        cx<T> v[stage_values<T>];
#pragma unroll
        for (int k = 0; k < stage_values<T>; ++k)
        {
            const int e = e0 + k * bs;
            if (e < total)
                v[k] = lds[lds_pad<PAD>(e, G.padshift)];
        }
        if (plain(st) && st.pdist == G.n)
        {
            cx<T>* dst = static_cast<cx<T>*>(st.p) + (first + st.b0) * (long long)G.n;
#pragma unroll
            for (int k = 0; k < stage_values<T>; ++k)
            {
                const int e = e0 + k * bs;
                if (e < lim)
                    dst[e] = v[k];
            }
        }
        else
        {
#pragma unroll
            for (int k = 0; k < stage_values<T>; ++k)
            {
                const int e = e0 + k * bs;
                if (e < lim)
                {
                    const int tb = (int)fdiv((uint32_t)e, ndiv);
                    st.store(first + tb, e - tb * G.n, v[k]);
                }
            }
        }
        e0 += stage_values<T> * bs;
    } while (!PAD && e0 < total);
}

// Waves per SIMD that the mixed-radix kernels are compiled for: f32 four, in 128 VGPRs and without spills (up to
// 165 unbounded, a wave fewer); f64 as many as it comes to
template <typename T, bool MIXED>
inline constexpr int mixed_waves = MIXED && sizeof(T) == 4 ? 4 : 1;

// whether a schedule has direct passes (its last passes)
inline bool has_direct(const stockham& s) { return !s.kind.empty() && s.kind.back() == pass_generic; }
// FL: the first pass reads HBM itself (plain loads; row kernels, whose input is the intermediate); FS: the
// last of two or more passes writes HBM itself (plain stores; column kernels). Mixed-radix builds only:
// powers of two with plain data have kernels of their own. GEN: whole transforms with direct passes, which
// stage both ends; compiled without the bound of mixed_waves, in which they spill 68 to 92 bytes per lane (f32 2910 =
// 30 * 97 points x 1441 565 -> 440 us, 190 such lengths 12% faster; short transforms without direct passes
// are 10 to 30% faster with it). The other builds of whole transforms hold no direct pass.
template <typename T, bool INV, int ROLE, bool MIXED, bool FL, bool FS, bool GEN>
__global__ void __launch_bounds__(max_block_of(MIXED), (GEN ? 1 : mixed_waves<T, MIXED>)) k_fft(lds_geom G, const cx<T>* __restrict__ tw, long long batch,
                                              xload<T> ld, xstore<T> st, fourstep_args<T> fs)
{
    constexpr bool PAD = !MIXED;
    constexpr int SV   = stage_values<T>;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    cx<T>* lds               = reinterpret_cast<cx<T>*>(smem_raw);
    const long long first    = (long long)blockIdx.x * G.tpb;
    const fft_ctx<T, PAD> c  = make_ctx<PAD, T>(G, lds, first, batch);
    [[maybe_unused]] uint32_t bl = 0;
    [[maybe_unused]] int col     = 0;
    if constexpr (ROLE == role_col)
    {
        // column col of batch item bl: elements col + n1*i; consecutive lanes take consecutive columns
        bl  = c.valid ? fdiv((uint32_t)c.g, fs.n1div) : 0u;
        col = c.valid ? (int)((uint32_t)c.g - bl * (uint32_t)fs.n1) : 0;
    }
    if constexpr (FL)
    {
        const cx<T>* src = static_cast<const cx<T>*>(ld.p);
        from_global<T> in{ nullptr, 1, c.valid };
        if constexpr (ROLE == role_direct)
            in.p = src + (c.valid ? c.g + ld.b0 : 0) * ld.pdist;
        else if constexpr (ROLE == role_col)
        {
            in.p      = src + ((long long)bl + ld.b0) * ld.pdist + col;
            in.stride = fs.n1;
        }
        else
            in.p = fs.scratch + (c.valid ? c.g : 0) * (long long)G.n; // row g of the intermediate, contiguous
        first_pass<T, INV, MIXED>(G, tw, c, in);
    }
    else
    {
        if constexpr (ROLE == role_direct)
            block_load<PAD>(G, lds, first, batch, ld, fs.ndiv);
        else
        {
            for (int i0 = c.t; i0 < G.n; i0 += SV * G.tpt)
            {
                cx<T> v[SV];
#pragma unroll
                for (int k = 0; k < SV; ++k)
                {
                    const int i = i0 + k * G.tpt;
                    v[k]        = { T(0), T(0) };
                    if (i < G.n && c.valid)
                    {
                        if constexpr (ROLE == role_col)
                            v[k] = ld.load(bl, (long long)col + (long long)fs.n1 * i);
                        else
                            v[k] = fs.scratch[c.g * (long long)G.n + i];
                    }
                }
#pragma unroll
                for (int k = 0; k < SV; ++k)
                {
                    const int i = i0 + k * G.tpt;
                    if (i < G.n)
                        c.at(i) = v[k];
                }
            }
        }
        __syncthreads();
    }
    fft_passes<T, INV, MIXED, (GEN || ROLE != role_direct)>(G, tw, c, FL ? 1 : 0, FS ? G.np - 1 : G.np);
    if constexpr (ROLE == role_direct)
    {
        if constexpr (FS)
            last_pass<T, INV, MIXED>(G, tw, c,
                                     to_global<T>{ static_cast<cx<T>*>(st.p) + (c.valid ? c.g + st.b0 : 0) * st.pdist, 1,
                                                   c.valid });
        else
            block_store<PAD>(G, lds, first, batch, st, fs.ndiv);
    }
    else if constexpr (ROLE == role_col)
    {
        to_column<T> out;
        out.p      = fs.scratch + (long long)bl * fs.n + col;
        out.stride = fs.n1;
        out.valid  = c.valid;
        out.ta     = fs.ta;
        out.tb     = fs.tb;
        out.lbits  = fs.lbits;
        out.col    = (unsigned)col;
        if constexpr (FS)
            last_pass<T, INV, MIXED>(G, tw, c, out);
        else if (c.valid)
            for (int i = c.t; i < G.n; i += G.tpt)
            {
                const cx<T> v = c.at(i);
                out.p[(long long)fs.n1 * i] =
                    out.ta ? ctw<INV>(v, out.table((unsigned long long)col * (unsigned)i)) : v;
            }
    }
    else
    {
        // transposed store: transform index fastest, so consecutive lanes write consecutive columns k2.
        // blockDim = tpt*tpb, so a thread keeps one transform and steps i by tpt.
        const int tid    = threadIdx.x;
        const int tb     = tid % G.tpb;
        const int t2     = tid / G.tpb;
        const long long g = first + tb;
        if (g < batch)
        {
            const uint32_t b2 = fdiv((uint32_t)g, fs.n2div);
            const int k2      = (int)((uint32_t)g - b2 * (uint32_t)fs.n2);
            cx<T>* dst        = static_cast<cx<T>*>(st.p) + ((long long)b2 + st.b0) * st.pdist + k2;
            for (int i0 = t2; i0 < G.n; i0 += SV * G.tpt)
            {
                cx<T> v[SV];
#pragma unroll
                for (int k = 0; k < SV; ++k)
                {
                    const int i = i0 + k * G.tpt;
                    if (i < G.n)
                        v[k] = c.slot(tb * G.ld + i);
                }
                if (plain(st))
                {
#pragma unroll
                    for (int k = 0; k < SV; ++k)
                    {
                        const int i = i0 + k * G.tpt;
                        if (i < G.n)
                            dst[(long long)fs.n2 * i] = v[k];
                    }
                }
                else
                {
#pragma unroll
                    for (int k = 0; k < SV; ++k)
                    {
                        const int i = i0 + k * G.tpt;
                        if (i < G.n)
                            st.store(b2, (long long)k2 + (long long)fs.n2 * i, v[k]);
                    }
                }
            }
        }
    }
}

// Bluestein tables of an n-point transform padded to M points: chirp[m] = exp(-i pi (m^2 mod 2n)/n)
// (n values) and H = FFT_M(h)/M with h the chirp mirrored into both ends of M points (M values), both
// computed in FP64 and rounded once. Synchronises s.
template <typename T>
void bluestein_tables(size_t n, size_t M, cx<T>* chirp, cx<T>* H, hipStream_t s);

// ------------------------------------------------------------------------------------------------
// A transform computed without Bluestein: one LDS kernel, or four-step in two kernels.

inline size_t lds_budget() { return 128 * 1024; }

inline bool is_mixed(const stockham& s)
{
    for (int r : s.radix)
        if (r & (r - 1))
            return true;
    return false;
}

// fft_passes runs a pass only if its build has the butterfly: radix 16 where a thread holds 16 values,
// odd radices and direct prime passes in the mixed-radix build. A schedule with any other pass would
// leave it out silently, so launches check on the host first.
template <typename T>
inline void check_pass_radices(const stockham& s, bool mixed_build)
{
    for (int r : s.radix)
    {
        const bool pow2 = (r & (r - 1)) == 0;
        const bool ok   = pow2 ? r == 2 || r == 4 || r == 8 || (r == 16 && pmax_of<T> >= 16) : mixed_build;
        if (!ok)
            throw std::logic_error("no butterfly for a radix-" + std::to_string(r) + " pass in this kernel build");
    }
}

template <typename T, bool INV, int ROLE, bool MIXED, bool FL, bool FS, bool GEN = false>
void launch_fft_as(const lds_geom& G, const cx<T>* tw, long long batch, const xload<T>& ld, const xstore<T>& st,
                   const fourstep_args<T>& fs, unsigned grid, unsigned block, size_t sh, hipStream_t s)
{
    // complex values in and out: batch items (columns or rows in the four-step roles) of G.n points
    timing::span ts([] { return timing::kernel_name("k_fft", timing::type_name<T>(), INV, ROLE, MIXED, FL, FS, GEN); },
                    2 * (long long)sizeof(cx<T>) * batch * G.n, s);
    allow_lds(k_fft<T, INV, ROLE, MIXED, FL, FS, GEN>, sh);
    hipLaunchKernelGGL((k_fft<T, INV, ROLE, MIXED, FL, FS, GEN>), dim3(grid), dim3(block), sh, s, G, tw, batch, ld, st, fs);
}

// launches the power-of-two or the mixed-radix build of a kernel role; mixed radices with the first
// and last pass on HBM directly where the data are plain. Transforms of fewer than 16 threads load and
// store through LDS in whole-workgroup runs instead (their lanes would touch a line each).
template <typename T, bool INV, int ROLE>
void launch_fft(bool mixed, const lds_geom& G, const cx<T>* tw, long long batch, const xload<T>& ld,
                const xstore<T>& st, const fourstep_args<T>& fs, unsigned grid, unsigned block, size_t sh,
                hipStream_t s)
{
    bool gen = false; // whole transforms with a direct pass
    for (int p = 0; p < G.np; ++p)
        gen = gen || (ROLE == role_direct && G.pass[p].kind == pass_generic);
    const bool wide = !gen && (ROLE != role_direct || G.tpt >= 16);
    const bool fl   = wide && G.pass[0].kind == pass_radix && (ROLE == role_row || plain(ld));
    const bool fl2  = fl && G.np >= 2;
    const bool fst  = wide && G.np >= 2 && G.pass[G.np - 1].kind == pass_radix && (ROLE == role_col || plain(st));
    if (!mixed)
        launch_fft_as<T, INV, ROLE, false, false, false>(G, tw, batch, ld, st, fs, grid, block, sh, s);
    else if constexpr (ROLE == role_row)
    {
        if (fl)
            launch_fft_as<T, INV, ROLE, true, true, false>(G, tw, batch, ld, st, fs, grid, block, sh, s);
        else
            launch_fft_as<T, INV, ROLE, true, false, false>(G, tw, batch, ld, st, fs, grid, block, sh, s);
    }
    else
    {
        if (fl2 && fst)
            launch_fft_as<T, INV, ROLE, true, true, true>(G, tw, batch, ld, st, fs, grid, block, sh, s);
        else if (fst)
            launch_fft_as<T, INV, ROLE, true, false, true>(G, tw, batch, ld, st, fs, grid, block, sh, s);
        else if (gen)
            launch_fft_as<T, INV, ROLE, true, false, false, ROLE == role_direct>(G, tw, batch, ld, st, fs, grid, block, sh, s);
        else
            launch_fft_as<T, INV, ROLE, true, false, false>(G, tw, batch, ld, st, fs, grid, block, sh, s);
    }
    hip_check(hipGetLastError(), "fft launch");
}

template <typename T>
struct core_fft
{
    size_t n      = 0;
    bool fourstep = false;
    // single LDS kernel
    stockham S;
    int tpb = 1;
    // four-step: n = n1 * n2; pass A = n2-point columns (C per block), pass B = n1-point rows (R per block)
    size_t n1 = 0, n2 = 0;
    stockham SA, SB;
    int C = 1, R = 1;
    int lbits       = 0;
    long long chunk = 1; // batch items per four-step round (intermediate = chunk*n)
    dev_mem tw;
    long long twA = 0, twB = 0, twTA = 0, twTB = 0;
    dev_mem scratch;
    // power-of-two lengths and mixed lengths built from the menu: specialised kernels for contiguous
    // batches (plain loads and stores)
    std::unique_ptr<pow2_fft<T>> pow2;
    std::unique_ptr<mixed_fft<T>> mixed;

    static bool fits_lds(size_t len)
    {
        const bool mixed = (len & (len - 1)) != 0;
        return len * sizeof(cx<T>) <= lds_budget() &&
               workgroup_threads((long long)len, pmax_of<T>, false) <= max_block_of(mixed);
    }

    static int pick_tpb(const stockham& s)
    {
        if (s.tpt >= 256)
            return 1;
        int t = std::max(1, 256 / s.tpt);
        // at most 64 KiB of LDS per block so that two blocks share a CU
        const size_t per = lds_padded_elems((size_t)s.n) * sizeof(cx<T>);
        t                = (int)std::max<size_t>(1, std::min<size_t>(t, 65536 / per));
        return t;
    }

    // Threads of one workgroup's schedule with direct passes (large primes), which are the longest by far and take
    // ceil(n / tpt) rounds in every wave: more than the least number where that saves a fifth of the rounds
    // times waves. f64 1032 = 24 * 43 points take 172 threads, 6 rounds of 3 waves, instead of 129 and 8 rounds (x
    // 4064: 200 -> 173 us); savings of an eighth, 1590 points in 228 threads instead of 199, measured slower.
    static void widen_direct(stockham& s)
    {
        if (!has_direct(s))
            return;
        auto cost = [](const stockham& c)
        {
            const int per = pick_tpb(c);
            return (double)((c.n + c.tpt - 1) / c.tpt) * ((c.tpt * per + 63) / 64) / per;
        };
        double best = 0.8 * cost(s);
        int tpt     = s.tpt;
        for (stockham c = s; c.tpt <= max_block_mixed; ++c.tpt)
            if (cost(c) <= best)
            {
                best = std::nextafter(cost(c), 0.0); // fewer threads where two are level
                tpt  = c.tpt;
            }
        s.tpt = tpt;
    }

    core_fft(size_t len, hipStream_t s)
    {
        n = len;
        if (pow2_fft<T>::supports(n))
            pow2.reset(new pow2_fft<T>(n, s));
        else if (mixed_fft<T>::supports(n))
            mixed.reset(new mixed_fft<T>(n, s));
        if (fits_lds(n))
        {
            make_stockham((long long)n, S, pmax_of<T>);
            widen_direct(S);
            check_pass_radices<T>(S, is_mixed(S));
            tpb = pick_tpb(S);
            tw.reset((size_t)std::max<long long>(1, S.tw_count) * sizeof(cx<T>));
            gen_stockham_twiddles(S, tw.as<cx<T>>(), s);
            return;
        }
        plan_fourstep();
        check_pass_radices<T>(SA, is_mixed(SA));
        check_pass_radices<T>(SB, is_mixed(SB));
        fourstep            = true;
        lbits               = (ilog2_ceil(n) + 1) / 2;
        const long long nTB = 1ll << lbits;
        const long long nTA = (long long)(n >> lbits) + 1;
        twA                 = 0;
        twB                 = SA.tw_count;
        twTA                = twB + SB.tw_count;
        twTB                = twTA + nTA;
        tw.reset((size_t)(twTB + nTB) * sizeof(cx<T>));
        cx<T>* t = tw.as<cx<T>>();
        gen_stockham_twiddles(SA, t + twA, s);
        gen_stockham_twiddles(SB, t + twB, s);
        gen_twiddles(t + twTA, nTA, (long long)n, nTB, 0, tw_linear, 0, s);
        gen_twiddles(t + twTB, nTB, (long long)n, 1, 0, tw_linear, 0, s);
        size_t cap = (size_t)256 << 20;
        if (const char* e = std::getenv("KFR_AMD_FOURSTEP_CHUNK_MB"))
            cap = (size_t)std::max(1, atoi(e)) << 20;
        chunk = (long long)std::max<size_t>(1, cap / (n * sizeof(cx<T>)));
    }

    static int ilog2_ceil(size_t v)
    {
        int l = 0;
        while ((size_t(1) << l) < v)
            ++l;
        return l;
    }

    // choose n = n1 * n2 maximising the narrower coalescing width (C columns in pass A, R rows in
    // pass B), then the balance of the two lengths
    void plan_fourstep()
    {
        size_t force_n2 = 0;
        if (const char* e = std::getenv("KFR_AMD_FOURSTEP_N2"))
            force_n2 = (size_t)atoll(e);
        size_t best_n2 = 0;
        int best_w = -1, best_C = 1, best_R = 1;
        double best_bal = 1e300;
        for (size_t d = 2; d * 2 <= n && d <= ((size_t)1 << 16); ++d)
        {
            if (n % d != 0 || (force_n2 && d != force_n2))
                continue;
            const size_t a = n / d;
            if (!fits_lds(d) || !fits_lds(a))
                continue;
            stockham sa, sb;
            make_stockham((long long)d, sa, pmax_of<T>);
            make_stockham((long long)a, sb, pmax_of<T>);
            // the columns (rows) of one workgroup may straddle two batch items: every transform computes
            // its own address and the last workgroup's surplus transforms are masked, so odd counts keep
            // full groups (one column per workgroup had made 3^10 points 1% of peak)
            int C = 16;
            const int bA = max_block_of(is_mixed(sa)), bB = max_block_of(is_mixed(sb));
            while (C > 1 && ((size_t)C * d * sizeof(cx<T>) > lds_budget() || C * sa.tpt > bA))
                C /= 2;
            int R = 16;
            while (R > 1 && ((size_t)R * (a + 1) * sizeof(cx<T>) > lds_budget() || R * sb.tpt > bB))
                R /= 2;
            const int w      = std::min(C, R);
            const double bal = std::fabs(std::log((double)a) - std::log((double)d));
            if (w > best_w || (w == best_w && bal < best_bal))
            {
                best_w   = w;
                best_bal = bal;
                best_n2  = d;
                best_C   = C;
                best_R   = R;
            }
        }
        if (!best_n2)
            throw std::runtime_error("transform length " + std::to_string(n) +
                                     " has no two-pass split on this device");
        n2 = best_n2;
        n1 = n / n2;
        C  = best_C;
        R  = best_R;
        if (const char* e = std::getenv("KFR_AMD_FOURSTEP_C"))
            C = std::max(1, std::min(C, atoi(e)));
        if (const char* e = std::getenv("KFR_AMD_FOURSTEP_R"))
            R = std::max(1, std::min(R, atoi(e)));
        make_stockham((long long)n2, SA, pmax_of<T>);
        make_stockham((long long)n1, SB, pmax_of<T>);
    }

    template <bool INV>
    void run(const xload<T>& ld, const xstore<T>& st, long long batch, hipStream_t s, workspace w = {})
    {
        if (batch <= 0)
            return;
        if ((pow2 || mixed) && plain_batch(ld) && plain_batch(st))
        {
            const cx<T>* x = static_cast<const cx<T>*>(ld.p) + ld.b0 * (long long)n;
            cx<T>* y       = static_cast<cx<T>*>(st.p) + st.b0 * (long long)n;
            if (pow2)
                pow2->run(INV, x, y, batch, s, w);
            else
                mixed->run(INV, x, y, batch, s, w);
            return;
        }
        const cx<T>* t = tw.as<cx<T>>();
        if (!fourstep)
        {
            lds_geom G      = make_geom(S, tpb, 0, 1, (int)n);
            const size_t sh = lds_padded_elems((size_t)tpb * n) * sizeof(cx<T>);
            fourstep_args<T> fs;
            fs.ndiv = make_fastdiv((uint32_t)n);
            launch_fft<T, INV, role_direct>(is_mixed(S), G, t, batch, ld, st, fs, nblocks(batch, tpb),
                                            (unsigned)(S.tpt * tpb), sh, s);
            return;
        }
        if (w.p)
        {
            run_fourstep<INV>(ld, st, batch, static_cast<cx<T>*>(w.p), 3, s,
                              rounds_in(w, chunk, n * sizeof(cx<T>), 1));
            return;
        }
        scratch.ensure((size_t)std::min<long long>(chunk, batch) * n * sizeof(cx<T>));
        run_fourstep<INV>(ld, st, batch, scratch.as<cx<T>>(), 3, s);
    }

    // columns or rows per workgroup of a launch of `count`: `most` (whole lines), halved down to `least` while
    // the launch has fewer workgroups than the card has CUs
    static int group_width(int most, long long count, int least = sizeof(T) == 4 ? 4 : 2)
    {
        while (most > least && (count + most - 1) / most < 256)
            most /= 2;
        return most;
    }

    // four-step in rounds of at most `chunk` items through `mid`: phases bit 0 runs the column kernels,
    // bit 1 the row kernels (one of them alone only within one round)
    template <bool INV>
    void run_fourstep(const xload<T>& ld, const xstore<T>& st, long long batch, cx<T>* mid, int phases,
                      hipStream_t s, long long round = 0)
    {
        const long long chunk = round > 0 ? round : this->chunk;
        const cx<T>* t   = tw.as<cx<T>>();
        fourstep_args<T> fs;
        fs.scratch = mid;
        fs.ta      = t + twTA;
        fs.tb      = t + twTB;
        fs.n1div   = make_fastdiv((uint32_t)n1);
        fs.n2div   = make_fastdiv((uint32_t)n2);
        fs.n1      = (int)n1;
        fs.n2      = (int)n2;
        fs.lbits   = lbits;
        fs.n       = (long long)n;
        const bool mA = is_mixed(SA), mB = is_mixed(SB);
        for (long long b0 = 0; b0 < batch; b0 += chunk)
        {
            const long long nb = std::min(chunk, batch - b0);
            xload<T> la        = ld;
            la.b0 += b0;
            xstore<T> sb = st;
            sb.b0 += b0;
            const long long ga = nb * (long long)n1, gb = nb * (long long)n2;
            const int cw = group_width(C, ga), rw = group_width(R, gb);
            const lds_geom GA = make_geom(SA, cw, 1, cw, 1);
            const lds_geom GB = make_geom(SB, rw, 0, 1, (int)n1 | 1); // an odd distance: the transposed reads spread
            fs.ndiv           = make_fastdiv((uint32_t)n2);
            if (phases & 1)
                launch_fft<T, INV, role_col>(mA, GA, t + twA, ga, la, st, fs, nblocks(ga, cw), (unsigned)(SA.tpt * cw),
                                             lds_padded_elems((size_t)cw * n2) * sizeof(cx<T>), s);
            fs.ndiv = make_fastdiv((uint32_t)n1);
            if (phases & 2)
                launch_fft<T, INV, role_row>(mB, GB, t + twB, gb, ld, sb, fs, nblocks(gb, rw), (unsigned)(SB.tpt * rw),
                                             lds_padded_elems((size_t)rw * (n1 + 1)) * sizeof(cx<T>), s);
        }
    }

    // ---- one axis of a multidimensional array in place along its stride: `outer` arrays of n rows of
    // `inner` values, every column transformed by the four-step column kernel without its twiddle.
    // Columns per workgroup: whole 128-byte lines (16 f32) and a wave of threads, fewer if that leaves CUs
    // without work (the 1080-point axis of a 1080 x 961 spectrum runs 4: 241 workgroups of 288 threads), but
    // 32-byte runs and a wave of threads
    int axis_columns(long long cols) const
    {
        const int most = max_block_of(is_mixed(S));
        int c          = 16;
        while (c * S.tpt < 64)
            c *= 2;
        while (c > 1 && ((size_t)c * n * sizeof(cx<T>) > lds_budget() || c * S.tpt > most))
            c /= 2;
        int least = sizeof(T) == 4 ? 4 : 2;
        while (least * S.tpt < 64)
            least *= 2;
        return group_width(c, cols, least);
    }
    // Lengths of one workgroup whose columns move in runs of 32 bytes or more; f32 powers of two from 256 points
    // (the staged build of the kernel, which spills) 64 bytes, and no f64 powers of two from 4096. What is left
    // takes contiguous transforms and transposes, whose runs are 256 bytes. Measured strided against
    // transposed: 8-byte runs 6000 x 1024 f32 185 and 92 us, 16-byte runs 3000 x 4000 237 and 150, 2400 x
    // 1024 f64 110 and 75, 3000 x 500 f32 45 and 47; 32-byte runs 1080 x 960 f32 34 and 59 (transposed by the kernels
    // of before), 2000 x 2000 58 and 61; f32 powers of two with 32-byte runs 4096 x 2049 273 and 227, 512 x 300 26 and 23, 2048 x
    // 700 41 and 43, with 64-byte runs 1024 x 2400 38 and 47; f64 4096 x 2049 482 and 418, 1024 x 1025 83 and 92.
    bool supports_axis(long long inner, long long outer) const
    {
        if (fourstep || inner <= 0 || outer <= 0 || inner > 0x7fffffffll / outer)
            return false;
        const long long run = std::min<long long>(axis_columns(inner * outer), inner) * (long long)sizeof(cx<T>);
        if (is_mixed(S))
            return run >= 32;
        return sizeof(T) == 4 ? run >= (n >= 256 ? 64 : 32) : run >= 32 && n < 4096;
    }
    template <bool INV>
    void run_axis(const cx<T>* in, cx<T>* out, long long inner, long long outer, hipStream_t s)
    {
        if (!supports_axis(inner, outer))
            throw std::logic_error("this plan cannot transform a strided axis");
        const long long cols = inner * outer;
        const int c          = axis_columns(cols);
        lds_geom G = make_geom(S, c, 1, c, 1);
        fourstep_args<T> fs;
        fs.scratch = out;
        fs.n1div   = make_fastdiv((uint32_t)inner);
        fs.n1      = (int)inner;
        fs.n       = (long long)n * inner;
        launch_fft<T, INV, role_col>(is_mixed(S), G, tw.as<cx<T>>(), cols, load_plain<T>(in, fs.n), xstore<T>{}, fs,
                                     nblocks(cols, c), (unsigned)(S.tpt * c), lds_padded_elems((size_t)c * n) * sizeof(cx<T>),
                                     s);
    }

    // ---- progressive execution (one reference stage per call, include/kfr/dft/fft.hpp:393-439): one
    // item in place on `data`, as units of one launch each. Lengths in one workgroup run one pass of a
    // finer Stockham schedule per unit (about `want` passes); four-step lengths run their column and
    // row kernels as two units through `mid` (n values, kept apart from the plan's scratch).
    stockham Sp;
    dev_mem twp;
    int tpbp = 1;
    void progressive_prepare(int want, hipStream_t s)
    {
        if (fourstep || !Sp.radix.empty())
            return;
        if (!make_stockham_progressive((long long)n, std::max(1, want), Sp, pmax_of<T>))
            throw std::logic_error("no progressive schedule for this length");
        check_pass_radices<T>(Sp, is_mixed(Sp));
        if (Sp.tpt > max_block_of(is_mixed(Sp)))
            throw std::logic_error("progressive schedule needs too many threads per transform");
        tpbp = 1; // one item per progressive execution
        twp.reset((size_t)std::max<long long>(1, Sp.tw_count) * sizeof(cx<T>));
        gen_stockham_twiddles(Sp, twp.as<cx<T>>(), s);
    }
    int progressive_units() const { return fourstep ? 2 : (int)Sp.radix.size(); }
    template <bool INV>
    void progressive_unit(int u, cx<T>* data, cx<T>* mid, hipStream_t s)
    {
        if (fourstep)
        {
            run_fourstep<INV>(load_plain<T>(data, (long long)n), store_plain<T>(data, (long long)n), 1, mid,
                              u == 0 ? 1 : 2, s);
            return;
        }
        lds_geom G = make_geom(Sp, tpbp, 0, 1, (int)n);
        G.pass[0]  = G.pass[u];
        G.np       = 1;
        const size_t sh = lds_padded_elems((size_t)tpbp * n) * sizeof(cx<T>);
        fourstep_args<T> fs;
        fs.ndiv = make_fastdiv((uint32_t)n);
        launch_fft<T, INV, role_direct>(is_mixed(Sp), G, twp.as<cx<T>>(), 1, load_plain<T>(data, (long long)n),
                                        store_plain<T>(data, (long long)n), fs, 1, (unsigned)(Sp.tpt * tpbp), sh,
                                        s);
    }

    // contiguous batch: item b at b*n, no element operation
    bool plain_batch(const xload<T>& l) const
    {
        return l.mode == ld_plain && l.pdist == (long long)n && l.mtab == nullptr && l.lim == LLONG_MAX;
    }
    bool plain_batch(const xstore<T>& st) const
    {
        return st.mode == st_plain && st.pdist == (long long)n && st.mtab == nullptr && st.lim == LLONG_MAX;
    }

    std::vector<int> radices() const
    {
        if (!fourstep)
            return S.radix;
        std::vector<int> r = SA.radix;
        r.insert(r.end(), SB.radix.begin(), SB.radix.end());
        return r;
    }
};

} // namespace kfr_amd
