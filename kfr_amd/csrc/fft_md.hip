// Multidimensional DFTs on device data. The last axis runs as contiguous rows; every other axis whose
// length fits one workgroup is transformed along its stride by a column kernel, one HBM round trip per
// axis. Shapes with an axis that needs contiguous transforms go the reference's way
// (dft_plan_md::execute_dim, include/kfr/dft/fft.hpp:641-690): every axis as contiguous rows, followed by
// an LDS-tiled transpose that rotates the next axis to the end, a second round trip per axis.
#include "fft_md.hpp"

#include "fft_core.hpp"

#include <stdexcept>

namespace kfr_amd
{

// 32x32 tiles through LDS (padded row), 256 threads, each moving 4 values in and 4 out
template <typename T>
__global__ void __launch_bounds__(256) k_transpose(const cx<T>* __restrict__ in, cx<T>* __restrict__ out,
                                                   long long rows, long long cols, long long tiles_x)
{
    __shared__ cx<T> tile[32][33];
    const long long t  = blockIdx.x;
    const long long ty = t / tiles_x;
    const long long tx = t - ty * tiles_x;
    const int lx       = threadIdx.x & 31;
    const int ly       = threadIdx.x >> 5;
    const long long c  = tx * 32 + lx;
#pragma unroll
    for (int k = 0; k < 32; k += 8)
    {
        const long long r = ty * 32 + ly + k;
        if (r < rows && c < cols)
            tile[ly + k][lx] = in[r * cols + c];
    }
    __syncthreads();
    const long long r2 = ty * 32 + lx;
#pragma unroll
    for (int k = 0; k < 32; k += 8)
    {
        const long long c2 = tx * 32 + ly + k;
        if (c2 < cols && r2 < rows)
            out[c2 * rows + r2] = tile[lx][ly + k];
    }
}

template <typename T>
void transpose(void* out, const void* in, size_t rows, size_t cols, hipStream_t s)
{
    if (rows == 0 || cols == 0)
        return;
    const long long tx = (long long)((cols + 31) / 32), ty = (long long)((rows + 31) / 32);
    if (tx * ty > 0xffffffffll)
        throw std::runtime_error("array too large to transpose in one launch");
    hipLaunchKernelGGL(k_transpose<T>, dim3((unsigned)(tx * ty)), dim3(256), 0, s, static_cast<const cx<T>*>(in),
                       static_cast<cx<T>*>(out), (long long)rows, (long long)cols, tx);
    hip_check(hipGetLastError(), "transpose launch");
}
template void transpose<float>(void*, const void*, size_t, size_t, hipStream_t);
template void transpose<double>(void*, const void*, size_t, size_t, hipStream_t);

namespace
{
size_t product(const std::vector<size_t>& v)
{
    size_t p = 1;
    for (size_t x : v)
        p *= x;
    return p;
}
void check_shape(const std::vector<size_t>& sh)
{
    if (sh.size() < 2)
        throw std::invalid_argument("a multidimensional plan needs at least two axes");
    for (size_t x : sh)
        if (x == 0)
            throw std::invalid_argument("every axis of a multidimensional plan must be positive");
    size_t p = 1;
    for (size_t x : sh)
    {
        if (p > ((size_t)1 << 40) / x)
            throw std::invalid_argument("multidimensional plan is too large");
        p *= x;
    }
}
template <typename T>
std::string axis_text(const std::map<size_t, std::unique_ptr<gpu_dft<T>>>& plans, const std::vector<size_t>& sh,
                      size_t axes)
{
    std::string s;
    for (size_t i = 0; i < axes; ++i)
    {
        const size_t n = sh[i];
        s += "axis " + std::to_string(i) + " (" + std::to_string(n) + "): ";
        auto it = plans.find(n);
        s += (n > 1 && it != plans.end()) ? it->second->schedule().text() : std::string("identity");
        s += "\n";
    }
    return s;
}
} // namespace

template <typename T>
bool axis_set<T>::plan(const std::vector<size_t>& shape, std::map<size_t, std::unique_ptr<gpu_dft<T>>>& plans)
{
    long long inner = (long long)shape.back(), total = 1;
    for (size_t n : shape)
        total *= (long long)n;
    hipStream_t s = library_stream();
    for (size_t i = shape.size() - 1; i-- > 0; inner *= (long long)shape[i])
    {
        const size_t n = shape[i];
        if (n == 1)
            continue;
        const long long outer = total / inner / (long long)n;
        if ((inner & (inner - 1)) == 0 && pow2_fft<T>::supports_axis(n))
        {
            auto& p = pow2[n];
            if (!p)
                p.reset(new pow2_fft<T>(n, s));
            list.push_back({ i, n, inner, outer, p.get(), nullptr });
            continue;
        }
        // columns of 64-byte runs and more: below that the transposes, whose runs are 256 bytes
        bool fits = inner * (long long)sizeof(cx<T>) >= 64;
        if (fits)
        {
            auto& g = plans[n];
            if (!g)
                g.reset(new gpu_dft<T>(n));
            fits = g->supports_axis(inner, outer);
            list.push_back({ i, n, inner, outer, nullptr, g.get() });
        }
        if (!fits)
        {
            hip_check(hipStreamSynchronize(s), "multidimensional plan initialisation");
            list.clear();
            pow2.clear();
            return false;
        }
    }
    hip_check(hipStreamSynchronize(s), "multidimensional plan initialisation");
    return true;
}

template <typename T>
bool axis_set<T>::run(void* out, const void* in, bool inverse, hipStream_t s) const
{
    for (const entry& e : list)
    {
        if (e.p2)
        {
            int l = 0;
            while ((1ll << l) < e.inner)
                ++l;
            e.p2->run_axis(inverse, in, out, l, e.outer, s);
        }
        else
            e.g->execute_axis(out, in, e.inner, e.outer, inverse, s);
        in = out;
    }
    return !list.empty();
}

template <typename T>
std::string axis_set<T>::describe(size_t i) const
{
    for (const entry& e : list)
        if (e.axis == i)
            return "in place along its stride, " + (e.p2 ? e.p2->describe() : e.g->schedule().text());
    return "identity";
}
template class axis_set<float>;
template class axis_set<double>;

template <typename T>
gpu_dft_md<T>::gpu_dft_md(const std::vector<size_t>& shape) : sh(shape)
{
    check_shape(sh);
    total = product(sh);
    if (sh.back() > 1)
        plans[sh.back()].reset(new gpu_dft<T>(sh.back()));
    strided = axes.plan(sh, plans);
    if (strided)
        return;
    for (size_t n : sh)
        if (n > 1 && !plans.count(n))
            plans[n].reset(new gpu_dft<T>(n));
}
template <typename T>
gpu_dft_md<T>::~gpu_dft_md() = default;

template <typename T>
size_t gpu_dft_md<T>::size() const
{
    return total;
}

template <typename T>
std::string gpu_dft_md<T>::schedule() const
{
    if (strided)
    {
        std::string t;
        const size_t n = sh.size() - 1;
        for (size_t i = 0; i < n; ++i)
            t += "axis " + std::to_string(i) + " (" + std::to_string(sh[i]) + "): " + axes.describe(i) + "\n";
        return t + "axis " + std::to_string(n) + " (" + std::to_string(sh.back()) + "): " +
               (sh.back() > 1 ? plans.at(sh.back())->schedule().text() : std::string("identity"));
    }
    return axis_text(plans, sh, sh.size()) + "transpose after every axis";
}

template <typename T>
void gpu_dft_md<T>::execute(void* out, const void* in, bool inverse, hipStream_t s)
{
    if (strided)
    {
        const size_t last = sh.back();
        if (last > 1)
            plans.at(last)->execute(out, in, (long long)(total / last), inverse, s);
        else if (out != in)
            hip_check(hipMemcpyAsync(out, in, total * sizeof(cx<T>), hipMemcpyDeviceToDevice, s), "copy");
        axes.run(out, out, inverse, s);
        return;
    }
    scratch.ensure(total * sizeof(cx<T>));
    std::vector<size_t> cur = sh; // current layout, last axis contiguous
    const void* src         = in;
    for (size_t k = 0; k < sh.size(); ++k)
    {
        const size_t len  = cur.back();
        const size_t rows = total / len;
        if (len > 1)
            plans.at(len)->execute(scratch.ptr, src, (long long)rows, inverse, s);
        else
            hip_check(hipMemcpyAsync(scratch.ptr, src, total * sizeof(cx<T>), hipMemcpyDeviceToDevice, s), "copy");
        transpose<T>(out, scratch.ptr, rows, len, s);
        // the transposed array has the transformed axis first
        cur.insert(cur.begin(), cur.back());
        cur.pop_back();
        src = out;
    }
}

template <typename T>
gpu_dft_md_real<T>::gpu_dft_md_real(const std::vector<size_t>& shape) : sh(shape)
{
    check_shape(sh);
    rtotal = product(sh);
    last.reset(new gpu_dft_real<T>(sh.back(), 1 /* CCs */));
    ctotal = rtotal / sh.back() * last->complex_size();
    std::vector<size_t> csh = sh;
    csh.back()              = last->complex_size();
    strided                 = axes.plan(csh, plans);
    if (strided)
        return;
    for (size_t i = 0; i + 1 < sh.size(); ++i)
        if (sh[i] > 1 && !plans.count(sh[i]))
            plans[sh[i]].reset(new gpu_dft<T>(sh[i]));
}
template <typename T>
gpu_dft_md_real<T>::~gpu_dft_md_real() = default;

template <typename T>
size_t gpu_dft_md_real<T>::size() const
{
    return rtotal;
}
template <typename T>
size_t gpu_dft_md_real<T>::complex_size() const
{
    return ctotal;
}

template <typename T>
std::string gpu_dft_md_real<T>::schedule() const
{
    const std::string lt = "axis " + std::to_string(sh.size() - 1) + " (" + std::to_string(sh.back()) +
                           ", real): " + last->schedule().text();
    if (strided)
    {
        std::string t;
        for (size_t i = 0; i + 1 < sh.size(); ++i)
            t += "axis " + std::to_string(i) + " (" + std::to_string(sh[i]) + "): " + axes.describe(i) + "\n";
        return t + lt;
    }
    return axis_text(plans, sh, sh.size() - 1) + lt + "\ntranspose after every axis";
}

template <typename T>
void gpu_dft_md_real<T>::forward(void* cout, const void* rin, hipStream_t s)
{
    a.ensure(ctotal * sizeof(cx<T>));
    const size_t ck    = last->complex_size();
    const size_t rows0 = rtotal / sh.back();
    // through `a`: the spectrum's rows are longer than the real rows, and the caller may pass one buffer
    last->forward(a.ptr, rin, (long long)rows0, s);
    if (strided)
    {
        if (!axes.run(cout, a.ptr, false, s))
            hip_check(hipMemcpyAsync(cout, a.ptr, ctotal * sizeof(cx<T>), hipMemcpyDeviceToDevice, s), "copy");
        return;
    }
    b.ensure(ctotal * sizeof(cx<T>));
    std::vector<size_t> cur(sh.begin(), sh.end() - 1);
    cur.insert(cur.begin(), ck); // after the transpose: (ck, d0, ..., d_{k-1})
    const size_t naxes = sh.size() - 1;
    transpose<T>(naxes == 0 ? cout : b.ptr, a.ptr, rows0, ck, s);
    for (size_t k = 0; k < naxes; ++k)
    {
        const size_t len  = cur.back();
        const size_t rows = ctotal / len;
        if (len > 1)
            plans.at(len)->execute(a.ptr, b.ptr, (long long)rows, false, s);
        else
            hip_check(hipMemcpyAsync(a.ptr, b.ptr, ctotal * sizeof(cx<T>), hipMemcpyDeviceToDevice, s), "copy");
        transpose<T>(k + 1 == naxes ? cout : b.ptr, a.ptr, rows, len, s);
        cur.insert(cur.begin(), cur.back());
        cur.pop_back();
    }
}

template <typename T>
void gpu_dft_md_real<T>::inverse(void* rout, const void* cin, hipStream_t s)
{
    a.ensure(ctotal * sizeof(cx<T>));
    if (strided)
    {
        if (!axes.run(a.ptr, cin, true, s))
            hip_check(hipMemcpyAsync(a.ptr, cin, ctotal * sizeof(cx<T>), hipMemcpyDeviceToDevice, s), "copy");
        last->inverse(rout, a.ptr, (long long)(rtotal / sh.back()), s);
        return;
    }
    b.ensure(ctotal * sizeof(cx<T>));
    const size_t ck    = last->complex_size();
    const size_t naxes = sh.size() - 1;
    // layout (d0, ..., d_{k-1}, ck); bring each complex axis to the end, transform it in place
    std::vector<size_t> cur(sh.begin(), sh.end() - 1);
    cur.push_back(ck);
    const void* src = cin;
    void* bufs[2]   = { a.ptr, b.ptr };
    int which       = 0;
    for (size_t k = 0; k < naxes; ++k)
    {
        const size_t front = cur.front();
        const size_t rest  = ctotal / front;
        void* dst          = bufs[which];
        transpose<T>(dst, src, front, rest, s);
        if (front > 1)
            plans.at(front)->execute(dst, dst, (long long)rest, true, s);
        cur.push_back(cur.front());
        cur.erase(cur.begin());
        src = dst;
        which ^= 1;
    }
    // layout (ck, d0, ..., d_{k-1}): back to (d0, ..., ck), then the real inverse of every row
    void* dst = bufs[which];
    transpose<T>(dst, src, ck, ctotal / ck, s);
    last->inverse(rout, dst, (long long)(rtotal / sh.back()), s);
}

template class gpu_dft_md<float>;
template class gpu_dft_md<double>;
template class gpu_dft_md_real<float>;
template class gpu_dft_md_real<double>;

} // namespace kfr_amd
