// Multidimensional DFTs (dft_plan_md / dft_plan_md_real, include/kfr/dft/fft.hpp:569-924) of
// row-major arrays on device data.
#pragma once

#include "fft_engine.hpp"
#include "fft_pow2.hpp"

#include <map>
#include <memory>
#include <string>
#include <vector>

namespace kfr_amd
{

// The axes of a row-major complex array of `shape` but its last one, each transformed along its stride:
// power-of-two axes before power-of-two dimensions by the power-of-two column kernel, other lengths of
// one workgroup by the mixed-radix one.
template <typename T>
class axis_set
{
public:
    // false if an axis needs contiguous transforms (Bluestein and four-step lengths) or its columns are
    // narrower than a 64-byte run; plans: the contiguous plans by length, to which it adds those of the
    // mixed-radix axes
    bool plan(const std::vector<size_t>& shape, std::map<size_t, std::unique_ptr<gpu_dft<T>>>& plans);
    // every axis longer than 1, the last of them first: the first one run reads `in`, the others run in
    // place on `out`; false if there is none
    bool run(void* out, const void* in, bool inverse, hipStream_t s) const;
    std::string describe(size_t i) const; // axis i

private:
    struct entry
    {
        size_t axis, n;
        long long inner, outer;
        pow2_fft<T>* p2; // power-of-two column kernel, or
        gpu_dft<T>* g;   // mixed-radix column kernel
    };
    std::vector<entry> list;
    std::map<size_t, std::unique_ptr<pow2_fft<T>>> pow2;
};

// Complex DFT over every axis of a row-major array of the given shape (two or more axes).
template <typename T>
class gpu_dft_md
{
public:
    explicit gpu_dft_md(const std::vector<size_t>& shape);
    ~gpu_dft_md();
    size_t size() const; // number of complex values
    const std::vector<size_t>& shape() const { return sh; }
    // one array; out == in allowed; no scaling
    void execute(void* out, const void* in, bool inverse, hipStream_t s);
    std::string schedule() const;

private:
    std::vector<size_t> sh;
    size_t total = 0;
    std::map<size_t, std::unique_ptr<gpu_dft<T>>> plans; // one per distinct axis length
    bool strided = false; // every axis but the last is transformed along its stride
    axis_set<T> axes;
    dev_mem scratch;
};

// Real DFT over every axis: real array of `shape` <-> complex array of the same shape with the last
// axis n/2+1 (the CCs format of the last axis, which must be even).
template <typename T>
class gpu_dft_md_real
{
public:
    explicit gpu_dft_md_real(const std::vector<size_t>& shape);
    ~gpu_dft_md_real();
    size_t size() const;         // real values
    size_t complex_size() const; // complex values
    const std::vector<size_t>& shape() const { return sh; }
    void forward(void* cout, const void* rin, hipStream_t s);
    void inverse(void* rout, const void* cin, hipStream_t s);
    std::string schedule() const;

private:
    std::vector<size_t> sh;
    size_t rtotal = 0, ctotal = 0;
    std::map<size_t, std::unique_ptr<gpu_dft<T>>> plans; // complex axes
    std::unique_ptr<gpu_dft_real<T>> last;               // real last axis
    bool strided = false;                                // the complex axes are transformed along their strides
    axis_set<T> axes;
    dev_mem a, b;
};

// out[c*rows + r] = in[r*cols + c] (complex values), LDS-tiled
template <typename T>
void transpose(void* out, const void* in, size_t rows, size_t cols, hipStream_t s);

extern template class gpu_dft_md<float>;
extern template class gpu_dft_md<double>;
extern template class gpu_dft_md_real<float>;
extern template class gpu_dft_md_real<double>;

} // namespace kfr_amd
