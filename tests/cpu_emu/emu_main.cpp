// Runs one transform of the engine on the CPU emulation of HIP (hip/hip_runtime.h beside this file):
//   emu_main dft  f32|f64 n batch inverse in.bin out.bin
//   emu_main real f32|f64 n fmt batch inverse in.bin out.bin
//   emu_main dct  f32|f64 n batch inverse in.bin out.bin
//   emu_main prog f32|f64 n want inverse in.bin out.bin   (progressive units of one transform)
//   emu_main ws   f32|f64 n batch inverse mb in.bin out.bin (execute with an mb-MiB caller workspace)
//   emu_main half bf16|f16 n batch inverse in.bin out.bin   (half-precision storage, 4-byte values)
//   emu_main constants f64 n out.bin   (cos and sin of 2*pi*k/n, k < n, as the butterflies' constants)
//   emu_main filter f32|f64|c32|c64 taps n,n,... taps.bin in.bin out.bin   (streaming filter, calls of n samples)
//   emu_main md f32|f64 d0,d1,.. real inverse in.bin out.bin   (axes; its schedule on standard output)
//   emu_main schedule f32|f64 n
//   emu_main conv f32|f64 nx nh batch shared in.bin out.bin   (signals, taps and output gradients to
//                                   outputs, signal gradients and tap gradients, one after the other)
//   emu_main order calls out.txt   (stream_order's launches, event records and waits for calls like 0-,5s,0-:
//                                   stream handle, then s with or - without scratch)
// The input is copied into a buffer of exactly its size and the output buffer holds exactly the
// output, so under AddressSanitizer every access beyond either is reported.
#include "../../kfr_amd/csrc/fft_device.hpp"
#include "../../kfr_amd/csrc/fft_engine.hpp"
#include "../../kfr_amd/csrc/fft_md.hpp"
#include "../../kfr_amd/csrc/fft_pow2.hpp"
#include "../../kfr_amd/csrc/stream_order.hpp"

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

using namespace kfr_amd;

static std::vector<char> read_file(const char* path)
{
    std::vector<char> v;
    FILE* f = std::fopen(path, "rb");
    if (!f)
        return v;
    char buf[1 << 16];
    size_t r;
    while ((r = std::fread(buf, 1, sizeof(buf), f)) > 0)
        v.insert(v.end(), buf, buf + r);
    std::fclose(f);
    return v;
}

template <typename T>
static int run(const std::string& kind, int argc, char** argv)
{
    const size_t n = std::strtoull(argv[3], nullptr, 10);
    int a          = 4;
    if (kind == "ws")
    {
        const long long batch = std::atoll(argv[4]);
        const bool inverse    = std::atoi(argv[5]) != 0;
        const size_t wbytes   = (size_t)std::atoll(argv[6]) << 20;
        const std::vector<char> in = read_file(argv[7]);
        const size_t bytes         = (size_t)batch * n * 2 * sizeof(T);
        if (in.size() != bytes)
            return 2;
        char* din  = static_cast<char*>(std::malloc(bytes));
        char* dout = static_cast<char*>(std::malloc(bytes));
        void* ws   = std::malloc(wbytes);
        std::memcpy(din, in.data(), bytes);
        try
        {
            gpu_dft<T>(n).execute_workspace(dout, din, batch, inverse, nullptr, workspace{ ws, wbytes });
        }
        catch (const std::exception& e)
        {
            std::fprintf(stderr, "error: %s\n", e.what());
            return 3;
        }
        FILE* f = std::fopen(argv[8], "wb");
        if (!f || std::fwrite(dout, 1, bytes, f) != bytes)
            return 4;
        std::fclose(f);
        std::free(din);
        std::free(dout);
        std::free(ws);
        return 0;
    }
    if (kind == "prog")
    {
        const int want     = std::atoi(argv[4]);
        const bool inverse = std::atoi(argv[5]) != 0;
        const std::vector<char> in = read_file(argv[6]);
        const size_t bytes         = n * 2 * sizeof(T);
        if (in.size() != bytes)
            return 2;
        char* d = static_cast<char*>(std::malloc(bytes));
        std::memcpy(d, in.data(), bytes);
        try
        {
            gpu_dft<T> f(n);
            const int units = f.progressive_prepare(want);
            void* mid       = f.progressive_mid_bytes() ? std::malloc(f.progressive_mid_bytes()) : nullptr;
            for (int u = 0; u < units; ++u)
                f.progressive_unit(u, d, mid, inverse, nullptr);
            std::free(mid);
            std::fprintf(stderr, "units=%d\n", units);
        }
        catch (const std::exception& e)
        {
            std::fprintf(stderr, "error: %s\n", e.what());
            return 3;
        }
        FILE* f = std::fopen(argv[7], "wb");
        if (!f || std::fwrite(d, 1, bytes, f) != bytes)
            return 4;
        std::fclose(f);
        std::free(d);
        return 0;
    }
    int fmt        = 1;
    if (kind == "real")
        fmt = std::atoi(argv[a++]);
    const long long batch = std::atoll(argv[a++]);
    const bool inverse    = std::atoi(argv[a++]) != 0;
    if (argc != a + 2)
        return 2;
    const std::vector<char> in = read_file(argv[a]);
    size_t in_bytes = 0, out_bytes = 0;
    const size_t cs = kind == "real" ? (fmt == 1 ? n / 2 + 1 : n / 2) : 0;
    if (kind == "dft")
        in_bytes = out_bytes = (size_t)batch * n * 2 * sizeof(T);
    else if (kind == "dct")
        in_bytes = out_bytes = (size_t)batch * n * sizeof(T);
    else
    {
        in_bytes  = (size_t)batch * (inverse ? cs * 2 : n) * sizeof(T);
        out_bytes = (size_t)batch * (inverse ? n : cs * 2) * sizeof(T);
    }
    if (in.size() != in_bytes)
    {
        std::fprintf(stderr, "input holds %zu bytes, expected %zu\n", in.size(), in_bytes);
        return 2;
    }
    char* din  = static_cast<char*>(std::malloc(in_bytes));
    char* dout = static_cast<char*>(std::malloc(out_bytes));
    std::memcpy(din, in.data(), in_bytes);
    std::memset(dout, 0x7f, out_bytes);
    try
    {
        if (kind == "dft")
            gpu_dft<T>(n).execute(dout, din, batch, inverse, nullptr);
        else if (kind == "dct")
            gpu_dct<T>(n).execute(dout, din, batch, inverse, nullptr);
        else if (inverse)
            gpu_dft_real<T>(n, fmt).inverse(dout, din, batch, nullptr);
        else
            gpu_dft_real<T>(n, fmt).forward(dout, din, batch, nullptr);
    }
    catch (const std::exception& e)
    {
        std::fprintf(stderr, "error: %s\n", e.what());
        return 3;
    }
    FILE* f = std::fopen(argv[a + 1], "wb");
    if (!f || std::fwrite(dout, 1, out_bytes, f) != out_bytes)
        return 4;
    std::fclose(f);
    std::free(din);
    std::free(dout);
    return 0;
}

// one stream through a filter, every call from and into buffers of exactly its samples
template <typename V, typename F>
static int run_filter(F&& f, const char* calls, const char* fin, const char* fout)
{
    const std::vector<char> in = read_file(fin);
    std::vector<V> res;
    size_t pos = 0;
    for (char* p = const_cast<char*>(calls); *p; p += *p == ',' ? 1 : 0)
    {
        const size_t n = std::strtoull(p, &p, 10);
        if ((pos + n) * sizeof(V) > in.size())
            return 2;
        V* din  = static_cast<V*>(std::malloc(n * sizeof(V)));
        V* dout = static_cast<V*>(std::malloc(n * sizeof(V)));
        std::memcpy(din, in.data() + pos * sizeof(V), n * sizeof(V));
        f.process(dout, din, n, nullptr);
        res.insert(res.end(), dout, dout + n);
        std::free(din);
        std::free(dout);
        pos += n;
    }
    FILE* f2 = std::fopen(fout, "wb");
    if (!f2 || std::fwrite(res.data(), sizeof(V), res.size(), f2) != res.size())
        return 4;
    std::fclose(f2);
    return 0;
}

template <typename T>
static int filter_main(bool complex, char** argv)
{
    const size_t nt         = std::strtoull(argv[3], nullptr, 10);
    const std::vector<char> h = read_file(argv[5]);
    if (h.size() != nt * sizeof(T) * (complex ? 2 : 1))
        return 2;
    if (complex)
    {
        struct value
        {
            T re, im;
        };
        return run_filter<value>(gpu_conv_filter_complex<T>(h.data(), nt, 1024), argv[4], argv[6], argv[7]);
    }
    return run_filter<T>(gpu_conv_filter<T>(reinterpret_cast<const T*>(h.data()), nt, 1024), argv[4], argv[6], argv[7]);
}

template <typename T>
static int conv_main(char** argv)
{
    const size_t nx = std::strtoull(argv[3], nullptr, 10), nh = std::strtoull(argv[4], nullptr, 10);
    const long long batch = std::atoll(argv[5]);
    const bool shared     = std::atoi(argv[6]) != 0;
    const size_t xn = batch * nx, hn = (shared ? 1 : batch) * nh, yn = batch * (nx + nh - 1);
    const std::vector<char> in = read_file(argv[7]);
    if (in.size() != (xn + hn + yn) * sizeof(T))
        return 2;
    size_t pos = 0;
    auto take  = [&](size_t n)
    {
        T* p = static_cast<T*>(std::malloc(n * sizeof(T)));
        std::memcpy(p, in.data() + pos * sizeof(T), n * sizeof(T));
        pos += n;
        return p;
    };
    T *x = take(xn), *h = take(hn), *g = take(yn);
    T* out[3]         = {};
    const size_t n[3] = { yn, xn, hn };
    for (int k = 0; k < 3; ++k)
    {
        out[k] = static_cast<T*>(std::malloc(n[k] * sizeof(T)));
        std::memset(out[k], 0x7f, n[k] * sizeof(T));
    }
    gpu_conv<T> c(nx, nh);
    c.forward(out[0], x, h, shared ? 0 : (long long)nh, batch, false, nullptr);
    c.backward(out[1], out[2], g, x, h, shared ? 0 : (long long)nh, batch, false, nullptr);
    FILE* f = std::fopen(argv[8], "wb");
    for (int k = 0; f && k < 3; ++k)
        if (std::fwrite(out[k], sizeof(T), n[k], f) != n[k])
            return 4;
    if (!f)
        return 4;
    std::fclose(f);
    for (T* p : { x, h, g, out[0], out[1], out[2] })
        std::free(p);
    return 0;
}

template <typename T>
static int md_main(char** argv)
{
    std::vector<size_t> shape;
    for (char* p = argv[3]; *p; p += *p == ',' ? 1 : 0)
        shape.push_back(std::strtoull(p, &p, 10));
    const bool real = std::atoi(argv[4]) != 0, inverse = std::atoi(argv[5]) != 0;
    const std::vector<char> in = read_file(argv[6]);
    size_t values = 1;
    for (size_t d : shape)
        values *= d;
    const size_t spectrum = (real ? values / shape.back() * (shape.back() / 2 + 1) : values) * 2 * sizeof(T);
    const size_t ib = real && !inverse ? values * sizeof(T) : spectrum, ob = real && inverse ? values * sizeof(T) : spectrum;
    if (in.size() != ib)
        return 2;
    char* din  = static_cast<char*>(std::malloc(ib));
    char* dout = static_cast<char*>(std::malloc(ob));
    std::memcpy(din, in.data(), ib);
    std::memset(dout, 0x7f, ob);
    if (real)
    {
        gpu_dft_md_real<T> f(shape);
        std::printf("%s\n", f.schedule().c_str());
        if (inverse)
            f.inverse(dout, din, nullptr);
        else
            f.forward(dout, din, nullptr);
    }
    else
    {
        gpu_dft_md<T> f(shape);
        std::printf("%s\n", f.schedule().c_str());
        f.execute(dout, din, inverse, nullptr);
    }
    FILE* f = std::fopen(argv[7], "wb");
    if (!f || std::fwrite(dout, 1, ob, f) != ob)
        return 4;
    std::fclose(f);
    std::free(din);
    std::free(dout);
    return 0;
}

int main(int argc, char** argv)
{
    if (argc < 4)
    {
        std::fprintf(stderr, "usage: emu_main dft|real|dct f32|f64 n [fmt] batch inverse in out\n");
        return 2;
    }
    const std::string kind = argv[1], t = argv[2];
    if (kind == "half")
    {
        if (argc != 8)
            return 2;
        const size_t n        = std::strtoull(argv[3], nullptr, 10);
        const long long batch = std::atoll(argv[4]);
        const bool inverse    = std::atoi(argv[5]) != 0;
        const std::vector<char> in = read_file(argv[6]);
        const size_t bytes         = (size_t)batch * n * 4;
        if (in.size() != bytes)
            return 2;
        char* din  = static_cast<char*>(std::malloc(bytes));
        char* dout = static_cast<char*>(std::malloc(bytes));
        std::memcpy(din, in.data(), bytes);
        try
        {
            pow2_fft<float> f(n, nullptr, t == "bf16" ? 1 : 2);
            f.reserve();
            f.run(inverse, din, dout, batch, nullptr);
        }
        catch (const std::exception& e)
        {
            std::fprintf(stderr, "error: %s\n", e.what());
            return 3;
        }
        FILE* f = std::fopen(argv[7], "wb");
        if (!f || std::fwrite(dout, 1, bytes, f) != bytes)
            return 4;
        std::fclose(f);
        std::free(din);
        std::free(dout);
        return 0;
    }
    if (kind == "filter" && argc == 8)
        return t == "f32" || t == "c32" ? filter_main<float>(t == "c32", argv) : filter_main<double>(t == "c64", argv);
    if (kind == "md" && argc == 8)
        return t == "f64" ? md_main<double>(argv) : md_main<float>(argv);
    if (kind == "conv" && argc == 9)
        return t == "f64" ? conv_main<double>(argv) : conv_main<float>(argv);
    if (kind == "schedule" && argc == 4)
    {
        const size_t n = std::strtoull(argv[3], nullptr, 10);
        std::printf("%s\n", (t == "f64" ? gpu_dft<double>(n).schedule() : gpu_dft<float>(n).schedule()).text().c_str());
        return 0;
    }
    if (kind == "order")
    {
        stream_order ord;
        char* p = argv[2];
        while (*p)
        {
            const auto s = reinterpret_cast<hipStream_t>((uintptr_t)std::strtoull(p, &p, 10));
            ord.run(s, *p == 's', [&] { emu::event_log.push_back("launch " + emu::stream_text(s)); });
            p += p[1] == ',' ? 2 : 1;
        }
        FILE* f = std::fopen(argv[3], "wb");
        if (!f)
            return 2;
        for (const std::string& l : emu::event_log)
            std::fprintf(f, "%s\n", l.c_str());
        std::fclose(f);
        return 0;
    }
    if (kind == "constants")
    {
        const long n = std::atol(argv[3]);
        FILE* f      = argc == 5 ? std::fopen(argv[4], "wb") : nullptr;
        if (!f)
            return 2;
        for (long k = 0; k < n; ++k)
        {
            const double v[2] = { ccos2pi(k, n), csin2pi(k, n) };
            std::fwrite(v, sizeof(v), 1, f);
        }
        std::fclose(f);
        return 0;
    }
    if (kind != "dft" && kind != "real" && kind != "dct" && kind != "prog" && kind != "ws")
        return 2;
    return t == "f64" ? run<double>(kind, argc, argv) : run<float>(kind, argc, argv);
}
