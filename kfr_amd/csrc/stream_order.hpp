// The order of one plan's calls across streams.
#pragma once

#include "fft_engine.hpp"

#include <hip/hip_runtime.h>

#include <mutex>

namespace kfr_amd
{

// Calls on one plan run in the order they were made, also on different streams: a call on another
// stream than the plan's last one waits for that stream's work on the plan. That orders the uses of the
// plan's device scratch (four-step intermediates, real and DCT half spectra, Bluestein buffers), and a
// transform on one stream before the one on another that reads its output. Enqueues from several host
// threads are serialised by the mutex, which also guards the lazily grown scratch. Inside a stream
// capture nothing is waited for or recorded (the captured stream orders its own work).
//
// A call is recorded by an event after its launches, and such an event holds back the next launch (4096 x
// 256 f32 forward and back on the default stream: 20.2 us with one after every call, 14.0 without). So
// calls without scratch on a stream that outlives every plan (the default stream and the library's
// own) are recorded only when a call on another stream has to wait for them; on a caller's stream, which may be gone
// by then, at once.
struct stream_order
{
    stream_order() { (void)hipGetDevice(&device); }
    stream_order(const stream_order&) = delete;
    ~stream_order()
    {
        if (ev)
            (void)hipEventDestroy(ev);
    }
    // scratch: fn's work uses the plan's scratch
    template <typename Fn>
    void run(hipStream_t s, bool scratch, Fn&& fn)
    {
        std::lock_guard<std::mutex> lock(mu);
        const bool late = !scratch && (!s || s == library_stream());
        if (late && (!used || last == s))
        {
            fn();
            unrecorded(s);
            return;
        }
        hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
        hip_check(hipStreamIsCapturing(s, &cs), "stream capture status");
        if (cs != hipStreamCaptureStatusNone)
        {
            fn();
            return;
        }
        if (used && last != s)
        {
            if (pending)
                record_pending();
            hip_check(hipStreamWaitEvent(s, ev, 0), "stream ordering");
        }
        fn();
        if (late)
            unrecorded(s);
        else
        {
            record(s);
            last    = s;
            used    = true;
            pending = false;
        }
    }

private:
    std::mutex mu;
    hipEvent_t ev    = nullptr;
    hipStream_t last = nullptr; // stream of the last call
    bool used        = false;
    bool pending     = false; // the last call is not recorded in ev
    int device       = 0;     // the plan's: its calls run with it current

    void unrecorded(hipStream_t s)
    {
        last = s;
        used = pending = true;
    }
    void record(hipStream_t s)
    {
        if (!ev)
            hip_check(hipEventCreateWithFlags(&ev, hipEventDisableTiming), "hipEventCreate");
        hip_check(hipEventRecord(ev, s), "stream ordering");
    }
    // the default stream is one per device
    void record_pending()
    {
        int now = 0;
        hip_check(hipGetDevice(&now), "hipGetDevice");
        if (now != device)
            hip_check(hipSetDevice(device), "hipSetDevice");
        try
        {
            record(last);
        }
        catch (...)
        {
            if (now != device)
                (void)hipSetDevice(now);
            throw;
        }
        if (now != device)
            hip_check(hipSetDevice(now), "hipSetDevice");
        pending = false;
    }
};

} // namespace kfr_amd
