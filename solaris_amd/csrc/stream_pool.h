// stream_pool.h -- the second streams of contexts, kept for the next context.
//
// Making and destroying one takes 50 us of a context's 540 (disk of 16,385
// bodies), so up to kKept idle ones per device stay for the rest of the process.
// A stream belongs to one context at a time and comes back idle.
#pragma once

#include <mutex>
#include <vector>

#include <hip/hip_runtime_api.h>

namespace sol {

class StreamPool {
public:
    static hipError_t take(int device, hipStream_t *s)
    {
        {
            Device &d = of(device);
            std::lock_guard<std::mutex> lock(d.m);
            if (!d.idle.empty()) {
                *s = d.idle.back();
                d.idle.pop_back();
                return hipSuccess;
            }
        }
        return hipStreamCreateWithFlags(s, hipStreamNonBlocking);
    }
    // Waits for the stream.  One that cannot be waited for is not kept.
    static void give_back(int device, hipStream_t s)
    {
        if (hipStreamSynchronize(s) == hipSuccess) {
            Device &d = of(device);
            std::lock_guard<std::mutex> lock(d.m);
            if (d.idle.size() < kKept) {
                d.idle.push_back(s);
                return;
            }
        }
        (void)hipStreamDestroy(s);
    }

private:
    static constexpr size_t kKept = 4;
    struct Device {
        std::mutex m;
        std::vector<hipStream_t> idle;
    };
    static Device &of(int device)
    {
        // never destroyed: a context may end after this library's statics would
        static Device *devices = new Device[64];
        return devices[device & 63];
    }
};

}  // namespace sol
