// unit_lease.h -- the compute units of a device that launches of this process
// hold while their workgroups wait for each other.
#pragma once

#include <algorithm>
#include <condition_variable>
#include <cstdint>
#include <mutex>

namespace sol {

// The compute units that launches whose workgroups wait for each other (grid,
// mesh and quad form) hold on a device.  Two such launches of this process that
// did not fit side by side could each hold a part of the device and wait for
// the rest, so a launch first takes as many units as it needs, waiting for
// those of the others' launches to end.
//
// Leases are served in the order they are asked for, so that one of many units
// is not passed over by smaller ones for ever.  How long one is held: a launch
// is cut to about 0.2 s of accepted steps at one attempt each; every rejected
// attempt adds its own time to that, and a launch that gives up holds its units
// for its whole wait budget (2 s unless set otherwise) on top.
class UnitLease {
public:
    UnitLease(int device, int units, int total) : d_(pool(device)), units_(std::min(units, total))
    {
        std::unique_lock<std::mutex> lock(d_.m);
        const uint64_t ticket = d_.asked++;
        d_.cv.wait(lock, [&] { return d_.served == ticket && d_.used + units_ <= total; });
        ++d_.served;
        d_.used += units_;
        lock.unlock();
        d_.cv.notify_all();       // the next in turn may fit too
    }
    ~UnitLease()
    {
        {
            std::lock_guard<std::mutex> lock(d_.m);
            d_.used -= units_;
        }
        d_.cv.notify_all();
    }
    UnitLease(const UnitLease &) = delete;
    UnitLease &operator=(const UnitLease &) = delete;
    // Leases asked for on a device so far, the waiting ones among them.
    static uint64_t asked(int device)
    {
        Device &d = pool(device);
        std::lock_guard<std::mutex> lock(d.m);
        return d.asked;
    }

private:
    struct Device {
        std::mutex m;
        std::condition_variable cv;
        int used = 0;
        uint64_t asked = 0, served = 0;
    };
    static Device &pool(int device)
    {
        static Device devices[64];
        return devices[device & 63];
    }
    Device &d_;
    int units_;
};

}  // namespace sol
