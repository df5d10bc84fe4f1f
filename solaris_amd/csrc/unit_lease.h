// unit_lease.h -- the compute units of a device that launches of this process
// hold while their workgroups wait for each other.
#pragma once

#include <algorithm>
#include <condition_variable>
#include <mutex>

namespace sol {

// The compute units that launches whose workgroups wait for each other (grid
// and mesh form) hold on a device.  Two such launches of this process that
// did not fit side by side could each hold a part of the device and wait for
// the rest, so a launch first takes as many units as it needs, waiting for
// those of the others' launches to end (each at most about 0.2 s).
class UnitLease {
public:
    UnitLease(int device, int units, int total) : d_(pool(device)), units_(std::min(units, total))
    {
        std::unique_lock<std::mutex> lock(d_.m);
        d_.cv.wait(lock, [&] { return d_.used + units_ <= total; });
        d_.used += units_;
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

private:
    struct Device {
        std::mutex m;
        std::condition_variable cv;
        int used = 0;
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
