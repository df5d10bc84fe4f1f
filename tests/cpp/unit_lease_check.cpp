// Host-side check of the leases of compute units (solaris_amd/csrc/unit_lease.h):
// a large one that waits is served before smaller ones asked for after it, and
// leases that fit side by side are held side by side.  Exit status 0 when every
// check holds.
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <memory>
#include <thread>
#include <vector>

#include "../../solaris_amd/csrc/unit_lease.h"

using namespace sol;

// (threads may still wait: no destructors)
static void fail(const char *what)
{
    std::printf("FAIL %s\n", what);
    std::fflush(stdout);
    std::_Exit(1);
}

static void until(int device, uint64_t asked)
{
    while (UnitLease::asked(device) < asked) std::this_thread::sleep_for(std::chrono::milliseconds(1));
    std::this_thread::sleep_for(std::chrono::milliseconds(50));     // the waiting thread waits
}

int main()
{
    constexpr int kUnits = 256;
    std::mutex m;
    std::vector<int> order;
    auto note = [&](int k) { std::lock_guard<std::mutex> lock(m); order.push_back(k); };
    {
        // one unit held; all of them asked for; then one more
        std::unique_ptr<UnitLease> first(new UnitLease(0, 1, kUnits));
        std::thread large([&] { UnitLease l(0, kUnits, kUnits); note(1); });
        until(0, 2);
        std::thread small([&] { UnitLease l(0, 1, kUnits); note(2); });
        until(0, 3);
        {
            std::lock_guard<std::mutex> lock(m);
            if (!order.empty()) fail("a small lease passed a large one");
        }
        first.reset();
        large.join();
        small.join();
    }
    if (order != std::vector<int>{1, 2}) fail("order of service");
    {
        // more than there are counts as all; side by side; another device is its own
        UnitLease a(1, 100, kUnits), b(1, 156, kUnits), c(2, 1000, kUnits);
        std::thread t([&] { UnitLease d(1, 1, kUnits); note(3); });
        until(1, 3);
        std::lock_guard<std::mutex> lock(m);
        if (order.size() != 2) fail("more units leased than there are");
        t.detach();
    }
    for (int k = 0; k < 1000; ++k) {
        std::this_thread::sleep_for(std::chrono::milliseconds(5));
        std::lock_guard<std::mutex> lock(m);
        if (order.size() == 3) break;
    }
    std::lock_guard<std::mutex> lock(m);
    if (order.size() != 3) fail("a lease given back is not served");
    std::printf("unit leases: ok\n");
    return 0;
}
