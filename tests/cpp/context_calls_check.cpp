// Host-side check of what creating and destroying a context asks of the
// runtime (fake_hip.h in place of the HIP library): its arrays in a few
// allocations, all given back; a second stream only where the neighbour search
// runs beside a symmetric pair sum, never shared by two contexts, kept for the
// next one; a context's memory and streams on its own device, whichever is
// current when it is called.  Exit status 0 when every check holds.
#include "fake_hip.h"

#include "../../include/solaris_amd.h"

static int g_fails = 0;
static void expect(const char *what, int n, long got, long most)
{
    if (got <= most) return;
    std::printf("FAIL %s, %d bodies: %ld, at most %ld\n", what, n, got, most);
    ++g_fails;
}

static sol_context *make(int planets, int particles, int device = 0)
{
    sol_nbodies nb{};
    nb.central_body = 1;
    nb.proto_planet = planets;
    nb.test_particle = particles;
    nb.total = 1 + planets + particles;
    sol_context *c = nullptr;
    if (sol_create(&c, &nb, 0, device) != SOL_OK) { std::printf("FAIL sol_create: %s\n", sol_last_error(nullptr)); std::exit(1); }
    return c;
}

static void check(int planets, int particles, long allocations, long streams)
{
    const int n = 1 + planets + particles;
    fake::forget();
    sol_context *c = make(planets, particles);
    const long made = fake::calls()["hipMalloc"] + fake::calls()["hipHostMalloc"];
    std::printf("%d bodies: %ld allocations, %ld streams\n", n, made, fake::calls()["hipStreamCreateWithFlags"]);
    expect("allocations", n, made, allocations);
    expect("streams", n, fake::calls()["hipStreamCreateWithFlags"], streams);
    sol_destroy(c);
    expect("allocations left", n, made - fake::calls()["hipFree"] - fake::calls()["hipHostFree"], 0);
    expect("device memory left", n, (long)fake::device_memory().size(), 0);
}

int main()
{
    check(2, 512, 3, 1);
    check(2, 16382, 3, 1);         // few sources: no symmetric sum, no second stream
    check(300, 0, 3, 1);
    check(4000, 0, 5, 1);
    check(9000, 0, 5, 2);
    check(9000, 0, 5, 1);          // the stream of the context before
    {
        fake::forget();
        sol_context *c[7];
        for (sol_context *&x : c) x = make(9000, 0);
        if (fake::calls()["hipStreamCreateWithFlags"] != 7 + 6) { std::printf("FAIL contexts share a stream\n"); ++g_fails; }
        for (sol_context *x : c) sol_destroy(x);
        expect("streams kept", 9001, (long)fake::streams().size(), 4);
    }
    {
        // test particles that become sources: the symmetric sum comes later
        fake::forget();
        sol_context *c = make(2, 9000, 1);
        (void)hipSetDevice(0);
        if (sol_set_source_ranges(c, 9003, 9003) != SOL_OK) { std::printf("FAIL %s\n", sol_last_error(c)); ++g_fails; }
        (void)hipSetDevice(0);
        if (sol_set_precision(c, SOL_PRECISION_MIXED, 0.0) != SOL_OK) { std::printf("FAIL %s\n", sol_last_error(c)); ++g_fails; }
        expect("of a context of device 1 on device 0", 9003, fake::made_on()[0], 0);
        if (fake::calls()["hipStreamCreateWithFlags"] != 2) { std::printf("FAIL no second stream\n"); ++g_fails; }
        (void)hipSetDevice(0);
        sol_destroy(c);
    }
    if (!g_fails) std::printf("context calls: ok\n");
    return g_fails != 0;
}
