// Host-side check of what runs of an ensemble ask of the runtime (fake_hip.h
// in place of the HIP library; its kernels only count steps): a launch of the
// mesh form, which holds compute units, is cut to about 0.2 s, and each queue's
// launch is captured once and replayed however many systems are left, in the
// next run too.  Exit status 0 when every check holds.
#include "fake_hip.h"

#include "../../include/solaris_amd.h"
#include "../../solaris_amd/csrc/mesh.h"

using namespace sol;

static int g_fails = 0;
static void expect(const char *what, long got, long most)
{
    if (got <= most) return;
    std::printf("FAIL %s: %ld, at most %ld\n", what, got, most);
    ++g_fails;
}

static ResSystem *g_systems = nullptr;      // the ensemble's, on the device
static int g_nsys = 0;
static long g_end = 0, g_longest = 0;       // steps a system takes in all; of the longest mesh launch

static void advance(ResSystem &S, long steps)
{
    if (S.status != RES_RUNNING) return;
    S.steps += steps;
    if (S.steps >= g_end) S.status = RES_DONE;
}

int main()
{
    const int nsys = 20, n = 257;
    g_nsys = nsys;
    fake::on_kernel() = [](const std::string &name, void **args) {
        if (name.find("k_resident_queue") != std::string::npos) {
            g_systems = *reinterpret_cast<ResSystem **>(args[0]);
        } else if (name.find("k_mesh_commit") != std::string::npos) {
            const MeshArgs &A = *reinterpret_cast<MeshArgs *>(args[0]);
            std::memcpy(*reinterpret_cast<ResSystem **>(args[1]), A.systems, g_nsys * sizeof(ResSystem));
        } else if (name.find("k_mesh") != std::string::npos && name.find("k_mesh_zero") == std::string::npos) {
            const MeshArgs &A = *reinterpret_cast<MeshArgs *>(args[0]);
            const int steps = *reinterpret_cast<int *>(args[1]);
            if (steps > g_longest) g_longest = steps;
            for (int k = 0; k < g_nsys; ++k) advance(A.systems[k], steps);
        }
    };
    // the queues' launches: the systems end one after the other
    fake::on_graph() = [] { for (int k = 0; k < g_nsys; ++k) advance(g_systems[k], 16 + k); };
    std::vector<sol_nbodies> nb(nsys);
    for (int k = 0; k < nsys; ++k) {
        nb[k] = sol_nbodies{};
        nb[k].central_body = 1;
        nb[k].total = k == 0 ? 5 : n;          // (one for the narrow queue)
        nb[k].proto_planet = nb[k].total - 1;
    }
    sol_ensemble *e = nullptr;
    if (sol_ensemble_create(&e, nsys, nb.data(), 0) != SOL_OK) { std::printf("FAIL %s\n", sol_ensemble_last_error(nullptr)); return 1; }
    std::vector<double> one(n, 1.0), y(6 * n, 1.0);
    std::vector<int32_t> type(n, 3);
    type[0] = 0;
    sol_body_params p{};
    p.mass = one.data();
    auto set = [&] {
        for (int k = 0; k < nsys; ++k) {
            sol_timeline tl{};
            tl.hNext = 1.0; tl.length = tl.output = 1e9;
            if (sol_ensemble_set_system(e, k, &p, y.data(), &tl)) { std::printf("FAIL %s\n", sol_ensemble_last_error(e)); ++g_fails; }
        }
    };
    set();
    if (sol_ensemble_tune(e, SOL_RUNGE_KUTTA_FEHLBERG78, 1e-10, 8) || !g_systems) { std::printf("FAIL tune\n"); return 1; }
    g_end = 20000;
    if (sol_ensemble_run(e, SOL_RUNGE_KUTTA_FEHLBERG78, 1e-10, 0, nullptr)) { std::printf("FAIL %s\n", sol_ensemble_last_error(e)); return 1; }
    std::printf("longest mesh launch %ld steps\n", g_longest);
    // 13 evaluations of 5 us and 1 ps a pair
    expect("steps of a mesh launch", g_longest, (long)(0.2 / (13 * (5.0e-6 + 1.0e-12 * n * n))));
    if (g_longest == 0) { std::printf("FAIL no mesh launch\n"); ++g_fails; }
    // a run of several launches, twice
    g_end = 300;
    long launches = 0;
    for (int run = 0; run < 2; ++run) {
        fake::forget();
        set();
        if (sol_ensemble_run(e, SOL_RUNGE_KUTTA4, 1e-10, 0, nullptr)) { std::printf("FAIL %s\n", sol_ensemble_last_error(e)); return 1; }
        launches += fake::calls()["hipGraphLaunch"];
        expect(run ? "captures of the second run" : "captures of the first run", fake::calls()["hipGraphInstantiate"], run ? 0 : 2);
    }
    std::printf("%ld graph launches\n", launches);
    if (launches < 8) { std::printf("FAIL few launches\n"); ++g_fails; }
    sol_ensemble_destroy(e);
    if (!g_fails) std::printf("ensemble calls: ok\n");
    return g_fails != 0;
}
