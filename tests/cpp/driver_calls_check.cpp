// Host-side check of what a single Driver call asks of the runtime
// (fake_hip.h in place of the HIP library): no more copies, launches and
// questions than the one-workgroup form it took the place of (one copy of the
// descriptor each way, one kernel), for small systems in quads, with one
// workgroup and several, and on the mesh.  Exit status 0 when every check holds.
#include "fake_hip.h"

#include "../../include/solaris_amd.h"
#include "../../solaris_amd/csrc/mesh.h"
#include "../../solaris_amd/csrc/quad.h"

using namespace sol;

static int g_fails = 0;
static void expect(const char *what, long got, long most)
{
    if (got <= most) return;
    std::printf("FAIL %s: %ld, at most %ld\n", what, got, most);
    ++g_fails;
}

// The driver kernels take one step.
static void one_step(ResSystem *S)
{
    S->status = RES_RUNNING;
    S->steps += 1;
    S->attempts += 1;
    S->t = 1.0;
    S->h_did = S->h_next = S->body_h = 1.0;
}

static void check(int planets, int particles, int integrator, long zeroings)
{
    sol_nbodies nb{};
    nb.central_body = 1;
    nb.proto_planet = planets;
    nb.test_particle = particles;
    nb.total = 1 + planets + particles;
    sol_context *c = nullptr;
    if (sol_create(&c, &nb, 0, 0) != SOL_OK) { std::printf("FAIL sol_create: %s\n", sol_last_error(nullptr)); ++g_fails; return; }
    std::vector<double> one(nb.total, 1.0), y(6 * (size_t)nb.total, 1.0);
    sol_body_params p{};
    p.mass = p.radius = one.data();
    if (sol_set_bodies(c, &p) || sol_set_state(c, y.data())) { std::printf("FAIL set-up\n"); ++g_fails; }
    auto call = [&] {
        sol_timeline tl{};
        tl.hNext = 1.0; tl.length = 1e9; tl.output = 1e9;
        if (sol_driver(c, integrator, 1e-9, &tl, nullptr)) { std::printf("FAIL driver: %s\n", sol_last_error(c)); ++g_fails; }
    };
    fake::forget();
    call();
    expect("allocations of the first call", fake::calls()["hipMalloc"] + fake::calls()["hipHostMalloc"], 1);
    fake::forget();
    call();
    std::printf("%d planets, %d particles, integrator %d: %ld copies to the device, %ld back, %ld kernels\n", planets,
                particles, integrator, fake::calls()["to device"], fake::calls()["to host"], fake::calls()["hipLaunchKernel"]);
    expect("copies to the device", fake::calls()["to device"], 1);
    expect("copies back", fake::calls()["to host"], 1);
    expect("launches", fake::calls()["hipLaunchKernel"], 1 + zeroings);
    expect("allocations", fake::calls()["hipMalloc"] + fake::calls()["hipHostMalloc"], 0);
    expect("questions for the occupancy", fake::calls()["hipOccupancyMaxActiveBlocksPerMultiprocessor"], 0);
    expect("attributes set", fake::calls()["hipFuncSetAttribute"], 0);
    if (fake::pending()) { std::printf("FAIL work left behind\n"); ++g_fails; }
    sol_destroy(c);
}

int main()
{
    fake::on_kernel() = [](const std::string &name, void **args) {
        if (name.find("k_quad_zero") != std::string::npos || name.find("k_mesh_zero") != std::string::npos) return;
        if (name.find("k_quad") != std::string::npos) {
            one_step(reinterpret_cast<QuadArgs *>(args[0])->system);
        } else if (name.find("k_mesh") != std::string::npos) {
            one_step(reinterpret_cast<MeshArgs *>(args[0])->systems);
        }
    };
    for (int integrator : {SOL_RUNGE_KUTTA_FEHLBERG78, SOL_RUNGE_KUTTA4, SOL_DORMAND_PRINCE}) {
        check(2, 1, integrator, 0);                                              // a workgroup of quads
        check(2, 512, integrator, integrator == SOL_RUNGE_KUTTA4 ? 0 : 1);       // ten, which exchange words
        check(40, 0, integrator, 0);                                             // mesh
    }
    if (!g_fails) std::printf("driver calls: ok\n");
    return g_fails != 0;
}
