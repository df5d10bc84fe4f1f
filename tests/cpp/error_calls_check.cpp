// Host-side check of calls that fail half-way (fake_hip.h in place of the HIP
// library, one of whose calls fails): they return the error, and nothing they
// queued on either stream is left running, as the next call fills the pinned
// rows and scratch that it uses.  Exit status 0 when every check holds.
#include "fake_hip.h"

#include "../../include/solaris_amd.h"
#include "../../solaris_amd/csrc/mesh.h"
#include "../../solaris_amd/csrc/quad.h"

static int g_fails = 0, g_errors = 0;

// `call` with every one of its runtime calls `name` failing in turn.
static void check(const char *what, sol_context *c, const char *name, const std::function<int()> &call)
{
    for (long k = 1; k < 200; ++k) {
        fake::fail_name() = name;
        fake::fail_at() = k;
        const int r = call();
        const bool failed = fake::fail_at() == 0;
        fake::fail_at() = 0;
        if (!failed) {
            if (r != SOL_OK) { std::printf("FAIL %s: %s\n", what, sol_last_error(c)); ++g_fails; }
            return;
        }
        if (r == SOL_OK) { std::printf("FAIL %s: no error from %s %ld\n", what, name, k); ++g_fails; }
        ++g_errors;
        if (fake::pending()) {
            std::printf("FAIL %s: %ld operations left behind by %s %ld\n", what, fake::pending(), name, k);
            ++g_fails;
            for (ihipStream_t *s : fake::streams()) s->done = s->queued;
        }
    }
}

int main()
{
    // a disk whose neighbour search runs on the second stream, and one in quads
    for (int small = 0; small < 2; ++small) {
        sol_nbodies nb{};
        nb.central_body = 1;
        nb.proto_planet = small ? 2 : 9000;
        nb.test_particle = small ? 300 : 0;
        nb.total = 1 + nb.proto_planet + nb.test_particle;
        fake::on_kernel() = [](const std::string &name, void **args) {
            if (name.find("k_quad") == std::string::npos || name.find("k_quad_zero") != std::string::npos) return;
            sol::ResSystem *S = reinterpret_cast<sol::QuadArgs *>(args[0])->system;
            S->status = sol::RES_RUNNING;
            S->steps += 1;
            S->t = S->h_next = S->h_did = 1.0;
        };
        sol_context *c = nullptr;
        if (sol_create(&c, &nb, 0, 0) != SOL_OK) { std::printf("FAIL sol_create\n"); return 1; }
        std::vector<double> one(nb.total, 1.0), y(6 * (size_t)nb.total, 1.0), out(y);
        sol_body_params p{};
        p.mass = p.radius = one.data();
        if (sol_set_bodies(c, &p) || sol_set_state(c, y.data()) || fake::pending()) { std::printf("FAIL set-up\n"); return 1; }
        for (const char *name : {"hipEventRecord", "hipStreamWaitEvent", "hipMemcpyAsync"}) {
            check("sol_compute", c, name, [&] { return sol_compute(c, 0.0, y.data(), out.data()); });
            check("sol_driver", c, name, [&] {
                sol_timeline tl{};
                tl.hNext = 1.0; tl.length = tl.output = 1e9;
                return sol_driver(c, SOL_RUNGE_KUTTA_FEHLBERG78, 1e-9, &tl, nullptr);
            });
            check("sol_step", c, name, [&] { return sol_step(c, SOL_RUNGE_KUTTA4, 0.0, 1.0); });
            check("sol_get_array", c, name, [&] { return sol_get_array(c, SOL_ARRAY_Y0, out.data()); });
            check("sol_set_state", c, name, [&] { return sol_set_state(c, y.data()); });
        }
        sol_destroy(c);
    }
    std::printf("%d errors\n", g_errors);
    if (!g_errors) ++g_fails;
    if (!g_fails) std::printf("error calls: ok\n");
    return g_fails != 0;
}
