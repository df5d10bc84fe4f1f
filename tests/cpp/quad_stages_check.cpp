// Host-side check of the stage derivatives of the quad form
// (solaris_amd/csrc/quad_stages.h): clearing a thread's column and writing
// every row of it stays inside the columns the host allots, for the rows of
// every integrator and the workgroups of 64 and 128 places, and every row of
// every thread keeps a place of its own.  Exit status 0 when every check holds.
#include <cstdio>
#include <vector>

#include "../../solaris_amd/csrc/quad_stages.h"

using namespace sol;

static const double kMark = -7.25;

template <int ROWS>
static int check(int places)
{
    const int threads = 4 * places;
    const size_t len = quad_column_bytes(ROWS, threads) / sizeof(double), guard = 64 * (size_t)threads;
    std::vector<double> lds(len + guard, kMark);
    auto column = [&](int t) {
        QStages<ROWS, true> d;
        d.col = lds.data() + t;
        d.stride = threads;
        return d;
    };
    for (int t = 0; t < threads; ++t) column(t).clear();
    size_t past = 0;
    for (size_t q = len; q < lds.size(); ++q) past += lds[q] != kMark;
    for (size_t q = 0; q < len; ++q)
        if (lds[q] != 0.0) { std::printf("FAIL rows %d, places %d: word %zu not cleared\n", ROWS, places, q); return 1; }
    if (past) { std::printf("FAIL rows %d, places %d: %zu words past the columns\n", ROWS, places, past); return 1; }
    for (int t = 0; t < threads; ++t)
        for (int l = 0; l < ROWS; ++l) column(t).put(l, 1.0 + 2.0 * (l * threads + t), 2.0 + 2.0 * (l * threads + t));
    for (int t = 0; t < threads; ++t)
        for (int l = 0; l < ROWS; ++l)
            if (column(t).V(l) != 1.0 + 2.0 * (l * threads + t) || column(t).F(l) != 2.0 + 2.0 * (l * threads + t)) {
                std::printf("FAIL rows %d, places %d: thread %d, row %d\n", ROWS, places, t, l);
                return 1;
            }
    for (size_t q = len; q < lds.size(); ++q)
        if (lds[q] != kMark) { std::printf("FAIL rows %d, places %d: written past the columns\n", ROWS, places); return 1; }
    return 0;
}

int main()
{
    for (int places : {16, 64, 128})
        // RKF78, Dormand-Prince, RK4
        if (check<13>(places) || check<9>(places) || check<4>(places)) return 1;
    std::printf("quad stages: ok\n");
    return 0;
}
