// A launch that fails in the middle of a linear solve: the launches before it still write the
// pinned progress words and the vectors, so the solve waits for them before it reports the error
// (the next solve on the context clears the words and would take a late write for its own).
#include "hip_calls.hpp"

using namespace cipc;

static int solve_fails(int preconditioner, int precision, int at) {
    Context c;
    const int V = 100;
    c.sc.V = V; c.sc.S = 1; c.sc.h_voff = {0, V};
    c.mrow.resize(V); c.mcol.resize(V); c.mval.resize(9 * V); c.mptr.resize(4 * V + 2); c.rhs.resize(3 * V);
    fake::launches = fake::in_flight = 0;
    fake::fail_launch = at;
    SolveResult r;
    bool failed = false;
    try {
        linear_solve_scenes(c, precision, preconditioner, 1e-6, 100, nullptr, &r);
    } catch (const Error& e) {
        failed = e.code == CIPC_ERR_HIP;
    }
    fake::fail_launch = -1;
    EXPECT(failed);
    EXPECT(fake::launches > at);
    EXPECT(fake::in_flight == 0);
    // the host polls the progress words while the kernels run: memory that is coherent whatever the
    // environment's default is
    if (c.pin_pcg.p) EXPECT(fake::pinned.at(c.pin_pcg.p) & hipHostMallocCoherent);
    return 0;
}

int main() {
    // every launch of the set-up, the start and the first iterations (six are enqueued before the
    // host looks at the device's progress)
    for (int preconditioner = 0; preconditioner < 2; ++preconditioner)
        for (int at = 0; at < (preconditioner ? 24 : 16); ++at)
            if (solve_fails(preconditioner, 0, at)) {
                std::printf("preconditioner %d, launch %d\n", preconditioner, at);
                return 1;
            }
    return 0;
}
