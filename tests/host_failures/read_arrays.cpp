// Pinned staging that cannot be allocated: the error is reported, and a later read of the same
// context allocates it then instead of copying through memory that is not there.
#include "hip_calls.hpp"

using namespace cipc;

static bool read_fails(Context& c, std::vector<double>& host, const std::vector<double>& dev) {
    try {
        read_arrays(c, {{host.data(), dev.data(), host.size() * sizeof(double)}});
    } catch (const Error& e) {
        return e.code == CIPC_ERR_HIP;
    }
    return false;
}

int main() {
    // smaller than a slot, several slots, more than every slot at once
    for (size_t n : {size_t(10), size_t(100000), size_t(2000000)}) {
        std::vector<double> dev(n), host(n);
        for (size_t i = 0; i < n; ++i) dev[i] = (double)i;
        Context c;
        fake::fail_pinned = true;
        bool failed = false;
        try {
            read_arrays_prepare(c, n * sizeof(double));
        } catch (const Error& e) {
            failed = e.code == CIPC_ERR_HIP;
        }
        EXPECT(failed);
        EXPECT(read_fails(c, host, dev));
        fake::fail_pinned = false;
        EXPECT(!read_fails(c, host, dev) && host == dev);
        // an allocation that fails as the slots grow
        Context d;
        read_arrays_prepare(d, 1);
        fake::fail_pinned = true;
        try {
            read_arrays_prepare(d, 1 << 20);
        } catch (const Error&) {
        }
        fake::fail_pinned = false;
        host.assign(n, -1.0);
        EXPECT(!read_fails(d, host, dev) && host == dev);
    }
    return 0;
}
