// rules_test.cpp -- the rules by which a range of iterations is launched
// (lbmcl_amd/csrc/lbm_range.hpp), asked without a device: this program is host code
// alone and takes the library's functions from liblbm_hip.so.  Exit status 0 when
// every check passes.
#include "lbm_range.hpp"

using namespace lbm_host;

namespace {

int failures = 0;
void check(bool ok, const char* what, long a = 0, long b = 0, long c = 0) {
    if (!ok) {
        std::fprintf(stderr, "FAIL %s (%ld, %ld, %ld)\n", what, a, b, c);
        ++failures;
    }
}

// The third lattice: an eighth of the memory at most, for short ranges what the
// pool keeps, and never more than is free beside it.
void third_lattices() {
    const size_t G = size_t(1) << 30, total = 288 * G;
    check(third_lattice_fits(G, 12, 200 * G, total), "1 GB, much is free");
    check(third_lattice_fits(total / 64, 63, 200 * G, total), "the pool's largest block");
    check(!third_lattice_fits(total / 64 + 1, 63, 200 * G, total), "larger, for a short range");
    check(third_lattice_fits(total / 64 + 1, 64, 200 * G, total), "larger, for a long range");
    check(third_lattice_fits(36 * G, 64, 200 * G, total), "an eighth");
    check(!third_lattice_fits(36 * G + 1, 1000, 200 * G, total), "more than an eighth");
    check(third_lattice_fits(G, 64, 2 * G, total), "as much again is free");
    check(!third_lattice_fits(G, 64, 2 * G - 1, total), "less is free");
}

}  // namespace

int main() {
    third_lattices();
    if (failures) return 1;
    std::printf("all checks passed\n");
    return 0;
}
