// stage_test.cpp -- blocking reads (lbmcl_amd/csrc/lbm_stage.hpp) on a runtime of host
// threads: the bytes arrive, behind the work before them, through the staging buffers
// into pageable memory and in one copy into memory that the device reaches itself; a
// copy that fails ends the read with its error; without pinned memory the runtime
// does it.  Exit status 0 when every check passes.
#include <chrono>
#include <cstdio>
#include <vector>

#include "lbm_stage.hpp"

namespace {

int failures = 0;
void check(bool ok, const char* what, size_t bytes) {
    if (!ok) {
        std::fprintf(stderr, "FAIL %s (%zu bytes)\n", what, bytes);
        ++failures;
    }
}

std::vector<char> pattern;

// One read of `bytes` into `to`: its copies, or -1 if the bytes are wrong or late.
long read(lbm_host::HostStage& stage, hipStream_t stream, char* to, size_t bytes) {
    std::vector<char> dev(bytes, 0);
    stream->add([&] {  // the work before the read
        std::this_thread::sleep_for(std::chrono::milliseconds(2));
        std::memcpy(dev.data(), pattern.data(), bytes);
    });
    const long before = host_hip::copies;
    int calls = 0;
    const hipError_t e = stage.copy(0, stream, to, dev.data(), bytes, [&] { ++calls; });
    if (e != hipSuccess || calls != 1) return -1;
    return std::memcmp(to, pattern.data(), bytes) ? -1 : host_hip::copies - before;
}

}  // namespace

int main() {
    host_hip::Stream stream;
    lbm_host::HostStage stage;
    const size_t K = 1024, M = K * K;
    for (size_t i = 0; i < 46 * M; ++i) pattern.push_back(char(i * 7 + i / 4093));
    for (const size_t bytes : {size_t(1), size_t(24), 256 * K - 1, 256 * K + 1, 2 * M, 2 * M + 1, 9 * M + 5, 16 * M, 45 * M + 3}) {
        std::vector<char> pageable(bytes);
        const long staged = read(stage, &stream, pageable.data(), bytes);
        check(staged >= 1, "into pageable memory", bytes);
        check(bytes <= 256 * K || staged > 1, "in pieces", bytes);
        void* p = nullptr;
        if (hipHostMalloc(&p, bytes + 64, 0) != hipSuccess) return 1;
        check(read(stage, &stream, static_cast<char*>(p) + 64, bytes) == 1, "into pinned memory in one copy", bytes);
        (void)hipHostFree(p);
        if (bytes < M) continue;
        for (const long k : {0L, 1L, staged - 1}) {  // a copy fails; the next read is whole again
            host_hip::copies_to_fail = host_hip::copies + k;
            check(read(stage, &stream, pageable.data(), bytes) == -1, "a failed copy is reported", bytes);
            host_hip::copies_to_fail = -1;
            check(read(stage, &stream, pageable.data(), bytes) > 1, "after a failed copy", bytes);
        }
    }
    lbm_host::g_pinned.free();
    host_hip::no_pinned_memory = true;
    std::vector<char> pageable(3 * M);
    check(read(stage, &stream, pageable.data(), 3 * M) == 1, "without pinned memory", 3 * M);
    host_hip::no_pinned_memory = false;
    stage.release();
    if (failures) return 1;
    std::printf("all checks passed\n");
    return 0;
}
