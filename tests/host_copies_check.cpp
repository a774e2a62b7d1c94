// Copies between the caller's host arrays and the device (host_copies) against a stand-in for the HIP calls they make:
// device memory is host memory, and the caller's own work on the null stream is done when that stream is waited for.
#include "../shiokaze_amd/csrc/shkz_runtime.hip"
#include "host_hip.hpp"

#include <chrono>
#include <cstdio>

static std::function<void()> null_stream_work;
static void wait_null_stream() {
    if (null_stream_work) std::exchange(null_stream_work, nullptr)();
}

extern "C" {
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
    static char streams[64];
    static int n;
    *s = (hipStream_t)&streams[n++];
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
    if (!s) wait_null_stream();
    return hipSuccess;
}
hipError_t hipMemcpy(void *dst, const void *src, size_t n, hipMemcpyKind) {
    wait_null_stream();
    std::memcpy(dst, src, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t n, hipMemcpyKind, hipStream_t) {
    if (*(const char *)src == 's') std::this_thread::sleep_for(std::chrono::milliseconds(20));  // a slow copy
    std::memcpy(dst, src, n);
    return hipSuccess;
}
}

// Allocations left before one fails (-1: none does).
static std::atomic<int> allocations_left{-1};
void *operator new(size_t n) {
    if (allocations_left >= 0 && allocations_left-- == 0) throw std::bad_alloc();
    return std::malloc(n);
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

// The caller's arrays are still being written by its own work on the null stream when it calls.
static bool after_null_stream(size_t bytes, hipMemcpyKind kind) {
    shkz_ctx C;
    std::vector<char> src(bytes, 'a'), other(100, 'a'), dst(bytes, 'x'), dst2(100, 'x');
    null_stream_work = [&]() {
        std::fill(src.begin(), src.end(), 'b');
        std::fill(other.begin(), other.end(), 'c');
    };
    const int rc = host_copies(&C, {{dst.data(), src.data(), bytes}, {dst2.data(), other.data(), other.size()}}, kind);
    null_stream_work = nullptr;
    return rc == SHKZ_OK && dst == std::vector<char>(bytes, 'b') && dst2 == std::vector<char>(100, 'c');
}

// Two grids of a batch share an output array, whole or in part: the last one's values stay.
static bool last_of_overlapping(size_t bytes, size_t offset) {
    shkz_ctx C;
    std::vector<char> first(bytes, 's'), last(bytes, 'b'), dst(offset + bytes, 'x'), want(dst);
    std::fill_n(want.begin(), bytes, 's');
    std::fill_n(want.begin() + (ptrdiff_t)offset, bytes, 'b');
    const int rc = host_copies(&C, {{dst.data(), first.data(), bytes}, {dst.data() + offset, last.data(), bytes}},
                               hipMemcpyDeviceToHost);
    return rc == SHKZ_OK && dst == want;
}

// Each allocation of a call fails in turn: the call copies everything with fewer threads, or ends with the exception,
// never with the process.
static bool short_of_memory() {
    bool ok = true;
    int copied = 0;
    for (int left = 0;; ++left) {
        shkz_ctx C;
        std::vector<char> src(2 * COPY_PARALLEL, 'b'), dst(src.size(), 'x');
        const std::vector<HostCopy> copies{{dst.data(), src.data(), src.size()}};
        allocations_left = left;
        try {
            const int rc = host_copies(&C, copies, hipMemcpyHostToDevice);
            const bool reached = allocations_left < 0;
            allocations_left = -1;
            ok = ok && rc == SHKZ_OK && dst == src;
            if (!reached) break;  // fewer allocations than that
            ++copied;
        } catch (const std::bad_alloc &) {
            allocations_left = -1;
        }
    }
    return ok && copied > 0;
}

int main(int, char **argv) {
    const std::string what = argv[1];
    bool ok = true;
    if (what == "null-stream")
        for (size_t bytes : {COPY_PARALLEL / 2, COPY_PARALLEL, 5 * COPY_PARALLEL / 2 + 17})
            for (hipMemcpyKind kind : {hipMemcpyHostToDevice, hipMemcpyDeviceToHost}) {
                const bool good = after_null_stream(bytes, kind);
                if (!good) std::printf("%zu bytes, kind %d: the arrays as they were before\n", bytes, (int)kind);
                ok = ok && good;
            }
    if (what == "overlap")
        for (size_t bytes : {COPY_PARALLEL / 4, 6 * COPY_PIECE})
            for (size_t offset : {(size_t)0, bytes / 2, bytes}) {
                const bool good = last_of_overlapping(bytes, offset);
                if (!good) std::printf("%zu bytes at %zu: values of the copy before\n", bytes, offset);
                ok = ok && good;
            }
    if (what == "memory") ok = short_of_memory();
    if (ok) std::printf("OK\n");
    return ok ? 0 : 1;
}
