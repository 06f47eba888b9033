// The memory of calls without a workspace (csrc/common.hpp TempBuffer) over a
// stand-in for the HIP runtime's memory and event calls, which these
// definitions replace in the process: addresses are numbers, never read, and
// an event is pending until the test says otherwise.
#include <cstdio>
#include <map>
#include <set>
#include <stdexcept>
#include <string>
#include <vector>

#include "common.hpp"

namespace {

std::map<void*, size_t> g_live;
size_t g_bytes = 0, g_limit = size_t(1) << 40;
uintptr_t g_next = 0x100000;
std::vector<size_t> g_freed;
std::set<hipEvent_t> g_pending;
std::vector<std::pair<hipStream_t, hipEvent_t>> g_waits;
hipStreamCaptureStatus g_capture = hipStreamCaptureStatusNone;
hipError_t g_device_sync = hipSuccess;
int g_failures = 0;

void expect(bool ok, const char* what) {
    if (ok) return;
    ++g_failures;
    std::printf("FAILED: %s\n", what);
}

}  // namespace

extern "C" {

hipError_t hipMalloc(void** p, size_t n) {
    if (g_bytes + n > g_limit) return hipErrorOutOfMemory;
    *p = reinterpret_cast<void*>(g_next);
    g_next += n + 4096;
    g_live[*p] = n;
    g_bytes += n;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    expect(g_live.count(p) == 1, "hipFree of live memory");
    g_bytes -= g_live[p];
    g_freed.push_back(g_live[p]);
    g_live.erase(p);
    return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceSynchronize(void) { return g_device_sync; }
hipError_t hipHostMalloc(void**, size_t, unsigned) { return hipErrorOutOfMemory; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    *e = reinterpret_cast<hipEvent_t>(g_next++);
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
    g_pending.erase(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
    g_pending.insert(e);
    return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t e) {
    return g_pending.count(e) ? hipErrorNotReady : hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
    g_waits.emplace_back(s, e);
    return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* st) {
    *st = g_capture;
    return hipSuccess;
}

}  // extern "C"

namespace {

const auto kA = reinterpret_cast<hipStream_t>(0xA), kB = reinterpret_cast<hipStream_t>(0xB);
constexpr size_t kMiB = size_t(1) << 20;

// A stream under capture, in any mode: a graph would hold the address of
// memory that is freed when the call returns.
void capture_is_refused() {
    for (auto st : {hipStreamCaptureStatusActive, hipStreamCaptureStatusInvalidated}) {
        g_capture = st;
        std::string msg;
        try {
            tg::TempBuffer t(kMiB, kA);
        } catch (const std::invalid_argument& e) {
            msg = e.what();
        }
        expect(msg.find("workspace") != std::string::npos, "capture refused, naming the workspace");
        expect(g_live.empty(), "capture: nothing allocated");
        tg::TempBuffer none(0, kA);  // a call that needs no memory
        expect(none.get() == nullptr, "capture: no memory, no error");
    }
    g_capture = hipStreamCaptureStatusNone;
    g_freed.clear();
}

// A freed block goes to the next call of its size, behind the stream that
// freed it; the oldest go back to the driver past 512 MiB.
void blocks_are_reused() {
    void* p;
    {
        tg::TempBuffer t(3 * kMiB, kA);
        p = t.get();
    }
    expect(g_freed.empty(), "kept");
    {
        tg::TempBuffer t(3 * kMiB, kB);
        expect(t.get() == p, "reused");
        expect(g_waits.size() == 1 && g_waits[0].first == kB, "the new stream waits for the old");
        g_pending.clear();
    }
    g_pending.clear();
    {
        tg::TempBuffer t(3 * kMiB, kA);
        expect(t.get() == p && g_waits.size() == 1, "no wait for an event that has passed");
        tg::TempBuffer u(3 * kMiB, kA);
        expect(u.get() != p, "not two users of one block");
    }
    {
        tg::TempBuffer a(300 * kMiB, kA), b(300 * kMiB, kA);
    }
    expect(g_bytes <= 512 * kMiB, "at most 512 MiB kept");
    g_waits.clear();
}

// Kept blocks are no reason for another allocation of the library to fail, and
// a program can have them back.
void kept_blocks_are_given_back() {
    expect(g_bytes > 100 * kMiB, "some memory kept");
    g_limit = g_bytes + kMiB;
    {
        tg::DeviceBuffer d;
        bool failed = false;
        try {
            d.resize(64 * kMiB);
        } catch (const tg::AllocError&) {
            failed = true;
        }
        expect(!failed, "a plan's allocation takes the kept memory back");
        try {
            d.resize(g_limit + kMiB);
        } catch (const tg::AllocError&) {
            failed = true;
        }
        expect(failed && d.get() == nullptr && d.size() == 0, "one that cannot be met fails");
    }
    {
        tg::TempBuffer t(8 * kMiB, kA);
    }
    expect(g_bytes == 8 * kMiB, "kept");
    expect(tg_trim() == TG_OK && g_bytes == 0 && g_live.empty(), "given back on request");
}

// A CSV handle's memory is kept, without an event, once its device is idle;
// where the device cannot be waited for it goes to the driver.  (Opening fails
// here at the pinned staging buffers, after the file's memory.)
void handles_wait_for_the_device(const char* file) {
    for (bool idle : {true, false}) {
        g_device_sync = idle ? hipSuccess : hipErrorStreamCaptureUnsupported;
        g_freed.clear();
        tg_csv_t csv = nullptr;
        expect(tg_csv_open(file, &csv, nullptr) == TG_ERR_ALLOC && csv == nullptr, "open fails");
        expect(g_freed.empty() == idle, idle ? "kept when idle" : "to the driver when not");
        expect(tg_trim() == TG_OK && g_live.empty(), "nothing left");
    }
    g_device_sync = hipSuccess;
}

}  // namespace

int main(int, char** argv) {
    capture_is_refused();
    blocks_are_reused();
    kept_blocks_are_given_back();
    handles_wait_for_the_device(argv[0]);
    std::printf(g_failures ? "%d failed\n" : "ok\n", g_failures);
    return g_failures != 0;
}
