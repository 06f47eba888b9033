// common.hip -- error plumbing, device buffers and the device-wide scan.
#include "common.hpp"
#include "device_utils.hpp"

#include <cstddef>
#include <mutex>
#include <string>
#include <vector>

namespace tg {

namespace {
thread_local std::string g_last_error;
}

void set_last_error(const std::string& msg) { g_last_error = msg; }
const char* last_error() { return g_last_error.c_str(); }

void throw_hip(hipError_t e, const char* what, const char* file, int line) {
    std::string msg = std::string("HIP error ") + hipGetErrorName(e) + " (" +
                      hipGetErrorString(e) + ") in " + what + " at " + file + ":" +
                      std::to_string(line);
    if (e == hipErrorOutOfMemory || e == hipErrorMemoryAllocation) throw AllocError(msg);
    throw HipError(msg);
}

namespace {

constexpr size_t kKeepBytes = size_t(512) << 20;
constexpr int kMaxDevices = 64;

struct Block {
    void* p;
    size_t bytes;
    hipEvent_t event;  // of the stream that freed it
    bool idle;         // freed with the device idle: no event to wait for
};

struct Blocks {
    std::mutex mu;
    std::vector<Block> list;  // oldest first
    size_t bytes = 0;
};

Blocks& blocks_of(int device) {
    static Blocks* all = new Blocks[kMaxDevices];  // never destroyed: the runtime may go first
    return all[device];
}

void give_back(const Block& b) {
    (void)hipFree(b.p);  // waits for the device
    (void)hipEventDestroy(b.event);
}

// Gives a device's kept blocks back to the driver: whether there were any.
bool give_back_kept(int device) {
    std::vector<Block> old;
    {
        Blocks& bl = blocks_of(device);
        std::lock_guard<std::mutex> lock(bl.mu);
        old.swap(bl.list);
        bl.bytes = 0;
    }
    for (const Block& b : old) give_back(b);
    return !old.empty();
}

// hipMalloc on the current device; where that fails for want of memory that
// the kept blocks hold, once more without them.
hipError_t device_malloc(void** p, size_t bytes) {
    hipError_t e = hipMalloc(p, bytes);
    int device = -1;
    if (e == hipErrorOutOfMemory && hipGetDevice(&device) == hipSuccess && device >= 0 &&
        device < kMaxDevices) {
        (void)hipGetLastError();
        if (give_back_kept(device)) e = hipMalloc(p, bytes);
    }
    if (e != hipSuccess) {
        *p = nullptr;
        (void)hipGetLastError();
    }
    return e;
}

// Sizes of a call vary a little from one to the next: whole 64 KB, or 2 MB.
size_t block_size(size_t bytes) {
    const size_t unit = bytes <= (size_t(1) << 20) ? size_t(64) << 10 : size_t(2) << 20;
    return (bytes + unit - 1) / unit * unit;
}

}  // namespace

void DeviceBuffer::resize(size_t bytes) {
    reset();
    if (bytes == 0) return;
    const hipError_t e = device_malloc(&p_, bytes);
    if (e != hipSuccess)
        throw AllocError("hipMalloc of " + std::to_string(bytes) + " bytes failed: " +
                         hipGetErrorString(e));
    n_ = bytes;
}

void DeviceBuffer::reset() {
    if (p_) (void)hipFree(p_);
    p_ = nullptr;
    n_ = 0;
}

void TempBuffer::allocate(size_t bytes, hipStream_t s) {
    reset();
    if (bytes == 0) return;
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    const bool known = hipStreamIsCapturing(s, &capture) == hipSuccess;
    // a graph would hold an address that is freed when the call returns (a
    // capture in relaxed mode lets hipMalloc and hipFree through)
    require(!known || capture == hipStreamCaptureStatusNone,
            "the stream is being captured and this call allocates its temporaries: pass it a "
            "workspace, or make it outside the capture");
    const bool keep =
        known && hipGetDevice(&device_) == hipSuccess && device_ >= 0 && device_ < kMaxDevices;
    if (!keep) (void)hipGetLastError();
    const size_t want = keep ? block_size(bytes) : bytes;
    if (keep) {
        Blocks& bl = blocks_of(device_);
        Block b{};
        {
            std::lock_guard<std::mutex> lock(bl.mu);
            size_t best = bl.list.size();
            for (size_t i = 0; i < bl.list.size(); ++i)
                if (bl.list[i].bytes >= want && bl.list[i].bytes / 2 <= want &&
                    (best == bl.list.size() || bl.list[i].bytes < bl.list[best].bytes))
                    best = i;
            if (best < bl.list.size()) {
                b = bl.list[best];
                bl.list.erase(bl.list.begin() + static_cast<std::ptrdiff_t>(best));
                bl.bytes -= b.bytes;
            }
        }
        if (b.p != nullptr) {
            hipError_t e = hipSuccess;
            if (!b.idle && hipEventQuery(b.event) != hipSuccess) {
                (void)hipGetLastError();  // not ready
                e = hipStreamWaitEvent(s, b.event, 0);
            }
            if (e != hipSuccess) {
                give_back(b);
                TG_HIP(e);
            }
            p_ = b.p;
            n_ = bytes;
            block_ = b.bytes;
            event_ = b.event;
            stream_ = s;
            return;
        }
        const hipError_t e = hipEventCreateWithFlags(&event_, hipEventDisableTiming);
        if (e != hipSuccess) {
            event_ = nullptr;
            TG_HIP(e);
        }
    }
    const hipError_t e = device_malloc(&p_, want);
    if (e != hipSuccess) {
        if (event_) (void)hipEventDestroy(event_);
        event_ = nullptr;
        throw AllocError("hipMalloc of " + std::to_string(bytes) + " bytes failed: " +
                         hipGetErrorString(e));
    }
    n_ = bytes;
    block_ = keep ? want : 0;
    stream_ = s;
}

void trim_memory() {
    for (int d = 0; d < kMaxDevices; ++d) give_back_kept(d);
}

void TempBuffer::reset() {
    if (p_) {
        const bool ordered =
            block_ > 0 && block_ <= kKeepBytes &&
            (idle_free_ || hipEventRecord(event_, stream_) == hipSuccess);
        if (ordered) {
            std::vector<Block> old;
            {
                Blocks& bl = blocks_of(device_);
                std::lock_guard<std::mutex> lock(bl.mu);
                bl.list.push_back(Block{p_, block_, event_, idle_free_});
                bl.bytes += block_;
                while (bl.bytes > kKeepBytes) {
                    old.push_back(bl.list.front());
                    bl.bytes -= bl.list.front().bytes;
                    bl.list.erase(bl.list.begin());
                }
            }
            for (const Block& b : old) give_back(b);
        } else {
            (void)hipGetLastError();
            (void)hipFree(p_);  // waits for the device
            if (event_) (void)hipEventDestroy(event_);
        }
    }
    p_ = nullptr;
    n_ = block_ = 0;
    stream_ = nullptr;
    event_ = nullptr;
    idle_free_ = false;
}

void PinnedBuffer::reserve(size_t bytes) {
    if (bytes <= n_) return;
    reset();
    hipError_t e = hipHostMalloc(&p_, bytes, hipHostMallocDefault);
    if (e != hipSuccess) {
        p_ = nullptr;
        (void)hipGetLastError();
        throw AllocError("hipHostMalloc of " + std::to_string(bytes) + " bytes failed: " +
                         hipGetErrorString(e));
    }
    n_ = bytes;
}

void PinnedBuffer::reset() {
    if (p_) (void)hipHostFree(p_);
    p_ = nullptr;
    n_ = 0;
}

// ---------------------------------------------------------------------------
// Exclusive scan of int32 counts (tiles of 1024 = 256 threads x 4 items).
// ---------------------------------------------------------------------------
namespace {

constexpr int kScanBlock = 256;
constexpr int kScanItems = 4;
constexpr int kScanTile = kScanBlock * kScanItems;

__global__ __launch_bounds__(kScanBlock) void scan_reduce_kernel(const int32_t* __restrict__ in,
                                                                 int64_t n,
                                                                 int64_t* __restrict__ part) {
    __shared__ int64_t lds[kScanBlock / kWave];
    const int64_t base = static_cast<int64_t>(blockIdx.x) * kScanTile;
    int64_t s = 0;
#pragma unroll
    for (int j = 0; j < kScanItems; ++j) {
        int64_t i = base + static_cast<int64_t>(j) * kScanBlock + threadIdx.x;
        if (i < n) s += in[i];
    }
    s = wave_sum(s);
    if ((threadIdx.x & (kWave - 1)) == 0) lds[threadIdx.x / kWave] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        int64_t t = 0;
        for (int w = 0; w < kScanBlock / kWave; ++w) t += lds[w];
        part[blockIdx.x] = t;
    }
}

// Single workgroup: exclusive scan of part[0..nb) in place, part[nb] = total.
// 256 threads (one wavefront per SIMD): the workgroup fits beside three
// workgroups of the MFMA GEMM on a compute unit, where a 1,024-thread one
// (62 registers x 4 wavefronts per SIMD) waited for the GEMM's last
// workgroups (0.5 ms in a reference-semantics forward, its plans' scans
// beside layer 0's transform).
__global__ __launch_bounds__(kScanBlock) void scan_parts_kernel(int64_t* __restrict__ part,
                                                                int64_t nb) {
    __shared__ int64_t lds[kScanBlock / kWave];
    int64_t carry = 0;
    for (int64_t base = 0; base < nb; base += kScanBlock) {
        int64_t i = base + threadIdx.x;
        int64_t v = (i < nb) ? part[i] : 0;
        int64_t tot;
        int64_t ex = block_exclusive_scan<kScanBlock>(v, lds, &tot);
        if (i < nb) part[i] = carry + ex;
        carry += tot;
    }
    if (threadIdx.x == 0) part[nb] = carry;
}

__global__ __launch_bounds__(kScanBlock) void scan_apply_kernel(const int32_t* __restrict__ in,
                                                                int32_t* __restrict__ out,
                                                                int64_t n,
                                                                const int64_t* __restrict__ part,
                                                                int64_t nb) {
    __shared__ int64_t lds[kScanBlock / kWave];
    const int64_t base = static_cast<int64_t>(blockIdx.x) * kScanTile +
                         static_cast<int64_t>(threadIdx.x) * kScanItems;
    int64_t v[kScanItems];
    int64_t s = 0;
#pragma unroll
    for (int j = 0; j < kScanItems; ++j) {
        int64_t i = base + j;
        v[j] = (i < n) ? in[i] : 0;
        s += v[j];
    }
    int64_t tot;
    int64_t ex = block_exclusive_scan<kScanBlock>(s, lds, &tot) + part[blockIdx.x];
#pragma unroll
    for (int j = 0; j < kScanItems; ++j) {
        int64_t i = base + j;
        if (i < n) out[i] = static_cast<int32_t>(ex);
        ex += v[j];
    }
    if (blockIdx.x == nb - 1 && threadIdx.x == 0) out[n] = static_cast<int32_t>(part[nb]);
}

__global__ void scan_empty_kernel(int32_t* out) { out[0] = 0; }

__global__ __launch_bounds__(256) void fill_i32_kernel(int32_t* __restrict__ p, int64_t n,
                                                       int32_t v) {
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
         i += static_cast<int64_t>(gridDim.x) * blockDim.x)
        p[i] = v;
}

__global__ __launch_bounds__(256) void fill_zero_2d_kernel(float* __restrict__ p, int64_t rows,
                                                           int64_t cols, int64_t ld) {
    const int64_t n = rows * cols;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
         i += static_cast<int64_t>(gridDim.x) * blockDim.x)
        p[(i / cols) * ld + (i % cols)] = 0.0f;
}

unsigned fill_grid(int64_t n) {
    int64_t b = ceil_div(n, 256);
    return static_cast<unsigned>(b < 8192 ? (b > 0 ? b : 1) : 8192);
}

}  // namespace

void fill_i32(int32_t* p, int64_t n, int32_t v, hipStream_t s) {
    if (n <= 0) return;
    fill_i32_kernel<<<fill_grid(n), 256, 0, s>>>(p, n, v);
    TG_LAUNCH_CHECK();
}

void fill_zero_2d(float* p, int64_t rows, int64_t cols, int64_t ld, hipStream_t s) {
    if (rows <= 0 || cols <= 0) return;
    fill_zero_2d_kernel<<<fill_grid(rows * cols), 256, 0, s>>>(p, rows, cols, ld);
    TG_LAUNCH_CHECK();
}

size_t scan_temp_elems(int64_t n) { return static_cast<size_t>(ceil_div(n, kScanTile) + 1); }

void exclusive_scan_i32(const int32_t* in, int32_t* out, int64_t n, int64_t* temp,
                        hipStream_t s) {
    if (n <= 0) {
        scan_empty_kernel<<<1, 1, 0, s>>>(out);
        TG_LAUNCH_CHECK();
        return;
    }
    const int64_t nb = ceil_div(n, kScanTile);
    scan_reduce_kernel<<<static_cast<unsigned>(nb), kScanBlock, 0, s>>>(in, n, temp);
    TG_LAUNCH_CHECK();
    scan_parts_kernel<<<1, kScanBlock, 0, s>>>(temp, nb);
    TG_LAUNCH_CHECK();
    scan_apply_kernel<<<static_cast<unsigned>(nb), kScanBlock, 0, s>>>(in, out, n, temp, nb);
    TG_LAUNCH_CHECK();
}

}  // namespace tg

extern "C" {

const char* tg_last_error(void) { return tg::last_error(); }

int tg_version(void) { return (0 << 16) | 1; }

int tg_trim(void) {
    return tg::guard([] { tg::trim_memory(); });
}

}  // extern "C"
