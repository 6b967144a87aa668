// host_stage.hpp -- large host arrays across the boundary, through pinned buffers.
//
// `rows` rows of row_bytes each, contiguous on the device, `pitch` bytes apart on the host.
// An array of at least kStageMin bytes goes through pinned buffers, kStageThreads threads each
// taking pieces of whole rows in turn: while one piece is on the link the others are copied
// between the caller's pageable memory and their buffers (which also faults fresh pages in
// parallel).  Smaller ones, and calls that find the buffers taken by another context's, go
// straight from or to the caller's memory.  The line lies where both directions together gain
// (two fields, us, straight / by pieces): out 115 / 255 at 0.9 MB a field, 330-1050 / 1220 at 2.2,
// 1800 / 1080-1390 at 5.7, 1900-2200 / 1280-1570 at 7.3, 3130 / 1750 at 12.9, 7030 / 2420 at 34
// (what varies is the first touch of the caller's pages); in 95 / 230 at 0.9, 330 / 445 at 4.9,
// 440 / 580 at 7.3, 750 / 865 at 12.9, 1000 / 1090 at 17.2, 2370 / 1960 at 34.  Both ways replace a zeroed std::vector filled by
// the runtime's pageable copy and then copied once more number by number.  Two 17.2 MB arrays
// (rpcf_get_state at 128x129x128): 6.5-8.5 ms -> 1.7 ms; a padded
// field to physical planes (75.8 MB, rpcf_spec_to_phys, which also made four device
// allocations per call): 10.0 -> 3.1 ms.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>

namespace rpcf_host {

constexpr size_t kStageMin = 8u << 20, kStagePiece = 2u << 20;
constexpr int kStageThreads = 6;
inline std::mutex g_stage_mu;    // held while the buffers are in use
inline char* g_stage = nullptr;  // kStageThreads pieces, pinned; freed with the last context
inline std::mutex g_ctx_mu;
inline int g_ctx_count = 0;

inline void stage_ref(int by) {
    std::lock_guard<std::mutex> lk(g_ctx_mu);
    g_ctx_count += by;
    if (g_ctx_count) return;
    std::lock_guard<std::mutex> ls(g_stage_mu);
    if (g_stage) (void)hipHostFree(g_stage);
    g_stage = nullptr;
}

inline void copy_rows(char* dst, size_t dst_pitch, const char* src, size_t src_pitch, size_t rows, size_t row_bytes) {
    if (dst_pitch == row_bytes && src_pitch == row_bytes) memcpy(dst, src, rows * row_bytes);
    else
        for (size_t r = 0; r < rows; r++) memcpy(dst + r * dst_pitch, src + r * src_pitch, row_bytes);
}

// `device` current while it lives (an event belongs to the device that is current when it is
// made), then again the one that was: piece 0 runs on the caller's thread
struct DeviceScope {
    int was = -1;  // to be restored
    hipError_t err;
    explicit DeviceScope(int device) {
        int now;
        err = hipGetDevice(&now);
        if (err != hipSuccess || now == device) return;
        err = hipSetDevice(device);
        if (err == hipSuccess) was = now;
    }
    ~DeviceScope() {
        if (was >= 0) (void)hipSetDevice(was);
    }
    DeviceScope(const DeviceScope&) = delete;
    DeviceScope& operator=(const DeviceScope&) = delete;
};

// the pieces t, t + kStageThreads, .. through buffer t
inline hipError_t stage_pieces(int device, hipStream_t stream, int t, char* dev, char* host, size_t rows,
                               size_t row_bytes, size_t pitch, bool out) {
    const DeviceScope scope(device);
    hipError_t e = scope.err;
    hipEvent_t ev = nullptr;
    if (e == hipSuccess) e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
    if (e != hipSuccess) return e;
    char* buf = g_stage + t * kStagePiece;
    const size_t per = kStagePiece / row_bytes;
    bool pending = false;
    for (size_t r = t * per; r < rows && e == hipSuccess; r += kStageThreads * per) {
        const size_t n = std::min(per, rows - r);
        if (!out) {
            if (pending) e = hipEventSynchronize(ev);  // the buffer's last piece has left
            if (e == hipSuccess) copy_rows(buf, row_bytes, host + r * pitch, pitch, n, row_bytes);
        }
        if (e == hipSuccess)
            e = hipMemcpyAsync(out ? buf : dev + r * row_bytes, out ? dev + r * row_bytes : buf, n * row_bytes,
                               out ? hipMemcpyDeviceToHost : hipMemcpyHostToDevice, stream);
        if (e == hipSuccess) e = hipEventRecord(ev, stream);
        pending = e == hipSuccess;
        if (out && pending) {
            e = hipEventSynchronize(ev);
            if (e == hipSuccess) copy_rows(host + r * pitch, pitch, buf, row_bytes, n, row_bytes);
        }
    }
    if (!out && pending) {
        const hipError_t w = hipEventSynchronize(ev);
        if (e == hipSuccess) e = w;
    }
    (void)hipEventDestroy(ev);
    return e;
}

// *done = false: the caller takes the direct way
inline hipError_t staged_copy(int device, hipStream_t stream, char* dev, char* host, size_t rows, size_t row_bytes,
                              size_t pitch, bool out, bool* done) {
    *done = false;
    if (rows * row_bytes < kStageMin || row_bytes > kStagePiece) return hipSuccess;
    std::unique_lock<std::mutex> lk(g_stage_mu, std::try_to_lock);
    if (!lk.owns_lock()) return hipSuccess;
    if (!g_stage && hipHostMalloc((void**)&g_stage, kStageThreads * kStagePiece, hipHostMallocPortable) != hipSuccess) {
        g_stage = nullptr;
        (void)hipGetLastError();
        return hipSuccess;
    }
    hipError_t err[kStageThreads];
    std::thread th[kStageThreads];
    auto pieces = [&](int t) { err[t] = stage_pieces(device, stream, t, dev, host, rows, row_bytes, pitch, out); };
    for (int t = 1; t < kStageThreads; t++) {
        try {
            th[t] = std::thread(pieces, t);
        } catch (const std::exception&) {  // no thread: its pieces are taken below
        }
    }
    pieces(0);
    for (int t = 1; t < kStageThreads; t++) {
        if (th[t].joinable()) th[t].join();
        else pieces(t);
    }
    *done = true;
    for (hipError_t e : err)
        if (e != hipSuccess) return e;
    return hipSuccess;
}

}  // namespace rpcf_host
