// The host side of the ABI: packed host arrays (x, y, z triples and masses)
// and their way to and from the device's 32-B rows.
//
// Bounds: the link to the host.  One kernel reads or writes the pinned host
// arrays directly, a double per lane in the host's order, so the link sees
// whole lines and the rows are packed on the way; nothing is staged, neither
// on the host nor on the device.  A 48 MB array takes 0.89 ms out and 0.85 ms
// in (54 and 57 GB/s; packing into device memory and a DMA copy: 0.87 and
// 0.88 ms, at 20 KB 19 us instead of 13).  Before, rows were packed by one
// host thread and copied through pageable memory: 80^3 cells (2,048,000
// atoms, and 267,000 ghosts on the way out) took 51 ms in and 62 ms out, now 2.1
// and 3.5 where the pinned arrays have been in use before; 864 atoms 60 and 160
// us, now 20 and 20.  Fresh pinned pages cost the first simulation more: create,
// upload, read and close at 80^3 together 35 ms, where it was 137 (a process's
// first: 39 and 198).
#include <algorithm>
#include <cstring>
#include <thread>

#include "tmd_internal.hpp"

namespace tmd {

void HostBuf::reserve(size_t need, size_t keep) {
    if (need <= doubles) return;
    double* np = nullptr;
    bool pin = true;
    if (hipHostMalloc(reinterpret_cast<void**>(&np), need * sizeof(double)) != hipSuccess) {
        // no more memory may be pinned: ordinary pages, and staged copies
        (void)hipGetLastError();
        pin = false;
        np = static_cast<double*>(std::malloc(need * sizeof(double)));
        if (!np) {
            set_error(__FILE__, __LINE__, "out of host memory");
            return;
        }
    }
    if (keep) std::memcpy(np, p, keep * sizeof(double));
    release();
    p = np;
    doubles = need;
    pinned = pin;
}

void HostBuf::release() {
    if (p && pinned) (void)hipHostFree(p);
    else std::free(p);
    p = nullptr;
    doubles = 0;
}

void HostAtoms::reserve(int atoms) {
    if (atoms <= cap) return;
    HostBuf old = buf;
    buf = HostBuf{};
    buf.reserve(10 * (size_t)atoms);
    if (!buf.p) {
        buf = old;
        return;
    }
    const size_t c = (size_t)cap, k = (size_t)count;
    double* const from[4] = {old.p, old.p + 3 * c, old.p + 6 * c, old.p + 9 * c};
    cap = atoms;
    double* const to[4] = {pos(), vel(), force(), mass()};
    for (int a = 0; a < 4 && k; ++a)
        if (a != 2 || !no_force) std::memcpy(to[a], from[a], sizeof(double) * (a < 3 ? 3 : 1) * k);
    old.release();
}

void HostAtoms::release() {
    buf.release();
    cap = count = 0;
    no_force = true;
}

// a.host[t] <-> component t % width of row t / width, zero beyond `have`
struct TransferArgs {
    HostArray a[kHostArrays];
};
template <bool OUT>
__global__ void __launch_bounds__(256) k_transfer(TransferArgs x) {
    const HostArray a = x.a[blockIdx.y];
    const size_t step = (size_t)gridDim.x * blockDim.x;
    for (size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x; t < a.count; t += step) {
        size_t d = t;
        if (a.width == 3) {
            const size_t i = t / 3;
            d = t + i;  // 4 i + t % 3
            if (!OUT && t - 3 * i == 2) a.dev[d + 1] = 0.0;
        }
        if (OUT) a.host[t] = t < a.have ? a.dev[d] : 0.0;
        else a.dev[d] = t < a.have ? a.host[t] : 0.0;
    }
}

template <bool OUT>
static void launch_transfer(const TransferArgs& x, int na, hipStream_t st) {
    size_t most = 0;
    for (int k = 0; k < na; ++k) most = std::max(most, x.a[k].count);
    if (most == 0) return;
    // 1,024 blocks an array keep the link full
    hipLaunchKernelGGL(k_transfer<OUT>, dim3((unsigned)std::min<size_t>((most + 255) / 256, 1024), na), dim3(256), 0, st, x);
    TMD_HIP(hipGetLastError());
}

template <bool OUT>
static void transfer(const HostArray* a, int na, bool pinned, hipStream_t st) {
    TransferArgs x{};
    for (int k = 0; k < na; ++k) x.a[k] = a[k];
    if (pinned) {
        launch_transfer<OUT>(x, na, st);
        return;
    }
    // host memory that the device cannot reach: packed on the device, copied
    // an array at a time
    DevBuf stage;
    for (int k = 0; k < na && !has_error(); ++k) {
        if (a[k].count == 0) continue;
        const size_t bytes = sizeof(double) * a[k].count, have = sizeof(double) * std::min(a[k].have, a[k].count);
        stage.reserve(bytes, false, st);
        if (has_error()) break;
        TransferArgs y{};
        y.a[0] = a[k];
        y.a[0].host = stage.as<double>();
        if (!OUT && have) TMD_HIP(hipMemcpyAsync(stage.p, a[k].host, have, hipMemcpyHostToDevice, st));
        launch_transfer<OUT>(y, 1, st);
        if (OUT) TMD_HIP(hipMemcpyAsync(a[k].host, stage.p, bytes, hipMemcpyDeviceToHost, st));
        TMD_HIP(hipStreamSynchronize(st));
    }
    stage.release();
}

void to_host(const HostArray* a, int na, bool pinned, hipStream_t st) { transfer<true>(a, na, pinned, st); }
void to_device(const HostArray* a, int na, bool pinned, hipStream_t st) { transfer<false>(a, na, pinned, st); }

// The user's arrays to and from the pinned ones.  One thread copies 48 MB in
// 1.8 ms, and in 4.5 ms (large pages) to 10.6 ms (small ones) where the
// target's pages are touched for the first time; four take 0.5, 1.1 and 3.7,
// eight 0.5, 1.0 and 2.1.  A thread costs about 20 us: each gets 2 MiB or more.
void host_copy(std::initializer_list<HostSpan> spans) {
    constexpr int kCopyThreads = 8;
    size_t total = 0;
    for (const HostSpan& s : spans) total += s.bytes;
    const size_t cores = std::max(1u, std::thread::hardware_concurrency() / 2);
    const int nt = (int)std::max<size_t>(1, std::min({(size_t)kCopyThreads, cores, total >> 21}));
    auto part = [&spans](size_t lo, size_t hi) {  // bytes [lo, hi) of the spans laid end to end
        size_t at = 0;
        for (const HostSpan& s : spans) {
            const size_t a = std::max(lo, at), b = std::min(hi, at + s.bytes);
            if (a < b) {
                char* to = static_cast<char*>(s.to) + (a - at);
                if (s.from) std::memcpy(to, static_cast<const char*>(s.from) + (a - at), b - a);
                else std::memset(to, 0, b - a);
            }
            at += s.bytes;
        }
    };
    std::thread th[kCopyThreads];
    const size_t each = (total / nt + 4095) & ~(size_t)4095;
    for (int k = 1; k < nt; ++k) {
        const size_t lo = std::min(total, k * each), hi = k + 1 < nt ? std::min(total, lo + each) : total;
        try {
            th[k] = std::thread(part, lo, hi);
        } catch (...) {
            part(lo, hi);  // no thread to be had
        }
    }
    part(0, nt > 1 ? std::min(total, each) : total);
    for (std::thread& t : th)
        if (t.joinable()) t.join();
}

}  // namespace tmd
