// Small device results on the host (fu_mail.h).
#include <string.h>

#include <mutex>
#include <vector>

#include "fu_mail.h"

namespace fu {

namespace {
std::mutex g_lock;
std::vector<std::pair<void*, void*>> g_free;  // (host, device) addresses of idle slots

__global__ __launch_bounds__(256) void k_mail(unsigned* dst, const unsigned* a, int na, const unsigned* b, int nb) {
    for (int i = threadIdx.x; i < na + nb; i += 256) dst[i] = i < na ? a[i] : b[i - na];
}
}  // namespace

Mail::Mail() {
    {
        std::lock_guard<std::mutex> g(g_lock);
        if (!g_free.empty()) {
            host = g_free.back().first;
            dev = g_free.back().second;
            g_free.pop_back();
            return;
        }
    }
    if (hipHostMalloc(&host, kMailBytes, hipHostMallocPortable | hipHostMallocMapped) != hipSuccess ||
        hipHostGetDevicePointer(&dev, host, 0) != hipSuccess) {
        (void)hipGetLastError();
        if (host) (void)hipHostFree(host);
        host = dev = nullptr;
        idle = true;
    }
}
Mail::~Mail() {
    if (!dev || !idle) return;  // a slot that a failed call may still write is never reused
    {
        std::lock_guard<std::mutex> g(g_lock);
        if (g_free.size() < kMailSlots) {
            g_free.push_back({host, dev});
            return;
        }
    }
    (void)hipHostFree(host);
}

int current_device() {
    int d = -1;
    return hipGetDevice(&d) == hipSuccess ? d : -1;
}

hipError_t mail_read(int dev, void* dst0, const void* src0, size_t bytes0, void* dst1, const void* src1, size_t bytes1,
                     hipStream_t s) {
    Mail mail;
    const bool post = mail.dev && bytes0 + bytes1 <= kMailBytes && !((bytes0 | bytes1) & 3) && dev == current_device();
    bool sent = false;
    if (post) {
        hipLaunchKernelGGL(k_mail, dim3(1), dim3(256), 0, s, (unsigned*)mail.dev, (const unsigned*)src0, (int)(bytes0 / 4),
                           (const unsigned*)src1, (int)(bytes1 / 4));
        sent = hipGetLastError() == hipSuccess;  // or an error that an earlier call left
    }
    if (!sent) {
        hipError_t e = hipMemcpyAsync(dst0, src0, bytes0, hipMemcpyDeviceToHost, s);
        if (e == hipSuccess && bytes1) e = hipMemcpyAsync(dst1, src1, bytes1, hipMemcpyDeviceToHost, s);
        const hipError_t es = hipStreamSynchronize(s);
        if (!post || es == hipSuccess) mail.done();
        return e == hipSuccess ? es : e;
    }
    const hipError_t e = hipStreamSynchronize(s);
    if (e != hipSuccess) return e;
    mail.done();
    memcpy(dst0, mail.host, bytes0);
    if (bytes1) memcpy(dst1, (const char*)mail.host + bytes0, bytes1);
    return hipSuccess;
}

}  // namespace fu
