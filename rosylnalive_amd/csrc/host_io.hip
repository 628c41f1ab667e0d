// The few words a call exchanges with the host, as kernels on the device's stream: a copy each way costs a call a stream
// wait and 12-14 us per transfer, however small, and a decode step had eight of them (4 bytes to 136).
//
// k_put_words carries words in its arguments (no staging buffer, nothing to wait for); k_collect writes what the call
// hands back (the fp16 range sites, taken and cleared; the argmax; the persistent step's abort words; the decoded ids) into
// the device's host-visible words, which the host reads once the call's last event has completed.
#include <hip/hip_runtime.h>

#include <cstring>

#include "device.hpp"

namespace lrm {

struct PutWords {
    uint32_t w[Device::kPutWords];
};

static __global__ __launch_bounds__(256) void k_put_words(uint32_t* dst, PutWords p, uint32_t n) {
    for (uint32_t i = threadIdx.x; i < n; i += 256u) dst[i] = p.w[i];
}

static __global__ __launch_bounds__(256) void k_collect(uint32_t* out, uint32_t* range0, uint32_t* range1,
                                                        const uint32_t* argmax, const uint32_t* abort_words,
                                                        const uint32_t* ids, uint32_t nids) {
    const uint32_t t = threadIdx.x;
    if (t < 2) {
        uint32_t* w = t ? range1 : range0;
        uint32_t v = w ? *w : 0u;
        if (v) v = atomicExch(w, 0u);
        out[Device::kHostRange + t] = v;
    } else if (t == 2) {
        out[Device::kHostArgmax] = argmax ? *argmax : 0u;
    } else if (t < 5) {
        out[Device::kHostAbort + t - 3u] = abort_words ? abort_words[t - 3u] : 0u;
    }
    for (uint32_t i = t; i < nids; i += 256u) out[Device::kHostIds + i] = ids[i];
}

void Device::put_words(void* dst, const uint32_t* src, size_t n) {
    hip_check(hipSetDevice(index_), "hipSetDevice");
    for (size_t i = 0; i < n; i += kPutWords) {
        PutWords p;
        const size_t m = n - i < kPutWords ? n - i : kPutWords;
        std::memcpy(p.w, src + i, m * 4);
        hipLaunchKernelGGL(k_put_words, dim3(1), dim3(256), 0, stream_, static_cast<uint32_t*>(dst) + i, p, uint32_t(m));
    }
    hip_check(hipGetLastError(), "k_put_words");
}

void Device::collect(bool range, const void* argmax, const void* abort_words, const void* ids, uint32_t nids) {
    if (nids > kHostIdWords) contract_fail("collect: %u ids", nids);
    hip_check(hipSetDevice(index_), "hipSetDevice");
    hipLaunchKernelGGL(k_collect, dim3(1), dim3(256), 0, stream_, host_words_,
                       static_cast<uint32_t*>(range ? f16_range_[0] : nullptr),
                       static_cast<uint32_t*>(range ? f16_range_[1] : nullptr), static_cast<const uint32_t*>(argmax),
                       static_cast<const uint32_t*>(abort_words), static_cast<const uint32_t*>(ids), nids);
    hip_check(hipGetLastError(), "k_collect");
}

}  // namespace lrm
