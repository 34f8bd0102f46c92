// Every kernel launch of the library but one goes through HCCLX_LAUNCH, which counts it for the calling host thread
// (hcclx_kernels_launched): the host runtime reports how many kernels a collective took from that count.  The one is
// the upload of a large launch table (upload_table), which stands for a copy and is not counted, as the copy is not.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace hcclx {
inline uint64_t &kernels_launched()
{
    static thread_local uint64_t n = 0;
    return n;
}
}  // namespace hcclx

#define HCCLX_LAUNCH(...)                    \
    do {                                     \
        ++::hcclx::kernels_launched();       \
        hipLaunchKernelGGL(__VA_ARGS__);     \
    } while (0)
