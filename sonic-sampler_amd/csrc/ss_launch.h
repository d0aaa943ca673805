// Host-side launch helpers shared by the entry points.
#pragma once

#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace ss {

// Launches `kernel`; with a (start, end) event pair, the events are recorded by the dispatch
// itself (hipExtLaunchKernelGGL), so they time exactly this kernel and add no packets to the
// stream between it and its neighbours.
template <class Kernel, class... Args>
inline void launch_timed(Kernel kernel, dim3 grid, dim3 block, size_t shared, hipStream_t stream,
                         void *start, void *end, Args... args) {
    if (start && end)
        hipExtLaunchKernelGGL(kernel, grid, block, shared, stream, (hipEvent_t)start, (hipEvent_t)end, 0, args...);
    else
        hipLaunchKernelGGL(kernel, grid, block, shared, stream, args...);
}

// Whether every row of a bf16 plane (or an absent one) starts on a dword.
inline bool half_rows_on_dwords(const void *p, int64_t stride) {
    return !p || ((uintptr_t)p % 4 == 0 && stride % 2 == 0);
}

}  // namespace ss
