/* qmsg_device.h - device helpers and the launch macro shared by the kernel sources. */
#ifndef QMSG_DEVICE_H
#define QMSG_DEVICE_H

#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>

#include "qmsg_internal.h"
#include "qmsg_libm.h"

/* Launch `kern` on `st`; with a timing hook installed the dispatch stamps its own events. */
#define QLAUNCH(name, kern, grid, block, lds, st, ...)                                          \
    do {                                                                                       \
        hipEvent_t qa_ = nullptr, qb_ = nullptr;                                               \
        if (qmsg::g_launch_timer)                                                              \
            qmsg::g_launch_timer->events(qmsg::g_launch_timer->ctx, (name), &qa_, &qb_);       \
        if (qa_)                                                                               \
            hipExtLaunchKernelGGL(kern, (grid), (block), (lds), (st), qa_, qb_, 0u, __VA_ARGS__); \
        else                                                                                   \
            hipLaunchKernelGGL(kern, (grid), (block), (lds), (st), __VA_ARGS__);              \
    } while (0)

namespace qmsg {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float h2f(uint32_t bits16)
{
    return (float)__builtin_bit_cast(_Float16, (uint16_t)bits16);
}

/* src/model.c:424 */
__device__ __forceinline__ float silu_ref(float a) { return a / (1.0f + qmsg_expf(-a)); }

/* Wait for this wave's LDS accesses only (global loads and DMA still in flight), then the block
 * barrier. The memory clobber keeps the compiler from moving LDS accesses across it. */
__device__ __forceinline__ void mx_lds_barrier()
{
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

}  // namespace qmsg

#endif /* QMSG_DEVICE_H */
