// One body's state packed for the host, in one launch.
//
// A read-back asks for up to six arrays of a body; a copy each, the error flag's and the body
// states' cost 10 to 15 us of launch and wait apiece, whatever the body's size (139 us for a body of
// 1,024 vertices, measured with the update idle).  This kernel writes everything the call needs
// straight into pinned host memory, already in the caller's layout, so a read is one launch, one
// wait and plain memory copies (about 25 us).  Bound by the launch for small bodies and by the bus for
// large ones: consecutive lanes write consecutive words, so stores leave as whole lines.
#include "xpbd_device.h"

namespace xpbd {

// out: ReadHeader, then the requested arrays one after the other (pos, prev, vel: 3 floats per
// vertex, plane: 4, idx, contact: 1 int); a null source is not wanted.
__global__ __launch_bounds__(256) void readback_kernel(ReadSources s, uint32_t nv, ReadHeader *header, uint32_t *out)
{
    const uint32_t t = blockIdx.x * 256u + threadIdx.x, stride = gridDim.x * 256u;
    if (t == 0)
    {
        header->error = *s.error;
        if (s.state)
            header->state = *s.state;
    }
    uint32_t base = 0;
    for (int a = 0; a < 3; ++a)
    {
        const float4 *src = a == 0 ? s.x : a == 1 ? s.prev : s.v;
        if (!src)
            continue;
        const uint32_t *words = reinterpret_cast<const uint32_t *>(src);
        for (uint32_t k = t; k < 3u * nv; k += stride)
            out[base + k] = words[k + k / 3u];
        base += 3u * nv;
    }
    if (s.plane)
    {
        const uint32_t *words = reinterpret_cast<const uint32_t *>(s.plane);
        for (uint32_t k = t; k < 4u * nv; k += stride)
            out[base + k] = words[k];
        base += 4u * nv;
    }
    for (int a = 0; a < 2; ++a)
    {
        const int32_t *src = a == 0 ? s.idx : s.contact;
        if (!src)
            continue;
        for (uint32_t k = t; k < nv; k += stride)
            out[base + k] = (uint32_t)src[k];
        base += nv;
    }
}

hipError_t launch_readback(const ReadSources &s, uint32_t nv, ReadHeader *header, uint32_t *out, hipStream_t stream)
{
    const uint32_t blocks = nv * 3u < 256u ? 1u : nv * 3u / 256u < 512u ? (nv * 3u + 255u) / 256u : 512u;
    hipLaunchKernelGGL(readback_kernel, dim3(blocks), dim3(256), 0, stream, s, nv, header, out);
    return hipGetLastError();
}

} // namespace xpbd
