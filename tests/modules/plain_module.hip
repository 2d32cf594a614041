// plain_module.hip — a fractal module with the ABI's kernels and no others, each in the
// reference's geometry: 32 x 32-thread blocks, one thread a pixel.  Its images name their
// pixels: record (x, y) has the value x + y * width, and compose colours it with
// palette[0] + value.
#include "../../chaos-ultra_amd/csrc/kernels/cu_types.hpp"

extern "C" {
__device__ unsigned long long cu_iteration_slots[CU_ITER_SLOTS];
__device__ bool VISUALIZE_SAMPLE_COUNT;
}

__device__ __forceinline__ Point<uint> pixel() {
    return {blockIdx.x * blockDim.x + threadIdx.x, blockIdx.y * blockDim.y + threadIdx.y};
}

__device__ void name_pixel(pixel_info_t *out, long pitch, Point<uint> size) {
    const Point<uint> p = pixel();
    if (p.x >= size.x || p.y >= size.y) return;
    ((pixel_info_t *)((char *)out + p.y * pitch))[p.x] = {(float)(p.x + p.y * size.x), 1.0f, false, 0.0f};
}

#define PLAIN_KERNELS(NAME, REAL)                                                                  \
    extern "C" __global__ __launch_bounds__(1024) void fractalRenderMain##NAME(                    \
        pixel_info_t *out, long pitch, Point<uint> size, Rectangle<REAL>, uint, float, uint) {     \
        name_pixel(out, pitch, size);                                                              \
    }                                                                                              \
    extern "C" __global__ __launch_bounds__(1024) void fractalRenderAdvanced##NAME(                \
        pixel_info_t *out, long pitch, Point<uint> size, Rectangle<REAL>, uint, float, uint,       \
        Rectangle<REAL>, const pixel_info_t *, long, Point<uint>) {                                \
        name_pixel(out, pitch, size);                                                              \
    }
PLAIN_KERNELS(Float, float)
PLAIN_KERNELS(Double, double)

extern "C" __global__ void init() {}
extern "C" __global__ void debug() {}
extern "C" __global__ void fractalRenderUnderSampled(pixel_info_t *, long, uint, uint, float, float,
                                                     float, float, uint, uint) {}

extern "C" __global__ __launch_bounds__(1024) void compose(const pixel_info_t *main, long pitch,
                                                           const pixel_info_t *, long, uint *output,
                                                           uint width, uint height,
                                                           const uint *palette, uint, float) {
    const Point<uint> p = pixel();
    if (p.x >= width || p.y >= height) return;
    const pixel_info_t *row = (const pixel_info_t *)((const char *)main + p.y * pitch);
    output[p.y * width + p.x] = palette[0] + (uint)row[p.x].value;
}
