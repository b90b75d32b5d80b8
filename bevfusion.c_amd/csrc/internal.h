// Launch-only forms the GPU runtime composes into one HIP graph (hidden,
// not part of the C ABI).  The point count is read from device memory and
// grids are sized by a host bound, so one captured graph serves frames of any
// point count up to the bound.
#pragma once

#include "bevfusion.h"
#include "bf_cuda_depth_raster.h"
#include "bf_cuda_ops.h"
#include "bf_cuda_transfusion.h"
#include "bf_cuda_voxel.h"

#include <stddef.h>

namespace bfhip {

__attribute__((visibility("hidden"))) int depth_rasterize_count_device(
    bf_cuda_depth_raster *raster, const float *points, const unsigned *count_device,
    size_t bound, const float *lidar_aug, const float *lidar_to_image, const float *image_aug,
    float *depth, void *stream, char *error, size_t cap);

__attribute__((visibility("hidden"))) int voxelize_count_device(
    bf_cuda_voxelizer *voxelizer, const float *points, const unsigned *count_device,
    size_t bound, bf_coord4 *coords, float *means, unsigned *voxel_count, void *stream,
    char *error, size_t cap);

// Decode kernel only; the detections stay in the decoder's device buffer.
__attribute__((visibility("hidden"))) int transfusion_decode_launch(
    bf_cuda_transfusion *decoder, const bf_transfusion_raw_outputs *outputs, float threshold,
    void *stream, const bf_detections **device_detections, char *error, size_t cap);

}  // namespace bfhip

// For tests: the largest feature plane, in bytes, that the sparse convolutions
// gather through 32-bit buffer offsets (at most, and by default, 2 GiB - 1);
// above it they read rows through 64-bit addresses.
struct bf_cuda_lidar_backbone;
extern "C" void bfhip_lidar_offset_limit(bf_cuda_lidar_backbone *backbone, unsigned bytes);

// For tests: the kernel that bf_cuda_gemm_f32 runs on these operands
// (GemmRoute in ops.hip; pointers for their alignment only, -1: refused as too
// large).
extern "C" int bfhip_gemm_route(const float *x, const float *w, const float *b, const float *y,
                                int rows, int in_f, int out_f);

// For tests: the kernel that bf_cuda_conv2d_f32 runs (ConvRoute in ops.hip, plus
// 8 where it loads weights as float4 and 16 where the patch too) and the
// threads of its launch (0 for the gather core).
extern "C" int bfhip_conv_route(const bf_cuda_conv2d_desc *desc, const float *x, const float *w,
                                const float *y, unsigned long long *threads);

// For tests: the launches that insert a cloud of at most this many points.
extern "C" int bfhip_voxel_insert_launches(unsigned points);
