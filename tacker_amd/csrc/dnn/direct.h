// Argument structures and tile constants of the direct DNN kernels (kernels/dnn_direct.hip), shared by host and device.
#pragma once
#include "../header/pets_common.h"

#define DNN_TILE 8                                     // a workgroup's pixels: 8 x 8
#define DNN_PATCH (DNN_TILE + 2)                       // ... and the input they need
#define DNN_PATCH_LOADS ((DNN_PATCH * DNN_PATCH + 7) / 8)   // LDS-direct loads (8 pixels x 64 channels) per 64 channels
#define DNN_PLANE_BYTES (DNN_PATCH_LOADS * 1024)
#define DNN_PARTIAL_BYTES (DNN_TILE * DNN_TILE * 16 * 4)    // one segment's partial tile of 16 channels

// where a layer's result goes
typedef struct DnnOutput {
    float *raw;          // [H * W][ld], 1.1 * A * B^T; null: nobody reads it
    const float *bias;
    void *act;           // f16, [..][act_pitch][act_C] with `border` zero pixels around: relu(raw + bias), pooled or not
    int H, W, ld;
    int act_pitch, act_C, border, pool;
} DnnOutput;

#define DNN_MAX_SEGMENTS 32
typedef struct DnnConv {
    const void *act;       // f16 [H + 2][W + 2][C], border of zeros
    const void *weights;   // fragments (pack_weight_fragments)
    DnnOutput out;
    int C;
    int chunks;            // 64-k chunks of the padded reduction
    int runs;              // pieces of the reduction: wavefronts of a workgroup that share its channels
    int tiles, tiles_x;    // pixel tiles, and per row of them
    unsigned per_group, per_row;   // reciprocals of tiles and tiles_x (dnn_div)
    int workgroups;        // tiles * channel groups
    int ct_count;          // a group: ct_count x 16 output channels
    int segment_begin[DNN_MAX_SEGMENTS + 1];   // first chunk of each segment tzgemm cuts the reduction into; no padding chunks
} DnnConv;

#define DNN_IMAGE_SIDE (DNN_PATCH + 2)
#define DNN_IMAGE_BYTES (DNN_IMAGE_SIDE * DNN_IMAGE_SIDE * 3 * 2)
// The first convolution as the second one computes it for itself (conv3x3_direct_image)
typedef struct DnnImage {
    const float *image;    // [H][W][3]
    float *keep;           // where the image is stored as well
    const void *weights;   // fragments of 64 channels, `chunks` chunks of 64 k
    const float *bias;
    int chunks;
    int lds;               // where in LDS the tile's image goes (DNN_IMAGE_BYTES)
} DnnImage;

typedef struct DnnFc {
    const void *x;         // f16 [64 * chunks]
    const void *weights;
    float *raw;
    const float *bias;     // of this layer
    void *act;             // f16 input vector of the next layer, or null
    int chunks, segments;
    int segment_begin[DNN_MAX_SEGMENTS + 1];
} DnnFc;
