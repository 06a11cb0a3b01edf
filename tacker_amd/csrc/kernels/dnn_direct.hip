// The layers of the latency-critical DNN task (VGG16, batch 1) as launches of their own: a convolution that reads
// its input activation where it lies instead of an im2col operand in memory, and a fully connected layer as the
// matrix-vector product it is.  They are what a layer runs when nothing is fused with it; a layer that shares its
// launch with a best-effort kernel goes through im2col and the tzgemm role (dnn_kernels.h, the generated fused
// kernels), and both give the same bits: every element of C is added up in the order of tzgemm_role --
// v_mfma_f32_16x16x32_f16 over ascending k, and for the shapes whose reduction tzgemm cuts (tz_use_ksplit) the
// same quarters of the same parts, ((w0 + w1) + w2) + w3, parts in order.
//
// Data.  An activation is f16 NHWC with a border of one zero pixel, [H + 2][W + 2][C], written by the layer before
// with bias, ReLU and -- where a pooling follows -- the 2x2 maximum applied; beside it a layer leaves its raw
// 1.1 * A * B^T in fp32 as the operand builders expect it, where somebody may read it (54 MB a query at 224 x 224, 20 us of it).  Weights are laid out once, at the task's creation, in the
// order the matrix instruction takes them (pack_weight_fragments): fragment (16 output channels, 32 k) is
// 1 KiB in a row, lane l's 16 bytes at 16 l.
#include <hip/hip_runtime.h>

#include "../../../include/tacker_amd.h"
#include "../header/tzgemm_header.h"
#include "../dnn/direct.h"

namespace tk {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) char lds_char;
typedef __attribute__((address_space(3))) const half8_t lds_half8;
typedef __attribute__((address_space(3))) half4_t lds_half4;
typedef __attribute__((address_space(3))) _Float16 lds_half;
typedef __attribute__((address_space(3))) float4_t lds_float4;
typedef __attribute__((address_space(3))) float lds_float;

#define DNN_VMCNT_IMM(n) (((n) & 15) | (((n) >> 4) << 14) | 0x0F70)   // s_waitcnt vmcnt(n), nothing else

template <int N>
struct dnn_int {
    static constexpr int value = N;
};

// One LDS-direct load of 16 bytes per lane: scalar base + 32-bit lane offset, to LDS address + 16 lane.
__device__ __forceinline__ void dnn_load_to_lds(const char *uniform_base, unsigned lane_offset, unsigned lds_address)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(lds_address), "v"(lane_offset), "s"(uniform_base)
                 : "memory");
}

__device__ __forceinline__ half4_t dnn_activate(float4_t v, float4_t bias)
{
    v += bias;
    half4_t h;
#pragma unroll
    for (int i = 0; i < 4; ++i) h[i] = (_Float16)(v[i] < 0.0f ? 0.0f : v[i]);
    return h;
}

// Where float4 q (channels 4 q ..) of pixel p of a tile of `quads` float4s a pixel lies in LDS, in units of 16 bytes: row p,
// with a key that spreads a matrix instruction's result (16 pixels, one q) and a row's reads alike over all banks
__device__ __forceinline__ int dnn_tile_at(int p, int q, int quads)
{
    return p * quads + (q ^ (quads >= 8 ? p & 7 : (p >> 1) & 3));
}

// The pixel p of an 8 x 8 tile: four 2x2 cells side by side per group of 16 (the rows of a matrix instruction), groups
// two image rows apart
__device__ __forceinline__ int dnn_tile_x(int p) { return 2 * ((p >> 2) & 3) + (p & 1); }
__device__ __forceinline__ int dnn_tile_y(int p) { return 2 * (p >> 4) + ((p >> 1) & 1); }

// n / d by the host's reciprocal (2^32 / d rounded up, 0 for d = 1): exact for the tile numbers of any image
__device__ __forceinline__ int dnn_div(int n, unsigned reciprocal) { return reciprocal ? (int)__umulhi((unsigned)n, reciprocal) : n; }

// A tile's results from LDS to memory, of its first 16 GROUPS pixels.  `partials` tiles of [pixel][quads] lie in LDS, to be added in tzgemm's order
// (parts of four segments, or -- parts_only -- sums of whole parts); n0: first channel.  Lanes take a pixel's channels
// side by side, so that a pixel's row goes out in one piece: the raw value to C, the activation -- of the pixel, or of its
// 2x2 cell -- to the next layer's input.
template <int GROUPS>
__device__ __forceinline__ void dnn_finish(lds_float4 *tile, int partials, bool parts_only, int quads, int y0, int x0, int n0,
                                           const float4_t bias, const DnnOutput &o)
{
    const int threads = (int)blockDim.x, quad_shift = __builtin_ctz(quads);
    const int stride = DNN_TILE * DNN_TILE * quads;
    for (int i = (int)threadIdx.x; i < 16 * GROUPS * quads; i += threads) {
        const int p = i >> quad_shift, q = i & (quads - 1);
        const int at = dnn_tile_at(p, q, quads);
        float4_t v = tile[at];
        if (parts_only) {
            for (int s = 1; s < partials; ++s) v += tile[s * stride + at];
        } else if (partials > 1) {
            for (int s = 0; s < partials; s += 4) {
                float4_t part = tile[s * stride + at];
                part += tile[(s + 1) * stride + at];
                part += tile[(s + 2) * stride + at];
                part += tile[(s + 3) * stride + at];
                v = s == 0 ? part : v + part;
            }
        }
        v *= TZ_ALPHA;
        const int y = y0 + dnn_tile_y(p), x = x0 + dnn_tile_x(p), n = n0 + 4 * q;
        if (y < o.H && x < o.W) {
            if (o.raw) *reinterpret_cast<float4_t *>(o.raw + (size_t)(y * o.W + x) * o.ld + n) = v;
            if (!o.pool)
                *reinterpret_cast<half4_t *>(reinterpret_cast<_Float16 *>(o.act) +
                                             (size_t)((y + o.border) * o.act_pitch + x + o.border) * o.act_C + n) =
                    dnn_activate(v, bias);
        }
        if (o.pool) tile[at] = v;
    }
    if (!o.pool) return;
    __syncthreads();
    for (int i = (int)threadIdx.x; i < 4 * GROUPS * quads; i += threads) {
        const int cell = i >> quad_shift, q = i & (quads - 1);
        float4_t v = tile[dnn_tile_at(4 * cell, q, quads)];
#pragma unroll
        for (int e = 1; e < 4; ++e) {
            const float4_t w = tile[dnn_tile_at(4 * cell + e, q, quads)];
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = fmaxf(v[j], w[j]);
        }
        const int y = y0 + dnn_tile_y(4 * cell), x = x0 + dnn_tile_x(4 * cell), n = n0 + 4 * q;
        if (y < o.H && x < o.W)
            *reinterpret_cast<half4_t *>(reinterpret_cast<_Float16 *>(o.act) +
                                         (size_t)((y / 2 + o.border) * o.act_pitch + x / 2 + o.border) * o.act_C + n) =
                dnn_activate(v, bias);
    }
}

// The bias of the channels a thread finishes, float4 threadIdx.x of the tile's `quads` a pixel (which divide the threads).
// Asked for as the kernel starts: where it is needed it would be one more trip to memory, at the end of a short kernel.
__device__ __forceinline__ float4_t dnn_bias(const DnnOutput &o, int n0, int quads)
{
    return *reinterpret_cast<const float4_t *>(o.bias + n0 + 4 * ((int)threadIdx.x & (quads - 1)));
}

// workgroup -> (pixel tile, channel group): every XCD takes a contiguous run of the order "channel group, then pixel
// tile", so that a group's weights come into few L2s
__device__ __forceinline__ int dnn_tile_of(int block, int tiles)
{
    const int per = (tiles + TK_XCD_NUM - 1) / TK_XCD_NUM;
    return (block % TK_XCD_NUM) * per + block / TK_XCD_NUM;
}

}  // namespace tk

using namespace tk;

// The input patch of a tile of ROWS rows of the second convolution, ROWS + 2 x 10 pixels of the first one's activation, computed
// from the image: groups of 16 pixels, 27 k in one matrix instruction for 16 channels each, rounded as the first convolution's own
// kernel rounds.  The image's ROWS + 4 x 12 pixels come to LDS once, in f16, where a pixel's k are three runs of nine values.
// The tiles of a layer compute 1.6 times its pixels that way (1.9 with four rows); a launch, and its activation written and read again, are gone.
// us, both layers: 14.0 at 224 x 224 and 6.1 at 64 x 96, where the first one took 8.6 and 5.4 and the second one 12.6 and 4.9 (17.6 and 9.8
// without the raw outputs).  With every lane gathering its k from the image in memory, 14.4 and 6.9.
template <int ROWS>
__device__ __forceinline__ void dnn_patch_of_image(const DnnImage &f, lds_char *lds, lds_half *image, int y0, int x0, int H, int W,
                                                   bool keeps, int wave, int waves, int lane)
{
    constexpr int PIXELS = (ROWS + 2) * DNN_PATCH, GROUPS = (PIXELS + 15) / 16, ROW = 3 * DNN_IMAGE_SIDE;
    const int r = lane & 15, kq = lane >> 4;
    const half8_t *weights = reinterpret_cast<const half8_t *>(f.weights) + lane;
    half8_t w[4];
    float4_t bias[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        w[j] = weights[(size_t)(j * f.chunks * 2) * 64];
        bias[j] = *reinterpret_cast<const float4_t *>(f.bias + 16 * j + 4 * kq);
    }
    for (int i = (int)threadIdx.x; i < (ROWS + 4) * ROW; i += 64 * waves) {
        const int row = i / ROW, column = i - row * ROW;
        const int y = y0 - 2 + row, at = 3 * (x0 - 2) + column;
        const bool there = y >= 0 && y < H && at >= 0 && at < 3 * W;
        const float v = there ? f.image[y * 3 * W + at] : 0.0f;
        image[i] = (_Float16)v;
        if (keeps && there && row >= 2 && row < ROWS + 2 && column >= 6 && column < 6 + 3 * DNN_TILE) f.keep[y * 3 * W + at] = v;
    }
    int tap_at[8];   // where this lane's eight k (of 32; the last 5 are padding) of a pixel lie
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int k = min(8 * kq + e, 26);
        tap_at[e] = k / 9 * ROW + k % 9;
    }
    __syncthreads();
    for (int group = wave; group < GROUPS; group += waves) {
        const int p = min(16 * group + r, PIXELS - 1);
        const int py = (p * 205) >> 11, px = p - py * DNN_PATCH;   // p / 10 for p < 1024
        half8_t a;
#pragma unroll
        for (int e = 0; e < 8; ++e) a[e] = image[py * ROW + 3 * px + tap_at[e]];
        if (kq == 3) a[3] = a[4] = a[5] = a[6] = a[7] = (_Float16)0.0f;
        const int y = y0 + py - 1, x = x0 + px - 1;
        const bool inside = y >= 0 && y < H && x >= 0 && x < W;   // the border is zeros
        const int key = ((px >> 1) + 4 * (py & 1)) & 7;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float4_t zero = {0.f, 0.f, 0.f, 0.f};
            float4_t raw = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[j], a, zero, 0, 0, 0);
            raw *= TZ_ALPHA;
            half4_t h = dnn_activate(raw, bias[j]);
            if (!inside) h = half4_t{0, 0, 0, 0};
            // (lanes past the last pixel compute and write it again)
            *(lds_half4 *)(lds + p * 128 + (((2 * j + (kq >> 1)) ^ key) << 4) + 8 * (kq & 1)) = h;
        }
    }
}

// 3x3 / pad 1 / stride 1 convolution of an activation with C a multiple of 64 channels.  A workgroup computes an 8 x 8
// pixel tile by 16 * ct_count output channels; wavefront (cp, kw) of it 16 * NT channels over a run of the reduction:
// one segment, a whole part (PART: its four segments one after the other, added as tzgemm adds them), or all of it
// where tzgemm does not cut it.
//
// The tile's input, 10 x 10 pixels x C, is brought into LDS once (im2col would read it nine times) and the k loop
// runs without a barrier: a wavefront reads its 64 pixels' fragments from LDS at the tap's offset and its own
// weights, which no other wavefront of the workgroup needs, straight from memory into registers, RING chunks ahead.
// LDS rows are a pixel's 64 channels (128 bytes), one plane per 64 channels; 16-byte segment s of a pixel lies in
// slot s ^ key, key = (x / 2 + 4 (y & 1)) & 7, which spreads the 16 pixels of a fragment read (8 x 2, at any
// tap) over all banks.
//
// What bounds it is a chain of short things one after the other.  Of the 9.2 us of 28 x 28, 512 -> 512 channels (a workgroup
// is 64 pixels x 32 channels, one per CU, and loads 104 KB of patch and 295 KB of weights) 4.1 are left where the patch
// and all chunks but one are left out -- launch, first load, barrier, last sums and stores --, 2 are the k loop where its
// loads are left out, 1.6 the patch and 1.5 the weights.  So a workgroup takes as many channels as leave every CU one,
// and two 16-channel slices a wavefront (NT = 2), which halves the fragment reads from LDS, where eight wavefronts are left (four
// are too few: conv2_2 10.3 -> 11.2 us); where there are workgroups for half of the CUs or fewer, tiles have four rows (GROUPS = 2
// pairs of rows instead of 4); the bias is asked for first, then the patch, then the weights; and a step's
// fragments are read from LDS while the matrix units work on those of the step before.  us a layer of VGG16 at 224 x 224,
// first through the operand in memory and tzgemm, then reading its fragments where it uses them, now: conv2_2 26, 10.5, 9.5,
// conv3_2 21, 9.5, 8.8, conv4_2 23, 9.7, 9.1, conv5_1 18, 8.4, 6.6; at 64 x 96 conv4_2 8.6, 6.8, conv5_1 8.2, 6.3 (the last two each).
template <int NT, bool PART, bool IMAGE, int GROUPS>
__device__ __forceinline__ void conv3x3_direct(const DnnConv &c, const DnnImage &first_layer, char *lds_generic)
{
    lds_char *const lds = (lds_char *)lds_generic;
    const int lane = (int)threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int waves = (int)blockDim.x >> 6;
    const int tile = dnn_tile_of((int)blockIdx.x, c.workgroups);
    if (tile >= c.workgroups) return;
    const int group = dnn_div(tile, c.per_group);
    const int pixel_tile = tile - group * c.tiles;
    const int tile_row = dnn_div(pixel_tile, c.per_row);
    const int y0 = tile_row * (2 * GROUPS), x0 = (pixel_tile - tile_row * c.tiles_x) * DNN_TILE;
    const int ct_shift = __builtin_ctz(c.ct_count / NT);
    const int cp = wave & ((1 << ct_shift) - 1), kw = wave >> ct_shift;
    const int n16 = group * c.ct_count + cp * NT;
    const int H = c.out.H, W = c.out.W;
    const int planes = c.C >> 6, plane_shift = __builtin_ctz(planes);

    // this wavefront's chunks, and with PART where its second, third and fourth segment begin
    const int *begin = c.segment_begin + (PART ? 4 * kw : kw);
    const int first = begin[0], last = begin[PART ? 4 : 1];
    const int second = PART ? begin[1] : last, third = PART ? begin[2] : last, fourth = PART ? begin[3] : last;

    const int quads = 4 * c.ct_count;
    const float4_t bias = dnn_bias(c.out, group * c.ct_count * 16, quads);
    if (IMAGE) dnn_patch_of_image<2 * GROUPS>(first_layer, lds, (lds_half *)(lds + first_layer.lds), y0, x0, H, W, group == 0, wave, waves, lane);
    // the patch: pieces of 8 pixels, every plane of a piece by one wavefront; what lies below the image's border is left out
    const int pieces = IMAGE ? 0 : (min(2 * GROUPS + 2, H + 2 - y0) * DNN_PATCH + 7) >> 3;
    const unsigned lds_base = (unsigned)(size_t)lds;
    for (int piece = wave; piece < pieces; piece += waves) {
        const int p = min(8 * piece + (lane >> 3), DNN_PATCH * DNN_PATCH - 1);
        const int py = (p * 205) >> 11, px = p - py * DNN_PATCH;   // p / 10 for p < 1024
        const int gy = min(y0 + py, H + 1), gx = min(x0 + px, W + 1);
        const int key = ((px >> 1) + 4 * (py & 1)) & 7;
        const unsigned at = (unsigned)((gy * (W + 2) + gx) * c.C + (((lane & 7) ^ key) << 3)) * 2u;
        for (int plane = 0; plane < planes; ++plane)
            dnn_load_to_lds(reinterpret_cast<const char *>(c.act) + plane * 128, at,
                            lds_base + plane * DNN_PLANE_BYTES + piece * 1024);
    }
    // behind it the first chunks of the weights; the patch has landed when only they are still on their way
    constexpr int RING = 2;
    static_assert(RING % 2 == 0, "a step's fragments are read into the set the step before does not use");
    const half8_t *weights = reinterpret_cast<const half8_t *>(c.weights) + (size_t)n16 * c.chunks * 2 * 64 + lane;
    half8_t b[RING][NT][2];
    const int final_chunk = max(last - 1, 0);   // an empty run fetches the first chunk, which is there
    const auto fetch = [&](half8_t (&w)[NT][2], int chunk) {
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int h = 0; h < 2; ++h) w[t][h] = weights[(size_t)(t * c.chunks * 2 + 2 * chunk + h) * 64];
    };
#pragma unroll
    for (int u = 0; u < RING; ++u) fetch(b[u], min(first + u, final_chunk));
    __builtin_amdgcn_sched_barrier(0);
    if (IMAGE) {
        __syncthreads();
    } else {
        __builtin_amdgcn_s_waitcnt(DNN_VMCNT_IMM(2 * NT * RING));
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    }

    const int r = lane & 15;
    const int tx = dnn_tile_x(r), ty = dnn_tile_y(r);
    float4_t acc[NT][GROUPS], sum[NT][GROUPS];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int g = 0; g < GROUPS; ++g) acc[t][g] = sum[t][g] = float4_t{0.f, 0.f, 0.f, 0.f};

    // The pixels' fragments of this step and the next, both halves of their 64 k.  (They make 108 registers out of 64: of workgroups of
    // 12 and 16 wavefronts with up to 256 channels one fits a CU where two did, and layers of 288 to 448 of those -- conv3_2 at 128 x
    // 160, conv4_1 at 160 x 224 -- take 8.4 and 7.8 us for 7.5 and 6.9.  All others gain, the queries of those sizes by 7 %.)
    half8_t a[2][2][GROUPS];
    const auto read = [&](half8_t (&to)[2][GROUPS], int chunk) {
        const int tap = chunk >> plane_shift, plane = chunk & (planes - 1);
        const int kh = (tap * 11) >> 5, kx = tap - 3 * kh;   // tap / 3 for tap < 9
        const int px = tx + kx, py = ty + kh;
        const int key = ((px >> 1) + 4 * (py & 1)) & 7;
        const unsigned at = (unsigned)(plane * DNN_PLANE_BYTES + (py * DNN_PATCH + px) * 128 + (((lane >> 4) ^ key) << 4));
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int g = 0; g < GROUPS; ++g) to[h][g] = *(lds_half8 *)(lds + (at ^ (64u * h)) + g * (2 * DNN_PATCH * 128));
    };
    const auto multiply = [&](const half8_t (&w)[NT][2], const half8_t (&p)[2][GROUPS]) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int g = 0; g < GROUPS; ++g) acc[t][g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[t][h], p[h][g], acc[t][g], 0, 0, 0);
    };
    int segment = 1;
    const auto segment_done = [&]() {   // ((w0 + w1) + w2) + w3
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int g = 0; g < GROUPS; ++g) {
                sum[t][g] = segment == 1 ? acc[t][g] : sum[t][g] + acc[t][g];
                acc[t][g] = float4_t{0.f, 0.f, 0.f, 0.f};
            }
        ++segment;
    };
    const auto next_begins = [&]() -> int { return segment == 1 ? second : (segment == 2 ? third : (segment == 3 ? fourth : last)); };
    const auto step = [&](const half8_t (&w)[NT][2], const half8_t (&now)[2][GROUPS], half8_t (&next)[2][GROUPS], int chunk) {
        if (PART)
            while (chunk == next_begins()) segment_done();
        read(next, min(chunk + 1, final_chunk));   // (behind the run the last ones again)
        __builtin_amdgcn_sched_barrier(0);
        multiply(w, now);
        __builtin_amdgcn_sched_barrier(0);
    };
    // A run is 9 chunks in most layers.  Its last RING chunks are told apart from the rest: nothing behind the run is
    // fetched (that was a third more weights than it has), and the loop's waits count exactly the loads behind the one they
    // need; with the end's condition inside the loop the compiler has to allow for a fetch left out, and waits for all of
    // them every time round.  More chunks in flight lose: with 4 a query takes 145.7 instead of 142.4 us at 224 x 224 and 90.7
    // instead of 89.1 at 64 x 96 (what is in front of the barrier, the patch, is what the wavefronts wait for).
    read(a[0], min(first, final_chunk));
    int base = first;
    for (; base + RING < last; base += RING) {
#pragma unroll
        for (int u = 0; u < RING; ++u) {
            step(b[u], a[u & 1], a[(u + 1) & 1], base + u);
            fetch(b[u], min(base + u + RING, final_chunk));
        }
    }
#pragma unroll
    for (int u = 0; u < RING; ++u)
        if (base + u < last) step(b[u], a[u & 1], a[(u + 1) & 1], base + u);   // uniform
    if (PART)
        while (segment <= 4) segment_done();

    // results to LDS, [run of the reduction][pixel][channels]; the patch is done with
    __syncthreads();
    lds_float4 *const results = (lds_float4 *)lds;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int g = 0; g < GROUPS; ++g)
            results[kw * DNN_TILE * DNN_TILE * quads + dnn_tile_at(16 * g + r, 4 * (cp * NT + t) + (lane >> 4), quads)] =
                PART ? sum[t][g] : acc[t][g];
    __syncthreads();
    dnn_finish<GROUPS>(results, c.runs, PART, quads, y0, x0, group * c.ct_count * 16, bias, c.out);
}

#define DNN_CONV_KERNEL(NAME_, NT_, PART_, GROUPS_, THREADS_)                                                          \
    extern "C" __global__ __launch_bounds__(THREADS_) void NAME_(DnnConv c)                                            \
    {                                                                                                                 \
        extern __shared__ __align__(16) char conv_lds[];                                                              \
        conv3x3_direct<NT_, PART_, false, GROUPS_>(c, DnnImage{}, conv_lds);                                           \
    }
DNN_CONV_KERNEL(conv3x3_direct_1_0, 1, false, 4, 1024)
DNN_CONV_KERNEL(conv3x3_direct_1_1, 1, true, 4, 512)
DNN_CONV_KERNEL(conv3x3_direct_2_0, 2, false, 4, 512)
// Tiles of four rows instead of eight, for layers of few workgroups: half the reads from LDS and matrix instructions, 62 instead of
// 104 KB of patch at 512 channels, twice the workgroups (conv5_1 at 224 x 224 8.0 -> 6.7 us, conv4_2 at 64 x 96 9.0 -> 7.3).
DNN_CONV_KERNEL(conv3x3_direct_1_0_low, 1, false, 2, 1024)
DNN_CONV_KERNEL(conv3x3_direct_1_1_low, 1, true, 2, 512)
// the first two convolutions, the first one's activation as patches in LDS only
#define DNN_IMAGE_KERNEL(NAME_, GROUPS_)                                                                               \
    extern "C" __global__ __launch_bounds__(512, 4) void NAME_(DnnImage first_layer, DnnConv c)                        \
    {                                                                                                                 \
        extern __shared__ __align__(16) char conv_lds[];                                                              \
        conv3x3_direct<1, false, true, GROUPS_>(c, first_layer, conv_lds);                                             \
    }
DNN_IMAGE_KERNEL(conv3x3_direct_image, 4)
DNN_IMAGE_KERNEL(conv3x3_direct_image_low, 2)

// The first convolution: the image, [H][W][3] fp32, 27 k in one matrix instruction.  A workgroup computes an 8 x 8 pixel
// tile by 64 channels, wavefront g the pixel group g; a lane gathers its 8 k (of 32; the last 5 are padding) of its pixel.
// keep: null, or where the image is stored as well.
extern "C" __global__ __launch_bounds__(256) void conv3x3_image(const float *image, float *keep, DnnConv c)
{
    __shared__ __align__(16) char image_lds[DNN_TILE * DNN_TILE * 64 * 4];
    lds_float4 *const results = (lds_float4 *)(lds_char *)image_lds;
    const int lane = (int)threadIdx.x & 63;
    const int g = (int)threadIdx.x >> 6;
    const int tile = dnn_tile_of((int)blockIdx.x, c.workgroups);
    if (tile >= c.workgroups) return;
    const int tile_row = dnn_div(tile, c.per_row);
    const int y0 = tile_row * DNN_TILE, x0 = (tile - tile_row * c.tiles_x) * DNN_TILE;
    const int H = c.out.H, W = c.out.W;
    const float4_t bias = dnn_bias(c.out, 0, 16);
    if (keep && threadIdx.x < 3 * DNN_TILE * DNN_TILE) {
        const int row = (int)threadIdx.x / (3 * DNN_TILE), column = (int)threadIdx.x - row * (3 * DNN_TILE);
        if (y0 + row < H && 3 * x0 + column < 3 * W) {
            const int at = ((y0 + row) * W + x0) * 3 + column;
            keep[at] = image[at];
        }
    }
    const int r = lane & 15;
    const int x = x0 + dnn_tile_x(r), y = y0 + 2 * g + dnn_tile_y(r);
    // all eight loads at once, from indices clamped to the image; what lies outside becomes zero afterwards
    float v[8];
    bool in[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int k = 8 * (lane >> 4) + e;
        const int tap = k / 3, ch = k - 3 * tap;
        const int kh = tap / 3, kx = tap - 3 * kh;
        const int yy = y + kh - 1, xx = x + kx - 1;
        in[e] = k < 27 && yy >= 0 && yy < H && xx >= 0 && xx < W;
        v[e] = image[(min(max(yy, 0), H - 1) * W + min(max(xx, 0), W - 1)) * 3 + ch];
    }
    const half8_t *weights = reinterpret_cast<const half8_t *>(c.weights) + lane;
    half8_t w[4], a;
#pragma unroll
    for (int j = 0; j < 4; ++j) w[j] = weights[(size_t)(j * c.chunks * 2) * 64];
#pragma unroll
    for (int e = 0; e < 8; ++e) a[e] = (_Float16)(in[e] ? v[e] : 0.0f);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const float4_t zero = {0.f, 0.f, 0.f, 0.f};
        results[dnn_tile_at(16 * g + r, 4 * j + (lane >> 4), 16)] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[j], a, zero, 0, 0, 0);
    }
    __syncthreads();
    dnn_finish<4>(results, 1, false, 16, y0, x0, 0, bias, c.out);
}

// A fully connected layer at batch 1: 16 outputs per workgroup, a wavefront takes SPW consecutive segments of the
// reduction and streams their weights past the caches (nontemporal: a query reads each of them once).  All 16 rows of the
// matrix instruction's other operand are the activation vector; its first row is the layer's.
//
// A segment is a few steps to a few dozen, and it is up to 8 steps' loads at a time, the last ones as well: a trip to
// memory is 1 to 2 us, and a segment of 6 steps (3072 -> 4096), or two of 4 (4096 -> 1000), two steps at a time made three or four
// of them.
template <int SPW>
__device__ __forceinline__ void fc_direct(const DnnFc &f)
{
    __shared__ float partial[16 * SPW][16];
    const float bias = f.act ? f.bias[blockIdx.x * 16 + (threadIdx.x & 15)] : 0.0f;   // (asked for first, as dnn_bias)
    const int lane = (int)threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const half8_t *weights = reinterpret_cast<const half8_t *>(f.weights) + ((size_t)blockIdx.x * f.chunks * 2) * 64 + lane;
    const half8_t *x = reinterpret_cast<const half8_t *>(f.x) + (lane >> 4);
    half8_t w[8], a[8];
    const auto load = [&](auto steps, int k) {   // steps of 32 k
#pragma unroll
        for (int u = 0; u < decltype(steps)::value; ++u) {
            w[u] = __builtin_nontemporal_load(weights + (size_t)(k + u) * 64);
            a[u] = x[4 * (k + u)];
        }
    };
    const auto multiply = [&](auto from, auto to, float4_t &acc) {
#pragma unroll
        for (int u = decltype(from)::value; u < decltype(to)::value; ++u)
            acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[u], a[u], acc, 0, 0, 0);
    };
    const auto store = [&](int s, const float4_t &acc) {
        if ((lane & 15) == 0) {
#pragma unroll
            for (int e = 0; e < 4; ++e) partial[s][4 * (lane >> 4) + e] = acc[e];
        }
    };
    const int s0 = wave * SPW;
    if (SPW == 2 && s0 + 1 < f.segments && f.segment_begin[s0 + 1] - f.segment_begin[s0] == 2 &&
        f.segment_begin[s0 + 2] - f.segment_begin[s0 + 1] == 2) {   // two of four steps: at once
        float4_t acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = acc0;
        load(dnn_int<8>(), 2 * f.segment_begin[s0]);
        multiply(dnn_int<0>(), dnn_int<4>(), acc0);
        multiply(dnn_int<4>(), dnn_int<8>(), acc1);
        store(s0, acc0);
        store(s0 + 1, acc1);
    } else {
#pragma unroll
        for (int i = 0; i < SPW; ++i) {
            const int s = s0 + i;
            if (s < f.segments) {
                int k = 2 * f.segment_begin[s];
                const int last = 2 * f.segment_begin[s + 1];
                float4_t acc = {0.f, 0.f, 0.f, 0.f};
                const auto step = [&](auto steps) {
                    load(steps, k);
                    multiply(dnn_int<0>(), steps, acc);
                    k += decltype(steps)::value;
                };
                while (k + 8 <= last) step(dnn_int<8>());
                if (k + 6 <= last) step(dnn_int<6>());
                else if (k + 4 <= last) step(dnn_int<4>());
                else if (k + 2 <= last) step(dnn_int<2>());
                store(s, acc);
            }
        }
    }
    __syncthreads();
    if (threadIdx.x < 16) {
        const int n = (int)blockIdx.x * 16 + (int)threadIdx.x;
        float v = partial[0][threadIdx.x];   // one segment (a reduction tzgemm does not cut) is its own sum
        for (int s = 0; f.segments > 1 && s < f.segments; s += 4) {
            float part = partial[s][threadIdx.x];
            part += partial[s + 1][threadIdx.x];
            part += partial[s + 2][threadIdx.x];
            part += partial[s + 3][threadIdx.x];
            v = s == 0 ? part : v + part;
        }
        v *= TZ_ALPHA;
        f.raw[n] = v;
        if (f.act) {
            v += bias;
            reinterpret_cast<_Float16 *>(f.act)[n] = (_Float16)(v < 0.0f ? 0.0f : v);
        }
    }
}
extern "C" __global__ __launch_bounds__(1024) void fc_direct_1(DnnFc f) { fc_direct<1>(f); }
extern "C" __global__ __launch_bounds__(1024) void fc_direct_2(DnnFc f) { fc_direct<2>(f); }

// The activation of a layer whose raw output another kernel wrote (a launch fused with a best-effort kernel), for a next
// layer that runs by itself: a thread per four channels of a pixel, or of a 2x2 cell.
extern "C" __global__ __launch_bounds__(256) void dnn_activation(DnnOutput o, int channels)
{
    const int Ho = o.pool ? o.H / 2 : o.H, Wo = o.pool ? o.W / 2 : o.W;
    const int quads = channels / 4;
    const int total = Ho * Wo * quads;
    for (int i = (int)(blockIdx.x * blockDim.x + threadIdx.x); i < total; i += (int)(gridDim.x * blockDim.x)) {
        const int p = i / quads, n = 4 * (i - p * quads);
        const int y = p / Wo, x = p - y * Wo;
        float4_t v;
        if (o.pool) {
            const float *at = o.raw + (size_t)(2 * y * o.W + 2 * x) * o.ld + n;
            const float4_t a = *reinterpret_cast<const float4_t *>(at);
            const float4_t b = *reinterpret_cast<const float4_t *>(at + o.ld);
            const float4_t d = *reinterpret_cast<const float4_t *>(at + (size_t)o.W * o.ld);
            const float4_t e = *reinterpret_cast<const float4_t *>(at + (size_t)o.W * o.ld + o.ld);
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = fmaxf(fmaxf(a[j], b[j]), fmaxf(d[j], e[j]));
        } else {
            v = *reinterpret_cast<const float4_t *>(o.raw + (size_t)p * o.ld + n);
        }
        *reinterpret_cast<half4_t *>(reinterpret_cast<_Float16 *>(o.act) + (size_t)((y + o.border) * o.act_pitch + x + o.border) * o.act_C + n) =
            dnn_activate(v, *reinterpret_cast<const float4_t *>(o.bias + n));
    }
}

// [rows][K] f16 (rows a multiple of 16, K of 64) -> fragments: 16-byte segment (n, k / 8) to fragment (n / 16, k / 32),
// lane n % 16 + 16 * (k / 8 % 4)
extern "C" __global__ __launch_bounds__(256) void pack_weight_fragments(const void *src_, void *dst_, int rows, int K)
{
    const half8_t *src = reinterpret_cast<const half8_t *>(src_);
    half8_t *dst = reinterpret_cast<half8_t *>(dst_);
    const size_t per_row = (size_t)K / 8, total = (size_t)rows * per_row;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x) {
        // i: destination segment, so that the writes are the contiguous side
        const size_t fragment = i >> 6;
        const int lane = (int)(i & 63);
        const size_t n16 = fragment / (per_row / 4), step = fragment - n16 * (per_row / 4);
        dst[i] = src[(n16 * 16 + (lane & 15)) * per_row + step * 4 + (lane >> 4)];
    }
}

extern "C" void tk_register_dnn_kernels(tk_kernel_insert_fn insert, void *ctx)
{
    insert("conv3x3_direct_1_0", (const void *)conv3x3_direct_1_0, ctx);
    insert("conv3x3_direct_1_1", (const void *)conv3x3_direct_1_1, ctx);
    insert("conv3x3_direct_2_0", (const void *)conv3x3_direct_2_0, ctx);
    insert("conv3x3_direct_1_0_low", (const void *)conv3x3_direct_1_0_low, ctx);
    insert("conv3x3_direct_1_1_low", (const void *)conv3x3_direct_1_1_low, ctx);
    insert("conv3x3_direct_image", (const void *)conv3x3_direct_image, ctx);
    insert("conv3x3_direct_image_low", (const void *)conv3x3_direct_image_low, ctx);
    insert("conv3x3_image", (const void *)conv3x3_image, ctx);
    insert("fc_direct_1", (const void *)fc_direct_1, ctx);
    insert("fc_direct_2", (const void *)fc_direct_2, ctx);
    insert("dnn_activation", (const void *)dnn_activation, ctx);
    insert("pack_weight_fragments", (const void *)pack_weight_fragments, ctx);
}
