// MRI-Q role: Q(x) += sum_k phiMag_k * exp(i 2 pi k.x).
//
// Replaces ori_mriq / g_general_ptb_mriq (src/ori_kernel/mriq_kernel.cu:56-105,
// src/gptb_kernel/mriq_kernel.cu:3-70).  The fused copy of the reference
// truncates cos/sin to int (src/mix_kernel/tzgemm_mriq.cu:57,63); parity is with
// the unfused kernel, so this role keeps float throughout.  Kept: one thread per
// voxel, blocks of 256 voxels, read-modify-write of Qr/Qi, the k table as an
// array of {Kx,Ky,Kz,PhiMag} in constant memory, fp32 order
//   arg = 2pi * ((Kx*x + Ky*y) + Kz*z); Qr += PhiMag*cos(arg); Qi += PhiMag*sin(arg)
// with k ascending.  The reference's loop "for QGrid < 1" handles only the first
// 1024-sample chunk; here all numK samples held in the table are used.
//
// gfx950: what bounds it is VALU issue.  The hardware sine and cosine take their argument in revolutions and reduce
// it themselves, at any size: the phase k.x goes to them as it is, cos(2 pi p) = v_cos(p).  (Over the whole range of
// floats they are within 1.3e-7 of sine and cosine; behind a v_fract, which rounds a negative phase to a whole turn's
// last bit, within 2.7e-7 at |p| < 300 and the same above.)  A (k, x) pair is the two transcendentals, 8.45 cycles of a SIMD each, two fused
// multiply-adds of 2.75 (Q + PhiMag*c, as nvcc contracts the reference's source with its default -fmad=true) and a 256th of a matrix
// instruction, 4 cycles that the vector units need not wait for while other wavefronts have something for them: the phase (mriq_put_point below).
// With the phase as three multiply-adds in the reference's order, ((Kx*x) + Ky*y) + Kz*z, 2032 records and 262144 voxels took 130 us alone and
// 144 to 160 beside tzgemm 2048^3, so 104 and 118 to 122, and with the transcendentals first 104 to 106 and 112 to 121; 700 records and 65536 voxels beside tzgemm 1024^3
// 21.2 to 22.1, now 18.5.
// The result differs from a float64 evaluation by about 1e-6 per term, far inside the 1e-3 + 1e-4 |Q| bar.
#pragma once
#include "role_common.h"
#include "../header/mriq_header.h"

__constant__ mriq_kValues ck[MRIQ_MAX_K];

namespace tk {

typedef __attribute__((address_space(3))) float4_t mriq_lds_float4;

// the LDS of the role's wavefronts, QUADS float4s each.  role_wave: the calling wavefront's number within the role
template <int WAVES, int QUADS>
__device__ __forceinline__ mriq_lds_float4 *mriq_stage_of_wave(int role_wave)
{
    __shared__ __align__(16) float4_t mriq_stage[WAVES][QUADS];
    return (mriq_lds_float4 *)&mriq_stage[role_wave][0];
}

// what a wavefront wrote to its own LDS is there for all its lanes (LDS serves a wavefront in order), and what it read is read
__device__ __forceinline__ void mriq_stage_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ int mriq_lane() { return (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)); }

// A phase k.x by the matrix units.  A float is the sum of three bf16 pieces, each the rest rounded to nearest, and products of
// pieces are exact in the matrix instruction's fp32 sum, so eight of the nine products of pieces of a coordinate (not the one of the two last,
// 2^-32 of it) for three coordinates are 24 of the 32 slots of one v_mfma_f32_16x16x32_bf16, which gives 256 phases in 16 cycles of a SIMD
// where three multiply-adds in fp32 take 32, and leaves the vector units to others part of the time.
//
// In LDS a point -- a record's K or a voxel -- is three tokens of four bf16, {x, y, z, 0} of its first, second and third pieces.  Lanes
// 16 g .. 16 g + 15 hold slots 8 g .. 8 g + 7 of an operand, two tokens; which ones decides how the products add up.  The sum
// runs from group 0 to 3, so the largest product comes last, with the smallest: phases then have less error than the chain of three
// multiply-adds (2-norm against 64 bits: |K|, |x| up to 0.5 4.2e-9 for 5.1e-9, up to 20 7.7e-6 for 8.3e-6; with the largest first 6.7e-9 and 11e-6).
typedef __bf16 mriq_bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 mriq_bf16x8 __attribute__((ext_vector_type(8)));
typedef float mriq_float2 __attribute__((ext_vector_type(2)));
typedef unsigned mriq_uint2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) mriq_uint2 mriq_lds_token;
#define MRIQ_TOKENS 3   // of a point
#define MRIQ_TILE 16    // records, and voxels, of a matrix instruction

struct MriqSlots {
    // tokens of lane group g, one digit of 8 bits a group
    static __device__ __forceinline__ int pick(unsigned digits, int group) { return (int)(digits >> (8 * group)) & 3; }
    int record[2], voxel[2];
    __device__ __forceinline__ explicit MriqSlots(int group)
        : record{pick(0x00000001u, group), pick(0x02010201u, group)}, voxel{pick(0x00010202u, group), pick(0x01000001u, group)} {}
};

// the next pieces of two values, which lose them
__device__ __forceinline__ unsigned mriq_pieces(float &a, float &b)
{
    const unsigned p = __builtin_bit_cast(unsigned, __builtin_convertvector(mriq_float2{a, b}, mriq_bf16x2));
    a -= __uint_as_float(p << 16);
    b -= __uint_as_float(p & 0xffff0000u);
    return p;
}

__device__ __forceinline__ void mriq_put_point(mriq_lds_token *tokens, float x, float y, float z)
{
    float nothing = 0.f;
#pragma unroll
    for (int i = 0; i < MRIQ_TOKENS; ++i) {
        const unsigned xy = mriq_pieces(x, y);
        tokens[i] = mriq_uint2{xy, mriq_pieces(z, nothing)};
    }
}

// Pieces hold a value exactly from 2^-109 to 3.39e38, and to 2^-134 below.  Beside a coordinate of 2^64 or more, where that may show in a phase or a
// piece round to infinity, phases are the chain of multiply-adds.  (Elsewhere 2^-134 is less than 2^-67 of a turn.)
__device__ __forceinline__ bool mriq_far(float x, float y, float z)
{
    return (__builtin_fabsf(x) >= 0x1p64f) | (__builtin_fabsf(y) >= 0x1p64f) | (__builtin_fabsf(z) >= 0x1p64f);
}

__device__ __forceinline__ mriq_bf16x8 mriq_slots(const mriq_lds_token *point, const int (&tokens)[2])
{
    const mriq_uint2 a = point[tokens[0]], b = point[tokens[1]];
    return __builtin_bit_cast(mriq_bf16x8, uint4_t{a.x, a.y, b.x, b.y});
}

// the halves of a wavefront, and the rows of 16 lanes, added by lane swaps that add two values at once
__device__ __forceinline__ float mriq_fold_halves(float a, float b)
{
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);   // lower half: sum of a's, upper half: of b's
}
__device__ __forceinline__ float mriq_fold_rows(float a, float b)
{
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);   // even rows: sum of a's pair, odd rows: of b's
}

// V times T tiles of 16 voxels of a wavefront, from voxel base[v] on, k records [k_begin, k_end) from a multiple of MRIQ_K_CHUNK.  The wavefront
// brings 64 records at a time through its LDS.  A lane has voxel 16 t + lane % 16 of every tile t of 16 and, of 16 records, the four
// 4 (lane / 16) ..: its sums over a chunk of records are added to the other three lane groups' at the chunk's end, and that to Q, so any
// split at chunks gives the same bits.  The last records of the table come in a whole tile of 16, with weights of zero behind them.
// stage: this wavefront's LDS.  Where a voxel or a record was far, nothing is written and the result is true: then FAR computes the voxels, 16 at a time,
// and differs in the phases of what is far alone, so that a voxel's bits do not depend on those beside it.
template <int V, int T, bool FAR = false>
__device__ __forceinline__ bool mriq_voxels(int k_begin, int k_end, const float *__restrict__ x,
                                            const float *__restrict__ y, const float *__restrict__ z,
                                            float *__restrict__ Qr, float *__restrict__ Qi,
                                            const int (&base)[V], mriq_lds_float4 *stage)
{
    static_assert(T == 1 || T == 2 || T == 4, "the folds leave a lane one voxel's sums");
    if (k_begin >= k_end) return false;
    constexpr int GROUPS = TK_WAVE_SIZE / MRIQ_TILE, TILES = T * V, AHEAD = TILES == 1 ? 1 : 2;
    int lane = mriq_lane();
    if (FAR) asm volatile("" : "+v"(lane));   // (what follows from it is not kept through a launch, in registers that it does not have)
    const int group = lane / MRIQ_TILE, column = lane % MRIQ_TILE;
    const MriqSlots slots(group);
    mriq_lds_token *const points = (mriq_lds_token *)stage;
    __attribute__((address_space(3))) float *const weights =
        (__attribute__((address_space(3))) float *)(points + MRIQ_TOKENS * TK_WAVE_SIZE);
    // the tile whose sum the folds leave here
    const int own_tile = T == 4 ? (group == 1 ? 2 : (group == 2 ? 1 : group)) : (T == 2 ? group / 2 : 0);

    mriq_bf16x8 voxel[TILES];
    unsigned long long far = 0;   // lanes that met a far voxel or record
    int own[V];   // this lane's voxel of each 64, whose sums the folds leave here
    float totalR[V], totalI[V];
    const float4_t *table = reinterpret_cast<const float4_t *>(ck);
    float4_t ahead = table[min(k_begin + lane, k_end - 1)];
#pragma unroll
    for (int v = 0; v < V; ++v) {
        const int i = base[v] + lane % (T * MRIQ_TILE);
        own[v] = base[v] + MRIQ_TILE * own_tile + column;
        totalR[v] = Qr[own[v]];
        totalI[v] = Qi[own[v]];
        mriq_put_point(points + MRIQ_TOKENS * lane, x[i], y[i], z[i]);
        if (!FAR) far |= __builtin_amdgcn_ballot_w64(mriq_far(x[i], y[i], z[i]));
        mriq_stage_fence();
#pragma unroll
        for (int t = 0; t < T; ++t)
            voxel[T * v + t] = mriq_slots(points + MRIQ_TOKENS * (MRIQ_TILE * t + column), slots.voxel);
        mriq_stage_fence();
    }
    float r[TILES], i[TILES];
    const auto phases = [&](const mriq_bf16x8 &k, int t) {
        const float4_t zero = {0.f, 0.f, 0.f, 0.f};
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(k, voxel[t], zero, 0, 0, 0);
    };
    // two tiles at a time, the matrix instructions of the next two in front of their sines.  (The next records' first ones in front of the last
    // tiles' sines as well, and records read another step ahead: 122 us for 112 beside tzgemm 2048^3.)
    // first: the lane's first record of the four.
    const auto add = [&](const mriq_bf16x8 &k, const float4_t &w, int first) {
        float4_t now[AHEAD];
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) now[u] = phases(k, u);
#pragma unroll
        for (int t = 0; t < TILES; t += AHEAD) {
            float4_t next[AHEAD];
#pragma unroll
            for (int u = 0; u < AHEAD; ++u) next[u] = t + AHEAD < TILES ? phases(k, t + AHEAD + u) : now[u];
            if (FAR) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int at = base[0] + column;
                    const float4_t of = table[min(first + e, k_end - 1)];
                    if (mriq_far(x[at], y[at], z[at]) || mriq_far(of.x, of.y, of.z))
                        now[0][e] = __builtin_fmaf(of.z, z[at], __builtin_fmaf(of.y, y[at], of.x * x[at]));
                }
            }
            float c[AHEAD][4], s[AHEAD][4];
            if (T == 4) transcendentals_begin();   // (with fewer tiles the compiler's order is worth more: 65536 voxels 27.0 us for 30.9)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int u = 0; u < AHEAD; ++u) {   // revolutions
                    c[u][e] = __builtin_amdgcn_cosf(now[u][e]);
                    s[u][e] = __builtin_amdgcn_sinf(now[u][e]);
                }
            if (T == 4) transcendentals_end();
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int u = 0; u < AHEAD; ++u) {
                    r[t + u] = __builtin_fmaf(w[e], c[u][e], r[t + u]);
                    i[t + u] = __builtin_fmaf(w[e], s[u][e], i[t + u]);
                }
#pragma unroll
            for (int u = 0; u < AHEAD; ++u) now[u] = next[u];
        }
    };
    for (int chunk = k_begin; chunk < k_end; chunk += MRIQ_K_CHUNK) {
        const int chunk_end = min(chunk + MRIQ_K_CHUNK, k_end);
#pragma unroll
        for (int t = 0; t < TILES; ++t) r[t] = i[t] = 0.f;
        for (int k0 = chunk; k0 < chunk_end; k0 += TK_WAVE_SIZE) {
            mriq_put_point(points + MRIQ_TOKENS * lane, ahead.x, ahead.y, ahead.z);
            if (!FAR) far |= __builtin_amdgcn_ballot_w64(mriq_far(ahead.x, ahead.y, ahead.z));
            weights[lane] = k0 + lane < k_end ? ahead.w : 0.f;
            ahead = table[min(k0 + TK_WAVE_SIZE + lane, k_end - 1)];
            mriq_stage_fence();
            const int tiles = (min(TK_WAVE_SIZE, chunk_end - k0) + MRIQ_TILE - 1) / MRIQ_TILE;
            const auto record = [&](int tile) { return mriq_slots(points + MRIQ_TOKENS * (MRIQ_TILE * tile + column), slots.record); };
            const auto weight = [&](int tile) { return ((mriq_lds_float4 *)weights)[GROUPS * tile + group]; };
            mriq_bf16x8 k = record(0);
            float4_t w = weight(0);
            for (int tile = 0; tile < tiles; ++tile) {
                const int next = (tile + 1) % GROUPS;   // (the last read is not used)
                const mriq_bf16x8 next_k = record(next);
                const float4_t next_w = weight(next);
                add(k, w, k0 + MRIQ_TILE * tile + 4 * group);
                k = next_k;
                w = next_w;
            }
            mriq_stage_fence();
        }
#pragma unroll
        for (int v = 0; v < V; ++v) {
            const auto fold = [&](const float (&of)[TILES]) {   // (g0 + g2) + (g1 + g3)
                const float *tile = of + T * v;
                const float a = mriq_fold_halves(tile[0], tile[T > 1 ? 1 : 0]);
                return mriq_fold_rows(a, T == 4 ? mriq_fold_halves(tile[T == 4 ? 2 : 0], tile[T == 4 ? 3 : 0]) : a);
            };
            totalR[v] += fold(r);
            totalI[v] += fold(i);
        }
    }
    if (!FAR && far != 0) return true;
    if (T < 4 && group != own_tile * (GROUPS / T)) return false;   // (with fewer tiles than lane groups several have the same voxel)
#pragma unroll
    for (int v = 0; v < V; ++v) {
        Qr[own[v]] = totalR[v];
        Qi[own[v]] = totalI[v];
    }
    return false;
}

// What a wavefront does for V times T tiles of 16 voxels and a run of k records: the part of the kernel that the
// walk over block positions below does not know about.  MRI-FHD (mrif_role.h) walks the
// same position grid with another body.
struct MriqBody {
    static constexpr bool SHARES = true;   // a block's voxels over more wavefronts than they fill
    static constexpr int AT_ONCE = 2;   // units of 64 voxels: eight tiles of a wavefront, 32 registers of pieces
    static constexpr int STAGE_QUADS = TK_WAVE_SIZE * (8 * MRIQ_TOKENS + 4) / 16;   // float4s of LDS a wavefront needs: 64 points and weights
    static __device__ __forceinline__ int chunk() { return MRIQ_K_CHUNK; }
    // Wavefronts a block of 256 voxels is shared out over, where `simds` SIMDs serve `blocks` blocks: 4 of 64 voxels each, or twice or four
    // times as many where that leaves less for the SIMD that has most, in three turns or fewer (a smaller unit prepares the records
    // for fewer voxels).  us, 1024 records beside a GEMM of four tiles, 64 / 32 / 16 voxels a wavefront, * = taken: 8192 voxels
    // 19.8 / 13.9 / 11.8*, 24576 20.1 / 14.9* / 15.2, 49152 20.4* / 20.8 / 27.5, 65536 31.9 / 27.0* / 30.9, 81920 32.2 / 27.2* / 40.3,
    // 98304 32.4* / 38.8 / 43.6, 131072 43.6* / 45.1 / 56.1, 262144 68.0* / 81.6 / 107.6.  A table of one chunk is over before units of 16 voxels are
    // worth it: 128 records, 8192 voxels beside 256^3 6.4 / 6.3* / 6.5, alone 4.5 / 3.9* / 4.0; 256 records beside 128^3 7.0 / 5.6 / 5.6*.
    static __device__ __forceinline__ int parts(int blocks, int chunks, int simds)
    {
        int p = KERNEL_Q_THREADS_PER_BLOCK / TK_WAVE_SIZE;
        while (p < KERNEL_Q_THREADS_PER_BLOCK / (chunks > 1 ? MRIQ_TILE : 2 * MRIQ_TILE)) {
            const int most = (blocks * p + simds - 1) / simds, halves = (blocks * 2 * p + simds - 1) / simds;
            if (halves >= 2 * most || halves > 3) break;
            p *= 2;
        }
        return p;
    }
    template <int V, int T>
    static __device__ __forceinline__ bool voxels(int k_begin, int k_end, const float *__restrict__ x,
                                                  const float *__restrict__ y, const float *__restrict__ z,
                                                  float *__restrict__ Qr, float *__restrict__ Qi,
                                                  const int (&base)[V], mriq_lds_float4 *stage)
    {
        return mriq_voxels<V, T>(k_begin, k_end, x, y, z, Qr, Qi, base, stage);
    }
    // `count` voxels from `first` on, some of which may be far (called in one place of a kernel: four more of them cost the others 1 to 2 %)
    static __device__ __forceinline__ void far_voxels(int k_begin, int k_end, const float *__restrict__ x,
                                                      const float *__restrict__ y, const float *__restrict__ z,
                                                      float *__restrict__ Qr, float *__restrict__ Qi, int first, int count,
                                                      mriq_lds_float4 *stage)
    {
#pragma unroll 1
        for (int t = 0; t < count; t += MRIQ_TILE) {
            const int one[1] = {first + t};
            mriq_voxels<1, 1, true>(k_begin, k_end, x, y, z, Qr, Qi, one, stage);
        }
    }
};

// the natural kernel's wavefront: 64 voxels, every record.  tid: thread of the workgroup, of WAVES wavefronts
template <int WAVES, class Body = MriqBody>
__device__ __forceinline__ void mriq_voxel(int numK, const float *__restrict__ x,
                                           const float *__restrict__ y, const float *__restrict__ z,
                                           float *__restrict__ Qr, float *__restrict__ Qi, int xIndex, int tid)
{
    const int one[1] = {xIndex - tid % TK_WAVE_SIZE};
    mriq_lds_float4 *stage = mriq_stage_of_wave<WAVES, Body::STAGE_QUADS>(__builtin_amdgcn_readfirstlane(tid / TK_WAVE_SIZE));
    if (Body::template voxels<1, 4>(0, numK, x, y, z, Qr, Qi, one, stage))
        Body::far_voxels(0, numK, x, y, z, Qr, Qi, one[0], TK_WAVE_SIZE, stage);
}

// One phase of a launch: units [lo, hi) of T tiles each take records [k_begin, k_end).  A wavefront serves the units it
// owns -- first_owned, first_owned + stride, ... -- up to AT_ONCE at a time, up to the first ones that are far.  Which that is, or hi or more.
template <class Body, int T, int AT_ONCE>
__device__ __forceinline__ int mriq_phase(int lo, int hi, int k_begin, int k_end,
                                           const float *__restrict__ x, const float *__restrict__ y,
                                           const float *__restrict__ z, float *__restrict__ Qr,
                                           float *__restrict__ Qi, int first_owned, int stride,
                                           mriq_lds_float4 *stage)
{
    constexpr int V = AT_ONCE;
    if (lo >= hi || k_begin >= k_end) return hi;
    int u = first_owned;
    if (u < lo) u += (lo - u + stride - 1) / stride * stride;
    for (; u < hi; u += V * stride) {
        int base[V];
        int count = 0;
#pragma unroll
        for (int v = 0; v < V; ++v) {
            const int uv = u + v * stride;
            if (uv < hi) count = v + 1;
            base[v] = (uv < hi ? uv : u) * (T * MRIQ_TILE);
        }
        if (count == V) {
            if (Body::template voxels<V, T>(k_begin, k_end, x, y, z, Qr, Qi, base, stage)) break;
        } else if constexpr (V > 1) {
            if constexpr (V > 2) {   // (a body that takes as many has nothing far: the first two would be added twice)
                if (count >= 2) {
                    const int two[2] = {base[0], base[1]};
                    Body::template voxels<2, T>(k_begin, k_end, x, y, z, Qr, Qi, two, stage);
                }
            }
            if (count & 1) {
                const int one[1] = {base[count - 1]};
                if (Body::template voxels<1, T>(k_begin, k_end, x, y, z, Qr, Qi, one, stage)) break;
            }
        }
    }
    return u;
}

// Block positions of the GPTB form are a grid of grid_dimension_x voxel blocks (256 voxels
// each) by grid_dimension_y chunks of MRIQ_K_CHUNK k records: position p adds chunk
// (p / grid_dimension_x) % grid_dimension_y to voxel block p % grid_dimension_x -- the
// reference's host loop over k chunks (one launch per chunk with kGlobalIndex,
// src/ori_kernel/mriq_kernel.cu:258-283) folded into the y index of the GPTB grid, so that
// a short range of positions is a short piece of work.  Q is carried through memory
// between chunks exactly as the reference carries it between launches, and a float stored
// and reloaded is unchanged, so any split of [0, x*y) into ranges gives the bits of the
// one k loop.
//
// A range [start, end) is a partial first row of the position grid, whole rows, and a
// partial last row.  A block is 4 units of 64 voxels, or where that leaves wavefronts without one 8 or 16 smaller
// ones.  Every unit has one owner wavefront for the whole launch (first_piece),
// and the owner walks the three parts in order: the chunks of a voxel are added in
// ascending position order without any synchronisation between wavefronts.  Whole rows that
// follow each other are one run of the k loop.
// WAVES: wavefronts of a workgroup that there is LDS for; those of a larger workgroup leave the units to them.
template <int WAVES, class Body = MriqBody>
__device__ __forceinline__ void mriq_role(int numK, const float *__restrict__ x,
                                          const float *__restrict__ y, const float *__restrict__ z,
                                          float *__restrict__ Qr, float *__restrict__ Qi,
                                          int grid_dimension_x, int grid_dimension_y, int role_block,
                                          int role_blocks, int start, int end, int tid, int role_threads)
{
    constexpr int UNITS = KERNEL_Q_THREADS_PER_BLOCK / TK_WAVE_SIZE;   // of 64 voxels a block
    const int waves = min(role_threads / TK_WAVE_SIZE, WAVES);
    const int wave = __builtin_amdgcn_readfirstlane(tid / TK_WAVE_SIZE);
    if (wave >= waves || start >= end) return;
    mriq_lds_float4 *stage = mriq_stage_of_wave<WAVES, Body::STAGE_QUADS>(wave);
    const int gx = grid_dimension_x;
    const int gy = grid_dimension_y;
    const int stride = role_blocks * waves;
    const int parts = Body::parts(gx, gy, min(role_blocks * min(waves, 4), 4 * TK_CU_NUM));   // (a CU has four SIMDs)
    const int first_owned = first_piece(gx * parts, 4 * TK_CU_NUM, wave, waves, role_block, role_blocks);
    if (first_owned >= gx * parts) return;   // (most, in small launches: 128 records, 8192 voxels alone 5.0 us, so 4.0)
    for (int pos = start; pos < end;) {
        const int row = pos / gx, chunk = row % gy;
        const int lo = pos - row * gx, hi = min(gx, lo + (end - pos));
        // rows up to the next multiple of grid_dimension_y are consecutive chunks
        const int rows = lo == 0 && hi == gx ? min((end - pos) / gx, gy - chunk) : 1;
        pos += rows == 1 ? hi - lo : rows * gx;
        const int k_begin = min(chunk * Body::chunk(), numK), k_end = min((chunk + rows) * Body::chunk(), numK);
        int u;
#define MRIQ_PHASE(T_, AT_ONCE_) \
    u = mriq_phase<Body, T_, AT_ONCE_>(lo * parts, hi * parts, k_begin, k_end, x, y, z, Qr, Qi, first_owned, stride, stage)
        if (Body::SHARES && parts == 4 * UNITS) MRIQ_PHASE(1, 1);
        else if (Body::SHARES && parts == 2 * UNITS) MRIQ_PHASE(2, 1);
        else MRIQ_PHASE(4, Body::AT_ONCE);
        const int voxels = MRIQ_TILE * (parts == 4 * UNITS ? 1 : (parts == 2 * UNITS ? 2 : 4));
        for (; __builtin_expect(u < hi * parts, 0); u += stride)
            Body::far_voxels(k_begin, k_end, x, y, z, Qr, Qi, u * voxels, voxels, stage);
#undef MRIQ_PHASE
    }
}

}  // namespace tk
