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
// last bit, within 2.7e-7 at |p| < 300 and the same above.)  The dot product and the two accumulations are fused
// multiply-adds in the reference's order (((Kx*x) + Ky*y) + Kz*z; Q + PhiMag*c) -- what nvcc makes of the reference's
// source with its default -fmad=true -- so a (k, x) pair is 5 such instructions and the two transcendentals.  The five
// take 2.5 to 2.8 cycles of a SIMD with two wavefronts at work if all their operands are vector registers and 4.4 with a
// scalar one (v_fract 4.3, sine and cosine 8.5 each), so a wavefront brings the records, 64 at a time, through LDS of its
// own and reads each back with one 16-byte broadcast.  2048 records and 262144 voxels: 130 us alone, 145 beside tzgemm
// 2048^3; 153 and 161 with the records in scalar registers and a v_fract.  (Without the v_fract alone: 152 and 153.)
// The result differs from a float64 evaluation by about 1e-6 per term, far inside the 1e-3 + 1e-4 |Q| bar.
#pragma once
#include "role_common.h"
#include "../header/mriq_header.h"

__constant__ mriq_kValues ck[MRIQ_MAX_K];

namespace tk {

template <int N>
struct mriq_count {
    static constexpr int value = N;
};

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

// V voxels per thread at once, k records [k_begin, k_end).  The k loop is a chain of
// dependent operations per voxel (dot product, sin/cos, accumulate) and a fused
// launch leaves the role at most two waves per SIMD, so the independent work that hides
// instruction latency has to come from inside the thread; V voxels also share each
// read of a k record.  stage: this wavefront's LDS.
template <int V>
__device__ __forceinline__ void mriq_voxels(int k_begin, int k_end, const float *__restrict__ x,
                                            const float *__restrict__ y, const float *__restrict__ z,
                                            float *__restrict__ Qr, float *__restrict__ Qi,
                                            const int (&xIndex)[V], mriq_lds_float4 *stage)
{
    if (k_begin >= k_end) return;
    float sX[V], sY[V], sZ[V], sQr[V], sQi[V];
#pragma unroll
    for (int v = 0; v < V; ++v) {
        const int i = xIndex[v];
        sX[v] = x[i];
        sY[v] = y[i];
        sZ[v] = z[i];
        sQr[v] = Qr[i];
        sQi[v] = Qi[i];
    }
    const int lane = mriq_lane();
    const float4_t *table = reinterpret_cast<const float4_t *>(ck);
    // (a voxel alone needs eight records to have enough chains: 2048 x 65536, one voxel a lane and one or two wavefronts a
    // SIMD, 51.9 us with four, 46.6 with eight; beside tzgemm 1024^3 57.2 and 48.9)
    constexpr int U = V == 1 ? 8 : 4;
    // U records at a time, written stage by stage (all phases, then all sines and cosines,
    // then the accumulation in ascending k): the U * V chains are independent until the last
    // stage, and the order of the source is already the interleaved one -- the compiler's
    // scheduler does not have to find it (for one of the instances in a fused kernel it did
    // not, and that loop ran one dependent chain at a time).
    const auto add = [&](const float4_t *k, auto records) {
        constexpr int N = decltype(records)::value;
        float c[N][V], s[N][V];
#pragma unroll
        for (int u = 0; u < N; ++u)
#pragma unroll
            for (int v = 0; v < V; ++v)   // revolutions
                c[u][v] = __builtin_fmaf(k[u].z, sZ[v], __builtin_fmaf(k[u].y, sY[v], k[u].x * sX[v]));
#pragma unroll
        for (int u = 0; u < N; ++u)
#pragma unroll
            for (int v = 0; v < V; ++v) {
                s[u][v] = __builtin_amdgcn_sinf(c[u][v]);
                c[u][v] = __builtin_amdgcn_cosf(c[u][v]);
            }
#pragma unroll
        for (int u = 0; u < N; ++u)
#pragma unroll
            for (int v = 0; v < V; ++v) {
                sQr[v] = __builtin_fmaf(k[u].w, c[u][v], sQr[v]);
                sQi[v] = __builtin_fmaf(k[u].w, s[u][v], sQi[v]);
            }
    };
    float4_t ahead = table[min(k_begin + lane, k_end - 1)];
    for (int k0 = k_begin; k0 < k_end; k0 += TK_WAVE_SIZE) {
        stage[lane] = ahead;
        ahead = table[min(k0 + TK_WAVE_SIZE + lane, k_end - 1)];
        mriq_stage_fence();
        const int count = min(TK_WAVE_SIZE, k_end - k0);
        const auto read = [&](float4_t (&r)[U], int first) {
#pragma unroll
            for (int u = 0; u < U; ++u) r[u] = stage[(first & (TK_WAVE_SIZE - 1)) + u];
            __builtin_amdgcn_sched_barrier(0);   // on its way while the records before it are used
        };
        float4_t ka[U], kb[U];
        read(ka, 0);
        int i = 0;
        for (; i + 2 * U <= count; i += 2 * U) {
            read(kb, i + U);
            add(ka, mriq_count<U>());
            __builtin_amdgcn_sched_barrier(0);
            read(ka, i + 2 * U);
            add(kb, mriq_count<U>());
            __builtin_amdgcn_sched_barrier(0);
        }
        // The table's last records: up to 15 one by one with a voxel alone, up to 7 with more.  They cost 0.4 to 1.1 us of a launch: 262144
        // voxels, 2032 records 130.3 us and 2047 131.4, 128 and 143 10.9 and 12.5; 65536 voxels 46.1 and 46.9, 5.9 and 6.7.  (The records
        // in scalar registers took 152.9 and 154.4, 12.3 and 13.1, 69.0 and 69.9, 6.8 and 7.4 there.)
        for (; i < count; ++i) {
            const float4_t one[1] = {stage[i]};
            add(one, mriq_count<1>());
        }
        mriq_stage_fence();
    }
#pragma unroll
    for (int v = 0; v < V; ++v) {
        Qr[xIndex[v]] = sQr[v];
        Qi[xIndex[v]] = sQi[v];
    }
}

// What a thread does for V voxels and a run of k records: the part of the kernel that the
// walk over block positions below does not know about.  MRI-FHD (mrif_role.h) walks the
// same position grid with another body.
struct MriqBody {
    static constexpr int STAGE_QUADS = TK_WAVE_SIZE;   // float4s of LDS a wavefront needs
    static __device__ __forceinline__ int chunk() { return MRIQ_K_CHUNK; }
    template <int V>
    static __device__ __forceinline__ void voxels(int k_begin, int k_end, const float *__restrict__ x,
                                                  const float *__restrict__ y, const float *__restrict__ z,
                                                  float *__restrict__ Qr, float *__restrict__ Qi,
                                                  const int (&xIndex)[V], mriq_lds_float4 *stage)
    {
        mriq_voxels<V>(k_begin, k_end, x, y, z, Qr, Qi, xIndex, stage);
    }
};

// the natural kernel's thread: one voxel, every record.  tid: thread of the workgroup, of WAVES wavefronts
template <int WAVES, class Body = MriqBody>
__device__ __forceinline__ void mriq_voxel(int numK, const float *__restrict__ x,
                                           const float *__restrict__ y, const float *__restrict__ z,
                                           float *__restrict__ Qr, float *__restrict__ Qi, int xIndex, int tid)
{
    const int one[1] = {xIndex};
    Body::template voxels<1>(0, numK, x, y, z, Qr, Qi, one,
                             mriq_stage_of_wave<WAVES, Body::STAGE_QUADS>(__builtin_amdgcn_readfirstlane(tid / TK_WAVE_SIZE)));
}

// One phase of a launch: voxel blocks [block_lo, block_hi) each take records
// [k_begin, k_end).  A thread serves the blocks it owns -- first_owned, first_owned +
// stride, ... -- up to MRIQ_VOXELS_PER_THREAD at a time.
#define MRIQ_VOXELS_PER_THREAD 4
template <class Body>
__device__ __forceinline__ void mriq_phase(int block_lo, int block_hi, int k_begin, int k_end,
                                           const float *__restrict__ x, const float *__restrict__ y,
                                           const float *__restrict__ z, float *__restrict__ Qr,
                                           float *__restrict__ Qi, int first_owned, int stride, int t,
                                           mriq_lds_float4 *stage)
{
    constexpr int V = MRIQ_VOXELS_PER_THREAD;
    if (block_lo >= block_hi || k_begin >= k_end) return;
    int b = first_owned;
    if (b < block_lo) b += (block_lo - b + stride - 1) / stride * stride;
    for (; b < block_hi; b += V * stride) {
        int idx[V];
        int count = 0;
#pragma unroll
        for (int v = 0; v < V; ++v) {
            const int bv = b + v * stride;
            if (bv < block_hi) count = v + 1;
            idx[v] = (bv < block_hi ? bv : b) * KERNEL_Q_THREADS_PER_BLOCK + t;
        }
        if (count == V) {
            Body::template voxels<V>(k_begin, k_end, x, y, z, Qr, Qi, idx, stage);
        } else {
            if (count >= 2) {
                const int two[2] = {idx[0], idx[1]};
                Body::template voxels<2>(k_begin, k_end, x, y, z, Qr, Qi, two, stage);
            }
            if (count & 1) {
                const int one[1] = {idx[count - 1]};
                Body::template voxels<1>(k_begin, k_end, x, y, z, Qr, Qi, one, stage);
            }
        }
    }
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
// partial last row.  Every voxel block has one owner thread group for the whole launch
// (slot-major over the role's workgroups, so a short range still spreads over all CUs),
// and the owner walks the three parts in order: the chunks of a voxel are added in
// ascending position order without any synchronisation between threads.  Whole rows that
// follow each other are one run of the k loop.
// WAVES: wavefronts of a workgroup that there is LDS for; those of a larger workgroup leave the blocks to them.
template <int WAVES, class Body = MriqBody>
__device__ __forceinline__ void mriq_role(int numK, const float *__restrict__ x,
                                          const float *__restrict__ y, const float *__restrict__ z,
                                          float *__restrict__ Qr, float *__restrict__ Qi,
                                          int grid_dimension_x, int grid_dimension_y, int role_block,
                                          int role_blocks, int start, int end, int tid, int role_threads)
{
    const int blocks_at_once = min(role_threads, WAVES * TK_WAVE_SIZE) / KERNEL_Q_THREADS_PER_BLOCK;
    const int slot = tid / KERNEL_Q_THREADS_PER_BLOCK;
    const int t = tid % KERNEL_Q_THREADS_PER_BLOCK;
    if (slot >= blocks_at_once || start >= end) return;
    mriq_lds_float4 *stage = mriq_stage_of_wave<WAVES, Body::STAGE_QUADS>(__builtin_amdgcn_readfirstlane(tid / TK_WAVE_SIZE));
    const int gx = grid_dimension_x;
    const int gy = grid_dimension_y;
    const int stride = role_blocks * blocks_at_once;
    const int first_owned = slot * role_blocks + role_block;
    const auto chunk_begin = [&](int row) { return min((row % gy) * Body::chunk(), numK); };
    const auto chunk_end = [&](int row) { return min((row % gy + 1) * Body::chunk(), numK); };

    const int first_row = start / gx;
    const int last_row = (end - 1) / gx;   // row of the last position
    if (first_row == last_row) {
        mriq_phase<Body>(start - first_row * gx, end - first_row * gx, chunk_begin(first_row), chunk_end(first_row),
                   x, y, z, Qr, Qi, first_owned, stride, t, stage);
        return;
    }
    int row = first_row;
    if (start != first_row * gx) {   // partial first row
        mriq_phase<Body>(start - first_row * gx, gx, chunk_begin(row), chunk_end(row), x, y, z, Qr, Qi,
                   first_owned, stride, t, stage);
        ++row;
    }
    const int whole_end = (end == (last_row + 1) * gx) ? last_row + 1 : last_row;   // whole rows [row, whole_end)
    while (row < whole_end) {
        // rows up to the next multiple of grid_dimension_y are consecutive chunks
        const int run_end = min(whole_end, (row / gy + 1) * gy);
        mriq_phase<Body>(0, gx, chunk_begin(row), chunk_end(run_end - 1), x, y, z, Qr, Qi, first_owned, stride, t, stage);
        row = run_end;
    }
    if (whole_end == last_row)       // partial last row
        mriq_phase<Body>(0, end - last_row * gx, chunk_begin(last_row), chunk_end(last_row), x, y, z, Qr, Qi,
                   first_owned, stride, t, stage);
}

}  // namespace tk
