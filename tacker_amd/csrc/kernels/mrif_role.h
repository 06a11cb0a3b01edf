// MRI-FHD role: FhD(x) += sum_k RhoPhi_k * exp(i 2 pi k.x), RhoPhi = conj(phi) * d.
//
// Replaces ComputeRhoPhiGPU / ori_mrif / general_ptb_mrif
// (src/ori_kernel/mrif_kernel.cu:62-152, src/gptb_kernel/mrif_kernel.cu:6-170).
// Kept: one thread per voxel, blocks of 256 voxels, read-modify-write of
// outR/outI, the k table as an array of {Kx,Ky,Kz,RhoPhiR,RhoPhiI} in constant
// memory, fp32 order
//   arg = 2pi * ((Kx*x + Ky*y) + Kz*z)
//   outR += RhoPhiR*cos(arg) - RhoPhiI*sin(arg);  outI += RhoPhiI*cos(arg) + RhoPhiR*sin(arg)
// with k ascending.  The reference's loop "for FHGrid < 1" handles only the first
// 256-sample grid of the table; here all numK samples held in the table are used.
//
// The kernel has the shape of MRI-Q (a voxel block times a run of k records) and
// shares its walk over block positions (mriq_role.h): x = blocks of 256 voxels,
// y = chunks of MRIF_K_CHUNK records, one owner thread group per voxel block.
// The hardware sine and cosine take the phase in revolutions, the records come through a wavefront's LDS, and the
// multiply-adds are fused the way the reference's source contracts under nvcc's
// default -fmad=true: the product on the left of each sum or difference is
// folded into it, fma(RhoPhiR, cos, -(RhoPhiI*sin)) and fma(RhoPhiI, cos,
// RhoPhiR*sin), and the result is then added to the running value.
#pragma once
#include "mriq_role.h"
#include "../header/mrif_header.h"

__constant__ mrif_kValues c_mrif[MRIF_MAX_K];

namespace tk {

template <int N>
struct mrif_count {
    static constexpr int value = N;
};

static_assert(MRIF_K_CHUNK == MRIQ_K_CHUNK && KERNEL_FH_THREADS_PER_BLOCK == KERNEL_Q_THREADS_PER_BLOCK,
              "MRI-FHD shares MRI-Q's position grid: same voxel block and k chunk");

// stage: this wavefront's LDS, 64 {Kx, Ky, Kz, RhoPhiR} and behind them 64 RhoPhiI
template <int V>
__device__ __forceinline__ void mrif_voxels(int k_begin, int k_end, const float *__restrict__ x,
                                            const float *__restrict__ y, const float *__restrict__ z,
                                            float *__restrict__ outR, float *__restrict__ outI,
                                            const int (&xIndex)[V], mriq_lds_float4 *stage)
{
    if (k_begin >= k_end) return;
    typedef __attribute__((address_space(3))) float lds_float;
    float sX[V], sY[V], sZ[V], sOutR[V], sOutI[V];
#pragma unroll
    for (int v = 0; v < V; ++v) {
        const int i = xIndex[v];
        sX[v] = x[i];
        sY[v] = y[i];
        sZ[v] = z[i];
        sOutR[v] = outR[i];
        sOutI[v] = outI[i];
    }
    // U records at a time, written stage by stage (all phases, then all sines and cosines, then the accumulation in ascending k): the
    // U * V chains are independent until the last stage, and the source's order is the interleaved one already.
    constexpr int U = 4;
    const auto add = [&](const float4_t *k, const float *imaginary, auto records) {
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
                const float re = __builtin_fmaf(k[u].w, c[u][v], -(imaginary[u] * s[u][v]));
                const float im = __builtin_fmaf(imaginary[u], c[u][v], k[u].w * s[u][v]);
                sOutR[v] += re;
                sOutI[v] += im;
            }
    };
    const int lane = mriq_lane();
    mrif_kValues ahead = c_mrif[min(k_begin + lane, k_end - 1)];
    lds_float *stage_imaginary = (lds_float *)(stage + TK_WAVE_SIZE);
    for (int k0 = k_begin; k0 < k_end; k0 += TK_WAVE_SIZE) {
        stage[lane] = float4_t{ahead.Kx, ahead.Ky, ahead.Kz, ahead.RhoPhiR};
        stage_imaginary[lane] = ahead.RhoPhiI;
        ahead = c_mrif[min(k0 + TK_WAVE_SIZE + lane, k_end - 1)];
        mriq_stage_fence();
        const int count = min(TK_WAVE_SIZE, k_end - k0);
        const auto read = [&](float4_t (&r)[U], float4_t &imaginary, int first) {
#pragma unroll
            for (int u = 0; u < U; ++u) r[u] = stage[(first & (TK_WAVE_SIZE - 1)) + u];
            imaginary = stage[TK_WAVE_SIZE + (first & (TK_WAVE_SIZE - 1)) / 4];
            __builtin_amdgcn_sched_barrier(0);   // on its way while the records before it are used
        };
        const auto use = [&](const float4_t (&r)[U], const float4_t &imaginary) {
            const float im[U] = {imaginary[0], imaginary[1], imaginary[2], imaginary[3]};
            add(r, im, mrif_count<U>());
            __builtin_amdgcn_sched_barrier(0);
        };
        float4_t ka[U], kb[U], ia, ib;
        read(ka, ia, 0);
        int i = 0;
        for (; i + 2 * U <= count; i += 2 * U) {
            read(kb, ib, i + U);
            use(ka, ia);
            read(ka, ia, i + 2 * U);
            use(kb, ib);
        }
        for (; i < count; ++i) {   // (the table's last records)
            const float4_t one[1] = {stage[i]};
            const float im[1] = {stage_imaginary[i]};
            add(one, im, mrif_count<1>());
        }
        mriq_stage_fence();
    }
#pragma unroll
    for (int v = 0; v < V; ++v) {
        outR[xIndex[v]] = sOutR[v];
        outI[xIndex[v]] = sOutI[v];
    }
}

struct MrifBody {
    static constexpr int AT_ONCE = 4;
    static constexpr bool SHARES = false;   // a block's voxels over more wavefronts than they fill
    static constexpr int STAGE_QUADS = TK_WAVE_SIZE + TK_WAVE_SIZE / 4;
    static __device__ __forceinline__ int chunk() { return MRIF_K_CHUNK; }
    static __device__ __forceinline__ int parts(int, int, int) { return KERNEL_FH_THREADS_PER_BLOCK / TK_WAVE_SIZE; }
    template <int V, int T>
    static __device__ __forceinline__ bool voxels(int k_begin, int k_end, const float *__restrict__ x,
                                                  const float *__restrict__ y, const float *__restrict__ z,
                                                  float *__restrict__ outR, float *__restrict__ outI,
                                                  const int (&base)[V], mriq_lds_float4 *stage)
    {
        if constexpr (T == 4) {
            int xIndex[V];
#pragma unroll
            for (int v = 0; v < V; ++v) xIndex[v] = base[v] + mriq_lane();
            mrif_voxels<V>(k_begin, k_end, x, y, z, outR, outI, xIndex, stage);
        }
        return false;
    }
    static __device__ __forceinline__ void far_voxels(int, int, const float *, const float *, const float *, float *, float *, int, int,
                                                      mriq_lds_float4 *) {}   // (phases are multiply-adds at any size)
};

// Block positions [start, end) of the (voxel blocks) x (k chunks) grid, as mriq_role.
template <int WAVES>
__device__ __forceinline__ void mrif_role(int numK, const float *__restrict__ x,
                                          const float *__restrict__ y, const float *__restrict__ z,
                                          float *__restrict__ outR, float *__restrict__ outI,
                                          int grid_dimension_x, int grid_dimension_y, int role_block,
                                          int role_blocks, int start, int end, int tid, int role_threads)
{
    mriq_role<WAVES, MrifBody>(numK, x, y, z, outR, outI, grid_dimension_x, grid_dimension_y, role_block, role_blocks,
                               start, end, tid, role_threads);
}

}  // namespace tk
