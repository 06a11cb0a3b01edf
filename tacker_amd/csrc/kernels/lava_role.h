// lavaMD role (Rodinia): for every particle of a home box, the potential and force it feels from
// the particles of the home box and of its up to 26 neighbour boxes,
//   r2 = vi + vj - (xi xj + yi yj + zi zj);  vij = exp(-a2 r2);  fs = 2 vij;
//   f.v += qj vij;  f.x += qj fs (xi - xj);  f.y, f.z likewise,        a2 = 2 alpha^2,
// accumulated onto the force array in the order home box, neighbour 1, 2, ... and particle 0 .. 99
// within a box.
//
// Replaces ori_lava / general_ptb_lava (src/ori_kernel/lava_kernel.cu:9-141,
// src/gptb_kernel/lava_kernel.cu:3-140 of the reference).  The reference gives a home box to a
// block of 128 threads and stages the home and the neighbour particles in shared memory between
// block barriers.  Here wavefronts serve a box without LDS and without a barrier.  fp32; the exponential is
// the hardware's 2^x of -r2 a2 log2(e) where the reference calls CUDA's expf, and multiply-adds are fused:
// results agree within a tolerance, not bit for bit.
//
// What bounds it is VALU issue, so two things count.
//  * Which registers an instruction reads: with all operands in vector registers a 32-bit multiply, add or
//    fused multiply-add takes about 2.3 cycles of a SIMD with two or more waves at work, with a scalar
//    register among them 4.4 (measured; the exponential 8.5 either way).  Neighbour particles are the same
//    for many lanes, but they arrive by vector loads (one address for 16 lanes), not by scalar ones.
//  * How full the lanes are: 100 particles on 64 lanes, one neighbour at a time, leave 22 % of the slots
//    empty.  The wavefront is four rows of 16 lanes: row g takes neighbours g, g + 4, g + 8, ... (25 of the
//    100), a lane LAVA_MAX_P = 7 home particles (112 slots for 100) -- 89 % of the slots work, and a load
//    serves seven pairs.
// A pair is 12 such instructions and the exponential.  At the end of a part the four rows' sums are added,
// (g0 + g2) + (g1 + g3), by lane swaps that add two values at once, which leaves component v, y, x, z of the
// total in row 0, 1, 2, 3; the total goes on from the output array.  24^3 boxes: 1.31 ms, 32^3: 3.1 ms (52 cycles a SIMD
// and step of 64 slots); 2.86 and 5.35 ms with neighbours by scalar loads, two particles a lane, 25
// instructions a pair.  (By counters the vector units issue all the time: 1.30 in the units in which a kernel that keeps all
// SIMDs busy reads 1.)
//
// Few boxes: a box is then split over several wavefronts (P home particles a lane instead of 7, every particle
// summed exactly as before), see LavaUnits.
//
// Block positions.  A box through its 27 boxes is 270 000 pair interactions, 180 us of one
// wavefront and far longer than a GEMM, so -- as for cutcp -- the position grid has a second
// dimension: position p adds part (p / boxes) % 27 (0 = the home box, k = neighbour k of the
// box's list; nothing where the box has fewer neighbours) to box p % boxes.  The forces rest in the
// output between parts.  Every box has one owner wavefront for the whole launch, which walks the
// rows of the grid in order, so a box's parts are added in ascending order without any
// synchronisation and whole rows that follow each other are one run through their parts.
#pragma once
#include "role_common.h"
#include "../header/lava_header.h"

namespace tk {

typedef __attribute__((address_space(4))) const box_str lava_const_box;

#define LAVA_ROWS 4                                     // rows of 16 lanes: neighbours are dealt to them in turn
#define LAVA_LANES 16                                   // home particles side by side in a row
#define LAVA_MAX_P 7                                    // home particles per lane when one wavefront serves a box
#define LAVA_WAVES_PER_SIMD 4                           // wavefronts of this role a SIMD holds (registers)
#define LAVA_STEPS (NUMBER_PAR_PER_BOX / LAVA_ROWS)     // neighbours a row takes per box
// of them in flight: a step of a lane with many particles outlasts a load by itself, and the registers of
// more would cost a wavefront of the SIMD
#define LAVA_AHEAD(P_) ((P_) >= 4 ? 1 : 5)
static_assert(NUMBER_PAR_PER_BOX % LAVA_ROWS == 0 && LAVA_STEPS % 5 == 0, "rows and fetches come out even");
static_assert(LAVA_LANES * LAVA_MAX_P >= NUMBER_PAR_PER_BOX, "a wavefront holds a box");

// the halves of a wavefront, and the rows of its halves, exchanged between two registers: after it a holds
// the lower half (even rows) of both, b the upper half (odd rows)
__device__ __forceinline__ float lava_fold_halves(float a, float b)
{
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);   // lower half: sum of a, upper half: sum of b
}
__device__ __forceinline__ float lava_fold_rows(float a, float b)
{
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);   // even rows: sum of a's pair, odd rows: of b's
}

// box `bx`, parts [part_begin, part_end) of its list, for the 16 P home particles from 16 P `sub` on, by one
// wavefront.  scale = -a2 log2(e).
template <int P>
__device__ __forceinline__ void lava_box(const float scale, const box_str *d_box_gpu, const FOUR_VECTOR *d_rv_gpu,
                                         const float *d_qv_gpu, FOUR_VECTOR *d_fv_gpu, int bx, int sub, int part_begin,
                                         int part_end, int lane)
{
    constexpr int AHEAD = LAVA_AHEAD(P);
    const lava_const_box *boxes = (const lava_const_box *)d_box_gpu;
    const long first_i = boxes[bx].offset;
    const int neighbours = boxes[bx].nn;
    if (part_end > 1 + neighbours) part_end = 1 + neighbours;
    if (part_begin >= part_end) return;
    const int row = lane >> 4;
    const int component = row == 1 ? 2 : (row == 2 ? 1 : row);   // of {v, x, y, z}: what this row's total is
    const float twice = row == 0 ? 1.0f : 2.0f;                   // fs = 2 vij in the force components
    const float4_t *rA = reinterpret_cast<const float4_t *>(d_rv_gpu + first_i);
    float *fA = reinterpret_cast<float *>(d_fv_gpu + first_i) + component;
    float4_t home[P];   // {scale v, x, y, z}
    float total[P];
#pragma unroll
    for (int k = 0; k < P; ++k) {
        const int i = (sub * P + k) * LAVA_LANES + (lane & (LAVA_LANES - 1));
        const int in = i < NUMBER_PAR_PER_BOX ? i : 0;   // slots past the box compute along and are not stored
        home[k] = rA[in];
        home[k][0] *= scale;
        total[k] = fA[4 * in];
    }
    // A neighbour is named by its number alone (its offset in the list is not read): two loads behind one another.  The
    // first is issued two parts ahead, the second one; where there is no such part, the home box's own are read.  Both at
    // the part's start took 1347 us at 24^3 boxes and 403 at 14^3, this 1315 and 379.
    const auto box_of = [&](int part) -> int { return part == 0 || part >= part_end ? bx : boxes[bx].nei[part - 1].number; };
    long next_j = boxes[box_of(part_begin)].offset;
    int after_next = box_of(part_begin + 1);
    for (int part = part_begin; part < part_end; ++part) {
        const long first_j = next_j;
        next_j = boxes[after_next].offset;
        after_next = box_of(part + 2);
        const float4_t *rB = reinterpret_cast<const float4_t *>(d_rv_gpu + first_j) + row;
        const float *qB = d_qv_gpu + first_j + row;
        float4_t f[P];
#pragma unroll
        for (int k = 0; k < P; ++k) f[k] = float4_t{0.f, 0.f, 0.f, 0.f};
        float4_t rb[AHEAD];
        float qb[AHEAD];
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
            rb[u] = rB[LAVA_ROWS * u];
            qb[u] = qB[LAVA_ROWS * u];
        }
        for (int t = 0; t < LAVA_STEPS; t += AHEAD) {
            const int next = t + AHEAD < LAVA_STEPS ? t + AHEAD : 0;   // (the last fetch is not used)
#pragma unroll
            for (int u = 0; u < AHEAD; ++u) {
                const float4_t b = rb[u];
                const float q = qb[u];
                rb[u] = rB[LAVA_ROWS * (next + u)];
                qb[u] = qB[LAVA_ROWS * (next + u)];
                // scale (vi + vj - (xi xj + yi yj + zi zj)) = -r2 a2 log2(e), stage by stage over the lane's
                // particles: their chains are independent, and in this order none waits for its own last result
                const float4_t sb = {scale * b[0], -scale * b[1], -scale * b[2], -scale * b[3]};
                float w[P];
#pragma unroll
                for (int k = 0; k < P; ++k) w[k] = home[k][0] + sb[0];
#pragma unroll
                for (int c = 1; c < 4; ++c)
#pragma unroll
                    for (int k = 0; k < P; ++k) w[k] = __builtin_fmaf(home[k][c], sb[c], w[k]);
#pragma unroll
                for (int k = 0; k < P; ++k) w[k] = __builtin_amdgcn_exp2f(w[k]);
#pragma unroll
                for (int k = 0; k < P; ++k) w[k] *= q;
#pragma unroll
                for (int k = 0; k < P; ++k) f[k][0] += w[k];
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int c = 1; c < 4; ++c) {
                    float d[P];
#pragma unroll
                    for (int k = 0; k < P; ++k) d[k] = home[k][c] - b[c];
#pragma unroll
                    for (int k = 0; k < P; ++k) f[k][c] = __builtin_fmaf(w[k], d[k], f[k][c]);
                    __builtin_amdgcn_sched_barrier(0);   // (fewer differences alive at a time)
                }
            }
        }
#pragma unroll
        for (int k = 0; k < P; ++k)
            total[k] += twice * lava_fold_rows(lava_fold_halves(f[k][0], f[k][1]), lava_fold_halves(f[k][2], f[k][3]));
    }
#pragma unroll
    for (int k = 0; k < P; ++k) {
        const int i = (sub * P + k) * LAVA_LANES + (lane & (LAVA_LANES - 1));
        if (i < NUMBER_PAR_PER_BOX) fA[4 * i] = total[k];
    }
}

// wavefronts a box is split over with P home particles a lane
__device__ __forceinline__ constexpr int lava_subs(int P)
{
    return (NUMBER_PAR_PER_BOX + LAVA_LANES * P - 1) / (LAVA_LANES * P);
}

// Which wavefront takes what.  A unit is a box, or a part of its home particles: the first `whole` boxes are one
// unit each (7 particles a lane), the boxes behind them `subs` units each of 16 P particles.  A wavefront serves
// the units it owns -- first_owned, first_owned + stride, ... -- through all phases of a launch.
struct LavaUnits {
    int whole;   // boxes of one unit each
    int p;       // particles per lane of the others' units
    int subs;    // units each of them makes

    // `waves` wavefronts serve `boxes` boxes.  Whole rounds of as many boxes as wavefronts are at work at a time
    // take a box each; what is left over -- all of it when the domain is small -- is cut as fine as makes no more
    // units than those wavefronts: a box is 0.1 to 0.4 ms of one wavefront, with up to 4 of them on a SIMD, and a
    // last round of few boxes would leave most of the chip idle that long.  (Cut finer throughout, lanes are
    // emptier -- 78 % of the slots work with 2 and 4 particles a lane -- and a load serves fewer pairs.)
    // Measured against one unit a box throughout: 24^3 boxes (three rounds and 1536 boxes) 1.32 against 1.62 ms, 18^3
    // 0.58 / 0.74; against the kernel without any split 8^3 0.10 / 0.30, 3^3 0.05 / 0.30, 2^3 0.016 / 0.093 ms.
    __device__ __forceinline__ LavaUnits(int boxes, int waves)
    {
        const int at_once = min(waves, LAVA_WAVES_PER_SIMD * 4 * TK_CU_NUM);
        whole = boxes / at_once * at_once;
        const int left = boxes - whole;
        p = left * lava_subs(1) <= at_once * 3 / 4 ? 1 : (left * lava_subs(2) <= at_once ? 2 : (left * lava_subs(4) <= at_once ? 4 : LAVA_MAX_P));
        subs = p == 1 ? lava_subs(1) : (p == 2 ? lava_subs(2) : (p == 4 ? lava_subs(4) : 1));
    }
    __device__ __forceinline__ int first_of(int box) const { return box <= whole ? box : whole + (box - whole) * subs; }
};

// One phase of a launch: boxes [box_lo, box_hi) each walk parts [part_begin, part_end).
__device__ __forceinline__ void lava_phase(const LavaUnits units, int box_lo, int box_hi, int part_begin, int part_end,
                                           const float scale, const box_str *d_box_gpu, const FOUR_VECTOR *d_rv_gpu,
                                           const float *d_qv_gpu, FOUR_VECTOR *d_fv_gpu, int first_owned, int stride,
                                           int lane)
{
    const int lo = units.first_of(box_lo), hi = units.first_of(box_hi);
    int c = first_owned;
    if (c < lo) c += (lo - c + stride - 1) / stride * stride;
    for (; c < hi; c += stride) {
        const int unit = __builtin_amdgcn_readfirstlane(c);
        const int left = unit - units.whole;
        const int box = left < 0 ? unit : units.whole + left / units.subs;
        const int sub = left < 0 ? 0 : left % units.subs;
        const int p = left < 0 ? LAVA_MAX_P : units.p;
#define LAVA_BOX(P_) lava_box<P_>(scale, d_box_gpu, d_rv_gpu, d_qv_gpu, d_fv_gpu, box, sub, part_begin, part_end, lane)
        if (p == LAVA_MAX_P) LAVA_BOX(LAVA_MAX_P);
        else if (p == 4) LAVA_BOX(4);
        else if (p == 2) LAVA_BOX(2);
        else LAVA_BOX(1);
#undef LAVA_BOX
    }
}

// grid_dimension_x: boxes (the reference's grid); the position grid has the boxes as columns and the
// LAVA_PARTS parts as rows.  A range that runs past the grid wraps.
__device__ __forceinline__ void lava_role(par_str d_par_gpu, dim_str d_dim_gpu, const box_str *d_box_gpu,
                                          const FOUR_VECTOR *d_rv_gpu, const float *d_qv_gpu, FOUR_VECTOR *d_fv_gpu,
                                          int grid_dimension_x, int role_block, int role_blocks, int start, int end,
                                          int tid, int role_threads)
{
    const int waves = role_threads / TK_WAVE_SIZE;
    const int wave = tid / TK_WAVE_SIZE;
    if (wave >= waves || start >= end) return;
    const int lane = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    // boxes past number_boxes do nothing in the reference (src/ori_kernel/lava_kernel.cu:21)
    const int gx = (long)grid_dimension_x < d_dim_gpu.number_boxes ? grid_dimension_x : (int)d_dim_gpu.number_boxes;
    if (gx <= 0 || grid_dimension_x <= 0) return;
    const float a2 = 2.0 * d_par_gpu.alpha * d_par_gpu.alpha;
    const float scale = -a2 * 1.44269504088896340736f;
    const int cols = grid_dimension_x;   // positions per row, including boxes past number_boxes
    const int stride = role_blocks * waves;
    const LavaUnits units(gx, stride);
    // many units: those of a workgroup follow each other, so that the fine ones of the last round start last; few:
    // those that follow each other lie in different workgroups, so that a short range uses every CU there is
    const int first_owned = units.first_of(gx) >= LAVA_WAVES_PER_SIMD * 4 * TK_CU_NUM ? role_block * waves + wave
                                                                                      : wave * role_blocks + role_block;
    // the range as phases: a partial row, or whole rows that follow each other up to the last part
    for (int pos = start; pos < end;) {
        const int row = pos / cols;
        const int part = row % LAVA_PARTS;
        const int lo = pos - row * cols;
        int rows = 1, hi = min(cols, lo + (end - pos));
        if (lo == 0 && hi == cols) rows = min((end - pos) / cols, LAVA_PARTS - part);
        pos += rows == 1 ? hi - lo : rows * cols;
        const int last = min(hi, gx);
        if (lo >= last) continue;
        lava_phase(units, lo, last, part, part + rows, scale, d_box_gpu, d_rv_gpu, d_qv_gpu, d_fv_gpu, first_owned, stride,
                   lane);
    }
}

}  // namespace tk
