// D3Q19 lattice-Boltzmann role (collide + scatter, one time step).
//
// Replaces ori_lbm / general_ptb_lbm / lbm_tzgemm_lbm0 of the reference
// (src/ori_kernel/lbm_kernel.cu:9-154, src/gptb_kernel/lbm_kernel.cu:3-178,
// src/mix_kernel/tzgemm_lbm.cu:6-181) with run-time grid extents.  Kept: SoA
// layout CALC_INDEX(x,y,z,e) = cells*e + x + y*sx + z*sx*sy, SCATTER streaming
// by linear index arithmetic without boundary clamping, obstacle bounce-back,
// ACCEL override, and the exact fp32 operation order of the collision.
//
// One departure, on purpose: a scatter whose linear target cell lies outside
// [0, cells) would land in the neighbouring entry plane, where the reference
// races with that plane's own writer.  Here such a store is dropped, i.e. the
// race is always resolved in favour of the in-range writer, so results are
// reproducible.
//
// gfx950 design: a block is one x-row (y,z), and rows that follow each other in the position grid follow each other in
// memory.  What a cell does depends on its linear index alone, so a range of blocks is a run of cells, whatever the
// rows' length: a wave takes 128 of them, two a lane, and each of its 20 loads and 19 stores is one contiguous piece of
// 8 bytes per lane.  No LDS, no barrier.  What bounds it is memory; us beside a GEMM, on grids that are not in the memory-side cache, with a wave a
// row (60 to 12 lanes of it at work, a cell a lane where the length is odd, whole lines at neither end) / so: 120 x 120 x 150 cells beside 4096 x 4096 x
// 1024 117.7 / 116.1, 128^3 beside 1024 x 4096 x 512 93.2 / 77.2, 127 x 128 x 128 beside 2048 x 1024 x 1024 155.6 / 98.9, 64 x 100 x 64
// beside 1024^3 25.0 / 21.1, 97^3 beside 128^3 43.5 / 32.6, 33 x 61 x 97 beside 1024 x 1024 x 512 16.6 / 11.5.  (The first three with other ways
// of dealing the pieces: no slabs an XCD 126, 90, 107; a wave's second piece a round further 121, 91, 120; a run of its own for every workgroup
// 132, 93, 112; one piece at a time 130, 76, 113; with nontemporal stores 121, 83, 108.  The first of the three moves by up to 8 % with what else is in
// the library: the same source 116 in the whole one and 126 in one of this pair alone.)
#pragma once
#include "role_common.h"
#include "../header/lbm_header.h"

namespace tk {

// All indices are 32-bit: the host refuses grids with 20*cells >= 2^31.

// Collision of one cell, in place (src/ori_kernel/lbm_kernel.cu:49-131): obstacle cells
// swap opposite directions, the others relax towards equilibrium.
__device__ __forceinline__ void lbm_collide(unsigned flags, float &tempC, float &tempN, float &tempS, float &tempE, float &tempW, float &tempT, float &tempB, float &tempNE, float &tempNW, float &tempSE, float &tempSW, float &tempNT, float &tempNB, float &tempST, float &tempSB, float &tempET, float &tempEB, float &tempWT, float &tempWB)
{
    if (flags & LBM_OBSTACLE) {
        float t;
        t = tempN; tempN = tempS; tempS = t;
        t = tempE; tempE = tempW; tempW = t;
        t = tempT; tempT = tempB; tempB = t;
        t = tempNE; tempNE = tempSW; tempSW = t;
        t = tempNW; tempNW = tempSE; tempSE = t;
        t = tempNT; tempNT = tempSB; tempSB = t;
        t = tempNB; tempNB = tempST; tempST = t;
        t = tempET; tempET = tempWB; tempWB = t;
        t = tempEB; tempEB = tempWT; tempWT = t;
    } else {
        float ux, uy, uz, rho, u2, temp1, temp2, temp_base;
        rho = tempC + tempN + tempS + tempE + tempW + tempT + tempB + tempNE + tempNW + tempSE +
              tempSW + tempNT + tempNB + tempST + tempSB + tempET + tempEB + tempWT + tempWB;
        ux = +tempE - tempW + tempNE - tempNW + tempSE - tempSW + tempET + tempEB - tempWT - tempWB;
        uy = +tempN - tempS + tempNE + tempNW - tempSE - tempSW + tempNT + tempNB - tempST - tempSB;
        uz = +tempT - tempB + tempNT - tempNB + tempST - tempSB + tempET - tempEB + tempWT - tempWB;
        ux /= rho;
        uy /= rho;
        uz /= rho;
        if (flags & LBM_ACCEL) {
            ux = 0.005f;
            uy = 0.002f;
            uz = 0.000f;
        }
        u2 = 1.5f * (ux * ux + uy * uy + uz * uz) - 1.0f;
        temp_base = LBM_OMEGA * rho;
        temp1 = LBM_DFL1 * temp_base;
        temp2 = 1.0f - LBM_OMEGA;
        tempC = temp2 * tempC + temp1 * (-u2);
        temp1 = LBM_DFL2 * temp_base;
        tempN = temp2 * tempN + temp1 * (uy * (4.5f * uy + 3.0f) - u2);
        tempS = temp2 * tempS + temp1 * (uy * (4.5f * uy - 3.0f) - u2);
        tempT = temp2 * tempT + temp1 * (uz * (4.5f * uz + 3.0f) - u2);
        tempB = temp2 * tempB + temp1 * (uz * (4.5f * uz - 3.0f) - u2);
        tempE = temp2 * tempE + temp1 * (ux * (4.5f * ux + 3.0f) - u2);
        tempW = temp2 * tempW + temp1 * (ux * (4.5f * ux - 3.0f) - u2);
        temp1 = LBM_DFL3 * temp_base;
        tempNT = temp2 * tempNT + temp1 * ((+uy + uz) * (4.5f * (+uy + uz) + 3.0f) - u2);
        tempNB = temp2 * tempNB + temp1 * ((+uy - uz) * (4.5f * (+uy - uz) + 3.0f) - u2);
        tempST = temp2 * tempST + temp1 * ((-uy + uz) * (4.5f * (-uy + uz) + 3.0f) - u2);
        tempSB = temp2 * tempSB + temp1 * ((-uy - uz) * (4.5f * (-uy - uz) + 3.0f) - u2);
        tempNE = temp2 * tempNE + temp1 * ((+ux + uy) * (4.5f * (+ux + uy) + 3.0f) - u2);
        tempSE = temp2 * tempSE + temp1 * ((+ux - uy) * (4.5f * (+ux - uy) + 3.0f) - u2);
        tempET = temp2 * tempET + temp1 * ((+ux + uz) * (4.5f * (+ux + uz) + 3.0f) - u2);
        tempEB = temp2 * tempEB + temp1 * ((+ux - uz) * (4.5f * (+ux - uz) + 3.0f) - u2);
        tempNW = temp2 * tempNW + temp1 * ((-ux + uy) * (4.5f * (-ux + uy) + 3.0f) - u2);
        tempSW = temp2 * tempSW + temp1 * ((-ux - uy) * (4.5f * (-ux - uy) + 3.0f) - u2);
        tempWT = temp2 * tempWT + temp1 * ((-ux + uz) * (4.5f * (-ux + uz) + 3.0f) - u2);
        tempWB = temp2 * tempWB + temp1 * ((-ux - uz) * (4.5f * (-ux - uz) + 3.0f) - u2);
    }
}

#define TK_LBM_DIRECTIONS(X)                                                                       \
    X(LBM_C, 0, 0, 0, tempC) \
    X(LBM_N, 0, +1, 0, tempN) \
    X(LBM_S, 0, -1, 0, tempS) \
    X(LBM_E, +1, 0, 0, tempE) \
    X(LBM_W, -1, 0, 0, tempW) \
    X(LBM_T, 0, 0, +1, tempT) \
    X(LBM_B, 0, 0, -1, tempB) \
    X(LBM_NE, +1, +1, 0, tempNE) \
    X(LBM_NW, -1, +1, 0, tempNW) \
    X(LBM_SE, +1, -1, 0, tempSE) \
    X(LBM_SW, -1, -1, 0, tempSW) \
    X(LBM_NT, 0, +1, +1, tempNT) \
    X(LBM_NB, 0, +1, -1, tempNB) \
    X(LBM_ST, 0, -1, +1, tempST) \
    X(LBM_SB, 0, -1, -1, tempSB) \
    X(LBM_ET, +1, 0, +1, tempET) \
    X(LBM_EB, +1, 0, -1, tempEB) \
    X(LBM_WT, -1, 0, +1, tempWT) \
    X(LBM_WB, -1, 0, -1, tempWB)

__device__ __forceinline__ void lbm_cell(const float *__restrict__ src, float *__restrict__ dst,
                                         int cells, int c, int sx, int sxy)
{
    float tempC = __builtin_nontemporal_load(src + cells * LBM_C + c);
    float tempN = __builtin_nontemporal_load(src + cells * LBM_N + c);
    float tempS = __builtin_nontemporal_load(src + cells * LBM_S + c);
    float tempE = __builtin_nontemporal_load(src + cells * LBM_E + c);
    float tempW = __builtin_nontemporal_load(src + cells * LBM_W + c);
    float tempT = __builtin_nontemporal_load(src + cells * LBM_T + c);
    float tempB = __builtin_nontemporal_load(src + cells * LBM_B + c);
    float tempNE = __builtin_nontemporal_load(src + cells * LBM_NE + c);
    float tempNW = __builtin_nontemporal_load(src + cells * LBM_NW + c);
    float tempSE = __builtin_nontemporal_load(src + cells * LBM_SE + c);
    float tempSW = __builtin_nontemporal_load(src + cells * LBM_SW + c);
    float tempNT = __builtin_nontemporal_load(src + cells * LBM_NT + c);
    float tempNB = __builtin_nontemporal_load(src + cells * LBM_NB + c);
    float tempST = __builtin_nontemporal_load(src + cells * LBM_ST + c);
    float tempSB = __builtin_nontemporal_load(src + cells * LBM_SB + c);
    float tempET = __builtin_nontemporal_load(src + cells * LBM_ET + c);
    float tempEB = __builtin_nontemporal_load(src + cells * LBM_EB + c);
    float tempWT = __builtin_nontemporal_load(src + cells * LBM_WT + c);
    float tempWB = __builtin_nontemporal_load(src + cells * LBM_WB + c);
    const unsigned flags = __float_as_uint(__builtin_nontemporal_load(src + cells * LBM_FLAGS + c));
    lbm_collide(flags, tempC, tempN, tempS, tempE, tempW, tempT, tempB, tempNE, tempNW, tempSE, tempSW, tempNT, tempNB, tempST, tempSB, tempET, tempEB, tempWT, tempWB);
#define TK_LBM_SCATTER(entry, dx, dy, dz, value)                          \
    do {                                                                  \
        const int t_ = c + (dx) + (dy) * sx + (dz) * sxy;                 \
        if (t_ >= 0 && t_ < cells) dst[cells * (entry) + t_] = (value);   \
    } while (0);
    TK_LBM_DIRECTIONS(TK_LBM_SCATTER)
#undef TK_LBM_SCATTER
}

// Two x-adjacent cells per lane (c even, c + 1 in the same row): every access is 8 bytes
// per lane, which halves the number of vector-memory instructions per byte moved -- the
// per-CU address/data-return unit is what a dword-per-lane streaming kernel saturates first,
// and in a fused launch that unit is shared with the GEMM's loads.  Scatter targets are
// shifted by +-1 cell for 10 of the 19 directions, so the 8-byte accesses are only 4-byte
// aligned; the vector type says so.
typedef float lbm_pair_t __attribute__((ext_vector_type(2), aligned(4)));
// The 20 values of a cell are read once per step and never again: nontemporal loads, so that they pass
// through the L2 without pushing out what has a second use -- the scattered stores, whose lines are
// completed by the waves of neighbouring rows a little later, and in a fused launch the GEMM's operand
// panels.  (Measured at 120 x 120 x 150: the step alone 73.6 instead of 79.5 us in 64-thread workgroups,
// the fused launch with the 4096 x 4096 x 1024 GEMM 95 instead of 113 us.  Nontemporal stores on top
// of that take it back: 96 us alone, 102 us fused.)
__device__ __forceinline__ lbm_pair_t lbm_load_pair(const float *p)
{
    return __builtin_nontemporal_load(reinterpret_cast<const lbm_pair_t *>(p));
}
__device__ __forceinline__ void lbm_store_pair(float *p, lbm_pair_t v)
{
    *reinterpret_cast<lbm_pair_t *>(p) = v;
}

__device__ __forceinline__ void lbm_cell_pair(const float *__restrict__ src, float *__restrict__ dst,
                                              int cells, int c, int sx, int sxy)
{
#define TK_LBM_LOAD(entry, dx, dy, dz, name) \
    const lbm_pair_t name##_in = lbm_load_pair(src + cells * (entry) + c);
    TK_LBM_DIRECTIONS(TK_LBM_LOAD)
#undef TK_LBM_LOAD
    const lbm_pair_t flags_in = lbm_load_pair(src + cells * LBM_FLAGS + c);
#define TK_LBM_SPLIT(entry, dx, dy, dz, name) float name##0 = name##_in.x, name##1 = name##_in.y;
    TK_LBM_DIRECTIONS(TK_LBM_SPLIT)
#undef TK_LBM_SPLIT
    lbm_collide(__float_as_uint(flags_in.x), tempC0, tempN0, tempS0, tempE0, tempW0, tempT0, tempB0, tempNE0, tempNW0, tempSE0, tempSW0, tempNT0, tempNB0, tempST0, tempSB0, tempET0, tempEB0, tempWT0, tempWB0);
    lbm_collide(__float_as_uint(flags_in.y), tempC1, tempN1, tempS1, tempE1, tempW1, tempT1, tempB1, tempNE1, tempNW1, tempSE1, tempSW1, tempNT1, tempNB1, tempST1, tempSB1, tempET1, tempEB1, tempWT1, tempWB1);
#define TK_LBM_SCATTER2(entry, dx, dy, dz, name)                                           \
    do {                                                                                   \
        const int t_ = c + (dx) + (dy) * sx + (dz) * sxy;                                  \
        float *o_ = dst + cells * (entry) + t_;                                            \
        if (t_ >= 0 && t_ + 1 < cells) {                                                   \
            lbm_store_pair(o_, lbm_pair_t{name##0, name##1});            \
        } else {                                                                           \
            if (t_ >= 0 && t_ < cells) o_[0] = name##0;                                    \
            if (t_ + 1 >= 0 && t_ + 1 < cells) o_[1] = name##1;                            \
        }                                                                                  \
    } while (0);
    TK_LBM_DIRECTIONS(TK_LBM_SCATTER2)
#undef TK_LBM_SCATTER2
}

// N pairs a lane at once, for a role that has few waves on its CU (inside a fused kernel): all 20 N loads
// are issued before the first collision, so a wave has N times the bytes in flight.
// Each destination word has one writer whichever cells are taken together, so the result is the
// same as one pair after the other.
template <int N>
__device__ __forceinline__ void lbm_cell_pairs(const float *__restrict__ src, float *__restrict__ dst,
                                                   int cells, const int (&c)[N], int sx, int sxy)
{
    lbm_pair_t in[N][20];
#pragma unroll
    for (int r = 0; r < N; ++r) {
#define TK_LBM_LOAD(entry, dx, dy, dz, name) in[r][entry] = lbm_load_pair(src + cells * (entry) + c[r]);
        TK_LBM_DIRECTIONS(TK_LBM_LOAD)
#undef TK_LBM_LOAD
        in[r][LBM_FLAGS] = lbm_load_pair(src + cells * LBM_FLAGS + c[r]);
    }
    // a pair is collided and scattered while the loads of those behind it are still on their way;
    // the scheduling fences keep the pairs' arithmetic apart (interleaved it needs more registers
    // than a fused kernel has)
#pragma unroll
    for (int r = 0; r < N; ++r) {
        __builtin_amdgcn_sched_barrier(0);
#define TK_LBM_SPLIT(entry, dx, dy, dz, name) float name##0 = in[r][entry].x, name##1 = in[r][entry].y;
        TK_LBM_DIRECTIONS(TK_LBM_SPLIT)
#undef TK_LBM_SPLIT
        lbm_collide(__float_as_uint(in[r][LBM_FLAGS].x), tempC0, tempN0, tempS0, tempE0, tempW0, tempT0, tempB0, tempNE0, tempNW0, tempSE0, tempSW0, tempNT0, tempNB0, tempST0, tempSB0, tempET0, tempEB0, tempWT0, tempWB0);
        lbm_collide(__float_as_uint(in[r][LBM_FLAGS].y), tempC1, tempN1, tempS1, tempE1, tempW1, tempT1, tempB1, tempNE1, tempNW1, tempSE1, tempSW1, tempNT1, tempNB1, tempST1, tempSB1, tempET1, tempEB1, tempWT1, tempWB1);
#define TK_LBM_SCATTER_ROW(entry, dx, dy, dz, name)                                        \
    do {                                                                                   \
        const int t_ = c[r] + (dx) + (dy) * sx + (dz) * sxy;                               \
        float *o_ = dst + cells * (entry) + t_;                                            \
        if (t_ >= 0 && t_ + 1 < cells) {                                                   \
            lbm_store_pair(o_, lbm_pair_t{name##0, name##1});                              \
        } else {                                                                           \
            if (t_ >= 0 && t_ < cells) o_[0] = name##0;                                    \
            if (t_ + 1 >= 0 && t_ + 1 < cells) o_[1] = name##1;                            \
        }                                                                                  \
    } while (0);
        TK_LBM_DIRECTIONS(TK_LBM_SCATTER_ROW)
#undef TK_LBM_SCATTER_ROW
    }
    __builtin_amdgcn_sched_barrier(0);
}

#define LBM_FEW_CELLS (2 * TK_CU_NUM * TK_WAVE_SIZE)

// grid_dimension_x = sy, grid_dimension_y = sz, block_dimension_x = sx
// (src/ori_kernel/lbm_kernel.cu:218-222).  PAIRS > 1: a wave takes that many pieces of 128 cells, which follow each other, at a
// time (see lbm_cell_pairs).
template <int PAIRS = 1>
__device__ __forceinline__ void lbm_role(const float *__restrict__ src, float *__restrict__ dst,
                                         int grid_dimension_x, int grid_dimension_y,
                                         int block_dimension_x, int role_block, int role_blocks,
                                         int start, int end, int tid, int role_threads)
{
    const int sx = block_dimension_x, sy = grid_dimension_x, sz = grid_dimension_y;
    const int sxy = sx * sy;
    const int rows = sy * sz, cells = sx * rows;
    const int lane = tid & (TK_WAVE_SIZE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / TK_WAVE_SIZE), waves = role_threads / TK_WAVE_SIZE;
    constexpr int PIECE = 2 * TK_WAVE_SIZE;
    if (__builtin_expect(role_threads < TK_WAVE_SIZE, 0)) {   // workgroups of less than a wavefront: a cell a thread
#pragma unroll 1
        for (int i = role_block * role_threads + tid; i < min(end - start, rows) * sx; i += role_blocks * role_threads) {
            int c = start % rows * sx + i;
            c = c < cells ? c : c - cells;
            asm volatile("" : "+v"(c)::"memory");   // (nothing of it in registers that the others do without)
            lbm_cell(src, dst, cells, c, sx, sxy);
        }
        return;
    }
    // Every XCD (workgroups go to them in turn) takes a slab of the run, in order: the lines that two waves' scattered pieces share
    // are completed in one L2.
    const int xcd_bits = role_blocks % TK_XCD_NUM == 0 ? __builtin_ctz(TK_XCD_NUM) : 0;
    const int groups = role_blocks >> xcd_bits, group = role_block >> xcd_bits, xcd = role_block - (group << xcd_bits);
    const auto slab_of = [&](int pieces) { return (pieces + (1 << xcd_bits) - 1) >> xcd_bits; };
    // A launch by itself has 16 wavefronts a SIMD, most of which have nothing to do in a short range: they leave before anything else.  Alone, us with a
    // wave a row / with three divisions in front of that / so: 281 rows of 120 cells 5.0 / 8.2 / 4.5, 1125 7.3 / 9.6 / 6.7, 2250 9.8 / 11.7 / 9.3, 18000
    // 57.2 / 54.4 / 54.4; 1125 rows of 97 cells 6.8 / 9.1 / 5.7.
    // Where there are cells for few wavefronts they are taken a cell a lane, which is over sooner than two: 64 rows of 120 4.4 / 3.5, 64 rows of 97 4.3 / 3.4,
    // 281 of 97 4.4 / 3.8; with twice as many cells 5.0 / 5.8.  (Beside a GEMM it is as often the slower way.)
    const int most = min(end - start, rows) * sx, cell = (wave * role_blocks + role_block) * TK_WAVE_SIZE + lane;
    const bool cell_a_lane = PAIRS == 1 && most <= min(LBM_FEW_CELLS, role_blocks * waves * TK_WAVE_SIZE);
    if (cell_a_lane ? cell - lane >= most : wave * groups + group >= slab_of((most + PIECE - 1) / PIECE)) return;
    // what of the range lies before the end of the grid, and again from its beginning
    for (int pos = start; pos < end;) {
        const int row = pos < rows ? pos : pos % rows, here = min(end - pos, rows - row);
        pos += here;
        const int first = row * sx, count = here * sx;
        const int pieces = (count + PIECE - 1) / PIECE;
        const int slab = slab_of(pieces), lo = xcd * slab, hi = min(pieces, lo + slab);
        // this lane's pair of a piece: the run's last lane takes its last two cells where it has an odd one left (both of a cell's
        // writers have the same bits), those behind it none
        const auto cell_of = [&](int piece) { return first + min(piece * PIECE + 2 * lane, count - 2); };
        const auto there = [&](int piece) { return piece * PIECE + 2 * lane < count; };
        if (cell_a_lane || count == 1) {
            if (cell < count) lbm_cell(src, dst, cells, first + cell, sx, sxy);
            continue;
        }
        const auto one = [&](int piece) {
            if (there(piece)) lbm_cell_pair(src, dst, cells, cell_of(piece), sx, sxy);
        };
        // Pieces that all waves take at a time: PAIRS each, as long as there are enough for all, and what is left one each, so that a last
        // round of few does not take as long as one of all.  us beside 2048^3 with what is left dealt PAIRS a wave / so: 120 x 120 x 150, an eighth
        // of a round left, 110.3 / 104.4, 4500 of its rows, a thirtieth left, 45.3 / 38.2.
        const int round = groups * waves * PAIRS;
        int from = lo;
        if (PAIRS > 1)
            for (; from + round <= hi; from += round) {
                const int piece = from + (group * waves + wave) * PAIRS;
                if ((piece + PAIRS) * PIECE <= count) {
                    int c[PAIRS];
#pragma unroll
                    for (int r = 0; r < PAIRS; ++r) c[r] = first + (piece + r) * PIECE + 2 * lane;
                    lbm_cell_pairs<PAIRS>(src, dst, cells, c, sx, sxy);
                } else {   // (the run's last piece may be a part of one)
                    for (int r = 0; r < PAIRS; ++r) one(piece + r);
                }
            }
        // What is left one at a time, over all workgroups before a second wave of one; where that is more than a round, a
        // workgroup's pieces side by side, so that the last ones are those of few workgroups.
        const bool few = PAIRS > 1 || hi - from < round;
        for (int piece = from + (few ? wave * groups + group : group * waves + wave); piece < hi; piece += groups * waves) one(piece);
    }
}

}  // namespace tk
