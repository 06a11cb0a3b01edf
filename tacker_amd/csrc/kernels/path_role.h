// pathfinder role (Rodinia): `iteration` rows of the dynamic programme
//   next[x] = wall[row][x] + min(prev[x-1], prev[x], prev[x+1])      (x clamped to the grid)
// evaluated block by block on overlapping 256-column windows (a pyramid: every row the window's
// computed part shrinks by one column on each side, and the PATH_BLOCK_SIZE - 2 * iteration
// columns left in the middle are the block's result).
//
// Replaces ori_path / general_ptb_path (src/ori_kernel/path_kernel.cu:9-86,
// src/gptb_kernel/path_kernel.cu:3-93 of the reference).  Integer work: the output is the
// reference's bit for bit.  A block position bx is the window of columns
//   [small * bx - border, small * bx - border + 255],   small = 256 - 2 * iteration,
// column tx of it takes part in row i when i + 1 <= tx <= 254 - i and the column lies on the grid,
// with the neighbours clamped to the window's columns on the grid; after the last row the columns
// that were computed in it are written to gpuResults.
//
// gfx950: a wavefront serves a position, a lane holds 4 consecutive columns of the window in
// registers.  The neighbours across lanes come by a one-lane DPP shift of the wavefront, so the two
// block barriers a row of the reference's block and its two shared arrays are gone.  The dynamic
// programme is a dependent chain of `iteration` steps issued by one wavefront, so what counts is how
// few instructions a step is and that it never waits for memory:
//  * every column is updated in every row without asking whether it still takes part -- a column
//    outside the shrinking pyramid holds a value nobody reads, since a column that takes part in row
//    i only reads columns that took part in row i - 1.
//  * the clamping at the grid's two edges is a maximum: a column off the grid is held at INT_MAX, which
//    its neighbour's minimum then ignores -- min(prev, prev, right) and min(INT_MAX, prev, right) are one
//    value.  min3, add, max for a column: 14 instructions a row with the two shifts.
//  * a row of the wall is one 16-byte load a lane, AHEAD rows ahead of the row being evaluated.  The
//    lane's four columns are read as they lie, also where the row ends between them: the elements beyond
//    it are the neighbouring rows', inside the array for every row but the first and the last one the
//    launch reads, and belong to columns off the grid.  Those two rows are read column by column, from
//    indices clamped to the grid.
// 1200 columns x 125 rows (200 windows on 200 CUs): 9 us, of which 3.4 are the launch; 25 us with two selects a
// column for the clamping and four 4-byte loads a lane and row, 32 instructions a row.  20000 x 122 rows (1667
// windows): 24 against 84 us.
#pragma once
#include "role_common.h"
#include "../header/path_header.h"

// rows of the wall a wavefront keeps in flight (16, 24 and 30 take the same time at 1200 x 125)
#define PATH_ROWS_AHEAD 8

namespace tk {

// value of the lane below / above in the wavefront (0 at the wavefront's ends, whose columns lie outside the pyramid)
__device__ __forceinline__ int path_from_lane_below(int v)
{
    return __builtin_amdgcn_mov_dpp(v, 0x138 /* wave_shr:1 */, 0xf, 0xf, true);
}
__device__ __forceinline__ int path_from_lane_above(int v)
{
    return __builtin_amdgcn_mov_dpp(v, 0x130 /* wave_shl:1 */, 0xf, 0xf, true);
}

typedef int path_int4 __attribute__((ext_vector_type(4), aligned(4)));   // a lane's columns start anywhere

// one position, whole pyramid; lane = lane of the wavefront
__device__ __forceinline__ void path_window(int iteration, const int *__restrict__ gpuWall,
                                            const int *__restrict__ gpuSrc, int *__restrict__ gpuResults, int cols,
                                            int startStep, int border, int bx, int lane)
{
    constexpr int C = PATH_COLS_PER_LANE, AHEAD = PATH_ROWS_AHEAD;
    static_assert(C == 4, "a lane's columns of a row are one 16-byte load");
    const int small_block_cols = PATH_BLOCK_SIZE - iteration * PATH_HALO * 2;
    const int blkX = small_block_cols * bx - border;
    const int x0 = blkX + C * lane;       // the lane's first column

    int prev[C], floor_[C];               // floor_: what a column may not fall below
    unsigned column[C];                   // the column clamped to the grid
#pragma unroll
    for (int k = 0; k < C; ++k) {
        const int x = x0 + k;
        const bool off = x < 0 || x > cols - 1;
        column[k] = (unsigned)(x < 0 ? 0 : (off ? cols - 1 : x));
        floor_[k] = off ? 0x7fffffff : (int)0x80000000;
    }
    const int *const first = gpuWall + (long long)cols * startStep;
    const auto clamped_row = [&](const int *row, int (&v)[C]) {
#pragma unroll
        for (int k = 0; k < C; ++k) v[k] = row[column[k]];
    };
    const auto step = [&](const int (&w)[C]) {
        const int from_left = path_from_lane_below(prev[C - 1]);
        const int from_right = path_from_lane_above(prev[0]);
        int next[C];
#pragma unroll
        for (int k = 0; k < C; ++k) {
            const int left = k == 0 ? from_left : prev[k > 0 ? k - 1 : 0];
            const int right = k == C - 1 ? from_right : prev[k < C - 1 ? k + 1 : k];
            // (wraps where the sum does not fit, as the reference's does)
            next[k] = (int)((unsigned)min(min(left, prev[k]), right) + (unsigned)w[k]);
        }
#pragma unroll
        for (int k = 0; k < C; ++k) prev[k] = max(next[k], floor_[k]);
    };
    clamped_row(gpuSrc, prev);
#pragma unroll
    for (int k = 0; k < C; ++k) prev[k] = max(prev[k], floor_[k]);
    int w_last[C];
    clamped_row(first + (long long)cols * (iteration - 1), w_last);
    if (cols < C) {   // rows shorter than a lane's columns: nothing to win, every row read column by column
        for (int i = 0; i < iteration - 1; ++i) {
            int w[C];
            clamped_row(first + (long long)cols * i, w);
            step(w);
        }
        step(w_last);
    } else {
        // rows 0 .. middle - 1 go through the ring; a lane whole columns off the grid reads next to it.  Address:
        // a pointer to the window's first column of a row, the same for the whole wavefront, and an unsigned 32-bit
        // lane offset (from there, since a row may have 2^30 columns).
        const int middle = iteration - 1;
        const int window = __builtin_amdgcn_readfirstlane(min(max(blkX, 0), cols - 1));
        const unsigned at = (unsigned)(max(-(C - 1), min(x0, cols - 1)) - window + (C - 1)) * (unsigned)sizeof(int);
        const char *ahead = reinterpret_cast<const char *>(first + window - (C - 1));   // the row the next fetch takes
        int fetched = 0;
        int wall[AHEAD][C];
        const auto fetch = [&](int (&w)[C]) {
            const path_int4 v = *reinterpret_cast<const path_int4 *>(ahead + at);
#pragma unroll
            for (int k = 0; k < C; ++k) w[k] = v[k];
        };
        const auto next_row = [&]() {   // the last row again once there is no other: no load asks whether it is needed
            ahead += ++fetched < middle ? (long long)cols * (long long)sizeof(int) : 0ll;
        };
        if (middle > 0) {
            clamped_row(first, wall[0]);
            next_row();
#pragma unroll
            for (int u = 1; u < AHEAD; ++u) {
                if (middle > 1) fetch(wall[u]);   // (a middle of one row is the row read above)
                next_row();
            }
        }
        int base = 0;
        for (; base + AHEAD <= middle; base += AHEAD) {
#pragma unroll
            for (int u = 0; u < AHEAD; ++u) {
                step(wall[u]);
                fetch(wall[u]);
                next_row();
            }
        }
#pragma unroll
        for (int u = 0; u < AHEAD; ++u)
            if (base + u < middle) step(wall[u]);   // uniform
        step(w_last);
    }
    // the columns that took part in the last row: the middle of the window, where it is on the grid
#pragma unroll
    for (int k = 0; k < C; ++k) {
        const int tx = C * lane + k;
        if (tx >= iteration && tx <= PATH_BLOCK_SIZE - 1 - iteration && x0 + k >= 0 && x0 + k <= cols - 1)
            gpuResults[x0 + k] = prev[k];
    }
}

// Block positions [start, end) are served by the role's role_blocks x (role_threads / 64)
// wavefronts in turn; the position is the reference's bx (it uses block_pos itself, no wrap).
__device__ __forceinline__ void path_role(int iteration, const int *__restrict__ gpuWall,
                                          const int *__restrict__ gpuSrc, int *__restrict__ gpuResults, int cols,
                                          int startStep, int border, int role_block, int role_blocks, int start,
                                          int end, int tid, int role_threads)
{
    const int waves = role_threads / TK_WAVE_SIZE;
    const int wave = tid / TK_WAVE_SIZE;
    if (wave >= waves || start >= end || iteration <= 0 || 2 * iteration >= PATH_BLOCK_SIZE) return;
    const int lane = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    for (long long pos = (long long)start + role_block + (long long)role_blocks * wave; pos < end;
         pos += (long long)role_blocks * waves)
        path_window(iteration, gpuWall, gpuSrc, gpuResults, cols, startStep, border, (int)pos, lane);
}

}  // namespace tk
