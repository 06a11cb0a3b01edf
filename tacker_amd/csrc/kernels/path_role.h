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
//  * the window is moved until all of it lies on the grid (path_window_on_grid): its columns off the grid are
//    not read, and the wavefront has as many others instead.  The grid's edge is then the wavefront's, where the shift across
//    lanes leaves the neighbour at INT_MAX, which the minimum ignores -- min(prev, prev, right) and min(INT_MAX, prev,
//    right) are one value.  Nothing is clamped: a min3 and an add a column and the two shifts, 10 instructions a row.
//  * a row of the wall is one 16-byte load a lane, AHEAD rows ahead of the row being evaluated, from a scalar row
//    pointer that two instructions move on; whether there is such a row is asked for the last 2 AHEAD rows only.
// 1200 columns x 125 rows (200 windows on 200 CUs): 9.05 -> 6.5 us; 20000 x 125 (3292 windows) 44.4 -> 26.9, 20000 x 118 (1000)
// 13.6 -> 12.7, where a maximum a column held those off the grid at INT_MAX and every fetch asked for its row (14 vector
// instructions a row and 6 scalar ones).  Narrower grids keep that form (path_window).
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

__device__ __forceinline__ int path_min3(int a, int b, int c)
{
    int v;   // (left to itself, the compiler shares minima of two between columns: five instructions for four)
    asm("v_min3_i32 %0, %1, %2, %3" : "=v"(v) : "v"(a), "v"(b), "v"(c));
    return v;
}

typedef int path_int4 __attribute__((ext_vector_type(4), aligned(4)));   // a lane's columns start anywhere
typedef __attribute__((address_space(1))) path_int4 path_global_int4;
typedef __attribute__((address_space(1))) char path_global_char;

// One position, whole pyramid, on a grid of at least PATH_BLOCK_SIZE columns; lane = lane of the wavefront.  The wavefront's
// columns are the window moved until it lies on the grid.  (Columns of the window that are not on the grid nobody reads, and
// those the wavefront has instead are right for longer than the pyramid's.)
__device__ __forceinline__ void path_window_on_grid(int iteration, const int *__restrict__ gpuWall,
                                                    const int *__restrict__ gpuSrc, int *__restrict__ gpuResults, int cols,
                                                    int startStep, int border, int bx, int lane)
{
    constexpr int C = PATH_COLS_PER_LANE, AHEAD = PATH_ROWS_AHEAD;
    static_assert(C == 4 && C * TK_WAVE_SIZE == PATH_BLOCK_SIZE, "a lane's columns of a row are one 16-byte load");
    const int blkX = (PATH_BLOCK_SIZE - iteration * PATH_HALO * 2) * bx - border;
    const int first = __builtin_amdgcn_readfirstlane(min(max(blkX, 0), cols - PATH_BLOCK_SIZE));
    unsigned at = (unsigned)(C * lane) * (unsigned)sizeof(int);
    size_t ahead = reinterpret_cast<size_t>(gpuWall + (long long)cols * startStep + first);   // the row the next fetch takes
    const size_t row_bytes = (size_t)cols * sizeof(int);
    path_int4 wall[AHEAD], prev = *reinterpret_cast<const path_int4 *>(reinterpret_cast<const char *>(gpuSrc + first) + at);
    const auto fetch = [&](path_int4 &w, size_t to_next) {
        asm volatile("" : "+s"(ahead), "+v"(at));   // (a scalar pointer and a lane's offset, not a 64-bit vector address)
        w = *(const path_global_int4 *)((const path_global_char *)ahead + at);
        ahead += to_next;
    };
    // the neighbouring lanes' columns; beyond the wavefront's ends, which keep what they had, INT_MAX: the grid's edge, or a
    // column outside the pyramid
    int left = 0x7fffffff, right = 0x7fffffff;
    const auto step = [&](const path_int4 &w) {
        left = __builtin_amdgcn_update_dpp(left, prev[3], 0x138 /* wave_shr:1 */, 0xf, 0xf, false);
        right = __builtin_amdgcn_update_dpp(right, prev[0], 0x130 /* wave_shl:1 */, 0xf, 0xf, false);
        const int m1 = path_min3(prev[0], prev[1], prev[2]), m2 = path_min3(prev[1], prev[2], prev[3]);
        const int m0 = path_min3(left, prev[0], prev[1]), m3 = path_min3(prev[2], prev[3], right);
        // (wraps where the sum does not fit, as the reference's does)
        prev[0] = (int)((unsigned)m0 + (unsigned)w[0]);
        prev[3] = (int)((unsigned)m3 + (unsigned)w[3]);
        prev[1] = (int)((unsigned)m1 + (unsigned)w[1]);
        prev[2] = (int)((unsigned)m2 + (unsigned)w[2]);
    };
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) fetch(wall[u], u + 1 < iteration ? row_bytes : 0);   // (the last row again where there is no other)
    int row = 0;
    for (; row + 2 * AHEAD <= iteration; row += AHEAD) {   // no fetch asks whether there is a row
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
            step(wall[u]);
            fetch(wall[u], row_bytes);
            __builtin_amdgcn_sched_barrier(0);   // (eight steps and then eight fetches would wait for all of them)
        }
    }
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
        if (row + u < iteration) step(wall[u]);
        if (row + AHEAD + u < iteration) fetch(wall[u], row_bytes);
    }
#pragma unroll
    for (int u = 0; u < AHEAD; ++u)
        if (row + AHEAD + u < iteration) step(wall[u]);
    // the columns that took part in the last row: the middle of the window, where it is on the grid
#pragma unroll
    for (int k = 0; k < C; ++k) {
        const int x = first + C * lane + k, tx = x - blkX;
        if (tx >= iteration && tx <= PATH_BLOCK_SIZE - 1 - iteration) gpuResults[x] = prev[k];
    }
}

// The same on a grid narrower than the window.  A column off the grid is held at INT_MAX by a maximum, and the first and the last row
// are read column by column, from indices clamped to the grid: the lane's four columns are read as they lie, also where
// the row ends between them, and the elements beyond it are the neighbouring rows', inside the array for every other row.
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
        if (cols >= PATH_BLOCK_SIZE)   // uniform
            path_window_on_grid(iteration, gpuWall, gpuSrc, gpuResults, cols, startStep, border, (int)pos, lane);
        else
            path_window(iteration, gpuWall, gpuSrc, gpuResults, cols, startStep, border, (int)pos, lane);
}

}  // namespace tk
