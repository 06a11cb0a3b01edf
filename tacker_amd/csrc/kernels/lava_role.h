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
// block barriers.  Here wavefronts serve a box without a barrier, each with LDS of its own.  fp32; the exponential is
// the hardware's 2^x of -r2 a2 log2(e) where the reference calls CUDA's expf, and multiply-adds are fused:
// results agree within a tolerance, not bit for bit.
//
// What bounds it is VALU issue (measured, cycles of a SIMD an instruction with two or more wavefronts at work: 32-bit
// add, multiply, fused multiply-add 2.1, 4.2 where all three sources lie in one of four register banks or one is scalar, conversions and
// shifts 4.4, the exponential and lane swaps 8), so four things count.
//  * How many instructions a pair takes.  The force on i is a sum of w (xi - xj), w = qj vij; it is computed as
//    (xi - c) sum w - sum vij [qj (xj - c)], which leaves four multiply-adds a pair (v and the force together)
//    where the difference, its product and the sum of w take eight instructions.  c is about the middle of the home box, on a
//    coarse grid (LavaCentre).  The two terms are of the size of |x - c| sum w, so this is as exact as the differences only
//    where no pair much closer than that matters more than the rest: where a2 |x - c|^2 <= 1/2 (LAVA_CENTRED), and weights differ
//    little across the box.  Forces against 64 bits, 2-norm over the middle box of 3^3, 60 systems, differences / this form
//    where it is taken: unit boxes around the origin, v = |x|^2 / 2, alpha 0.35 12.3 / 12.0e-8, 0.5 13.3 / 13.0e-8; x and v in
//    0.1 ... 1 in every box, alpha 0.35 8.0 / 8.1e-8, 0.5 7.9 / 8.1e-8.  Where it is not taken it would be off by more: unit boxes,
//    alpha 1 25.8 / 30.7e-8, 2 58 / 86e-8 (with a centre off the grid, which cost 8 % at 0.5).  Those boxes take the differences, and
//    so does one in which v differ so much (LAVA_CENTRED_V) that a particle's weight on itself, which no force comes from, could
//    be larger than all the others' together: with one v of -30 among 0.1 ... 1 the form about the centre is off by 3.9e-4, they by 5.9e-7.
//    A total that is not finite is computed once more from them.
//  * What is computed per neighbour and not per pair.  A wavefront prepares the 100 neighbours of a part once, a lane
//    each: {scale v, -scale x, -scale y, -scale z} and {q, q (x - cx), q (y - cy), q (z - cz)} go to LDS and
//    come back as two 16-byte broadcast reads a step.  (By a vector load for every step and row of lanes, and four multiplies
//    behind it, this was a tenth of the time.)
//  * How full the lanes are.  The wavefront is four rows of 16 lanes: row g takes neighbours g, g + 4, g + 8, ... (25 of the
//    100), a lane LAVA_MAX_P = 6 of the first 96 home particles: 150 steps without an empty slot.  The last four
//    particles are four lanes side by side, 16 neighbours at a time: 7 steps, where a seventh particle a lane would take 25.
//  * What else could compute.  In domains of LAVA_TILES_FROM boxes or more the exponents come from the matrix units (below), and
//    a pair is four multiply-adds and the exponential.  Preparing a neighbour is 45 instructions then, which few home particles a wavefront do not
//    pay for: with three a lane 3^3 boxes 49 us for 37, 8^3 68 for 57, 12^3 146 for 138, 13^3 141 for 143, with six 16^3 225 for 257, 24^3 705 for 772.  (The bits
//    differ in the last place, so that the domain alone decides, and neither the launch nor the number of CUs; the figures are of 256.)
// A pair is 8 short instructions and the exponential otherwise, 12 from the differences; the exponentials go first (transcendentals_begin) where a
// lane has several.  At the end of a part the four rows' sums are added,
// (g0 + g2) + (g1 + g3), by lane swaps that add two values at once, which leaves component v, y, x, z of the
// total in row 0, 1, 2, 3; the total goes on from the output array.  24^3 boxes: 690 to 740 us (772 without the matrix units, 833 with neither, 1325 with
// neighbours by vector loads and seven particles a lane); 18^3 319 / - / 359 / 577, 9^3 65 / - / 71 / 116, 3^3 36.1 / - / 36.6 / 46.
//
// Few boxes: a box is then split over several wavefronts (P home particles a lane instead of 6, every particle
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
#include <cfloat>

#include "role_common.h"
#include "../header/lava_header.h"

namespace tk {

typedef __attribute__((address_space(4))) const box_str lava_const_box;

#define LAVA_ROWS 4                                     // rows of 16 lanes: neighbours are dealt to them in turn
#define LAVA_LANES 16                                   // home particles side by side in a row
#define LAVA_MAX_P 6                                    // home particles per lane when one wavefront serves a box
#define LAVA_TILES_P 3                                  // ... at least, where exponents come from the matrix units:
#define LAVA_TILES_FROM 2049                            // in domains of as many boxes
#define LAVA_WAVES_PER_SIMD 4                           // wavefronts of this role a SIMD holds (registers)
#define LAVA_STEPS (NUMBER_PAR_PER_BOX / LAVA_ROWS)     // neighbours a row takes per box
#define LAVA_CENTRED 0.72f                              // a2 log2(e) |x - c|^2 up to which forces are computed about the centre
#define LAVA_CENTRED_V 4.f                              // ... and a2 log2(e) times how far v - c x may differ: a weight on itself of 2^4 of the usual
#define LAVA_REST 4                                     // home particles behind the lanes' own ...
#define LAVA_REST_FROM (NUMBER_PAR_PER_BOX - LAVA_REST)
#define LAVA_REST_STEP (TK_WAVE_SIZE / LAVA_REST)       // ... and the neighbours they take a step
static_assert(NUMBER_PAR_PER_BOX % LAVA_ROWS == 0 && LAVA_LANES * LAVA_MAX_P == LAVA_REST_FROM, "rows and lanes come out even");
static_assert(NUMBER_PAR_PER_BOX > TK_WAVE_SIZE && NUMBER_PAR_PER_BOX <= 2 * TK_WAVE_SIZE, "two neighbours a lane are staged");

typedef __attribute__((address_space(3))) float4_t lava_lds_float4;
typedef __attribute__((address_space(3))) float lava_lds_float;
typedef unsigned lava_uint2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) lava_uint2 lava_lds_token;
typedef __bf16 lava_bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 lava_bf16x8 __attribute__((ext_vector_type(8)));
typedef float lava_float2 __attribute__((ext_vector_type(2)));

// The LDS of a wavefront, in float4s.  From the differences: two a neighbour.  About the centre: four tokens of 8 bytes a neighbour of
// half a box, a float4 each, and the home particles' x - c, y - c, z - c.  Behind either the last home particles.
#define LAVA_TOKENS 4
#define LAVA_HALF 48                                    // neighbours of a box's first half, three matrix instructions' rows; the second has four more
#define LAVA_STAGED (NUMBER_PAR_PER_BOX - LAVA_HALF)
#define LAVA_CHARGES (LAVA_STAGED * LAVA_TOKENS / 2)    // where what comes: {q, q (x - cx), ...} of the staged neighbours,
#define LAVA_OFFSETS (LAVA_CHARGES + LAVA_STAGED)       // the home particles' x - c,
#define LAVA_LAST (LAVA_OFFSETS + 3 * LAVA_REST_FROM / 4)   // the last home particles,
#define LAVA_LAST_SLOTS (LAVA_LAST + LAVA_REST)         // and their operand, [lane group][particle]
static_assert(LAVA_HALF % LAVA_LANES == 0 && LAVA_STAGED - LAVA_HALF == LAVA_REST, "the last four neighbours are a step of their own");
static_assert(LAVA_LAST >= 2 * NUMBER_PAR_PER_BOX && LAVA_STAGED <= TK_WAVE_SIZE, "a lane stages one neighbour of a half");

// role_wave: the calling wavefront's number within the role
template <int WAVES>
__device__ __forceinline__ lava_lds_float4 *lava_stage_of_wave(int role_wave)
{
    __shared__ __align__(16) float4_t lava_stage[WAVES][LAVA_LAST_SLOTS + LAVA_ROWS * LAVA_REST];
    return (lava_lds_float4 *)&lava_stage[role_wave][0];
}

// what a wavefront wrote to its own LDS is there for all its lanes (LDS serves a wavefront in order), and what it read is read
__device__ __forceinline__ void lava_stage_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

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

// v plus the value n lanes further along the row of 16 (around its end)
template <int N>
__device__ __forceinline__ float lava_add_along_row(float v)
{
    return v + __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(v), 0x120 + N, 0xf, 0xf, false));
}

template <int N>
__device__ __forceinline__ float lava_max_along_row(float v)
{
    return __builtin_fmaxf(v, __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(v), 0x120 + N, 0xf, 0xf, false)));
}

// The median of three thirds' means of a value that every home particle has -- lo of particle `lane`, hi of particle 64 + lane --
// which one particle far away, or one that is no number, does not move; 0 where that is not finite either.
__device__ __forceinline__ float lava_middle(float lo, float hi, int lane)
{
    float v = lo + (lane + TK_WAVE_SIZE < NUMBER_PAR_PER_BOX ? hi : 0.f);
    v = lava_add_along_row<8>(v);
    v = lava_add_along_row<4>(v);
    v = lava_add_along_row<2>(v);
    v = lava_add_along_row<1>(v);
    float row[LAVA_ROWS];
#pragma unroll
    for (int g = 0; g < LAVA_ROWS; ++g)
        row[g] = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), LAVA_LANES * g));
    // particles 0 - 15 and 64 - 79, 16 - 31 and 80 - 95, 32 - 63 and 96 - 99
    const float m = __builtin_amdgcn_fmed3f(row[0] * (1.f / 32), row[1] * (1.f / 32), (row[2] + row[3]) * (1.f / 36));
    return __builtin_fabsf(m) <= FLT_MAX ? m : 0.f;
}

// the largest of a value of every lane
__device__ __forceinline__ float lava_largest(float v)
{
    v = lava_max_along_row<8>(v);
    v = lava_max_along_row<4>(v);
    v = lava_max_along_row<2>(v);
    v = lava_max_along_row<1>(v);
    float most = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), 0));
#pragma unroll
    for (int g = 1; g < LAVA_ROWS; ++g)
        most = __builtin_fmaxf(most, __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), LAVA_LANES * g)));
    return most;
}

// a value that all lanes have, in a scalar register
__device__ __forceinline__ float lava_scalar(float v) { return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(v))); }

// About the middle of the home box, which its forces are computed about, the same for every wavefront that serves a part of it.
struct LavaCentre {
    float at[3];
    bool use;   // the box allows it
    __device__ __forceinline__ LavaCentre(const float4_t *rA, float scale, int lane)
    {
        const float4_t lo = rA[lane], hi = rA[min(lane + TK_WAVE_SIZE, NUMBER_PAR_PER_BOX - 1)];
        float across = 0.f;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            at[c] = lava_middle(lo[c + 1], hi[c + 1], lane);
            across = __builtin_fmaxf(across, __builtin_fmaxf(__builtin_fabsf(lo[c + 1] - at[c]), __builtin_fabsf(hi[c + 1] - at[c])));
        }
        // on a grid of an eighth to a quarter of the box's half width: x - c is then exact for most coordinates, and its
        // rounding was what the form about the centre lost most by
        const int grid = __builtin_amdgcn_frexp_expf(lava_largest(across)) - 3;
        float lo2 = 0.f, hi2 = 0.f;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            at[c] = lava_scalar(__builtin_ldexpf(__builtin_rintf(__builtin_ldexpf(at[c], -grid)), grid));
            lo2 += (lo[c + 1] - at[c]) * (lo[c + 1] - at[c]);
            hi2 += (hi[c + 1] - at[c]) * (hi[c + 1] - at[c]);
        }
        use = -scale * lava_largest(__builtin_fmaxf(lo2, hi2)) <= LAVA_CENTRED;   // (not where a2 is no number)
        // what the v of its particles make of their weights beside the others': v - c x
        lo2 = lo[0], hi2 = hi[0];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            lo2 = __builtin_fmaf(-at[c], lo[c + 1], lo2);
            hi2 = __builtin_fmaf(-at[c], hi[c + 1], hi2);
        }
        const float most = lava_largest(__builtin_fmaxf(lo2, hi2)), least = -lava_largest(__builtin_fmaxf(-lo2, -hi2));
        use = use && -scale * (most - least) <= LAVA_CENTRED_V;
    }
};

// The exponent -r2 a2 log2(e) = scale vi + scale vj + xi (-scale xj) + yi (-scale yj) + zi (-scale zj) by the matrix units.  A float is
// the sum of three bf16 pieces, each the rest rounded to nearest, whose products are exact in a matrix instruction's fp32 sum:
// eight of the nine products of pieces of a coordinate (not the one of the two last, 2^-32 of it), three coordinates, and the pieces of the
// two v are 30 of the 32 slots of one v_mfma_f32_16x16x32_bf16, which gives 256 exponents in 16 cycles of a SIMD where an add and
// three multiply-adds take 44, and leaves the vector units to other wavefronts part of the time.  A lane gets the exponents of one home
// particle, lane % 16 of a tile, and four neighbours, 4 (lane / 16) .. of 16.
//
// A neighbour is four tokens of four bf16 in LDS, pieces 1, 2, 2 and 3 of its coordinates beside 1 and pieces 1, 2, 3 of its v; lanes
// 16 g .. hold slots 8 g .. of an operand, two tokens, in the order in which the sum of products has least error (2-norm against 64 bits, of
// the add and multiply-adds / of this: v and x in 0.1 ... 1, alpha 0.5 3.4 / 2.4e-8; unit boxes, v = |x|^2 / 2, alpha 0.5 2.9 / 1.8e-8, 2 46 / 28e-8;
// with the largest products last 2.4, 2.0 and 32e-8, with both v as the sum the instruction starts from 3.1, 2.5 and 41e-8).

// the next pieces of two values, which lose them
__device__ __forceinline__ unsigned lava_pieces(float &a, float &b)
{
    const unsigned p = __builtin_bit_cast(unsigned, __builtin_convertvector(lava_float2{a, b}, lava_bf16x2));
    a -= __uint_as_float(p << 16);
    b -= __uint_as_float(p & 0xffff0000u);
    return p;
}
#define LAVA_ONE 0x3f80u   // 1 in bf16

__device__ __forceinline__ void lava_put_neighbour(lava_lds_token *to, float v, float x, float y, float z)
{
    unsigned xy[3], zv[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        xy[i] = lava_pieces(x, y);
        zv[i] = lava_pieces(z, v);
    }
    to[0] = lava_uint2{xy[0], (zv[0] & 0xffffu) | LAVA_ONE << 16};
    to[1] = lava_uint2{xy[1], (zv[1] & 0xffffu) | (zv[0] & 0xffff0000u)};
    to[2] = lava_uint2{xy[1], zv[1]};
    to[3] = lava_uint2{xy[2], zv[2]};
}

// the home particle's operand: slots of lane group g
__device__ __forceinline__ lava_bf16x8 lava_home_slots(float4_t home, int g)
{
    float v = home[0], x = home[1], y = home[2], z = home[3];
    unsigned xy[3], zv[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        xy[i] = lava_pieces(x, y);
        zv[i] = lava_pieces(z, v);
    }
    // lane masks in place of selects, which become branches around the pieces
    const unsigned is0 = 0u - (unsigned)(g == 0), is1 = 0u - (unsigned)(g == 1), late = ~(is0 | is1), odd = 0u - (unsigned)(g & 1);
    const unsigned a_xy = (xy[0] & is0) | (xy[1] & is1) | (xy[2] & late);
    const unsigned a_zv = (zv[0] & is0) | (zv[1] & is1) | (zv[2] & late & (g == 3 ? 0xffffu : ~0u));
    const unsigned b_xy = (xy[1] & odd) | (xy[0] & ~odd);
    const unsigned b_zv = ((zv[1] & odd) | (zv[0] & ~odd)) & 0xffffu;
    return __builtin_bit_cast(lava_bf16x8, uint4_t{a_xy, a_zv, b_xy, b_zv | (g == 3 ? 0u : LAVA_ONE << 16)});
}

// The neighbour's operand of lane group g: tokens 0 and 1 + g, of the last group 2 and 3
struct LavaSlots {
    const lava_lds_token *first, *second;   // of neighbour lane % 16
    __device__ __forceinline__ LavaSlots(const lava_lds_token *tokens, int neighbour, int g)
        : first(tokens + LAVA_TOKENS * neighbour + (g == 3 ? 2 : 0)), second(tokens + LAVA_TOKENS * neighbour + (g == 3 ? 3 : 1 + g)) {}
    __device__ __forceinline__ lava_bf16x8 at(int from) const
    {
        const lava_uint2 a = first[LAVA_TOKENS * from], b = second[LAVA_TOKENS * from];
        return __builtin_bit_cast(lava_bf16x8, uint4_t{a.x, a.y, b.x, b.y});
    }
};

// P home particles a lane about the centre: their operands and sums, and the last four's
template <int P>
struct LavaTiles {
    lava_bf16x8 home[P];
    float4_t f[P], g;   // sums of w, and of vij q (x - c), component by component
    lava_lds_float4 *stage;
    int lane;
    bool rest;

    __device__ __forceinline__ static float4_t exponents(const lava_bf16x8 &neighbours, const lava_bf16x8 &of)
    {
        const float4_t zero = {0.f, 0.f, 0.f, 0.f};
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(neighbours, of, zero, 0, 0, 0);
    }
    // ROWS exponents a lane (4: of 16 neighbours; 1: of the last four, every fourth row of the operand), charges from `at` on
    template <int ROWS>
    __device__ __forceinline__ void add(const lava_bf16x8 &neighbours, const lava_lds_float4 *at)
    {
        float4_t b[ROWS];
#pragma unroll
        for (int r = 0; r < ROWS; ++r) b[r] = at[r];
        constexpr int AHEAD = P == 1 ? 1 : 2;
        float4_t now[AHEAD];
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) now[u] = exponents(neighbours, home[u]);
#pragma unroll
        for (int k = 0; k < P; k += AHEAD) {
            float4_t next[AHEAD];
#pragma unroll
            for (int u = 0; u < AHEAD; ++u)
                next[u] = k + AHEAD + u < P ? exponents(neighbours, home[k + AHEAD + u < P ? k + AHEAD + u : 0]) : now[u];
            transcendentals_begin();
#pragma unroll
            for (int r = 0; r < ROWS; ++r)
#pragma unroll
                for (int u = 0; u < AHEAD; ++u) now[u][r] = __builtin_amdgcn_exp2f(now[u][r]);
            transcendentals_end();
#pragma unroll
            for (int r = 0; r < ROWS; ++r)
#pragma unroll
                for (int c = 0; c < 4; ++c)
#pragma unroll
                    for (int u = 0; u < AHEAD; ++u)
                        if (k + u < P) f[k + u][c] = __builtin_fmaf(now[u][r], b[r][c], f[k + u][c]);
#pragma unroll
            for (int u = 0; u < AHEAD; ++u) now[u] = next[u];
        }
    }
    // the last four home particles: every fourth column of a tile is the same one, and takes a row of its own
    __device__ __forceinline__ void add_last(const lava_bf16x8 &neighbours, const lava_lds_float4 *of, bool all)
    {
        const float4_t e = exponents(neighbours, __builtin_bit_cast(lava_bf16x8, stage[LAVA_LAST_SLOTS + lane / LAVA_LANES * LAVA_REST + lane % LAVA_REST]));
        const int r = (lane / LAVA_REST) & 3;
        const float lo = r & 1 ? e[1] : e[0], hi = r & 1 ? e[3] : e[2];
        const float w = __builtin_amdgcn_exp2f(r & 2 ? hi : lo);
        if (all || r == 0) {
            const float4_t b = *of;
#pragma unroll
            for (int c = 0; c < 4; ++c) g[c] = __builtin_fmaf(w, b[c], g[c]);
        }
    }
    // half a box's neighbours, which are staged
    template <bool SECOND>
    __device__ __forceinline__ void half()
    {
        const int row = lane / LAVA_LANES, column = lane % LAVA_LANES;
        const lava_lds_token *tokens = (const lava_lds_token *)stage;
        const lava_lds_float4 *charges = stage + LAVA_CHARGES;
        const LavaSlots slots(tokens, column, row);
        lava_bf16x8 n = slots.at(0);
#pragma unroll 1
        for (int t = 0; t < LAVA_HALF; t += LAVA_LANES) {
            const lava_bf16x8 now = n;
            n = slots.at(t + LAVA_LANES < LAVA_HALF ? t + LAVA_LANES : 0);   // (the last read is not used)
            add<4>(now, charges + t + LAVA_ROWS * row);
        }
        __builtin_amdgcn_sched_barrier(0);
        const LavaSlots end(tokens, LAVA_HALF + column / LAVA_ROWS, row);
        if (SECOND) add<1>(end.at(0), charges + LAVA_HALF + row);
        __builtin_amdgcn_sched_barrier(0);
        if (!rest) return;   // uniform
#pragma unroll
        for (int t = 0; t < LAVA_HALF; t += LAVA_LANES) add_last(slots.at(t), charges + t + lane / LAVA_REST, true);
        if (SECOND) add_last(end.at(0), charges + LAVA_HALF + row, false);
    }
};

// Where the particles of a box's parts begin.  A neighbour is named by its number alone (its offset in the list is not read): two loads behind
// one another, and the particles behind them.  The number is fetched three parts ahead, the offset two, the particles up to one; where there
// is no such part, the home box's own are read.
struct LavaWalk {
    const lava_const_box *boxes;
    int bx, part_end, after_next;
    long now, next;
    __device__ __forceinline__ int box_of(int part) const { return part == 0 || part >= part_end ? bx : boxes[bx].nei[part - 1].number; }
    __device__ __forceinline__ LavaWalk(const lava_const_box *boxes_, int box, int part_begin, int part_end_) : boxes(boxes_), bx(box), part_end(part_end_)
    {
        now = boxes[box_of(part_begin)].offset;
        next = boxes[box_of(part_begin + 1)].offset;
        after_next = box_of(part_begin + 2);
    }
    __device__ __forceinline__ void go_on(int part)   // to the part behind `part`
    {
        now = next;
        next = boxes[after_next].offset;
        after_next = box_of(part + 3);
    }
};

// Parts [part_begin, part_end) of box `bx` about the centre, added to the totals of P home particles a lane (first: the
// wavefront's first one) and of the last four.
template <int P>
__device__ __forceinline__ void lava_parts_centred(const float scale, LavaWalk walk, const FOUR_VECTOR *d_rv_gpu,
                                                   const float *d_qv_gpu, int part_begin, int part_end, const float4_t *rA, int first,
                                                   const float (&centre)[3], bool rest, int lane, lava_lds_float4 *stage,
                                                   float (&total)[P], float &last_total)
{
    float4_t r;   // the half that is staged next
    float q;
    const auto fetch = [&](unsigned j) {
        r = reinterpret_cast<const float4_t *>(d_rv_gpu + walk.now)[j];
        q = d_qv_gpu[walk.now + j];
    };
    fetch(lane);
    LavaTiles<P> tiles;
    tiles.stage = stage;
    tiles.lane = lane;
    tiles.rest = rest;
    lava_lds_float *const offsets = (lava_lds_float *)(stage + LAVA_OFFSETS);
    const int row = lane / LAVA_LANES, column = lane % LAVA_LANES;
    const float4_t *own = rA + (first + column);
#pragma unroll
    for (int k = 0; k < P; ++k) {
        float4_t home = own[k * LAVA_LANES];
#pragma unroll
        for (int c = 0; c < 3; ++c) offsets[c * LAVA_REST_FROM + k * LAVA_LANES + column] = home[c + 1] - centre[c];   // (the rows alike)
        home[0] *= scale;
        tiles.home[k] = lava_home_slots(home, row);
    }
    lava_stage_fence();
    const float4_t last = stage[LAVA_LAST + (lane & (LAVA_REST - 1))];   // {scale v, x, y, z}
    stage[LAVA_LAST_SLOTS + row * LAVA_REST + lane % LAVA_REST] = __builtin_bit_cast(float4_t, lava_home_slots(last, row));   // (four lanes alike)
    for (int part = part_begin; part < part_end; ++part) {
        const auto put = [&]() {
            lava_put_neighbour((lava_lds_token *)stage + LAVA_TOKENS * lane, scale * r[0], -scale * r[1], -scale * r[2], -scale * r[3]);
            stage[LAVA_CHARGES + lane] = float4_t{q, q * (r[1] - centre[0]), q * (r[2] - centre[1]), q * (r[3] - centre[2])};
        };
#pragma unroll
        for (int k = 0; k < P; ++k) tiles.f[k] = float4_t{0.f, 0.f, 0.f, 0.f};
        tiles.g = float4_t{0.f, 0.f, 0.f, 0.f};
        transcendentals_begin();
        if (lane < LAVA_HALF) put();
        transcendentals_end();
        fetch(min(lane + LAVA_HALF, NUMBER_PAR_PER_BOX - 1));
        lava_stage_fence();
        tiles.template half<false>();
        lava_stage_fence();
        transcendentals_begin();
        if (lane < LAVA_STAGED) put();
        transcendentals_end();
        walk.go_on(part);
        fetch(lane);
        lava_stage_fence();
        tiles.template half<true>();
        asm volatile("" : "+v"(lane));   // (what follows from it here needs no registers up there)
        transcendentals_begin();
        const lava_lds_float *offset = offsets + lane % LAVA_LANES;
        const float twice = lane < LAVA_LANES ? 1.0f : 2.0f;   // row 0 has v; fs = 2 vij in the force components
#pragma unroll
        for (int k = 0; k < P; ++k) {
            float4_t &f = tiles.f[k];
#pragma unroll
            for (int c = 1; c < 4; ++c)
                f[c] = __builtin_fmaf(offset[(c - 1) * LAVA_REST_FROM + k * LAVA_LANES], f[0], -f[c]);
            total[k] += twice * lava_fold_rows(lava_fold_halves(f[0], f[1]), lava_fold_halves(f[2], f[3]));
        }
        lava_stage_fence();
        if (!rest) {   // uniform
            transcendentals_end();
            continue;
        }
        float4_t g = tiles.g;
        const float4_t end = stage[LAVA_LAST + (lane & (LAVA_REST - 1))];
#pragma unroll
        for (int c = 1; c < 4; ++c) g[c] = __builtin_fmaf(end[c] - centre[c - 1], g[0], -g[c]);
#pragma unroll
        for (int c = 0; c < 4; ++c) g[c] = lava_add_along_row<4>(lava_add_along_row<8>(g[c]));
        last_total += twice * lava_fold_rows(lava_fold_halves(g[0], g[1]), lava_fold_halves(g[2], g[3]));
        transcendentals_end();
    }
}

// The forces of the staged part on P home particles a lane -- and on the last four, if `rest` -- added to their totals: about
// the centre c (CENTRED), or from the differences of the coordinates.
template <int P, bool CENTRED>
__device__ __forceinline__ void lava_part(const float4_t (&home)[P], const float (&centre)[3], int row, float twice, bool rest,
                                          const lava_lds_float4 *rest_home, int lane, const lava_lds_float4 *stage,
                                          float (&total)[P], float &last_total)
{
    float4_t f[P];   // sums of w, and of vij q (x - c) -- or of w (xi - xj) -- component by component
#pragma unroll
    for (int k = 0; k < P; ++k) f[k] = float4_t{0.f, 0.f, 0.f, 0.f};
    const lava_lds_float4 *at = stage + 2 * row;
    float4_t a = at[0], b = at[1];
    // Six particles a lane are chains enough for the compiler to interleave as it likes (24^3 boxes, when they took this loop, 829 us, with the step's
    // read held in front of it 871); with fewer, the reads stay in front of a step's work and every step is written out (3^3 boxes
    // 36.5 us; 42.1 in a loop of five steps, 43.2 as the compiler likes).
#pragma unroll P < LAVA_MAX_P ? LAVA_STEPS : 5
    for (int t = 0; t < LAVA_STEPS; ++t) {
        at += 2 * LAVA_ROWS;
        const lava_lds_float4 *next = t + 1 < LAVA_STEPS ? at : stage;   // (the last read is not used)
        const float4_t na = next[0], nb = next[1];
        if (P < LAVA_MAX_P) __builtin_amdgcn_sched_barrier(0);
        // scale (vi + vj - (xi xj + yi yj + zi zj)) = -r2 a2 log2(e), stage by stage over the lane's
        // particles: their chains are independent, and in this order none waits for its own last result.  With one particle a lane there is one
        // exponential, and holding it in front of the rest gains nothing where wavefronts share a SIMD (8^3 boxes 56.8 us for 57.2, 9^3 72.1 for 72.2, 11^3
        // 117.5 for 116.4) and costs where they do not (2^3 to 5^3 14.5 to 40.2 for 13.7 to 38.0); with two, 12^3 boxes 133.4 for 135.4.
        float w[P];
#pragma unroll
        for (int k = 0; k < P; ++k) w[k] = home[k][0] + a[0];
#pragma unroll
        for (int c = 1; c < 4; ++c)
#pragma unroll
            for (int k = 0; k < P; ++k) w[k] = __builtin_fmaf(home[k][c], a[c], w[k]);
        if (P > 1) transcendentals_begin();
#pragma unroll
        for (int k = 0; k < P; ++k) w[k] = __builtin_amdgcn_exp2f(w[k]);
        if (P > 1) transcendentals_end();
        if (CENTRED) {
#pragma unroll
            for (int c = 0; c < 4; ++c)
#pragma unroll
                for (int k = 0; k < P; ++k) f[k][c] = __builtin_fmaf(w[k], b[c], f[k][c]);
        } else {
#pragma unroll
            for (int k = 0; k < P; ++k) w[k] *= b[0];
#pragma unroll
            for (int k = 0; k < P; ++k) f[k][0] += w[k];
#pragma unroll
            for (int c = 1; c < 4; ++c)
#pragma unroll
                for (int k = 0; k < P; ++k) f[k][c] = __builtin_fmaf(w[k], home[k][c] - b[c], f[k][c]);
        }
        if (P < LAVA_MAX_P) __builtin_amdgcn_sched_barrier(0);
        a = na;
        b = nb;
    }
#pragma unroll
    for (int k = 0; k < P; ++k) {
        if (CENTRED) {
#pragma unroll
            for (int c = 1; c < 4; ++c) f[k][c] = __builtin_fmaf(home[k][c] - centre[c - 1], f[k][0], -f[k][c]);
        }
        total[k] += twice * lava_fold_rows(lava_fold_halves(f[k][0], f[k][1]), lava_fold_halves(f[k][2], f[k][3]));
    }
    if (!rest) return;   // uniform
    const float4_t last = rest_home[lane & (LAVA_REST - 1)];
    float4_t g = {0.f, 0.f, 0.f, 0.f};
    const auto pair = [&](int j) {
        const float4_t a = stage[2 * j], b = stage[2 * j + 1];
        float w = last[0] + a[0];
#pragma unroll
        for (int c = 1; c < 4; ++c) w = __builtin_fmaf(last[c], a[c], w);
        w = __builtin_amdgcn_exp2f(w);
        if (!CENTRED) w *= b[0];
        g[0] = CENTRED ? __builtin_fmaf(w, b[0], g[0]) : g[0] + w;
#pragma unroll
        for (int c = 1; c < 4; ++c) g[c] = __builtin_fmaf(w, CENTRED ? b[c] : last[c] - b[c], g[c]);
    };
    const int from = lane / LAVA_REST;
#pragma unroll
    for (int j = 0; j + LAVA_REST_STEP <= NUMBER_PAR_PER_BOX; j += LAVA_REST_STEP) pair(j + from);
    if (from < NUMBER_PAR_PER_BOX % LAVA_REST_STEP) pair(NUMBER_PAR_PER_BOX / LAVA_REST_STEP * LAVA_REST_STEP + from);
    if (CENTRED) {
#pragma unroll
        for (int c = 1; c < 4; ++c) g[c] = __builtin_fmaf(last[c] - centre[c - 1], g[0], -g[c]);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) g[c] = lava_add_along_row<4>(lava_add_along_row<8>(g[c]));
    last_total += twice * lava_fold_rows(lava_fold_halves(g[0], g[1]), lava_fold_halves(g[2], g[3]));
}

// Parts [part_begin, part_end) of box `bx`, added to the totals of its home particles as lava_part does.
template <int P, bool CENTRED>
__device__ __forceinline__ void lava_parts(const float scale, LavaWalk walk, const FOUR_VECTOR *d_rv_gpu,
                                           const float *d_qv_gpu, int part_begin, int part_end, const float4_t (&home)[P],
                                           const float (&centre)[3], bool rest, int lane, lava_lds_float4 *stage,
                                           float (&total)[P], float &last_total)
{
    const int row = lane / LAVA_LANES;
    const float twice = row == 0 ? 1.0f : 2.0f;   // fs = 2 vij in the force components
    const int second = min(lane + TK_WAVE_SIZE, NUMBER_PAR_PER_BOX - 1);   // a lane's second neighbour (past the last: not used)
    float4_t r0, r1;
    float q0, q1;
    const auto fetch = [&]() {
        const float4_t *rB = reinterpret_cast<const float4_t *>(d_rv_gpu + walk.now);
        const float *qB = d_qv_gpu + walk.now;
        r0 = rB[lane];
        r1 = rB[second];
        q0 = qB[lane];
        q1 = qB[second];
    };
    fetch();
    for (int part = part_begin; part < part_end; ++part) {
        const auto put = [&](int j, const float4_t &r, float q) {
            stage[2 * j] = float4_t{scale * r[0], -scale * r[1], -scale * r[2], -scale * r[3]};
            stage[2 * j + 1] = CENTRED ? float4_t{q, q * (r[1] - centre[0]), q * (r[2] - centre[1]), q * (r[3] - centre[2])}
                                       : float4_t{q, r[1], r[2], r[3]};
        };
        // the wavefront's reads of the part before are behind it: LDS serves a wavefront in order
        put(lane, r0, q0);
        if (lane < NUMBER_PAR_PER_BOX - TK_WAVE_SIZE) put(lane + TK_WAVE_SIZE, r1, q1);
        walk.go_on(part);
        fetch();
        lava_stage_fence();
        lava_part<P, CENTRED>(home, centre, row, twice, rest, stage + LAVA_LAST, lane, stage, total, last_total);
        lava_stage_fence();
    }
}

// box `bx`, parts [part_begin, part_end) of its list, for the 16 P home particles from 16 P `sub` on -- and the last four,
// if `rest` -- by one wavefront.  scale = -a2 log2(e).  stage: this wavefront's LDS.
template <int P>
__device__ __forceinline__ void lava_box(const float scale, const box_str *d_box_gpu, const FOUR_VECTOR *d_rv_gpu,
                                         const float *d_qv_gpu, FOUR_VECTOR *d_fv_gpu, bool tiles, int bx, int sub, bool rest,
                                         int part_begin, int part_end, int lane, lava_lds_float4 *stage)
{
    asm volatile("" : "+v"(lane));   // what follows from it is not kept through a launch, in registers that it does not have
    const lava_const_box *boxes = (const lava_const_box *)d_box_gpu;
    const long first_i = boxes[bx].offset;
    const int neighbours = boxes[bx].nn;
    if (part_end > 1 + neighbours) part_end = 1 + neighbours;
    if (part_begin >= part_end) return;
    const LavaWalk walk(boxes, bx, part_begin, part_end);   // (first of all: two trips to memory one after the other)
    const float4_t *rA = reinterpret_cast<const float4_t *>(d_rv_gpu + first_i);
    const int first = sub * P * LAVA_LANES;
    // where a lane's totals go: component v, y, x, z in row 0, 1, 2, 3
    const auto out = [&]() {
        const int row = lane / LAVA_LANES, component = row == 1 ? 2 : (row == 2 ? 1 : row);
        return reinterpret_cast<float *>(d_fv_gpu + first_i) + component;
    };
    float total[P], last_total;
    float *fA = out();
    const auto slot = [&](int k) -> float & { return fA[4 * (first + lane % LAVA_LANES) + 4 * LAVA_LANES * k]; };
    const auto last_slot = [&]() -> float & { return fA[4 * (LAVA_REST_FROM + lane % LAVA_REST)]; };
#pragma unroll
    for (int k = 0; k < P; ++k) total[k] = slot(k);
    last_total = last_slot();
    float4_t home[P];   // {scale v, x, y, z}; of six a lane only where they are used next, for want of registers
    const auto load_home = [&]() {
        const float4_t *own = rA + (first + lane % LAVA_LANES);
#pragma unroll
        for (int k = 0; k < P; ++k) {
            home[k] = own[k * LAVA_LANES];
            home[k][0] *= scale;
        }
    };
    if (P < LAVA_MAX_P) load_home();
    if (lane < LAVA_REST) {
        float4_t r = rA[LAVA_REST_FROM + lane];
        r[0] *= scale;
        stage[LAVA_LAST + lane] = r;
    }
    const LavaCentre centre(rA, scale, lane);
    unsigned todo = ~0u;   // bit k, or P: this total is still to be computed
    if (centre.use) {
        if constexpr (P >= LAVA_TILES_P) {
            if (tiles) lava_parts_centred<P>(scale, walk, d_rv_gpu, d_qv_gpu, part_begin, part_end, rA, first, centre.at, rest, lane, stage, total, last_total);
        }
        if (P < LAVA_TILES_P || !tiles) {
            if (P == LAVA_MAX_P) load_home();
            lava_parts<P, true>(scale, walk, d_rv_gpu, d_qv_gpu, part_begin, part_end, home, centre.at, rest, lane, stage, total, last_total);
        }
        // What is not finite is computed once more from the differences, from where it began: they are finite where a charge and a distance
        // whose product is not meet a weight of zero, and have signs where weights are infinite.
        asm volatile("" : "+v"(lane));   // (as above)
        fA = out();
        todo = 0;
        const auto keep = [&](int k, float &in_memory, float &value) {
            if (__builtin_fabsf(value) <= FLT_MAX) {
                in_memory = value;
            } else {
                value = in_memory;
                todo |= 1u << k;
            }
        };
#pragma unroll
        for (int k = 0; k < P; ++k) keep(k, slot(k), total[k]);
        if (rest && lane % LAVA_LANES < LAVA_REST) keep(P, last_slot(), last_total);
        if (__builtin_amdgcn_ballot_w64(todo != 0) == 0) return;
    }
    if (P == LAVA_MAX_P) load_home();
    lava_parts<P, false>(scale, walk, d_rv_gpu, d_qv_gpu, part_begin, part_end, home, centre.at, rest, lane, stage, total, last_total);
#pragma unroll
    for (int k = 0; k < P; ++k)
        if (todo >> k & 1) slot(k) = total[k];
    if (rest && lane % LAVA_LANES < LAVA_REST && (todo >> P & 1)) last_slot() = last_total;
}

// wavefronts a box is split over with P home particles a lane
__device__ __forceinline__ constexpr int lava_subs(int P)
{
    return LAVA_REST_FROM / (LAVA_LANES * P);
}

// Which wavefront takes what.  A unit is a box, or a part of its home particles: the first `whole` boxes are one
// unit each (6 particles a lane), the boxes behind them `subs` units each of 16 P particles.  A wavefront serves
// the units it owns -- first_owned, first_owned + stride, ... -- through all phases of a launch.
struct LavaUnits {
    int whole;   // boxes of one unit each
    int p;       // particles per lane of the others' units
    int subs;    // units each of them makes
    bool tiles;  // exponents from the matrix units

    // `waves` wavefronts serve `boxes` boxes.  Whole rounds of as many boxes as wavefronts are at work at a time
    // take a box each; what is left over -- all of it when the domain is small -- is cut: a box is 0.1 to 0.3 ms of
    // one wavefront, with up to 4 of them on a SIMD, and a last round of few boxes would leave most of the chip idle that
    // long.  Finer cuts spread better, but every wavefront prepares the neighbours again and a read serves fewer pairs.  Taken is the finest cut
    // that gives no wavefront at work two units (*).  us with everything left over in units of 6 / 3 / 2 / 1 particles a lane, in a launch of more
    // wavefronts than are at work at a time:
    //     8^3 (512 boxes) 110 / 65 / 64 / 57*,  9^3 (729) 109 / 81 / 66* / 72,  10^3 (1000) 110 / 82 / 85* / 95,  11^3 (1331) 144 / 109 / 105* / 116,
    //     12^3 (1728) 145 / 129* / 135 / 144;  with exponents from the matrix units, 6 or 3: 13^3 (2197) 133* / 143,  15^3 (3375) 210* / 219,
    //     18^3 (4096 + 1736) 335 / 319*,  24^3 (3 x 4096 + 1536) 731 / 737*.
    __device__ __forceinline__ LavaUnits(int boxes, int waves, bool tiles_) : tiles(tiles_)
    {
        const int at_once = min(waves, LAVA_WAVES_PER_SIMD * 4 * TK_CU_NUM);
        whole = boxes / at_once * at_once;
        const int left = boxes - whole;
        p = left * lava_subs(LAVA_TILES_P) <= at_once ? LAVA_TILES_P : LAVA_MAX_P;
        if (!tiles && left * lava_subs(2) <= at_once) p = left * lava_subs(1) <= at_once ? 1 : 2;
        subs = p == 1 ? lava_subs(1) : (p == 2 ? lava_subs(2) : (p == 3 ? lava_subs(3) : 1));
    }
    __device__ __forceinline__ int first_of(int box) const { return box <= whole ? box : whole + (box - whole) * subs; }
};

// One phase of a launch: boxes [box_lo, box_hi) each walk parts [part_begin, part_end).
__device__ __forceinline__ void lava_phase(const LavaUnits units, int box_lo, int box_hi, int part_begin, int part_end,
                                           const float scale, const box_str *d_box_gpu, const FOUR_VECTOR *d_rv_gpu,
                                           const float *d_qv_gpu, FOUR_VECTOR *d_fv_gpu, int first_owned, int stride,
                                           int lane, lava_lds_float4 *stage)
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
        const bool rest = left < 0 || sub == units.subs - 1;
#define LAVA_BOX(P_) lava_box<P_>(scale, d_box_gpu, d_rv_gpu, d_qv_gpu, d_fv_gpu, units.tiles, box, sub, rest, part_begin, part_end, lane, stage)
        if (p == LAVA_MAX_P) LAVA_BOX(LAVA_MAX_P);
        else if (p == 3) LAVA_BOX(3);
        else if (p == 2) LAVA_BOX(2);
        else LAVA_BOX(1);
#undef LAVA_BOX
    }
}

// grid_dimension_x: boxes (the reference's grid); the position grid has the boxes as columns and the
// LAVA_PARTS parts as rows.  A range that runs past the grid wraps.
// WAVES: wavefronts of a workgroup that there is LDS for; those of a larger workgroup leave the units to them.
template <int WAVES>
__device__ __forceinline__ void lava_role(par_str d_par_gpu, dim_str d_dim_gpu, const box_str *d_box_gpu,
                                          const FOUR_VECTOR *d_rv_gpu, const float *d_qv_gpu, FOUR_VECTOR *d_fv_gpu,
                                          int grid_dimension_x, int role_block, int role_blocks, int start, int end,
                                          int tid, int role_threads)
{
    const int waves = min(role_threads / TK_WAVE_SIZE, WAVES);
    const int wave = __builtin_amdgcn_readfirstlane(tid / TK_WAVE_SIZE);
    if (wave >= waves || start >= end) return;
    lava_lds_float4 *stage = lava_stage_of_wave<WAVES>(wave);
    const int lane = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    // boxes past number_boxes do nothing in the reference (src/ori_kernel/lava_kernel.cu:21)
    const int gx = (long)grid_dimension_x < d_dim_gpu.number_boxes ? grid_dimension_x : (int)d_dim_gpu.number_boxes;
    if (gx <= 0 || grid_dimension_x <= 0) return;
    const float a2 = 2.0 * d_par_gpu.alpha * d_par_gpu.alpha;
    const float scale = lava_scalar(-a2 * 1.44269504088896340736f);
    const int cols = grid_dimension_x;   // positions per row, including boxes past number_boxes
    const int stride = role_blocks * waves;
    const LavaUnits units(gx, stride, d_dim_gpu.number_boxes >= LAVA_TILES_FROM);
    // Many units: those of a workgroup follow each other, so that the fine ones of the last round start last; fewer: as first_piece says.  (By the
    // units of the range instead of the domain's, which spreads short ranges over more workgroups, they are slower: 64 and 512 boxes of 11^3 6.9 and
    // 9.5 us, so 7.9 and 10.5.)
    const int first_owned = units.first_of(gx) >= LAVA_WAVES_PER_SIMD * 4 * TK_CU_NUM ? role_block * waves + wave
                                                                                      : first_piece(units.first_of(gx), 4 * TK_CU_NUM, wave, waves, role_block, role_blocks);
    if (first_owned >= units.first_of(gx)) return;   // (most, in a launch of 32 wavefronts a SIMD: 64 and 512 boxes of 11^3 10.1 and 12.7 us, so 6.9 and 9.5)
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
                   lane, stage);
    }
}

}  // namespace tk
