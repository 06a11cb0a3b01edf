// Cutoff Coulomb potential role: the potential of binned point charges on a lattice, every charge
// acting within the cutoff only (src/ori_kernel/cutcp_kernel.cu:19-158,
// src/gptb_kernel/cutcp_kernel.cu:12-183 of the reference).
//
// The reference's block position is a region of 8 x 8 x 8 lattice points, given to a block of
// 128 threads (8, 2, 8): thread (tx, ty, tz) owns the points (tx, ty + 2 e, tz), e = 0 .. 3, and all
// threads walk the same atoms -- the bins the neighbour list names around the region's centre bin,
// staged 32 bins at a time in shared memory between two block barriers.  Here a wavefront serves a piece of
// a region on its own -- 64 of the reference's threads, some or all of their four points each -- so the
// role lives in a fused kernel next to roles that own the workgroup barrier.
//   dx = ax - x; dz = az - z; dy = ay - y; r2 = dx dx + dy dy + dz dz;
//   if (r2 < cutoff2) { s = 1 - r2 * inv_cutoff2; energy += aq * rsqrt(r2) * s * s; }
// with the hardware's reciprocal square root where the reference has CUDA's rsqrtf and fused multiply-adds
// (results agree within rounding, not bit for bit).
//
// What bounds it is VALU issue, so what counts is how many atoms are looked at and what an atom costs.
//  * Atoms.  The neighbour list names every bin that may matter to some region: 335 bins, 1340 atoms at 4 an
//    occupied bin, of which 450 are within 12 Angstroms of a point and 725 of some point of a half region.  A
//    wavefront therefore looks at 64 slots (8 bins) at a time, a lane each: an atom that can reach none of the
//    wavefront's points is dropped -- an exact zero is all it would have added -- and the others are appended, in
//    order, to a list in LDS, of which whole groups of 4 are used; what is left over waits for the next 64 slots.  Looking
//    through 64 slots is 60 instructions, none of them a 32-bit product: the list's entries are walked with a counter.
//  * An atom.  It is read back from that list with one 16-byte broadcast read into vector registers (an
//    instruction with a scalar register among its operands takes 4.2 cycles of a SIMD, one without 2.1), and a
//    point takes 7 such instructions and the reciprocal square root, 8 cycles, which goes first
//    (transcendentals_begin): where inv_cutoff2 is 1 / cutoff2 the cutoff
//    is the clamp of s to [0, 1], a modifier of the instruction that computes it, instead of a comparison and
//    an execution mask.
// The atoms' order, and so every point's sum, is the same in every form of the kernel.
// 208^3 lattice, two layers of regions: 99 to 103 us (123 with the square roots where they fall and a workgroup's pieces far apart); 136 us with every batch filled up to whole groups
// (a twelfth of the atoms) and the place in the list divided anew for each, in 95 instructions with five 32-bit products at a quarter of
// the rate.  Where inv_cutoff2 is not 1 / cutoff2 every point walks the list by itself: 169 us where the clamp took 123 (185 before).
#pragma once
#include <cfloat>

#include "role_common.h"
#include "../header/cutcp_header.h"

// the neighbour list: offsets (i, j, k) of the bins to visit around a region's centre bin
// (cudaMemcpyToSymbol(NbrListLen / NbrList, ...), src/ori_kernel/cutcp_kernel.cu:12-13,241-242)
__constant__ int NbrListLen;
__constant__ int NbrList[NBRLIST_MAXLEN][3];

namespace tk {

typedef __attribute__((address_space(3))) float4_t cutcp_lds_float4;

#define CUTCP_GROUP 4   // atoms read from the list at a time
#define CUTCP_BATCH_BINS (TK_WAVE_SIZE / BIN_DEPTH)   // bins whose slots a wavefront looks at at a time
#define CUTCP_RING (2 * TK_WAVE_SIZE)                 // atoms the list in LDS holds: those left over of less than a group, and 64
static_assert(CUTCP_NBR_CHUNK >= 2 * CUTCP_BATCH_BINS, "a part of several is no shorter than a batch");

// The neighbour list dealt to `parts` parts: part p holds the entries p, p + parts, p + 2 parts, ... (every part a
// sample of the whole neighbourhood, so that parts cost the same wherever the atoms are).  Walked part by part
// it is a sequence; these give the place in it where a part begins, and the entry at a place.
struct CutcpWalk {
    int len, parts, each, more;   // entries per part: each + 1 in the first `more` parts, each in the others
    float inv_each, inv_each1;
    __device__ __forceinline__ CutcpWalk(int len_, int parts_) : len(len_), parts(parts_)
    {
        each = len / parts;
        more = len - each * parts;
        inv_each = 1.0f / (float)max(each, 1);
        inv_each1 = 1.0f / (float)(each + 1);
    }
    __device__ __forceinline__ int begin_of(int part) const { return part * each + min(part, more); }
    // the entry at a place, as part and number within it
    struct Entry {
        int part, within;
    };
    __device__ __forceinline__ Entry entry_at(int place) const
    {
        // divisions of numbers below 2^12 by numbers below 2^11: exact with the half added
        const int split = more * (each + 1);
        const bool first = place < split;
        const int f = first ? place : place - split;
        const int part = (int)(((float)f + 0.5f) * (first ? inv_each1 : inv_each));
        return Entry{part + (first ? 0 : more), f - part * (first ? each + 1 : each)};
    }
    // ... a batch further (past the last one: any entry)
    __device__ __forceinline__ void advance(Entry &e) const
    {
        e.within += CUTCP_BATCH_BINS;
        const int entries = each + (e.part < more ? 1 : 0);
        const bool next = e.within >= entries;
        e.within -= next ? entries : 0;
        e.part += next ? 1 : 0;
    }
    __device__ __forceinline__ int number_of(const Entry &e) const { return min(e.part + __mul24(e.within, parts), len - 1); }
};

// The piece `sub` of half `half` of region (xr, yr, zr): the reference's threads 64 half + lane, points e = PTS sub ..
// PTS sub + PTS - 1 of each, over parts [part_begin, part_end) of the neighbour list.  A range that does not start
// with part 0 goes on from the energies in memory, where the range before it left them (a float stored and reloaded
// is unchanged, so consecutive ranges give the bits of one walk through all parts).  CLAMP: the cutoff is the clamp
// of s.  stage: CUTCP_RING x 16 bytes of LDS, this wavefront's own.
template <int PTS, bool CLAMP>
__device__ __forceinline__ void cutcp_piece(int binDim_x, int binDim_y, const float *binZeroAddr, float h, float cutoff2,
                                            float inv_cutoff2, float *regionZeroAddr, int gdx, int gdy, int xr, int yr,
                                            int zr, int half, int sub, int lane, int part_begin, int part_end,
                                            const CutcpWalk walk, cutcp_lds_float4 *stage)
{
    const int tid = 64 * half + lane;
    const int tx = tid & 7, ty = (tid >> 3) & 1, tz = tid >> 4;
    float *region = regionZeroAddr + (size_t)((zr * gdy + yr) * gdx + xr) * REGION_SIZE;
    const float x = (8 * xr + tx) * h;
    const float z = (8 * zr + tz) * h;
    float y[PTS], energy[PTS];
    float *mine = region + (tid >> 4) * 64 + (tid & 15) + 16 * PTS * sub;
#pragma unroll
    for (int e = 0; e < PTS; ++e) {
        y[e] = (8 * yr + ty + 2 * (PTS * sub + e)) * h;
        energy[e] = part_begin > 0 ? mine[16 * e] : 0.f;
    }
    // bin of the region's centre
    const int bx = (int)floorf((8 * xr + 4) * h * BIN_INVLEN);
    const int by = (int)floorf((8 * yr + 4) * h * BIN_INVLEN);
    const int bz = (int)floorf((8 * zr + 4) * h * BIN_INVLEN);
    // the box around the wavefront's points, and how far from it an atom may lie (rounded outwards)
    const float box_x0 = (8 * xr) * h, box_x1 = (8 * xr + 7) * h;
    const float box_y0 = (8 * yr + 2 * PTS * sub) * h, box_y1 = (8 * yr + 2 * PTS * sub + 2 * PTS - 1) * h;
    const float box_z0 = (8 * zr + 4 * half) * h, box_z1 = (8 * zr + 4 * half + 3) * h;
    const float reach2 = cutoff2 * 1.0001f;
    float inv = inv_cutoff2;
    asm volatile("" : "+v"(inv));   // (in a vector register)
    const int end = walk.begin_of(part_end);
    const int slot = lane & (BIN_DEPTH - 1);
    // this lane's slot of the centre bin, and a bin's distance from it in bins: (k binDim_y + j) binDim_x + i, in factors of 24
    // bits unless the bins' grid is half a million long (a 32-bit product is a quarter of the rate)
    const float4_t *centre = reinterpret_cast<const float4_t *>(binZeroAddr) +
                             ((((long long)bz * binDim_y + by) * binDim_x + bx) * BIN_DEPTH + slot);
    const bool short_sides = binDim_x < (1 << 19) && binDim_y < (1 << 19);
    // The batch that starts at `place`: the list's entry of this lane's bin, then the slot this lane looks at.  A place
    // past the end is not used.  Entries are fetched two batches ahead, slots one.
    struct Offset {
        int i, j, k;
    };
    CutcpWalk::Entry upcoming;   // of the next fetch from the list
    const auto entry = [&]() -> Offset {
        const unsigned at = (unsigned)__mul24(walk.number_of(upcoming), (int)sizeof(NbrList[0]));
        const int *n = reinterpret_cast<const int *>(reinterpret_cast<const char *>(&NbrList[0][0]) + at);
        walk.advance(upcoming);
        return Offset{n[0], n[1], n[2]};
    };
    const auto fetch = [&](const Offset &n) -> float4_t {
        long long bin;
        if (short_sides) bin = __mul24(__mul24(n.k, binDim_y) + n.j, binDim_x) + n.i;   // uniform
        else bin = ((long long)n.k * binDim_y + n.j) * binDim_x + n.i;
        return centre[bin * BIN_DEPTH];
    };
    // the lanes whose slot is an atom that a bin holds: its atoms end with the first charge of zero
    const auto held = [&](const float4_t &a, int place) -> unsigned long long {
        const unsigned long long zeros = __ballot(a.w == 0.f);
        const unsigned before = (unsigned)(zeros >> (lane & ~(BIN_DEPTH - 1))) & (2u * (1u << slot) - 1u);
        return __ballot(before == 0u) & __ballot(place + (lane >> 3) < end);
    };
    // ... and those whose charge is a finite number
    const auto finite = [](const float4_t &a) -> unsigned long long { return __ballot(__builtin_fabsf(a.w) <= FLT_MAX); };
    const int begin = walk.begin_of(part_begin);
    unsigned long long all = ~0ull;   // the lanes that have met finite charges only
    float4_t next = {0.f, 0.f, 0.f, 0.f};
    Offset ahead = {0, 0, 0};
    const auto start = [&]() {   // at the first batch
        upcoming = walk.entry_at(min(begin + (lane >> 3), end - 1));
        next = fetch(entry());
        ahead = entry();
    };
    if (begin < end) start();
    int first = 0, behind = 0;   // the list: atoms first .. behind - 1, atom n at n modulo its size; first is a multiple of a group
    const auto fence = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    const auto use_groups = [&]() {   // the whole groups there are
        float4_t ga[CUTCP_GROUP], gb[CUTCP_GROUP];
        const auto read = [&](float4_t (&g)[CUTCP_GROUP], int at) {
#pragma unroll
            for (int u = 0; u < CUTCP_GROUP; ++u) g[u] = stage[(at & (CUTCP_RING - 1)) + u];
            __builtin_amdgcn_sched_barrier(0);   // on its way while the group before it is used
        };
        const auto use = [&](const float4_t (&g)[CUTCP_GROUP]) {
            float r2[CUTCP_GROUP][PTS], inverse[CUTCP_GROUP][PTS];
#pragma unroll
            for (int u = 0; u < CUTCP_GROUP; ++u) {
                const float dx = g[u].x - x;
                const float dz = g[u].z - z;
                const float dxdz2 = __builtin_fmaf(dx, dx, dz * dz);
#pragma unroll
                for (int e = 0; e < PTS; ++e) {
                    const float dy = g[u].y - y[e];
                    r2[u][e] = __builtin_fmaf(dy, dy, dxdz2);
                }
            }
            // (Where a wavefront has its SIMD to itself they might as well not go first: in an instance of its own for up to 4 * TK_CU_NUM pieces, 48 points
            // 23.8 us for 24.0, but 72 to 104 points 2 to 3 % more, with more code around theirs.)
            transcendentals_begin();
#pragma unroll
            for (int u = 0; u < CUTCP_GROUP; ++u)
#pragma unroll
                for (int e = 0; e < PTS; ++e) inverse[u][e] = __builtin_amdgcn_rsqf(r2[u][e]);
            transcendentals_end();
#pragma unroll
            for (int u = 0; u < CUTCP_GROUP; ++u)
#pragma unroll
                for (int e = 0; e < PTS; ++e) {
                    float s = __builtin_fmaf(-r2[u][e], inv, 1.f);
                    if (CLAMP) s = __builtin_amdgcn_fmed3f(s, 0.f, 1.f);
                    const float add = __builtin_fmaf(g[u].w * inverse[u][e], s * s, energy[e]);
                    energy[e] = CLAMP || r2[u][e] < cutoff2 ? add : energy[e];
                }
            __builtin_amdgcn_sched_barrier(0);
        };
        if (first + CUTCP_GROUP <= behind) read(ga, first);
        while (first + CUTCP_GROUP <= behind) {   // uniform
            read(gb, first + CUTCP_GROUP);
            use(ga);
            first += CUTCP_GROUP;
            if (first + CUTCP_GROUP > behind) break;
            read(ga, first + CUTCP_GROUP);
            use(gb);
            first += CUTCP_GROUP;
        }
    };
    for (int place = begin; place < end; place += CUTCP_BATCH_BINS) {
        const float4_t a = next;
        next = fetch(ahead);
        ahead = entry();
        // how far the atom is from the box (no number, and so out of reach, where a coordinate is none)
        const float ex = a.x - __builtin_amdgcn_fmed3f(a.x, box_x0, box_x1);
        const float ey = a.y - __builtin_amdgcn_fmed3f(a.y, box_y0, box_y1);
        const float ez = a.z - __builtin_amdgcn_fmed3f(a.z, box_z0, box_z1);
        const float e2 = ex * ex + ey * ey + ez * ez;
        // beyond a point's cutoff the clamp makes s zero, and the term with it unless the charge is infinite or no number
        // (whole masks, so that no branch and no mask made into numbers and back comes of it)
        const unsigned long long usable = CLAMP ? finite(a) : ~0ull;
        all &= usable;
        const unsigned long long kept = held(a, place) & __ballot(e2 < reach2) & usable;
        const bool keep = __builtin_amdgcn_inverse_ballot_w64(kept);
        const int at = (int)__builtin_amdgcn_mbcnt_hi((unsigned)(kept >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)kept, (unsigned)behind));
        // the wavefront's reads of the list before are behind it: LDS serves a wavefront in order
        if (keep) stage[at & (CUTCP_RING - 1)] = a;
        behind += __popcll(kept);
        if (place + CUTCP_BATCH_BINS >= end) {   // uniform: the last ones, up to a whole group with charges of zero out of everybody's reach
            const int pad = (first - behind) & (CUTCP_GROUP - 1);
            if (lane < pad) stage[(behind + lane) & (CUTCP_RING - 1)] = float4_t{1e18f, 1e18f, 1e18f, 0.f};
            behind += pad;
        }
        fence();
        use_groups();
        fence();
    }
    // The atoms left out are compared with the cutoff, on a walk of their own: a sum they are part of is infinite or no
    // number whenever they are added.  (As a second form of the loop above, chosen for every 64 slots, this cost 1.5 us of
    // 26 at 36 regions and 2.3 of 45 at 361.)
    if (CLAMP && all != ~0ull) {   // uniform
        start();
        for (int place = begin; place < end; place += CUTCP_BATCH_BINS) {
            const float4_t a = next;
            next = fetch(ahead);
            ahead = entry();
            unsigned long long those = held(a, place) & ~finite(a);
            while (those != 0) {
                const int from = __builtin_ctzll(those);
                those &= those - 1;
                float c[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) c[i] = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(a[i]), from));
                const float dx = c[0] - x, dz = c[2] - z;
                const float dxdz2 = __builtin_fmaf(dx, dx, dz * dz);
#pragma unroll
                for (int e = 0; e < PTS; ++e) {
                    const float dy = c[1] - y[e];
                    const float r2 = __builtin_fmaf(dy, dy, dxdz2);
                    const float s = __builtin_fmaf(-r2, inv, 1.f);
                    const float add = __builtin_fmaf(c[3] * __builtin_amdgcn_rsqf(r2), s * s, energy[e]);
                    energy[e] = r2 < cutoff2 ? add : energy[e];
                }
            }
        }
    }
#pragma unroll
    for (int e = 0; e < PTS; ++e) mine[16 * e] = energy[e];
}

// How the regions are cut into units of a wavefront each: half regions with all four points a thread, or pieces of
// a quarter or a half of those.  A smaller piece is more wavefronts -- one that has its SIMD to itself issues at
// half the rate of two -- and evener shares, and has fewer atoms in reach (725 of a half region, 620 of a quarter of
// it); against it stand what a wavefront spends on looking for them, about 60 instructions for every 64 slots, and
// the four instructions and the read an atom costs before its points.  Measured with 1 and 2 points, us: 361 regions
// 39.5 / 45.5, 400 42.5 / 45.7, 450 49.4 / 51.3, 484 44.7 / 46.9, 576 53.9 / 48.1, 722 73.1 / 63.6; with 2 and 4, before the square roots went first, 4056
// 321 / 326, 5408 456 / 444, 17576 1352 / 1337.
struct CutcpPieces {
    int pts, subs;
    __device__ __forceinline__ CutcpPieces(int regions, int waves)
    {
        pts = regions * 8 <= min(waves, 16 * TK_CU_NUM) ? 1 : (regions <= 16 * TK_CU_NUM ? 2 : 4);
        subs = 4 / pts;
    }
    __device__ __forceinline__ int first_of(int region) const { return region * 2 * subs; }
};

// One phase of a launch: regions [region_lo, region_hi) (in position order) each walk parts
// [part_begin, part_end) of the neighbour list.  A wavefront serves the units it owns: first_owned,
// first_owned + stride, ...
__device__ __forceinline__ void cutcp_phase(const CutcpPieces pieces, int region_lo, int region_hi, int part_begin, int part_end,
                                            const CutcpWalk walk, int binDim_x, int binDim_y, const float *binZeroAddr,
                                            float h, float cutoff2, float inv_cutoff2, float *regionZeroAddr, int gdx,
                                            int gdy, int gdz, int first_owned, int stride, int lane,
                                            cutcp_lds_float4 *stage)
{
    // (1e-4: a shell where the two disagree has s below 1e-4 and adds less than 1e-8 of a term)
    const bool clamp = fabsf(cutoff2 * inv_cutoff2 - 1.f) <= 1e-4f;
    const int lo = pieces.first_of(region_lo), hi = pieces.first_of(region_hi);
    int c = first_owned;
    if (c < lo) c += (lo - c + stride - 1) / stride * stride;
    for (; c < hi; c += stride) {
        const int unit = __builtin_amdgcn_readfirstlane(c);
        const int sub = unit % pieces.subs, half = (unit / pieces.subs) & 1;
        const int r = unit / (2 * pieces.subs);
        // region r of the reference's GPTB order, x slowest (src/gptb_kernel/cutcp_kernel.cu:61-63)
#define CUTCP_PIECE(PTS_, CLAMP_, sub_)                                                                                 \
    cutcp_piece<PTS_, CLAMP_>(binDim_x, binDim_y, binZeroAddr, h, cutoff2, inv_cutoff2, regionZeroAddr, gdx, gdy,       \
                              r / (gdy * gdz), (r / gdz) % gdy, r % gdz, half, sub_, lane, part_begin, part_end, walk, stage)
        if (clamp && pieces.pts == 4) CUTCP_PIECE(4, true, sub);
        else if (clamp && pieces.pts == 2) CUTCP_PIECE(2, true, sub);
        else if (clamp) CUTCP_PIECE(1, true, sub);
        else CUTCP_PIECE(1, false, sub * pieces.pts);
        if (!clamp)
            for (int e = 1; e < pieces.pts; ++e) CUTCP_PIECE(1, false, sub * pieces.pts + e);
#undef CUTCP_PIECE
    }
}

// the LDS of the role's wavefronts: CUTCP_RING atoms each.  role_wave: the calling wavefront's number within the role
template <int WAVES>
__device__ __forceinline__ cutcp_lds_float4 *cutcp_stage_of_wave(int role_wave)
{
    __shared__ __align__(16) float4_t cutcp_stage[WAVES][CUTCP_RING];
    return (cutcp_lds_float4 *)&cutcp_stage[role_wave][0];
}

// grid_dimension_x, _y: regions along x and y; grid_dimension_z: regions along z times the parts of
// the neighbour list (ceil(NbrListLen / CUTCP_NBR_CHUNK) parts of at most CUTCP_NBR_CHUNK entries, dealt
// round-robin; 1 part when the list is empty).  The position grid has the regions as columns and the
// parts as rows: position p adds part (p / regions) % parts to region p % regions.  Every unit has one owner
// wavefront for the whole launch, which walks the rows in order, so the parts of a region are added in ascending
// order without any synchronisation, whole rows that follow each other are one run through their parts, and
// a range that runs past the grid wraps.
// WAVES: wavefronts of a workgroup that there is LDS for; those of a larger workgroup leave the units to them.
template <int WAVES>
__device__ __forceinline__ void cutcp_role(int binDim_x, int binDim_y, const float *binZeroAddr, float h, float cutoff2,
                                           float inv_cutoff2, float *regionZeroAddr, int grid_dimension_x,
                                           int grid_dimension_y, int grid_dimension_z, int role_block, int role_blocks,
                                           int start, int end, int tid, int role_threads)
{
    const int waves = min(role_threads / TK_WAVE_SIZE, WAVES);
    const int wave = __builtin_amdgcn_readfirstlane(tid / TK_WAVE_SIZE);
    if (wave >= waves || start >= end) return;
    const int lane = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    const int len = NbrListLen;
    const int gy = max(1, (len + CUTCP_NBR_CHUNK - 1) / CUTCP_NBR_CHUNK);   // parts = rows
    const int gdz = grid_dimension_z / gy;                                     // regions along z
    const int gx = grid_dimension_x * grid_dimension_y * gdz;                  // regions = columns
    if (gx <= 0) return;
    const int stride = role_blocks * waves;
    const CutcpPieces pieces(gx, stride);
    const int first_owned = first_piece(pieces.first_of(gx), 8 * TK_CU_NUM, wave, waves, role_block, role_blocks);
    if (first_owned >= pieces.first_of(gx)) return;   // (most, in small lattices: 48 points 24.7 us, so 24.0, 104 points 29.6 and 28.8)
    const CutcpWalk walk(len, gy);
    cutcp_lds_float4 *stage = cutcp_stage_of_wave<WAVES>(wave);
    // the range as phases: a partial row, or whole rows that follow each other up to the last part
    for (int pos = start; pos < end;) {
        const int row = pos / gx;
        const int part = row % gy;
        const int lo = pos - row * gx;
        int rows = 1;
        const int hi = min(gx, lo + (end - pos));
        if (lo == 0 && hi == gx) rows = min((end - pos) / gx, gy - part);
        pos += rows == 1 ? hi - lo : rows * gx;
        cutcp_phase(pieces, lo, hi, part, part + rows, walk, binDim_x, binDim_y, binZeroAddr, h, cutoff2, inv_cutoff2,
                    regionZeroAddr, grid_dimension_x, grid_dimension_y, gdz, first_owned, stride, lane, stage);
    }
}

}  // namespace tk
