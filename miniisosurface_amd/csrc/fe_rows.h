/*
 * fe_rows.h -- Flying Edges passes 2 and 4 with (grid row, mask word) pairs on the lanes.
 *
 * A wavefront covers RPW consecutive grid rows of W mask words each (RPW = 64 / Wp, Wp a power of
 * two >= W, so nx <= 4096 voxels per row); lane (q, w) owns word w of row q. Row
 * totals and offsets are segmented wave reductions and prefix sums over the Wp lanes of a row.
 * Consecutive grid rows own consecutive vertex blocks, so a wavefront's vertices form one
 * contiguous range of the output, and its triangles one contiguous range too.
 *
 *   k_fe_count_rows  pass 1b + 2 (trims, x/y/z cut counts, triangle counts per row)
 *   k_fe_emit_rows   pass 4: vertices (voxels with a cut edge listed in output order in LDS, one per
 *                    lane, its up to three vertices from one set of voxel loads), and triangles
 *                    (active cells listed in output order, one per lane its case and its twelve
 *                    vertex ids into LDS, then one triangle per lane)
 */
#ifndef MINIISO_FE_ROWS_H
#define MINIISO_FE_ROWS_H

#include "fe_kernels.h"

namespace miso {

struct RowLanes {
    int Wp;       // lanes per row (power of two, >= W)
    int rpw;      // rows per wavefront
    int q;        // this lane's row within the wavefront
    int w;        // this lane's word within the row
};

/* lg of the lanes per row: the fewest that hold a row's words (at most 64), and more, so that a wavefront
 * has fewer rows, where `waves` wavefronts of those would be less than kFillWaves. Passes 2 and 4 of a
 * small volume are as long as one wavefront's chain of loads, lists and stores (64^3 with 64 rows per
 * wavefront: 64 wavefronts for 256 CUs). Whole extractions without allocation, with the fewest lanes and at
 * least 1024, 2048, 4096 or 8192 wavefronts: 64^3 gyroid 154, 54, 55, 62, 62 us; 96^3 noise 105, 64, 61, 67, 80;
 * 128^3 gyroid 102, 74, 63, 61, 75; 160^3 noise 82, 82, 72, 77, 92; 200^3 gyroid 92, 92, 92, 98, 97. More
 * wavefronts than that repeat the setup and leave lanes empty. */
constexpr int64_t kFillWaves = 2048;

inline int fewest_lanes(int64_t W)
{
    int lg = 0;
    while (lg < 6 && (int64_t(1) << lg) < W) ++lg;
    return lg;
}

/* lg of how many times the fewest: `lanes` is the rows' sum of the fewest */
inline int more_lanes(int64_t lanes)
{
    int more = 0;
    while (more < 6 && (lanes << more) >> 6 < kFillWaves) ++more;
    return more;
}

inline int plan_lanes(int64_t ny, int64_t nz, int64_t W)
{
    const int lg = fewest_lanes(W), most = lg + more_lanes((ny * nz) << lg);
    return most < 6 ? most : 6;
}

/* The same for a batch: one `more` for every job, from all jobs' lanes together. Added up in wavefronts,
 * rounded down per job, jobs of less than a wavefront count as nothing however many there are: 20000 of 7x7x7
 * then got 13 blocks each in the place of one (2521 us against 711). */
struct BatchLanes {
    int64_t lanes = 0;
    void add(int64_t ny, int64_t nz, int64_t W) { lanes += (ny * nz) << fewest_lanes(W); }
    int job(int64_t W) const
    {
        const int lg = fewest_lanes(W) + more_lanes(lanes);
        return lg < 6 ? lg : 6;
    }
};

__device__ __forceinline__ RowLanes row_lanes(const Geom& g)
{
    RowLanes L;
    const int lg = g.lg_wp;
    L.Wp = 1 << lg;
    L.rpw = 64 >> lg;
    const int lane = lane_id();
    L.q = lane >> lg;
    L.w = lane & (L.Wp - 1);
    return L;
}

/* the first row of lane-row block blk */
__device__ __forceinline__ int64_t block_row(const Geom& g, int64_t blk) { return blk * 4 * (64 >> g.lg_wp); }

/* This wavefront's index within its 256-thread block, in a scalar register. */
__device__ __forceinline__ int wave_in_block() { return __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)); }

/* a / b for values that are the same in every lane (scalar code; 32-bit when both fit) */
__host__ __device__ __forceinline__ int64_t uniform_div(int64_t a, int64_t b)
{
    if (((uint64_t)a | (uint64_t)b) >> 32 == 0) return (int64_t)((uint32_t)a / (uint32_t)b);
    return a / b;
}

/* (j, k) of grid row r0 + q, for a wavefront whose first row r0 is the same in every lane and
 * 0 <= q < 64: one division per wavefront, then carries per lane (at most one once ny >= 64). */
struct RowJK {
    int64_t j, k;
};

__host__ __device__ __forceinline__ RowJK split_row(int64_t r0, int q, int64_t ny)
{
    RowJK p;
    p.k = uniform_div(r0, ny);
    p.j = r0 - p.k * ny + q;
    while (p.j >= ny) {
        p.j -= ny;
        ++p.k;
    }
    return p;
}

/* Where a wavefront's rows lie, the same in every lane, so that what a lane works out from it is 32-bit:
 * the wavefront's first row r0 = (j0, k0), how many of its rows are there, and how many planes lie
 * above plane k0 (at most 128; the rows span fewer than 66). */
struct WaveRows {
    int64_t r0, k0;
    int j0, ny, n, above;
};

__device__ __forceinline__ WaveRows wave_rows(const Geom& g, int64_t r0, int rpw)
{
    WaveRows A;
    A.r0 = r0;
    const RowJK first = split_row(r0, 0, g.ny);
    A.k0 = first.k;
    A.j0 = (int)first.j;
    A.ny = (int)g.ny;
    const int64_t left = g.ny * g.nz - r0, up = g.nz - 1 - A.k0;
    A.n = (int)(left < rpw ? left : rpw);
    A.above = (int)(up < 128 ? up : 128);
    return A;
}

/* Row r0 + q: its j, and the planes from k0 on */
struct LaneRow {
    int j, dk;
    bool has_y, has_z;
};

__device__ __forceinline__ LaneRow lane_row(const WaveRows& A, int q)
{
    LaneRow p;
    p.j = A.j0 + q;
    p.dk = 0;
    if (A.ny >= 64) {
        const bool wrap = p.j >= A.ny;
        p.j -= wrap ? A.ny : 0;
        p.dk = wrap ? 1 : 0;
    } else {
        while (p.j >= A.ny) {
            p.j -= A.ny;
            ++p.dk;
        }
    }
    p.has_y = p.j < A.ny - 1;
    p.has_z = p.dk < A.above;
    return p;
}

/* A lane's entry of a per-row array: row r0 + q + `ahead`, r0 the same in every lane */
template <typename T>
__device__ __forceinline__ T& row_entry(T* __restrict__ rows, const WaveRows& A, int q, int64_t ahead = 0)
{
    return *reinterpret_cast<T*>(const_cast<char*>(reinterpret_cast<const char*>(rows + (A.r0 + ahead)) +
                                                   (uint32_t)q * (uint32_t)sizeof(T)));
}

/* Bits of a lane's word that are voxels (vb), and x-edges or cells (eb): all but in the row's last word */
struct WordBits {
    uint64_t vb, eb;
};

__device__ __forceinline__ WordBits word_bits(const Geom& g, int w)
{
    const int last = (int)g.W - 1, in_last = (int)(g.nx - 64 * (int64_t)last);   // 1 .. 64 voxels in the last word
    const uint64_t vb = ~0ull >> (64 - in_last);
    return w == last ? WordBits{vb, vb >> 1} : WordBits{~0ull, ~0ull};
}

/* Prefix sums over the lanes of a row: a scan of the whole wavefront (six DPP adds, no lane masks) less
 * what comes before the row's first lane. Two counts may share a value, 16 bits each, as long as the
 * wavefront's totals fit 16 bits (its 4096 voxels have at most 4096 cut edges along an axis and
 * 20480 triangles). */
__device__ __forceinline__ uint32_t seg_before(uint32_t incl, const RowLanes& rl)
{
    const int head = lane_id() - rl.w;
    const uint32_t before = (uint32_t)__shfl((int)incl, (head - 1) & 63);
    return head ? before : 0u;
}

__device__ __forceinline__ uint32_t seg_excl_scan(uint32_t v, const RowLanes& rl)
{
    const uint32_t incl = wave_incl_scan_u32(v);
    return incl - v - seg_before(incl, rl);
}

/* the row's total, in every lane of the row; all: the wavefront's */
__device__ __forceinline__ uint32_t seg_sum(uint32_t v, const RowLanes& rl, uint32_t& all)
{
    const uint32_t incl = wave_incl_scan_u32(v);
    all = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
    return (uint32_t)__shfl((int)incl, lane_id() - rl.w + rl.Wp - 1) - seg_before(incl, rl);
}

/* the larger of each 16-bit half */
__device__ __forceinline__ uint32_t max_halves(uint32_t a, uint32_t b)
{
    typedef unsigned short Pair __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t,
                              __builtin_elementwise_max(__builtin_bit_cast(Pair, a), __builtin_bit_cast(Pair, b)));
}

/* The row's xl and xr of pass 1, in the row's first lane, from the 32-bit halves of the lanes' trim words:
 * a lane's first bit, counted down from 4096, and its last one, a half each, and the maximum of both over
 * the row's lanes, to which a lane's window has grown after log2(Wp) moves. nx and 0 for a row without a
 * bit. */
__device__ __forceinline__ RowTrim seg_trim(uint32_t lo, uint32_t hi, const RowLanes& rl, int64_t nx)
{
    const uint32_t first = lo ? (uint32_t)__builtin_ctz(lo) : 32u + (uint32_t)__builtin_ctz(hi);
    const uint32_t last = hi ? 64u - (uint32_t)__builtin_clz(hi) : 32u - (uint32_t)__builtin_clz(lo);
    uint32_t key = (lo | hi) ? (4096u - 64u * (uint32_t)rl.w - first) << 16 | (64u * (uint32_t)rl.w + last) : 0u;
    if (rl.Wp > 1) key = max_halves(key, dpp_u32<kDppRowShl1>(key));
    if (rl.Wp > 2) key = max_halves(key, dpp_u32<kDppRowShl2>(key));
    if (rl.Wp > 4) key = max_halves(key, dpp_u32<kDppRowShl4>(key));
    if (rl.Wp > 8) key = max_halves(key, dpp_u32<kDppRowShl8>(key));
    if (rl.Wp > 16) key = max_halves(key, (uint32_t)__shfl((int)key, (lane_id() + 16) & 63));
    if (rl.Wp > 32) key = max_halves(key, (uint32_t)__shfl((int)key, (lane_id() + 32) & 63));
    return key ? RowTrim{4096u - (key >> 16), key & 0xFFFFu} : RowTrim{(uint32_t)nx, 0u};
}

/* Sign-mask words around lane (row r, word w): rows (j,k) (j+1,k) (j,k+1) (j+1,k+1). n holds the
 * lowest bit of each row's next word (the +1 neighbour of bit 63), taken from the next lane, which
 * holds that word of the same row, or 0 in the row's last word. Rows outside the grid read as zero. */
struct LaneWords {
    uint64_t m[4];
    uint32_t n[4];
};

__device__ __forceinline__ LaneWords load_lane_words(const uint64_t* __restrict__ mask, const Geom& g,
                                                     const WaveRows& A, const RowLanes& rl, bool ok, bool has_y,
                                                     bool has_z)
{
    LaneWords L;
    // scalar bases for the four rows, one 32-bit offset per lane (below 2^15)
    const uint64_t* __restrict__ base = mask + A.r0 * g.W;
    const uint32_t off = 8u * ((uint32_t)rl.q * (uint32_t)g.W + (uint32_t)rl.w);
    const uint64_t* __restrict__ rows[4] = {base, base + g.W, base + g.ny * g.W, base + (g.ny + 1) * g.W};
    const bool rok[4] = {ok, ok && has_y, ok && has_z, ok && has_y && has_z};
    uint32_t low = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        L.m[q] = 0ull;
        if (rok[q]) __builtin_memcpy(&L.m[q], reinterpret_cast<const char*>(rows[q]) + off, 8);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) low |= ((uint32_t)L.m[q] & 1u) << q;
    const uint32_t of_next = dpp_u32<kDppWaveShl1>(low);   // every lane takes part
    low = rl.w + 1 < (int)g.W ? of_next : 0u;
#pragma unroll
    for (int q = 0; q < 4; ++q) L.n[q] = __builtin_amdgcn_ubfe(low, q, 1);
    return L;
}

/* the word's bits moved down by one, `next` (bit 0) moving in at the top */
__device__ __forceinline__ uint64_t shifted(uint64_t m, uint32_t next)
{
    const uint32_t lo = (uint32_t)m, hi = (uint32_t)(m >> 32);
    return (uint64_t)__builtin_amdgcn_alignbit(next, hi, 1) << 32 | __builtin_amdgcn_alignbit(hi, lo, 1);
}

/* The 8 corner words of a lane: sign bits at i (m) and at i+1 (s) of the 4 rows. */
struct CornerWords {
    uint64_t m[4], s[4];
};

__device__ __forceinline__ CornerWords corner_words(const LaneWords& L)
{
    CornerWords C;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        C.m[q] = L.m[q];
        C.s[q] = shifted(L.m[q], L.n[q]);
    }
    return C;
}

/* A cell's marching-cubes case has corner bit q = v_q, in the reference's order
 * (FlyingEdgesAlgorithm.cpp:138-157): v0..v7 = m0 s0 s1 m1 m2 s2 s3 m3 of CornerWords, i.e. rows
 * (j,k), (j+1,k), (j,k+1), (j+1,k+1) at x = i (m) and i + 1 (s), taken (i,j) (i+1,j) (i+1,j+1)
 * (i,j+1) in plane k, then the same in plane k + 1. */

__device__ __forceinline__ uint64_t active_cells(const CornerWords& C, uint64_t eb)
{
    const uint64_t all = C.m[0] & C.m[1] & C.m[2] & C.m[3] & C.s[0] & C.s[1] & C.s[2] & C.s[3];
    const uint64_t any = C.m[0] | C.m[1] | C.m[2] | C.m[3] | C.s[0] | C.s[1] | C.s[2] | C.s[3];
    return any & ~all & eb;
}

__device__ __forceinline__ uint64_t active_cells(const LaneWords& L, uint64_t eb)
{
    return active_cells(corner_words(L), eb);
}

/* Triangles of the marching-cubes cases of a cell row, bit-sliced over the 64 cells of a lane's word: the
 * lane's share, modulo 2^32, of a count that only the row's sum makes. For a cell with corners on both
 * sides of the isovalue, the case table's triangle count (numTris,
 * flyingEdges/util/MarchingCubesTables.h:23-41) equals V - 2F - 4S: V the corners >= iso, F the faces
 * whose four corners are >= iso, S = 1 for the six-corner rings (both ends of a body diagonal below
 * iso, the other six corners >= iso); a cell with all corners >= iso has 8 - 12, so each adds 4 back.
 * Corners and x-faces at x = i + 1 are those at x = i of the next cell, so that over the row they count
 * twice but at its two ends: V = sum over the four rows of 2 P - (first voxel) - (last voxel), and the
 * x-faces likewise, which takes one popcount for two. Bits past the row are 0, and no x-pair, ring or
 * inner face has one there. Word halves, so that three-operand logic takes one instruction: pass 2 at
 * 1024^3, bound by its vector instructions, 160 -> 142 us with 342 -> 290 of them per wavefront (before the
 * row sums 176 us, with every corner and face masked and counted). */
__device__ __forceinline__ uint32_t word_tri_count(const LaneWords& L, const Geom& g, int w)
{
    uint32_t P = 0, F = 0, A = 0, Q = 0;       // corners, faces, x-faces and rings, full cells
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        uint32_t m[4], s[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint32_t lo = (uint32_t)L.m[q], hi = (uint32_t)(L.m[q] >> 32);
            m[q] = h ? hi : lo;
            s[q] = h ? __builtin_amdgcn_alignbit(L.n[q], hi, 1) : __builtin_amdgcn_alignbit(hi, lo, 1);
            P += (uint32_t)__popc(m[q]);
        }
        const uint32_t p0 = m[0] & s[0], p1 = m[1] & s[1], p2 = m[2] & s[2], p3 = m[3] & s[3];
        const uint32_t f01 = p0 & p1, f23 = p2 & p3;
        F += (uint32_t)__popc(f01);
        F += (uint32_t)__popc(f23);
        F += (uint32_t)__popc(p0 & p2);
        F += (uint32_t)__popc(p1 & p3);
        A += (uint32_t)__popc(m[0] & m[1] & m[2] & m[3]);
        Q += (uint32_t)__popc(f01 & f23);
        // rings about v0-v6 or v1-v7 (rows 0 and 3), about v2-v4 or v3-v5 (rows 1 and 2): the rows' two diagonals
        // have equal ends each and differ, the other two rows' four corners are set
        const uint32_t u = ~(m[0] ^ s[3]) & ~(s[0] ^ m[3]) & (m[0] ^ s[0]);
        const uint32_t v = ~(m[1] ^ s[2]) & ~(s[1] ^ m[2]) & (m[1] ^ s[1]);
        A += (uint32_t)__popc(p1 & p2 & u);
        A += (uint32_t)__popc(p0 & p3 & v);
    }
    // the row's first voxels (bits 0 .. 3) and last ones (4 .. 7), a bit per row
    const int last = (int)g.W - 1, top = (int)(g.nx - 64 * (int64_t)last) - 1;
    uint32_t lo = 0, hi = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        lo |= ((uint32_t)L.m[q] & 1u) << q;
        hi |= ((top & 32 ? (uint32_t)(L.m[q] >> 32) : (uint32_t)L.m[q]) >> (top & 31)) << (4 + q);
    }
    const uint32_t e = (w == 0 ? lo : 0u) | (w == last ? hi : 0u);
    const uint32_t xends = (uint32_t)((e & 15u) == 15u) + (uint32_t)(e >= 0xF0u);
    return 2 * (P - F + xends) - (uint32_t)__popc(e) - 4 * (A - Q);
}

/* ------------------------------------------------------------------ pass 1b + 2 */
/* per-row count beside these (none here; first-visit Marching Cubes adds its owned-edge counts,
 * k_fe_mc_count_rows): called by every lane with its words and row, and `empty` when every word the wavefront loaded is zero; the row's count, in every lane of the row */
struct NoRowExtra {
    static constexpr bool kCounts = false;
    __device__ uint32_t operator()(const LaneWords&, const RowLanes&, const WaveRows&, bool, const LaneRow&, bool) const
    {
        return 0u;
    }
};

/* The 4 wavefronts of lane-row block blk (rows 4 rpw blk ..); the wavefront's sums for pass 3. In a slab,
 * rows below emit_lo belong to the slab before it (counts 0, so that the slab's offsets start at 0),
 * and cells from row emit_hi on to the next (triangle counts 0); the vertices of those rows keep their
 * counts, the slab's last cell row names them. xy, zt: the row's counts, packed, in the row's first
 * lane (0 in the others). */
template <class Extra>
__device__ __forceinline__ WaveSums fe_count_rows_block(const uint64_t* __restrict__ mask, const Geom& g,
                                                        RowCounts* __restrict__ counts, RowTrim* __restrict__ trims,
                                                        int64_t blk, Extra extra, uint32_t& xy, uint32_t& zt)
{
    WaveSums sums{0u, 0u, 0u};
    xy = zt = 0u;
    const RowLanes rl = row_lanes(g);
    const int64_t r0 = (blk * 4 + wave_in_block()) * rl.rpw;
    if (r0 >= g.ny * g.nz) return sums;
    const WaveRows A = wave_rows(g, r0, rl.rpw);
    const bool there = rl.q < A.n, ok = there && rl.w < (int)g.W, head = there && rl.w == 0;
    const LaneRow at = lane_row(A, rl.q);
    const bool has_y = at.has_y, has_z = at.has_z;
    const LaneWords L = load_lane_words(mask, g, A, rl, ok, has_y, has_z);
    uint32_t lo[4], hi[4], any = L.n[0] | L.n[1] | L.n[2] | L.n[3];   // bit 0 of the next words: corner i + 1 of bit 63
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        lo[q] = (uint32_t)L.m[q];
        hi[q] = (uint32_t)(L.m[q] >> 32);
        any |= lo[q] | hi[q];
    }
    if (__ballot(any != 0u) == 0ull) {
        // every voxel the wavefront's rows see is below the isovalue (most wavefronts at a
        // sparse, high isovalue): no cut edge, no triangle, an empty trim
        if (head) {
            row_entry(counts, A, rl.q) = RowCounts{0u, 0u, 0u, 0u};
            row_entry(trims, A, rl.q) = RowTrim{(uint32_t)g.nx, 0u};
        }
        extra(L, rl, A, ok, at, true);
        return sums;
    }
    const uint64_t eb = word_bits(g, rl.w).eb;
    const uint32_t e[2] = {(uint32_t)eb, (uint32_t)(eb >> 32)};
    const uint32_t ym = has_y ? ~0u : 0u, zm = has_z ? ~0u : 0u;
    const uint32_t next[2] = {__builtin_amdgcn_alignbit(hi[0], lo[0], 1), __builtin_amdgcn_alignbit(L.n[0], hi[0], 1)};
    uint32_t nx = 0, ny = 0, nz = 0, trim[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const uint32_t* m = h ? hi : lo;
        const uint32_t x = (m[0] ^ next[h]) & e[h], y = (m[0] ^ m[1]) & ym, z = (m[0] ^ m[2]) & zm;
        nx += (uint32_t)__popc(x);
        ny += (uint32_t)__popc(y);
        nz += (uint32_t)__popc(z);
        trim[h] = x | ((y | z) & e[h]);
    }
    const uint32_t tc = word_tri_count(L, g, rl.w) & ym & zm;
    uint32_t all_xy, all_zt;
    xy = seg_sum(nx | ny << 16, rl, all_xy);
    zt = seg_sum(nz | tc << 16, rl, all_zt);
    const bool whole = r0 >= g.emit_lo && r0 + rl.rpw <= g.emit_hi;   // no row of another slab
    if (!whole) {
        if (r0 + rl.q < g.emit_lo) xy = zt = 0u;
        if (r0 + rl.q >= g.emit_hi) zt &= 0xFFFFu;
    }
    const RowTrim tr = seg_trim(trim[0], trim[1], rl, g.nx);
    if (head) {
        row_entry(counts, A, rl.q) = RowCounts{xy & 0xFFFFu, xy >> 16, zt & 0xFFFFu, zt >> 16};
        row_entry(trims, A, rl.q) = tr;
    }
    const uint32_t own = extra(L, rl, A, ok, at, false);
    if (!head) xy = zt = 0u;
    sums.xy = whole ? all_xy : wave_sum_u32(xy);
    sums.zt = whole ? all_zt : wave_sum_u32(zt);
    if (Extra::kCounts) sums.own = wave_sum_u32(head ? own : 0u);
    return sums;
}

/* The sums of a block's four wavefronts into those of the block's tile (2^shift rows hold whole
 * blocks). One atomic per block and kind: with one per wavefront, pass 2 took 215 us at 1024^3 and
 * 34 us at 512^3 against 162 and 25 without (atomics on one tile's line follow one another). */
__device__ __forceinline__ void add_block_sums(const WaveSums& w, uint64_t* __restrict__ tile_sums)
{
    __shared__ WaveSums s_sums[4];
    if (lane_id() == 0) s_sums[threadIdx.x >> 6] = w;
    __syncthreads();
    const int a = (int)threadIdx.x;
    if (a >= kTileSums) return;
    uint32_t v = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) v += sum_of_kind(s_sums[q], a);
    if (v) add_sum(&tile_sums[a], v);
}

__global__ __launch_bounds__(256) void k_fe_count_rows(const uint64_t* __restrict__ mask, Geom g,
                                                       RowCounts* __restrict__ counts,
                                                       RowTrim* __restrict__ trims,
                                                       uint64_t* __restrict__ sums, int shift)
{
    uint32_t xy, zt;
    const WaveSums w = fe_count_rows_block(mask, g, counts, trims, blockIdx.x, NoRowExtra(), xy, zt);
    add_block_sums(w, sums + (block_row(g, blockIdx.x) >> shift) * kTileSums);
}

/* ------------------------------------------------------------------ pass 4: edge points */

/* One gradient component at the grid vertex *v, the reference's formula ((lower - upper) / run,
 * one-sided at the faces; flyingEdges/util/Image3D.cpp:116-188). With unit spacing the divisions
 * by 1 and 2 are exact and written as such. */
template <bool Unit>
__device__ __forceinline__ float grad_at(const float* __restrict__ v, int pos, int n, int stride, float s)
{
    const bool first = pos == 0, last = pos == n - 1;
    const float hi = v[last ? 0 : stride];
    const float lo = v[first ? 0 : -stride];
    const bool one_sided = first || last;
    if (Unit) return one_sided ? (lo - hi) : (lo - hi) * 0.5f;
    return (lo - hi) / (one_sided ? s : 2.0f * s);
}

template <bool Unit>
__device__ __forceinline__ float grad_interior(const float* __restrict__ v, int stride, float s)
{
    const float hi = v[stride], lo = v[-stride];
    if (Unit) return (lo - hi) * 0.5f;
    return (lo - hi) / (2.0f * s);
}

/* Point and normal of the crossing on the edge from grid vertex (i,j,k) along `axis`, with the
 * Flying Edges corner coordinates (fe_edge_corners). `v` points at the voxel of (i,j,k); strides
 * are 32-bit (the launch checks nx * ny < 2^31). Edges whose both ends are interior take a
 * branch without the face tests; it computes the same formulas. */
template <bool Unit>
__device__ __forceinline__ void fe_edge_point(const float* __restrict__ v, const Geom& g, float iso, int axis, int i,
                                              int j, int k, float p[3], float nrm[3])
{
    const int nx = (int)g.nx, ny = (int)g.ny, nz = (int)g.nz;
    const int sy = nx, sz = nx * ny;
    const int step = axis == 0 ? 1 : (axis == 1 ? sy : sz);
    const float* __restrict__ vb = v + step;
    const float v0 = v[0], v1 = vb[0];
    const float w = (iso - v0) / (v1 - v0);
    float A[3], B[3];
    if (Unit) {
        A[0] = (float)i; A[1] = (float)j; A[2] = (float)(k + (int)g.kofs);
        B[0] = A[0]; B[1] = A[1]; B[2] = A[2];
        B[axis] = A[axis] + 1.0f;
    } else {
        fe_edge_corners(g, axis, i, j, k, A, B);
    }
    const int ib = i + (axis == 0), jb = j + (axis == 1), kb = k + (axis == 2);
    float ga0, ga1, ga2, gb0, gb1, gb2;
    if (i >= 1 && j >= 1 && k >= 1 && ib <= nx - 2 && jb <= ny - 2 && kb <= nz - 2) {
        ga0 = grad_interior<Unit>(v, 1, g.sp[0]);
        ga1 = grad_interior<Unit>(v, sy, g.sp[1]);
        ga2 = grad_interior<Unit>(v, sz, g.sp[2]);
        gb0 = grad_interior<Unit>(vb, 1, g.sp[0]);
        gb1 = grad_interior<Unit>(vb, sy, g.sp[1]);
        gb2 = grad_interior<Unit>(vb, sz, g.sp[2]);
    } else {
        ga0 = grad_at<Unit>(v, i, nx, 1, g.sp[0]);
        ga1 = grad_at<Unit>(v, j, ny, sy, g.sp[1]);
        ga2 = grad_at<Unit>(v, k, nz, sz, g.sp[2]);
        gb0 = grad_at<Unit>(vb, ib, nx, 1, g.sp[0]);
        gb1 = grad_at<Unit>(vb, jb, ny, sy, g.sp[1]);
        gb2 = grad_at<Unit>(vb, kb, nz, sz, g.sp[2]);
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) p[c] = A[c] + w * (B[c] - A[c]);
    nrm[0] = ga0 + w * (gb0 - ga0);
    nrm[1] = ga1 + w * (gb1 - ga1);
    nrm[2] = ga2 + w * (gb2 - ga2);
}

/* interior central difference (lower - upper) / (2 h), exact as * 0.5 for unit spacing */
template <bool Unit>
__device__ __forceinline__ float central(float lo, float hi, float s)
{
    if (Unit) return (lo - hi) * 0.5f;
    return (lo - hi) / (2.0f * s);
}

/* Corner coordinates of the edges from an origin (i,j,k) below the last index of each axis, and the end
 * of edge_point with them: p = a + w (b - a), where b - a is 1 or spacing along the edge and a - a (0, or
 * NaN) across it. Flying Edges' are fe_edge_corners; Marching Cubes' (Mc) those of the cell that first
 * visits the edge, one back across it where there is one: that cell's corner plus one spacing
 * (marchingCubes/util/Image3D.cpp:22-65). With unit spacing and zero origin both are the indices. */
template <bool Unit, bool Mc = false>
struct CornerCoords {
    float A[3], P[3];   // along the edge, and (Mc) across it
    __device__ __forceinline__ CornerCoords(const Geom& g, int i, int j, int k)
    {
        if (Unit) {
            A[0] = (float)i; A[1] = (float)j; A[2] = (float)(k + (int)g.kofs);
        } else {
            A[0] = g.org[0] + (float)i * g.sp[0];
            A[1] = g.org[1] + (float)j * g.sp[1];
            A[2] = g.org[2] + (float)(k + (int)g.kofs) * g.sp[2];
            if (Mc) {
                P[0] = i > 0 ? g.org[0] + (float)(i - 1) * g.sp[0] + g.sp[0] : A[0];
                P[1] = j > 0 ? g.org[1] + (float)(j - 1) * g.sp[1] + g.sp[1] : A[1];
                P[2] = k > 0 ? g.org[2] + (float)(k - 1) * g.sp[2] + g.sp[2] : A[2];
            }
        }
    }
    __device__ __forceinline__ float across(int c) const { return Mc && !Unit ? P[c] : A[c]; }
    __device__ __forceinline__ void finish(const Geom& g, int axis, float w, const float ga[3], const float gb[3],
                                           float p[3], float nrm[3]) const
    {
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            if (Unit)
                p[c] = A[c] + (c == axis ? w : w * 0.0f);
            else if (c == axis)
                p[c] = A[c] + w * (A[c] + g.sp[c] - A[c]);
            else
                p[c] = across(c) + w * (across(c) - across(c));
            nrm[c] = ga[c] + w * (gb[c] - ga[c]);
        }
    }
};

/* ------------------------------------------------------------------ pass 4: fused emit */
constexpr int kEmitCellCap = 576;   // active-cell entries per wavefront and round
constexpr int kEmitTriCap = 64 * 5; // triangles of one group of 64 cells (at most 5 each)
constexpr int kIdStride = 7;        // dwords per cell of ids: odd, so that cells spread over the banks
constexpr int kOriginCap = 640;     // origin entries per wavefront and round

/* LDS of one wavefront. words: the mask bits of a lane's four rows by 32-voxel halves (half h of lane
 * l at 2 l + h, followed by the next half's for the corner i + 1; a row that is not there repeats
 * row 0, so that it shows no cut). rank: per half, the id ranks of the eight edge combinations before
 * it, 16 bits each, (0,1) (2,3) (4,5) (6,7). origins: the vertices' list. t: the triangles' cell list
 * and, for the current 64 cells, their ids and the map of their triangles. The cell list takes what LDS four
 * blocks leave: listing is done again for every round (of 240 cells instead of 576: 333x257x190 spaced 123
 * us against 117, a 256^3 gyroid at 16 isovalues 1061 against 1043, 512^3 466.5 against 463, 1024^3 2.238
 * ms against 2.228). Four blocks share a CU; a
 * fifth (the list in t's bytes, made again after the triangles) measured 1.48 against 1.445 ms at
 * 1024^3, three 1.73. */
struct EmitRowsLds {
    uint4 rank[128];
    uint32_t words[4][130];
    uint16_t origins[kOriginCap];
    struct {
        uint32_t ids[64 * kIdStride];
        uint32_t map[kEmitTriCap];
        uint16_t cells[kEmitCellCap];
    } t;
};
static_assert(sizeof(EmitRowsLds) * 4 + 256 * 8 <= 40960, "four blocks of pass 4 share a CU's 160 KB");

/* Pass 4 for the (row, word) lane layout in one launch: each wavefront writes the vertices of its
 * rows, then the triangles of its cell rows. */

/* Per-wavefront state of pass 4 in the lane-row layout: rows r0 .. r0 + rpw - 1, lane (q, w)
 * holding word w of row r0 + q. */
struct EmitRows {
    RowLanes rl;
    int lane, wv, wp_log2;
    int64_t r0;
    uint64_t v0, v2, t0;           // first vertex of row r0 and of row r0 + ny, first triangle of row r0
    uint64_t origins, act;         // this lane's voxels with a cut edge that pass 4 writes; its active cells
    int64_t k0;                    // the wavefront's first row is (j0, k0)
    int j0;
};

/* Loads the wavefront's mask words and row state and fills words and rank. False: nothing to write.
 * The row state comes from one lane per row and reaches the others by lane moves: a load that 64
 * lanes make of their row's entry costs the L1 one access per four lanes, 1024^3 about 100 of a
 * wavefront's 1320. */
template <class Lds>
__device__ __forceinline__ bool emit_rows_setup(EmitRows& E, Lds* s_w, const uint64_t* __restrict__ mask,
                                                const Geom& g, const RowCounts* __restrict__ counts,
                                                const uint64_t* __restrict__ voff, const uint64_t* __restrict__ toff,
                                                int64_t blk)
{
    E.lane = lane_id();
    E.wv = wave_in_block();
    E.rl = row_lanes(g);
    const RowLanes& rl = E.rl;
    const int64_t R = g.ny * g.nz;
    E.r0 = (blk * 4 + E.wv) * rl.rpw;
    if (E.r0 >= R) return false;
    // a wavefront whose rows have no vertex and no triangle leaves before anything else (most of
    // them at a sparse isovalue)
    RowCounts c{0u, 0u, 0u, 0u};
    const bool ok = E.r0 + rl.q < R && rl.w < (int)g.W;
    const bool first = ok && rl.w == 0;        // the lane that holds the row's state
    if (first) c = counts[E.r0 + rl.q];
    if (__ballot((c.x | c.y | c.z | c.t) != 0u) == 0ull) return false;
    const WaveRows A = wave_rows(g, E.r0, rl.rpw);
    const LaneRow at = lane_row(A, rl.q);
    const bool has_y = at.has_y, has_z = at.has_z;
    const LaneWords L = load_lane_words(mask, g, A, rl, ok, has_y, has_z);
    E.v0 = voff[E.r0];
    E.t0 = toff[E.r0];
    E.k0 = A.k0;
    E.j0 = A.j0;
    // the row's vertex offset and, in the plane above, that row's, from v0 and v2: below 2^16, since the wavefront's at
    // most 4096 voxels have 12288 edges, and the row after them puts up to 8192 x- and y-edges before its z-edges,
    // which rank up to 4096 among themselves: 24576
    const int64_t left_above = R - E.r0 - g.ny;             // rows from the one above the wavefront's first
    E.v2 = left_above > 0 ? voff[E.r0 + g.ny] : 0ull;
    uint32_t own = 0, above = 0, above_x = 0;
    if (first) {
        own = (uint32_t)(row_entry(voff, A, rl.q) - E.v0);
        if (rl.q < left_above) {
            above = (uint32_t)(row_entry(voff, A, rl.q, g.ny) - E.v2);
            above_x = row_entry(counts, A, rl.q, g.ny).x;
        }
    }
    // first ids of the row's x-edges (a, low), z-edges (a, high), y-edges (b); x- and y-edges above (c)
    uint32_t a = own | (own + c.x + c.y) << 16, b = own + c.x, cc = above | (above + above_x) << 16;
    const int head = rl.q << (6 - __builtin_ctz((unsigned)rl.rpw)), next = head + rl.Wp;
    uint32_t a1 = (uint32_t)__shfl((int)a, next & 63), c1 = (uint32_t)__shfl((int)cc, next & 63);
    if (next >= 64) {
        // the row after the wavefront's last one
        const int64_t rn = E.r0 + rl.rpw;
        a1 = c1 = 0;
        if (rn < R) {
            const uint32_t o = (uint32_t)(voff[rn] - E.v0);
            const RowCounts cn = counts[rn];
            a1 = o | (o + cn.x + cn.y) << 16;
        }
        if (rn + g.ny < R) c1 = (uint32_t)(voff[rn + g.ny] - E.v2);
    }
    a = (uint32_t)__shfl((int)a, head);
    b = (uint32_t)__shfl((int)b, head);
    cc = (uint32_t)__shfl((int)cc, head);
    E.wp_log2 = 6 - __builtin_ctz((unsigned)rl.rpw);

    const auto [vb, eb] = word_bits(g, rl.w);
    const uint64_t cw[8] = {(L.m[0] ^ shifted(L.m[0], L.n[0])) & eb, (L.m[1] ^ shifted(L.m[1], L.n[1])) & eb,
                            (L.m[2] ^ shifted(L.m[2], L.n[2])) & eb, (L.m[3] ^ shifted(L.m[3], L.n[3])) & eb,
                            (L.m[0] ^ L.m[1]) & vb, (L.m[2] ^ L.m[3]) & vb,
                            (L.m[0] ^ L.m[2]) & vb, (L.m[1] ^ L.m[3]) & vb};
    const uint32_t base[4] = {(a & 0xFFFFu) | a1 << 16, (cc & 0xFFFFu) | c1 << 16, b | (cc & 0xFFFF0000u),
                              a >> 16 | (a1 & 0xFFFF0000u)};
    uint32_t lo[4], hi[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        // two combinations per segmented scan and per dword
        lo[q] = base[q] + seg_excl_scan((uint32_t)__popcll(cw[2 * q]) | (uint32_t)__popcll(cw[2 * q + 1]) << 16, rl);
        hi[q] = lo[q] + ((uint32_t)__popc((uint32_t)cw[2 * q]) | (uint32_t)__popc((uint32_t)cw[2 * q + 1]) << 16);
    }
    Lds& S = s_w[E.wv];
    S.rank[2 * E.lane] = uint4{lo[0], lo[1], lo[2], lo[3]};
    S.rank[2 * E.lane + 1] = uint4{hi[0], hi[1], hi[2], hi[3]};
    const uint64_t m[4] = {L.m[0], has_y ? L.m[1] : L.m[0], has_z ? L.m[2] : L.m[0], L.m[3]};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        S.words[q][2 * E.lane] = (uint32_t)m[q];
        S.words[q][2 * E.lane + 1] = (uint32_t)(m[q] >> 32);
    }
    const bool emit = ok && E.r0 + rl.q >= g.emit_lo && E.r0 + rl.q < g.emit_hi;
    E.origins = emit ? cw[0] | (m[0] ^ m[1]) | (m[0] ^ m[2]) : 0ull;
    E.act = emit && has_y && has_z ? active_cells(L, eb) : 0ull;
    wave_sync();
    return true;
}

/* bits below position b (0 .. 31) */
__device__ __forceinline__ uint32_t bits_below(uint32_t b) { return __builtin_amdgcn_ubfe(0xFFFFFFFFu, 0, b); }

/* Appends the positions (lane << 6 | bit) of a lane's set bits to list, from entry `first` on as far
 * as they fall in [win, win + Cap); total: those of the wavefront, which a list that holds them all takes
 * without a test per entry. A lane's loop is a chain of branches, and its length the fullest lane's: without
 * the test 333x257x190 spaced 116.9 -> 113.9 us, 1024^3 2.238 -> 2.215 ms, 1000x900x700 at iso 0.8 608 -> 604. In
 * its place every lane writing in every step, both halves' bits in one loop, took 2.264 ms at 1024^3. */
template <int Cap>
__device__ __forceinline__ void list_bits(uint64_t bits, uint32_t first, uint32_t win, uint32_t total, int lane,
                                          uint16_t* list)
{
    if (total <= (uint32_t)Cap) {
        uint16_t* to = list + first;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint32_t ent = (uint32_t)lane << 6 | (uint32_t)h << 5;
            for (uint32_t a = h ? (uint32_t)(bits >> 32) : (uint32_t)bits; a; a &= a - 1)
                *to++ = (uint16_t)(ent | (uint32_t)__builtin_ctz(a));
        }
        return;
    }
    uint32_t p = first - win;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const uint32_t ent = (uint32_t)lane << 6 | (uint32_t)h << 5;
        for (uint32_t a = h ? (uint32_t)(bits >> 32) : (uint32_t)bits; a; a &= a - 1, ++p)
            if (p < (uint32_t)Cap) list[p] = (uint16_t)(ent | (uint32_t)__builtin_ctz(a));
    }
}

/* The voxels around an inner origin (i,j,k): its row from i - 1 to i + 2, the rows j + 1 and k + 1
 * from i - 1 to i + 1, the rows j - 1 and k - 1 from i to i + 1; then, for a y-edge, (j + 2),
 * (j + 1, k - 1), for a z-edge, (k + 2), (j - 1, k + 1), and for either, (j + 1, k + 1), each at i. */
struct Around {
    Vox4 r;
    Vox3 yp, zp;
    Vox2 ym, zm, y2, yz, z2, zy, d;
};

/* The first voxel of a pair, the second one kept as read (the compiler would narrow the load). */
__device__ __forceinline__ float of_pair(const Vox2& v)
{
    asm volatile("" ::"v"(v.y));
    return v.x;
}

/* Vertices: one origin -- a voxel with a cut edge along x, y or z -- per lane; its up to three vertices
 * share the voxels around it. The gathers are bound by the L1, which takes one access per 128-byte
 * line and four lanes (a 4-byte gather mostly one per lane, so single voxels are read in pairs): 3.6
 * accesses per vertex by origin against 6.1 with an edge per lane (value noise at 1024^3, counted
 * from the mask; all of pass 4, from the L1's counter: 5.5 against 8.8). Pass 4 at 1024^3, with the
 * triangles of emit_rows_triangles: 1.59 -> 1.37-1.40 ms (now 1.35-1.37); 512^3 gyroid 0.41 -> 0.34 ms. Vertices are
 * stored from the lanes: put in windows of 192 at their place in LDS and stored in 16-byte pieces
 * they took the same time at 1024^3 and 3% more at 512^3, where a wavefront has several windows. */

/* One step of the vertices: a lane's origin, its cut edges and their ids (from v0), its voxels. */
struct VertexStep {
    uint32_t ent, at[3];
    bool any, inner, cut[3];
    int j, k;
    Around a;
};

/* Where the wavefront's rows lie, and its origins: in output order, so that a step's x-, y- and z-edge
 * vertices leave in runs of neighbouring ids (1024^3: 1.405 ms against 1.445 ms with word w of all rows
 * before word w + 1, whose gathers share more lines). */
struct VertexRows {
    const float* __restrict__ vol;
    const float* __restrict__ row0;   // voxel (0, j0, k0)
    bool rows_inner;                  // every row at least one row from a near face, two from a far one
    uint32_t n, first;                // the wavefront's origins; this lane's first in their order
};

__device__ __forceinline__ VertexRows vertex_rows(const EmitRows& E, const float* __restrict__ vol, const Geom& g)
{
    VertexRows R;
    R.vol = vol;
    R.row0 = vol + E.r0 * g.nx;
    R.rows_inner = E.j0 >= 1 && E.j0 + E.rl.rpw <= (int)g.ny - 2 && E.k0 >= 1 && E.k0 <= (int)g.nz - 3;
    const uint32_t cnt = (uint32_t)__popcll(E.origins);
    const uint32_t incl = wave_incl_scan_u32(cnt);
    R.n = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
    R.first = incl - cnt;
    return R;
}

/* base + off bytes, off per lane and base the same in every lane: a scalar base and a 32-bit offset */
template <typename T>
__device__ __forceinline__ T load_at(const float* __restrict__ base, uint32_t off)
{
    T t;
    __builtin_memcpy(&t, reinterpret_cast<const char*>(base) + off, sizeof(T));
    return t;
}

/* Takes this lane's origin (list entry e, if below n) and requests its voxels. */
__device__ __forceinline__ void vertex_load(VertexStep& V, const EmitRows& E, const EmitRowsLds& S, const VertexRows& R,
                                            const Geom& g, uint32_t e, uint32_t n)
{
    const int nx = (int)g.nx, ny = (int)g.ny, nz = (int)g.nz;
    const int64_t sy = g.nx, sz = g.nx * g.ny;
    V.any = e < n;
    V.ent = V.any ? (uint32_t)S.origins[e] : 0u;
    const uint32_t h2 = V.ent >> 5, b = V.ent & 31;
    const int i = (int)(V.ent & ((64u << E.wp_log2) - 1u)), q = (int)(V.ent >> (6 + E.wp_log2));
    const uint32_t w0 = S.words[0][h2], n0 = S.words[0][h2 + 1];
    const uint32_t x = w0 ^ __builtin_amdgcn_alignbit(n0, w0, 1), y = w0 ^ S.words[1][h2], z = w0 ^ S.words[2][h2];
    const uint4 rk = S.rank[h2];
    const uint32_t below = bits_below(b);
    V.cut[0] = V.any && ((x >> b) & 1u) && i < nx - 1;
    V.cut[1] = V.any && ((y >> b) & 1u);
    V.cut[2] = V.any && ((z >> b) & 1u);
    V.at[0] = (rk.x & 0xFFFFu) + (uint32_t)__popc(x & below);
    V.at[1] = (rk.z & 0xFFFFu) + (uint32_t)__popc(y & below);
    V.at[2] = (rk.w & 0xFFFFu) + (uint32_t)__popc(z & below);
    V.j = E.j0 + q;
    V.k = (int)E.k0;
    V.inner = V.any && (uint32_t)(i - 1) < (nx > 3 ? (uint32_t)(nx - 3) : 0u);
    if (!R.rows_inner) {
        while (V.j >= ny) {
            V.j -= ny;
            ++V.k;
        }
        V.inner = V.inner && V.j >= 1 && V.j <= ny - 3 && V.k >= 1 && V.k <= nz - 3;
    }
    if (V.inner) {
        const float* __restrict__ v = R.row0;
        const uint32_t off = 4 * ((uint32_t)q * (uint32_t)nx + (uint32_t)i);   // below 2^20
        Around& a = V.a;
        a.r = load_at<Vox4>(v - 1, off);
        a.yp = load_at<Vox3>(v + sy - 1, off);
        a.zp = load_at<Vox3>(v + sz - 1, off);
        a.ym = load_at<Vox2>(v - sy, off);
        a.zm = load_at<Vox2>(v - sz, off);
        if (V.cut[1]) {
            a.y2 = load_at<Vox2>(v + 2 * sy, off);
            a.yz = load_at<Vox2>(v + sy - sz, off);
        }
        if (V.cut[2]) {
            a.z2 = load_at<Vox2>(v + 2 * sz, off);
            a.zy = load_at<Vox2>(v + sz - sy, off);
        }
        if (V.cut[1] || V.cut[2]) a.d = load_at<Vox2>(v + sy + sz, off);
    }
}

/* Computes and stores the step's vertices. */
template <bool Unit, bool Map, typename Index>
__device__ __forceinline__ void vertex_store(const VertexStep& V, const EmitRows& E, const VertexRows& R, const Geom& g,
                                             float iso, float* __restrict__ pts, float* __restrict__ nrm,
                                             const Index* __restrict__ vmap)
{
    const int i = (int)(V.ent & ((64u << E.wp_log2) - 1u)), q = (int)(V.ent >> (6 + E.wp_log2));
    auto put = [&](uint32_t v, const float p[3], const float nn[3]) {
        const Vox3 vp{p[0], p[1], p[2]}, vn{nn[0], nn[1], nn[2]};
        if (Map) {
            const uint64_t id = (uint64_t)vmap[E.v0 + v];
            __builtin_memcpy(pts + 3 * id, &vp, sizeof(vp));
            __builtin_memcpy(nrm + 3 * id, &vn, sizeof(vn));
        } else {
            const uint32_t off = 12 * v;   // below 2^20
            __builtin_memcpy(reinterpret_cast<char*>(pts + 3 * E.v0) + off, &vp, sizeof(vp));
            __builtin_memcpy(reinterpret_cast<char*>(nrm + 3 * E.v0) + off, &vn, sizeof(vn));
        }
    };
    if (V.inner) {
        const Around& a = V.a;
        const float ga[3] = {central<Unit>(a.r.x, a.r.z, g.sp[0]), central<Unit>(a.ym.x, a.yp.y, g.sp[1]),
                             central<Unit>(a.zm.x, a.zp.y, g.sp[2])};
        const CornerCoords<Unit, Map> cc(g, i, V.j, V.k);
        const float num = iso - a.r.y;
        float p[3], nn[3];
        if (V.cut[0]) {
            const float gb[3] = {central<Unit>(a.r.y, a.r.w, g.sp[0]), central<Unit>(a.ym.y, a.yp.z, g.sp[1]),
                                 central<Unit>(a.zm.y, a.zp.z, g.sp[2])};
            cc.finish(g, 0, num / (a.r.z - a.r.y), ga, gb, p, nn);
            put(V.at[0], p, nn);
        }
        if (V.cut[1]) {
            const float gb[3] = {central<Unit>(a.yp.x, a.yp.z, g.sp[0]), central<Unit>(a.r.y, of_pair(a.y2), g.sp[1]),
                                 central<Unit>(of_pair(a.yz), of_pair(a.d), g.sp[2])};
            cc.finish(g, 1, num / (a.yp.y - a.r.y), ga, gb, p, nn);
            put(V.at[1], p, nn);
        }
        if (V.cut[2]) {
            const float gb[3] = {central<Unit>(a.zp.x, a.zp.z, g.sp[0]), central<Unit>(of_pair(a.zy), of_pair(a.d), g.sp[1]),
                                 central<Unit>(a.r.y, of_pair(a.z2), g.sp[2])};
            cc.finish(g, 2, num / (a.zp.y - a.r.y), ga, gb, p, nn);
            put(V.at[2], p, nn);
        }
    } else if (V.any) {
        const float* __restrict__ v = R.row0 + ((uint32_t)q * (uint32_t)g.nx + (uint32_t)i);
#pragma unroll
        for (int ax = 0; ax < 3; ++ax) {
            if (!V.cut[ax]) continue;
            float p[3], nn[3];
            if (Map && !Unit) {
                // Marching Cubes' corner coordinates, the general edge_point
                const CornerCoords<Unit, Map> cc(g, i, V.j, V.k);
                float A[3] = {cc.across(0), cc.across(1), cc.across(2)};
                A[ax] = cc.A[ax];
                float B[3] = {A[0], A[1], A[2]};
                B[ax] = A[ax] + g.sp[ax];
                edge_point(R.vol, g, iso, ax, i, V.j, V.k, A, B, p, nn);
            } else {
                fe_edge_point<Unit>(v, g, iso, ax, i, V.j, V.k, p, nn);
            }
            put(V.at[ax], p, nn);
        }
    }
}

/* Triangles of the wavefront's cell rows: active cells listed per lane in output order, then 64 at a
 * time one cell per lane (its case and its twelve vertex ids, into LDS), then one triangle per lane
 * (three ids from LDS, stored at consecutive addresses). Ids are written less vbias, or through
 * remap.
 * A cell needs the bits b and b + 1 of four rows and the ranks of eight edge combinations at b,
 * which one alignbit and one popcount each give from the 32-bit half that holds b; ranks of the
 * wavefront's own rows count from its first vertex v0, those of the plane above from v2, the first
 * vertex of the row above the wavefront's first, so that both fit 16 bits. */
template <typename Index, bool Remap>
__device__ __forceinline__ void emit_rows_triangles(const EmitRows& E, EmitRowsLds& S, const uint64_t* __restrict__ s_case,
                                                    Index* __restrict__ tris, uint64_t vbias,
                                                    const Index* __restrict__ remap)
{
    const int lane = E.lane;
    const uint64_t v0 = E.v0;
    const uint32_t ncell = (uint32_t)__popcll(E.act);
    const uint32_t cincl = wave_incl_scan_u32(ncell);
    const uint32_t ctotal = (uint32_t)__builtin_amdgcn_readlane((int)cincl, 63);
    if (ctotal == 0) return;
    const uint32_t cfirst = cincl - ncell;
    const uint64_t vrel = v0 - vbias;
    const uint32_t dv = (uint32_t)(E.v2 - v0);
    Index* __restrict__ out = tris + 3 * E.t0;
    for (uint32_t win = 0; win < ctotal; win += kEmitCellCap) {
        list_bits<kEmitCellCap>(E.act, cfirst, win, ctotal, lane, S.t.cells);
        wave_sync();
        const uint32_t n = min((uint32_t)kEmitCellCap, ctotal - win);
        for (uint32_t g0 = 0; g0 < n; g0 += 64) {
            const uint32_t idx = g0 + (uint32_t)lane;
            const uint32_t ent = idx < n ? (uint32_t)S.t.cells[idx] : 0u;
            const uint32_t h2 = ent >> 5, b = ent & 31;
            uint32_t w[4], t[4], x[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t lo = S.words[q][h2], hi = S.words[q][h2 + 1];
                w[q] = lo;
                t[q] = __builtin_amdgcn_alignbit(hi, lo, b);           // bits b and b + 1 of the row, at 0 and 1
                x[q] = lo ^ __builtin_amdgcn_alignbit(hi, lo, 1);      // cut x-edges of the half
            }
            const uint4 rk = S.rank[h2];
            const uint32_t cs = (t[0] & 3) | (t[1] & 3) << 2 | (t[2] & 3) << 4 | (t[3] & 3) << 6;
            uint64_t packed = s_case[cs];
            const uint32_t nt = idx < n ? (uint32_t)case_tri_count(packed) : 0u;
            const uint32_t below = bits_below(b);
            auto cnt = [&](uint32_t bits) { return (uint32_t)__popc(bits & below); };
            uint32_t* id = S.t.ids + kIdStride * lane;
            id[0] = rk.x + (cnt(x[0]) | cnt(x[1]) << 16);
            id[4] = rk.y + (cnt(x[2]) | cnt(x[3]) << 16);
            auto pair = [&](uint32_t r16, uint32_t bits, uint32_t cut) {
                const uint32_t at = r16 + cnt(bits);
                return at | (at + (cut & 1)) << 16;                    // at x = i and at x = i + 1
            };
            id[1] = pair(rk.z & 0xFFFFu, w[0] ^ w[1], t[0] ^ t[1]);
            id[5] = pair(rk.z >> 16, w[2] ^ w[3], t[2] ^ t[3]);
            id[2] = pair(rk.w & 0xFFFFu, w[0] ^ w[2], t[0] ^ t[2]);
            id[3] = pair(rk.w >> 16, w[1] ^ w[3], t[1] ^ t[3]);
            const uint32_t tincl = wave_incl_scan_u32(nt);
            const uint32_t ttot = (uint32_t)__builtin_amdgcn_readlane((int)tincl, 63);
            // the group's triangles in output order: byte offset of the cell's ids | its 3 slots << 12
            uint32_t* m = S.t.map + (tincl - nt);
            for (uint32_t tt = 0; tt < nt; ++tt, packed >>= 12)
                m[tt] = (uint32_t)(4 * kIdStride * lane) | (uint32_t)packed << 12;
            wave_sync();
            for (uint32_t e = lane; e < ttot; e += 64) {
                const uint32_t me = S.t.map[e];
                const uint32_t at = me & 0xFFFu;
                uint64_t id3[3];
#pragma unroll
                for (int s = 0; s < 3; ++s) {
                    const uint32_t slot = __builtin_amdgcn_ubfe(me, 12 + 4 * s, 4);
                    const uint32_t up = (uint32_t)__builtin_amdgcn_sbfe((int)me, 15 + 4 * s, 1);   // slots 8 .. 11
                    uint16_t rel;
                    __builtin_memcpy(&rel, reinterpret_cast<const char*>(S.t.ids) + (at + 2 * slot), 2);
                    id3[s] = vrel + ((uint32_t)rel + (up & dv));
                }
                if (Remap)
                    store_tri<Index>(out, e, remap[id3[0]], remap[id3[1]], remap[id3[2]]);
                else
                    store_tri<Index>(out, e, id3[0], id3[1], id3[2]);
            }
            out += 3 * ttot;
            wave_sync();
        }
    }
}

/* The wavefront's vertices and triangles. The first step's voxels are requested before the
 * triangles, which work from LDS (1024^3: 1.44 ms against 1.48 ms with the vertices first). */
template <typename Index, bool Unit, bool Map>
__device__ __forceinline__ void emit_rows_both(const EmitRows& E, EmitRowsLds& S, const uint64_t* __restrict__ s_case,
                                               const float* __restrict__ vol, const Geom& g, float iso,
                                               float* __restrict__ pts, float* __restrict__ nrm,
                                               Index* __restrict__ tris, uint64_t vbias,
                                               const Index* __restrict__ vmap)
{
    const VertexRows R = vertex_rows(E, vol, g);
    const uint32_t lane = (uint32_t)E.lane;
    VertexStep V;
    uint32_t n = min((uint32_t)kOriginCap, R.n);
    list_bits<kOriginCap>(E.origins, R.first, 0, R.n, E.lane, S.origins);
    wave_sync();
    vertex_load(V, E, S, R, g, lane, n);
    wave_sync();
    emit_rows_triangles<Index, Map>(E, S, s_case, tris, vbias, vmap);
    for (uint32_t win = 0;;) {
        for (uint32_t e0 = 0; e0 < n; e0 += 64) {
            vertex_store<Unit, Map, Index>(V, E, R, g, iso, pts, nrm, vmap);
            if (e0 + 64 < n) vertex_load(V, E, S, R, g, e0 + 64 + lane, n);
        }
        win += kOriginCap;
        if (win >= R.n) break;
        n = min((uint32_t)kOriginCap, R.n - win);
        wave_sync();
        list_bits<kOriginCap>(E.origins, R.first, win, R.n, E.lane, S.origins);
        wave_sync();
        vertex_load(V, E, S, R, g, lane, n);
    }
}

/* Lane-row block blk. s_case holds kCaseSlots; vertex ids are written less vbias (the first
 * vertex of this volume's output when several volumes share one buffer). */
template <typename Index, bool Unit>
__device__ __forceinline__ void fe_emit_rows_block(const uint64_t* __restrict__ s_case, EmitRowsLds* s_w,
                                                   const float* __restrict__ vol, const uint64_t* __restrict__ mask,
                                                   const Geom& g, float iso, const RowCounts* __restrict__ counts,
                                                   const uint64_t* __restrict__ voff,
                                                   const uint64_t* __restrict__ toff, float* __restrict__ pts,
                                                   float* __restrict__ nrm, Index* __restrict__ tris,
                                                   uint64_t vbias, int64_t blk)
{
    EmitRows E;
    if (!emit_rows_setup(E, s_w, mask, g, counts, voff, toff, blk)) return;
    emit_rows_both<Index, Unit, false>(E, s_w[E.wv], s_case, vol, g, iso, pts, nrm, tris, vbias, (const Index*)nullptr);
}

/* The order in which pass 4's blocks take the rows, across the 8 XCDs. The hardware hands blocks
 * to the XCDs round-robin (block b to XCD b mod 8); this gives each XCD tiles of TG consecutive
 * row blocks (about 64 grid rows) by TP = 3 planes instead of every eighth block, so that the
 * rows around a wavefront's own that its vertices read (j - 1 .. j + 2, k - 1 .. k + 2) are
 * mostly in the same XCD's L2, while all XCDs still move through the planes together (they share
 * the MALL). At 1024^3 pass 4 takes 1.63 ms in this order against 1.84 ms in dispatch order.
 * Identity when the blocks do not split the planes evenly. A bijection on [0, n) otherwise:
 * block b is the i-th (i = b / 8) of XCD x = b % 8, which takes tile t = i / (TG TP) of its
 * column of tiles, TP planes by TG blocks, planes first.
 * The plan (plan_block_order) is made on the host with the geometry, and a block maps its index
 * with shifts, multiplications and one 32-bit division. That matters at a sparse isovalue, where
 * most blocks write nothing: with the plan worked out in every block in 64-bit arithmetic, pass 4
 * at 1024^3, iso 0.95 took 0.15 ms against 0.08 ms. */
constexpr uint32_t kBlockOrderTP = 3;

inline BlockOrder plan_block_order(int64_t ny, int64_t nz, int64_t W, int lg_wp = -1)
{
    BlockOrder o{0u, 1u, 1u, 0u};
    if (W < 1 || W > 64 || ny >= (1ll << 30)) return o;
    const int64_t per_block = 4 * (64 >> (lg_wp < 0 ? fewest_lanes(W) : lg_wp));   // 4 wavefronts of lane rows: 4 .. 256
    const int64_t n = (ny * nz + per_block - 1) / per_block;
    if (ny % per_block || n > 0xFFFFFFFFll) return o;
    const int64_t G = ny / per_block;                       // blocks per plane
    int64_t TG = per_block >= 64 ? 1 : 64 / per_block;
    while (TG > 1 && G % (8 * TG)) TG >>= 1;
    if (G % (8 * TG)) return o;
    o.n0 = (uint32_t)(n / (G * kBlockOrderTP) * (G * kBlockOrderTP));   // whole tile rows
    o.G = (uint32_t)G;
    o.U = (uint32_t)(G / (8 * TG));
    o.lg_tg = (uint32_t)__builtin_ctzll((unsigned long long)TG);
    return o;
}

__host__ __device__ __forceinline__ uint32_t apply_block_order(const BlockOrder& o, uint32_t b)
{
    constexpr uint32_t TP = kBlockOrderTP;
    const uint32_t TG = 1u << o.lg_tg;
    const uint32_t x = b & 7u, i = b >> 3;
    const uint32_t q = (i >> o.lg_tg) / TP;                 // i / (TG TP): the XCD's tile
    const uint32_t t = i - q * (TG * TP), c = q / o.U, u = q - c * o.U;
    return (c * TP + t % TP) * o.G + (x + 8 * u) * TG + t / TP;
}

__device__ __forceinline__ int64_t emit_block_order(int64_t b, int64_t n, const Geom& g)
{
    // a bijection on [0, n0) and the identity above it, so also on any grid of at least n0 blocks
    if (b >= (int64_t)g.bo.n0 || n < (int64_t)g.bo.n0) return b;
    return apply_block_order(g.bo, (uint32_t)b);
}

/* The row block of block b of a single-volume pass 4 of n blocks: the order above from the end, where
 * the voxels lie that pass 1 read last (kKeepVoxels). */
__device__ __forceinline__ int64_t emit_block(int64_t b, int64_t n, const Geom& g)
{
    return n - 1 - emit_block_order(b, n, g);
}

template <typename Index, bool Unit>
__global__ __launch_bounds__(256) void k_fe_emit_rows(const float* __restrict__ vol,
                                                      const uint64_t* __restrict__ mask, Geom g, float iso,
                                                      const RowCounts* __restrict__ counts,
                                                      const uint64_t* __restrict__ voff,
                                                      const uint64_t* __restrict__ toff,
                                                      float* __restrict__ pts, float* __restrict__ nrm,
                                                      Index* __restrict__ tris, uint64_t vbias = 0,
                                                      const uint64_t* __restrict__ need = nullptr,
                                                      uint64_t cap_v = 0, uint64_t cap_t = 0)
{
    // with need (pass 3's totals, on the device), write nothing unless they fit the buffers and
    // the index width (the host then grows the buffers and runs this pass again)
    if (need && !output_fits<Index>(need, cap_v, cap_t)) return;
    __shared__ uint64_t s_case[256];
    __shared__ EmitRowsLds s_w[4];
    s_case[threadIdx.x] = kCaseSlots.v[threadIdx.x];
    __syncthreads();
    const int64_t blk = emit_block(blockIdx.x, gridDim.x, g);
    fe_emit_rows_block<Index, Unit>(s_case, s_w, vol, mask, g, iso, counts, voff, toff, pts, nrm, tris, vbias, blk);
}

/* Marching Cubes: the Flying Edges pass 4 with Marching Cubes' corner coordinates, every vertex written at
 * fe_to_mc[its Flying Edges id] and every triangle's ids read through the same map. */
template <typename Index, bool Unit>
__global__ __launch_bounds__(256) void k_mc_emit_rows(const float* __restrict__ vol,
                                                      const uint64_t* __restrict__ mask, Geom g, float iso,
                                                      const RowCounts* __restrict__ counts,
                                                      const uint64_t* __restrict__ voff,
                                                      const uint64_t* __restrict__ toff,
                                                      const Index* __restrict__ fe_to_mc, float* __restrict__ pts,
                                                      float* __restrict__ nrm, Index* __restrict__ tris,
                                                      const uint64_t* __restrict__ need = nullptr,
                                                      uint64_t cap_v = 0, uint64_t cap_t = 0)
{
    if (need && !output_fits<Index>(need, cap_v, cap_t)) return;   // as k_fe_emit_rows
    __shared__ uint64_t s_case[256];
    __shared__ EmitRowsLds s_w[4];
    s_case[threadIdx.x] = kCaseSlots.v[threadIdx.x];
    __syncthreads();
    const int64_t blk = emit_block(blockIdx.x, gridDim.x, g);
    EmitRows E;
    if (!emit_rows_setup(E, s_w, mask, g, counts, voff, toff, blk)) return;
    emit_rows_both<Index, Unit, true>(E, s_w[E.wv], s_case, vol, g, iso, pts, nrm, tris, 0, fe_to_mc);
}

}  // namespace miso

#endif
