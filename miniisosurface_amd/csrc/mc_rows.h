/*
 * mc_rows.h -- Marching Cubes with the serial reference's vertex numbering, in the (grid row,
 * mask word) lane layout of fe_rows.h.
 *
 * Vertex order (marchingCubes/serial/main.cpp:145-177, first visit through a hash map): the
 * owner of a cut edge is its adjacent cell with the smallest (k, j, i); ids run over owner cells
 * in linear order and, within a cell, over its owned edges in order of first appearance in the
 * cell's case triangle list. Triangles are the Flying Edges triangle stream with each vertex id
 * mapped to its Marching Cubes id.
 *
 *   k_fe_mc_count_rows Flying Edges pass 2 and the owned cut edges per cell row, bit-sliced over
 *                      the 64 cells of a word, in one pass over the mask words
 *   k_mc_ids_rows      the map from Flying Edges vertex id to Marching Cubes id
 *   k_mc_emit_rows     (fe_rows.h) Flying Edges pass 4 through that map
 */
#ifndef MINIISO_MC_ROWS_H
#define MINIISO_MC_ROWS_H

#include "fe_rows.h"

namespace miso {

/* Edges a cell owns: always 5, 6, 11; with k == 0 also 1, 2; with j == 0 also 4, 9; with
 * i == 0 also 7, 10; and 0 (j, k == 0), 3 (i, k == 0), 8 (i, j == 0). */
__device__ __forceinline__ uint32_t mc_owned_edges(bool i0, bool j0, bool k0)
{
    uint32_t m = (1u << 5) | (1u << 6) | (1u << 11);
    if (k0) m |= (1u << 1) | (1u << 2);
    if (j0) m |= (1u << 4) | (1u << 9);
    if (i0) m |= (1u << 7) | (1u << 10);
    if (j0 && k0) m |= 1u << 0;
    if (i0 && k0) m |= 1u << 3;
    if (i0 && j0) m |= 1u << 8;
    return m;
}

/* corner plane q (v0..v7) of the cells of a word */
__device__ __forceinline__ uint64_t corner_plane(const CornerWords& C, int q)
{
    switch (q) {
    case 0: return C.m[0];
    case 1: return C.s[0];
    case 2: return C.s[1];
    case 3: return C.m[1];
    case 4: return C.m[2];
    case 5: return C.s[2];
    case 6: return C.s[3];
    default: return C.m[3];
    }
}

/* Owned cut edges of the cell row of lane words L (row `at` from (j0, k0)), summed over the row's lanes
 * (valid in every lane of the row): bit-sliced over the 64 cells of a word. Lanes without cells (the
 * last row or plane, or past the row) count nothing, whatever their words. */
__device__ __forceinline__ uint32_t mc_owned_row_count(const LaneWords& L, const Geom& g, const RowLanes& rl,
                                                       const WaveRows& A, bool ok, const LaneRow& at)
{
    const int j = at.j;
    const bool k_first = A.k0 == 0 && at.dk == 0;
    const CornerWords C = corner_words(L);
    const uint64_t eb = (ok && at.has_y && at.has_z) ? word_bits(g, rl.w).eb : 0ull;
    const uint64_t first_cell = rl.w == 0 ? 1ull : 0ull;
    uint32_t cnt = 0;
#pragma unroll
    for (int e = 0; e < 12; ++e) {
        const uint64_t cut = corner_plane(C, kEdgeLo[e]) ^ corner_plane(C, kEdgeHi[e]);
        const bool need_i = (0x588u >> e) & 1u, need_j = (0x311u >> e) & 1u, need_k = (0x00Fu >> e) & 1u;
        // e: 0(j,k) 1(k) 2(k) 3(i,k) 4(j) 7(i) 8(i,j) 9(j) 10(i); always 5 6 11
        uint64_t own = eb;
        if (need_j && j != 0) own = 0;
        if (need_k && !k_first) own = 0;
        if (need_i) own &= first_cell;
        cnt += (uint32_t)__popcll(cut & own);
    }
    uint32_t all;
    return seg_sum(cnt, rl, all);
}

/* the owned-edge counts beside pass 2's (NoRowExtra) */
struct OwnedEdges {
    static constexpr bool kCounts = true;
    const Geom& g;
    uint32_t* __restrict__ owned;
    __device__ uint32_t operator()(const LaneWords& L, const RowLanes& rl, const WaveRows& A, bool ok, const LaneRow& at,
                                   bool empty) const
    {
        const uint32_t cnt = empty ? 0u : mc_owned_row_count(L, g, rl, A, ok, at);
        if (rl.q < A.n && rl.w == 0) row_entry(owned, A, rl.q) = cnt;
        return cnt;
    }
};

/* Flying Edges pass 2 (k_fe_count_rows) and the first-visit owned-edge counts per cell row in
 * one pass over the mask words, each row's words loaded once. */
__global__ __launch_bounds__(256) void k_fe_mc_count_rows(const uint64_t* __restrict__ mask, Geom g,
                                                          RowCounts* __restrict__ counts,
                                                          RowTrim* __restrict__ trims,
                                                          uint64_t* __restrict__ sums, int shift,
                                                          uint32_t* __restrict__ owned)
{
    uint32_t xy, zt;
    const WaveSums w = fe_count_rows_block(mask, g, counts, trims, blockIdx.x, OwnedEdges{g, owned}, xy, zt);
    add_block_sums(w, sums + (block_row(g, blockIdx.x) >> shift) * kTileSums);
}

/* Per case: for each cut edge e, its rank in order of first appearance in the case's triangle
 * list (nibble e, bits 4e .. 4e + 3), and the 12-bit mask of cut edges (bits 48 .. 59). */
__device__ __forceinline__ uint64_t first_appearance(uint64_t packed)
{
    uint64_t pos = 0;
    uint32_t seen = 0;
    int n = 0;
    const int ns = 3 * case_tri_count(packed);
    for (int s = 0; s < ns; ++s) {
        const int e = case_edge(packed, s);
        if ((seen >> e) & 1u) continue;
        seen |= 1u << e;
        pos |= (uint64_t)n << (4 * e);
        ++n;
    }
    return pos | (uint64_t)seen << 48;
}

/* Edge order (the order of util::duplicateRemover, marchingCubes/util/DuplicateRemover.h:34-70:
 * vertices sorted by global edge id, marchingCubes/util/Image3D.cpp:170-253): all cut x-edges in
 * (k, j, i) order, then all y-edges, then all z-edges. perm maps each Flying Edges vertex id
 * (row blocks [x][y][z]) to that order; xyz holds the per-row exclusive scans of the x, y and z
 * counts (R each) and tot their totals. Sixteen lanes per row, four rows per wavefront: the
 * lanes run over the row's ids [x][y][z] together (64-byte store runs). */
template <typename Index>
__global__ __launch_bounds__(256) void k_edge_order_perm(const RowCounts* __restrict__ counts,
                                                         const uint64_t* __restrict__ voff,
                                                         const uint64_t* __restrict__ xyz,
                                                         const uint64_t* __restrict__ tot, int64_t R,
                                                         Index* __restrict__ perm,
                                                         const uint64_t* __restrict__ need = nullptr,
                                                         uint64_t cap_v = 0, uint64_t cap_t = 0)
{
    if (need && !output_fits<Index>(need, cap_v, cap_t)) return;
    const int64_t r = (int64_t)blockIdx.x * 16 + (threadIdx.x >> 4);
    if (r >= R) return;
    const uint32_t l = threadIdx.x & 15;
    const RowCounts c = counts[r];
    const uint32_t n = c.x + c.y + c.z;
    if (n == 0) return;
    const uint64_t f0 = voff[r];
    // what each axis adds to t, modulo the ids' type: a selection and an addition per id (16x128x65536 noise
    // 258 us; 410 with each axis's own 64-bit sum)
    const Index dx = (Index)xyz[r], dy = (Index)(tot[0] + xyz[R + r] - c.x),
                dz = (Index)(tot[0] + tot[1] + xyz[2 * R + r] - c.x - c.y);
    const uint32_t cxy = c.x + c.y;
    for (uint32_t t = l; t < n; t += 16) perm[f0 + t] = (Index)((t < c.x ? dx : (t < cxy ? dy : dz)) + (Index)t);
}

/* The edges that a cell off the near faces may own (5, 6, 11) as a case has them: bits 0, 1, 2 that they are
 * cut, bits 4, 6, 8 on their places among them in order of first appearance. */
__device__ __forceinline__ uint16_t inner_order(uint64_t order)
{
    const int edge[3] = {5, 6, 11};
    uint32_t r = 0;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        if (!((order >> (48 + edge[a])) & 1ull)) continue;
        uint32_t before = 0;
#pragma unroll
        for (int b = 0; b < 3; ++b)
            before += ((order >> (48 + edge[b])) & 1ull) && ((order >> (4 * edge[b])) & 0xF) < ((order >> (4 * edge[a])) & 0xF);
        r |= 1u << a | before << (4 + 2 * a);
    }
    return (uint16_t)r;
}

/* LDS of one wavefront of k_mc_ids_rows: as EmitRowsLds. With this alone, not pass 4's whole struct, seven
 * blocks share a CU. A shorter list only costs a second round of listing: at the 512^3 gyroid the kernel takes
 * 82 us, 87 with 240 cells (seven blocks too), 87 with 176 (eight). */
constexpr int kMcIdsCells = 384;
struct McIdsLds {
    uint4 rank[128];
    uint32_t words[4][130];
    uint16_t cells[kMcIdsCells];
};
static_assert((sizeof(McIdsLds) * 4 + 256 * (8 + 2)) * 7 <= 163840, "seven blocks of k_mc_ids_rows share a CU's 160 KB");

/* First-visit order: the map from Flying Edges vertex id to Marching Cubes id. Active cells one per lane
 * in order, as in pass 4's triangles, from the same words and ranks: a scan of the owned edges' counts
 * gives a cell's first id, the edges' order of first appearance the ids within the cell. Cells off the
 * near faces own at most the three edges that meet at their far corner (5, 6, 11), whose Flying Edges
 * ids run on from cell to cell: the stores of 64 lanes are runs. 64 such cells take their edges' places
 * from a table by case (with the general order for all of them 84.5 us against 79 at the 512^3 gyroid). */
template <typename Index>
__global__ __launch_bounds__(256) void k_mc_ids_rows(const uint64_t* __restrict__ mask, Geom g,
                                                     const RowCounts* __restrict__ counts,
                                                     const uint64_t* __restrict__ voff,
                                                     const uint64_t* __restrict__ toff,
                                                     const uint64_t* __restrict__ moff, Index* __restrict__ fe_to_mc,
                                                     const uint64_t* __restrict__ need = nullptr,
                                                     uint64_t cap_v = 0, uint64_t cap_t = 0)
{
    if (need && !output_fits<Index>(need, cap_v, cap_t)) return;
    __shared__ uint64_t s_first[256];
    __shared__ uint16_t s_inner[256];
    __shared__ McIdsLds s_w[4];
    {
        // by the bits as the mask words give them (make_case_slots)
        const uint32_t c = threadIdx.x;
        s_first[c] = first_appearance(kCaseEdges[(c & 0x33) | (c & 0x44) << 1 | (c & 0x88) >> 1]);
        s_inner[c] = inner_order(s_first[c]);
    }
    __syncthreads();
    EmitRows E;
    if (!emit_rows_setup(E, s_w, mask, g, counts, voff, toff, emit_block(blockIdx.x, gridDim.x, g))) return;
    McIdsLds& S = s_w[E.wv];
    const uint32_t ncell = (uint32_t)__popcll(E.act);
    const uint32_t cincl = wave_incl_scan_u32(ncell);
    const uint32_t ctotal = (uint32_t)__builtin_amdgcn_readlane((int)cincl, 63);
    uint64_t mid = moff[E.r0];
    for (uint32_t win = 0; win < ctotal; win += kMcIdsCells) {
        list_bits<kMcIdsCells>(E.act, cincl - ncell, win, ctotal, E.lane, S.cells);
        wave_sync();
        const uint32_t n = min((uint32_t)kMcIdsCells, ctotal - win);
        for (uint32_t g0 = 0; g0 < n; g0 += 64) {
            const uint32_t idx = g0 + (uint32_t)E.lane;
            const uint32_t ent = idx < n ? (uint32_t)S.cells[idx] : 0u;
            const uint32_t h2 = ent >> 5, b = ent & 31;
            uint32_t w[4], t[4], x[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t lo = S.words[q][h2], hi = S.words[q][h2 + 1];
                w[q] = lo;
                t[q] = __builtin_amdgcn_alignbit(hi, lo, b);
                x[q] = lo ^ __builtin_amdgcn_alignbit(hi, lo, 1);
            }
            const uint4 rk = S.rank[h2];
            const uint32_t cs = (t[0] & 3) | (t[1] & 3) << 2 | (t[2] & 3) << 4 | (t[3] & 3) << 6;
            const int i = (int)(ent & ((64u << E.wp_log2) - 1u));
            int j = E.j0 + (int)(ent >> (6 + E.wp_log2));
            int64_t k = E.k0;
            while (j >= (int)g.ny) {
                j -= (int)g.ny;
                ++k;
            }
            const uint32_t below = bits_below(b);
            auto cnt = [&](uint32_t bits) { return (uint32_t)__popc(bits & below); };
            const uint32_t y1 = (rk.z >> 16) + cnt(w[2] ^ w[3]), z1 = (rk.w >> 16) + cnt(w[1] ^ w[3]);
            const uint64_t at5 = E.v2 + (y1 + ((t[2] ^ t[3]) & 1u)), at6 = E.v2 + ((rk.y >> 16) + cnt(x[3]));
            const uint64_t at11 = E.v0 + (z1 + ((t[1] ^ t[3]) & 1u));
            if (__ballot(idx < n && (i == 0 || j == 0 || k == 0)) == 0ull) {
                const uint32_t in = idx < n ? (uint32_t)s_inner[cs] : 0u, no = (uint32_t)__popc(in & 7u);
                const uint32_t incl = wave_incl_scan_u32(no);
                const uint64_t first = mid + (incl - no);
                if (in & 1u) fe_to_mc[at5] = (Index)(first + __builtin_amdgcn_ubfe(in, 4, 2));
                if (in & 2u) fe_to_mc[at6] = (Index)(first + __builtin_amdgcn_ubfe(in, 6, 2));
                if (in & 4u) fe_to_mc[at11] = (Index)(first + __builtin_amdgcn_ubfe(in, 8, 2));
                mid += (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
                continue;
            }
            const uint64_t order = s_first[cs];
            const uint32_t own = idx < n ? (uint32_t)(order >> 48) & 0xFFFu & mc_owned_edges(i == 0, j == 0, k == 0) : 0u;
            const uint32_t no = (uint32_t)__popc(own);
            const uint32_t incl = wave_incl_scan_u32(no);
            uint32_t place = 0;      // bit p: the edge that appears p-th is owned
            for (uint32_t o = own; o; o &= o - 1) place |= 1u << ((order >> (4 * __builtin_ctz(o))) & 0xF);
            const uint64_t first = mid + (incl - no);
            auto put = [&](int e, uint64_t fe) {
                if (!((own >> e) & 1u)) return;
                const uint32_t p = (uint32_t)(order >> (4 * e)) & 0xF;
                fe_to_mc[fe] = (Index)(first + (uint32_t)__popc(place & bits_below(p)));
            };
            const uint32_t y0 = (rk.z & 0xFFFFu) + cnt(w[0] ^ w[1]), z0 = (rk.w & 0xFFFFu) + cnt(w[0] ^ w[2]);
            put(6, at6);
            put(5, at5);
            put(11, at11);
            if (own & ~((1u << 5) | (1u << 6) | (1u << 11))) {
                put(0, E.v0 + ((rk.x & 0xFFFFu) + cnt(x[0])));
                put(2, E.v0 + ((rk.x >> 16) + cnt(x[1])));
                put(4, E.v2 + ((rk.y & 0xFFFFu) + cnt(x[2])));
                put(3, E.v0 + y0);
                put(1, E.v0 + (y0 + ((t[0] ^ t[1]) & 1u)));
                put(7, E.v2 + y1);
                put(8, E.v0 + z0);
                put(9, E.v0 + (z0 + ((t[0] ^ t[2]) & 1u)));
                put(10, E.v0 + z1);
            }
            mid += (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
        }
        wave_sync();
    }
}

}  // namespace miso

#endif
