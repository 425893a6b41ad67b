/*
 * mc_kernels.h -- Marching Cubes with the serial reference's vertex numbering, as HIP kernels.
 *
 * The serial reference (marchingCubes/serial/main.cpp:42-192) visits every cell in z, y, x
 * order and numbers a cut edge the first time a cell's triangle list names it (through a hash
 * map keyed by the global edge id, :145-177). Every cut edge is named by each adjacent cell, so
 * the first visitor is the adjacent cell with the smallest (k, j, i): the "owner". A cell owns
 * its edges on the far side of each axis, plus those on the near side where it is the first
 * cell along that axis (i == 0, j == 0 or k == 0). Vertex ids therefore follow (owner cell in
 * linear order, first slot of the edge in the owner's case triangle list) -- no hash map needed.
 *
 *   k_mc_count      owned cut edges per cell row
 *   k_fe_scan       scans those counts too (vertex offsets per cell row)
 *   k_mc_vertices   owners write point and normal (with the owner's corner coordinates,
 *                   marchingCubes/util/Image3D.cpp:22-65) and record, at the edge's Flying Edges
 *                   rank, the Marching Cubes id
 *   k_mc_triangles  triangles in the same order as Flying Edges, ids read through that map
 */
#ifndef MINIISO_MC_KERNELS_H
#define MINIISO_MC_KERNELS_H

#include "fe_kernels.h"

namespace miso {

/* Edges a cell owns under first-visit numbering, given whether it is first along x, y, z. */
__device__ __forceinline__ uint32_t owned_edges(bool i0, bool j0, bool k0)
{
    uint32_t m = (1u << 6) | (1u << 5) | (1u << 11);
    if (k0) m |= (1u << 2) | (1u << 1);
    if (j0) m |= (1u << 4) | (1u << 9);
    if (i0) m |= (1u << 7) | (1u << 10);
    if (j0 && k0) m |= 1u << 0;
    if (i0 && k0) m |= 1u << 3;
    if (i0 && j0) m |= 1u << 8;
    return m;
}

/* owned edges of cell row r, which has triangles, in every lane */
__device__ __forceinline__ uint32_t mc_count_row(const uint64_t* __restrict__ mask, const Geom& g,
                                                 const uint16_t* __restrict__ s_cut, EmitLds& L, int64_t r)
{
    const int lane = lane_id();
    const int64_t j = r % g.ny, k = r / g.ny;
    RowWalker rw(L, mask, g, r, true, true);
    uint32_t total = 0;
    for (int64_t s0w = 0; s0w < g.W; s0w += kSegWords) {
        rw.stage(s0w);
        const int na = rw.prepare_cells();
        for (int e = lane; e < na; e += 64) {
            const int li = L.list[e];
            const int64_t i = s0w * 64 + li;
            const int cs = rw.cell_case(li);
            total += __popc(s_cut[cs] & owned_edges(i == 0, j == 0, k == 0));
        }
        wave_sync();
    }
    return wave_sum_u32(total);
}

/* Rows of a wavefront of k_mc_count, one after the other: four where there are blocks enough all the same. The time
 * of a volume with few triangles is that of handing out the blocks: 700x700x4100 without one takes 541 us with a
 * row per wavefront, 150 with four. */
inline int mc_count_rows(int64_t R) { return R >= (int64_t(1) << 16) ? 4 : 1; }

__global__ __launch_bounds__(256) void k_mc_count(const uint64_t* __restrict__ mask, Geom g,
                                                  const RowCounts* __restrict__ counts,
                                                  uint32_t* __restrict__ owned, uint64_t* __restrict__ sums, int shift,
                                                  int per)
{
    __shared__ EmitLds lds_all[kRowsPerBlock];
    __shared__ uint16_t s_cut[256];
    __shared__ uint64_t s_sums[kRowsPerBlock][1];
    const int lane = lane_id(), wave = threadIdx.x >> 6;
    const int64_t first = (int64_t)blockIdx.x * kRowsPerBlock * per, r0 = first + wave * per;
    const bool there = lane < per && r0 + lane < g.ny * g.nz;      // a lane per row
    const uint64_t live = __ballot(there && counts[r0 + lane].t != 0);   // no triangles on the last row or plane
    if (!__syncthreads_or(live != 0)) {
        if (there) owned[r0 + lane] = 0;
        return;
    }
    s_cut[threadIdx.x] = kCaseCuts.v[threadIdx.x];
    __syncthreads();
    uint32_t mine = 0;
    uint64_t total = 0;
    for (uint64_t rest = live; rest; rest &= rest - 1) {
        const int q = __builtin_ctzll(rest);
        const uint32_t n = mc_count_row(mask, g, s_cut, lds_all[wave], r0 + q);
        if (lane == q) mine = n;
        total += n;
    }
    if (there) owned[r0 + lane] = mine;
    if (lane == 0) s_sums[wave][0] = total;
    add_rows_sums<1>(s_sums, sums + (first >> shift) * kTileSums + 4);
}

/* EdgeOrder: each owned edge's point goes to fe_to_mc[its Flying Edges id] (an edge-order
 * permutation made beforehand), which this kernel then only reads; moff is not used. */
template <typename Index, bool EdgeOrder = false>
__global__ __launch_bounds__(256) void k_mc_vertices(const float* __restrict__ vol,
                                                     const uint64_t* __restrict__ mask, Geom g, float iso,
                                                     const RowCounts* __restrict__ counts,
                                                     const uint64_t* __restrict__ voff,
                                                     const uint64_t* __restrict__ moff,
                                                     float* __restrict__ pts, float* __restrict__ nrm,
                                                     Index* __restrict__ fe_to_mc)
{
    __shared__ EmitLds lds_all[kRowsPerBlock];
    __shared__ uint16_t s_cut[256];
    s_cut[threadIdx.x] = kCaseCuts.v[threadIdx.x];
    __syncthreads();
    const int lane = lane_id();
    const int wave = threadIdx.x >> 6;
    const int64_t r = (int64_t)blockIdx.x * kRowsPerBlock + wave;
    if (r >= g.ny * g.nz) return;
    const int64_t j = r % g.ny, k = r / g.ny;
    const bool has_y = j < g.ny - 1, has_z = k < g.nz - 1;
    if (!(has_y && has_z) || counts[r].t == 0) return;
    RowWalker rw(lds_all[wave], mask, g, r, has_y, has_z);
    EmitLds& L = lds_all[wave];
    uint64_t cbase[8];
    combo_bases(counts, voff, rw.rows, cbase);
    uint64_t mrun = EdgeOrder ? 0 : moff[r];
    const float Y = g.org[1] + (float)j * g.sp[1], Z = g.org[2] + (float)k * g.sp[2];
    for (int64_t s0w = 0; s0w < g.W; s0w += kSegWords) {
        rw.stage(s0w);
        const int na = rw.prepare_cells();
        for (int e0 = 0; e0 < na; e0 += 64) {
            const int e = e0 + lane;
            int li = 0, cs = 0;
            uint32_t own = 0;
            if (e < na) {
                li = L.list[e];
                cs = rw.cell_case(li);
                own = s_cut[cs] & owned_edges(s0w * 64 + li == 0, j == 0, k == 0);
            }
            const uint32_t o = (uint32_t)__popc(own);
            const uint32_t incl = wave_incl_scan_u32(o);
            if (own) {
                const int64_t i = s0w * 64 + li;
                const float X = g.org[0] + (float)i * g.sp[0];
                const uint64_t packed = kCaseEdges[cs];
                uint64_t vid = mrun + incl - o;
                uint32_t seen = 0;
                const int ne = 3 * case_tri_count(packed);
                for (int s = 0; s < ne; ++s) {
                    const int ed = case_edge(packed, s);
                    if (!((own >> ed) & 1u) || ((seen >> ed) & 1u)) continue;
                    seen |= 1u << ed;
                    const int a = edge_axis(ed);
                    const int dx = edge_dx(ed), dy = edge_dy(ed), dz = edge_dz(ed);
                    // corner coordinates as the owner cell computes them (getPosCube)
                    float A[3] = {dx ? X + g.sp[0] : X, dy ? Y + g.sp[1] : Y, dz ? Z + g.sp[2] : Z};
                    float B[3] = {A[0], A[1], A[2]};
                    B[a] = A[a] + g.sp[a];
                    float p[3], nn[3];
                    edge_point(vol, g, iso, a, i + dx, j + dy, k + dz, A, B, p, nn);
                    const uint64_t fe = rw.fe_vertex_id(cbase, ed, li);
                    if (EdgeOrder) vid = (uint64_t)fe_to_mc[fe];
                    pts[3 * vid + 0] = p[0];
                    pts[3 * vid + 1] = p[1];
                    pts[3 * vid + 2] = p[2];
                    nrm[3 * vid + 0] = nn[0];
                    nrm[3 * vid + 1] = nn[1];
                    nrm[3 * vid + 2] = nn[2];
                    if (!EdgeOrder) fe_to_mc[fe] = (Index)vid;
                    ++vid;
                }
            }
            mrun += __shfl(incl, 63);
        }
        rw.advance_bases(cbase);
        wave_sync();
    }
}

template <typename Index>
__global__ __launch_bounds__(256) void k_mc_triangles(const uint64_t* __restrict__ mask, Geom g,
                                                      const RowCounts* __restrict__ counts,
                                                      const uint64_t* __restrict__ voff,
                                                      const uint64_t* __restrict__ toff,
                                                      const Index* __restrict__ fe_to_mc,
                                                      Index* __restrict__ tris)
{
    __shared__ EmitLds lds_all[kRowsPerBlock];
    const int lane = lane_id();
    const int wave = threadIdx.x >> 6;
    const int64_t r = (int64_t)blockIdx.x * kRowsPerBlock + wave;
    if (r >= g.ny * g.nz) return;
    const int64_t j = r % g.ny, k = r / g.ny;
    const bool has_y = j < g.ny - 1, has_z = k < g.nz - 1;
    if (!(has_y && has_z) || counts[r].t == 0) return;
    RowWalker rw(lds_all[wave], mask, g, r, has_y, has_z);
    EmitLds& L = lds_all[wave];
    uint64_t cbase[8];
    combo_bases(counts, voff, rw.rows, cbase);
    uint64_t tri_run = toff[r];
    for (int64_t s0w = 0; s0w < g.W; s0w += kSegWords) {
        rw.stage(s0w);
        const int na = rw.prepare_cells();
        for (int e0 = 0; e0 < na; e0 += 64) {
            const int e = e0 + lane;
            int cs = 0, nt = 0, li = 0;
            if (e < na) {
                li = L.list[e];
                cs = rw.cell_case(li);
                nt = case_tri_count(kCaseEdges[cs]);
            }
            const uint32_t incl = wave_incl_scan_u32((uint32_t)nt);
            const uint64_t slot0 = tri_run + incl - (uint32_t)nt;
            if (nt) {
                const uint64_t packed = kCaseEdges[cs];
                for (int t = 0; t < nt; ++t) {
                    const uint64_t a = fe_to_mc[rw.fe_vertex_id(cbase, case_edge(packed, 3 * t + 0), li)];
                    const uint64_t b = fe_to_mc[rw.fe_vertex_id(cbase, case_edge(packed, 3 * t + 1), li)];
                    const uint64_t c = fe_to_mc[rw.fe_vertex_id(cbase, case_edge(packed, 3 * t + 2), li)];
                    store_tri<Index>(tris, slot0 + t, a, b, c);
                }
            }
            tri_run += __shfl(incl, 63);
        }
        rw.advance_bases(cbase);
        wave_sync();
    }
}

}  // namespace miso

#endif
