/*
 * fe_batch.h -- Flying Edges over many volumes (or one volume at many isovalues) in one launch
 * per pass.
 *
 * The jobs' grid rows are concatenated into one row space: the per-row arrays (sign masks,
 * counts, trims, offsets) of job j start at row_base / mask_base. An item is one block of the
 * single-volume kernels (4 wavefronts of lane rows for counting and emission) of one job, found in the
 * jobs' item prefix. Pass 1 and pass 4 are one block per item, pass 2 one per few consecutive items (their
 * sums are added up once), and the dispatcher hands the blocks out as others end. Classification works
 * on groups of consecutive jobs that read the same volume (one volume at several isovalues): an item is
 * a block of the group's rows, loaded once for all its jobs. Pass 3 is the single-volume scan over the
 * concatenated rows, so job j's output is the contiguous range [voff[row_base_j], voff[row_base_{j+1}])
 * of one shared buffer; its triangles index its own vertices from 0. k_batch_fused runs the same block
 * functions for all four passes in one cooperative launch, with grid barriers between the passes.
 */
#ifndef MINIISO_FE_BATCH_H
#define MINIISO_FE_BATCH_H

#include <hip/hip_cooperative_groups.h>

#include "fe_rows.h"

namespace miso {

constexpr int kClassifyGroup = 16;   // jobs of one volume classified together (pass 1 of a batch)

struct BatchJob {
    Geom g;
    const float* vol;
    float iso;
    int unit;            // unit spacing and zero origin (the exact fast path of pass 4)
    int64_t row_base;    // first row of the job in the concatenated row arrays
    int64_t mask_base;   // first sign-mask word
};

/* The job's volume pointer, read from memory as what it is, a pointer to device memory: as a plain
 * pointer its loads become flat ones, for which LDS operations wait too. */
__device__ __forceinline__ const float* job_volume(const BatchJob& J)
{
    typedef const __attribute__((address_space(1))) float* GlobalFloats;
    GlobalFloats p;
    __builtin_memcpy(&p, &J.vol, sizeof(p));
    return (const float*)p;
}

/* The job whose item range holds `item` (the largest j < njobs with prefix[j] <= item), for a whole
 * wavefront: 64 ranges at a time. */
__device__ __forceinline__ int find_job(const int64_t* __restrict__ prefix, int njobs, int64_t item)
{
    int lo = 0, end = njobs;
    while (end - lo > 1) {
        const int step = (end - lo + 63) >> 6, at = lo + lane_id() * step;
        const int below = __popcll(__ballot(at < end && prefix[at < end ? at : lo] <= item));   // 1 .. 64
        lo += (below - 1) * step;
        end = min(end, lo + step);
    }
    return lo;
}

/* The items of block b of nblocks: the chunks b, b + nblocks, ... of `chunk` consecutive items each, or chunk b
 * alone (not Again); item i of job j after next(). Every wavefront walks the same items by itself: no barrier, and no queue's counter
 * to wait for (a counter gives out a ticket every 14 ns: pass 1 of 256 mixed volumes, then 170,000 items,
 * took 600 us with tickets). A chunk's job is looked up, not walked to: between two chunks lie as many jobs as
 * items where a job is one item, each a load that waits for the one before (20000 volumes of 3x3x3, fused launch:
 * 2254 us walked, 623 looked up). */
template <bool Again>
struct ItemWalk {
    const int64_t* __restrict__ prefix;
    int64_t nitems, stride, it, end, i;
    int chunk, njobs, j;

    __device__ __forceinline__ ItemWalk(const int64_t* __restrict__ p, int njobs, int64_t n, int c, int64_t b,
                                        int64_t nblocks)
        : prefix(p), nitems(n), stride((nblocks - 1) * c), it(b * c - 1), end(b * c + c), i(0), chunk(c), njobs(njobs),
          j(0)
    {
        if (b * c < n) j = find_job(p, njobs, b * c);
    }
    __device__ __forceinline__ bool next()
    {
        const bool jump = ++it == end;
        if (jump) {
            if (!Again) return false;
            it += stride;
            end = it + chunk;
        }
        if (it >= nitems) return false;
        if (it >= prefix[j + 1]) j = Again && jump ? find_job(prefix, njobs, it) : j + 1;   // no job is without items
        i = it - prefix[j];
        return true;
    }
};

/* Pass 2 of the batch's row blocks of this block's items, into the scan's tile sums: a wavefront keeps the
 * sums of the items it takes one after the other, as long as they lie in one tile, and adds them at
 * once (lane a, 0 .. 3, those of kind a). */
template <class Walk>
__device__ __forceinline__ void batch_count_items(const BatchJob* __restrict__ jobs, Walk walk,
                                                  const uint64_t* __restrict__ mask, RowCounts* __restrict__ counts,
                                                  RowTrim* __restrict__ trims, uint64_t* __restrict__ sums, int shift)
{
    const int lane = lane_id();
    int64_t tile = -1;
    uint64_t mine = 0;
    while (walk.next()) {
        const BatchJob& J = jobs[walk.j];
        uint32_t xy, zt;                   // per row, in one lane per row
        const WaveSums w = fe_count_rows_block(mask + J.mask_base, J.g, counts + J.row_base, trims + J.row_base, walk.i,
                                               NoRowExtra(), xy, zt);
        const RowLanes rl = row_lanes(J.g);
        const int64_t r0 = J.row_base + (walk.i * 4 + wave_in_block()) * rl.rpw;
        // a job's rows start anywhere in a tile, so a wavefront's may lie in two
        const int64_t first = r0 >> shift, last = (r0 + rl.rpw - 1) >> shift;
        for (int64_t t = first; t <= last; ++t) {
            WaveSums s = w;
            if (first != last) {
                const bool in = (r0 + rl.q) >> shift == t;
                s = WaveSums{wave_sum_u32(in ? xy : 0u), wave_sum_u32(in ? zt : 0u), 0u};
            }
            if ((s.xy | s.zt) == 0) continue;
            if (t != tile) {
                if (mine) add_sum(&sums[tile * kTileSums + lane], mine);
                mine = 0;
                tile = t;
            }
            mine += lane < 4 ? sum_of_kind(s, lane) : 0u;
        }
    }
    if (mine) add_sum(&sums[tile * kTileSums + lane], mine);
}

/* clears the scan's tile sums for the fused launch (a kernel, so it can sit in a graph) */
__global__ __launch_bounds__(256) void k_batch_zero(uint64_t* __restrict__ words, int64_t n)
{
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (int64_t)gridDim.x * blockDim.x)
        words[t] = 0;
}

/* Pass 1 item blk of classify group q: the jobs [group_job[q], group_job[q + 1]), consecutive jobs that
 * read the same volume with the same dimensions (one volume at several isovalues); a block of its rows
 * is loaded once and every job's sign-mask words written. bits: kFlatBits words of LDS per wavefront. */
__device__ __forceinline__ void batch_classify_item(const BatchJob* __restrict__ jobs,
                                                    const int* __restrict__ group_job, uint64_t* __restrict__ mask,
                                                    int q, int64_t blk, uint32_t* __restrict__ bits)
{
    const int j0 = group_job[q], n = group_job[q + 1] - j0;
    const BatchJob& J = jobs[j0];
    auto sink = [&](int t, float& iso, uint64_t*& m) {
        iso = jobs[j0 + t].iso;
        m = mask + jobs[j0 + t].mask_base;
    };
    if (J.g.W <= kFlatWords)
        fe_classify_flat_n(job_volume(J), J.g, n, sink, blk, flat_rows_per_wave(J.g.nx), bits);
    else
        fe_classify_block_n(job_volume(J), J.g, n, sink, blk, INT64_MAX);
}

/* Pass 1, one item per block, from item `first`. A wavefront's item is one chain of loads (its job, then 2048
 * voxels), which only other wavefronts' hide: 256 mixed volumes (1.24 GB) take 234 us with a block per item,
 * 253 with four items per block one after the other, 265 with 2048 blocks that walk all of them; a 256^3
 * volume at 16 isovalues 41, 59 and 59 us. */
__global__ __launch_bounds__(256) void k_batch_classify(const BatchJob* __restrict__ jobs,
                                                        const int* __restrict__ group_job,
                                                        const int64_t* __restrict__ prefix, int ngroups,
                                                        int64_t first, uint64_t* __restrict__ mask,
                                                        uint64_t* __restrict__ sums, int64_t nsums)
{
    __shared__ uint32_t s_bits[4][kFlatBits];
    // pass 2 adds up the scan's tile sums: clear them here
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < nsums; t += (int64_t)gridDim.x * blockDim.x)
        sums[t] = 0;
    const int64_t it = first + blockIdx.x;
    const int q = find_job(prefix, ngroups, it);
    batch_classify_item(jobs, group_job, mask, q, it - prefix[q], s_bits[threadIdx.x >> 6]);
}

/* Pass 2, a chunk of items per block, from chunk `first` of nchunks. 256 mixed volumes: 67 us with chunks of
 * four, 80 with one item per block (an atomic per item and kind), 87 with 2048 blocks that walk all chunks. */
__global__ __launch_bounds__(256) void k_batch_count(const BatchJob* __restrict__ jobs,
                                                     const int64_t* __restrict__ prefix, int njobs, int64_t nitems,
                                                     int chunk, int64_t first, int64_t nchunks,
                                                     const uint64_t* __restrict__ mask, RowCounts* __restrict__ counts,
                                                     RowTrim* __restrict__ trims, uint64_t* __restrict__ sums, int shift)
{
    batch_count_items(jobs, ItemWalk<false>(prefix, njobs, nitems, chunk, first + blockIdx.x, nchunks), mask, counts,
                      trims, sums, shift);
}

/* Job j's first vertex, first triangle, vertex and triangle counts (from the scan). */
__device__ __forceinline__ void batch_job_counts_one(const BatchJob* __restrict__ jobs, int njobs, int64_t R,
                                                     const uint64_t* __restrict__ voff,
                                                     const uint64_t* __restrict__ toff,
                                                     const uint64_t* __restrict__ totals, uint64_t* __restrict__ out,
                                                     uint64_t* __restrict__ host, int j)
{
    const int64_t b = jobs[j].row_base;
    const int64_t e = j + 1 < njobs ? jobs[j + 1].row_base : R;
    const uint64_t vb = b < R ? voff[b] : totals[0], tb = b < R ? toff[b] : totals[1];
    const uint64_t ve = e < R ? voff[e] : totals[0], te = e < R ? toff[e] : totals[1];
    const uint64_t c[4] = {vb, tb, ve - vb, te - tb};
    for (int q = 0; q < 4; ++q) {
        out[4 * j + q] = c[q];
        host[4 * j + q] = c[q];      // pinned memory
    }
}

__global__ __launch_bounds__(256) void k_batch_job_counts(const BatchJob* __restrict__ jobs, int njobs, int64_t R,
                                                          const uint64_t* __restrict__ voff,
                                                          const uint64_t* __restrict__ toff,
                                                          const uint64_t* __restrict__ totals,
                                                          uint64_t* __restrict__ out, uint64_t* __restrict__ host)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j < njobs) batch_job_counts_one(jobs, njobs, R, voff, toff, totals, out, host, j);
}

/* Which geometries a batch's jobs have: pass 4 holds the code of those only (with both, it takes 129
 * registers, and 3 wavefronts share a SIMD where 4 do otherwise). */
enum BatchUnits { kAllUnit, kNoneUnit, kSomeUnit };

/* Pass 4 of job j's row block blk into the shared output; the job's triangles index its own
 * vertices, from its first one, voff at its first row. */
template <BatchUnits Units>
__device__ __forceinline__ void batch_emit_item(const uint64_t* __restrict__ s_case, EmitRowsLds* s_w,
                                                const BatchJob* __restrict__ jobs, const uint64_t* __restrict__ mask,
                                                const RowCounts* __restrict__ counts,
                                                const uint64_t* __restrict__ voff, const uint64_t* __restrict__ toff,
                                                float* __restrict__ pts, float* __restrict__ nrm,
                                                uint32_t* __restrict__ tris, int j, int64_t blk)
{
    const BatchJob& J = jobs[j];
    const float* __restrict__ vol = job_volume(J);
    const uint64_t vbias = voff[J.row_base];
    if (Units == kAllUnit || (Units == kSomeUnit && J.unit))
        fe_emit_rows_block<uint32_t, true>(s_case, s_w, vol, mask + J.mask_base, J.g, J.iso, counts + J.row_base,
                                           voff + J.row_base, toff + J.row_base, pts, nrm, tris, vbias, blk);
    else
        fe_emit_rows_block<uint32_t, false>(s_case, s_w, vol, mask + J.mask_base, J.g, J.iso, counts + J.row_base,
                                            voff + J.row_base, toff + J.row_base, pts, nrm, tris, vbias, blk);
}

/* Item b of pass 4 for the first nemit jobs (nitems items): in dispatch order the items in job order,
 * from the last one, whose volume the caches may still hold; with xprefix, XCD b mod 8 (the dispatcher
 * hands workgroups to the 8 XCDs in turn) takes its own items: within job j the dispatch indices
 * 8 t + x < n_j, which emit_block_order maps to the job's row blocks as it maps the single-volume
 * kernel's blocks, so that each XCD's L2 sees tiles of neighbouring rows, and all XCDs move through a
 * job's planes together. xprefix[x (njobs + 1) + j]: XCD x's items before job j. */
template <BatchUnits Units>
__device__ __forceinline__ void batch_emit_nth(const uint64_t* __restrict__ s_case, EmitRowsLds* s_w,
                                               const BatchJob* __restrict__ jobs, const int64_t* __restrict__ prefix,
                                               int njobs, int64_t nitems, const uint64_t* __restrict__ mask,
                                               const RowCounts* __restrict__ counts, const uint64_t* __restrict__ voff,
                                               const uint64_t* __restrict__ toff, float* __restrict__ pts,
                                               float* __restrict__ nrm, uint32_t* __restrict__ tris,
                                               const int64_t* __restrict__ xprefix, int nemit, int64_t b)
{
    const int x = xprefix ? (int)(b & 7) : 0;
    const int64_t* __restrict__ pre = xprefix ? xprefix + (int64_t)x * (njobs + 1) : prefix;
    const int64_t it = xprefix ? b >> 3 : nitems - 1 - b;
    if (it < 0 || it >= pre[nemit]) return;
    const int j = find_job(pre, nemit, it);
    const int64_t i = it - pre[j];
    const int64_t blk = xprefix ? emit_block_order(8 * i + x, prefix[j + 1] - prefix[j], jobs[j].g) : i;
    batch_emit_item<Units>(s_case, s_w, jobs, mask, counts, voff, toff, pts, nrm, tris, j, blk);
}

/* Pass 4 for the first nemit jobs, one item per block, from item `first`; writes nothing when their output
 * exceeds the capacity (the host then grows the buffers and runs this pass again). The items' costs
 * differ, and the dispatcher evens them out for nothing: with tickets from a queue, one gyroid 256^3
 * volume at 16 isovalues took 1360 us for the batch, now 1080; 12 clients' jobs of one serving step 618, now
 * 505. */
template <BatchUnits Units>
__global__ __launch_bounds__(256) void k_batch_emit(const BatchJob* __restrict__ jobs,
                                                    const int64_t* __restrict__ prefix, int njobs, int64_t nitems,
                                                    const uint64_t* __restrict__ mask,
                                                    const RowCounts* __restrict__ counts,
                                                    const uint64_t* __restrict__ voff,
                                                    const uint64_t* __restrict__ toff,
                                                    const uint64_t* __restrict__ need, uint64_t cap_v,
                                                    uint64_t cap_t, float* __restrict__ pts, float* __restrict__ nrm,
                                                    uint32_t* __restrict__ tris, const int64_t* __restrict__ xprefix,
                                                    int nemit, int64_t first)
{
    __shared__ uint64_t s_case[256];
    __shared__ EmitRowsLds s_w[4];
    // need: vertices and triangles of the emitted jobs (the totals, or the first vertex and
    // triangle of the first job not emitted)
    if (need[0] > cap_v || need[1] > cap_t) return;
    s_case[threadIdx.x] = kCaseSlots.v[threadIdx.x];
    __syncthreads();
    batch_emit_nth<Units>(s_case, s_w, jobs, prefix, njobs, nitems, mask, counts, voff, toff, pts, nrm, tris, xprefix,
                          nemit, first + blockIdx.x);
}

/* Everything batch_run does on the device after clearing the tile sums, in one cooperative launch: the
 * grid (every block resident at once) runs pass 1 over the classify groups, pass 2, the scan and pass 4
 * (when the totals fit the output), with a grid-wide barrier between the phases, which also orders
 * every block's writes before the next phase's reads; the per-job counts for the host are written
 * beside pass 4, which does not read them. The block functions are those of the separate kernels, so
 * the output is theirs. state: [0..1] totals, [2..] the scan's tile sums. */
__global__ __launch_bounds__(256) void k_batch_fused(const BatchJob* __restrict__ jobs,
                                                     const int* __restrict__ group_job,
                                                     const int64_t* __restrict__ cls_prefix, int ngroups, int64_t ncls,
                                                     const int64_t* __restrict__ lane_prefix, int njobs,
                                                     int64_t nlane, int chunk, uint64_t* __restrict__ mask,
                                                     RowCounts* __restrict__ counts, RowTrim* __restrict__ trims,
                                                     uint64_t* __restrict__ voff, uint64_t* __restrict__ toff,
                                                     uint64_t* __restrict__ state, int64_t R, int shift,
                                                     int64_t ntiles, uint64_t* __restrict__ jobout,
                                                     uint64_t* __restrict__ host, uint64_t cap_v, uint64_t cap_t,
                                                     float* __restrict__ pts, float* __restrict__ nrm,
                                                     uint32_t* __restrict__ tris, const int64_t* __restrict__ xprefix,
                                                     int64_t nemit_items)
{
    namespace cg = cooperative_groups;
    cg::grid_group grid = cg::this_grid();
    __shared__ uint64_t s_case[256];
    __shared__ EmitRowsLds s_w[4];
    s_case[threadIdx.x] = kCaseSlots.v[threadIdx.x];
    ItemWalk<true> walk(cls_prefix, ngroups, ncls, chunk, blockIdx.x, gridDim.x);
    // pass 1's bits where pass 4 has its lists
    uint32_t* bits = reinterpret_cast<uint32_t*>(&s_w[wave_in_block()]);
    while (walk.next()) batch_classify_item(jobs, group_job, mask, walk.j, walk.i, bits);
    grid.sync();
    batch_count_items(jobs, ItemWalk<true>(lane_prefix, njobs, nlane, chunk, blockIdx.x, gridDim.x), mask, counts,
                      trims, state + 2, shift);
    grid.sync();
    for (int64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x)
        fe_scan_tile(counts, R, voff, toff, state + 2, shift, ntiles, state, host + 4 * (int64_t)njobs, ScanMore(), tile);
    grid.sync();
    for (int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; j < njobs; j += (int64_t)gridDim.x * blockDim.x)
        batch_job_counts_one(jobs, njobs, R, voff, toff, state, jobout, host, (int)j);
    if (state[0] > cap_v || state[1] > cap_t) return;
    // block b's items: b, b + the grid's blocks (a multiple of 8 with the XCD order), ...
    for (int64_t b = blockIdx.x; b < nemit_items; b += gridDim.x) {
        batch_emit_nth<kSomeUnit>(s_case, s_w, jobs, lane_prefix, njobs, nlane, mask, counts, voff, toff, pts, nrm, tris,
                                  xprefix, njobs, b);
        wave_sync();
    }
}

}  // namespace miso

#endif
