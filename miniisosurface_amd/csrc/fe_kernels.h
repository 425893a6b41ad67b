/*
 * fe_kernels.h -- Flying Edges passes 1-4 as HIP kernels for gfx950 (wave64).
 *
 *   k_fe_classify  pass 1a: a wavefront per grid row, or for several short ones, coalesced loads,
 *                  v >= iso into the 1-bit sign mask (replaces FlyingEdgesAlgorithm.cpp:31-45).
 *   k_fe_count     pass 1b + pass 2: from the masks of rows (j,k), (j+1,k), (j,k+1), (j+1,k+1):
 *                  xl/xr trims (cpp:47-65 with isCutEdge :515-554), cut-edge counts per grid
 *                  row and triangle counts per cell row (cpp:72-190) with popcounts.
 *   k_fe_scan      pass 3: exclusive scan of the per-row vertex and triangle counts into 64-bit
 *                  offsets (cpp:196-269), tile by tile on the tile sums that pass 2 adds up.
 *   k_fe_emit      pass 4: per grid row, the cut edges are compacted into an LDS list already in
 *                  output order, so lanes write consecutive vertices; per cell row, the active
 *                  cells are compacted, a wave prefix sum of numTris gives triangle slots, and
 *                  vertex ids come from row offsets plus popcount ranks (cpp:275-497).
 */
#ifndef MINIISO_FE_KERNELS_H
#define MINIISO_FE_KERNELS_H

#include "fe_common.h"

namespace miso {

constexpr int kRowsPerBlock = 4;        // one wavefront per grid row, 4 waves per block
constexpr int kSegWords = 16;           // pass 4 processes a row in segments of 16 words (1024 voxels)

/* Pass 3 works on tiles of 2^shift rows: at least 1024 (256 threads, four rows each), and so many that
 * a scan has at most 1024 tiles as long as tiles of 2^22 rows do: each tile's block adds up the sums of
 * the tiles before it. Per tile, the sums of the rows' x, y, z, triangle and (first-visit Marching
 * Cubes) owned-edge counts. */
constexpr int kTileSums = 5;
constexpr int kScanStep = 1024;      // rows per block and step
struct ScanPlan {
    int shift;
    int64_t ntiles;
    // words for the tile sums of up to this many rows: fewer rows may have up to 1024 tiles all the same
    int64_t sum_words() const { return kTileSums * (ntiles > 1024 ? ntiles : 1024); }
};
inline ScanPlan plan_scan(int64_t R)
{
    ScanPlan p{10, 0};
    while (p.shift < 22 && (R >> p.shift) >= 1024) ++p.shift;
    p.ntiles = (R + (int64_t(1) << p.shift) - 1) >> p.shift;
    return p;
}

/* adds v to a tile sum (pass 1 or the batch's first kernel has cleared them) */
__device__ __forceinline__ void add_sum(uint64_t* __restrict__ sum, uint64_t v)
{
    (void)__hip_atomic_fetch_add((unsigned long long*)sum, (unsigned long long)v, __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_AGENT);
}

/* A wavefront's counts, the same in every lane: xy = x | y << 16, zt = z | t << 16 (a wavefront's totals stay
 * below 2^16), and its owned edges. */
struct WaveSums {
    uint32_t xy, zt, own;
};

/* kind a of a wavefront's sums: x, y, z, t, owned */
__device__ __forceinline__ uint32_t sum_of_kind(const WaveSums& w, int a)
{
    return a == 4 ? w.own : ((a & 2) ? w.zt : w.xy) >> ((a & 1) * 16) & 0xFFFFu;
}

/* ------------------------------------------------------------------ pass 1a: sign mask */
/* Voxels at the end of a volume that pass 1 leaves in the 256 MB cache beside the HBM, where pass 4,
 * which takes the rows from the end (emit_block), finds them: 128 MB. Streamed past the caches as the
 * rest is, pass 4 reads them from HBM again: 512^3 gyroid 496 us against 475 us, 333x257x190 144
 * against 131, 1024^3 2.284 ms against 2.267. 256 MB: 482 us and 2.279 ms (pass 1 slows down by more
 * than pass 4 gains); every voxel, and pass 4 from the start: 515 us and 2.340 ms. The kernels of wider rows
 * take them from the start, so that only a volume that is kept whole gains: 64x64x4097 noise at 0.98 200 us
 * against 210, 16x128x65536 1960 us against 1946 with its last 128 MB kept. */
constexpr int64_t kKeepVoxels = int64_t(1) << 25;

inline int64_t keep_from_row(const Geom& g, bool from_end)
{
    const int64_t r = g.ny * g.nz - (kKeepVoxels + g.nx - 1) / g.nx;
    return from_end || r <= 0 ? r : g.ny * g.nz;
}

/* Rows 4 blk .. 4 blk + 3, one per wavefront. Each lane loads 4 consecutive voxels (one 16-byte
 * non-temporal load, so a wavefront step covers 256 voxels = 4 mask words); its 4 sign bits are placed at
 * bit 4 * (lane % 16) and OR-reduced over each 16-lane row with DPP, so lane 16 t + 15 ends up
 * holding mask word t of the step. Rows from keep_row on are read with plain loads instead, so that
 * they stay in the caches for pass 4 (kKeepVoxels). Voxels past nx read as below the isovalue.
 * The voxels are loaded once and classified against n isovalues of the same volume:
 * sink(t, iso, mask) names isovalue t and the mask array it writes (n = 1 for one extraction). */
template <class Sink>
__device__ __forceinline__ void fe_classify_block_n(const float* __restrict__ vol, const Geom& g, int n, Sink sink,
                                                    int64_t blk, int64_t keep_row)
{
    const int lane = lane_id();
    const int64_t r = blk * kRowsPerBlock + (threadIdx.x >> 6);
    if (r >= g.ny * g.nz) return;
    const float* __restrict__ row = vol + r * g.nx;
    const int sub = lane & 15;
    constexpr int kSteps = 4;                      // 1024 voxels in flight per wavefront
    for (int64_t c0 = 0; c0 < g.nx; c0 += 256 * kSteps) {
        float v[kSteps][4];
        uint32_t in[kSteps];                       // bit c: voxel i + c lies in the row
#pragma unroll
        for (int u = 0; u < kSteps; ++u) {
#pragma unroll
            for (int c = 0; c < 4; ++c) v[u][c] = 0.0f;
            in[u] = 0;
            if (c0 + 256 * u >= g.nx) continue;    // wavefront-uniform: short rows skip whole steps
            const int64_t i = c0 + 256 * u + 4 * lane;
            if (i + 4 <= g.nx) {
                const Vox4 q = r < keep_row ? load_vox4_stream(row + i) : load_vox<Vox4>(row + i);
                v[u][0] = q.x; v[u][1] = q.y; v[u][2] = q.z; v[u][3] = q.w;
                in[u] = 15u;
            } else {
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    v[u][c] = i + c < g.nx ? row[i + c] : 0.0f;
                    in[u] |= (uint32_t)(i + c < g.nx) << c;
                }
            }
        }
        for (int t = 0; t < n; ++t) {
            float iso;
            uint64_t* mask;
            sink(t, iso, mask);
            uint64_t* __restrict__ mrow = mask + r * g.W;
#pragma unroll
            for (int u = 0; u < kSteps; ++u) {
                if (c0 + 256 * u >= g.nx) break;
                uint32_t nib = 0;
#pragma unroll
                for (int c = 0; c < 4; ++c) nib |= (uint32_t)(v[u][c] >= iso) << c;
                nib &= in[u];
                // bits of lane sub go to 4 sub .. 4 sub + 3 of the (lo, hi) 32-bit halves of the word
                uint32_t lo = sub < 8 ? nib << (4 * sub) : 0u;
                uint32_t hi = sub < 8 ? 0u : nib << (4 * (sub - 8));
                lo |= dpp_u32<kDppRowShr1>(lo);
                hi |= dpp_u32<kDppRowShr1>(hi);
                lo |= dpp_u32<kDppRowShr2>(lo);
                hi |= dpp_u32<kDppRowShr2>(hi);
                lo |= dpp_u32<kDppRowShr4>(lo);
                hi |= dpp_u32<kDppRowShr4>(hi);
                lo |= dpp_u32<kDppRowShr8>(lo);
                hi |= dpp_u32<kDppRowShr8>(hi);
                const int64_t w = (c0 + 256 * u) / 64 + (lane >> 4);
                if (sub == 15 && w < g.W) mrow[w] = (uint64_t)hi << 32 | lo;
            }
        }
    }
}

/* Short rows (W <= kFlatWords): a wavefront takes `per` whole rows, at most 2048 voxels, which lie one after
 * the other, and classifies them as one run, eight voxels per lane and step: a byte of sign bits, put in
 * LDS. A row's words are then cut from the run of bits wherever they start. All steps are in flight at
 * once, and no lane waits at a row's end: with a row's words loaded one voxel per lane, 16 words a
 * wavefront, pass 1 of 256 mixed volumes (32 to 256 a side, 1.24 GB) was bound by its instructions and took
 * 385 us, then 265, and 235 with a block per item. 1024, 1536 or 3072 voxels a wavefront: the batch 500, 493
 * and 512 us against 495; streaming loads 575 against 552 (neighbouring lanes' halves of a line are read
 * twice). Longer rows (up to 512 or 1024 voxels) gain nothing (400x300x280: 212 us either way), and large
 * volumes of them lose the streaming loads of the row kernel (512^3: 103 us against 85). */
constexpr int kFlatWords = 4;
constexpr int kFlatSteps = 4;
constexpr int kFlatVoxels = 512 * kFlatSteps;
constexpr int kFlatBits = kFlatVoxels / 32 + 4;    // LDS words of a wavefront
__host__ __device__ __forceinline__ int flat_rows_per_wave(int64_t nx) { return kFlatVoxels / (int)nx; }

template <class Sink>
__device__ __forceinline__ void fe_classify_flat_n(const float* __restrict__ vol, const Geom& g, int n, Sink sink,
                                                   int64_t blk, int per, uint32_t* __restrict__ bits)
{
    const int lane = lane_id(), wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int64_t r0 = (blk * 4 + wv) * per, left = g.ny * g.nz - r0;
    if (left <= 0) return;
    const int nx = (int)g.nx, W = (int)g.W, rows = (int)(left < per ? left : per), voxels = rows * nx;
    const int64_t there = left * g.nx;                  // voxels to the volume's end
    const float* __restrict__ base = vol + r0 * g.nx;
    float v[kFlatSteps][8];
#pragma unroll
    for (int u = 0; u < kFlatSteps; ++u) {
        const int p = 512 * u + 8 * lane;
        if (512 * u >= voxels) {
#pragma unroll
            for (int c = 0; c < 8; ++c) v[u][c] = 0.0f;
        } else if (p + 8 <= there) {
            const Vox4 a = load_vox<Vox4>(base + p), b = load_vox<Vox4>(base + p + 4);
            v[u][0] = a.x; v[u][1] = a.y; v[u][2] = a.z; v[u][3] = a.w;
            v[u][4] = b.x; v[u][5] = b.y; v[u][6] = b.z; v[u][7] = b.w;
        } else {
#pragma unroll
            for (int c = 0; c < 8; ++c) v[u][c] = p + c < there ? base[p + c] : 0.0f;
        }
    }
    for (int t = 0; t < n; ++t) {
        float iso;
        uint64_t* mask;
        sink(t, iso, mask);
#pragma unroll
        for (int u = 0; u < kFlatSteps; ++u) {
            if (512 * u >= voxels) break;
            uint32_t byte = 0;
#pragma unroll
            for (int c = 7; c >= 0; --c) byte = byte + byte + (uint32_t)(v[u][c] >= iso);
            reinterpret_cast<uint8_t*>(bits)[64 * u + lane] = (uint8_t)byte;
        }
        wave_sync();
        uint64_t* __restrict__ out = mask + r0 * W;
        for (int e = lane; e < rows * W; e += 64) {
            const int q = W == 1 ? e : (W == 2 ? e >> 1 : (W == 3 ? (e * 43691) >> 17 : e >> 2));
            const int w = e - q * W, at = q * nx + 64 * w, in = nx - 64 * w;      // voxels from the word on
            const uint32_t* d = bits + (at >> 5);
            const uint32_t lo = __builtin_amdgcn_alignbit(d[1], d[0], at & 31);
            const uint32_t hi = __builtin_amdgcn_alignbit(d[2], d[1], at & 31);
            const uint64_t word = (uint64_t)hi << 32 | lo;
            out[e] = in < 64 ? word & ((1ull << in) - 1ull) : word;
        }
        wave_sync();
    }
}

/* rows of a pass 1 block */
inline int64_t classify_rows(const Geom& g)
{
    return g.W <= kFlatWords ? 4 * flat_rows_per_wave(g.nx) : kRowsPerBlock;
}

__global__ __launch_bounds__(256) void k_fe_classify(const float* __restrict__ vol, Geom g, float iso,
                                                     uint64_t* __restrict__ mask, int64_t keep_row,
                                                     uint64_t* __restrict__ sums, int64_t nsums)
{
    __shared__ uint32_t s_bits[4][kFlatBits];
    // pass 2 adds up the tile sums of pass 3: clear them here
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < nsums; t += (int64_t)gridDim.x * blockDim.x)
        sums[t] = 0;
    auto sink = [&](int, float& is, uint64_t*& m) { is = iso; m = mask; };
    if (g.W <= kFlatWords)
        fe_classify_flat_n(vol, g, 1, sink, blockIdx.x, flat_rows_per_wave(g.nx), s_bits[threadIdx.x >> 6]);
    else
        fe_classify_block_n(vol, g, 1, sink, blockIdx.x, keep_row);
}

/* ------------------------------------------------------------------ pass 1b + 2: counts */
/* The counts of a block's wavefronts (kind q of wavefront w in s_sums[w][q], 0 where it has no row) into the block's
 * tile: one atomic per block and kind, called by every thread. Atomics on one tile's line follow one another: with
 * one per row and kind, an extraction of 64x64x4097 noise at 0.98 takes 236 us, so 200 (211 with a look-back
 * scan, which needs no sums). */
template <int Kinds>
__device__ __forceinline__ void add_rows_sums(const uint64_t (*s_sums)[Kinds], uint64_t* __restrict__ tile_sums)
{
    __syncthreads();
    const int a = (int)threadIdx.x;
    if (a >= Kinds) return;
    uint64_t v = 0;
#pragma unroll
    for (int w = 0; w < kRowsPerBlock; ++w) v += s_sums[w][a];
    if (v) add_sum(&tile_sums[a], v);
}

__device__ __forceinline__ void fe_count_row(const uint64_t* __restrict__ mask, const Geom& g,
                                             RowCounts* __restrict__ counts, RowTrim* __restrict__ trims,
                                             const uint8_t* __restrict__ s_ntri, int64_t r, uint64_t* __restrict__ sum)
{
    const int lane = lane_id();
    const int64_t j = r % g.ny, k = r / g.ny;
    const bool has_y = j < g.ny - 1, has_z = k < g.nz - 1, cells = has_y && has_z;
    const int64_t W = g.W;
    const uint64_t* __restrict__ m0p = mask + r * W;
    const uint64_t* __restrict__ m1p = m0p + W;            // row (j+1, k)
    const uint64_t* __restrict__ m2p = m0p + g.ny * W;     // row (j, k+1)
    const uint64_t* __restrict__ m3p = m2p + W;            // row (j+1, k+1)

    uint32_t xc = 0, yc = 0, zc = 0, tc = 0;
    int64_t first = INT64_MAX, last = -1;
    for (int64_t w0 = 0; w0 < W; w0 += 64) {
        const int64_t w = w0 + lane;
        if (w >= W) break;
        const bool nxt = w + 1 < W;
        const uint64_t m0 = m0p[w], m0n = nxt ? m0p[w + 1] : 0;
        const uint64_t my = has_y ? m1p[w] : 0, myn = (has_y && nxt) ? m1p[w + 1] : 0;
        const uint64_t mz = has_z ? m2p[w] : 0, mzn = (has_z && nxt) ? m2p[w + 1] : 0;
        const uint64_t vb = low_bits(g.nx - 64 * w);          // vertices i < nx
        const uint64_t eb = low_bits(g.nx - 1 - 64 * w);      // x-edges / cells i < nx-1
        const uint64_t s0 = (m0 >> 1) | (m0n << 63);           // bit i -> vertex i+1
        const uint64_t xcut = (m0 ^ s0) & eb;
        const uint64_t ycut = has_y ? ((m0 ^ my) & vb) : 0;
        const uint64_t zcut = has_z ? ((m0 ^ mz) & vb) : 0;
        xc += __popcll(xcut);
        yc += __popcll(ycut);
        zc += __popcll(zcut);
        // isCutEdge tests i in [0, nx-2] only (FlyingEdgesAlgorithm.cpp:52-63)
        const uint64_t trim = (xcut | ycut | zcut) & eb;
        if (trim) {
            first = min(first, 64 * w + (int64_t)__builtin_ctzll(trim));
            last = max(last, 64 * w + 63 - (int64_t)__builtin_clzll(trim));
        }
        if (cells) {
            const uint64_t myz = m3p[w], myzn = nxt ? m3p[w + 1] : 0;
            const uint64_t sy = (my >> 1) | (myn << 63);
            const uint64_t sz = (mz >> 1) | (mzn << 63);
            const uint64_t syz = (myz >> 1) | (myzn << 63);
            const uint64_t all = m0 & s0 & sy & my & mz & sz & syz & myz;
            const uint64_t any = m0 | s0 | sy | my | mz | sz | syz | myz;
            uint64_t act = any & ~all & eb;
            while (act) {
                const int b = __builtin_ctzll(act);
                act &= act - 1;
                const int c = (int)((m0 >> b) & 1) | (int)((s0 >> b) & 1) << 1 | (int)((sy >> b) & 1) << 2 |
                              (int)((my >> b) & 1) << 3 | (int)((mz >> b) & 1) << 4 |
                              (int)((sz >> b) & 1) << 5 | (int)((syz >> b) & 1) << 6 |
                              (int)((myz >> b) & 1) << 7;
                tc += s_ntri[c];
            }
        }
    }
    xc = wave_sum_u32(xc);
    yc = wave_sum_u32(yc);
    zc = wave_sum_u32(zc);
    tc = wave_sum_u32(tc);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        first = min(first, (int64_t)__shfl_xor((long long)first, o));
        last = max(last, (int64_t)__shfl_xor((long long)last, o));
    }
    if (r < g.emit_lo) xc = yc = zc = tc = 0u;   // a slab's ghost rows, as in fe_count_rows_block
    if (r >= g.emit_hi) tc = 0u;
    if (lane < 4) sum[lane] = lane == 0 ? xc : (lane == 1 ? yc : (lane == 2 ? zc : tc));
    if (lane == 0) {
        counts[r] = RowCounts{xc, yc, zc, tc};
        trims[r] = RowTrim{last < 0 ? (uint32_t)g.nx : (uint32_t)first, last < 0 ? 0u : (uint32_t)(last + 1)};
    }
}

__global__ __launch_bounds__(256) void k_fe_count(const uint64_t* __restrict__ mask, Geom g,
                                                  RowCounts* __restrict__ counts,
                                                  RowTrim* __restrict__ trims,
                                                  uint64_t* __restrict__ sums, int shift)
{
    __shared__ uint8_t s_ntri[256];
    __shared__ uint64_t s_sums[kRowsPerBlock][4];
    for (int c = threadIdx.x; c < 256; c += blockDim.x) s_ntri[c] = (uint8_t)case_tri_count(kCaseEdges[c]);
    __syncthreads();

    const int wave = threadIdx.x >> 6;
    const int64_t r0 = (int64_t)blockIdx.x * kRowsPerBlock, r = r0 + wave;
    if (r < g.ny * g.nz)
        fe_count_row(mask, g, counts, trims, s_ntri, r, s_sums[wave]);
    else if (lane_id() < 4)
        s_sums[wave][lane_id()] = 0;
    add_rows_sums<4>(s_sums, sums + (r0 >> shift) * kTileSums);
}

/* ------------------------------------------------------------------ pass 3: scan */
/* What a scan writes beside the vertex and triangle offsets: for first-visit Marching Cubes the offsets
 * of the owned edges (owned -> moff), for its edge order those of the x, y and z counts (xyz, R each). */
struct ScanMore {
    const uint32_t* owned = nullptr;
    uint64_t* moff = nullptr;
    uint64_t* xyz = nullptr;
};

/* Tile `tile` of the scan: first the sums of the tiles before it (wavefront a takes every fourth kind),
 * then its own rows, kScanStep at a time, four per thread. The last tile's block writes totals: V, T,
 * and with xyz the totals of x, y and z after them; V and T also to host (pinned memory), if given.
 * Latency-bound: no tile waits for another one. 6 us at 512^3 and 12 us at 1024^3, against 17 and 28 with
 * look-back over tiles of 4096 rows (event pairs; pass 2, which adds up the sums, then took 2 and 15 us
 * more). Eight tile sums in flight per lane and the next rows requested a step ahead measured the same. A
 * step's sums are of type
 * S, 64 bits where 1024 rows of 5 nx triangles may pass 2^32. */
template <typename S = uint32_t>
__device__ __forceinline__ void fe_scan_tile(const RowCounts* __restrict__ counts, int64_t R,
                                             uint64_t* __restrict__ voff, uint64_t* __restrict__ toff,
                                             const uint64_t* __restrict__ sums, int shift, int64_t ntiles,
                                             uint64_t* __restrict__ totals, uint64_t* __restrict__ host,
                                             const ScanMore& more, int64_t tile)
{
    __shared__ uint64_t s_base[8];
    __shared__ S s_w[kTileSums][4];
    const int lane = lane_id(), wave = threadIdx.x >> 6;
    __syncthreads();   // the block's previous tile is done with the LDS
    for (int a = wave; a < kTileSums; a += 4) {
        uint64_t b = 0;
        if (a < 4 || more.owned)
            for (int64_t t = lane; t < tile; t += 64) b += sums[t * kTileSums + a];
        b = wave_sum_u64(b);
        if (lane == 0) s_base[a] = b;
    }
    __syncthreads();
    uint64_t base[kTileSums];
#pragma unroll
    for (int a = 0; a < kTileSums; ++a) base[a] = s_base[a];
    const int64_t r_lo = tile << shift, r_hi = min(R, (tile + 1) << shift);
    for (int64_t r0 = r_lo; r0 < r_hi; r0 += kScanStep) {
        const int64_t r = r0 + 4 * (int64_t)threadIdx.x;
        uint32_t v[4][kTileSums];
        S own[kTileSums] = {0, 0, 0, 0, 0};
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            RowCounts c{0u, 0u, 0u, 0u};
            if (r + u < r_hi) c = counts[r + u];
            v[u][0] = c.x;
            v[u][1] = c.y;
            v[u][2] = c.z;
            v[u][3] = c.t;
            v[u][4] = more.owned && r + u < r_hi ? more.owned[r + u] : 0u;
#pragma unroll
            for (int a = 0; a < kTileSums; ++a) own[a] += v[u][a];
        }
        uint64_t ex[kTileSums];
        S incl[kTileSums];
#pragma unroll
        for (int a = 0; a < kTileSums; ++a) {
            incl[a] = wave_incl_scan(own[a]);
            if (lane == 63) s_w[a][wave] = incl[a];
        }
        __syncthreads();
#pragma unroll
        for (int a = 0; a < kTileSums; ++a) {
            uint64_t before = 0, all = 0;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                before += q < wave ? s_w[a][q] : 0u;
                all += s_w[a][q];
            }
            ex[a] = base[a] + before + (incl[a] - own[a]);
            base[a] += all;
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if (r + u < r_hi) {
                voff[r + u] = ex[0] + ex[1] + ex[2];
                toff[r + u] = ex[3];
                if (more.owned) more.moff[r + u] = ex[4];
                if (more.xyz) {
                    more.xyz[r + u] = ex[0];
                    more.xyz[R + r + u] = ex[1];
                    more.xyz[2 * R + r + u] = ex[2];
                }
            }
#pragma unroll
            for (int a = 0; a < kTileSums; ++a) ex[a] += v[u][a];
        }
    }
    if (tile == ntiles - 1 && threadIdx.x == 0) {
        totals[0] = base[0] + base[1] + base[2];
        totals[1] = base[3];
        if (more.xyz)
            for (int a = 0; a < 3; ++a) totals[2 + a] = base[a];
        if (host) {
            host[0] = base[0] + base[1] + base[2];
            host[1] = base[3];
        }
    }
}

template <typename S>
__global__ __launch_bounds__(256) void k_fe_scan(const RowCounts* __restrict__ counts, int64_t R,
                                                 uint64_t* __restrict__ voff, uint64_t* __restrict__ toff,
                                                 const uint64_t* __restrict__ sums, int shift, int64_t ntiles,
                                                 uint64_t* __restrict__ totals, uint64_t* __restrict__ host,
                                                 ScanMore more)
{
    fe_scan_tile<S>(counts, R, voff, toff, sums, shift, ntiles, totals, host, more, blockIdx.x);
}

inline bool scan_is_wide(int64_t nx) { return nx > (int64_t(1) << 19); }   // 1024 rows of 5 nx triangles

/* ------------------------------------------------------------------ pass 4: emit */

struct EmitLds {
    uint64_t m[4][kSegWords + 1];         // sign-mask words of rows (j,k) (j+1,k) (j,k+1) (j+1,k+1)
    uint64_t cut[8][kSegWords + 1];       // cut words per (axis,row) combination, see combo_of_edge
    uint32_t pre[8][kSegWords + 1];       // exclusive popcount prefix of cut[q] within the segment
    uint16_t list[3 * 64 * kSegWords];    // compacted cut edges (axis << 14 | i) or active cells
};

/* Vertex id combination of a cube edge: which of the four grid rows holds the edge and along
 * which axis. 0-3: x-edges of rows (j,k) (j+1,k) (j,k+1) (j+1,k+1); 4-5: y-edges of rows (j,k)
 * (j,k+1); 6-7: z-edges of rows (j,k) (j+1,k). */
__device__ __forceinline__ int combo_of_edge(int e)
{
    // e:      0  1  2  3  4  5  6  7  8  9  10 11
    // combo:  0  4  1  4  2  5  3  5  6  6  7  7
    return (int)((0x776653524140ull >> (4 * e)) & 0xF);
}

/* Walks one row of the grid (j,k) segment by segment; holds the four sign-mask rows of the
 * cell row (j,k) in LDS. Each wavefront owns one RowWalker and its EmitLds slice. */
struct RowWalker {
    EmitLds& L;
    const uint64_t* __restrict__ mask;
    const Geom& g;
    int64_t rows[4];
    bool row_ok[4];
    int64_t s0w = 0;   // first word of the current segment
    int nw = 0;        // words in the current segment

    __device__ RowWalker(EmitLds& l, const uint64_t* __restrict__ m, const Geom& gg, int64_t r, bool has_y, bool has_z)
        : L(l), mask(m), g(gg)
    {
        rows[0] = r; rows[1] = r + 1; rows[2] = r + g.ny; rows[3] = r + g.ny + 1;
        row_ok[0] = true; row_ok[1] = has_y; row_ok[2] = has_z; row_ok[3] = has_y && has_z;
    }

    /* stage mask words [s0w, s0w + nw] (one extra word for the +1 neighbours) of the 4 rows */
    __device__ void stage(int64_t seg_w0)
    {
        const int lane = lane_id();
        s0w = seg_w0;
        nw = (int)min((int64_t)kSegWords, g.W - s0w);
        for (int t = lane; t < 4 * (kSegWords + 1); t += 64) {
            const int q = t / (kSegWords + 1), w = t % (kSegWords + 1);
            const int64_t gw = s0w + w;
            L.m[q][w] = (row_ok[q] && w <= nw && gw < g.W) ? mask[rows[q] * g.W + gw] : 0ull;
        }
        wave_sync();
    }

    /* Compacts the cut edges of grid row (j,k) in this segment into L.list: x-edges, then
     * y-edges, then z-edges, each by increasing i. Returns the count; per-axis starts/counts. */
    __device__ int compact_row_edges(bool has_y, bool has_z, int start[3], int cnt[3])
    {
        const int lane = lane_id();
        int n = 0;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            start[a] = n;
            if ((a == 1 && !has_y) || (a == 2 && !has_z)) {
                cnt[a] = 0;
                continue;
            }
            for (int w = 0; w < nw; ++w) {
                const int64_t gw = s0w + w;
                const uint64_t m0 = L.m[0][w];
                uint64_t bits;
                if (a == 0) {
                    const uint64_t sh = (m0 >> 1) | (L.m[0][w + 1] << 63);
                    bits = (m0 ^ sh) & low_bits(g.nx - 1 - 64 * gw);
                } else {
                    bits = (m0 ^ L.m[a][w]) & low_bits(g.nx - 64 * gw);
                }
                if ((bits >> lane) & 1ull)
                    L.list[n + __popcll(bits & __lanemask_lt())] = (uint16_t)((a << 14) | (w * 64 + lane));
                n += __popcll(bits);
            }
            cnt[a] = n - start[a];
        }
        wave_sync();
        return n;
    }

    /* Cut words of the 8 (axis,row) combinations and their popcount prefix for this segment,
     * then the compacted list of active cells (cells with at least one cut edge). */
    __device__ int prepare_cells()
    {
        const int lane = lane_id();
        if (lane <= nw) {
            const int w = lane;
            const int64_t gw = s0w + w;
            const uint64_t vb = low_bits(g.nx - 64 * gw), eb = low_bits(g.nx - 1 - 64 * gw);
            const bool has_next = w < nw;   // word w+1 staged (word nw is only read at bit 0)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint64_t m = L.m[q][w];
                const uint64_t nb = has_next ? L.m[q][w + 1] : 0ull;
                L.cut[q][w] = (m ^ ((m >> 1) | (nb << 63))) & eb;
            }
            L.cut[4][w] = (L.m[0][w] ^ L.m[1][w]) & vb;
            L.cut[5][w] = (L.m[2][w] ^ L.m[3][w]) & vb;
            L.cut[6][w] = (L.m[0][w] ^ L.m[2][w]) & vb;
            L.cut[7][w] = (L.m[1][w] ^ L.m[3][w]) & vb;
        }
        wave_sync();
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const uint32_t pc = lane <= nw ? (uint32_t)__popcll(L.cut[q][lane]) : 0u;
            const uint32_t inc = wave_incl_scan_u32(pc);
            if (lane <= nw) L.pre[q][lane] = inc - pc;
        }
        int na = 0;
        for (int w = 0; w < nw; ++w) {
            const int64_t gw = s0w + w;
            const uint64_t eb = low_bits(g.nx - 1 - 64 * gw);
            const uint64_t a0 = L.m[0][w], a1 = L.m[1][w], a2 = L.m[2][w], a3 = L.m[3][w];
            const uint64_t b0 = (a0 >> 1) | (L.m[0][w + 1] << 63);
            const uint64_t b1 = (a1 >> 1) | (L.m[1][w + 1] << 63);
            const uint64_t b2 = (a2 >> 1) | (L.m[2][w + 1] << 63);
            const uint64_t b3 = (a3 >> 1) | (L.m[3][w + 1] << 63);
            const uint64_t all = a0 & a1 & a2 & a3 & b0 & b1 & b2 & b3;
            const uint64_t any = a0 | a1 | a2 | a3 | b0 | b1 | b2 | b3;
            const uint64_t act = any & ~all & eb;
            if ((act >> lane) & 1ull) L.list[na + __popcll(act & __lanemask_lt())] = (uint16_t)(w * 64 + lane);
            na += __popcll(act);
        }
        wave_sync();
        return na;
    }

    /* marching-cubes case of the cell at local index li of this segment */
    __device__ int cell_case(int li) const
    {
        const int w = li >> 6, b = li & 63;
        auto bit = [&](int q, int dx) -> int {
            const int p = b + dx;
            return (int)((L.m[q][w + (p >> 6)] >> (p & 63)) & 1ull);
        };
        return bit(0, 0) | bit(0, 1) << 1 | bit(1, 1) << 2 | bit(1, 0) << 3 | bit(2, 0) << 4 |
               bit(2, 1) << 5 | bit(3, 1) << 6 | bit(3, 0) << 7;
    }

    /* Flying Edges vertex id of cube edge `e` of the cell at local index li: the row offset plus
     * axis-block offset (cbase) plus the rank of the edge among the row's cut edges. */
    __device__ uint64_t fe_vertex_id(const uint64_t cbase[8], int e, int li) const
    {
        const int q = combo_of_edge(e);
        const int p = li + edge_dx(e);
        const int w = p >> 6, b = p & 63;
        const uint64_t below = L.cut[q][w] & ((1ull << b) - 1ull);
        return cbase[q] + L.pre[q][w] + (uint64_t)__popcll(below);
    }

    __device__ void advance_bases(uint64_t cbase[8]) const
    {
#pragma unroll
        for (int q = 0; q < 8; ++q) cbase[q] += L.pre[q][nw - 1] + __popcll(L.cut[q][nw - 1]);
    }
};

/* Row-offset plus axis-block bases of the 8 combinations for cell row r. */
__device__ __forceinline__ void combo_bases(const RowCounts* __restrict__ counts, const uint64_t* __restrict__ voff,
                                            const int64_t rows[4], uint64_t cbase[8])
{
    RowCounts cq[4];
    uint64_t pq[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        cq[q] = counts[rows[q]];
        pq[q] = voff[rows[q]];
    }
    cbase[0] = pq[0]; cbase[1] = pq[1]; cbase[2] = pq[2]; cbase[3] = pq[3];
    cbase[4] = pq[0] + cq[0].x;
    cbase[5] = pq[2] + cq[2].x;
    cbase[6] = pq[0] + cq[0].x + cq[0].y;
    cbase[7] = pq[1] + cq[1].x + cq[1].y;
}

template <typename Index>
__global__ __launch_bounds__(256) void k_fe_emit(const float* __restrict__ vol,
                                                 const uint64_t* __restrict__ mask, Geom g, float iso,
                                                 const RowCounts* __restrict__ counts,
                                                 const uint64_t* __restrict__ voff,
                                                 const uint64_t* __restrict__ toff,
                                                 float* __restrict__ pts, float* __restrict__ nrm,
                                                 Index* __restrict__ tris, uint64_t vbias = 0,
                                                 const uint64_t* __restrict__ need = nullptr, uint64_t cap_v = 0,
                                                 uint64_t cap_t = 0)
{
    if (need && !output_fits<Index>(need, cap_v, cap_t)) return;   // as k_fe_emit_rows
    __shared__ EmitLds lds_all[kRowsPerBlock];
    const int lane = lane_id();
    const int wave = threadIdx.x >> 6;
    const int64_t r = (int64_t)blockIdx.x * kRowsPerBlock + wave;
    if (r >= g.ny * g.nz || r < g.emit_lo || r >= g.emit_hi) return;
    const RowCounts c0 = counts[r];
    if (c0.x + c0.y + c0.z == 0 && c0.t == 0) return;
    const int64_t j = r % g.ny, k = r / g.ny;
    const bool has_y = j < g.ny - 1, has_z = k < g.nz - 1, cells = has_y && has_z && c0.t;
    RowWalker rw(lds_all[wave], mask, g, r, has_y, has_z);
    EmitLds& L = lds_all[wave];

    const uint64_t p0 = voff[r];
    uint64_t vb_run[3] = {p0, p0 + c0.x, p0 + c0.x + c0.y};
    uint64_t cbase[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    uint64_t tri_run = 0;
    if (cells) {
        combo_bases(counts, voff, rw.rows, cbase);
        tri_run = toff[r];
    }

    for (int64_t s0w = 0; s0w < g.W; s0w += kSegWords) {
        rw.stage(s0w);
        // ---- vertices of grid row r, already in output order
        int start[3], cnt[3];
        const int n = rw.compact_row_edges(has_y, has_z, start, cnt);
        for (int e = lane; e < n; e += 64) {
            const uint32_t ent = L.list[e];
            const int a = (int)(ent >> 14);
            const int64_t i = s0w * 64 + (int64_t)(ent & 0x3FFF);
            const uint64_t vid = vb_run[a] + (uint64_t)(e - start[a]);
            float A[3], B[3], p[3], nn[3];
            fe_edge_corners(g, a, i, j, k, A, B);
            edge_point(vol, g, iso, a, i, j, k, A, B, p, nn);
            pts[3 * vid + 0] = p[0];
            pts[3 * vid + 1] = p[1];
            pts[3 * vid + 2] = p[2];
            nrm[3 * vid + 0] = nn[0];
            nrm[3 * vid + 1] = nn[1];
            nrm[3 * vid + 2] = nn[2];
        }
        wave_sync();
        vb_run[0] += cnt[0];
        vb_run[1] += cnt[1];
        vb_run[2] += cnt[2];

        // ---- triangles of cell row (j,k)
        if (cells) {
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
                        const uint64_t a = rw.fe_vertex_id(cbase, case_edge(packed, 3 * t + 0), li);
                        const uint64_t b = rw.fe_vertex_id(cbase, case_edge(packed, 3 * t + 1), li);
                        const uint64_t c = rw.fe_vertex_id(cbase, case_edge(packed, 3 * t + 2), li);
                        store_tri<Index>(tris, slot0 + t, a - vbias, b - vbias, c - vbias);
                    }
                }
                tri_run += __shfl(incl, 63);
            }
            rw.advance_bases(cbase);
        }
        wave_sync();
    }
}

}  // namespace miso

#endif
