// Table gradient through binned records: the hash-grid backward for batches
// large enough to stream.
//
// A float atomic straight into the table costs one memory request per 64-byte
// block a wave instruction touches, about 21 G requests/s whatever their width,
// and the fine hashed levels share no block between samples: 4.5 requests per
// sample and level (3-D), two thirds of a training step.  Here no sample's
// contribution goes to memory as an atomic:
//
//   k_scatter_emit   one thread per sample; per level, a record for each of the
//                    2^(D-1) x-neighbour corner pairs: the pair's place in its
//                    bin, x's fraction and the pair's weight times dL/dfeature.
//                    A bin is a part of the level's table whose gradient fits
//                    in 64 KiB of LDS.  The workgroup sorts its records by bin
//                    in LDS, reserves their places in the bins' lists with one
//                    atomic per bin, and writes them as contiguous runs.
//   k_scatter_apply  a workgroup takes one bin (or a share of a long list), adds
//                    its records up in LDS and then the touched entries to the
//                    table's gradient, one request per 64-byte block.
//
// Both stream: 16 bytes (two features) or 24 (four) written and read per corner
// pair.  The batch is taken in chunks so that the record buffer stays bounded.
// Scatter per step, atomics into the table (with the coarse levels summed per
// block in LDS) -> records: 256^3 cone, 10.7 M samples x 16 levels 19.0 -> 6.0 ms;
// 4-D, 2^21 entries 45.0 -> 8.6 ms; four QuadCubes grids 22.8 -> 6.5 ms; a million
// random points 3.48 -> 0.6 ms.  The emission is bound by its writes (3.0-3.3 TB/s),
// the sums by their LDS atomics and the records' reads (3.5 TB/s) about equally.
//
// The sums are float64 because gfx950 performs a wave's float64 LDS adds in about
// 28 cycles and its float32 ones in about 195 (hash-drawn addresses; uint32 11):
// with float32 sums the 256^3 scatter took 19.3 ms.
// A bin's list holds a multiple of its even share; records past it (a batch
// whose samples crowd into few bins) are added straight to the gradient, so
// every distribution is correct.
//
// Folding.  Where the grid's last dimension reads the time t, which is one value
// for all rays of a batch, the two corners along t get (1 - f_t) and f_t times
// the same sum over the samples: the records are formed over the other
// dimensions only (half as many), summed, and each sum is added to both entries.
#include <algorithm>
#include <type_traits>

#include "sources.hpp"

namespace nect {

constexpr int kEmitThreads = 512;
constexpr int kApplyThreads = 512;
constexpr int kBinLog2Floats = 13;     // a bin's gradient in float64: 64 KiB of LDS, two workgroups per CU
constexpr int kBinFloats = 1 << kBinLog2Floats;
constexpr int kMaxBins = 4096;         // per level
constexpr int kGroupBins = 2048;       // most per group of levels: the emission's counters in LDS
constexpr int kFillBlocks = 768;       // emission workgroups that fill the device
constexpr int64_t kWholeListBytes = (int64_t)256 << 20;
constexpr int kPartRecords = 16384;
constexpr int kCounterLead = 64;       // counters per chunk are rounded up to this many

// Record word: place of the pair's first entry in its bin (13 bits), how the
// second follows from it (5), the bin (14).
constexpr int kPlaceBits = 13, kKindBits = 5;
constexpr uint32_t kKindNext = 0;      // second = first + 1; k = 1..13: first ^ (2^k - 1)
constexpr uint32_t kKindAlone = 31;    // no second entry (it lies in another bin)

// The samples of the rays' tiles, under a column map (see place_sample).
template <int D>
struct RayColsSource {
    const NectRay *rays;
    const int32_t *tile_offsets;
    const int32_t *tile_ray;
    const int32_t *n_tiles;
    int64_t max_tiles;
    float t;
    uint32_t cmap;
    // slots [s0, s1) of chunk c of n_chunks
    __device__ __forceinline__ void bounds(int c, int n_chunks, int64_t &s0, int64_t &s1) const {
        const int64_t n = min((int64_t)n_tiles[0], max_tiles);
        s0 = n * c / n_chunks * kTile;
        s1 = n * (c + 1) / n_chunks * kTile;
    }
    __device__ __forceinline__ bool get(int64_t slot, float (&p)[D]) const {
        const int64_t tile = slot / kTile;
        const int r = tile_ray[tile];
        const int i = (int)(tile - tile_offsets[r]) * kTile + (int)(slot % kTile);
        const NectRay d = rays[r];
        float q[3];
        const bool ok = ray_sample(d, i, q);
        place_sample<D>(cmap, q, t, p);
        return ok;
    }
};

template <int D>
struct PointRowsSource {
    const float *x;
    int64_t n;
    int64_t stride;
    __device__ __forceinline__ void bounds(int c, int n_chunks, int64_t &s0, int64_t &s1) const {
        const int64_t t = (n + kTile - 1) / kTile;
        s0 = t * c / n_chunks * kTile;
        s1 = min(n, t * (c + 1) / n_chunks * kTile);
    }
    __device__ __forceinline__ bool get(int64_t slot, float (&p)[D]) const {
        const float *r = x + slot * stride;
#pragma unroll
        for (int d = 0; d < D; ++d) p[d] = r[d];
        return true;
    }
};

// Per level: 2^bins bins of `entries` table entries each; entry i belongs to bin
// (i >> granule) mod 2^bins.  A hashed level's bins are contiguous (its entries
// are spread evenly anyway, and a pair almost never straddles two; but see
// plan_bins for a caller's points); a dense level's interleave in runs of
// 2^granule entries, so that a batch confined to a part of the volume or to one
// time still uses every bin.
struct BinPlan {
    int32_t n_chunks;
    uint32_t hashed;                  // bit l: level l is hashed
    uint32_t size[NECT_MAX_LEVELS];   // entries the bins cover: the level's, or (folded, dense) one t's
    int32_t n_counters;               // per chunk
    int32_t n_bins;                   // of all levels
    int32_t n_groups;                 // of levels whose counters fit the emission's LDS
    uint8_t group0[NECT_MAX_LEVELS + 1];
    uint8_t log2_bins[NECT_MAX_LEVELS];
    uint8_t granule[NECT_MAX_LEVELS];
    uint8_t log2_splits[NECT_MAX_LEVELS];
    int32_t entries[NECT_MAX_LEVELS];
    int32_t n_lists;                  // lists per bin: the workgroups of one XCD append to one
    uint32_t cap[NECT_MAX_LEVELS];    // records per list
    int32_t bin0[NECT_MAX_LEVELS];    // counter of the level's first bin
    int32_t task0[NECT_MAX_LEVELS + 1];
    int64_t rec0[NECT_MAX_LEVELS];    // first record of the level's first bin
    float t;                          // folded: the last coordinate
};

// Adds v to an entry of a level (bins' numbering): itself, or (folded) the two
// entries at t's corners.
template <bool FOLD>
struct LevelAdd {
    float *lvl;
    uint32_t size;
    bool hashed;
    uint32_t at[2];   // FOLD: what the corners along t contribute to the entry
    float f;          // FOLD: t's fraction
    __device__ __forceinline__ uint32_t entry(uint32_t e, int k) const {
        if constexpr (!FOLD) return e;
        return hashed ? e ^ at[k] : (e + at[k]) % size;
    }
    template <int F>
    __device__ __forceinline__ void add(uint32_t e, int j, double v) const {
#pragma unroll
        for (int k = 0; k < (FOLD ? 2 : 1); ++k) {
            const float x = (float)(FOLD ? v * (double)(k ? f : 1.0f - f) : v);
            if (x != 0.0f) unsafeAtomicAdd(lvl + (size_t)entry(e, k) * F + j, x);
        }
    }
};

// FOLD: D spatial dimensions of a D + 1-dimensional grid.
template <int D, bool FOLD>
__device__ __forceinline__ LevelAdd<FOLD> level_add(const NectGridDesc &g, const BinPlan &P, int l, float *grad) {
    LevelAdd<FOLD> a;
    a.lvl = grad + (size_t)g.offset[l] * g.n_features;
    a.size = g.level_size[l];
    a.hashed = (P.hashed >> l) & 1u;
    if constexpr (FOLD) {
        uint32_t c;
        grid_pos(g.scale[l], P.t, c, a.f);
        uint32_t mul = 1;
#pragma unroll
        for (int d = 0; d < D; ++d) mul *= g.resolution[l];
        if (a.hashed) mul = hash_prime(D) & (a.size - 1);
        a.at[0] = c * mul;
        a.at[1] = (c + 1) * mul;
        if (a.hashed) {
            a.at[0] &= a.size - 1;
            a.at[1] &= a.size - 1;
        }
    }
    return a;
}

// Index constants of a level's bins' numbering (folded: over the D spatial dimensions).
template <int D, bool FOLD>
__device__ __forceinline__ LevelIndex<D> bin_index(const NectGridDesc &g, const BinPlan &P, int l) {
    if constexpr (!FOLD) return level_index<D>(g.resolution[l], g.level_size[l]);
    LevelIndex<D> li;
    li.hashed = (P.hashed >> l) & 1u;
    uint32_t m = 1;
#pragma unroll
    for (int d = 0; d < D; ++d) {
        li.mul[d] = li.hashed ? hash_prime(d) : m;
        m *= g.resolution[l];
    }
    // a dense level's spatial index is taken as it is (P.size covers the upper corners of the far faces)
    li.size = li.hashed ? g.level_size[l] : 0u;
    li.pow2 = true;
    return li;
}

__device__ __forceinline__ uint32_t bin_of(uint32_t entry, int granule, int log2_bins) {
    return (entry >> granule) & ((1u << log2_bins) - 1u);
}
__device__ __forceinline__ uint32_t place_of(uint32_t entry, int granule, int log2_bins) {
    return ((entry >> (granule + log2_bins)) << granule) | (entry & ((1u << granule) - 1u));
}
__device__ __forceinline__ uint32_t entry_of(uint32_t place, uint32_t bin, int granule, int log2_bins) {
    return ((((place >> granule) << log2_bins) | bin) << granule) | (place & ((1u << granule) - 1u));
}
__device__ __forceinline__ uint32_t second_place(uint32_t place, uint32_t kind) {
    return kind == kKindNext ? place + 1u : place ^ ((1u << kind) - 1u);
}

template <int F>
struct BinRecord {
    uint32_t word;
    float fx;
    float v[F];  // weight of the pair's other coordinates times dL/dfeature
};

__global__ __launch_bounds__(256) void k_scatter_zero(uint32_t *counts, int n) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) counts[i] = 0u;
}

// Up to N values of a dL/dfeature row from column c (past `cols`: zero), in
// pieces of P elements of type T read at once.
template <typename T, int P, int N>
__device__ __forceinline__ void load_pieces(const T *row, float sc, int c, int cols, float (&b)[N]) {
    struct __attribute__((aligned(P * sizeof(T)))) Piece {
        T e[P];
    };
#pragma unroll
    for (int u = 0; u < N; u += P) {
        if (c + u + P <= cols) {
            const Piece q = *reinterpret_cast<const Piece *>(row + c + u);
#pragma unroll
            for (int k = 0; k < P; ++k) b[u + k] = to_f32(q.e[k]) * sc;
        } else {
#pragma unroll
            for (int k = 0; k < P; ++k) b[u + k] = c + u + k < cols ? to_f32(row[c + u + k]) * sc : 0.0f;
        }
    }
}

// `align`: bytes the rows and column c are aligned to (4 or less: one element at a time).
template <typename T, int N>
__device__ __forceinline__ void load_row(const DoutView &d, float sc, int align, int64_t row, int c, int cols,
                                         float (&b)[N]) {
    const T *r = static_cast<const T *>(d.p) + row * d.stride;
    if (align >= 16) load_pieces<T, 16 / sizeof(T)>(r, sc, c, cols, b);
    else if (align >= 8) load_pieces<T, 8 / sizeof(T)>(r, sc, c, cols, b);
    else load_pieces<T, 1>(r, sc, c, cols, b);
}

template <int N>
__device__ __forceinline__ void load_dout(const DoutView &d, float sc, int align, int64_t row, int c, int cols,
                                          float (&b)[N]) {
    if (d.dtype == NECT_F32) load_row<float>(d, sc, align, row, c, cols, b);
    else if (d.dtype == NECT_F16) load_row<_Float16>(d, sc, align, row, c, cols, b);
    else load_row<bf16_t>(d, sc, align, row, c, cols, b);
}

// Runs of samples of one ray in one cell, within rows of 16 lanes: whether this
// lane starts one, and its last lane.
template <int D>
__device__ __forceinline__ bool run_head(const uint32_t (&c)[D], bool live, int lane) {
    // every lane takes part in the row shifts: no short-circuit around them
    uint32_t diff = (uint32_t)row_up<1>((int)live) ^ (uint32_t)live;
#pragma unroll
    for (int d = 0; d < D; ++d) diff |= (uint32_t)row_up<1>((int)c[d]) ^ c[d];
    return ((lane & 15) == 0) | (diff != 0u);
}
__device__ __forceinline__ int run_end(bool head, int lane) {
    const uint64_t heads = __ballot(head);
    const uint64_t after = lane == kWave - 1 ? 0ull : heads & (~0ull << (lane + 1));
    return after ? __builtin_ctzll(after) - 1 : kWave - 1;
}

// One step of the run sums: lane i adds the values of lane i + OFF of its row of
// 16 lanes (a run never leaves its row) when `add`.
template <int OFF, int K, int F>
__device__ __forceinline__ void run_step(float (&v)[K][F], bool add) {
#pragma unroll
    for (int k = 0; k < K; ++k)
#pragma unroll
        for (int f = 0; f < F; ++f) {
            const float t = row_down<OFF>(v[k][f]);
            v[k][f] += add ? t : 0.0f;
        }
}

template <int F>
__device__ __forceinline__ void store_record(uint32_t *recs, int64_t i, const BinRecord<F> &r) {
    constexpr int W = (int)(sizeof(BinRecord<F>) / 4);
    if constexpr (F == 2) {
        *reinterpret_cast<uint4 *>(recs + i * W) = __builtin_bit_cast(uint4, r);
    } else {
        const uint2 *w = reinterpret_cast<const uint2 *>(&r);
        uint2 *d = reinterpret_cast<uint2 *>(recs + i * W);
#pragma unroll
        for (int k = 0; k < W / 2; ++k) d[k] = w[k];
    }
}

// A record whose bin's list is full: straight to the gradient.
template <int F, bool FOLD>
__device__ __noinline__ void add_record(const LevelAdd<FOLD> to, const BinRecord<F> r, int gr, int lb) {
    const uint32_t bin = r.word >> (kPlaceBits + kKindBits);
    const uint32_t a = r.word & ((1u << kPlaceBits) - 1u);
    const uint32_t kind = (r.word >> kPlaceBits) & ((1u << kKindBits) - 1u);
    const uint32_t e0 = entry_of(a, bin, gr, lb);
#pragma unroll
    for (int k = 0; k < F; ++k) to.template add<F>(e0, k, (double)((1.0f - r.fx) * r.v[k]));
    if (kind != kKindAlone) {
        const uint32_t e1 = entry_of(second_place(a, kind), bin, gr, lb);
#pragma unroll
        for (int k = 0; k < F; ++k) to.template add<F>(e1, k, (double)(r.fx * r.v[k]));
    }
}

// Emission (bound by its record writes).  Writing each record where its atomic
// says, unsorted, cost the 4-D batch 7.9 ms against 6.5 for eight levels; one
// list per bin instead of one per XCD 2.34 against 1.93 ms (3-D).  Runs of
// samples in one cell are summed first where they halve the records: without,
// the 256^3 scatter takes 7.2 ms.
// A workgroup takes 512 samples and a group of levels whose bins'
// counters fit in LDS (host: P.group0).  Pass 1 counts every level's records per
// bin; one round of atomics then reserves the places of all of them; pass 2 forms
// the records.
// The records of a level are sorted by bin in LDS and written as runs.
template <int D, int F, bool FOLD, typename Src>
__global__ __launch_bounds__(kEmitThreads, D <= 3 && F == 2 ? 6 : (D == 4 && F == 4 ? 2 : 4)) void k_scatter_emit(NectGridDesc g, BinPlan P, Src src, int chunk,
                                                               DoutView dv, int align, uint32_t *__restrict__ counts,
                                                               uint32_t *__restrict__ recs, float *__restrict__ grad,
                                                               int group_bins) {
    constexpr int Q = 1 << (D - 1), LB = 16 / F;
    static_assert(sizeof(BinRecord<F>) == 8 + 4 * F, "records are packed");
    extern __shared__ __align__(16) char smem_raw[];
    BinRecord<F> *stage = reinterpret_cast<BinRecord<F> *>(smem_raw);
    uint32_t *cursor = reinterpret_cast<uint32_t *>(stage + kEmitThreads * Q);
    uint32_t *delta = cursor + group_bins;
    __shared__ uint32_t wave_total[kEmitThreads / kWave];
    __shared__ uint32_t level_first[NECT_MAX_LEVELS + 1];
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    int64_t s0, s1;
    src.bounds(chunk, P.n_chunks, s0, s1);
    // workgroup -> (samples, group of levels): the groups of one block of samples follow one another on one XCD, whose
    // L2 then holds their dL/dfeature rows
    const int xcd = (int)(blockIdx.x % kXcds), turn = (int)(blockIdx.x / kXcds);
    const int grp = turn % P.n_groups;
    const int64_t first = s0 + ((int64_t)(turn / P.n_groups) * kXcds + xcd) * kEmitThreads;
    if (first >= s1) return;
    const int64_t slot = first + tid;
    float p[D];
#pragma unroll
    for (int d = 0; d < D; ++d) p[d] = 0.0f;
    const bool live = slot < s1 && src.get(slot, p);
    if (__syncthreads_or(live) == 0) return;
    // consecutive workgroups run on the XCDs in turn, so a list is written through one L2 and its lines fill up
    // there; with one list for all, neighbouring runs of a line came from different L2s as partial writes
    const int list = xcd % P.n_lists;
    counts += ((int64_t)chunk * P.n_lists + list) * P.n_counters;
    const float gsc = dv.scale ? dv.scale[0] : 1.0f;
    const int l0 = P.group0[grp], l1 = P.group0[grp + 1];   // at most LB levels
    const int b0 = P.bin0[l0], nb_all = (l1 < g.n_levels ? P.bin0[l1] : P.n_bins) - b0;
    // the group's dL/dfeature, read once (a second pass over the rows would fetch them again: the records written
    // in between have replaced them in L2), and which levels this lane has a record of
    float buf[16];
    uint32_t emits = 0;
    if (live) {
        const int at = l0 * F * (dv.dtype == NECT_F32 ? 4 : 2);
        load_dout(dv, gsc, at % 16 == 0 ? align : min(align, at % 8 == 0 ? 8 : 4), slot, l0 * F, l1 * F, buf);
#pragma unroll
        for (int u = 0; u < LB; ++u) {
            bool any = false;
#pragma unroll
            for (int f = 0; f < F; ++f) any |= buf[u * F + f] != 0.0f;
            emits |= any ? 1u << u : 0u;
        }
    } else {
#pragma unroll
        for (int u = 0; u < 16; ++u) buf[u] = 0.0f;
    }
    uint32_t merged = 0;   // levels whose runs this wave sums
    bool runs = true;
    for (int b = tid; b < nb_all; b += kEmitThreads) cursor[b] = 0u;
    lds_barrier();
    // pass 1: records per bin
    for (int l = l0; l < l1; ++l) {
        const bool any = (emits >> (l - l0)) & 1u;
        if (__ballot(any) == 0) continue;
        const LevelIndex<D> li = bin_index<D, FOLD>(g, P, l);
        const float scale = g.scale[l];
        const int gr = P.granule[l], lb = P.log2_bins[l];
        uint32_t *cnt = cursor + (P.bin0[l] - b0);
        uint32_t c[D], ct[D], e[Q];
        float f[D];
#pragma unroll
        for (int d = 0; d < D; ++d) grid_pos(scale, p[d], c[d], f[d]);
        corner_terms<D>(li, c, ct);
        corner_entries<D>(li, ct, 0, e);
        if (runs) {
            // runs are summed while half the live lanes or fewer start one; the next level's cells are
            // smaller, so a wave that is past that does not look again
            const bool head = run_head<D>(c, live, lane);
            runs = 2 * __popcll(__ballot(head && live)) <= __popcll(__ballot(live));
            if (runs) {
                merged |= 1u << (l - l0);
                if (head && live) {
#pragma unroll
                    for (int q = 0; q < Q; ++q) atomicAdd(&cnt[bin_of(e[q], gr, lb)], 1u);
                    corner_entries<D>(li, ct, 1, e);
#pragma unroll
                    for (int q = 0; q < Q; ++q) atomicAdd(&cnt[bin_of(e[q], gr, lb)], 1u);
                }
                continue;
            }
        }
        if (any) {
#pragma unroll
            for (int q = 0; q < Q; ++q) atomicAdd(&cnt[bin_of(e[q], gr, lb)], 1u);
        }
    }
    lds_barrier();
    // places in the bins' lists, and the exclusive scan of the counts over the group
    const int per = (nb_all + kEmitThreads - 1) / kEmitThreads;
    const int bb = min(nb_all, tid * per), be = min(nb_all, bb + per);
    uint32_t sum = 0;
    for (int b = bb; b < be; ++b) {
        const uint32_t h = cursor[b];
        delta[b] = h ? atomicAdd(&counts[b0 + b], h) : 0u;
        cursor[b] = sum;
        sum += h;
    }
    uint32_t inc = sum;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
        const uint32_t v = __shfl_up(inc, off, kWave);
        if (lane >= off) inc += v;
    }
    if (lane == kWave - 1) wave_total[wave] = inc;
    lds_barrier();
    uint32_t before = inc - sum, total = 0;
#pragma unroll
    for (int w = 0; w < kEmitThreads / kWave; ++w) {
        const uint32_t v = wave_total[w];
        if (w < wave) before += v;
        total += v;
    }
    for (int b = bb; b < be; ++b) {
        const uint32_t st = cursor[b] + before;
        cursor[b] = st;
        delta[b] -= st;
    }
    if (tid == 0) level_first[l1 - l0] = total;
    lds_barrier();
    if (tid < l1 - l0) level_first[tid] = cursor[P.bin0[l0 + tid] - b0];
    lds_barrier();
    // pass 2: the records
    for (int l = l0; l < l1; ++l) {
        float gv[F];
#pragma unroll
        for (int f = 0; f < F; ++f) gv[f] = buf[f];
#pragma unroll
        for (int u = 0; u + F < 16; ++u) buf[u] = buf[u + F];
        const float scale = g.scale[l];
        const int gr = P.granule[l], lb = P.log2_bins[l];
        const uint32_t cap = P.cap[l];
        const int64_t rec0 = P.rec0[l] + ((int64_t)list << lb) * cap;
        const LevelAdd<FOLD> to = level_add<D, FOLD>(g, P, l, grad);
        uint32_t *cur = cursor + (P.bin0[l] - b0);
        const uint32_t lf = level_first[l - l0];
        auto put = [&](BinRecord<F> r, uint32_t place, uint32_t kind, uint32_t bin) {
            r.word = place | (kind << kPlaceBits) | (bin << (kPlaceBits + kKindBits));
            stage[atomicAdd(&cur[bin], 1u) - lf] = r;
        };
        const bool any = (emits >> (l - l0)) & 1u;
        if (__ballot(any) != 0) {
            const LevelIndex<D> li = bin_index<D, FOLD>(g, P, l);
            uint32_t c[D], ct[D];
            float fr[D];
#pragma unroll
            for (int d = 0; d < D; ++d) grid_pos(scale, p[d], c[d], fr[d]);
            corner_terms<D>(li, c, ct);
            if ((merged >> (l - l0)) & 1u) {
                const bool head = run_head<D>(c, live, lane);
                const int end = run_end(head, lane);
#pragma unroll 1
                for (int cx = 0; cx < 2; ++cx) {
                    uint32_t e[Q];
                    corner_entries<D>(li, ct, cx, e);
                    float v[Q][F];
#pragma unroll
                    for (int q = 0; q < Q; ++q) {
                        const float w = corner_weight<D>(fr, cx | (q << 1));
#pragma unroll
                        for (int f = 0; f < F; ++f) v[q][f] = live ? w * gv[f] : 0.0f;
                    }
                    run_step<1>(v, lane + 1 <= end);
                    run_step<2>(v, lane + 2 <= end);
                    run_step<4>(v, lane + 4 <= end);
                    run_step<8>(v, lane + 8 <= end);
                    if (head && live) {
#pragma unroll
                        for (int q = 0; q < Q; ++q) {
                            BinRecord<F> r;
                            r.fx = 0.0f;
#pragma unroll
                            for (int f = 0; f < F; ++f) r.v[f] = v[q][f];
                            put(r, place_of(e[q], gr, lb), kKindAlone, bin_of(e[q], gr, lb));
                        }
                    }
                }
            } else if (any) {
                uint32_t i0[Q], i1[Q];
                corner_entries<D>(li, ct, 0, i0);
                corner_entries<D>(li, ct, 1, i1);
#pragma unroll
                for (int q = 0; q < Q; ++q) {
                    // the weight of the pair: the product over the other coordinates, then dL/dfeature
                    float w = 1.0f;
#pragma unroll
                    for (int d = 1; d < D; ++d) w = w * (((q >> (d - 1)) & 1) ? fr[d] : 1.0f - fr[d]);
                    BinRecord<F> r;
                    r.fx = fr[0];
#pragma unroll
                    for (int k = 0; k < F; ++k) r.v[k] = w * gv[k];
                    const uint32_t bin = bin_of(i0[q], gr, lb), a = place_of(i0[q], gr, lb);
                    uint32_t kind = kKindAlone;
                    if (bin_of(i1[q], gr, lb) == bin) {
                        const uint32_t b = place_of(i1[q], gr, lb), x = a ^ b;
                        if (b == a + 1u) kind = kKindNext;
                        else if (x != 0u && (x & (x + 1u)) == 0u) kind = (uint32_t)__popc(x);
                    }
                    if (kind == kKindAlone) {
                        // the second entry lies in another bin: straight to the gradient
#pragma unroll
                        for (int k = 0; k < F; ++k) to.template add<F>(i1[q], k, (double)(r.fx * r.v[k]));
                    }
                    put(r, a, kind, bin);
                }
            }
        }
        lds_barrier();
        const uint32_t total = level_first[l - l0 + 1] - lf;
        const uint32_t *dl = delta + (P.bin0[l] - b0);
        for (uint32_t i = tid; i < total; i += kEmitThreads) {
            const BinRecord<F> r = stage[i];
            const uint32_t bin = r.word >> (kPlaceBits + kKindBits);
            const uint32_t pos = i + lf + dl[bin];
            if (pos < cap) store_record<F>(recs, rec0 + (int64_t)bin * cap + pos, r);
            else add_record<F, FOLD>(to, r, gr, lb);
        }
        lds_barrier();
    }
}

// Adds a wave's records to the bin's sums (the 16^3 level of the 256^3 batch:
// 3.19 ms with one LDS add per record, 0.31 with the runs summed here and there).  LDS atomics on one address take their
// turns, and neighbouring records of a coarse or middle level often share their
// entries (neighbouring samples' records follow one another in a list): where a
// quarter of the lanes repeat their left neighbour's place, the repeats within a
// row of 16 lanes are summed first and only each run's first lane adds.
template <int F>
__device__ __forceinline__ void apply_records(double *acc, const BinRecord<F> &r, bool on, int lane) {
    constexpr uint32_t kWhere = (1u << (kPlaceBits + kKindBits)) - 1u;
    const uint32_t key = on ? r.word & kWhere : ~0u;
    const uint32_t a = r.word & ((1u << kPlaceBits) - 1u);
    const uint32_t kind = (r.word >> kPlaceBits) & ((1u << kKindBits) - 1u);
    float v[2][F];
#pragma unroll
    for (int k = 0; k < F; ++k) {
        v[0][k] = on ? (1.0f - r.fx) * r.v[k] : 0.0f;
        v[1][k] = on ? r.fx * r.v[k] : 0.0f;
    }
    const uint32_t left = (uint32_t)row_up<1>((int)key);  // on every lane: no short-circuit around the row shift
    const bool head = ((lane & 15) == 0) | (left != key);
    bool add = on;
    if (4 * __popcll(__ballot(!head)) >= kWave) {
        const int end = run_end(head, lane);
        run_step<1>(v, lane + 1 <= end);
        run_step<2>(v, lane + 2 <= end);
        run_step<4>(v, lane + 4 <= end);
        run_step<8>(v, lane + 8 <= end);
        add = on && head;
    }
    if (add) {
#pragma unroll
        for (int k = 0; k < F; ++k) unsafeAtomicAdd(acc + a * F + k, (double)v[0][k]);
        if (kind != kKindAlone) {
            const uint32_t b = second_place(a, kind);
#pragma unroll
            for (int k = 0; k < F; ++k) unsafeAtomicAdd(acc + b * F + k, (double)v[1][k]);
        }
    }
}

template <int F>
__device__ __forceinline__ BinRecord<F> load_record(const uint32_t *recs, int64_t i) {
    constexpr int W = (int)(sizeof(BinRecord<F>) / 4);
    if constexpr (F == 2) {
        return __builtin_bit_cast(BinRecord<F>, *reinterpret_cast<const uint4 *>(recs + i * W));
    } else {
        BinRecord<F> r;
        uint2 *w = reinterpret_cast<uint2 *>(&r);
        const uint2 *s = reinterpret_cast<const uint2 *>(recs + i * W);
#pragma unroll
        for (int k = 0; k < W / 2; ++k) w[k] = s[k];
        return r;
    }
}

template <int D, int F, bool FOLD>
__global__ __launch_bounds__(kApplyThreads) void k_scatter_apply(NectGridDesc g, BinPlan P, int chunk,
                                                                 const uint32_t *__restrict__ counts,
                                                                 const uint32_t *__restrict__ recs,
                                                                 float *__restrict__ grad) {
    __shared__ double acc[kBinFloats];
    const int task = blockIdx.x;
    int l = 0;
    while (task >= P.task0[l + 1]) ++l;
    const int gr = P.granule[l], lb = P.log2_bins[l], ls = P.log2_splits[l];
    const int bin = (task - P.task0[l]) >> ls, part = (task - P.task0[l]) & ((1 << ls) - 1);
    const uint32_t cap = P.cap[l];
    // with a list per XCD, wave w takes list w (they hold even shares); else the waves share the one list.  Of each
    // list, this workgroup takes its part
    constexpr int U = 4, kWaves = kApplyThreads / kWave;
    static_assert(kWaves == kXcds, "a wave per list");
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int list = wave % P.n_lists, turn = wave / P.n_lists, turns = kWaves / P.n_lists;
    const int64_t n = min(counts[((int64_t)chunk * P.n_lists + list) * P.n_counters + P.bin0[l] + bin], cap);
    const int64_t r0 = (n * part) >> ls, r1 = (n * (part + 1)) >> ls;
    if (__syncthreads_or(r0 < r1) == 0) return;
    const int floats = P.entries[l] * F;
    for (int i = threadIdx.x; i < floats; i += kApplyThreads) acc[i] = 0.0;
    __syncthreads();
    const int64_t base = P.rec0[l] + (((int64_t)list << lb) + bin) * cap;
    // whole waves stay in the loop: apply_records reads neighbouring lanes
    for (int64_t i0 = r0 + turn * kWave; i0 < r1; i0 += U * turns * kWave) {
        BinRecord<F> r[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t i = i0 + u * turns * kWave + lane;
            r[u] = load_record<F>(recs, base + min(i, r1 - 1));
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t i = i0 + u * turns * kWave;
            if (i < r1) apply_records<F>(acc, r[u], i + lane < r1, lane);
        }
    }
    __syncthreads();
    // the touched entries: consecutive lanes take consecutive floats, one request per 64-byte block
    const LevelAdd<FOLD> to = level_add<D, FOLD>(g, P, l, grad);
    const uint32_t size = P.size[l];
    for (int k = threadIdx.x; k < floats; k += kApplyThreads) {
        const double v = acc[k];
        if (v != 0.0) {
            const uint32_t e = entry_of((uint32_t)k / F, (uint32_t)bin, gr, lb);
            if (e < size) to.template add<F>(e, (int)((uint32_t)k % F), v);
        }
    }
}

// ------------------------------------------------------------------- host

int32_t check_grid(const NectGridDesc *g);

static int ceil_log2(uint32_t v) {
    int l = 0;
    while (((uint64_t)1 << l) < v) ++l;
    return l;
}

static bool level_is_hashed(const NectGridDesc &g, int l) {
    uint64_t stride = 1;
    for (int d = 0; d < g.n_dims && stride <= g.level_size[l]; ++d) stride *= g.resolution[l];
    return stride > g.level_size[l];
}

// Runs of 2^granule table entries along the first coordinate that a slice of a level, its last coordinate held, touches.
static int64_t runs_per_slice(uint32_t res, int granule) {
    return (int64_t)res * std::max<int64_t>(1, ((int64_t)res >> granule));
}

// Fills P for batches of at most `slots` samples per chunk; returns the record
// buffer's records, or -1 when a level needs more bins than the kernels take.
// `points`: a caller's (their number and sizes do not depend on it).
static int64_t plan_bins(const NectGridDesc &g, bool fold, bool points, int64_t slots, BinPlan &P, int &group_bins) {
    const int dims = g.n_dims - (fold ? 1 : 0);
    const int64_t pairs = slots << (dims - 1);
    // small batches (a few rays, a region) crowd into few bins more often, and lists that hold the whole batch cost
    // them little: within kWholeListBytes in all, no list can overflow.  (Taken for the grid as it is, folded or not: a
    // folded batch then never needs more than the same chunks of the unfolded one, which the workspace is sized for.)
    int64_t all = 0;
    for (int l = 0; l < g.n_levels; ++l) {
        const int lb = std::max(0, ceil_log2(g.level_size[l]) - (kBinLog2Floats - (g.n_features == 2 ? 1 : 2)));
        all += (slots << (g.n_dims - 1 + lb)) * (8 + 4 * g.n_features);
    }
    const bool whole = all <= kWholeListBytes;
    // a list per XCD once every XCD has many workgroups of the chunk (their shares are even then)
    P.n_lists = !whole && slots >= (int64_t)kXcds * 32 * kEmitThreads ? kXcds : 1;
    const int log2_entries = kBinLog2Floats - (g.n_features == 2 ? 1 : 2);
    int64_t rec = 0;
    int counter = 0, task = 0;
    group_bins = 0;
    P.hashed = 0;
    // a group's counters leave room for two workgroups' records on a CU (three dimensions, two features: three);
    // a batch of few workgroups is spread over the device by smaller groups
    const int most = dims == 4 || g.n_features == 4 ? 1024 : kGroupBins;
    const int64_t blocks = (slots + kEmitThreads - 1) / kEmitThreads;
    const int most_levels = (int)std::max<int64_t>(1, std::min<int64_t>(16 / g.n_features, blocks * g.n_levels / kFillBlocks));
    int groups = 0, in_group = kGroupBins;
    for (int l = 0; l < g.n_levels; ++l) {
        const bool hashed = level_is_hashed(g, l);
        uint32_t size = g.level_size[l];
        if (fold && !hashed) {
            // one t's entries, up to the upper corners of the far faces: c_d <= res in every dimension
            uint64_t n = 0, stride = 1;
            for (int d = 0; d < dims; ++d) {
                n += stride * g.resolution[l];
                stride *= g.resolution[l];
            }
            size = (uint32_t)(n + 1);
        }
        P.size[l] = size;
        P.hashed |= hashed ? 1u << l : 0u;
        const int lb = std::max(0, ceil_log2(size) - log2_entries);
        const int nb = 1 << lb;
        if (nb > kMaxBins) return -1;
        if (in_group + nb > most || l - P.group0[groups - 1] >= most_levels) {
            P.group0[groups++] = (uint8_t)l;
            in_group = 0;
        }
        in_group += nb;
        group_bins = std::max(group_bins, in_group);
        // (two dimensions: a hashed index holds few values of its second term, which alone would choose the bin)
        const bool spread = hashed && dims > 2 && (size & (size - 1)) == 0;
        int gr = lb == 0 || spread ? log2_entries : 6;
        // A caller's points may all have one last coordinate (a model over (z, y, t) at one time): the second term alone
        // then chooses the bin here, too, and where it has few values for the bins (four features: twice as many bins,
        // and a record past its list costs twice the atomics) lists overflow.  Such levels' bins interleave in runs short
        // enough for four runs of a slice per bin, and no shorter than 64 entries: a pair across two runs adds its second
        // entry by itself.  A million random points, 16 x 4, T = 2^19: last coordinate held 4.86 -> 1.97 ms (atomics
        // without records: 5.14), all varying 1.31 -> 1.40; 23 levels of growth 1.17, T = 2^21: 7.91 -> 3.67 (6.67)
        // and 2.47 -> 2.54.
        if (points && dims == 3 && g.n_features == 4 && spread && nb >= 256)
            while (gr > 6 && runs_per_slice(g.resolution[l], gr) < 4 * (int64_t)nb) --gr;
        P.log2_bins[l] = (uint8_t)lb;
        P.granule[l] = (uint8_t)gr;
        const int64_t rows = ((int64_t)size + ((int64_t)1 << (gr + lb)) - 1) >> (gr + lb);
        P.entries[l] = lb == 0 ? (int32_t)size : (int32_t)std::min<int64_t>(rows << gr, (int64_t)1 << log2_entries);
        // room for 1.5 (contiguous bins) or 2.5 (interleaved) times a bin's even share of the records
        const int64_t share = (pairs / P.n_lists + nb - 1) / nb;
        int64_t cap = whole ? pairs : std::min(pairs, spread ? share + share / 2 : 2 * share + share / 2);
        cap = (cap + 15) / 16 * 16;
        if (cap >= ((int64_t)1 << 32)) return -1;
        P.cap[l] = (uint32_t)cap;
        P.bin0[l] = counter;
        P.rec0[l] = rec;
        counter += nb;
        rec += cap * nb * P.n_lists;
        // about 64 workgroups per level at least, of kPartRecords records at least: every part adds its sums to the
        // gradient by itself
        int ls = 0;
        while (lb + ls < 6 && (pairs >> (lb + ls + 1)) >= kPartRecords) ++ls;
        P.log2_splits[l] = (uint8_t)ls;
        P.task0[l] = task;
        task += nb << ls;
    }
    for (int l = g.n_levels; l <= NECT_MAX_LEVELS; ++l) P.task0[l] = task;
    P.group0[groups] = (uint8_t)g.n_levels;
    P.n_groups = groups;
    P.n_bins = counter;
    P.n_counters = (counter + kCounterLead - 1) / kCounterLead * kCounterLead;
    return rec;
}

// Chunks so that counters and records fit in `bytes`; 0 when they cannot.  The counts tried do not depend on `bytes`, so
// that the size found for one limit is enough for the launch, whose limit it is.
static int plan_chunks(const NectGridDesc &g, bool fold, bool points, int64_t slots, int64_t bytes, BinPlan &P,
                       int &group_bins, int64_t &chunk_slots, int64_t &need) {
    const int64_t rec_bytes = 8 + 4 * g.n_features;
    const int64_t tiles = (slots + kTile - 1) / kTile;
    for (int64_t k = 1; k <= tiles && k <= 4096; k += std::max<int64_t>(1, k / 16)) {
        chunk_slots = ((tiles + k - 1) / k) * kTile;
        const int64_t rec = plan_bins(g, fold, points, chunk_slots, P, group_bins);
        if (rec < 0) return 0;
        need = rec * rec_bytes + k * (int64_t)P.n_counters * P.n_lists * 4;
        if (need <= bytes) {
            P.n_chunks = (int32_t)k;
            return (int)k;
        }
    }
    return 0;
}

template <int D, int F, bool FOLD, typename Src>
static int32_t launch_binned(const NectGridDesc &g, const Src &src, float t, int64_t slots, const DoutView &dv,
                             float *grad, void *ws, int64_t ws_bytes, hipStream_t st) {
    BinPlan P = {};
    P.t = t;
    int group_bins;
    int64_t chunk_slots, need;
    constexpr bool kPoints = std::is_same<Src, PointRowsSource<D>>::value;
    const int chunks = plan_chunks(g, FOLD, kPoints, slots, ws_bytes, P, group_bins, chunk_slots, need);
    NECT_REQUIRE(chunks > 0, "workspace too small for this grid and batch");
    uint32_t *counts = static_cast<uint32_t *>(ws);
    const int n_counts = chunks * P.n_lists * P.n_counters;
    uint32_t *recs = counts + n_counts;
    const int64_t esz = dv.dtype == NECT_F32 ? 4 : 2;
    const uintptr_t lead = (uintptr_t)dv.p | (uintptr_t)(dv.stride * esz);
    const int align = lead % 16 == 0 ? 16 : (lead % 8 == 0 ? 8 : 4);
    const size_t lds = (size_t)kEmitThreads * (1 << (D - 1)) * sizeof(BinRecord<F>) + (size_t)group_bins * 8;
    const auto emit = k_scatter_emit<D, F, FOLD, Src>;
    const auto apply = k_scatter_apply<D, F, FOLD>;
    if (lds > 64 * 1024) {
        const hipError_t e = hipFuncSetAttribute((const void *)emit, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) {
            set_error(std::string("k_scatter_emit: cannot reserve LDS: ") + hipGetErrorString(e));
            return 1;
        }
    }
    hipLaunchKernelGGL(k_scatter_zero, dim3((n_counts + 255) / 256), dim3(256), 0, st, counts, n_counts);
    if (check_launch("k_scatter_zero")) return 1;
    const int64_t sample_blocks = (chunk_slots + kEmitThreads - 1) / kEmitThreads;
    const unsigned blocks = (unsigned)((sample_blocks + kXcds - 1) / kXcds * kXcds * P.n_groups);
    for (int c = 0; c < chunks; ++c) {
        hipLaunchKernelGGL(emit, dim3(blocks), dim3(kEmitThreads), lds, st, g, P, src, c, dv, align, counts, recs, grad,
                           group_bins);
        if (check_launch("k_scatter_emit")) return 1;
        hipLaunchKernelGGL(apply, dim3(P.task0[g.n_levels]), dim3(kApplyThreads), 0, st, g, P, c, counts,
                           recs, grad);
        if (check_launch("k_scatter_apply")) return 1;
    }
    return 0;
}

// Whether the grid's last dimension reads t (column 3) and its levels can be folded over it.
static bool can_fold(const NectGridDesc &g, const int32_t *src_cols) {
    if (!(src_cols ? src_cols[g.n_dims - 1] == 3 : g.n_dims == 4)) return false;
    for (int d = 0; d + 1 < g.n_dims && src_cols; ++d)
        if (src_cols[d] == 3) return false;
    for (int l = 0; l < g.n_levels; ++l) {
        const uint32_t size = g.level_size[l];
        // the xor of t's term commutes with the mask of a power-of-two size only; a dense level's spatial index
        // stays within its resolution (positions lie in [0, 1])
        if (level_is_hashed(g, l) ? (size & (size - 1)) != 0 : !((double)g.scale[l] + 0.5 < (double)g.resolution[l]))
            return false;
    }
    return true;
}

static int32_t check_binned(const DoutView &dv, const NectGridDesc &g, const float *grad, const void *ws) {
    NECT_REQUIRE(dv.p && grad && ws, "NULL pointer");
    NECT_REQUIRE(dv.dtype == NECT_F32 || dv.dtype == NECT_F16 || dv.dtype == NECT_BF16,
                 "dout_dtype must be NECT_F32, NECT_F16 or NECT_BF16");
    NECT_REQUIRE(dv.stride >= (int64_t)g.n_levels * g.n_features, "dout_stride smaller than L*F");
    NECT_REQUIRE(((uintptr_t)ws & 255) == 0, "workspace must be 256-byte aligned");
    return 0;
}

}  // namespace nect

using namespace nect;

extern "C" int64_t nect_grid_binned_workspace(const NectGridDesc *desc, int64_t n_slots, int64_t max_bytes) {
    clear_error();
    if (check_grid(desc)) return -1;
    if (n_slots <= 0) return 0;
    BinPlan P = {};
    int group_bins;
    int64_t chunk_slots, need;
    // (a folded batch needs no more, and takes fewer chunks where it needs less)
    if (plan_chunks(*desc, false, false, n_slots, max_bytes, P, group_bins, chunk_slots, need) == 0) return 0;
    return need;
}

extern "C" int32_t nect_grid_backward_binned_rays(const NectGridDesc *desc, const int32_t *src_cols,
                                                  const NectRay *rays, const int32_t *tile_offsets,
                                                  const int32_t *tile_ray, const int32_t *n_tiles, int64_t max_tiles,
                                                  float t, int32_t dout_dtype, const void *dout, int64_t dout_stride,
                                                  const float *dout_scale, float *grad, void *workspace,
                                                  int64_t workspace_bytes, void *stream) {
    clear_error();
    if (check_grid(desc)) return 1;
    NECT_REQUIRE(rays && tile_offsets && tile_ray && n_tiles, "NULL pointer");
    NECT_REQUIRE(max_tiles >= 1 && max_tiles < ((int64_t)1 << 31) / kTile, "max_tiles out of range");
    const DoutView dv = {dout, dout_stride, dout_dtype, dout_scale};
    if (check_binned(dv, *desc, grad, workspace)) return 1;
    uint32_t cmap = 0;
    for (int d = 0; d < desc->n_dims && src_cols; ++d) {
        NECT_REQUIRE(src_cols[d] >= 0 && src_cols[d] <= 3, "src_cols entries must be 0 (z), 1 (y), 2 (x) or 3 (t)");
        cmap |= ((uint32_t)src_cols[d] ^ (uint32_t)d) << (2 * d);
    }
    const int64_t slots = max_tiles * kTile;
    const hipStream_t st = as_stream(stream);
    const int D = desc->n_dims, F = desc->n_features;
    const bool fold = can_fold(*desc, src_cols);
#define NECT_BINNED(DS, FF, FOLD)                                                                                  \
    launch_binned<DS, FF, FOLD>(*desc, RayColsSource<DS>{rays, tile_offsets, tile_ray, n_tiles, max_tiles, t, cmap}, \
                                t, slots, dv, grad, workspace, workspace_bytes, st)
    if (D == 3 && fold) return F == 2 ? NECT_BINNED(2, 2, true) : NECT_BINNED(2, 4, true);
    if (D == 3) return F == 2 ? NECT_BINNED(3, 2, false) : NECT_BINNED(3, 4, false);
    if (fold) return F == 2 ? NECT_BINNED(3, 2, true) : NECT_BINNED(3, 4, true);
    return F == 2 ? NECT_BINNED(4, 2, false) : NECT_BINNED(4, 4, false);
#undef NECT_BINNED
}

extern "C" int32_t nect_grid_backward_binned(const NectGridDesc *desc, const float *x, int64_t n, int64_t x_stride,
                                             int32_t dout_dtype, const void *dout, int64_t dout_stride,
                                             const float *dout_scale, float *grad, void *workspace,
                                             int64_t workspace_bytes, void *stream) {
    clear_error();
    if (check_grid(desc)) return 1;
    NECT_REQUIRE(n >= 0, "n must be >= 0");
    if (n == 0) return 0;
    NECT_REQUIRE(x, "NULL pointer");
    NECT_REQUIRE(x_stride >= desc->n_dims, "x_stride smaller than n_dims");
    const DoutView dv = {dout, dout_stride, dout_dtype, dout_scale};
    if (check_binned(dv, *desc, grad, workspace)) return 1;
    const hipStream_t st = as_stream(stream);
    const int D = desc->n_dims, F = desc->n_features;
#define NECT_BINNED(DS, FF)                                                                                       \
    launch_binned<DS, FF, false>(*desc, PointRowsSource<DS>{x, n, x_stride}, 0.0f, n, dv, grad, workspace,        \
                                 workspace_bytes, st)
    if (D == 3) return F == 2 ? NECT_BINNED(3, 2) : NECT_BINNED(3, 4);
    return F == 2 ? NECT_BINNED(4, 2) : NECT_BINNED(4, 4);
#undef NECT_BINNED
}
