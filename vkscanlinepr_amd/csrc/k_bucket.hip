// k_bucket.hip -- (path, cell row) buckets: the MSD step of the segmented sort (gfx950).
//
// A path's sort keys are (row, x) cell keys, so its entries split into one bucket per cell row,
// followed by an off-canvas bucket and the row-0 bucket (the reference compares keys as signed
// int32: rows 2..h-2, then the off-canvas sentinel, then row 0; gen_fragment.comp:180-187,
// naive_seg_sort_pairs.comp:69).  The transform pass bounds each path's rows from its control
// points (a Bezier curve stays inside their hull), so each path owns a small, exactly sized
// bucket range.  Entries are counted per bucket while their keys are generated, and the buckets
// are packed into bands of at most 2048 entries that one workgroup sorts in LDS.  The scatter
// only has to bring each entry into its band (the band sort orders by bucket, then x), so the
// entries of a run that fall into one band take their slots with one atomic and are stored
// contiguously.  After the sort the per-bucket ranges give the composite each path's records of
// each cell row without any further sorting.
#include "device_common.hpp"
#include "kernels.hpp"
#include "scan_common.hpp"

namespace spr {

namespace {

constexpr int kBlock = 256;

inline unsigned grid_for(int64_t n) {
    int64_t g = (n + kBlock - 1) / kBlock;
    return (unsigned)(g < 1 ? 1 : g);
}

// Scatter into band order.  The wide sort word orders exactly like the reference's signed
// (key, index) pair and carries the winding change in its two low bits.  The narrow word (used
// when no stage is exported) drops the index: (bucket inside its path) << 17 | (x + 2) << 2 |
// (winding change + 1); inside a band (whole buckets of one path) it orders like the key, and the
// order among equal keys changes no record, no span and no pixel (no span starts between equal
// keys, and the winding number after a run of equal keys is the sum over the whole run).  The
// band of bucket b is flag_scan[b + 1] - 1 (flag_scan: exclusive scan of the band-start flags).
// Each wave takes kRounds chunks of 64 consecutive entries and issues every load, then every
// slot atomic (one per run of equal bands, on the band's fill counter), of all chunks before it
// waits on any of them.  The head of a run also adds the run's winding changes to the band's sum
// (bsum), from which one scan gives every band its exclusive prefix before the band sort.
// PACKED (narrow only): the piece kernels already stored each entry's global bucket (in key) and
// its narrow word (in epath), so the path-table gathers are skipped.
constexpr int kRounds = 4;

template <bool NARROW, bool PACKED>
__global__ __launch_bounds__(kBlock) void k_bucket_scatter(const int32_t* __restrict__ key,
                                                           const int8_t* __restrict__ wn,
                                                           const uint32_t* __restrict__ epath, int64_t N,
                                                           const int32_t* __restrict__ bucket_base,
                                                           const int2* __restrict__ prow,
                                                           const int32_t* __restrict__ flag_scan,
                                                           const int32_t* __restrict__ band_start,
                                                           int32_t* __restrict__ fill,
                                                           int32_t* __restrict__ bsum,
                                                           unsigned long long* __restrict__ out,
                                                           uint32_t* __restrict__ out32,
                                                           int32_t* __restrict__ err,
                                                           const int32_t* __restrict__ n_dev) {
    const int64_t n = n_dev ? min((int64_t)*n_dev, N) : N;
    const int lane = threadIdx.x & 63;
    const int64_t g0 = ((int64_t)blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6)) * (64 * kRounds);
    uint32_t pth[kRounds];
    int32_t k[kRounds], wv[kRounds];
    bool valid[kRounds];
    uint32_t b[kRounds], loc[kRounds];
    bool sent[kRounds];
#pragma unroll
    for (int r = 0; r < kRounds; ++r) {
        const int64_t i = g0 + r * 64 + lane;
        valid[r] = i < n;
        pth[r] = kNoPath; k[r] = 0; wv[r] = 0;
        b[r] = 0; loc[r] = 0; sent[r] = false;
        if constexpr (PACKED) {
            // k = the narrow word, b = the global bucket
            if (valid[r]) {
                b[r] = (uint32_t)key[i];
                k[r] = (int32_t)epath[i];
                wv[r] = (int32_t)((uint32_t)k[r] & 3u) - 1;
            }
        } else {
            if (valid[r]) { pth[r] = epath[i]; k[r] = key[i]; wv[r] = wn[i]; }
            if (pth[r] == kNoPath) { valid[r] = false; wv[r] = 0; }  // an entry without a fragment
        }
    }
    if constexpr (!PACKED) {
#pragma unroll
        for (int r = 0; r < kRounds; ++r) {
            if (valid[r]) {
                const int2 pr = prow[pth[r]];
                loc[r] = bucket_local(k[r], pr, err);
                sent[r] = loc[r] == (uint32_t)pr.y;
                b[r] = (uint32_t)bucket_base[pth[r]] + loc[r];
            }
        }
    }
#pragma unroll
    for (int r = 0; r < kRounds; ++r)
        if (valid[r]) b[r] = (uint32_t)(flag_scan[b[r] + 1] - 1);  // bucket -> band
    // runs of equal bands: heads take their run's slots with one atomic each, and add the run's
    // winding changes (an inclusive wave scan read at the run's last lane) to the band's sum
    unsigned long long vm[kRounds], hd[kRounds];
    int32_t base[kRounds];
#pragma unroll
    for (int r = 0; r < kRounds; ++r) {
        vm[r] = __ballot(valid[r]);
        hd[r] = run_heads(b[r], valid[r], vm[r]);
        const int32_t inc = wave_inclusive_add(wv[r]);
        const bool head = (hd[r] >> lane) & 1ull;
        const int len = head ? run_length(lane, hd[r], vm[r]) : 1;
        const int32_t at_end = __shfl(inc, lane + len - 1);
        base[r] = 0;
        if (head) {
            base[r] = band_start[b[r]] + atomicAdd(&fill[b[r]], len);
            const int32_t rs = at_end - inc + wv[r];
            if (rs != 0) atomicAdd(&bsum[b[r]], rs);
        }
    }
#pragma unroll
    for (int r = 0; r < kRounds; ++r) {
        const unsigned long long mine = hd[r] & ((2ull << lane) - 1ull);
        const int h = (valid[r] && mine) ? 63 - __clzll((long long)mine) : lane;
        const int32_t slot = __shfl(base[r], h) + (lane - h);
        if (valid[r]) {
            const int64_t i = g0 + r * 64 + lane;
            if constexpr (PACKED) {
                out32[slot] = (uint32_t)k[r];
            } else if constexpr (NARROW) {
                // the off-canvas bucket holds one key: its x is left at 0
                const uint32_t xl = sent[r] ? 0u : ((uint32_t)k[r] & 0xFFFFu) - kNarrowX0;
                out32[slot] = (loc[r] << 17) | (xl << 2) | (uint32_t)(wv[r] + 1);
            } else {
                const unsigned long long w = ((unsigned long long)((uint32_t)k[r] ^ 0x80000000u) << 32) |
                                             ((unsigned long long)i << 2) | (unsigned long long)(uint32_t)(wv[r] + 1);
                out[slot] = w;
            }
        }
    }
}

// What a run of buckets tells the buckets after it: its entries and the size of its last non-empty
// bucket since the last path start (0: none since then), if it holds either.
struct OpBands {
    struct T {
        uint32_t sum, last;
        bool defined;
    };
    __device__ static T zero() { return {0u, 0u, false}; }
    __device__ static T add(const T& a, const T& b) {  // b follows a
        return {a.sum + b.sum, b.defined ? b.last : a.last, a.defined || b.defined};
    }
    // sums and sizes are at most 2^30, a size with an entry after it less
    __device__ static uint64_t encode(uint64_t st, const T& v) {
        return (st << 62) | ((uint64_t)(v.defined ? 1u : 0u) << 61) | ((uint64_t)min(v.last, (1u << 30) - 1u) << 31) |
               (v.sum & 0x7FFFFFFFu);
    }
    __device__ static uint64_t state(uint64_t w) { return w >> 62; }
    __device__ static T value(uint64_t w) {
        return {(uint32_t)(w & 0x7FFFFFFFu), (uint32_t)(w >> 31) & 0x3FFFFFFFu, ((w >> 61) & 1u) != 0};
    }
};

__device__ inline OpBands::T shfl_up_bands(const OpBands::T& v, int d) {
    return {(uint32_t)__shfl_up((int)v.sum, d), (uint32_t)__shfl_up((int)v.last, d), __shfl_up(v.defined ? 1 : 0, d) != 0};
}

// The exclusive prefix of a tile by decoupled look-back, 64 predecessors at a time (first wave only);
// as lookback() of scan_common.hpp for an operation that does not commute.
__device__ inline OpBands::T lookback_bands(unsigned long long* status, int64_t tile, const OpBands::T& agg) {
    const int lane = threadIdx.x & 63;
    if (lane == 0) store_status(&status[tile], OpBands::encode(tile == 0 ? kStInclusive : kStAggregate, agg));
    OpBands::T excl = OpBands::zero();
    for (int64_t pred = tile - 1; pred >= 0;) {
        const int64_t idx = pred - lane;
        const unsigned long long st = idx >= 0 ? load_status(&status[idx]) : OpBands::encode(kStInclusive, OpBands::zero());
        const uint64_t state = OpBands::state(st);
        const unsigned long long inc_mask = __ballot(state == kStInclusive), bad_mask = __ballot(state == 0);
        const int first_inc = inc_mask ? __ffsll((long long)inc_mask) - 1 : 64;
        const unsigned long long upto = first_inc >= 63 ? ~0ull : ((2ull << first_inc) - 1ull);
        if (bad_mask & upto) {
            __builtin_amdgcn_s_sleep(1);
            continue;
        }
        // lane 0 holds the nearest predecessor: combine from the highest lane down
        OpBands::T v = lane <= first_inc ? OpBands::value(st) : OpBands::zero();
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const OpBands::T u = {(uint32_t)__shfl_down((int)v.sum, o), (uint32_t)__shfl_down((int)v.last, o),
                                  __shfl_down(v.defined ? 1 : 0, o) != 0};
            if (lane + o < 64) v = OpBands::add(u, v);
        }
        const OpBands::T all = {(uint32_t)__shfl((int)v.sum, 0), (uint32_t)__shfl((int)v.last, 0),
                                __shfl(v.defined ? 1 : 0, 0) != 0};
        excl = OpBands::add(all, excl);
        if (first_inc < 64) break;
        pred -= 64;
    }
    if (lane == 0 && tile > 0) store_status(&status[tile], OpBands::encode(kStInclusive, OpBands::add(excl, agg)));
    return excl;
}

// Bucket offsets and bands in one pass over the bucket counts (in place: `hist` becomes the
// exclusive offsets, total at [NB]).  A band is a run of consecutive buckets of one path whose
// entries start in the same 512-entry window (kBandWindowLog); a bucket of more than 512 entries is
// a band of its own.  Every band therefore holds at most 1024 entries (sorted by one wave, 16 per
// lane) unless it is a single larger bucket.  A bucket starts a band when it is not empty and the
// last non-empty bucket of its path before it started in another window, or either exceeds the
// window, or there is none; that bucket ends where this one starts, so its size is all that the
// look-back has to carry besides the offset.  A second look-back numbers the bands: flag_scan[b] =
// bands before bucket b (total at [NB]), and each band's start, path and path rows are written.
constexpr int kBandItems = 8, kBandTile = kBlock * kBandItems;
constexpr int kBandPaths = kBandTile / 2 + 2;  // paths of a tile at most: a path owns two buckets or more
static_assert(kBandTile == kBucketBandTile, "status arrays of the band pass");
__global__ __launch_bounds__(kBlock) void k_bands(const BandArgs K) {
    __shared__ int32_t s_base[kBandPaths];
    __shared__ int32_t s_w[kBlock / 64], s_tile, s_p0;
    __shared__ uint32_t s_sum[kBlock / 64], s_last[kBlock / 64];
    __shared__ bool s_def[kBlock / 64];
    const int32_t NB = K.nb_dev ? min(*K.nb_dev, K.NB) : K.NB;
    if ((int64_t)blockIdx.x * kBandTile >= (NB > 0 ? NB : 1)) return;  // past the live buckets: no ticket
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t tile = ordered_tile_id(K.counter, &s_tile);
    const int64_t b0 = tile * kBandTile;
    // the paths of the tile's buckets: the path that holds b0, by a 64-way search of the first wave
    if (wave == 0) {
        int64_t lo = 0, hi = K.Np;  // bucket_base[lo] <= b0 < bucket_base[hi]
        while (hi - lo > 1) {
            const int64_t step = (hi - lo + 63) / 64;
            const int64_t at = min(lo + (lane + 1) * step, hi);
            const unsigned long long above = __ballot(at >= (int64_t)K.Np || (int64_t)K.bucket_base[at] > b0);
            const int f = above ? __ffsll((long long)above) - 1 : 63;
            const int64_t base = lo;
            hi = min(base + (f + 1) * step, hi);
            lo = base + f * step;
        }
        if (lane == 0) s_p0 = (int32_t)lo;
    }
    __syncthreads();
    const int32_t p0 = s_p0;
    for (int i = tid; i < kBandPaths; i += kBlock)
        s_base[i] = p0 + i <= (int32_t)K.Np ? K.bucket_base[p0 + i] : 0x7FFFFFFF;
    __syncthreads();
    // thread t owns kBandItems consecutive buckets
    const int64_t my = b0 + (int64_t)tid * kBandItems;
    int pl = 0;  // path (local) of bucket my: s_base[pl] <= my < s_base[pl + 1]
    {
        int hi = kBandPaths - 1;
        while (hi - pl > 1) {
            const int mid = (pl + hi) >> 1;
            if ((int64_t)s_base[mid] <= my) pl = mid; else hi = mid;
        }
    }
    int32_t sz[kBandItems];
#pragma unroll
    for (int k = 0; k < kBandItems; ++k) sz[k] = my + k < NB ? K.hist[my + k] : 0;
    OpBands::T agg = OpBands::zero();
    {
        int q = pl;
#pragma unroll
        for (int k = 0; k < kBandItems; ++k) {
            while (q + 1 < kBandPaths && (int64_t)s_base[q + 1] <= my + k) ++q;
            if ((int64_t)s_base[q] == my + k) { agg.last = 0; agg.defined = true; }
            if (sz[k] > 0) { agg.last = (uint32_t)sz[k]; agg.defined = true; }
            agg.sum += (uint32_t)sz[k];
        }
    }
    OpBands::T inc = agg;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const OpBands::T u = shfl_up_bands(inc, o);
        if (lane >= o) inc = OpBands::add(u, inc);
    }
    if (lane == 63) { s_sum[wave] = inc.sum; s_last[wave] = inc.last; s_def[wave] = inc.defined; }
    __syncthreads();
    OpBands::T before = OpBands::zero(), total = OpBands::zero();
#pragma unroll
    for (int k = 0; k < kBlock / 64; ++k) {
        const OpBands::T x = {s_sum[k], s_last[k], s_def[k]};
        if (k < wave) before = OpBands::add(before, x);
        total = OpBands::add(total, x);
    }
    __syncthreads();
    if (wave == 0) {
        const OpBands::T pre = lookback_bands(K.status, tile, total);
        if (lane == 0) { s_sum[0] = pre.sum; s_last[0] = pre.last; s_def[0] = pre.defined; }
    }
    __syncthreads();
    const OpBands::T tile_pre = {s_sum[0], s_last[0], s_def[0]};
    OpBands::T ex = shfl_up_bands(inc, 1);
    if (lane == 0) ex = OpBands::zero();
    ex = OpBands::add(tile_pre, OpBands::add(before, ex));
    // flags
    const int32_t win = 1 << K.window_log;
    uint32_t flags = 0;
    {
        int32_t o = (int32_t)ex.sum, last = (int32_t)ex.last;
        int q = pl;
#pragma unroll
        for (int k = 0; k < kBandItems; ++k) {
            while (q + 1 < kBandPaths && (int64_t)s_base[q + 1] <= my + k) ++q;
            if ((int64_t)s_base[q] == my + k) last = 0;
            if (sz[k] > 0) {
                const bool f = last == 0 || (o >> K.window_log) != ((o - last) >> K.window_log) || last > win || sz[k] > win;
                flags |= f ? 1u << k : 0u;
                last = sz[k];
            }
            o += sz[k];
        }
    }
    const int32_t mine = __popc(flags);
    const int32_t binc = wave_inclusive_add(mine);
    if (lane == 63) s_w[wave] = binc;
    __syncthreads();
    int32_t bbefore = 0, btotal = 0;
#pragma unroll
    for (int k = 0; k < kBlock / 64; ++k) {
        if (k < wave) bbefore += s_w[k];
        btotal += s_w[k];
    }
    __syncthreads();
    if (wave == 0) {
        const int32_t pre = lookback<OpI32>(K.status2, tile, btotal);
        if (lane == 0) s_w[0] = pre;
    }
    __syncthreads();
    int32_t band = s_w[0] + bbefore + binc - mine;
    {
        int32_t o = (int32_t)ex.sum;
        int q = pl;
#pragma unroll
        for (int k = 0; k < kBandItems; ++k) {
            if (my + k >= NB) break;
            while (q + 1 < kBandPaths && (int64_t)s_base[q + 1] <= my + k) ++q;
            K.hist[my + k] = o;
            K.flag_scan[my + k] = band;
            if ((flags >> k) & 1u) {
                K.band_start[band] = o;
                if (K.band_pr) {
                    K.band_pr[band] = K.prow[p0 + q];
                    K.band_path[band] = p0 + q;
                }
                ++band;
            }
            o += sz[k];
            if (my + k == NB - 1) {
                K.hist[NB] = o;
                K.flag_scan[NB] = band;
                K.band_start[band] = o;
                if (K.n_sorted) *K.n_sorted = o;
                if (K.n_bands) *K.n_bands = band;
            }
        }
    }
}

}  // namespace

hipError_t launch_bucket_scatter(const int32_t* key, const int8_t* wn, const uint32_t* epath, int64_t N,
                                 const int32_t* bucket_base, const int2* prow, const int32_t* flag_scan,
                                 const int32_t* band_start, int32_t* fill, int32_t* bsum, unsigned long long* out,
                                 int32_t* err, hipStream_t s, const int32_t* n_dev, bool narrow, bool packed) {
    if (N == 0) return hipSuccess;
    if (packed && !narrow) return hipErrorInvalidValue;
    const unsigned g = grid_for((N + kRounds - 1) / kRounds);
    if (packed)
        k_bucket_scatter<true, true><<<g, kBlock, 0, s>>>(key, wn, epath, N, bucket_base, prow, flag_scan,
                                                          band_start, fill, bsum, nullptr,
                                                          reinterpret_cast<uint32_t*>(out), err, n_dev);
    else if (narrow)
        k_bucket_scatter<true, false><<<g, kBlock, 0, s>>>(key, wn, epath, N, bucket_base, prow, flag_scan,
                                                           band_start, fill, bsum, nullptr,
                                                           reinterpret_cast<uint32_t*>(out), err, n_dev);
    else
        k_bucket_scatter<false, false><<<g, kBlock, 0, s>>>(key, wn, epath, N, bucket_base, prow, flag_scan,
                                                            band_start, fill, bsum, out, nullptr, err, n_dev);
    return hipGetLastError();
}

hipError_t launch_bands(const BandArgs& K, hipStream_t s) {
    if (K.Np == 0 || K.NB == 0) return hipSuccess;
    if (K.window_log < kBandWindowLog || K.window_log > 10) return hipErrorInvalidValue;  // bands <= max_bands_for
    k_bands<<<(unsigned)((K.NB + kBandTile - 1) / kBandTile), kBlock, 0, s>>>(K);
    return hipGetLastError();
}

}  // namespace spr
