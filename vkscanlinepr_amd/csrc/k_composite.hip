// k_composite.hip -- records to RGBA8 pixels (gfx950).
//
// Replaces the reference's line-list draw (scanlinepr.vert:18-50, scanlinepr.frag:7-14, pipeline
// state scanline_rasterizer.cpp:881-944): every record (yx, width, fill) covers canvas rows y and
// y+1 over columns [x, x+width), records are applied in order (blending disabled: the later one
// wins), and canvas row y lands on image row h-1-y.  All records sit on even rows, so the image
// is a stack of independent two-pixel "cell rows".
//
// One workgroup owns one chunk of CHUNK columns of one cell row; each thread keeps PIX of its
// pixels in registers, one in every CHUNK / PIX columns.  The chunk follows the canvas (launch_composite): a canvas
// row that fills a quarter of a chunk leaves three quarters of the threads without a pixel
// and gives the others four times the pixels to fold one after another.  The (path, row) bucket
// table gives each path's records on
// this row as one contiguous range of non-overlapping compact records (x | width << 16) with one
// colour.  Paths are taken in order, 64 at a time: a record toggles its path's bit at its first
// column and at its end column in a 64-bit event word per column (LDS), and a prefix XOR over
// the columns turns the events into each pixel's coverage mask (the records of one path never
// overlap, so the XOR of the toggles left of a pixel is exactly "inside one of them").  Each
// thread then folds the set bits of its pixels in path order (overwrite: the last one wins;
// src-over: d = s*a + d*(1-a), from the last opaque path on).  A record costs two LDS operations
// whatever its width, and each image row is written once.
//
// The prefix takes consecutive columns in one thread, the fold in consecutive lanes, through LDS: 64
// neighbouring pixels are mostly covered by the same paths, so a wave's lanes take the same number of
// steps, read the same colours and evaluate the same paints.  Folding PIX consecutive pixels per thread, a
// wave's lanes lay PIX pixels apart, each step lasted as long as the most covered of them, and
// 4096^2 pixels under 55 paths each took 611 us instead of 457; 64 opaque paths on 1024^2 30 instead of
// 16; a drawing with gradients at 1800x1200 289 instead of 94; anti-aliased 4096^2 1,597 instead of 1,281.
//
// Gradient paints (no reference counterpart: the reference draws solid colours only): a path
// with a paint takes, at each covered pixel, the paint's colour at that pixel's centre, packed
// like a solid fill, so the two rows of a cell row get their own colours; the variant that
// evaluates them keeps a second row of pixels per thread.  An evaluation is some 150 dependent
// operations per pixel and path, so this variant runs few pixels per thread (more waves), maps each
// pixel centre back to the scene once for all its paths, and reads the batch's paints and stops
// from LDS instead of through two dependent loads per evaluation.
//
// Anti-aliased coverage (src-over): a boundary cell record whose 64-sample mask (k_aa.hip) is not
// full appends, at each of its two columns, an entry (path of the batch, covered samples of row y,
// of row y + 1) to that column's list in LDS (kAaSlots per column, and kAaMore more in a list for the
// whole chunk); the fold scales such a path's premultiplied colour by count/16 in each row.  A batch
// whose lists would overflow is redone with half as many paths (kAaSlots paths can never overflow).
#include "device_common.hpp"
#include "kernels.hpp"
#include "scan_common.hpp"

namespace spr {

namespace {

constexpr int kStops = 512;                // gradient stops of one batch in LDS
constexpr int kBatch = 64;                 // paths per coverage mask
constexpr int kAaSlots = 4;                // partial-coverage entries per column and batch
// entries of one batch beyond their column's: without them one column of 4,096 with a fifth entry had
// half of all batches done over (4096^2: 1,284 us, with 16 more 1,150); a pixel with more than its slots
// reads them all, so a long list (64, 128) costs denser scenes more than the batches it saves
constexpr int kAaMore = 16;
constexpr int kList = 512;                 // paths listed before their batches are folded
constexpr int kListSub = 256;              // a listing step examines candidate paths in parts of this many
constexpr int kUnroll = 4;                 // records loaded per thread before applying
typedef unsigned long long u64;

// LDS slot of chunk column c: PIX consecutive columns per thread and consecutive columns in
// consecutive lanes both touch every bank once (a permutation inside each 32 columns).
template <int PIX>
__device__ inline int ev_slot(int c) { return c ^ ((c >> 5) & (PIX - 1)); }

__device__ inline u64 shfl_up_u64(u64 v, int d) {
    const uint32_t lo = (uint32_t)v, hi = (uint32_t)(v >> 32);
    return (u64)(uint32_t)__shfl_up((int)lo, d) | ((u64)(uint32_t)__shfl_up((int)hi, d) << 32);
}

// Exclusive prefix XOR of one value per thread over a workgroup of BLOCK threads.
template <int BLOCK>
__device__ inline u64 block_exclusive_xor(u64 v, u64* lds) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    u64 inc = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const u64 u = shfl_up_u64(inc, d);
        if (lane >= d) inc ^= u;
    }
    if (lane == 63) lds[wave] = inc;
    __syncthreads();
    u64 off = 0;
#pragma unroll
    for (int k = 0; k < BLOCK / 64; ++k)
        if (k < wave) off ^= lds[k];
    __syncthreads();
    return off ^ inc ^ v;
}

// The scene point under the centre of canvas pixel (x, y); h: the inverse MVP's rows.
__device__ __forceinline__ float2 scene_point(const float* h, int x, int y) {
    const float px = (float)x + 0.5f, py = (float)y + 0.5f;
    const float u = (h[0] * px + h[1] * py) + h[2];
    const float v = (h[3] * px + h[4] * py) + h[5];
    const float q = (h[6] * px + h[7] * py) + h[8];
    return make_float2(u / q, v / q);
}

// A gradient's colour at scene point (sx, sy), packed like a solid fill (channel times 255
// truncated, alpha times opacity, 0 when the alpha byte is 0).  st: the paint's stops.  Every
// float operation is written out in order (the library is built without contraction).
__device__ __forceinline__ uint32_t paint_color(const Paint& g, const float* st, float sx, float sy) {
    const float gx = (g.xform[0] * sx + g.xform[1] * sy) + g.xform[2];
    const float gy = (g.xform[3] * sx + g.xform[4] * sy) + g.xform[5];
    float t;
    bool degenerate = false;
    if (g.kind == kPaintLinear) {
        const float dx = g.geom[2] - g.geom[0], dy = g.geom[3] - g.geom[1];
        const float den = dx * dx + dy * dy;
        if (den > 0.0f) {
            t = ((gx - g.geom[0]) * dx + (gy - g.geom[1]) * dy) / den;
        } else {
            t = 1.0f;  // both points equal: the last stop's colour
            degenerate = true;
        }
    } else {
        // |g - f - t (c - f)| = t r: (d.d - r^2) t^2 - 2 (q.d) t + q.q = 0, a < 0, largest root
        const float qx = gx - g.geom[2], qy = gy - g.geom[3];
        const float dx = g.geom[0] - g.geom[2], dy = g.geom[1] - g.geom[3];
        const float r = g.geom[4];
        const float a = (dx * dx + dy * dy) - r * r;
        const float b = qx * dx + qy * dy;
        const float c = qx * qx + qy * qy;
        t = (b - sqrtf(b * b - a * c)) / a;
    }
    if (!(t == t)) t = 0.0f;
    if (!degenerate) {
        if (g.spread == kSpreadPad) {
            t = t < 0.0f ? 0.0f : (t > 1.0f ? 1.0f : t);
        } else if (g.spread == kSpreadRepeat) {
            t = t - floorf(t);
        } else if (g.spread == kSpreadReflect) {
            const float m = t - 2.0f * floorf(t * 0.5f);
            t = m > 1.0f ? 2.0f - m : m;
        } else if (t < 0.0f || t > 1.0f) {
            return 0u;  // transparent outside [0, 1]
        }
        if (!(t == t)) t = 0.0f;
    }
    const uint32_t n = g.n_stops;
    float c[4];
    if (t <= st[0]) {
        c[0] = st[1]; c[1] = st[2]; c[2] = st[3]; c[3] = st[4];
    } else if (t >= st[5 * (n - 1)]) {
        const float* e = st + 5 * (n - 1);
        c[0] = e[1]; c[1] = e[2]; c[2] = e[3]; c[3] = e[4];
    } else {
        uint32_t i = 0;
        while (i + 1 < n && st[5 * (i + 1)] <= t) ++i;  // off[i] <= t < off[i + 1]
        const float* e0 = st + 5 * i;
        const float* e1 = e0 + 5;
        const float f = (t - e0[0]) / (e1[0] - e0[0]);
#pragma unroll
        for (int k = 0; k < 4; ++k) c[k] = lerp(e0[1 + k], e1[1 + k], f);
    }
    c[3] = c[3] * g.opacity;
    uint32_t out = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const float vv = c[k] * 255.0f;
        const int iv = (vv != vv) ? 0 : (vv <= 0.0f ? 0 : (vv >= 255.0f ? 255 : (int)vv));
        out |= (uint32_t)iv << (8 * k);
    }
    return (out & 0xFF000000u) ? out : 0u;
}

// The colours of a pixel of each row of a cell row, from a paint and stops in memory (a paint
// with more stops than LDS holds).
__device__ __noinline__ uint2 paint_pair_far(const PaintArgs pa, uint32_t pi, float2 s0, float2 s1) {
    const Paint g = pa.paints[pi];
    const float* st = pa.stops + 5 * (size_t)g.first_stop;
    return make_uint2(paint_color(g, st, s0.x, s0.y), paint_color(g, st, s1.x, s1.y));
}

// (r*a, g*a, b*a, a) of a packed colour, as the blend uses it.
__device__ inline float4 premul(uint32_t col) {
    const float a = (float)((col >> 24) & 0xFFu) / 255.0f;
    return make_float4(((float)(col & 0xFFu) / 255.0f) * a, ((float)((col >> 8) & 0xFFu) / 255.0f) * a,
                       ((float)((col >> 16) & 0xFFu) / 255.0f) * a, a);
}

// A premultiplied colour times a coverage share.
__device__ inline float4 scale(const float4 s, float c) { return make_float4(s.x * c, s.y * c, s.z * c, s.w * c); }

__device__ inline void blend(float* d, const float4 sa) {
    const float ia = 1.0f - sa.w;
    d[0] = sa.x + d[0] * ia;
    d[1] = sa.y + d[1] * ia;
    d[2] = sa.z + d[2] * ia;
    d[3] = sa.w + d[3] * ia;
}

// The first workgroups of the launch: the cells and spans of the bands summed into totals, and, by the
// last of them to end, the frame's counters gathered into host memory.  (On their own the two were
// a launch each, and a copy.)
template <int BLOCK>
__device__ inline void tally(const TallyArgs& T) {
    __shared__ int32_t s_c[BLOCK / 64], s_s[BLOCK / 64];
    __shared__ uint32_t s_rank;
    const int tid = threadIdx.x;
    if (T.band_cnt) {
        const int32_t nb = *T.n_bands;
        int32_t c = 0, sp = 0;
        for (int32_t t = (int32_t)blockIdx.x * BLOCK + tid; t < nb; t += T.blocks * BLOCK) {
            const int2 v = T.band_cnt[t];
            c += v.x;
            sp += v.y;
        }
        c = wave_sum(c);
        sp = wave_sum(sp);
        if ((tid & 63) == 0) { s_c[tid >> 6] = c; s_s[tid >> 6] = sp; }
        __syncthreads();
        if (tid == 0) {
            int32_t tc = 0, ts = 0;
            for (int k = 0; k < BLOCK / 64; ++k) { tc += s_c[k]; ts += s_s[k]; }
            if (tc) atomicAdd(&T.totals[0], tc);
            if (ts) atomicAdd(&T.totals[1], ts);
            if (tc + ts) atomicAdd(&T.totals[2], tc + ts);
        }
    }
    if (tid == 0) {
        __threadfence();
        s_rank = atomicAdd(T.done, 1u);
    }
    __syncthreads();
    if (s_rank != (uint32_t)T.blocks - 1u || tid >= T.src.n) return;
    const int32_t* p = T.src.p[tid];
    const int32_t v = p ? __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0;
    __hip_atomic_store(&T.out[tid], v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

template <int COMPOSE, int GRAD, int AA, int PIX, int CHUNK>
__global__ __launch_bounds__(CHUNK / PIX) __attribute__((amdgpu_waves_per_eu(GRAD ? 1 : 4))) void k_composite(const uint32_t* __restrict__ records,
                                                      const int2* __restrict__ brec,
                                                      const int32_t* __restrict__ bucket_base,
                                                      const int2* __restrict__ prow,
                                                      const uint32_t* __restrict__ fill, uint32_t Np,
                                                      int w, int h, int64_t rec_cap,
                                                      uint8_t* __restrict__ image,
                                                      const DocDev* __restrict__ docs, int n_docs,
                                                      const PaintArgs pa,
                                                      const unsigned long long* __restrict__ cmask,
                                                      const TallyArgs T) {
    constexpr int TWO = (GRAD || AA) ? 1 : 0;            // the two rows of a cell row differ
    constexpr int BLOCK = CHUNK / PIX;                   // threads; each keeps PIX pixels, BLOCK columns apart
    static_assert(PIX <= 32 && PIX % (AA ? 4 : 2) == 0 && BLOCK % kListSub == 0, "composite shape");
    // Parts of a listing step.  Four at a time, their rows loaded a step ahead, took the composite of
    // 20,000 paths on 2048^2 from 70 to 58 us (one at a time: 79 steps that wait on two loads each);
    // the wide chunks have no registers left for that (4096^2, 5,000 paths: two parts 457 us, four 497,
    // four loaded ahead 542).
    constexpr bool kAhead = CHUNK <= 2048;
    constexpr int kListSubs = kAhead ? 4 : 2;
    constexpr int kCand = kListSub * kListSubs / BLOCK;  // candidate paths per thread of a listing step
    static_assert(kCand >= 1 && kList >= kListSub, "listing step");
    // partial coverage: entry k of column c at lslot[k * CHUNK + c], q | n0 << 6 | n1 << 11; byte c of
    // lcnt counts the column's entries
    __shared__ uint16_t lslot[AA ? kAaSlots * CHUNK : 1];
    __shared__ uint32_t lcnt[AA ? CHUNK / 4 : 1];
    __shared__ uint32_t lmore[AA ? kAaMore : 1];  // the others: column << 16 | entry
    __shared__ int32_t lmore_n;
    __shared__ u64 ev[CHUNK];
    __shared__ int2 list[kList];
    __shared__ uint32_t lcol[kList];
    __shared__ uint32_t lpaint[GRAD ? kList : 1];  // each listed path's paint (kSolidPaint: its colour)
    __shared__ u64 lgrad;                          // the batch's paths that have a paint
    __shared__ Paint lpnt[GRAD ? kBatch : 1];      // their paints (first_stop: the first in lstop, ~0: in memory)
    __shared__ float lstop[GRAD ? 5 * kStops : 1];
    __shared__ int32_t lfit;                       // paths of the batch whose stops fit in lstop
    __shared__ float4 lsa[kBatch];   // (r*a, g*a, b*a, a) of each path of the batch, as the blend uses them
    __shared__ u64 lopaque;                        // the batch's paths that hide what lies under them
    __shared__ int32_t wcount[kListSub * kListSubs / 64];
    __shared__ int32_t bpre[kBatch + 1];
    __shared__ u64 xlds[BLOCK / 64];
    if ((int)blockIdx.x < T.blocks) {
        if (blockIdx.y == 0) tally<BLOCK>(T);
        return;
    }
    int r = (int)blockIdx.x - T.blocks;
    uint32_t pbeg = 0, pend = Np;
    if (docs) {
        // batch: find this cell row's document (documents are numbered by first row)
        int lo = 0, hi = n_docs;
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (docs[mid].row0 <= r) lo = mid; else hi = mid;
        }
        const DocDev d = docs[lo];
        r -= d.row0;
        w = d.w; h = d.h;
        pbeg = (uint32_t)d.p0; pend = (uint32_t)d.p1;
        image += d.img_off;
    }
    const int y = 2 * r;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int c0 = (int)blockIdx.y * CHUNK;
    if (c0 >= w) return;  // a narrower document of a batch
    {
        const int cw = w - c0 < CHUNK ? w - c0 : CHUNK;
        uint32_t pix[PIX], pix1[TWO ? PIX : 1];  // rows y and, with paints or coverage, y + 1
        float acc[COMPOSE ? PIX : 1][4], acc1[(COMPOSE && TWO) ? PIX : 1][4];
#pragma unroll
        for (int j = 0; j < PIX; ++j) {
            pix[j] = 0xFFFFFFFFu;
            if constexpr (TWO != 0) pix1[j] = 0xFFFFFFFFu;
            if constexpr (COMPOSE != 0) { acc[j][0] = acc[j][1] = acc[j][2] = acc[j][3] = 1.0f; }
            if constexpr (COMPOSE != 0 && TWO != 0) { acc1[j][0] = acc1[j][1] = acc1[j][2] = acc1[j][3] = 1.0f; }
        }
        uint32_t p0 = pbeg;
        // the candidates' rows, loaded one listing step ahead
        int2 ahead[kCand];
        uint32_t ahead_p0 = ~0u;
        auto load_rows = [&](uint32_t from) {
            ahead_p0 = from;
#pragma unroll
            for (int u = 0; u < kCand; ++u) {
                const uint32_t p = from + (uint32_t)(u * BLOCK + tid);
                ahead[u] = p < pend ? prow[p] : make_int2(0, -2);  // no row, not even row 0
            }
        };
        while (p0 < pend) {
            // ordered list of the paths with records on this cell row, up to kListSub * kListSubs
            // candidates at a time until the list could overflow: batches are then full whatever the
            // path numbering
            int n = 0;
            while (p0 < pend && n + kListSub <= kList) {
                int2 rng[kCand];
                int at[kCand];
                if (!kAhead || ahead_p0 != p0) load_rows(p0);
#pragma unroll
                for (int u = 0; u < kCand; ++u) {
                    const int2 pr = ahead[u];
                    const int loc = r == 0 ? pr.y + 1 : ((r >= pr.x && r < pr.x + pr.y) ? r - pr.x : -1);
                    at[u] = loc >= 0 ? bucket_base[p0 + (uint32_t)(u * BLOCK + tid)] + loc : -1;
                }
                if (kAhead && p0 + kListSub * kListSubs < pend) load_rows(p0 + kListSub * kListSubs);
                u64 m[kCand];
#pragma unroll
                for (int u = 0; u < kCand; ++u) {
                    rng[u] = at[u] >= 0 ? brec[at[u]] : make_int2(0, 0);
                    // ranges never reach past the records actually stored (a frame whose record
                    // budget overflowed must still read in bounds)
                    rng[u].y = (int64_t)rng[u].y < rec_cap ? rng[u].y : (int32_t)rec_cap;
                    rng[u].x = rng[u].x < rng[u].y ? rng[u].x : rng[u].y;
                }
#pragma unroll
                for (int u = 0; u < kCand; ++u) {
                    m[u] = __ballot(rng[u].y > rng[u].x);
                    if (lane == 0) wcount[u * (BLOCK / 64) + wave] = (int32_t)__popcll(m[u]);
                }
                __syncthreads();
                // the parts that fit, the first one always
                int upto[kListSubs], fit = 0, add = 0;
#pragma unroll
                for (int k = 0; k < kListSubs; ++k) {
                    upto[k] = add;
                    int c = 0;
#pragma unroll
                    for (int v = 0; v < kListSub / 64; ++v) c += wcount[k * (kListSub / 64) + v];
                    if (fit == k && n + add + c <= kList) { ++fit; add += c; }
                }
#pragma unroll
                for (int u = 0; u < kCand; ++u) {
                    const int group = u * (BLOCK / 64) + wave, sub = group / (kListSub / 64);
                    if (sub < fit && rng[u].y > rng[u].x) {
                        int off = n;
#pragma unroll
                        for (int k = 0; k < kListSubs; ++k) off += k == sub ? upto[k] : 0;
                        for (int v = sub * (kListSub / 64); v < group; ++v) off += wcount[v];
                        const int slot = off + (int)__popcll(m[u] & ((1ull << lane) - 1ull));
                        const uint32_t p = p0 + (uint32_t)(u * BLOCK + tid);
                        list[slot] = rng[u];
                        lcol[slot] = fill[p];
                        if constexpr (GRAD != 0) lpaint[slot] = pa.path_paint[p];
                    }
                }
                __syncthreads();
                n += add;
                p0 += (uint32_t)(fit * kListSub);
            }
            int qn = 0;
            for (int q0 = 0; q0 < n; q0 += qn) {
                qn = n - q0 < kBatch ? n - q0 : kBatch;
            batch:
                if constexpr (AA != 0) {
                    for (int k = tid; k < CHUNK / 4; k += BLOCK) lcnt[k] = 0u;
                    if (tid == 0) lmore_n = 0;
                }
                // clear the event words; the batch's colours; its records as one flat index space
#pragma unroll
                for (int j = 0; j < PIX; ++j) ev[j * BLOCK + tid] = 0ull;
                if (wave == 0) {
                    if constexpr (COMPOSE != 0) {
                        bool opaque = false;
                        if (lane < qn) {
                            lsa[lane] = premul(lcol[q0 + lane]);
                            opaque = (lcol[q0 + lane] >> 24) == 255u;
                            if constexpr (GRAD != 0) opaque = opaque && lpaint[q0 + lane] == kSolidPaint;
                        }
                        const u64 om = __ballot(opaque);
                        if (lane == 0) lopaque = om;
                    }
                    if constexpr (GRAD != 0) {
                        const uint32_t pi = lane < qn ? lpaint[q0 + lane] : kSolidPaint;
                        const u64 gm = __ballot(pi != kSolidPaint);
                        if (lane == 0) lgrad = gm;
                        Paint g;
                        g.n_stops = 0;
                        if (pi != kSolidPaint) g = pa.paints[pi];
                        int upto = (int)min(g.n_stops, (uint32_t)kStops + 1u);
#pragma unroll
                        for (int d = 1; d < 64; d <<= 1) {
                            const int u = __shfl_up(upto, d);
                            if (lane >= d) upto += u;
                        }
                        // the paths up to the first whose stops no longer fit (that one alone, if
                        // it is the first: its stops stay in memory)
                        const u64 over = __ballot(upto > kStops);
                        const int fit = max(1, over ? __ffsll((long long)over) - 1 : 64);
                        if (lane == 0) lfit = fit;
                        if (pi != kSolidPaint && lane < fit) {
                            const float* src = pa.stops + 5 * (size_t)g.first_stop;
                            const int at = upto - (int)g.n_stops;
                            const bool near = upto <= kStops;
                            if (near)
                                for (uint32_t k = 0; k < 5u * g.n_stops; ++k) lstop[5 * at + (int)k] = src[k];
                            g.first_stop = near ? (uint32_t)at : ~0u;
                            lpnt[lane] = g;
                        }
                    }
                    const int2 rg = lane < qn ? list[q0 + lane] : make_int2(0, 0);
                    int inc = rg.y - rg.x;
#pragma unroll
                    for (int d = 1; d < 64; d <<= 1) {
                        const int u = __shfl_up(inc, d);
                        if (lane >= d) inc += u;
                    }
                    bpre[lane + 1] = inc;
                    if (lane == 0) bpre[0] = 0;
                }
                __syncthreads();
                if constexpr (GRAD != 0) qn = min(qn, lfit);
                const int total = bpre[qn];
                for (int f0 = tid; f0 < total; f0 += BLOCK * kUnroll) {
                    uint32_t rec[kUnroll];
                    int qi[kUnroll];
                    int64_t ri[kUnroll];
#pragma unroll
                    for (int u = 0; u < kUnroll; ++u) {
                        const int f = f0 + u * BLOCK;
                        qi[u] = -1;
                        if (f < total) {
                            int lo = 0, hi = qn;
                            while (hi - lo > 1) {
                                const int mid = (lo + hi) >> 1;
                                if (bpre[mid] <= f) lo = mid; else hi = mid;
                            }
                            qi[u] = lo;
                            ri[u] = (int64_t)list[q0 + lo].x + (f - bpre[lo]);
                            rec[u] = records[ri[u]];
                        }
                    }
#pragma unroll
                    for (int u = 0; u < kUnroll; ++u) {
                        if (qi[u] < 0) continue;
                        const u64 bit = 1ull << qi[u];
                        int xs = (int)(rec[u] & 0xFFFFu) - c0;
                        int xe = xs + (int)(rec[u] >> 16);
                        xs = xs < 0 ? 0 : xs;
                        xe = xe > cw ? cw : xe;
                        if (xs < xe) {
                            atomicXor(&ev[ev_slot<PIX>(xs)], bit);
                            if (xe < cw) atomicXor(&ev[ev_slot<PIX>(xe)], bit);  // ends past the chunk change nothing
                        }
                        if constexpr (AA != 0) {
                            const unsigned long long cm = cmask[ri[u]];
                            if (cm != ~0ull) {  // a boundary cell (2 wide): its pixels' sample counts
                                const int x0 = (int)(rec[u] & 0xFFFFu) - c0;
#pragma unroll
                                for (int px = 0; px < 2; ++px) {
                                    const int col = x0 + px;
                                    if (col < 0 || col >= cw) continue;
                                    const uint32_t n0 = __popcll((cm >> (16 * px)) & 0xFFFFull);
                                    const uint32_t n1 = __popcll((cm >> (16 * (2 + px))) & 0xFFFFull);
                                    const uint32_t k = (atomicAdd(&lcnt[col >> 2], 1u << (8 * (col & 3))) >>
                                                        (8 * (col & 3))) & 0xFFu;
                                    const uint32_t e = (uint32_t)qi[u] | (n0 << 6) | (n1 << 11);
                                    if (k < (uint32_t)kAaSlots) {
                                        lslot[k * CHUNK + col] = (uint16_t)e;
                                    } else {
                                        const int at = atomicAdd(&lmore_n, 1);
                                        if (at < kAaMore) lmore[at] = ((uint32_t)col << 16) | e;
                                    }
                                }
                            }
                        }
                    }
                }
                __syncthreads();
                if constexpr (AA != 0) {
                    if (lmore_n > kAaMore) {  // more partial cells than the lists hold: fewer paths
                        qn = qn / 2;
                        __syncthreads();
                        goto batch;
                    }
                }
                // coverage = prefix XOR of the events, each thread over PIX consecutive columns
                {
                    u64 run = 0;
#pragma unroll
                    for (int j = 0; j < PIX; ++j) run ^= ev[ev_slot<PIX>(tid * PIX + j)];
                    u64 cov = block_exclusive_xor<BLOCK>(run, xlds);
#pragma unroll
                    for (int j = 0; j < PIX; ++j) {
                        u64* e = &ev[ev_slot<PIX>(tid * PIX + j)];
                        cov ^= *e;
                        *e = cov;
                    }
                }
                __syncthreads();
                // the fold in path order, consecutive columns in consecutive lanes: they are mostly
                // covered by the same paths, so the lanes of a wave take the same number of steps and
                // read the same colours
                const u64 gmask = GRAD ? lgrad : 0ull;
                const u64 omask = COMPOSE ? lopaque : 0ull;
#pragma unroll
                for (int j = 0; j < PIX; ++j) {
                    const int c = j * BLOCK + tid;
                    u64 mm = ev[ev_slot<PIX>(c)];
                    if (mm == 0ull) continue;
                    // the scene points of the pixel's centres, for its gradients
                    float2 g0, g1;
                    auto pair = [&](int k) -> uint2 {  // colours of path k of the batch
                        const Paint& g = lpnt[k];
                        if (g.first_stop == ~0u) return paint_pair_far(pa, lpaint[q0 + k], g0, g1);
                        const float* st = lstop + 5 * g.first_stop;
                        return make_uint2(paint_color(g, st, g0.x, g0.y), paint_color(g, st, g1.x, g1.y));
                    };
                    if constexpr (GRAD != 0) {
                        if (mm & gmask) {
                            const int x = c0 + c;  // the pixel's canvas column
                            g0 = scene_point(pa.inv, x, y);
                            g1 = scene_point(pa.inv, x, y + 1);
                        }
                    }
                    // this pixel's partial-coverage entries (AA), and the paths they belong to
                    uint32_t pe[AA ? kAaSlots : 1];
                    uint32_t np = 0;
                    u64 pm = 0ull;
                    if constexpr (AA != 0) {
                        np = (lcnt[c >> 2] >> (8 * (c & 3))) & 0xFFu;
#pragma unroll
                        for (int k = 0; k < kAaSlots; ++k) pe[k] = 0u;
                        if (np) {
#pragma unroll
                            for (int k = 0; k < kAaSlots; ++k) {
                                if ((uint32_t)k < np) {
                                    pe[k] = (uint32_t)lslot[k * CHUNK + c];
                                    pm |= 1ull << (pe[k] & 63u);
                                }
                            }
                            if (np > (uint32_t)kAaSlots)
                                for (int i = 0; i < lmore_n; ++i)
                                    if ((int)(lmore[i] >> 16) == c) pm |= 1ull << (lmore[i] & 63u);
                        }
                    }
                    if constexpr (COMPOSE == 0) {
                        const int q = 63 - __clzll((long long)mm);
                        if (GRAD && ((gmask >> q) & 1ull)) {
                            const uint2 pc = pair(q);
                            pix[j] = pc.x;
                            pix1[j] = pc.y;
                        } else {
                            pix[j] = lcol[q0 + q];
                            if constexpr (GRAD != 0) pix1[j] = pix[j];
                        }
                    } else {
                        // what lies under an opaque path changes nothing: with a = 1, d = s + d * 0 = s
                        if (omask) {
                            const u64 mo = mm & omask & ~pm;
                            if (mo) mm &= ~0ull << (63 - __clzll((long long)mo));
                        }
                        // src-over, d = s*a + d*(1-a) per channel, the paths in order
                        // the mask's two words in turn: 32-bit bit scans and clears
#pragma unroll
                        for (int hw = 0; hw < 2; ++hw) {
                            uint32_t m32 = (uint32_t)(mm >> (32 * hw));
                            const float4* L = lsa + 32 * hw;
                            while (m32) {
                                const int q = __builtin_ctz(m32);
                                m32 &= m32 - 1u;
                                if constexpr (TWO != 0) {
                                    float4 s0 = L[q], s1 = L[q];
                                    if (GRAD && ((gmask >> (32 * hw + q)) & 1ull)) {
                                        const uint2 pc = pair(32 * hw + q);
                                        s0 = premul(pc.x);
                                        s1 = premul(pc.y);
                                    }
                                    if constexpr (AA != 0) {
                                        const uint32_t qq = (uint32_t)(32 * hw + q);
                                        if ((pm >> qq) & 1ull) {
                                            uint32_t e = 0;
#pragma unroll
                                            for (int k = 0; k < kAaSlots; ++k)
                                                if ((uint32_t)k < np && (pe[k] & 63u) == qq) e = pe[k];
                                            if (np > (uint32_t)kAaSlots)
                                                for (int i = 0; i < lmore_n; ++i)
                                                    if (lmore[i] >> 16 == (uint32_t)c && (lmore[i] & 63u) == qq) e = lmore[i];
                                            s0 = scale(s0, (float)((e >> 6) & 31u) / 16.0f);
                                            s1 = scale(s1, (float)((e >> 11) & 31u) / 16.0f);
                                        }
                                    }
                                    blend(acc[j], s0);
                                    blend(acc1[j], s1);
                                } else {
                                    blend(acc[j], L[q]);
                                }
                            }
                        }
                    }
                }
                __syncthreads();
            }
        }
        auto round8 = [](const float* a) -> uint32_t {
            uint32_t o = 0;
#pragma unroll
            for (int ch = 0; ch < 4; ++ch) {
                float q = a[ch] * 255.0f + 0.5f;
                q = q < 0.0f ? 0.0f : (q > 255.0f ? 255.0f : q);
                o |= (uint32_t)q << (8 * ch);
            }
            return o;
        };
        if constexpr (COMPOSE != 0) {
#pragma unroll
            for (int j = 0; j < PIX; ++j) {
                pix[j] = round8(acc[j]);
                if constexpr (TWO != 0) pix1[j] = round8(acc1[j]);
            }
        }
        for (int yy = y; yy < y + 2 && yy < h; ++yy) {
            uint32_t* row = reinterpret_cast<uint32_t*>(image) + (int64_t)(h - 1 - yy) * w + c0;
#pragma unroll
            for (int j = 0; j < PIX; ++j) {
                const int c = j * BLOCK + tid;
                uint32_t out = pix[j];
                if constexpr (TWO != 0) out = yy == y ? pix[j] : pix1[j];
                if (c < cw) row[c] = out;
            }
        }
        __syncthreads();
    }
}

}  // namespace

// Chunk and pixels per thread by the widest row: the narrowest of 512, 1024 and 2048 columns in
// workgroups of 256 threads that holds it, else 4096 columns at 8 pixels per thread (512 threads; with
// coverage two rows of accumulators, 128 VGPRs, 4 waves per SIMD, and 27 VGPRs spilled, 112 bytes a
// lane).  Above kFewPaths paths, where
// listing them is most of the work, src-over takes 16 pixels in 256 threads.  4096^2, three frames in
// turn: 5,000 paths 2.33 ms against 2.48 with 16 (6 VGPRs spilled), 20,000 glyphs 370 us against 330; the
// line lies somewhere between these two, and what it stands for is the paths on a row.  Overwrite takes
// 16 (its pixels need one register each).  With paints always 1024 columns at 4 per thread.
constexpr uint32_t kFewPaths = 8192;
hipError_t launch_composite(const uint32_t* records, const int2* brec, const int32_t* bucket_base,
                            const int2* prow, const uint32_t* fill, uint32_t Np, int w, int h, int compose,
                            uint8_t* image, hipStream_t s, int64_t rec_cap, const DocDev* docs, int n_docs,
                            int total_rows, const PaintArgs* paint, const unsigned long long* cmask, const TallyArgs* tally) {
    const TallyArgs T = tally ? *tally : TallyArgs{};
    int rows = docs ? total_rows : (h + 1) / 2;
    if (w == 0) rows = 0;
    if (rows + T.blocks == 0) return hipSuccess;
    if (rows == 0) w = 1;  // the tally alone
    if (cmask && !compose) return hipErrorInvalidValue;  // coverage needs the src-over blend
    const PaintArgs pa = paint ? *paint : PaintArgs{nullptr, nullptr, nullptr, nullptr};
#define SPR_COMPOSITE(C, G, A, PIX, CHUNK)                                                                      \
    k_composite<C, G, A, PIX, CHUNK><<<dim3((unsigned)(rows + T.blocks), (unsigned)((w + (CHUNK) - 1) / (CHUNK))), (CHUNK) / (PIX), 0, s>>>( \
        records, brec, bucket_base, prow, fill, Np, w, h, rec_cap, image, docs, n_docs, pa, cmask, T)
    if (paint) {
        if (cmask) SPR_COMPOSITE(1, 1, 1, 4, 1024);
        else if (compose) SPR_COMPOSITE(1, 1, 0, 4, 1024);
        else SPR_COMPOSITE(0, 1, 0, 4, 1024);
    } else if (cmask) {
        if (w <= 1024) SPR_COMPOSITE(1, 0, 1, 4, 1024);
        else if (w <= 2048) SPR_COMPOSITE(1, 0, 1, 8, 2048);
        else SPR_COMPOSITE(1, 0, 1, 8, 4096);
    } else if (compose) {
        if (w <= 512) SPR_COMPOSITE(1, 0, 0, 2, 512);
        else if (w <= 1024) SPR_COMPOSITE(1, 0, 0, 4, 1024);
        else if (w <= 2048) SPR_COMPOSITE(1, 0, 0, 8, 2048);
        else if (Np <= kFewPaths) SPR_COMPOSITE(1, 0, 0, 8, 4096);
        else SPR_COMPOSITE(1, 0, 0, 16, 4096);
    } else {
        if (w <= 512) SPR_COMPOSITE(0, 0, 0, 2, 512);
        else if (w <= 1024) SPR_COMPOSITE(0, 0, 0, 4, 1024);
        else if (w <= 2048) SPR_COMPOSITE(0, 0, 0, 8, 2048);
        else SPR_COMPOSITE(0, 0, 0, 16, 4096);
    }
#undef SPR_COMPOSITE
    return hipGetLastError();
}

}  // namespace spr
