// k_aa.hip -- anti-aliased coverage of the boundary cells (gfx950).
//
// No reference counterpart: the reference leaves the boundary fragments' "comb-like
// multisampling" stencil mask TODO (gen_fragment.comp:202); its draw would fetch one mask per
// cell record (scanlinepr.vert:48-50, draw.w - 1) and set gl_SampleMask from it
// (scanlinepr.frag:13-14), and today sets all samples.  Here every boundary cell record gets a
// 64-bit mask: 16 samples in each of its 2x2 pixels, sample j of a pixel at
// ((7j mod 16) + 1/2)/16 across and (j + 1/2)/16 up (each sample row and column used once, an
// N-rooks "comb"), bit (2 py + px) * 16 + j.  Spans keep full coverage: a pixel that no edge of
// the path crosses lies in no boundary cell of that path, so the winding number is constant over
// it.
//
// The path inside a cell is its chord polygon (the segments pf -> pl between consecutive
// intersections, as gen_fragment forms them; the fragment stage stores them for these frames).
// The winding number at a sample is the cell's
// centre-row winding number at its left edge (the exclusive scan at the cell's first sorted
// entry), plus the changes met on the way to the sample: along the centre row to the sample's
// column, the winding change of each chord crossing the row (gen_fragment's half-open rule),
// then along that column to the sample's height, +1 for a chord going right and -1 for a chord
// going left when moving up (the reverse when moving down).  Both legs stay inside the cell, so
// only the cell's own chords (one sorted run of entries) are met.
//
// k_cell_cover gives spans their full masks, computes which samples each chord changes, one lane
// per chord, and adds those up per cell, one lane per cell.  Every float expression has a fixed
// operation order (no contraction).
#include "device_common.hpp"
#include "kernels.hpp"
#include "scan_common.hpp"

namespace spr {

namespace {

constexpr int kBlock = 256;
constexpr int kRecs = 4;                // records per thread and pass
constexpr int kChunk = kRecs * kBlock;  // records per workgroup pass of the cover kernel
// Cells of up to kRunMax chords (the run of sorted entries with the cell's key and path) keep what
// their chords change in LDS; the cells of more come in a list, and a wave covers each.
constexpr int kRunMax = kAaRunMax;
constexpr int kDenseBlocks = 256;       // workgroups of the listed cells, in front of the others
constexpr int kSlots = 5 * kBlock;      // chords in LDS at a time, besides the last cell's overhang
constexpr uint32_t kNoEntry = 0xFFFFFFFFu;
static_assert(kChunk <= 1024 && kRunMax < 32 && kChunk * kRunMax < 65536, "cell words");
static_assert(kSlots >= 256 * (kBlock / 64), "words of the waves' listed cells");

// Columns c of two pixels (32 of them, sample x = x0 + (c + 1/2) / 16) whose sample x lies above z:
// those from the returned one on.  x32 = 32 x0, an integer below 2^20.  All values are exact: x > z
// when the odd integer x32 + 2c + 1 lies above 32 z, that is above its floor.  No sample lies above a
// NaN.
__device__ inline int first_above(float z, float x32) {
    const float k = fmaxf(fminf(floorf(32.0f * z), x32 + 64.0f), x32 - 1.0f) - x32;  // -1 .. 64
    return ((int)k + 1) >> 1;                                                        // 0 .. 32
}
__device__ inline uint32_t columns_from(int first) { return first < 32 ? 0xFFFFFFFFu << first : 0u; }

// What a chord changes in a cell's 64 samples:
//  - the centre-row crossing adds its change to the columns whose xs lies above its x, in both rows;
//  - a chord spanning column c (ax < xs <= bx or bx < xs <= ax) crosses it at height
//    yx = ay + (xs - ax) * slope, which counts in the upper pixel when yc <= yx < ys and in the
//    lower one (with the opposite sign) when ys < yx <= yc.
// head: first column of the crossing's change | 64 when it is -1 | 128 when the chord goes right;
// low, high: bit c set when column c's sample of the lower, upper pixel row (sample j = 7c mod 16 of a
// pixel sits in its column c, (7 * 7) mod 16 = 1) changes.
struct ChordBits {
    uint32_t head, low, high;
};
__device__ inline ChordBits chord_bits(const float4 ch, int32_t key) {
    const int rx = (key & 0xFFFF) - 0x7FFF, ry = ((key >> 16) & 0xFFFF) - 0x7FFF;
    const float y0 = (float)ry, yc = y0 + 1.0f, x0 = (float)rx, x32 = 32.0f * x0;
    const float ax = ch.x, ay = ch.y, bx = ch.z, by = ch.w;
    const bool down = ay < yc && yc <= by, up = by < yc && yc <= ay;
    const float xc = ax + (yc - ay) * ((bx - ax) / (by - ay));  // meaningless when the row is not crossed
    const bool rightward = ax < bx;
    const float lo = rightward ? ax : bx, hi = rightward ? bx : ax;
    // a NaN end fails the tests on the heights below
    const uint32_t span = columns_from(first_above(lo, x32)) & ~columns_from(first_above(hi, x32));
    const float sl = (by - ay) / (bx - ax);
    uint32_t low = 0u, high = 0u;
#pragma unroll
    for (int c = 31; c >= 0; --c) {
        const float xs = x0 + ((float)c + 0.5f) / 16.0f;
        // the height above the cell's lower edge, an even integer >= 0: exact inside the cell (it is
        // 0, or the height lies within a factor of two of it), and rounding keeps the order outside
        const float v = (ay + (xs - ax) * sl) - y0;
        const float yl = ((float)((7 * (c & 15)) & 15) + 0.5f) / 16.0f, yu = yl + 1.0f;  // the column's samples
        // no short circuit: no branches
        low = low + low + (uint32_t)((yl < v) & (v <= 1.0f));
        high = high + high + (uint32_t)((1.0f <= v) & (v < yu));
    }
    ChordBits r;
    r.head = (uint32_t)((down || up) ? first_above(xc, x32) : 32) | (down ? 64u : 0u) | (rightward ? 128u : 0u);
    r.low = low & span;
    r.high = high & span;
    return r;
}

// Winding numbers of the 32 samples of one pixel row of a cell, less a common start: plane p
// holds bit p of every sample's number (two's complement).
template <int PLANES>
struct Planes {
    uint32_t w[PLANES];
    // adds +1 (or -1 where neg) to the samples of m
    __device__ void add(uint32_t m, bool neg) {
        const uint32_t s = neg ? 0xFFFFFFFFu : 0u;
#pragma unroll
        for (int p = 0; p < PLANES; ++p) {
            const uint32_t carry = (w[p] ^ s) & m;
            w[p] ^= m;
            m = carry;
        }
    }
};

// The mask of a cell from the changes of its n chords at head[0..n), low[..], high[..] in LDS.
// PLANES: 2^(PLANES - 1) > 2 n.
template <int PLANES>
__device__ inline unsigned long long cell_mask(const uint32_t* head, const uint32_t* low, const uint32_t* high, int n,
                                               int32_t w0, bool even_odd) {
    Planes<PLANES> W[2];
#pragma unroll
    for (int p = 0; p < PLANES; ++p) W[0].w[p] = W[1].w[p] = 0u;
#pragma unroll 1
    for (int k = 0; k < n; ++k) {
        const uint32_t e = head[k];
        const uint32_t right = columns_from((int)(e & 63u));
        W[0].add(right, (e & 64u) != 0u);
        W[1].add(right, (e & 64u) != 0u);
        W[0].add(low[k], (e & 128u) != 0u);
        W[1].add(high[k], (e & 128u) == 0u);
    }
    // inside: an odd winding number, or one that is not 0 (its plane bits differ from those of -w0)
    const int32_t z = (int32_t)(0u - (uint32_t)w0);
    const bool out_of_reach = z >= (1 << (PLANES - 1)) || z < -(1 << (PLANES - 1));
    unsigned long long m = 0ull;
#pragma unroll
    for (int row = 0; row < 2; ++row) {
        uint32_t in = W[row].w[0] ^ ((w0 & 1) ? 0xFFFFFFFFu : 0u);
        if (!even_odd) {
            in = out_of_reach ? 0xFFFFFFFFu : 0u;
#pragma unroll
            for (int p = 0; p < PLANES; ++p) in |= W[row].w[p] ^ (((z >> p) & 1) ? 0xFFFFFFFFu : 0u);
        }
        // column c holds sample 7c mod 16 of its pixel: bits (2 py + px) * 16 .. + 15 of the mask
        uint32_t r = 0u;
#pragma unroll
        for (int c = 0; c < 16; ++c) r |= ((in >> c) & 0x10001u) << ((7 * c) & 15);
        m |= (unsigned long long)r << (32 * row);
    }
    return m;
}

// Orders within one wave: LDS written by some lanes and then read by others.
__device__ inline void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// A cell of any number of chords by a whole wave, 64 chords at a time: each chord's own values one lane per
// chord, into the wave's words of `at` and `of` (LDS, four and three rows of 64), then what the chords change
// one sample per lane (lane = its bit in the mask).  All lanes take part.
__device__ inline unsigned long long cover_dense(int32_t f, const int32_t* __restrict__ skey,
                                                const int32_t* __restrict__ sidx,
                                                const int32_t* __restrict__ winding,
                                                const uint32_t* __restrict__ epath,
                                                const float4* __restrict__ chord, int64_t N,
                                                const uint32_t* __restrict__ rule, uint32_t* at, uint32_t* of) {
    const int lane = threadIdx.x & 63;
    const int32_t key = skey[f];
    const uint32_t path = epath[f] & 0x3FFFFFFFu;
    const int rx = (key & 0xFFFF) - 0x7FFF, ry = ((key >> 16) & 0xFFFF) - 0x7FFF;
    const int j = lane & 15, px = (lane >> 4) & 1, py = lane >> 5;
    const float yc = (float)(ry + 1);
    const float xs = (float)(rx + px) + ((float)((7 * j) & 15) + 0.5f) / 16.0f;
    const float ys = (float)(ry + py) + ((float)j + 0.5f) / 16.0f;
    const bool upper = py != 0;
    int32_t W = winding[f];
    int n = 64;
    for (int64_t g0 = f; n == 64; g0 += 64) {
        const int64_t g = g0 + lane;
        const bool own = g < N && skey[g] == key && (epath[g] & 0x3FFFFFFFu) == path;
        const unsigned long long other = __ballot(!own);
        n = other ? __ffsll((long long)other) - 1 : 64;
        if (own) {
            const float4 ch = chord[sidx[g]];
            const float ax = ch.x, ay = ch.y, bx = ch.z, by = ch.w;
            const int sr = (ay < yc && yc <= by) ? -1 : ((by < yc && yc <= ay) ? 1 : 0);
            const bool rightward = ax < bx;
            at[lane] = fbits(ax + (yc - ay) * ((bx - ax) / (by - ay)));
            at[64 + lane] = fbits(rightward ? ax : bx);
            at[128 + lane] = fbits(rightward ? bx : ax);
            at[192 + lane] = (uint32_t)(sr + 1) | (rightward ? 4u : 0u);
            of[lane] = fbits(ax);
            of[64 + lane] = fbits(ay);
            of[128 + lane] = fbits((by - ay) / (bx - ax));
        }
        wave_sync();
        // four chords a step, their words loaded together; those past the last one change nothing
        for (int k = 0; k < n; k += 4) {
            float xc[4], lo[4], hi[4], ax[4], ay[4], sl[4];
            uint32_t e[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                xc[u] = bitsf(at[k + u]); lo[u] = bitsf(at[64 + k + u]); hi[u] = bitsf(at[128 + k + u]);
                e[u] = at[192 + k + u];
                ax[u] = bitsf(of[k + u]); ay[u] = bitsf(of[64 + k + u]); sl[u] = bitsf(of[128 + k + u]);
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const float v = ay[u] + (xs - ax[u]) * sl[u];
                // no short circuit: no branches
                const bool in = (lo[u] < xs) & (xs <= hi[u]);
                const bool hit = in & (((ys < v) & (v <= yc) & !upper) | ((yc <= v) & (v < ys) & upper));
                const int32_t row = ((int)(e[u] & 3u) - 1) & -(int)(xs > xc[u]);
                const int32_t column = (1 - 2 * (int)((e[u] >> 2) ^ (uint32_t)py)) & -(int)hit;
                W = wadd(W, (row + column) & -(int)(k + u < n));
            }
        }
        wave_sync();  // the words are used again
    }
    return __ballot(rule[path] == 1u ? (W & 1) != 0 : W != 0);
}

// Four entries from f on, in one load each; those at or beyond N (N > f) repeat the last one.
struct Four {
    int32_t key[4];
    uint32_t path[4];
};
__device__ inline Four four_entries(int64_t f, const int32_t* __restrict__ skey, const uint32_t* __restrict__ epath,
                                    int64_t N) {
    Four q;
    if (f + 4 <= N) {
        __builtin_memcpy(q.key, skey + f, 16);  // 4-byte aligned: global_load_dwordx4 takes that
        __builtin_memcpy(q.path, epath + f, 16);
    } else {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int64_t g = f + u < N ? f + u : N - 1;
            q.key[u] = skey[g];
            q.path[u] = epath[g];
        }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) q.path[u] &= 0x3FFFFFFFu;
    return q;
}

// The number of chords of the cell whose run starts at entry f with the entries q, or more than
// kRunMax.
__device__ inline int run_length(int32_t f, const Four& q, const int32_t* __restrict__ skey,
                                 const uint32_t* __restrict__ epath, int64_t N) {
    int k = 0;
    Four at = q;
    for (;;) {
        int n = 0;
#pragma unroll
        for (int u = 0; u < 4; ++u)
            n += n == u && f + k + u < N && at.key[u] == q.key[0] && at.path[u] == q.path[0] ? 1 : 0;
        k += n;
        if (n < 4 || k > kRunMax || f + k >= N) return k;
        at = four_entries((int64_t)f + k, skey, epath, N);
    }
}

// A workgroup takes kChunk records at a time.  The chords of its cells are laid out in LDS, kSlots at a
// time and each cell's side by side, and every lane computes the changes of one chord (all lanes the
// same straight line of about 550 instructions, the next chord on its way); then every lane adds up
// the changes of one cell (about 40 instructions a chord).  Bound by that arithmetic.  On 48.7 M chords in
// 36.6 M cells of a 4096^2 frame 1.43 ms (1.21 with the dense cells in a list, below).  Four lanes per cell
// with 16 integer winding numbers each, every lane walking the cell's chords: 2.5 ms; one lane per cell with the
// bits below: 1.9 ms, of which 0.4 ms were arithmetic, since the longest cell of a wave held the other lanes back
// and each of its chords waited on two dependent loads.  Five waves per SIMD: four or six were 6% slower.
// Cells of more than kRunMax chords are few, but lie side by side (a path's dense spots): taken by the waves
// whose records they were, one after another, 54 of them made this kernel 534 us instead of 130 in a
// drawing at four times its size.  k_mark_emit lists them, and waves of their own spread over the chip.
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(5)))
void k_cell_cover(const int32_t* __restrict__ cell_first, const int32_t* __restrict__ totals, int64_t rec_cap,
                  const int32_t* __restrict__ skey, const int32_t* __restrict__ sidx,
                  const int32_t* __restrict__ winding, const uint32_t* __restrict__ epath,
                  const float4* __restrict__ chord, int64_t N, const uint32_t* __restrict__ rule,
                  unsigned long long* __restrict__ cmask, const int2* __restrict__ dense,
                  const int32_t* __restrict__ n_dense) {
    // per chord: its entry and its cell's key, then its ChordBits
    __shared__ uint32_t s_head[kSlots + kRunMax], s_low[kSlots + kRunMax], s_high[kSlots + kRunMax];
    // per cell: place of its chords | chords << 16 | even-odd << 21 | record << 22, winding number
    __shared__ uint2 s_cell[kChunk];
    __shared__ int32_t s_wave[kBlock / 64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (blockIdx.x < kDenseBlocks) {
        const int32_t nd = *n_dense;
        for (int32_t i = (int32_t)blockIdx.x + kDenseBlocks * wave; i < nd; i += kDenseBlocks * (kBlock / 64)) {
            const int2 d = dense[i];
            const unsigned long long m = cover_dense(__builtin_amdgcn_readfirstlane(d.y), skey, sidx, winding, epath,
                                                     chord, N, rule, s_head + 256 * wave, s_low + 256 * wave);
            if (lane == 0) cmask[d.x] = m;
        }
        return;
    }
    const int64_t R = min((int64_t)totals[0] + (int64_t)totals[1], rec_cap);
    const int64_t stride = (int64_t)(gridDim.x - kDenseBlocks) * kChunk;
    for (int64_t c0 = (int64_t)(blockIdx.x - kDenseBlocks) * kChunk; c0 < R; c0 += stride) {
        // what a cell needs of its entries, all records of a thread at once (a span loads entry 0)
        int32_t fr[kRecs], key[kRecs];
        int n[kRecs], at[kRecs];
        uint2 cell[kRecs];
        {
            Four q[kRecs];
#pragma unroll
            for (int u = 0; u < kRecs; ++u) {
                const int64_t o = c0 + u * kBlock + tid;
                fr[u] = o < R ? cell_first[o] : -1;
                if (o < R && fr[u] < 0) cmask[o] = ~0ull;  // a span: every sample
            }
#pragma unroll
            for (int u = 0; u < kRecs; ++u) {
                q[u] = four_entries(max(fr[u], 0), skey, epath, N);
                cell[u].y = (uint32_t)winding[max(fr[u], 0)];
            }
#pragma unroll
            for (int u = 0; u < kRecs; ++u) {
                cell[u].x = (rule[q[u].path[0]] == 1u ? 1u << 21 : 0u) | ((uint32_t)(u * kBlock + tid) << 22);
                key[u] = q[u].key[0];
            }
#pragma unroll
            for (int u = 0; u < kRecs; ++u) n[u] = fr[u] >= 0 ? run_length(fr[u], q[u], skey, epath, N) : 0;
        }
        int mine = 0;  // chords | cells << 16
#pragma unroll
        for (int u = 0; u < kRecs; ++u) {
            if (n[u] > kRunMax) n[u] = 0;  // listed
            mine += n[u] + (n[u] > 0 ? 1 << 16 : 0);
        }
        // the cells' places among the chunk's chords
        const int upto = wave_inclusive_add(mine);
        if (lane == 63) s_wave[wave] = upto;
        __syncthreads();
        int off = upto - mine, all = 0;
#pragma unroll
        for (int k = 0; k < kBlock / 64; ++k) {
            if (k < wave) off += s_wave[k];
            all += s_wave[k];
        }
        const int total = all & 0xFFFF, cells = all >> 16;
#pragma unroll
        for (int u = 0; u < kRecs; ++u) {
            at[u] = off & 0xFFFF;
            if (n[u] > 0) {
                s_cell[off >> 16] = make_uint2(cell[u].x | (uint32_t)at[u] | ((uint32_t)n[u] << 16), cell[u].y);
                off += n[u] + (1 << 16);
            }
        }
        for (int t0 = 0; t0 < total; t0 += kSlots) {
            // the cells that start in [t0, t0 + kSlots), whole; slots of other rounds' cells hold none
            if (total > kSlots) {
                if (tid < kRunMax) s_head[tid] = s_head[kSlots + tid] = kNoEntry;
                __syncthreads();
            }
#pragma unroll
            for (int u = 0; u < kRecs; ++u)
                if (at[u] >= t0 && at[u] < t0 + kSlots)
                    for (int k = 0; k < n[u]; ++k) {
                        s_head[at[u] - t0 + k] = (uint32_t)(fr[u] + k);
                        s_low[at[u] - t0 + k] = (uint32_t)key[u];
                    }
            __syncthreads();
            const int count = min(total - t0, kSlots + kRunMax);
            // the chord one step ahead, its index two (entry 0 where there is none)
            auto index = [&](int i) -> int32_t {
                const uint32_t e = i < count ? s_head[i] : kNoEntry;
                return sidx[e == kNoEntry ? 0u : e];
            };
            float4 ch = chord[index(tid)];
            int32_t next = index(tid + kBlock);
#pragma unroll 1
            for (int i = tid; i < count; i += kBlock) {
                const float4 ahead = chord[next];
                next = index(i + 2 * kBlock);
                if (s_head[i] != kNoEntry) {
                    const ChordBits b = chord_bits(ch, (int32_t)s_low[i]);
                    s_head[i] = b.head;
                    s_low[i] = b.low;
                    s_high[i] = b.high;
                }
                ch = ahead;
            }
            __syncthreads();
#pragma unroll 1
            for (int t = tid; t < cells; t += kBlock) {
                const uint2 c = s_cell[t];
                const int i = (int)(c.x & 0xFFFFu) - t0, m = (int)((c.x >> 16) & 31u);
                const bool on = i >= 0 && i < kSlots;
                const bool many = __any(on && m > 3);
                if (on) {
                    const bool odd = (c.x & (1u << 21)) != 0u;
                    const int32_t w0 = (int32_t)c.y;
                    cmask[c0 + (c.x >> 22)] = many ? cell_mask<7>(s_head + i, s_low + i, s_high + i, m, w0, odd)
                                                   : cell_mask<4>(s_head + i, s_low + i, s_high + i, m, w0, odd);
                }
            }
            __syncthreads();
        }
        if (total == 0) __syncthreads();  // s_wave is used again
    }
}

}  // namespace

hipError_t launch_cell_cover(const int32_t* cell_first, const int32_t* totals, int64_t rec_cap,
                             const int32_t* skey, const int32_t* sidx, const int32_t* winding,
                             const uint32_t* epath, const float4* chord, int64_t N, const uint32_t* rule,
                             unsigned long long* cmask, const int2* dense, const int32_t* n_dense, hipStream_t s) {
    if (rec_cap <= 0 || N <= 0) return hipSuccess;
    int64_t g = (rec_cap + kChunk - 1) / kChunk;
    g = g < 65536 ? g : 65536;  // few passes each: passes differ in cost (3% faster than 4,096 workgroups)
    k_cell_cover<<<(unsigned)g + kDenseBlocks, kBlock, 0, s>>>(cell_first, totals, rec_cap, skey, sidx, winding, epath, chord, N,
                                                rule, cmask, dense, n_dense);
    return hipGetLastError();
}

}  // namespace spr
