// k_geometry.hip -- transform + cull, monotonisation + count, and fragment-key generation
// (gfx950).  The intersection write between count and keys lives in k_curves.hip.
#include "device_common.hpp"
#include "kernels.hpp"
#include "scan_common.hpp"
#include "wave_solve.hpp"

namespace spr {

namespace {

constexpr int kBlock = 256;

inline unsigned grid_for(int64_t n, int block = kBlock) {
    int64_t g = (n + block - 1) / block;
    return (unsigned)(g < 1 ? 1 : g);
}

__global__ void k_fill_u32(uint32_t* __restrict__ p, int64_t n, uint32_t v) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        p[i] = v;
}

// Clears what the second half of a frame counts in, finds the curve that holds each window's
// first entry and holds the exact total against the budget: one launch for all of it.
__global__ __launch_bounds__(kBlock) void k_frame_init(const FrameInit I) {
    const int64_t stride = (int64_t)gridDim.x * kBlock, t0 = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    for (int k = 0; k < I.n_fills; ++k) {
        const FrameInit::Fill& f = I.fill[k];
        int64_t n = f.n;
        if (f.n_dev) n = min(n, (int64_t)f.mult * *f.n_dev + f.add);
        for (int64_t i = t0; i < n; i += stride) f.p[i] = f.value;
    }
    for (int64_t c = t0; c < (int64_t)I.C; c += stride) {
        const int64_t o0 = I.offsets[c], o1 = I.offsets[c + 1];
        if (o0 < 0) continue;
        for (int64_t b = (o0 + I.window - 1) / I.window; b < I.n_first && b * I.window < o1; ++b)
            I.first[b] = (int32_t)c;
    }
    if (I.budget.entries && t0 == 0) {
        const int32_t total = I.offsets[I.C];
        const bool skip = total < 0 || (int64_t)total > I.budget.entries;
        *I.budget.live = skip ? 0 : total;
        *I.budget.over = skip ? 1 : 0;
    }
}

// transform_pos.comp:33-85.  The per-path outcode OR is reduced inside the wave first (points of
// one path are contiguous), then one atomicOr per (wave, path).
// It also bounds each path's cell rows from its transformed control points (the curves stay
// inside their hull; the margin of 1 px plus 2^-20 of the magnitude covers the rounding of the
// curve evaluation), which sizes the path's (path, row) buckets of the sort.
__global__ __launch_bounds__(kBlock) void k_transform(const float2* __restrict__ pos,
                                                      const uint32_t* __restrict__ pos_path,
                                                      uint32_t P, Mvp m, float fw, float fh, int rmax,
                                                      float2* __restrict__ tpos,
                                                      int32_t* __restrict__ visible,
                                                      int32_t* __restrict__ row_lo,
                                                      int32_t* __restrict__ row_hi,
                                                      const int2* __restrict__ pcanvas,
                                                      const float* __restrict__ mvp_dev) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    const bool valid = i < P;
    if (mvp_dev) {  // the matrix in device memory (a captured frame that follows setMVP)
#pragma unroll
        for (int k = 0; k < 16; ++k) m.m[k] = mvp_dev[k];
    }
    int32_t bits = 0, lo = 0, hi = 0;
    uint32_t path = 0xFFFFFFFFu;
    if (valid) {
        if (pcanvas) {  // documents of a batch: each path has its own canvas
            const int2 cv = pcanvas[pos_path[i]];
            fw = (float)cv.x; fh = (float)cv.y; rmax = (cv.y - 1) / 2;
        }
        float2 p = pos[i];
        float o[4];
#pragma unroll
        for (int r = 0; r < 4; ++r)
            o[r] = ((p.x * m.m[4 * r] + p.y * m.m[4 * r + 1]) + 0.0f * m.m[4 * r + 2]) + 1.0f * m.m[4 * r + 3];
        float ox = o[0] / o[3], oy = o[1] / o[3];
        tpos[i] = make_float2(ox, oy);
        bits = outcode_bits(ox, oy, fw, fh);
        path = pos_path[i];
        const float mg = 1.0f + fabsf(oy) * 0x1p-20f;
        lo = sat_f2i(floorf((oy - mg) * 0.5f));
        hi = sat_f2i(floorf((oy + mg) * 0.5f));
        lo = lo < -1 ? -1 : (lo > rmax + 1 ? rmax + 1 : lo);
        hi = hi < -1 ? -1 : (hi > rmax + 1 ? rmax + 1 : hi);
        if (!(oy == oy)) { lo = -1; hi = rmax + 1; }
    }
    unsigned long long todo = __ballot(valid && bits != 0);
    while (todo) {
        const int leader = __ffsll((long long)todo) - 1;
        const uint32_t lp = __shfl(path, leader);
        const bool match = valid && bits != 0 && path == lp;
        todo &= ~__ballot(match);
        int32_t v = match ? bits : 0;
        int32_t vlo = match ? lo : 0x7FFFFFFF, vhi = match ? hi : (int32_t)0x80000000;
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) {
            v |= __shfl_xor(v, o);
            vlo = min(vlo, __shfl_xor(vlo, o));
            vhi = max(vhi, __shfl_xor(vhi, o));
        }
        if ((int)(threadIdx.x & 63) == leader) {
            atomicOr(&visible[lp], v);
            atomicMin(&row_lo[lp], vlo);
            atomicMax(&row_hi[lp], vhi);
        }
    }
}

// Exclusive scan of one value per thread over the tiles of a launch (256 values a tile), with the
// decoupled look-back of the tile's first wave.  Returns the thread's exclusive prefix; `upto`
// receives the prefix after the tile.
__device__ inline int32_t tile_scan(int32_t v, int64_t tile, unsigned long long* status, int32_t* s_w, int32_t& upto) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int32_t inc = wave_inclusive_add(v);
    if (lane == 63) s_w[wave] = inc;
    __syncthreads();
    int32_t before = 0, total = 0;
#pragma unroll
    for (int k = 0; k < kBlock / 64; ++k) {
        const int32_t x = s_w[k];
        if (k < wave) before = wadd(before, x);
        total = wadd(total, x);
    }
    __syncthreads();
    if (wave == 0) {
        const int32_t pre = lookback<OpI32>(status, tile, total);
        if (lane == 0) s_w[0] = pre;
    }
    __syncthreads();
    const int32_t pre = s_w[0];
    upto = wadd(pre, total);
    return wadd(pre, wadd(before, (int32_t)((uint32_t)inc - (uint32_t)v)));
}

// make_intersection_0.comp:226-411 and the scans after it in one launch: the last K.curve_tiles
// workgroups take 256 curves each (monotone cuts, cut cache, intersection count and its exclusive
// scan, total at counts[C]; where each path's entries start, the sort segments of
// gen_fragment.comp:227-244, falls out of it), the first K.path_tiles 256 paths each (their bucket rows from the row
// bounds, and the exclusive scan of the bucket counts, total at bucket_base[Np]).  A count takes
// microseconds and a scan by itself little but its launch, so the tiles' look-backs hide behind
// the counting of the tiles after them.  The totals also go to host memory when the host waits
// for them.  What bounds a small frame's prefix is its launches (about 4.5 us each, back to back, and
// 8 us for a copy and its wait): with this kernel in the place of five launches and two copies, and
// its fills in one launch instead of four, the 512 x 512 sketch's frame went from 375 us to 345 us.
__global__ __launch_bounds__(kBlock) void k_count(const CountArgs K) {
    __shared__ int32_t s_w[kBlock / 64], s_tile;
    int32_t upto;
    if ((int)blockIdx.x < K.path_tiles) {
        // in-canvas rows r >= 1 get buckets first..first+nrows-1, then the off-canvas bucket, then row 0
        const int64_t tile = ordered_tile_id(K.path_counter, &s_tile);
        const int64_t p = tile * kBlock + threadIdx.x;
        int32_t n = 0;
        if (p < (int64_t)K.Np) {
            const int rmax = K.pcanvas ? (K.pcanvas[p].y - 1) / 2 : K.rmax;
            const int lo = K.row_lo[p], hi = K.row_hi[p];
            int first = lo < 1 ? 1 : lo;
            const int last = hi > rmax ? rmax : hi;
            int nrows = last >= first ? last - first + 1 : 0;
            if (lo > hi) { first = 1; nrows = 0; }  // no points
            K.prow[p] = make_int2(first, nrows);
            n = nrows + 2;
        }
        const int32_t at = tile_scan(n, tile, K.path_status, s_w, upto);
        if (p < (int64_t)K.Np) K.bucket_base[p] = at;
        if (tile == K.path_tiles - 1 && threadIdx.x == 0) {
            K.bucket_base[K.Np] = upto;
            if (K.host) __hip_atomic_store(&K.host[1], upto, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
        return;
    }
    const int64_t tile = ordered_tile_id(K.curve_counter, &s_tile);
    const int64_t c = tile * kBlock + threadIdx.x;
    int32_t cnt = 0;
    if (c < (int64_t)K.C) {
        const uint32_t path = K.cpath[c];
        int w = K.w, h = K.h;
        if (K.pcanvas) { w = K.pcanvas[path].x; h = K.pcanvas[path].y; }  // a batch: the path's document canvas
        const CurvePts cv = load_curve(K.tpos, K.cpos[c], K.ctype[c], K.cweight, (uint32_t)c);
        const bool vis = visible_mask(K.visible[path]);
        float q[4];
        const uint32_t n = monotone_cuts(cv, vis, q);
        K.cuts[c] = make_float4(q[0], q[1], q[2], q[3]);
        K.ncuts[c] = n;
        if (vis) {
            float p0x = cv.x[0], p0y = cv.y[0], t_first = -1.0f, end_x = 0.0f, end_y = 0.0f;
            // a piece beyond the curve pass's windows, perhaps: its grid rounds differently from the count far
            // outside any canvas
            const float far = 1e9f;
            bool big = !(fabsf(p0x) < far) | !(fabsf(p0y) < far);
#pragma unroll
            for (uint32_t k = 0; k < 5; ++k) {
                if (k > n) break;
                const float t = k < n ? q[k < 4 ? k : 3] : 1.0f;
                const float p1x = cv.ex(t), p1y = cv.ey(t);
                const int pc = piece_count(p0x, p0y, p1x, p1y, w, h);
                cnt += pc;
                big = big | (pc > kCurvePieceMax) | !(fabsf(p1x) < far) | !(fabsf(p1y) < far);
                if (k == 0 && pc > kLongHead && cv.type != kLine) { t_first = t; end_x = p1x; end_y = p1y; }
                p0x = p1x; p0y = p1y;
            }
            if (big) {
                uint32_t pieces = 0;
                p0x = cv.x[0]; p0y = cv.y[0];
#pragma unroll 1
                for (uint32_t k = 0; k <= n && k < 5; ++k) {
                    const float qk = k < 2 ? (k == 0 ? q[0] : q[1]) : (k == 2 ? q[2] : q[3]);
                    const float t = k < n ? qk : 1.0f;
                    const float p1x = cv.ex(t), p1y = cv.ey(t);
                    const PieceGrid G = piece_grid(p0x, p0y, p1x, p1y, w, h);
                    pieces |= 1 + G.nx + G.ny > kCurvePieceMax ? 1u << k : 0u;
                    p0x = p1x; p0y = p1y;
                }
                if (pieces) {
                    int32_t at = atomicAdd(K.n_big, (int32_t)__popc(pieces));
                    if (at == 0 && K.host)  // one store: an illustration of 34 M entries lost 110 us to one for each
                        __hip_atomic_store(&K.host[2], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                    for (; pieces; pieces &= pieces - 1u) K.big[at++] = (int32_t)(5 * c + (uint32_t)__ffs(pieces) - 1u);
                }
            }
            // the first piece's chains with many crossings before t1 / 32 (only the choice of a pass hangs on them)
            int n_long = 0;
            float reach = cv.type == kArc ? INFINITY : 0.0f;  // 128 pixels before t / 32 need 1,400 in all
#pragma unroll
            for (int i = 1; i < 4; ++i)
                reach = fmaxf(reach, fmaxf(fabsf(cv.x[i] - cv.x[0]), fabsf(cv.y[i] - cv.y[0])));
            if (t_first >= 0.0f && reach > 1024.0f) {
                const PieceGrid G = piece_grid(cv.x[0], cv.y[0], end_x, end_y, w, h);
                const float t32 = kHeadTau * t_first, x32 = cv.ex(t32), y32 = cv.ey(t32);
                n_long = (G.nx > kLongHead && 0.25f * G.dx * (x32 - G.x0) > (float)kLongHead ? 1 : 0) +
                         (G.ny > kLongHead && 0.25f * G.dy * (y32 - G.y0) > (float)kLongHead ? 1 : 0);
            }
            if (n_long) {
                const int before = atomicAdd(K.n_long, n_long);
                if (K.host && before <= kManyLong && before + n_long > kManyLong)
                    __hip_atomic_store(&K.host[3], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            }
        }
    }
    const int32_t at = tile_scan(cnt, tile, K.curve_status, s_w, upto);
    if (c < (int64_t)K.C) {
        K.counts[c] = at;
        if (K.seg) {
            // the paths that start with this curve (and the empty ones before them)
            const uint32_t path = K.cpath[c];
            for (uint32_t j = c == 0 ? 0u : K.cpath[c - 1] + 1u; j <= path; ++j) K.seg[j] = at;
            if (c == (int64_t)K.C - 1)
                for (uint32_t j = path + 1; j <= K.Np; ++j) K.seg[j] = upto;
        }
    }
    if (tile == K.curve_tiles - 1 && threadIdx.x == 0) {
        K.counts[K.C] = upto;
        if (K.host) __hip_atomic_store(&K.host[0], upto, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

__global__ void k_segment_stats(const int32_t* __restrict__ seg, uint32_t Np, int32_t* __restrict__ max_len) {
    const uint32_t p = blockIdx.x * kBlock + threadIdx.x;
    int32_t len = p < Np ? seg[p + 1] - seg[p] : 0;
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) len = max(len, __shfl_xor(len, o));
    if ((threadIdx.x & 63) == 0 && len > 0) atomicMax(max_len, len);
}

// gen_fragment.comp:90-224: cell key of the segment between consecutive intersections of one
// curve, and its winding change across the cell's centre row.  Returns the entry's bucket.
__device__ inline uint32_t gen_one(const int2* __restrict__ inter, int64_t N, int64_t i,
                                   const uint32_t* __restrict__ cpos, const uint32_t* __restrict__ ctype,
                                   const float* __restrict__ cweight, const uint32_t* __restrict__ cpath,
                                   const float2* __restrict__ tpos, int w,
                                   int h, int32_t* __restrict__ key, int8_t* __restrict__ wn,
                                   uint32_t* __restrict__ epath, const int32_t* __restrict__ bucket_base,
                                   const int2* __restrict__ prow, int32_t* __restrict__ err,
                                   float4* __restrict__ chord) {
    const int2 a = inter[i];
    const int2 b = (i + 1 != N) ? inter[i + 1] : make_int2(-1, 0x3f800000);
    float t0 = glmax(bitsf((uint32_t)a.y & 0xFFFFFFFCu), 0.0f);
    float t1 = glmax(bitsf((uint32_t)b.y & 0xFFFFFFFCu), 0.0f);
    const uint32_t c = (uint32_t)a.x;
    const uint32_t path = cpath[c];
    if (a.x != b.x) t1 = 1.0f;
    uint32_t yx;
    int swn;
    if (t0 < t1) {
        const CurvePts cv = load_curve(tpos, cpos[c], ctype[c], cweight, c);
        const float pfx = cv.ex(t0), pfy = cv.ey(t0), plx = cv.ex(t1), ply = cv.ey(t1);
        segment_cell_pts(true, pfx, pfy, plx, ply, w, h, yx, swn);
        if (chord) chord[i] = make_float4(pfx, pfy, plx, ply);
    } else {
        yx = kSentinelKey;
        swn = 0;
    }
    key[i] = (int32_t)yx;
    wn[i] = (int8_t)swn;
    epath[i] = path;
    return (uint32_t)bucket_base[path] + bucket_local((int32_t)yx, prow[path], err);
}


// Keys of all entries, counted per (path, row) bucket while they are produced.
__global__ __launch_bounds__(kBlock) void k_gen_fragment(const int2* __restrict__ inter, int64_t N,
                                                         const uint32_t* __restrict__ cpos,
                                                         const uint32_t* __restrict__ ctype,
                                                         const float* __restrict__ cweight,
                                                         const uint32_t* __restrict__ cpath,
                                                         const float2* __restrict__ tpos, int w,
                                                         int h, int32_t* __restrict__ key,
                                                         int8_t* __restrict__ wn,
                                                         uint32_t* __restrict__ epath,
                                                         const int32_t* __restrict__ bucket_base,
                                                         const int2* __restrict__ prow,
                                                         int32_t* __restrict__ hist,
                                                         int32_t* __restrict__ err,
                                                         const int32_t* __restrict__ n_dev,
                                                         const int2* __restrict__ pcanvas,
                                                         float4* __restrict__ chord) {
    const int64_t n = n_dev ? min((int64_t)*n_dev, N) : N;
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    bool valid = i < n;
    uint32_t bucket = 0;
    if (valid && inter[i].x < 0) {
        // a gap of a predicted-allocation layout: no fragment, no bucket
        epath[i] = kNoPath;
        valid = false;
    }
    if (valid) {
        int cw = w, ch = h;
        if (pcanvas) { const int2 cv = pcanvas[cpath[inter[i].x]]; cw = cv.x; ch = cv.y; }
        bucket = gen_one(inter, n, i, cpos, ctype, cweight, cpath, tpos, cw, ch, key, wn, epath, bucket_base, prow, err,
                         chord);
    }
    wave_count(hist, bucket, valid);
}

}  // namespace

hipError_t launch_frame_init(const FrameInit& I, hipStream_t s) {
    int64_t n = I.C;
    for (int k = 0; k < I.n_fills; ++k) n = n > I.fill[k].n ? n : I.fill[k].n;
    unsigned g = grid_for(n);
    if (g > 2048u) g = 2048u;
    k_frame_init<<<g, kBlock, 0, s>>>(I);
    return hipGetLastError();
}

hipError_t launch_fill_u32(uint32_t* p, int64_t n, uint32_t v, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    int64_t g = (n + kBlock - 1) / kBlock;
    if (g > 4096) g = 4096;
    k_fill_u32<<<(unsigned)g, kBlock, 0, s>>>(p, n, v);
    return hipGetLastError();
}

hipError_t launch_transform(const float2* pos, const uint32_t* pos_path, uint32_t P, const Mvp& m,
                            int w, int h, float2* tpos, int32_t* visible, int32_t* row_lo, int32_t* row_hi,
                            hipStream_t s, const int2* pcanvas, const float* mvp_dev) {
    if (P == 0) return hipSuccess;
    k_transform<<<grid_for(P), kBlock, 0, s>>>(pos, pos_path, P, m, (float)w, (float)h, (h - 1) / 2, tpos,
                                               visible, row_lo, row_hi, pcanvas, mvp_dev);
    return hipGetLastError();
}

hipError_t launch_count(const CountArgs& K, hipStream_t s) {
    k_count<<<(unsigned)(K.path_tiles + K.curve_tiles), kBlock, 0, s>>>(K);
    return hipGetLastError();
}

hipError_t launch_segment_stats(const int32_t* seg, uint32_t Np, int32_t* max_len, hipStream_t s) {
    if (Np == 0) return hipSuccess;
    k_segment_stats<<<grid_for(Np), kBlock, 0, s>>>(seg, Np, max_len);
    return hipGetLastError();
}

hipError_t launch_gen_fragment(const int2* inter, int64_t N, const uint32_t* cpos,
                               const uint32_t* ctype, const float* cweight, const uint32_t* cpath, const float2* tpos,
                               int w, int h, int32_t* key, int8_t* wn, uint32_t* epath,
                               const int32_t* bucket_base, const int2* prow, int32_t* hist, int32_t* err,
                               hipStream_t s, const int32_t* n_dev, const int2* pcanvas, float4* chord) {
    if (N == 0) return hipSuccess;
    k_gen_fragment<<<grid_for(N), kBlock, 0, s>>>(inter, N, cpos, ctype, cweight, cpath, tpos, w, h, key, wn, epath,
                                                  bucket_base, prow, hist, err, n_dev, pcanvas, chord);
    return hipGetLastError();
}

}  // namespace spr
