// k_curves.hip -- intersection write (make_intersection_1.comp:217-447) and fragment keys
// (gen_fragment.comp:90-224) in one pass over the curves, for gfx950.
//
// Inside one monotone piece the reference interleaves x-grid and y-grid crossings, but every
// bisection for the next crossing on one axis starts from the previous crossing of the SAME axis
// (the t_min it starts from is that axis' pending value, :338-359, :402).  So each (piece, axis)
// is a chain of dependent solves, and the reference's output order is a merge of the two chains
// (ties to x, :338) followed by its equal-t OR-merge (:361-375).  This file keeps every float
// operation of the reference and only changes who computes what.
//
// The entries of a frame are cut into windows, and one workgroup takes the pieces whose first entry
// lies in its window, whole, from the curve data to the fragment keys:
//
//  1. One lane per curve, of one wave, walks its pieces (their grid ranges, flagged end parameters and places)
//     into a table in LDS.
//  2. The chains are cut into segments of a few crossings, one thread each.  A chain carries only
//     one value from crossing to crossing, the last parameter with its two low bits replaced, so
//     a segment that guesses that value right computes exactly the chain's results.  It guesses by
//     solving the crossings before it, the first of them from the piece's start: a bisection
//     depends on its start only through the rounding of its midpoints, so two runs from
//     different starts mostly fall together within a few crossings and then stay together.  Every
//     guess is compared with what the segment before it ended on; a segment whose guess differs
//     is solved again from there until it meets the values it had, which repeats until all
//     guesses hold.  The values are therefore the sequential chain's, bit for bit, whatever the
//     guesses were worth.
//  3. The pieces are checked for order and merged by rank in LDS, and every entry becomes its
//     cell key (or sort word), winding change and bucket count.
//
// Runs fall together more slowly where t is small beside the bracket that is left: the 24
// halvings of [t, t1] then end on a grid of (t1 - t) 2^-24, coarser than the masked values around
// t, and that grid moves with its start: about 2, 4, 8.. values are possible below t1 / 8, t1 / 16,
// t1 / 32.  Segments that start there solve more crossings before their own (8 and 16 instead of
// 4), and a chain's first segment reaches past t = t1 / 32.
//
// A view of the first part of large curves has hundreds of crossings there, and hardly a guess comes true:
// segments corrected one after another cost more than the chain solved in order.  A chain with a long start
// (more than 64 crossings before t1 / 32) therefore has all those before t1 / 8 in its first segment, and a whole
// wave solves that (wave_solve.hpp).  us a frame: 64 scribbles at 32 and 8 times their size on 1024^2 813 -> 432
// and 767 -> 490, an illustration at 8 times its size on 4096^2 3,343 -> 1,758.
//
// This is the pass of small frames (launch_curves' caller chooses), whose span would otherwise be
// their longest chain: whole chains take about 1 us a crossing one after another, and the passes
// over the chains (k_chain.hip) cost a launch each.  The speculation costs about twice the
// arithmetic, so frames that fill the chip with chains take k_chain.hip.
//
// Pieces of more than kBigPiece entries, which the count pass lists, take k_big_pieces, one workgroup each.
#include "device_common.hpp"
#include "fragments.hpp"
#include "kernels.hpp"
#include "scan_common.hpp"
#include "wave_solve.hpp"

#include <type_traits>

namespace spr {

namespace {

constexpr int kBigPiece = kCurvePieceMax;       // longer pieces take a workgroup
constexpr int kCap = kCurveWindowMax + kBigPiece;  // LDS slots: a window plus its last piece's overhang
constexpr int kLanes = 64;                      // curves of a batch: one wave walks them
constexpr int kThreads = 256;                   // of a window
constexpr int kWaves = kThreads / 64;
constexpr int kSlots = 5 * kLanes;              // piece slots: piece k of lane l's curve at 5 l + k
constexpr int kPerLane = kBigPiece / kThreads;  // merged slots per thread and step
constexpr int kBigThreads = 256;
constexpr int kStage = 4096;                    // big pieces up to this many entries stay in LDS
// Crossings solved before a segment to guess its start, the least length of a segment, and the
// segments that a batch is cut into (besides one per chain).
constexpr int kWarm = 4, kWarm8 = 8, kWarm16 = 16, kSegMin = 4, kSegTarget = 112;
constexpr int kSegs = 832;
// A chain with a long start has all crossings before t1 / 8 in its first segment, which a whole wave solves; a
// batch has at most so many.
constexpr int kLongHeads = 8;
constexpr int kBigLongHead = 16;                // for kLongHead in k_big_pieces, whose waves would wait anyway
constexpr uint32_t kByWave = 1u << 20;          // on a chain's first segment in the list
// Candidate starts of a batch's slow segments (a multiple of 8 each), and the chains that have any.
constexpr int kCands = 384, kWalks = 16;
constexpr int kCand16 = 16, kCand8 = 8;         // below t1 / 16, t1 / 8
constexpr uint32_t kNoValue = 0xFFFFFFFFu;      // no entry, no value (solved values carry side bits 0 or 1)
constexpr int64_t kFewWindows = 1024, kLongCurves = 8;  // k_curves
static_assert(kCands / 8 < 64, "a segment's first candidate in 6 bits");
// chains are 2 * 320; the segments after a chain's first hold X / kSegTarget or more of the
// batch's X crossings in all but one of a chain, and only chains of 1.5 of them have any
static_assert(2 * kSlots + kSegTarget + (2 * kSegTarget) / 3 <= kSegs, "segment list");
static_assert(2 * kSlots <= 1024, "chain numbers of 10 bits");
constexpr uint32_t kNoPiece = 0xFFFFu;          // slot field of an empty piece slot
static_assert(kFrag == 2, "piece records keep only the sign of the grid step");
static_assert(kCap <= 2048 && kBigPiece % kThreads == 0, "slots of a batch");

// Bits of a piece record's second word above ny.
constexpr uint32_t kPwX = 1u << 22, kPwY = 1u << 23;            // grid step -2 on x, y
constexpr int kPwType = 24;                                     // curve type: 0 line, 1 quad, 2 cubic, 3 arc
constexpr uint32_t kPwFalls = 1u << 26, kPwRises = 1u << 27;    // the piece's sequences go down / up somewhere

__device__ inline uint32_t type_code(uint32_t type) { return type == kArc ? 3u : type - 2u; }
__device__ inline uint32_t type_of_code(uint32_t code) { return code == 3u ? kArc : code + 2u; }

// Orders within one wave: LDS written by some lanes and then read by others.
__device__ inline void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// A piece with what its fragments need besides its merged entries.
struct PieceSeq {
    int32_t base, nx, ny, curve;
    float t0;           // flagged start parameter
};
struct PieceMeta {
    PieceSeq pd;
    float t_end;        // parameter where the last entry's segment ends
    uint32_t path, bb;  // path, its first bucket
    int32_t w, h;
    int2 pr;            // the path's row range
    CurvePts cv;
};

// Merges one piece held in LDS (X = xs[0..nx), Y = xs[nx..nx+ny)) into out[0..n) with nthr
// threads (a wave or a workgroup; lane = the thread's index among them), in the order of
// make_intersection_1.comp:310-359, ties to x.
__device__ inline void wave_merge(const PieceSeq& pd, uint8_t mode, const float* X, uint32_t* out, int lane,
                                  int nthr = 64) {
    const int nx = pd.nx, ny = pd.ny;
    const float* Y = X + nx;
    const bool head_in_a = ny == 0;
    const int na = nx + (head_in_a ? 1 : 0), nb = head_in_a ? 0 : ny + 1;
    const float t0 = pd.t0;
    // loads always from the staged chains (index clamped), the piece start selected after: the
    // accessors must not form a pointer to t0, which would turn every access into a flat load
    auto Aat = [&](int i) -> float {
        if (!head_in_a) return X[i];
        const float x = X[i > 0 ? i - 1 : 0];
        return i == 0 ? t0 : x;
    };
    auto Bat = [&](int j) -> float {
        const float y = Y[j > 0 ? j - 1 : 0];
        return j == 0 ? t0 : y;
    };
    const int n = na + nb;
    if (mode == 2) {
        if (lane == 0) {
            const float kX2 = bitsf(kTwoBits), kY2 = bitsf(kTwoBits | 1u);
            float tx = pd.t0, ty = pd.t0;
            int xi = 0, yi = 0;
            if (nx == 0) tx = kX2;
            else if (ny == 0) ty = kY2;
            else { tx = X[0]; xi = 1; }
            for (int i = 0; i < n; ++i) {
                float tmin;
                if (tx <= ty) { tmin = tx; tx = xi < nx ? X[xi++] : kX2; }
                else { tmin = ty; ty = yi < ny ? Y[yi++] : kY2; }
                out[i] = fbits(tmin);
            }
        }
    } else if (mode == 1) {
        const bool a_first = nb == 0 || (na > 0 && Aat(0) <= Bat(0));
        for (int o = lane; o < n; o += nthr) {
            float v;
            if (a_first) v = o < na ? Aat(o) : Bat(o - na);
            else v = o < nb ? Bat(o) : Aat(o - nb);
            out[o] = fbits(v);
        }
    } else {
        const int per = (n + nthr - 1) / nthr;
        const int o0 = lane * per;
        const int o1 = o0 + per < n ? o0 + per : n;
        if (o0 < n) {
            int lo = o0 > nb ? o0 - nb : 0, hi = o0 < na ? o0 : na;
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                if (Aat(mid) <= Bat(o0 - 1 - mid)) lo = mid + 1; else hi = mid;
            }
            int i = lo, j = o0 - lo;
            for (int o = o0; o < o1; ++o) {
                const bool takeA = j >= nb || (i < na && Aat(i) <= Bat(j));
                const float v = takeA ? Aat(i) : Bat(j);
                i += takeA; j += !takeA;
                out[o] = fbits(v);
            }
        }
    }
}

// The reference's OR of equal t inside a piece (make_intersection_1.comp:361-375): within a run
// [s, e) of equal masked t, entry o ends up as the OR of raw values s..min(o+1, e-1).  Runs never
// leave the piece (its first entry starts a run).  `v` is the merged piece in LDS.
__device__ inline uint32_t or_merged(const uint32_t* v, int n, int o) {
    const uint32_t m = v[o] & 0xFFFFFFFCu;
    uint32_t acc = v[o];
    for (int s = o; s > 0 && (v[s - 1] & 0xFFFFFFFCu) == m; --s) acc |= v[s - 1];
    if (o + 1 < n && (v[o + 1] & 0xFFFFFFFCu) == m) acc |= v[o + 1];
    return acc;
}

// gen_fragment for the entries of one piece, v[0..n) = their merged t bits: entry o's segment
// runs to entry o+1, the last one's to m.t_end.  Keys, winding changes and paths are written
// coalesced; bucket counts are aggregated over runs of the wave.  Every lane of the n_waves
// waves calls it; wave w takes the chunks w, w + n_waves, ...
__device__ inline void piece_fragments(const PieceMeta& m, const uint32_t* v, int n, const FragArgs& A, int lane,
                                       int wave = 0, int n_waves = 1) {
    // lane l evaluates point o0 + l (point o is entry o's parameter, point n is t_end); entry o's
    // segment runs from point o to point o + 1, so a chunk of 64 points serves 63 entries
    for (int o0 = wave * 63; o0 < n; o0 += n_waves * 63) {
        const int o = o0 + lane;
        float t = 0.0f;
        uint32_t f = 0;
        if (o < n) { f = v[o]; t = glmax(bitsf(f & 0xFFFFFFFCu), 0.0f); }
        else if (o == n) t = m.t_end;
        const float px = m.cv.ex(t), py = m.cv.ey(t);
        const float t1 = __shfl_down(t, 1), qx = __shfl_down(px, 1), qy = __shfl_down(py, 1);
        const bool valid = lane < 63 && o < n;
        uint32_t bucket = 0;
        if (valid) {
            uint32_t yx;
            int swn;
            segment_cell_pts(t < t1, px, py, qx, qy, m.w, m.h, yx, swn);
            const int64_t i = (int64_t)m.pd.base + o;
            bucket = store_fragment(A, i, yx, swn, m.path, m.bb, m.pr);
            if (A.inter) A.inter[i] = make_int2(m.pd.curve, (int32_t)or_merged(v, n, o));
            if (A.chord) A.chord[i] = make_float4(px, py, qx, qy);
        }
        wave_count(A.hist, bucket, valid);
    }
}

// One monotone piece of a curve as the write pass walks it.
struct PieceGeom {
    int base, nx, ny;   // first entry, crossings per axis
    float x0, y0;       // first grid line crossed on each axis
    bool xneg, yneg;    // grid step -2
    float t0, t1;       // flagged start and end parameters
    bool ok;            // written: count and write passes agree on it
    __device__ int n() const { return 1 + nx + ny; }
};

// The pieces of a curve in order (at most 5): piece k runs from the end of piece k-1 (flagged end
// parameter and end point) to its own end, and its entries start after the 1 + nx + ny entries of
// each earlier piece.
template <class F>
__device__ inline void walk_pieces(const CurvePts& cv, const float4 q, uint32_t n_cuts, int base0, int limit, int w,
                                   int h, F&& f) {
    float t0 = 0.0f, p0x = cv.x[0], p0y = cv.y[0];
    int base = base0;
#pragma unroll 1
    for (uint32_t k = 0; k <= n_cuts && k < 5; ++k) {
        const float qk = k < 2 ? (k == 0 ? q.x : q.y) : (k == 2 ? q.z : q.w);
        const float traw = k < n_cuts ? qk : 1.0f;
        const float p1x = cv.ex(traw), p1y = cv.ey(traw);
        const PieceGrid G = piece_grid(p0x, p0y, p1x, p1y, w, h);
        PieceGeom g;
        g.base = base; g.nx = G.nx; g.ny = G.ny; g.x0 = G.x0; g.y0 = G.y0;
        g.xneg = G.dx < 0.0f; g.yneg = G.dy < 0.0f;
        g.t0 = t0;
        g.t1 = flag_piece_end(traw, p1x);
        g.ok = base + G.nx + G.ny + 1 <= limit;
        f((int)k, g);
        base += g.n();
        t0 = g.t1; p0x = p1x; p0y = p1y;
    }
}

// Masked parameter of a piece's first entry, where the last entry of the piece before it ends.
// The merges of make_intersection_1.comp:310-359 all start with the smaller of X[0] and the piece
// start when the piece has crossings on both axes (ties to x), and with the piece start
// otherwise; a piece that runs backwards in t (unsorted cuts) can therefore start with X[0].
__device__ inline float first_entry_t(const CurvePts& cv, const PieceGeom& g) {
    float first = g.t0;
    if (g.nx > 0 && g.ny > 0) {
        const CurveAxis ax = {{cv.x[0], cv.x[1], cv.x[2], cv.x[3]}};
        const float ts = solve_axis(cv.type, ax, g.x0, g.t0, g.t1);
        const float v = bitsf(fbits(ts) & 0xFFFFFFFCu);
        if (v <= g.t0) first = v;
    }
    return glmax(bitsf(fbits(first) & 0xFFFFFFFCu), 0.0f);
}

// Crossings k0..i1-1 of a chain, in order, the first solved from tstart; values i0..i1-1 go to
// vs[i0..i1-1].  Returns the value before crossing i0 (the guess of a segment's start when
// k0 < i0).  redo: the values are already there; stops at the first that comes out equal, since
// everything after it is then equal too.
template <uint32_t T, class P>
__device__ inline float solve_run(const CurveAxis& a, float line0, bool neg, uint32_t side, float t1, int k0, int i0,
                                  int i1, float tstart, bool redo, P vs) {
    const float step = neg ? -2.0f : 2.0f;
    float tprev = tstart, line = line0 + step * (float)k0, g = tstart;  // lines are small integers: exact
    ChainSolver<T, 6> solver(a, step, t1);  // six steps at a time: most waves run this code once or twice
    for (int k = k0; k < i1; ++k) {
        // the usual case in every lane: the straight-line form, no divergent branches
        const float ts = __all(solver.common(tprev)) ? solver.next_common(line, tprev, t1) : solver.next(line, tprev, t1);
        const float v = bitsf((fbits(ts) & 0xFFFFFFFCu) | side);
        if (k >= i0) {
            if (redo && fbits(vs[k]) == fbits(v)) break;
            vs[k] = v;
        } else {
            g = v;
        }
        tprev = v;
        line += step;
    }
    return g;
}

template <class P>
__device__ inline float solve_run_any(uint32_t type, const CurveAxis& a, float line0, bool neg, uint32_t side, float t1,
                                      int k0, int i0, int i1, float tstart, bool redo, P vs) {
    if (type == kCubic) return solve_run<kCubic>(a, line0, neg, side, t1, k0, i0, i1, tstart, redo, vs);
    if (type == kLine) return solve_run<kLine>(a, line0, neg, side, t1, k0, i0, i1, tstart, redo, vs);
    if (type == kQuad) return solve_run<kQuad>(a, line0, neg, side, t1, k0, i0, i1, tstart, redo, vs);
    return solve_run<kArc>(a, line0, neg, side, t1, k0, i0, i1, tstart, redo, vs);
}

// Segment j of a chain of n crossings cut into k equal parts.
__device__ inline int seg_begin(int n, int k, int j) { return (int)(((uint32_t)n * (uint32_t)j) / (uint32_t)k); }

// LDS of one batch: up to 64 curves, their pieces and the entries of the pieces.
struct CurveBatch {
    float v[kCap];                       // entry slots: piece start, x chain, y chain; then merged
    uint4 pa[kSlots];                    // slot | nx << 16; ny | curve | flags; x0 | y0 << 16; t1
    float tend[kSlots];                  // parameter after the last entry, or -1: the next slot's
    uint16_t by_rank[kSlots];            // piece slots in entry order
    float4 cx[kLanes], cy[kLanes];       // control values
    int4 cm[kLanes];                     // first bucket, row range, path
    int2 canvas[kLanes];
    unsigned long long starts[kCap / 64];  // bit per entry slot: a piece starts there
    uint16_t starts_before[kCap / 64];
    uint16_t head[2 * kSlots];           // length of each chain's first segment
    // chain | segment << 10 | crossings to guess its start from << 20, kHasCands | first candidate / 8 << 26
    uint32_t seg[kSegs];
    int n_segs;
    int n_pieces, longest, n_slots, crossings;  // of the batch
    int n_long;                          // chains with a long start
    uint16_t longs[kLongHeads];          // those that waves solve
};

struct Candidates {
    uint32_t cand[kCands];   // chain | segment << 10 | candidate << 20; then the value it ends on
    uint32_t start[kCands];  // the value it starts from; a segment's first: its predicted start
    uint2 walk[kWalks];      // chain | segments of kCand16 << 10, of kCand8 << 20; first candidate
    int n_cands, n_walks;
};
constexpr uint32_t kHasCands = 1u << 25;

// The piece that entry slot e lies in or after, -1 before the first.
__device__ inline int piece_of(const CurveBatch& B, int e) {
    const unsigned long long m = B.starts[e >> 6] & (~0ull >> (63 - (e & 63)));
    const int rank = (int)B.starts_before[e >> 6] + (int)__popcll(m) - 1;
    return rank < 0 ? -1 : (int)B.by_rank[rank];
}

// Merges the pieces of slots [s0, s1) in place (s1 - s0 <= kBigPiece; whole pieces): every
// slot's place is its index in its own sequence plus its rank in the other one.  Sequences: A =
// X, B = [t0, Y]; with one axis only the slots are already in order.  A piece whose sequences both
// fall is the sequence with the smaller head (ties to x) followed by the other; one that
// goes both ways is merged by the sequential walk, through scratch.
__device__ inline void merge_slots(CurveBatch& B, int s0, int s1, int longest, bool any_falls,
                                   uint32_t* __restrict__ scratch) {
    const int tid = threadIdx.x;
    if (any_falls) {
        for (int p = tid; p < kSlots; p += kThreads) {
            const uint32_t w0 = B.pa[p].x, w1 = B.pa[p].y;
            const int base = (int)(w0 & 0xFFFFu), nx = (int)(w0 >> 16), ny = (int)(w1 & 0xFFFFu);
            if (base < s0 || base >= s1 || (w1 & (kPwFalls | kPwRises)) != (kPwFalls | kPwRises)) continue;
            const float kX2 = bitsf(kTwoBits), kY2 = bitsf(kTwoBits | 1u);
            float tx = B.v[base], ty = B.v[base];
            int xi = 0, yi = 0;
            if (nx == 0) tx = kX2;
            else if (ny == 0) ty = kY2;
            else { tx = B.v[base + 1]; xi = 1; }
            for (int i = 0; i < 1 + nx + ny; ++i) {
                float tmin;
                if (tx <= ty) { tmin = tx; tx = xi < nx ? B.v[base + 1 + xi] : kX2; ++xi; }
                else { tmin = ty; ty = yi < ny ? B.v[base + 1 + nx + yi] : kY2; ++yi; }
                scratch[base + i] = fbits(tmin);
            }
        }
        __threadfence_block();
        __syncthreads();
    }
    float v[kPerLane];
    int from[kPerLane], len[kPerLane], rank[kPerLane], dest[kPerLane];
    uint32_t le = 0;  // bit j: rank counts equal values too
#pragma unroll
    for (int j = 0; j < kPerLane; ++j) {
        const int e = s0 + tid + kThreads * j;
        v[j] = 0.0f; from[j] = 0; len[j] = 0; rank[j] = 0; dest[j] = -1;
        if (s0 + kThreads * j >= s1) continue;
        if (e < s1) {
            const int p = piece_of(B, e);
            if (p < 0) continue;
            const uint2 w = make_uint2(B.pa[p].x, B.pa[p].y);
            const int base = (int)(w.x & 0xFFFFu), nx = (int)(w.x >> 16), ny = (int)(w.y & 0xFFFFu);
            const int idx = e - base;
            v[j] = B.v[e];
            if (idx <= nx + ny) {
                const bool in_a = idx >= 1 && idx <= nx;
                if ((w.y & (kPwFalls | kPwRises)) == (kPwFalls | kPwRises)) {
                    v[j] = bitsf(scratch[e]);
                    dest[j] = e;
                } else if (nx > 0 && ny > 0) {
                    const float t0 = B.v[base];
                    if (w.y & kPwFalls) {
                        const bool a_first = B.v[base + 1] <= t0;
                        if (in_a) dest[j] = base + idx - 1 + (a_first ? 0 : ny + 1);
                        else dest[j] = base + (idx == 0 ? 0 : idx - nx) + (a_first ? nx : 0);
                    } else if (in_a) {
                        from[j] = base + 1 + nx;
                        len[j] = ny;
                        dest[j] = e - 1 + (t0 < v[j] ? 1 : 0);
                    } else {
                        from[j] = base + 1;
                        len[j] = nx;
                        dest[j] = base + (idx == 0 ? 0 : idx - nx);
                        le |= 1u << j;
                    }
                }
            }
        }
    }
    for (int bit = longest ? 1 << (31 - __clz(longest)) : 0; bit; bit >>= 1) {
#pragma unroll
        for (int j = 0; j < kPerLane; ++j) {
            if (s0 + kThreads * j >= s1) continue;
            const int r = rank[j] + bit;
            if (r <= len[j]) {
                const float x = B.v[from[j] + r - 1];
                if (x < v[j] || (((le >> j) & 1u) && x == v[j])) rank[j] = r;
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kPerLane; ++j)
        if (dest[j] >= 0) B.v[dest[j] + rank[j]] = v[j];
    __syncthreads();
}

// Segments of a chain of n crossings whose first one has `head` of them: 1 + rest, the others of
// (nearly) equal lengths near `len`.
__device__ inline int seg_rest(int n, int head, int len) { return (n - head + len - 1) / len; }

// A chain of the batch: its piece's values for one axis.
struct ChainRef {
    CurveAxis a;
    float line0, t0, t1;
    uint32_t type, side;
    bool neg;
    int n, at;  // crossings, slot of the first
};
__device__ inline ChainRef chain_of(const CurveBatch& B, int ch) {
    const uint4 w = B.pa[ch >> 1];
    const bool ys = (ch & 1) != 0;
    const int base = (int)(w.x & 0xFFFFu), nx = (int)(w.x >> 16), lc = (int)((w.y >> 16) & 63u);
    const float4 cc = ys ? B.cy[lc] : B.cx[lc];
    ChainRef r;
    r.a = {{cc.x, cc.y, cc.z, cc.w}};
    r.line0 = (float)(ys ? w.z >> 16 : w.z & 0xFFFFu);
    r.neg = (w.y & (ys ? kPwY : kPwX)) != 0u;
    r.side = ys ? 1u : 0u;
    r.type = type_of_code((w.y >> kPwType) & 3u);
    r.t1 = bitsf(w.w);
    r.t0 = B.v[base];
    r.n = ys ? (int)(w.y & 0xFFFFu) : nx;
    r.at = base + 1 + (ys ? nx : 0);
    return r;
}
__device__ inline void seg_range(const CurveBatch& B, int ch, int j, int n, int len, int& i0, int& i1) {
    const int head = B.head[ch];
    i0 = 0; i1 = head;
    if (j > 0) {
        const int m = seg_rest(n, head, len);
        i0 = head + seg_begin(n - head, m, j - 1);
        i1 = head + seg_begin(n - head, m, j);
    }
}

// Where t is small, a guess rarely comes true (see above), and correcting one segment after another
// takes a round each.  The value before such a segment is one of few: the last midpoint of
// a bisection lies within 2^-24 of its bracket from the root, and masked values are 4 ulp apart.  So the
// idle threads solve these segments from each of the 16 (t < t1 / 16) or 8 (t < t1 / 8) masked
// values around the root, one thread each, and one thread per chain then walks its segments from
// candidate to candidate, which predicts every segment's start at once.  The predictions are
// checked like all guesses.
__device__ inline void try_candidates(const CurveBatch& B, Candidates& Q, int n_cands, int S, int len, float* none) {
    // the waves without segments first; none: nothing is stored there
    for (int c = ((int)threadIdx.x + kThreads - ((S + 63) & ~63)) & (kThreads - 1); c < n_cands; c += kThreads) {
        const uint32_t e = Q.cand[c];
        if (e == kNoValue) continue;
        const int ch = (int)(e & 1023u), k = (int)(e >> 20);
        const ChainRef r = chain_of(B, ch);
        int i0, i1;
        seg_range(B, ch, (int)((e >> 10) & 1023u), r.n, len, i0, i1);
        const float root = solve_run_any(r.type, r.a, r.line0, r.neg, r.side, r.t1, i0 - 1, i0, i0, r.t0, false, none);
        const uint32_t v = ((fbits(root) & 0xFFFFFFFCu) + (uint32_t)(4 * (k - kCand16))) | r.side;
        Q.start[c] = v;
        Q.cand[c] = fbits(solve_run_any(r.type, r.a, r.line0, r.neg, r.side, r.t1, i0, i1, i1, bitsf(v), false, none));
    }
}

__device__ inline void walk_candidates(const CurveBatch& B, Candidates& Q, const uint2 w) {
    const int ch = (int)(w.x & 1023u), n16 = (int)((w.x >> 10) & 1023u), n8 = (int)(w.x >> 20);
    const ChainRef r = chain_of(B, ch);
    uint32_t v = fbits(B.v[r.at + (int)B.head[ch] - 1]);
    int c = (int)w.y;
    for (int j = 0; j < n16 + n8; ++j) {
        const int n = j < n16 ? kCand16 : kCand8;
        uint32_t end = kNoValue;
        if (v != kNoValue) {
#pragma unroll 8
            for (int k = 0; k < n; ++k)
                if (Q.start[c + k] == v) end = Q.cand[c + k];
        }
        Q.start[c] = v;
        v = end;
        c += n;
    }
}

// One workgroup per window of K.window entries.  first[b] is the curve that holds entry b * window.
// Its span is latency (loads behind each other, chains of dependent solves, LDS searches), so the
// waves that fit a CU decide its rate: one wave a window left 6 waves on a CU (23 KB of LDS each,
// 160 VGPRs); four waves to the same LDS put 24 there (6 per SIMD: at most 80 VGPRs, for which 22 are
// spilled, 84 bytes a lane; with CANDS 5 per SIMD, 96 VGPRs and 17 spilled, 72 bytes).  Four waves
// also take a window of 1024 entries in about the time that one took 128, with a quarter of
// the speculative solves per entry.  Frames in turn on three handles, us a frame, one wave and four:
// 0.8 M entries on a few long curves 203 -> 134, 1.9 M on 20,000 glyphs 299 -> 261.  Two waves a
// window: 138, 255; four to five per SIMD (96 to 128 VGPRs): 2 to 15% slower.
// CANDS: frames of at most kFewWindows windows, which last as long as their slowest window (a dozen rounds
// of corrections: 109 us, the mean 42, for 16 paths at 512^2), try candidate starts.  us a frame without
// and with: 16 paths at 512^2 250 and 229, 64 at 1024^2 126 and 119, a drawing of 0.15 M entries alone 311
// and 291.  Frames of more windows fill the chip anyway, and the candidates' arithmetic costs more than the
// rounds: 1.9 M entries 259 and 265, 6.2 M 894 and 939.  So do frames of very short curves, whose chains
// are not cut: 0.4 M entries on 125,000 curves 203 and 210.  Both lines lie somewhere between two measured
// scenes: kFewWindows between 670 windows and 1,860, kLongCurves between 3 entries a curve and 13.
template <bool CANDS>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(CANDS ? 5 : 6)))
void k_curves(const CurveArgs K, const FragArgs A) {
    __shared__ CurveBatch B;
    __shared__ typename std::conditional<CANDS, Candidates, int>::type cands;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t total = K.n_dev ? min((int64_t)*K.n_dev, K.n) : K.n;
    const int64_t wb64 = (int64_t)blockIdx.x * K.window;
    if (wb64 >= total) return;
    const int wb = (int)wb64, wend = (int)min(wb64 + K.window, total);
    int n_split = 0;
    int64_t next_cb = 0;
    for (int64_t cb = K.first[blockIdx.x]; cb < (int64_t)K.C; cb = next_cb) {
        next_cb = cb + kLanes;
        // ---- the curves of the batch, one per lane, and the pieces that start in the window
        const int64_t c = cb + lane;
        int o0 = wend, o1 = wend;
        if (c < (int64_t)K.C) { o0 = K.offsets[c]; o1 = K.offsets[c + 1]; }
        const int bo = __builtin_amdgcn_readfirstlane(o0);
        if (bo >= wend) break;
        if (!__any(o1 > o0) && next_cb < (int64_t)K.C) {
            // 64 culled curves: on to the next curve with entries (the total lies above bo)
            int64_t lo = next_cb, hi = K.C;
            while (hi - lo > 1) {
                const int64_t step = (hi - lo + kLanes - 1) / kLanes;
                const int64_t at = min(lo + (lane + 1) * step, hi);
                const unsigned long long above = __ballot(at >= (int64_t)K.C || K.offsets[at] > bo);
                const int f = above ? __ffsll((long long)above) - 1 : kLanes - 1;
                const int64_t base = lo;
                hi = min(base + (f + 1) * step, hi);
                lo = base + f * step;
            }
            next_cb = lo;
            continue;
        }
        const int bb0 = max(wb, bo);  // the entry of slot 0
        if constexpr (CANDS) {
            for (int c = tid; c < kCands; c += kThreads) cands.cand[c] = kNoValue;
            if (tid == 0) cands.n_cands = cands.n_walks = 0;
        }
        const bool mine = o0 < wend && o1 > o0 && o1 > wb;
        if (wave == 0) {
            if (lane < kCap / 64) B.starts[lane] = 0ull;
#pragma unroll
            for (int k = 0; k < 5; ++k) { B.pa[5 * lane + k].x = kNoPiece; B.pa[5 * lane + k].y = 0u; }
            wave_sync();
            int np = 0, x_lane = 0, longest = 0, n_slots = 0;
            uint32_t in_set = 0;  // bit k: piece k of the lane's curve is in the batch
            if (mine) {
                const uint32_t path = A.cpath[c];
                int w = A.w, h = A.h;
                if (A.pcanvas) { const int2 cw = A.pcanvas[path]; w = cw.x; h = cw.y; }
                const uint32_t type = A.ctype[c];
                const CurvePts cv = load_curve(A.tpos, A.cpos[c], type, A.cweight, (uint32_t)c);
                const int2 pr = A.prow[path];
                const int bb = A.bucket_base[path];
                B.cx[lane] = make_float4(cv.x[0], cv.x[1], cv.x[2], cv.x[3]);
                B.cy[lane] = make_float4(cv.y[0], cv.y[1], cv.y[2], cv.y[3]);
                B.cm[lane] = make_int4(bb, pr.x, pr.y, (int)path);
                B.canvas[lane] = make_int2(w, h);
                int written = o0, prev = -1;  // prev: the piece before, when it is in the batch
                bool needs = false;           // a piece of the batch ends at the first entry of one outside
                PieceGeom after;
                after.nx = after.ny = 0; after.t0 = after.t1 = after.x0 = 0.0f;
                int needs_at = 0;
                walk_pieces(cv, K.cuts[c], K.ncuts[c], o0, o1, w, h, [&](int k, const PieceGeom& g) {
                    if (!g.ok) { prev = -1; return; }
                    written = g.base + g.n();
                    const bool starts = g.base >= wb && g.base < wend;
                    const bool in = starts && g.n() <= kBigPiece;
                    const int at = 5 * lane + k;
                    if (prev >= 0) {
                        if (in) B.tend[prev] = -1.0f;
                        else { needs = true; needs_at = prev; after = g; }
                    }
                    prev = in ? at : -1;
                    if (in) {
                        const int rel = g.base - bb0;
                        // a grid line is only meaningful (and then in [0, 16386]) on an axis with crossings
                        B.pa[at] = make_uint4((uint32_t)rel | ((uint32_t)g.nx << 16),
                                              (uint32_t)g.ny | ((uint32_t)lane << 16) | (g.xneg ? kPwX : 0u) |
                                                  (g.yneg ? kPwY : 0u) | (type_code(type) << kPwType),
                                              (g.nx ? (uint32_t)(int)g.x0 : 0u) | ((g.ny ? (uint32_t)(int)g.y0 : 0u) << 16),
                                              fbits(g.t1));
                        B.tend[at] = 1.0f;
                        B.v[rel] = g.t0;
                        atomicOr(&B.starts[rel >> 6], 1ull << (rel & 63));
                        ++np;
                        in_set |= 1u << k;
                        x_lane += g.nx + g.ny;
                        longest = max(longest, max(g.nx, g.ny));
                        n_slots = rel + g.n();
                    }
                });
                // counted but not written (the passes round differently only far outside any canvas)
                if (o0 >= wb)
                    for (int i = written; i < o1; ++i) store_gap(A, i, (int)c, path, (uint32_t)bb, pr);
                if (needs) B.tend[needs_at] = first_entry_t(cv, after);
            }
            const int before = wave_inclusive_add(np);
            const int x_upto = wave_inclusive_add(x_lane);
            int rank = before - np;
            for (; in_set; in_set &= in_set - 1) B.by_rank[rank++] = (uint16_t)(5 * lane + __ffs((int)in_set) - 1);
#pragma unroll
            for (int o = 32; o >= 1; o >>= 1) {
                longest = max(longest, __shfl_xor(longest, o));
                n_slots = max(n_slots, __shfl_xor(n_slots, o));
            }
            wave_sync();
            const int here = lane < kCap / 64 ? (int)__popcll(B.starts[lane]) : 0;
            const int upto = wave_inclusive_add(here);
            if (lane < kCap / 64) B.starts_before[lane] = (uint16_t)(upto - here);
            if (lane == 63) {
                B.n_pieces = before; B.crossings = x_upto; B.longest = longest; B.n_slots = n_slots;
                B.n_segs = B.n_long = 0;
            }
        }
        __syncthreads();
        if (B.n_pieces == 0) { __syncthreads(); continue; }
        const int longest = __builtin_amdgcn_readfirstlane(B.longest), n_slots = __builtin_amdgcn_readfirstlane(B.n_slots);
        const int crossings = __builtin_amdgcn_readfirstlane(B.crossings);

        // ---- segments: those of a chain side by side in the list and in order, the chains in any
        const int len = max(kSegMin, (crossings + kSegTarget - 1) / kSegTarget);
#pragma unroll 1
        for (int ch = tid; ch < 2 * kSlots; ch += kThreads) {
            if ((B.pa[ch >> 1].x & 0xFFFFu) == kNoPiece) continue;
            const ChainRef r = chain_of(B, ch);
            if (r.n == 0) continue;
            int head = r.n, k8 = 0;
            uint32_t by_wave = 0;
            if (r.n > len + len / 2) {
                head = len;
                if (r.type != kLine) {
                    k8 = crossings_before(r.type, r.a, r.line0, r.neg, r.t0, kEighth * r.t1, r.n);
                    if (k8) head = max(len, crossings_before(r.type, r.a, r.line0, r.neg, r.t0, kHeadTau * r.t1, r.n));
                    int w = kLongHeads;
                    if (head > kLongHead || k8 > kLongEighth) w = atomicAdd(&B.n_long, 1);
                    if (w < kLongHeads) {
                        B.longs[w] = (uint16_t)ch;
                        by_wave = kByWave;
                        head = max(head, k8);
                    }
                }
                if (r.n - head < len / 2) head = r.n;
            }
            B.head[ch] = (uint16_t)head;
            const int m = seg_rest(r.n, head, len);
            int at = atomicAdd(&B.n_segs, 1 + m);
            B.seg[at++] = (uint32_t)ch | by_wave;
            if (head >= r.n) continue;
            const int first = at;
            ++n_split;
            int k16 = 0, n8 = 0, n16 = 0;
            if (k8) k16 = crossings_before(r.type, r.a, r.line0, r.neg, r.t0, 0.0625f * r.t1, r.n);
            for (int j = 0; j < m; ++j) {
                const int i0 = head + seg_begin(r.n - head, m, j);
                const int warm = i0 >= k8 ? kWarm : (i0 >= k16 ? kWarm8 : kWarm16);
                B.seg[at++] = (uint32_t)ch | ((uint32_t)(j + 1) << 10) | ((uint32_t)warm << 20);
                n16 += i0 < k16 ? 1 : 0;
                n8 += i0 >= k16 && i0 < k8 ? 1 : 0;
            }
            if constexpr (CANDS) {
                // candidate starts for the segments below t1 / 8, as long as there is room
                const int want = n16 * kCand16 + n8 * kCand8;
                if (want == 0 || want > kCands) continue;
                const int c0 = atomicAdd(&cands.n_cands, want);
                if (c0 + want > kCands) continue;
                const int w = atomicAdd(&cands.n_walks, 1);
                if (w >= kWalks) continue;
                cands.walk[w] = make_uint2((uint32_t)ch | ((uint32_t)n16 << 10) | ((uint32_t)n8 << 20), (uint32_t)c0);
                for (int j = 0, c = c0; j < n16 + n8; ++j) {
                    B.seg[first + j] |= kHasCands | ((uint32_t)(c >> 3) << 26);
                    const int n = j < n16 ? kCand16 : kCand8;
                    for (int k = 0; k < n; ++k, ++c)  // numbered around kCand16
                        cands.cand[c] = (uint32_t)ch | ((uint32_t)(j + 1) << 10) | ((uint32_t)(kCand16 - n / 2 + k) << 20);
                }
            }
        }
        __syncthreads();
        const int S = __builtin_amdgcn_readfirstlane(B.n_segs);
        int n_cands = 0, n_walks = 0;
        if constexpr (CANDS) {
            // only beside a single round of segments
            if (S <= kThreads) n_cands = min(__builtin_amdgcn_readfirstlane(cands.n_cands), kCands);
            if (n_cands) n_walks = min(__builtin_amdgcn_readfirstlane(cands.n_walks), kWalks);
        }

        // ---- the long starts, a wave each
        const int n_long = min(__builtin_amdgcn_readfirstlane(B.n_long), kLongHeads);
        if (n_long) {
            const TreeNode N = tree_node(lane);
#pragma unroll 1
            for (int i = wave; i < n_long; i += kWaves) {
                const int ch = __builtin_amdgcn_readfirstlane((int)B.longs[i]);
                const ChainRef r = chain_of(B, ch);
                float* vs = B.v + r.at;
                solve_wave_any(N, r.type, r.a, r.line0, r.neg ? -2.0f : 2.0f, r.side, r.t1, (int)B.head[ch], r.t0,
                               [&](int k, float v) { if (lane == 0) vs[k] = v; });
            }
        }

        // ---- the crossings, one segment per lane
        for (int s0 = 0; s0 < S; s0 += kThreads) {
            const bool on = s0 + tid < S;
            const uint32_t e = B.seg[on ? s0 + tid : s0];
            const int ch = (int)(e & 1023u);
            const ChainRef r = chain_of(B, ch);
            int i0, i1;
            seg_range(B, ch, (int)((e >> 10) & 1023u), r.n, len, i0, i1);
            float* vs = B.v + r.at;
            // solve, then the guesses against what the segments before ended on: a segment whose
            // guess was off is solved again from there
            float g = r.t0, start = r.t0;
            int k0 = max(0, i0 - (int)((e >> 20) & 31u));
            bool run = on && !(i0 == 0 && (e & kByWave)), redo = false;
            for (;;) {
                if (run) {
                    const float got = solve_run_any(r.type, r.a, r.line0, r.neg, r.side, r.t1, k0, i0, i1, start, redo, vs);
                    if (!redo) g = got;
                }
                if constexpr (CANDS) {
                    if (n_walks && !redo) try_candidates(B, cands, n_cands, S, len, B.v);
                }
                __syncthreads();
                float is = on && i0 > 0 ? vs[i0 - 1] : g;
                if constexpr (CANDS) {
                    if (n_walks && !redo) {
                        if (tid < n_walks) walk_candidates(B, cands, cands.walk[tid]);
                        __syncthreads();
                        if (on && (e & kHasCands)) {
                            const uint32_t p = cands.start[(e >> 26) * 8];
                            if (p != kNoValue) is = bitsf(p);
                        }
                    }
                }
                run = fbits(is) != fbits(g);
                if (!__syncthreads_or(run ? 1 : 0)) break;
                g = start = is;
                k0 = i0;
                redo = true;
            }
        }

        // ---- the order of each piece's sequences, then the merge
        bool falls = false;
        for (int e = tid; e < n_slots; e += kThreads) {
            const int p = piece_of(B, e);
            if (p < 0) continue;
            const int base = (int)(B.pa[p].x & 0xFFFFu), nx = (int)(B.pa[p].x >> 16), ny = (int)(B.pa[p].y & 0xFFFFu);
            const int idx = e - base;
            if (idx < 1 || idx > nx + ny) continue;
            const float v = B.v[e];
            // the y chain follows the piece start, the x chain only without a y chain; a NaN goes both ways
            const float prev = idx == 1 + nx ? B.v[base] : (idx == 1 && ny > 0 ? v : B.v[e - 1]);
            if (!(v >= prev)) { falls = true; atomicOr(&B.pa[p].y, kPwFalls); }
        }
        const bool any_falls = __syncthreads_or(falls ? 1 : 0) != 0;
        if (any_falls) {
            for (int e = tid; e < n_slots; e += kThreads) {
                const int p = piece_of(B, e);
                if (p < 0) continue;
                const uint32_t w1 = B.pa[p].y;
                if (!(w1 & kPwFalls)) continue;
                const int base = (int)(B.pa[p].x & 0xFFFFu), nx = (int)(B.pa[p].x >> 16), ny = (int)(w1 & 0xFFFFu);
                const int idx = e - base;
                if (idx < 1 || idx > nx + ny) continue;
                const float v = B.v[e];
                const float prev = idx == 1 + nx ? B.v[base] : (idx == 1 && ny > 0 ? v : B.v[e - 1]);
                if (!(v <= prev)) atomicOr(&B.pa[p].y, kPwRises);
            }
            __syncthreads();
        }
        for (int s0 = 0; s0 < n_slots;) {
            int s1 = n_slots;
            if (n_slots - s0 > kBigPiece) {
                // the pieces that end within kBigPiece slots of s0
                int end_max = 0, next = n_slots;
                for (int p = lane; p < kSlots; p += kLanes) {
                    const uint32_t w0 = B.pa[p].x;
                    const int base = (int)(w0 & 0xFFFFu);
                    if (base == (int)kNoPiece) continue;
                    const int end = base + 1 + (int)(w0 >> 16) + (int)(B.pa[p].y & 0xFFFFu);
                    if (base >= s0 && end <= s0 + kBigPiece) end_max = max(end_max, end);
                    if (base > s0) next = min(next, base);
                }
#pragma unroll
                for (int o = 32; o >= 1; o >>= 1) {
                    end_max = max(end_max, __shfl_xor(end_max, o));
                    next = min(next, __shfl_xor(next, o));
                }
                s1 = __builtin_amdgcn_readfirstlane(end_max);
                if (s1 <= s0) {  // slots that no piece holds: on to the next piece
                    s0 = __builtin_amdgcn_readfirstlane(next);
                    continue;
                }
            }
            merge_slots(B, s0, s1, longest, any_falls, K.scratch + bb0);
            s0 = s1;
        }

        // ---- fragments: lane l evaluates the point of slot e0 + l; a slot's segment runs to the
        // next slot's point, so 64 points serve 63 slots
        for (int e0 = 63 * wave; e0 < n_slots; e0 += 63 * kWaves) {
            const int e = e0 + lane;
            const int p = e < n_slots ? piece_of(B, e) : -1;
            const uint32_t w0 = B.pa[max(p, 0)].x, w1 = B.pa[max(p, 0)].y;
            const int base = (int)(w0 & 0xFFFFu), n = 1 + (int)(w0 >> 16) + (int)(w1 & 0xFFFFu);
            const bool slot = p >= 0 && e - base < n;
            const int lc = (int)((w1 >> 16) & 63u);
            const float4 cx = B.cx[lc], cy = B.cy[lc];
            const int4 cm = B.cm[lc];
            const uint32_t type = type_of_code((w1 >> kPwType) & 3u);
            const uint32_t raw = slot ? fbits(B.v[e]) : 0u;
            const float t = glmax(bitsf(raw & 0xFFFFFFFCu), 0.0f);
            const float px = eval_axis(type, t, cx.x, cx.y, cx.z, cx.w);
            const float py = eval_axis(type, t, cy.x, cy.y, cy.z, cy.w);
            float t1 = __shfl_down(t, 1), qx = __shfl_down(px, 1), qy = __shfl_down(py, 1);
            const bool valid = slot && lane < 63;
            if (valid && e - base == n - 1) {
                const float te = B.tend[p];
                if (te >= 0.0f) {
                    t1 = te;
                    qx = eval_axis(type, te, cx.x, cx.y, cx.z, cx.w);
                    qy = eval_axis(type, te, cy.x, cy.y, cy.z, cy.w);
                }
            }
            uint32_t bucket = 0;
            if (valid) {
                const int2 wh = B.canvas[lc];
                uint32_t yx;
                int swn;
                segment_cell_pts(t < t1, px, py, qx, qy, wh.x, wh.y, yx, swn);
                const int64_t i = (int64_t)bb0 + e;
                bucket = store_fragment(A, i, yx, swn, (uint32_t)cm.w, (uint32_t)cm.x, make_int2(cm.y, cm.z));
                if (A.inter)
                    A.inter[i] = make_int2((int)(cb + lc),
                                           (int)or_merged(reinterpret_cast<const uint32_t*>(B.v) + base, n, e - base));
                if (A.chord) A.chord[i] = make_float4(px, py, qx, qy);
            }
            wave_count(A.hist, bucket, valid);
        }
        __syncthreads();  // the LDS is used again
    }
    n_split = wave_sum(n_split);
    if (lane == 0 && n_split) atomicAdd(K.split_count, n_split);
}

// One workgroup per piece of more than kBigPiece entries.  Pieces up to kStage entries stay in
// LDS; longer ones are solved into chain_t, merged into scratch[base..] and read back from there.
__global__ __launch_bounds__(kBigThreads) void k_big_pieces(const CurveArgs K, const FragArgs A) {
    __shared__ float st_in[kStage];
    __shared__ uint32_t st_out[kStage];
    __shared__ uint32_t s_flags;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int32_t count = K.n_dev && *K.n_dev == 0 ? 0 : *K.big_count;  // a frame over its budget has no entries
    int n_split = 0;
    for (int32_t item = (int32_t)blockIdx.x; item < count; item += (int32_t)gridDim.x) {
        const int32_t slot = K.big[item];
        const uint32_t c = (uint32_t)slot / 5u;
        const int kk = slot - (int)(5u * c);
        const uint32_t path = A.cpath[c];
        int w = A.w, h = A.h;
        if (A.pcanvas) { const int2 cw = A.pcanvas[path]; w = cw.x; h = cw.y; }
        const CurvePts cv = load_curve(A.tpos, A.cpos[c], A.ctype[c], A.cweight, c);
        const float4 qq = K.cuts[c];
        const uint32_t bb = (uint32_t)A.bucket_base[path];
        const int2 pr = A.prow[path];
        PieceGeom g, after;
        g.base = g.nx = g.ny = 0; g.x0 = g.y0 = g.t0 = g.t1 = 0.0f; g.xneg = g.yneg = g.ok = false;
        after = g;
        bool has_after = false;
        walk_pieces(cv, qq, K.ncuts[c], K.offsets[c], K.offsets[c + 1], w, h, [&](int k, const PieceGeom& x) {
            if (k == kk) g = x;
            if (k == kk + 1 && x.ok) { after = x; has_after = true; }
        });
        if (!g.ok) continue;  // counted but not written: left to k_curves as gaps
        const float t_end = has_after ? first_entry_t(cv, after) : 1.0f;
        const int nv = g.nx + g.ny, n = g.n();
        const bool local = n <= kStage;
        // segments: one per thread (as in k_curves)
        const int len = max(kSegMin, (nv + kBigThreads - 5) / (kBigThreads - 4));
        const CurveAxis ax = {{cv.x[0], cv.x[1], cv.x[2], cv.x[3]}}, ay = {{cv.y[0], cv.y[1], cv.y[2], cv.y[3]}};
        const int kx = crossings_before(cv.type, ax, g.x0, g.xneg, g.t0, kEighth * g.t1, g.nx);
        const int ky = crossings_before(cv.type, ay, g.y0, g.yneg, g.t0, kEighth * g.t1, g.ny);
        int hx = min(g.nx, max(len, crossings_before(cv.type, ax, g.x0, g.xneg, g.t0, kHeadTau * g.t1, g.nx)));
        int hy = min(g.ny, max(len, crossings_before(cv.type, ay, g.y0, g.yneg, g.t0, kHeadTau * g.t1, g.ny)));
        const bool wx = cv.type != kLine && hx > kBigLongHead, wy = cv.type != kLine && hy > kBigLongHead;  // by a wave
        if (wx) hx = max(hx, kx);
        if (wy) hy = max(hy, ky);
        const int sx = g.nx ? 1 + seg_rest(g.nx, hx, len) : 0, sy = g.ny ? 1 + seg_rest(g.ny, hy, len) : 0;
        n_split += (sx > 1 ? 1 : 0) + (sy > 1 ? 1 : 0);
        const bool on = tid < sx + sy, ys = tid >= sx;
        const int j = ys ? tid - sx : tid, nn = ys ? g.ny : g.nx, head = ys ? hy : hx, rest = max(1, (ys ? sy : sx) - 1);
        int i0 = 0, i1 = on ? head : 0;
        if (on && j > 0) {
            i0 = head + seg_begin(nn - head, rest, j - 1);
            i1 = head + seg_begin(nn - head, rest, j);
        }
        CurveAxis a;
#pragma unroll
        for (int i = 0; i < 4; ++i) a.c[i] = ys ? ay.c[i] : ax.c[i];
        const float line0 = ys ? g.y0 : g.x0;
        const bool neg = ys ? g.yneg : g.xneg;
        const uint32_t side = ys ? 1u : 0u;
        const int v0 = ys ? g.nx : 0;
        float* gt = K.chain_t + g.base + 1;
        if (tid == 0) s_flags = 0u;
        float gs = g.t0, start = g.t0;
        const float line = line0 + (neg ? -2.0f : 2.0f) * (float)i0;  // the axis' value where this segment starts
        auto beyond = [&](float tau) {
            const float v = eval_axis(cv.type, tau, a.c[0], a.c[1], a.c[2], a.c[3]);
            return neg ? line <= v : line >= v;
        };
        const int warm = beyond(0.125f * g.t1) ? kWarm : (beyond(0.0625f * g.t1) ? kWarm8 : kWarm16);
        int k0 = max(0, i0 - warm);
        // the long first segments by a wave each (as in k_curves)
        if (wave == 0 ? wx : (wave == 1 && wy)) {
            const TreeNode N = tree_node(lane);
            const CurveAxis aw = wave ? ay : ax;
            const int at = wave ? g.nx : 0;
            const float line_w = wave ? g.y0 : g.x0, step_w = (wave ? g.yneg : g.xneg) ? -2.0f : 2.0f;
            const int head_w = wave ? hy : hx;
            if (local) solve_wave_any(N, cv.type, aw, line_w, step_w, (uint32_t)wave, g.t1, head_w, g.t0,
                                      [&](int k, float v) { if (lane == 0) st_in[at + k] = v; });
            else solve_wave_any(N, cv.type, aw, line_w, step_w, (uint32_t)wave, g.t1, head_w, g.t0,
                                [&](int k, float v) { if (lane == 0) gt[at + k] = v; });
        }
        bool run = on && !(j == 0 && (ys ? wy : wx)), redo = false;
        for (;;) {
            if (run) {
                // the two branches keep every pointer in one address space (no flat accesses)
                const float r = local ? solve_run_any(cv.type, a, line0, neg, side, g.t1, k0, i0, i1, start, redo, st_in + v0)
                                      : solve_run_any(cv.type, a, line0, neg, side, g.t1, k0, i0, i1, start, redo, gt + v0);
                if (!redo) gs = r;
            }
            __threadfence_block();
            __syncthreads();
            float is = gs;
            if (on && i0 > 0) is = local ? st_in[v0 + i0 - 1] : gt[v0 + i0 - 1];
            run = fbits(is) != fbits(gs);
            if (!__syncthreads_or(run ? 1 : 0)) break;
            gs = start = is;
            k0 = i0;
            redo = true;
        }
        // the order of the sequences (as in k_curves)
        uint32_t fl = 0;
        for (int i = tid; i < nv; i += kBigThreads) {
            const float v = local ? st_in[i] : gt[i];
            const float before = i == 0 ? v : (local ? st_in[i - 1] : gt[i - 1]);
            const float prev = i == g.nx ? g.t0 : (i == 0 && g.ny == 0 ? g.t0 : before);
            if (!(v >= prev)) fl |= 1u;
            if (!(v <= prev)) fl |= 2u;
        }
        if (fl) atomicOr(&s_flags, fl);
        __syncthreads();
        const uint32_t flags = s_flags;
        const uint8_t mode = (flags & 1u) == 0u ? 0 : ((flags & 2u) == 0u ? 1 : 2);
        PieceMeta m;
        m.pd.base = g.base; m.pd.nx = g.nx; m.pd.ny = g.ny; m.pd.curve = (int32_t)c; m.pd.t0 = g.t0;
        m.t_end = t_end; m.path = path; m.bb = bb; m.w = w; m.h = h; m.pr = pr; m.cv = cv;
        if (local) {
            wave_merge(m.pd, mode, st_in, st_out, tid, kBigThreads);
            __syncthreads();
            piece_fragments(m, st_out, n, A, lane, wave, kBigThreads / 64);
        } else {
            uint32_t* vout = K.scratch + g.base;
            wave_merge(m.pd, mode, gt, vout, tid, kBigThreads);
            __threadfence_block();
            __syncthreads();
            piece_fragments(m, vout, n, A, lane, wave, kBigThreads / 64);
        }
        __syncthreads();
    }
    if (tid == 0 && n_split) atomicAdd(K.split_count, n_split);
}

}  // namespace

hipError_t launch_curves(const CurveArgs& K, const FragArgs& A, hipStream_t s) {
    if (K.C == 0 || K.n == 0) return hipSuccess;
    if (K.window < kCurveWindowMin || K.window > kCurveWindowMax) return hipErrorInvalidValue;
    const int64_t g = (K.n + K.window - 1) / K.window;
    // entries per curve: with a few each, hardly a chain is long enough to be cut (see k_curves)
    if (g <= kFewWindows && K.n >= kLongCurves * (int64_t)K.C) k_curves<true><<<(unsigned)g, kThreads, 0, s>>>(K, A);
    else k_curves<false><<<(unsigned)g, kThreads, 0, s>>>(K, A);
    return hipGetLastError();
}

hipError_t launch_big_pieces(const CurveArgs& K, const FragArgs& A, int n_cu, hipStream_t s) {
    if (K.C == 0 || K.n == 0) return hipSuccess;
    k_big_pieces<<<(unsigned)(n_cu * 4), kBigThreads, 0, s>>>(K, A);
    return hipGetLastError();
}

}  // namespace spr
