// Keypoint relocalisation without the detector: the parts of Frame::ExtractKeyPoints
// (Core/Frame.cc:93-212) and Tracker::Relocalise (Tracking/Tracking.cc:411-467) that do not
// depend on OpenCV's SURF.  The caller supplies the keypoints (pixel positions) and their
// descriptors; the library lifts them to 3-D with the frame's depth and normal maps, matches
// them against the key map's records (the role of cv::cuda::BFMatcher's knnMatch, k = 2, L2)
// and estimates the pose with the reference's RANSAC / Kabsch loop (Optimization/Solver.cc).
#include <hip/hip_runtime.h>
#include <math.h>
#include <stddef.h>
#include <stdint.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "fu_api.h"
#include "fu_keys.h"
#include "fu_mail.h"

using namespace fu;

namespace {

// ---------------------------------------------------------------------------- lifting
// The bounds test of InterpDepth / InterpNormal (Frame.cc:96, :133) compares y with the width
// and x with the height, as written; where it would let the four neighbours fall outside the
// image (y >= rows - 1 on a landscape frame: the reference reads past the image) or the
// position is NaN, the keypoint is refused.
__device__ __forceinline__ bool in_frame(float x, float y, int cols, int rows) {
    if (x <= 1 || y <= 1 || y >= cols - 1 || x >= rows - 1) return false;
    return !(isnan(x) || isnan(y) || x >= cols - 1 || y >= rows - 1);
}

// Frame::InterpDepth (Core/Frame.cc:93-129): bilinear depth at (x, y) from the four
// neighbours, NaN when any is invalid or outside [0.3, cutoff] or the result strays more than
// 5 mm from the upper-left one.
__device__ __forceinline__ float interp_depth(const float* d, int cols, int rows, float x, float y, float cutoff) {
    const float nan = __int_as_float(0x7fffffff);
    if (!in_frame(x, y, cols, rows)) return nan;
    const float cx = x - floorf(x), cy = y - floorf(y);
    const int x0 = (int)floorf(x), x1 = (int)ceilf(x), y0 = (int)floorf(y), y1 = (int)ceilf(y);
    const float d00 = d[y0 * cols + x0];
    if (isnan(d00) || (double)d00 < 0.3 || d00 > cutoff) return nan;
    const float d10 = d[y1 * cols + x0];
    if (isnan(d10) || (double)d10 < 0.3 || d10 > cutoff) return nan;
    const float d01 = d[y0 * cols + x1];
    if (isnan(d01) || (double)d01 < 0.3 || d01 > cutoff) return nan;
    const float d11 = d[y1 * cols + x1];
    if (isnan(d11) || (double)d11 < 0.3 || d11 > cutoff) return nan;
    const float e0 = d01 * cx + d00 * (1 - cx);
    const float e1 = d11 * cx + d10 * (1 - cx);
    const float fin = (1 - cy) * e0 + cy * e1;
    return (double)fabsf(fin - d00) <= 0.005 ? fin : nan;
}

// Frame::InterpNormal (Frame.cc:131-165): the same blend of the four normals (4-D), NaN when
// it differs from the upper-left one by more than 0.1 (4-D norm)
__device__ __forceinline__ f4 interp_normal(const f4* n, int cols, int rows, float x, float y) {
    const float nan = __int_as_float(0x7fffffff);
    const f4 bad = mk4(nan, nan, nan, nan);
    if (!in_frame(x, y, cols, rows)) return bad;
    const float cx = x - floorf(x), cy = y - floorf(y);
    const int x0 = (int)floorf(x), x1 = (int)ceilf(x), y0 = (int)floorf(y), y1 = (int)ceilf(y);
    const f4 d00 = n[y0 * cols + x0], d10 = n[y1 * cols + x0], d01 = n[y0 * cols + x1], d11 = n[y1 * cols + x1];
    const float ax = 1 - cx, ay = 1 - cy;
    const f4 e0 = mk4(d01.x * cx + d00.x * ax, d01.y * cx + d00.y * ax, d01.z * cx + d00.z * ax, d01.w * cx + d00.w * ax);
    const f4 e1 = mk4(d11.x * cx + d10.x * ax, d11.y * cx + d10.y * ax, d11.z * cx + d10.z * ax, d11.w * cx + d10.w * ax);
    const f4 fin = mk4(e0.x * ay + e1.x * cy, e0.y * ay + e1.y * cy, e0.z * ay + e1.z * cy, e0.w * ay + e1.w * cy);
    const f4 df = mk4(fin.x - d00.x, fin.y - d00.y, fin.z - d00.z, fin.w - d00.w);
    const float nm = sqrtf(df.x * df.x + df.y * df.y + df.z * df.z + df.w * df.w);
    return (double)nm <= 0.1 ? fin : bad;
}

struct LiftArgs {
    const float* xy;     // n keypoints (x, y) in pixels
    const float* depth;  // level-0 filtered depth
    const f4* nmap;      // level-0 normals
    int cols, rows, n;
    float fx, fy, cx, cy, cutoff;
    float* pos;          // n x 3
    float* normal;       // n x 4
    unsigned char* ok;   // n
};

// the per-keypoint test and back-projection of ExtractKeyPoints (Frame.cc:184-200)
__global__ void k_lift_keys(LiftArgs a) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.n) return;
    const float x = a.xy[2 * i], y = a.xy[2 * i + 1];
    const float nan = __int_as_float(0x7fffffff);
    float p[3] = {nan, nan, nan};
    f4 nr = mk4(nan, nan, nan, nan);
    bool ok = false;
    const float dp = interp_depth(a.depth, a.cols, a.rows, x, y, a.cutoff);
    if (!isnan(dp) && (double)dp > 0.3 && dp < a.cutoff) {
        const f4 n = interp_normal(a.nmap, a.cols, a.rows, x, y);
        if (!isnan(n.x)) {
            p[0] = dp * (x - a.cx) / a.fx;
            p[1] = dp * (y - a.cy) / a.fy;
            p[2] = dp;
            nr = n;
            ok = true;
        }
    }
    a.pos[3 * i + 0] = p[0];
    a.pos[3 * i + 1] = p[1];
    a.pos[3 * i + 2] = p[2];
    a.normal[4 * i + 0] = nr.x;
    a.normal[4 * i + 1] = nr.y;
    a.normal[4 * i + 2] = nr.z;
    a.normal[4 * i + 3] = nr.w;
    a.ok[i] = ok;
}

// ---------------------------------------------------------------------------- matching
// The two nearest train descriptors of every query descriptor by L2 distance (sqrt of the sum
// of the 64 squared differences, in dimension order); ties go to the lower train index.  All forms
// keep the two smallest (distance, index) pairs in lexicographic order, a total order over the
// candidates (NaN and +inf distances never enter), so the result is that of one lane scanning the
// train set in index order with strict comparisons, whatever the form, the chunks and the order of
// merges:
//   k_match_tile  all pairs by the exact sum.  Work-group: 256 queries, one per lane (its
//                 descriptor in registers), against a chunk of train descriptors staged through
//                 LDS kTile at a time (every lane reads the same record: LDS broadcast); the
//                 chunks' best two are merged by k_match_merge.  Bound by VALU issue, 192
//                 operations a pair;
//   k_match_scan  alone: a wave per query, a lane per train descriptor, for few of both;
//   k_match_bound and k_match_scan, where they leave most pairs out.
// Few of the pairs need the exact sum.  k_match_bound prices every pair on the matrix cores
// (|t|^2 - 2 q.t, FP32) and keeps, per query and chunk of train descriptors, the least lower and
// the least upper bound; k_match_scan, a wave per query, takes the second least upper bound and
// evaluates the chunks whose lower bound does not exceed it, a lane per train descriptor, with
// the sum's own operations and order.  How many remain depends on the descriptors: equal ones,
// distances far below the norms and magnitudes near overflow leave most of them.  A query with
// more than max_scan chunks left goes on a list instead, whose queries k_match_tile takes.
//
// The bounds.  u = 2^-24, Q = |q|^2, T = |t|^2: the price errs by at most 64 u (Q + T) (the dot
// product, doubled, with 2 |q||t| <= Q + T) + 64 u T + 4 u (Q + 3 T) from |q - t|^2 - Q, and the
// exact sum by 67 u |q - t|^2 <= 134 u (Q + T), its root's rounding (ties) by another 8 u (Q + T).
// kSlack = 512 u times (2 T + Q) covers twice that; kTiny covers sums that round towards zero
// below the normal range.  The chunk of a T of kHuge and more (products may overflow) is always
// evaluated, a query with a Q that is not below it evaluates all of them; a T that is NaN is that of a
// descriptor with a NaN, whose distances never enter.
//
// 900 queries against 20,000: all pairs by the exact sum take 153 us; the two passes take 43 + 14.
// The first is bound by its matrix instructions
// (17 us) and the loads under them: with a quarter of the instructions it still takes 28 us.
constexpr int kDesc = 64;
constexpr int kTile = 128;
constexpr int kChunkMin = kTile, kChunkMax = 8192;  // train descriptors
constexpr int kTargetGroups = 4096;
constexpr float kSlack = 0x1p-15f, kTiny = 0x1p-100f, kHuge = 1e37f;

struct Best2 {
    float d0, d1;
    int i0, i1;
};

__device__ __forceinline__ bool lex_less(float d, int i, float e, int j) { return d < e || (d == e && i < j); }

// (d, i) into the best two; the empty slots are (+inf, -1), which no candidate with a finite
// distance ties
__device__ __forceinline__ void push2(Best2& b, float d, int i) {
    if (lex_less(d, i, b.d0, b.i0)) {
        b.d1 = b.d0;
        b.i1 = b.i0;
        b.d0 = d;
        b.i0 = i;
    } else if (lex_less(d, i, b.d1, b.i1)) {
        b.d1 = d;
        b.i1 = i;
    }
}

typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef v4f v4f_word __attribute__((aligned(4)));  // descriptors are aligned as floats are

// A wave: 32 queries (its A operand: lane l holds of query l & 31 the four dimensions of every
// eight from 4 (l >> 5) on, in both operands, so that a load takes 32-byte pieces; the sum's order
// is free) against its chunk, 32 train
// descriptors at a time.  Four waves a SIMD hide each other's loads better than the next
// descriptors loaded ahead, which leave registers for three (44 and 50 us); a chunk's work-groups
// share an XCD's L2 (43 us).
// bound[chunk * nq + query] = {lower, upper}, without the query's own share.
// todo: the list's length, zero for the scan behind.
__global__ __launch_bounds__(256, 4) void k_match_bound(const float* q, int nq, const float* t, int nt, int chunk,
                                                        float2* bound, int* todo) {
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) *todo = 0;
    const int lane = threadIdx.x & 63, n = lane & 31, half = lane >> 5;
    // work-groups go to the eight XCDs in turn: each XCD takes every eighth chunk, all its queries
    const int c = blockIdx.y * 8 + (blockIdx.x & 7);
    const int q0 = ((blockIdx.x >> 3) * 4 + (threadIdx.x >> 6)) * 32;
    const int c0 = c * chunk, c1 = min(nt, c0 + chunk);
    if (q0 >= nq || c0 >= nt) return;  // uniform
    auto fetch = [&](const float* base, int row, v4f (&x)[8]) {
        const auto p = FU_G(const v4f_word, base + (size_t)row * kDesc + half * 4);
#pragma unroll
        for (int k = 0; k < 8; ++k) x[k] = p[2 * k];
    };
    v4f a[8], cur[8];
    fetch(q, min(q0 + n, nq - 1), a);
    float lo[16], hi[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) lo[r] = hi[r] = INFINITY;
    bool bad = false;
#pragma unroll 1
    for (int base = c0; base < c1; base += 32) {
        fetch(t, min(base + n, nt - 1), cur);
        v16f acc = {0.f};
        float T = 0.f;
#pragma unroll
        for (int k = 0; k < 8; ++k)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[k][e], cur[k][e], acc, 0, 0, 0);
                T = fmaf(cur[k][e], cur[k][e], T);
            }
        T += __shfl_xor(T, 32);
        const bool in = base + n < c1, sane = T < kHuge;
        bad = bad || (in && T >= kHuge);
        const float tl = in && sane ? fmaf(T, -2.f * kSlack, T) : INFINITY;
        const float th = in && sane ? fmaf(T, 2.f * kSlack, T) : INFINITY;
        // an infinite price or NaN (columns outside, or whose chunk is evaluated anyway) is no bound
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            lo[r] = fminf(lo[r], fmaf(-2.f, acc[r], tl));
            hi[r] = fminf(hi[r], fmaf(-2.f, acc[r], th));
        }
    }
    // the least over the 32 columns: halves of the rows are exchanged, so that lane n ends with
    // row n >> 1 of its 16
    if (bad)
#pragma unroll
        for (int r = 0; r < 16; ++r) lo[r] = -INFINITY;
#pragma unroll
    for (int h = 8; h >= 1; h >>= 1) {
        const int off = 2 * h;
        const bool up = (n & off) != 0;
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            if (r >= h) break;
            const float gl = up ? lo[r] : lo[r + h], gh = up ? hi[r] : hi[r + h];
            const float kl = up ? lo[r + h] : lo[r], kh = up ? hi[r + h] : hi[r];
            lo[r] = fminf(kl, __shfl_xor(gl, off));
            hi[r] = fminf(kh, __shfl_xor(gh, off));
        }
    }
    const float l = fminf(lo[0], __shfl_xor(lo[0], 1)), h = fminf(hi[0], __shfl_xor(hi[0], 1));
    const int r = n >> 1;                                 // the row, of query:
    const int qi = q0 + 8 * (r >> 2) + 4 * half + (r & 3);
    if (!(n & 1) && qi < nq) bound[(size_t)c * nq + qi] = make_float2(l, h);
}

// distance of train descriptor p to the wave's query
template <class Q>
__device__ __forceinline__ float exact_dist(const Q& q, FU_GPTR(const v4f_word) p) {
    v4f x[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) x[k] = p[k];
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < 16; ++k)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float d = q[4 * k + e] - x[k][e];
            s = s + d * d;
        }
    return sqrtf(s);
}

// the queries that a scan leaves to k_match_tile, and their number (null: there is no list)
struct Todo {
    int* n;
    int* list;
};

// a wave per query; without bounds (null) every chunk is evaluated
__global__ __launch_bounds__(256) void k_match_scan(const float* q, int nq, const float* t, int nt, int chunk, int nchunks,
                                                    const float2* bound, int max_scan, Todo todo, int* idx, float* dist) {
    const int qi = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
    const int lane = threadIdx.x & 63;
    if (qi >= nq) return;  // uniform
    typedef const __attribute__((address_space(4))) float CF;
    CF* qc = (CF*)(q + (size_t)qi * kDesc);
    constexpr int kKeep = 4;  // of the lane's chunks the lower bounds kept, others are read again
    unsigned long long left[kKeep];
    float limit = INFINITY;  // NaN or +inf: all chunks
    if (bound) {
        const float mine = q[(size_t)qi * kDesc + lane];
        float Q = mine * mine;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) Q += __shfl_xor(Q, off);
        // the two least upper bounds
        float h0 = INFINITY, h1 = INFINITY, lo[kKeep];
        auto upper = [&](float h) {
            h1 = fminf(h1, fmaxf(h0, h));
            h0 = fminf(h0, h);
        };
#pragma unroll
        for (int k = 0; k < kKeep; ++k) {
            const int c = k * 64 + lane;
            const float2 b = c < nchunks ? bound[(size_t)c * nq + qi] : make_float2(INFINITY, INFINITY);
            lo[k] = b.x;
            upper(b.y);
        }
        for (int c = kKeep * 64 + lane; c < nchunks; c += 64) upper(bound[(size_t)c * nq + qi].y);
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            const float g0 = __shfl_xor(h0, off), g1 = __shfl_xor(h1, off);
            h1 = fminf(fminf(h1, g1), fmaxf(h0, g0));
            h0 = fminf(h0, g0);
        }
        limit = Q < kHuge ? h1 + 2.f * fmaf(Q, kSlack, kTiny) : INFINITY;
        int count = 0;
#pragma unroll
        for (int k = 0; k < kKeep; ++k) {
            left[k] = __ballot(k * 64 + lane < nchunks && !(lo[k] > limit));
            count += __popcll(left[k]);
        }
        for (int c = kKeep * 64 + lane; c - lane < nchunks; c += 64)
            count += __popcll(__ballot(c < nchunks && !(bound[(size_t)min(c, nchunks - 1) * nq + qi].x > limit)));
        if (count > max_scan) {  // uniform
            if (lane == 0) todo.list[atomicAdd(todo.n, 1)] = qi;
            return;
        }
    }
    Best2 b{INFINITY, INFINITY, -1, -1};
    for (int base = 0; base < nchunks; base += 64) {
        const int c = base + lane;
        unsigned long long m;
        if (!bound)
            m = __ballot(c < nchunks);
        else if (base >= kKeep * 64)
            m = __ballot(c < nchunks && !(bound[(size_t)min(c, nchunks - 1) * nq + qi].x > limit));
        else
            m = base == 0 ? left[0] : base == 64 ? left[1] : base == 128 ? left[2] : left[3];
        while (m) {
            const int k = base + __builtin_ctzll(m);
            m &= m - 1;
            const int c0 = k * chunk, c1 = min(nt, c0 + chunk);
            for (int r = c0 + lane; r < c1; r += 128) {
                const int r2 = min(r + 64, nt - 1);
                const float d = exact_dist(qc, FU_G(const v4f_word, t + (size_t)r * kDesc));
                const float e = exact_dist(qc, FU_G(const v4f_word, t + (size_t)r2 * kDesc));
                push2(b, d, r);
                if (r + 64 < c1) push2(b, e, r + 64);
            }
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const float d0 = __shfl_xor(b.d0, off), d1 = __shfl_xor(b.d1, off);
        const int i0 = __shfl_xor(b.i0, off), i1 = __shfl_xor(b.i1, off);
        if (i0 >= 0) push2(b, d0, i0);
        if (i1 >= 0) push2(b, d1, i1);
    }
    if (lane == 0) {
        idx[2 * qi] = b.i0;
        idx[2 * qi + 1] = b.i1;
        dist[2 * qi] = b.d0;
        dist[2 * qi + 1] = b.d1;
    }
}

__device__ __forceinline__ void merge(Best2& b, const Best2& p) {
    if (p.i0 >= 0) push2(b, p.d0, p.i0);
    if (p.i1 >= 0) push2(b, p.d1, p.i1);
}

// A chunk's best two as the merge reads them: the indices count from the chunk's first descriptor, 16 bits
// each, kNone where there is none.  12 bytes: an allocation of 2 MB and more takes the stream's pool 45 us
// longer, and 900 queries against 20,000 stay below with these.
struct PartBest {
    float d0, d1;
    unsigned i;
};
constexpr int kNone = 0xFFFF;
static_assert(kChunkMax <= kNone && sizeof(PartBest) >= sizeof(float2), "indices in a chunk; the bounds' place");
// The best two of each query in each chunk, part[chunk * nq + query]; of the queries of the list
// (todo.n not null), in its order.  Launch: a work-group per 256 queries and chunk, of a chunk one after
// the other, or with a list, whose first groups alone may hold queries, of a group, so that all XCDs
// have some.
__global__ __launch_bounds__(256) void k_match_tile(const float* q, int nq, const float* t, int nt, int chunk, int nchunks,
                                                    Todo todo, PartBest* part) {
    __shared__ float tile[kTile * kDesc];
    const unsigned groups = (nq + 255) / 256, id = blockIdx.x;
    const int c = (int)(todo.n ? id % nchunks : id / groups), g = (int)(todo.n ? id / nchunks : id % groups);
    const int at = g * 256 + threadIdx.x, total = todo.n ? *todo.n : nq;
    if (g * 256 >= total) return;  // uniform
    const int c0 = c * chunk, c1 = min(nt, c0 + chunk);
    const int qi = at < total ? (todo.n ? todo.list[at] : at) : -1;
    float mine[kDesc];
#pragma unroll
    for (int j = 0; j < kDesc; ++j) mine[j] = qi >= 0 ? q[(size_t)qi * kDesc + j] : 0.f;
    Best2 b{INFINITY, INFINITY, -1, -1};
    const bool any = __any(qi >= 0);
    for (int base = c0; base < c1; base += kTile) {
        const int cnt = min(kTile, c1 - base);
        __syncthreads();
        for (int k = threadIdx.x; k < cnt * kDesc; k += 256) tile[k] = t[(size_t)base * kDesc + k];
        __syncthreads();
        if (!any) continue;  // uniform in the wave, which only helps to bring the tiles
        for (int r = 0; r < cnt; ++r) {
            float s = 0.f;
#pragma unroll
            for (int j = 0; j < kDesc; ++j) {
                const float dj = mine[j] - tile[r * kDesc + j];
                s = s + dj * dj;
            }
            const float d = sqrtf(s);
            if (d < b.d1) push2(b, d, base + r);  // indices rise within the chunk: d < d1 is the test
        }
    }
    if (qi >= 0)
        part[(size_t)c * nq + at] = PartBest{b.d0, b.d1, (unsigned)(b.i0 >= 0 ? b.i0 - c0 : kNone) |
                                                             (unsigned)(b.i1 >= 0 ? b.i1 - c0 : kNone) << 16};
}
// the chunks' best merged, a wave per query
__global__ __launch_bounds__(256) void k_match_merge(const PartBest* part, int nq, int chunk, int nchunks, Todo todo,
                                                     int* idx, float* dist) {
    const int at = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (at >= (todo.n ? *todo.n : nq)) return;
    Best2 b{INFINITY, INFINITY, -1, -1};
    for (int c = lane; c < nchunks; c += 64) {
        const PartBest p = part[(size_t)c * nq + at];
        const int i0 = (int)(p.i & 0xFFFFu), i1 = (int)(p.i >> 16);
        merge(b, Best2{p.d0, p.d1, i0 == kNone ? -1 : c * chunk + i0, i1 == kNone ? -1 : c * chunk + i1});
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
        merge(b, Best2{__shfl_xor(b.d0, off), __shfl_xor(b.d1, off), __shfl_xor(b.i0, off), __shfl_xor(b.i1, off)});
    if (lane == 0) {
        const int qi = todo.n ? todo.list[at] : at;
        idx[2 * qi] = b.i0;
        idx[2 * qi + 1] = b.i1;
        dist[2 * qi] = b.d0;
        dist[2 * qi + 1] = b.d1;
    }
}

// train descriptors per chunk: about kTargetGroups chunks of 256 queries in all, at least
// kChunkMin and at most kChunkMax, a whole number of kChunkMin
static int match_chunk_len(int nq, int nt) {
    const long long qgroups = (nq + 255) / 256;
    long long want = ((long long)nt * qgroups + kTargetGroups - 1) / kTargetGroups;
    want = (want + kChunkMin - 1) / kChunkMin * kChunkMin;
    return (int)std::min<long long>(kChunkMax, std::max<long long>(kChunkMin, want));
}

// Which form a call takes, by times of all three in us (all pairs / scan alone / bounds, random unit
// descriptors):
//     1000 x 512     98 /  18 /  28      8000 x 256    102 /   61 /   84     16000 x 1000   132 /  438 /  156
//     1000 x 1000    99 /  33 /  28      8000 x 512    104 /  116 /   85     20000 x 2100   271 / 1150 /  242
//     1000 x 20000  157 /  -  /  62     16000 x 256    106 /  116 /  154     20000 x 4000   409 /    - /  290
//     4000 x 4000   121 / 439 /  74     16000 x 20000 1285 /    - /  817    100000 x 4000  1574 /    - / 2877
// A scan alone costs by the pair, all pairs at least 95 us, which 2^22 pairs fill; the bounds need chunks
// to leave out, and many queries make few long ones.
enum MatchForm : int { kAll, kScan, kBounds };
static MatchForm match_form(int nq, int nt, int nchunks) {
    if (nt <= 512 && nq <= 16384 && (long long)nq * nt <= 1ll << 21) return kScan;
    return nq <= 8192 || nchunks >= 32 ? kBounds : kAll;
}
// The most chunks that a query's scan takes: those that take as long as the list would if every query
// were on it.  A scan takes 3.7 us per 128 descriptors while its waves find SIMDs of their own, then
// 4.9 ns per query; the list 95 us, then 0.67 ns per query and 128 descriptors.  Two chunks hold a
// query's nearest, so three at least.  Equal descriptors in every chunk, of which none can be left out,
// 900 x 20000: 590 us with every chunk scanned, now 215, where all pairs take 156; 4000 x 600: 174 and 98.
static int match_max_scan(int nq, int chunk, int nchunks) {
    const double scan = std::max(3.7, nq * 0.0049) * (chunk / kTile);
    const double list = std::max(95.0, (double)nq * nchunks * (chunk / kTile) * 0.00067);
    return std::max(3, (int)std::min(list / scan, (double)nchunks));
}

// ---------------------------------------------------------------------------- graph selection
// Tracker::GenerateGraph's choice of mutually consistent pairs (Tracking.cc:515-596) over the
// consistency matrix C (row-major n x n, C[a * n + b] = conMatrix(a, b)), without reading the
// matrix back to the host as the reference does:
//   k_rank_sums   the column sums (cv::cuda::reduce over rows): each column's rows in order,
//                 summed in double and rounded to float (OpenCV's order is its own).  A
//                 work-group takes 16 columns: all its lanes stage tiles of kSumRows rows in
//                 LDS, and 16 lanes add them, one per column;
//   k_rank_order  the pairs by rank, largest first (cv::sortIdx descending): a pair's position
//                 is the number of ranks above its own, ties going to the lower index
//                 (std::sort leaves them in no fixed order), counted against LDS tiles of the
//                 ranks by sixteen waves a part each and added; a NaN rank counts as -inf, so
//                 the positions are a permutation;
//   k_select      one 1024-lane work-group per list: the head and the pairs ranked after it
//                 with C[head][pair] > min_score, kept in rank order by a block-wide ballot
//                 prefix until max_sel are selected;
//   k_refine      the refinement test of each selected pair against every later pair of the list,
//                 one wave per pair, its lanes over the later pairs (the test is an "any", so
//                 their order is free).  Bound by the latency of its gathers: the ten work-groups
//                 of k_select took 89 us for both parts of ten lists of 400, most CUs idle, the
//                 two launches take 19 us.
constexpr int kSelLanes = 1024;
constexpr int kMaxSelect = 1024;

constexpr int kSumCols = 16, kSumRows = 512;  // columns and rows per LDS tile of k_rank_sums (32 KB)

// launch: ceil(n / kSumCols) work-groups of 256 lanes.  Lane t loads columns 4 (t & 3) .. +3 of
// rows t >> 2, (t >> 2) + 64, ... of a tile (eight 16-byte loads when the row is whole and
// aligned), the next tile's loads issued before the current one is added from LDS.  Bound by the
// columns' serial sums; with 64 columns and 128 rows a tile the trips for the tiles came to more:
// n = 1125, 20 -> 14 us.
__global__ __launch_bounds__(256) void k_rank_sums(const float* C, int n, float* rank) {
    __shared__ __align__(16) float tile[kSumRows][kSumCols];  // written as 16-byte words
    const int tid = threadIdx.x, col = tid & (kSumCols - 1);
    const int c0 = blockIdx.x * kSumCols;
    constexpr int kLoad = 256 / (kSumCols / 4);  // rows loaded at once
    const int q = tid % (kSumCols / 4) * 4, r_lane = tid / (kSumCols / 4);
    // whole 16-byte words: an aligned matrix and n a multiple of 4 keep every row start aligned
    const bool vec = ((uintptr_t)C & 15) == 0 && (n & 3) == 0 && c0 + q + 3 < n;
    float4 buf[kSumRows / kLoad];
    auto fetch = [&](int r0) {
#pragma unroll
        for (int k = 0; k < kSumRows / kLoad; ++k) {
            const int r = r0 + r_lane + kLoad * k;
            float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
            if (r < n) {
                const float* row = C + (size_t)r * n + c0 + q;
                if (vec) {
                    v = *reinterpret_cast<const float4*>(row);
                } else {
                    v.x = c0 + q < n ? row[0] : 0.f;
                    v.y = c0 + q + 1 < n ? row[1] : 0.f;
                    v.z = c0 + q + 2 < n ? row[2] : 0.f;
                    v.w = c0 + q + 3 < n ? row[3] : 0.f;
                }
            }
            buf[k] = v;
        }
    };
    double s = 0;  // the first lanes: column c0 + col
    fetch(0);
    for (int r0 = 0; r0 < n; r0 += kSumRows) {
        __syncthreads();  // the previous tile is summed
#pragma unroll
        for (int k = 0; k < kSumRows / kLoad; ++k) *reinterpret_cast<float4*>(&tile[r_lane + kLoad * k][q]) = buf[k];
        __syncthreads();
        if (r0 + kSumRows < n) fetch(r0 + kSumRows);
        // rows past n hold +0, which leaves the sum as it is (it starts at +0 and so is never
        // -0), so the last tile is summed to a multiple of 16 rows
        if (tid < kSumCols) {
            const int rows = min(kSumRows, (n - r0 + 15) & ~15);
#pragma unroll 16
            for (int r = 0; r < rows; ++r) s += (double)tile[r][col];
        }
    }
    if (tid < kSumCols && c0 + col < n) rank[c0 + col] = (float)s;
}

__device__ __forceinline__ float rank_key(float v) { return isnan(v) ? -INFINITY : v; }

// launch: ceil(n / 64) work-groups of 1024 lanes; lane (w, l) counts for pair 64 * group + l
// against entries w * 64 .. w * 64 + 63 of every 1024-rank tile (with four waves a tile's 256
// entries a lane were 20 us at n = 1125, now 7)
__global__ __launch_bounds__(1024) void k_rank_order(const float* rank, int n, int* order) {
    __shared__ float tile[1024];
    __shared__ int part[16][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int x = blockIdx.x * 64 + lane;
    const float kx = x < n ? rank_key(rank[x]) : 0.f;
    int pos = 0;
    for (int base = 0; base < n; base += 1024) {
        __syncthreads();
        // slots past n hold -inf: never above a rank, and equal to one only with an index
        // above it, so they never count
        const int k0 = base + threadIdx.x;
        tile[threadIdx.x] = k0 < n ? rank_key(rank[k0]) : -INFINITY;
        __syncthreads();
        const int lo = w * 64;
#pragma unroll 16
        for (int k = lo; k < lo + 64; ++k) {
            const float ky = tile[k];
            pos += (ky > kx) || (ky == kx && base + k < x);
        }
    }
    part[w][lane] = pos;
    __syncthreads();
    if (w == 0 && x < n) {
        int p = 0;
#pragma unroll
        for (int k = 0; k < 16; ++k) p += part[k][lane];
        order[p] = x;
    }
}

struct SelArgs {
    const float* C;
    const int* order;
    int n, max_sel;
    float min_score;
    int* n_selected;  // per list
    int* n_refined;   // per list; k_refine's count of ended work-groups until the last ends
    int* refined;     // max_sel per list; the selected pairs until then, the kept ones marked
};

// the exclusive prefix of `flag` over the work-group (lanes in order) and the total
__device__ __forceinline__ int block_prefix(bool flag, int* wsum, int& total) {
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const unsigned long long bal = __ballot(flag);
    const int in_wave = __popcll(bal & ((1ull << lane) - 1ull));
    __syncthreads();
    if (lane == 0) wsum[wid] = __popcll(bal);
    __syncthreads();
    int before = 0, all = 0;
    for (int w = 0; w < kSelLanes / 64; ++w) {
        const int c = wsum[w];
        before += w < wid ? c : 0;
        all += c;
    }
    total = all;
    return before + in_wave;
}

__global__ __launch_bounds__(kSelLanes) void k_select(SelArgs a) {
    __shared__ int wsum[kSelLanes / 64];
    const int i = blockIdx.x, tid = threadIdx.x;
    if (tid == 0) a.n_refined[i] = 0;
    if (i >= a.n) {  // no pairs from this rank on (Tracking.cc:538)
        if (tid == 0) a.n_selected[i] = 0;
        return;
    }
    const int head = a.order[i];
    const float* Ch = a.C + (size_t)head * a.n;
    int* sel = a.refined + (size_t)i * a.max_sel;
    int count = 1;  // the head is always taken (:544-548)
    if (tid == 0) sel[0] = head;
    for (int base = i + 1; base < a.n && count < a.max_sel; base += kSelLanes) {
        const int j = base + tid;
        int idx = 0;
        bool f = false;
        if (j < a.n) {
            idx = a.order[j];
            f = Ch[idx] > a.min_score;  // :551-555
        }
        int total;
        const int slot = count + block_prefix(f, wsum, total);
        if (f && slot < a.max_sel) sel[slot] = idx;
        count = min(count + total, a.max_sel);  // the same in every lane
    }
    if (tid == 0) a.n_selected[i] = count;
}

// launch: (work-groups per list, lists) of 256 lanes, a wave per pair: as many per list as it has pairs
// in fours, up to kRefineGroups in all; beyond that, with kStage, about kStagedGroups, four per list at
// least, whose waves take several pairs and have the list and its scores with the head in LDS (their
// gathers from C meet in the caches, which more waves at once overrun).  200 lists of 1024 of 3000 pairs:
// 962 us with a wave per pair, 842 with 4096 groups, now 690; 10 lists of 400: 73.
// The work-group that ends last of a list's (counted in its n_refined, the marks written through to the
// memory that all XCDs share) moves the marked pairs together.
constexpr int kRefineGroups = 4096, kStagedGroups = 800;
constexpr int kMark = (int)0x80000000u;  // pair indices are below 46340
template <bool kStage>
__global__ __launch_bounds__(256) void k_refine(SelArgs a) {
    __shared__ int last, wsum[4];
    __shared__ int staged[kStage ? kMaxSelect : 1];
    __shared__ float score[kStage ? kMaxSelect : 1];
    const int i = blockIdx.y, x = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int count = a.n_selected[i];
    if (count < 3) return;  // no PoseEstimate from fewer than three (:565)
    const int groups = min((count + 2) / 4, (int)gridDim.x);
    if (x >= groups) return;
    int* sel = a.refined + (size_t)i * a.max_sel;
    const float* Ch = a.C + (size_t)(sel[0] & ~kMark) * a.n;
    if constexpr (kStage) {
        for (int l = tid; l < count; l += 256) {
            const int b = sel[l] & ~kMark;
            staged[l] = b;
            score[l] = Ch[b];
        }
        __syncthreads();
    }
    // the t-th pair is kept unless a later one is nearly exclusive with it and scores higher
    // with the head (:567-582); the head (t = 0) is never kept
    for (int t = 1 + x * 4 + wid; t < count; t += groups * 4) {
        const int av = kStage ? staged[t] : sel[t] & ~kMark;
        const float ha = kStage ? score[t] : Ch[av];
        const float* Ca = a.C + (size_t)av * a.n;
        bool drop = false;
#pragma unroll 4
        for (int l = t + 1 + lane; l < count; l += 64) {
            const int b = kStage ? staged[l] : sel[l] & ~kMark;
            const bool x = Ca[b] < 5e-3f || a.C[(size_t)b * a.n + av] < 5e-3f;
            drop = drop || ((kStage ? score[l] : Ch[b]) > ha && x);
        }
        if (__ballot(drop) == 0ull && lane == 0)
            __hip_atomic_store(FU_G(int, sel + t), av | kMark, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the wave's marks are in place
    __syncthreads();
    if (tid == 0)
        last = __hip_atomic_fetch_add(FU_G(int, a.n_refined + i), 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == groups - 1;
    __syncthreads();
    if (!last) return;  // uniform
    int v[kMaxSelect / 256];
#pragma unroll
    for (int k = 0; k < kMaxSelect / 256; ++k) {
        const int p = k * 256 + tid;
        v[k] = p < count ? __hip_atomic_load(FU_G(int, sel + p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0;
    }
    unsigned long long m[kMaxSelect / 256];
#pragma unroll
    for (int k = 0; k < kMaxSelect / 256; ++k) m[k] = __ballot((v[k] & kMark) != 0);  // every pair has been read
    int total = 0;
#pragma unroll
    for (int k = 0; k < kMaxSelect / 256; ++k) {
        __syncthreads();  // by every wave; the previous sums are read
        if (lane == 0) wsum[wid] = __popcll(m[k]);
        __syncthreads();
        int at = total + __popcll(m[k] & ((1ull << lane) - 1ull));
        for (int w = 0; w < 4; ++w) {
            at += w < wid ? wsum[w] : 0;
            total += wsum[w];
        }
        if ((v[k] & kMark) != 0) sel[at] = v[k] & ~kMark;
    }
    if (tid == 0) a.n_refined[i] = total;
}

// ---------------------------------------------------------------------------- pose
// PoseEstimate (Optimization/Solver.cc:6-183) in double.  A hypothesis is a function of its draw
// alone, so the device counts the inliers of many at once (k_hypotheses) and the host walks the
// counts as the reference walks its iterations.  Both sides run the functions below, every
// operation of which is an IEEE one: the same counts and the same pose, whichever side counts.
#define FU_HD __host__ __device__ __forceinline__

// 3x3 helpers, row-major
struct M3d {
    double a[9];
};
FU_HD M3d mul(const M3d& x, const M3d& y) {
    M3d r;
    for (int i = 0; i < 3; ++i)
        for (int j = 0; j < 3; ++j) r.a[i * 3 + j] = x.a[i * 3] * y.a[j] + x.a[i * 3 + 1] * y.a[3 + j] + x.a[i * 3 + 2] * y.a[6 + j];
    return r;
}
FU_HD M3d transpose(const M3d& x) {
    M3d r;
    for (int i = 0; i < 3; ++i)
        for (int j = 0; j < 3; ++j) r.a[i * 3 + j] = x.a[j * 3 + i];
    return r;
}
FU_HD double det(const M3d& m) {
    const double* a = m.a;
    return a[0] * (a[4] * a[8] - a[5] * a[7]) - a[1] * (a[3] * a[8] - a[5] * a[6]) + a[2] * (a[3] * a[7] - a[4] * a[6]);
}

// R = U V^T for Ab = U S V^T (the Kabsch rotation of Solver.cc, R = (V U^T)^T).  One-sided
// Jacobi on the columns of Ab gives Ab V = U S; a singular vector of a zero singular value
// (three points of a sample span a plane) is completed as the cross product of the other two,
// on both sides, so such a sample yields the proper rotation.
FU_HD M3d kabsch(const M3d& Ab) {
    double A[9], V[9] = {1, 0, 0, 0, 1, 0, 0, 0, 1};
    for (int k = 0; k < 9; ++k) A[k] = Ab.a[k];
    for (int sweep = 0; sweep < 40; ++sweep) {
        double off = 0;
#pragma unroll
        for (int pq = 0; pq < 3; ++pq) {
                const int p = pq < 2 ? 0 : 1, q = pq < 1 ? 1 : 2;
                double al = 0, be = 0, ga = 0;
                for (int i = 0; i < 3; ++i) {
                    al += A[i * 3 + p] * A[i * 3 + p];
                    be += A[i * 3 + q] * A[i * 3 + q];
                    ga += A[i * 3 + p] * A[i * 3 + q];
                }
                if (ga == 0 || fabs(ga) <= 1e-15 * sqrt(al * be)) continue;
                off = fmax(off, fabs(ga) / sqrt(al * be));
                const double z = (be - al) / (2 * ga);
                const double t = (z >= 0 ? 1.0 : -1.0) / (fabs(z) + sqrt(1 + z * z));
                const double c = 1 / sqrt(1 + t * t), s = c * t;
                for (int i = 0; i < 3; ++i) {
                    const double ap = A[i * 3 + p], aq = A[i * 3 + q];
                    A[i * 3 + p] = c * ap - s * aq;
                    A[i * 3 + q] = s * ap + c * aq;
                    const double vp = V[i * 3 + p], vq = V[i * 3 + q];
                    V[i * 3 + p] = c * vp - s * vq;
                    V[i * 3 + q] = s * vp + c * vq;
                }
            }
        if (off < 1e-15) break;
    }
    // singular values (column norms), largest first: the columns in order, a later one ahead of an
    // earlier where it is strictly larger
    double sv[3];
    for (int k = 0; k < 3; ++k) sv[k] = sqrt(A[k] * A[k] + A[3 + k] * A[3 + k] + A[6 + k] * A[6 + k]);
    auto exchange = [&](int x, int y) {
        auto swap = [](double& u, double& v) {
            const double w = u;
            u = v;
            v = w;
        };
        swap(sv[x], sv[y]);
        for (int i = 0; i < 3; ++i) {
            swap(A[i * 3 + x], A[i * 3 + y]);
            swap(V[i * 3 + x], V[i * 3 + y]);
        }
    };
    if (sv[1] > sv[0]) exchange(0, 1);
    if (sv[2] > sv[0]) {
        exchange(1, 2);
        exchange(0, 1);
    } else if (sv[2] > sv[1]) {
        exchange(1, 2);
    }
    double U[9], W[9];
    for (int c = 0; c < 3; ++c) {
        const double inv = sv[c] > 0 ? 1 / sv[c] : 0;
        for (int i = 0; i < 3; ++i) {
            W[i * 3 + c] = V[i * 3 + c];
            U[i * 3 + c] = A[i * 3 + c] * inv;
        }
    }
    if (sv[2] <= 1e-12 * fmax(sv[0], 1e-300)) {
        // rank <= 2: third columns as cross products of the first two
        U[2] = U[3] * U[7] - U[6] * U[4];
        U[5] = U[6] * U[1] - U[0] * U[7];
        U[8] = U[0] * U[4] - U[3] * U[1];
        W[2] = W[3] * W[7] - W[6] * W[4];
        W[5] = W[6] * W[1] - W[0] * W[7];
        W[8] = W[0] * W[4] - W[3] * W[1];
    }
    M3d u, w;
    for (int k = 0; k < 9; ++k) {
        u.a[k] = U[k];
        w.a[k] = W[k];
    }
    return mul(u, transpose(w));
}

struct V3d {
    double x, y, z;
};
FU_HD V3d operator-(V3d a, V3d b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
FU_HD V3d operator+(V3d a, V3d b) { return {a.x + b.x, a.y + b.y, a.z + b.z}; }
FU_HD V3d operator/(V3d a, double s) { return {a.x / s, a.y / s, a.z / s}; }
FU_HD V3d rot(const M3d& R, V3d v) {
    return {R.a[0] * v.x + R.a[1] * v.y + R.a[2] * v.z, R.a[3] * v.x + R.a[4] * v.y + R.a[5] * v.z,
            R.a[6] * v.x + R.a[7] * v.y + R.a[8] * v.z};
}
FU_HD double vnorm(V3d v) { return sqrt(v.x * v.x + v.y * v.y + v.z * v.z); }
FU_HD V3d vcross(V3d a, V3d b) { return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x}; }
FU_HD void outer_add(M3d& m, V3d a, V3d b) {
    const double av[3] = {a.x, a.y, a.z}, bv[3] = {b.x, b.y, b.z};
    for (int i = 0; i < 3; ++i)
        for (int j = 0; j < 3; ++j) m.a[i * 3 + j] += av[i] * bv[j];
}

// number k (from 0) of the sample generator, below n: splitmix64 in place of the reference's
// srand(clock) / rand(), whose state is seed + (k + 1) times a constant
FU_HD int sample(uint64_t seed, uint64_t k, uint32_t n) {
    uint64_t z = seed + (k + 1) * 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    return (int)((uint32_t)((z >> 32) % n));
}

// src = R * ref + t
struct Model {
    M3d R;
    V3d t;
};
FU_HD bool inlier(const Model& m, V3d s, V3d r) {
    const float thresh_inlier = 0.05f;
    return vnorm(s - (rot(m.R, r) + m.t)) <= thresh_inlier;
}

// The model of draw d, three samples of the n pairs p.s(i) / p.r(i): false where the draw gives
// none, with its verdict: kNoModel, or kReflected, after which the iteration is not counted.
enum { kNoModel = -1, kReflected = -2 };
template <class P>
FU_HD bool draw_model(const P& p, int n, uint64_t seed, long long d, Model& m, int& verdict) {
    verdict = kNoModel;
    const int i = sample(seed, 3 * (uint64_t)d, (uint32_t)n), j = sample(seed, 3 * (uint64_t)d + 1, (uint32_t)n),
              k = sample(seed, 3 * (uint64_t)d + 2, (uint32_t)n);
    const bool bad = i == j || j == k || k == i;
    const V3d sa = p.s(i), sb = p.s(j), sc = p.s(k);
    const V3d ra = p.r(i), rb = p.r(j), rc = p.r(k);
    const float sd = (float)vnorm(vcross(sb - sa, sa - sc));  // stored in floats (Solver.cc:52-53)
    const float rd = (float)vnorm(vcross(rb - ra, ra - rc));
    if (bad || (double)sd < 1e-6 || (double)rd < 1e-6) return false;
    const V3d sm = (sa + sb + sc) / 3, rm = (ra + rb + rc) / 3;
    M3d Ab{{0, 0, 0, 0, 0, 0, 0, 0, 0}};
    outer_add(Ab, sa - sm, ra - rm);
    outer_add(Ab, sb - sm, rb - rm);
    outer_add(Ab, sc - sm, rc - rm);
    m.R = kabsch(Ab);
    if (det(m.R) < 0) {  // as Solver.cc:82: a new sample
        verdict = kReflected;
        return false;
    }
    m.t = sm - rot(m.R, rm);
    return true;
}

// The pairs on the device: those of the ratio test (a frame point by its index, the map's point) ...
struct RatioPair {
    int query;
    float pos[3];
};
struct RatioPoints {
    const int* count;
    const RatioPair* pair;
    const double* frame;
    __device__ int begin() { return *count; }
    __device__ V3d s(int i) const {
        const double* f = frame + 3 * (size_t)pair[i].query;
        return V3d{f[0], f[1], f[2]};
    }
    __device__ V3d r(int i) const {
        const RatioPair& k = pair[i];
        return V3d{(double)k.pos[0], (double)k.pos[1], (double)k.pos[2]};
    }
};
// ... or the refined pairs of the first list that selected three or more
struct ListPoints {
    const int* n_selected;
    const int* n_refined;
    const int* list;
    int lists, max_sel;
    const SurfHead* frame;
    const SurfHead* map;
    __device__ int begin() {
        for (int i = 0; i < lists; ++i)
            if (n_selected[i] >= 3) {
                list += (size_t)i * max_sel;
                return n_refined[i];
            }
        return 0;
    }
    __device__ V3d s(int i) const {
        const float* f = frame[list[i]].pos;
        return V3d{(double)f[0], (double)f[1], (double)f[2]};
    }
    __device__ V3d r(int i) const {
        const float* f = map[list[i]].pos;
        return V3d{(double)f[0], (double)f[1], (double)f[2]};
    }
};

// The inliers of draws first .. first + gridDim.x - 1 of call blockIdx.y (which draws from seed +
// blockIdx.y), a wave each: its lanes run the serial model side by side, then take the pairs 64 at
// a time.  Bound by the model's chain of divisions and roots.  100 draws of five calls over 380
// pairs took a host thread per call 500 us, here 14 us.
template <class P>
__global__ __launch_bounds__(64) void k_hypotheses(P p, uint64_t seed, long long first, int stride, int* verdict) {
    const int n = p.begin();
    if (n < 3) return;  // uniform
    Model m;
    int v;
    if (draw_model(p, n, seed + blockIdx.y, first + blockIdx.x, m, v)) {
        v = 0;
        for (int i = threadIdx.x; i - (int)threadIdx.x < n; i += 64) {
            const bool in = i < n && inlier(m, p.s(min(i, n - 1)), p.r(min(i, n - 1)));
            v += __popcll(__ballot(in));
        }
    }
    if (threadIdx.x == 0) verdict[blockIdx.y * stride + blockIdx.x] = v;
}

// the pairs on the host
struct HostPoints {
    const double* src;
    const double* ref;
    FU_HD V3d s(int i) const { return V3d{src[3 * i], src[3 * i + 1], src[3 * i + 2]}; }
    FU_HD V3d r(int i) const { return V3d{ref[3 * i], ref[3 * i + 1], ref[3 * i + 2]}; }
};

// Solver::PoseEstimate (Optimization/Solver.cc:6-183), checkAngle = false, over the verdicts of its
// draws: verdict(d, v) gives draw d's kNoModel, kReflected or count of inliers.  Only the last
// accepted hypothesis' refined model and the last evaluated one's outliers reach the result, so
// only those two are worked out here.
template <class V>
fu_status pose_estimate(const HostPoints& p, int n, int iterations, uint64_t seed, V&& verdict, double T[16],
                        uint8_t* inliers, int32_t* ok) {
    *ok = 0;
    for (int k = 0; k < 16; ++k) T[k] = (k % 5 == 0) ? 1.0 : 0.0;
    if (n < 3) return FU_OK;
    const float thresh_confidence = 0.95f;
    const int min_iter = 20;
    int inliers_best = 0, it = 0;
    long long best = -1, evaluated = -1;
    // a reflection re-draws without counting the iteration (as the reference); a three-point
    // sample spans at most a plane and its completed bases are right-handed, so that does not
    // repeat, but the draws are bounded all the same
    long long draws = 0;
    const long long max_draws = 64ll * (iterations > 0 ? iterations : 1);
    while (it < iterations && draws < max_draws) {
        const long long d = draws++;
        int nin = 0;
        const fu_status st = verdict(d, nin);
        if (st) return st;
        if (nin == kReflected) continue;
        if (nin >= 0) evaluated = d;
        if (nin > inliers_best) {
            best = d;
            inliers_best = nin;
            const float ratio = (float)nin / (float)n;
            // pow of a float and an int is the double pow (Solver.cc:124)
            const float confidence = (float)(1 - pow(1 - pow((double)ratio, 3), (double)(it + 1)));
            if (it >= min_iter && confidence >= thresh_confidence) break;
        }
        ++it;
    }
    if (evaluated < 0) return FU_OK;  // no hypothesis was evaluated
    std::vector<char> outlier(n);
    auto mark = [&](long long d) {  // the outliers of draw d's model (Solver.cc:84-93)
        Model m;
        int v;
        (void)draw_model(p, n, seed, d, m, v);
        for (int i = 0; i < n; ++i) outlier[i] = !inlier(m, p.s(i), p.r(i));
    };
    // the model of the pairs that are not outliers: false if there are none
    auto refit = [&](Model& m) {
        V3d smn{0, 0, 0}, rmn{0, 0, 0};
        int N = 0;
        for (int i = 0; i < n; ++i)
            if (!outlier[i]) {
                smn = smn + p.s(i);
                rmn = rmn + p.r(i);
                ++N;
            }
        if (N == 0) return false;
        smn = smn / N;
        rmn = rmn / N;
        M3d Ab{{0, 0, 0, 0, 0, 0, 0, 0, 0}};
        for (int i = 0; i < n; ++i)
            if (!outlier[i]) outer_add(Ab, p.s(i) - smn, p.r(i) - rmn);
        m.R = kabsch(Ab);
        m.t = smn - rot(m.R, rmn);
        return true;
    };
    Model m{M3d{{1, 0, 0, 0, 1, 0, 0, 0, 1}}, V3d{0, 0, 0}};
    if (best >= 0) {
        mark(best);
        refit(m);
    }
    // the final set: the best model's inliers added to the last evaluated hypothesis' (the
    // reference does not reset the flags first, Solver.cc:138-143)
    mark(evaluated);
    for (int i = 0; i < n; ++i)
        if (inlier(m, p.s(i), p.r(i))) outlier[i] = 0;
    if (!refit(m) || det(m.R) < 0) return FU_OK;
    for (int i = 0; i < 3; ++i) {
        for (int j = 0; j < 3; ++j) T[i * 4 + j] = m.R.a[i * 3 + j];
    }
    T[3] = m.t.x;
    T[7] = m.t.y;
    T[11] = m.t.z;
    if (inliers)
        for (int i = 0; i < n; ++i) inliers[i] = !outlier[i];
    *ok = 1;
    return FU_OK;
}

}  // namespace

// ---------------------------------------------------------------------------- C ABI
extern "C" fu_status fu_lift_keypoints(const float* xy, int32_t n, const float* depth, const float* nmap, int32_t cols,
                                       int32_t rows, float fx, float fy, float cx, float cy, float depth_cutoff,
                                       float* pos, float* normal, uint8_t* ok, fu_stream s) {
    if (n < 0 || cols < 1 || rows < 1) return api_error(FU_ERR_ARG, "fu_lift_keypoints: bad sizes");
    if (n == 0) return FU_OK;
    if (!xy || !depth || !nmap || !pos || !normal || !ok) return api_error(FU_ERR_ARG, "fu_lift_keypoints: null argument");
    LiftArgs a{xy, depth, (const f4*)nmap, cols, rows, n, fx, fy, cx, cy, depth_cutoff, pos, normal, ok};
    hipLaunchKernelGGL(k_lift_keys, dim3((n + 255) / 256), dim3(256), 0, (hipStream_t)s, a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return api_error(FU_ERR_HIP, "fu_lift_keypoints: %s", hipGetErrorString(e));
    return FU_OK;
}

extern "C" fu_status fu_match_knn2(const float* query, int32_t nq, const float* train, int32_t nt, int32_t* idx,
                                   float* dist, fu_stream s) {
    if (nq < 0 || nt < 0) return api_error(FU_ERR_ARG, "fu_match_knn2: bad sizes");
    if (nq == 0) return FU_OK;
    if (!query || !idx || !dist || (nt > 0 && !train)) return api_error(FU_ERR_ARG, "fu_match_knn2: null argument");
    if ((long long)nq * kDesc > (1ll << 31) || (long long)nt * kDesc > (1ll << 31))
        return api_error(FU_ERR_ARG, "fu_match_knn2: %d x %d descriptors (at most 2^25 each)", nq, nt);
    hipStream_t hs = (hipStream_t)s;
    const int chunk = match_chunk_len(nq, nt);
    const int nchunks = (nt + chunk - 1) / chunk;
    const MatchForm form = match_form(nq, nt, nchunks);
    const int max_scan = match_max_scan(nq, chunk, nchunks);
    // every chunk's best two of every query (the bounds, read before any of them is written, lie in the
    // same place), then the list
    char* scratch = nullptr;
    const size_t parts = sizeof(PartBest) * (size_t)nchunks * nq, ints = form == kBounds ? 1 + (size_t)nq : 0;
    if (form != kScan && hipMallocAsync((void**)&scratch, parts + sizeof(int) * ints, hs) != hipSuccess) {
        (void)hipGetLastError();
        return api_error(FU_ERR_NOMEM, "fu_match_knn2: %d partial lists", nchunks);
    }
    PartBest* part = reinterpret_cast<PartBest*>(scratch);
    float2* bound = nullptr;
    Todo todo{nullptr, nullptr};
    if (form == kBounds) {
        bound = reinterpret_cast<float2*>(scratch);
        todo.n = reinterpret_cast<int*>(scratch + parts);
        todo.list = todo.n + 1;
        hipLaunchKernelGGL(k_match_bound, dim3((nq + 127) / 128 * 8, (nchunks + 7) / 8), dim3(256), 0, hs, query, nq, train, nt,
                           chunk, bound, todo.n);
    }
    if (form != kAll)
        hipLaunchKernelGGL(k_match_scan, dim3((nq + 3) / 4), dim3(256), 0, hs, query, nq, train, nt, chunk, nchunks, bound,
                           max_scan, todo, idx, dist);
    if (form == kAll || (form == kBounds && nchunks > max_scan)) {
        hipLaunchKernelGGL(k_match_tile, dim3((unsigned)((nq + 255) / 256) * nchunks), dim3(256), 0, hs, query, nq, train, nt,
                           chunk, nchunks, todo, part);
        hipLaunchKernelGGL(k_match_merge, dim3((nq + 3) / 4), dim3(256), 0, hs, part, nq, chunk, nchunks, todo, idx, dist);
    }
    hipError_t e = hipGetLastError();
    if (scratch) {
        const hipError_t ef = hipFreeAsync(scratch, hs);
        if (e == hipSuccess) e = ef;
    }
    if (e != hipSuccess) return api_error(FU_ERR_HIP, "fu_match_knn2: %s", hipGetErrorString(e));
    return FU_OK;
}

// the counts made here, on the host
extern "C" fu_status fu_pose_estimate(const double* src, const double* ref, int32_t n, int32_t iterations,
                                      uint64_t seed, double T[16], uint8_t* inliers, int32_t* ok) {
    if (!src || !ref || !T || !ok || n < 0 || iterations < 0) return api_error(FU_ERR_ARG, "fu_pose_estimate: bad argument");
    const HostPoints p{src, ref};
    auto count = [&](long long d, int& v) {
        Model m;
        if (!draw_model(p, n, seed, d, m, v)) return FU_OK;
        v = 0;
        for (int i = 0; i < n; ++i) v += inlier(m, p.s(i), p.r(i));
        return FU_OK;
    };
    return pose_estimate(p, n, iterations, seed, count, T, inliers, ok);
}

namespace {
// parts of one stream-ordered allocation, 256-byte aligned
struct Block {
    hipStream_t stream;
    char* base = nullptr;
    size_t size = 0;
    explicit Block(hipStream_t s) : stream(s) {}
    Block(const Block&) = delete;
    Block& operator=(const Block&) = delete;
    ~Block() {
        if (base) (void)hipFreeAsync(base, stream);
    }
    size_t part(size_t bytes) {
        const size_t at = size;
        size += (bytes + 255) & ~(size_t)255;
        return at;
    }
    bool allocate() {
        if (hipMallocAsync((void**)&base, size, stream) == hipSuccess) return true;
        (void)hipGetLastError();
        base = nullptr;
        return false;
    }
    template <class T>
    T* at(size_t part) const {
        return reinterpret_cast<T*>(base + part);
    }
};

// The exclusive prefix over a 1024-lane work-group (lanes in order) of c, 0 to 2 per lane as the
// sum of two flags, and the total.
__device__ __forceinline__ int pair_prefix(bool f, bool g, int* wsum, int& total) {
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const unsigned long long bf = __ballot(f), bg = __ballot(g), below = (1ull << lane) - 1ull;
    __syncthreads();
    if (lane == 0) wsum[wid] = __popcll(bf) + __popcll(bg);
    __syncthreads();
    int before = 0, all = 0;
    for (int w = 0; w < 16; ++w) {
        const int c = wsum[w];
        before += w < wid ? c : 0;
        all += c;
    }
    total = all;
    return before + __popcll(bf & below) + __popcll(bg & below);
}

struct PairArgs {
    const int* idx;          // the two nearest map keys of each query
    const float* dist;
    int nq;
    const int* slot;         // of each map key, -1 for key 0
    const SurfHead* heads;   // the map's slots, kSlotHeads apart
};
// The pairs that pass the ratio test (Tracking.cc:437-444; with one map key the second distance is
// infinite) in query order.  One work-group: the prefix is over hundreds of queries.
__global__ __launch_bounds__(1024) void k_ratio_pairs(PairArgs a, RatioPair* out, int* count) {
    __shared__ int wsum[16];
    int n = 0;
    for (int base = 0; base < a.nq; base += 1024) {
        const int i = base + threadIdx.x;
        const int key = i < a.nq ? a.idx[2 * i] : -1;
        const bool f = key >= 0 && (double)a.dist[2 * i] < 0.90 * (double)a.dist[2 * i + 1];
        int total;
        const int at = n + pair_prefix(f, false, wsum, total);
        if (f) {
            const int s = a.slot[key];
            RatioPair p{i, {0.f, 0.f, 0.f}};
            if (s >= 0)
                for (int c = 0; c < 3; ++c) p.pos[c] = a.heads[(size_t)s * kSlotHeads].pos[c];
            out[at] = p;
        }
        n += total;
    }
    if (threadIdx.x == 0) *count = n;
}
// The match list of graph matching (Tracking.cc:437-444): both nearest keys of a query that fails the
// ratio test.  counts[0]: its length; counts[1]: the pairs whose key is valid (:485-505), which are
// written as the frame's and the map's records (without descriptors) and their distance.
__global__ __launch_bounds__(1024) void k_graph_pairs(PairArgs a, const float* fpos, const float* fnrm, SurfHead* fk,
                                                      SurfHead* mk, float* dd, int* counts) {
    __shared__ int wsum[16];
    int listed = 0, n = 0;
    for (int base = 0; base < a.nq; base += 1024) {
        const int i = base + threadIdx.x;
        int key[2] = {-1, -1}, slot[2] = {-1, -1};
        float d[2] = {0.f, 0.f};
        if (i < a.nq) {
            key[0] = a.idx[2 * i];
            d[0] = a.dist[2 * i];
            d[1] = a.dist[2 * i + 1];
            if (key[0] >= 0 && !((double)d[0] < 0.90 * (double)d[1])) key[1] = a.idx[2 * i + 1];
        }
#pragma unroll
        for (int k = 0; k < 2; ++k)
            if (key[k] >= 0) slot[k] = a.slot[key[k]];
        int total;
        (void)pair_prefix(key[0] >= 0, key[1] >= 0, wsum, total);
        listed += total;
        int at = n + pair_prefix(slot[0] >= 0, slot[1] >= 0, wsum, total);
#pragma unroll
        for (int k = 0; k < 2; ++k)
            if (slot[k] >= 0) {
                SurfHead f;
                f.valid = 1;  // the reference leaves this record's flag unset
                f.pad[0] = f.pad[1] = f.pad[2] = 0;
                for (int c = 0; c < 3; ++c) f.pos[c] = fpos[3 * i + c];
                for (int c = 0; c < 4; ++c) f.normal[c] = fnrm[4 * i + c];
                fk[at] = f;
                mk[at] = a.heads[(size_t)slot[k] * kSlotHeads];
                dd[at] = d[k];
                ++at;
            }
        n += total;
    }
    if (threadIdx.x == 0) {
        counts[0] = listed;
        counts[1] = n;
    }
}
// what the host needs of the selection: the lists' counts, then the points of the list whose pose is
// estimated (frame and map, 6 floats a pair)
__global__ __launch_bounds__(1024) void k_list_points(ListPoints p, int* counts, float* points) {
    if ((int)threadIdx.x < p.lists) {
        counts[threadIdx.x] = p.n_selected[threadIdx.x];
        counts[p.lists + threadIdx.x] = p.n_refined[threadIdx.x];
    }
    const int n = p.begin();
    for (int i = threadIdx.x; i < n; i += 1024)
        for (int c = 0; c < 3; ++c) {
            points[6 * i + c] = p.frame[p.list[i]].pos[c];
            points[6 * i + 3 + c] = p.map[p.list[i]].pos[c];
        }
}

// the map's keys (UpdateMapKeys, Mapping.cc:142-151; the first record is never written by
// CollectKeyPoints and reads as zeros here) and the two nearest of them to each frame descriptor,
// on the device.  `out`: idx and dist, 2 per query (-1 / +inf where the map has fewer keys), and the
// keys' slots, which live in `keys`.
fu_status collect_and_match(fu_keymap* km, const KeyScratch& scratch, const float* frame_desc, int32_t nq, uint32_t nk,
                            Block& keys, int32_t* idx, float* dist, PairArgs& out, hipStream_t hs, const char* who) {
    const size_t desc = keys.part(sizeof(float) * kDesc * nk), slot = keys.part(sizeof(int32_t) * nk);
    if (!keys.allocate()) return api_error(FU_ERR_NOMEM, "%s: %u keys", who, nk);
    fu_status st = keymap_pack(km, scratch, keys.at<float>(desc), keys.at<int32_t>(slot), nk, hs);
    if (st) return st;
    if ((st = fu_match_knn2(frame_desc, nq, keys.at<float>(desc), (int32_t)nk, idx, dist, (fu_stream)hs))) return st;
    out = PairArgs{idx, dist, nq, keys.at<int32_t>(slot), keymap_heads(km)};
    return FU_OK;
}

// The draws of the first launch of counts; a call that needs more has the next kMoreDraws counted.
constexpr int kFirstDraws = 256, kMoreDraws = 4096;
template <class P>
struct Counts {
    P points;
    uint64_t seed;
    int dev;
    hipStream_t stream;
    std::vector<int> have;  // of draws base .. base + have.size() - 1 (the walk asks for them in order)
    long long base = 0;
    fu_status operator()(long long d, int& v) {
        if (d >= base + (long long)have.size()) {
            Block block(stream);
            const size_t part = block.part(sizeof(int) * kMoreDraws);
            if (!block.allocate()) return api_error(FU_ERR_NOMEM, "PoseEstimate: %d draws", kMoreDraws);
            hipLaunchKernelGGL(k_hypotheses<P>, dim3(kMoreDraws), dim3(64), 0, stream, points, seed, d, 0,
                               block.at<int>(part));
            base = d;
            have.resize(kMoreDraws);
            hipError_t e = hipGetLastError();
            const hipError_t er = mail_read(dev, have.data(), block.at<int>(part), sizeof(int) * kMoreDraws, stream);
            if (e == hipSuccess) e = er;
            if (e != hipSuccess) return api_error(FU_ERR_HIP, "PoseEstimate: %s", hipGetErrorString(e));
        }
        v = have[(size_t)(d - base)];
        return FU_OK;
    }
};

// the camera pose of a PoseEstimate transform T (frame point = R * map point + t): T^-1
void rigid_inverse(const double T[16], double pose[16]) {
    for (int i = 0; i < 3; ++i) {
        for (int j = 0; j < 3; ++j) pose[i * 4 + j] = T[j * 4 + i];
        pose[i * 4 + 3] = -(T[0 * 4 + i] * T[3] + T[1 * 4 + i] * T[7] + T[2 * 4 + i] * T[11]);
    }
    pose[12] = pose[13] = pose[14] = 0;
    pose[15] = 1;
}
}  // namespace

// Tracker::Relocalise with useGraphMatching off, its default (Tracking.cc:411-467): the map's
// keys, the two nearest map descriptors of every frame descriptor, the ratio test
// d0 < 0.9 d1, PoseEstimate over the surviving pairs (frame point <- map point) and the pose
// as the inverse of its transform.  frame_desc: nq x 64 floats in device memory; frame_pos:
// nq x 3 doubles on the host (the lifted keypoints).
extern "C" fu_status fu_relocalise_keys(fu_keymap* km, const float* frame_desc, const double* frame_pos, int32_t nq,
                                        int32_t iterations, uint64_t seed, double pose[16], int32_t* n_pairs,
                                        int32_t* ok, fu_stream s) {
    if (!km || !pose || !ok || nq < 0 || (nq > 0 && (!frame_desc || !frame_pos)))
        return api_error(FU_ERR_ARG, "fu_relocalise_keys: bad argument");
    *ok = 0;
    if (n_pairs) *n_pairs = 0;
    for (int k = 0; k < 16; ++k) pose[k] = (k % 5 == 0) ? 1.0 : 0.0;
    hipStream_t hs = (hipStream_t)s;
    uint32_t nk = 0;
    fu_status st = keymap_count(km, nk, hs);
    if (st) return st;
    if (nk == 0 || nq == 0) return FU_OK;  // no map keys (Tracking.cc:417-418)
    KeyScratch scratch(km, hs);
    const int draws = std::max(0, std::min(iterations, kFirstDraws));
    Block keys(hs), work(hs);
    const size_t fpos = work.part(sizeof(double) * 3 * nq), idx = work.part(sizeof(int32_t) * 2 * nq),
                 dist = work.part(sizeof(float) * 2 * nq), head = work.part(sizeof(int) * (1 + kFirstDraws)),
                 pairs = work.part(sizeof(RatioPair) * nq);
    if (!work.allocate()) return api_error(FU_ERR_NOMEM, "fu_relocalise_keys: %d keypoints", nq);
    PairArgs pa{};
    if ((st = collect_and_match(km, scratch, frame_desc, nq, nk, keys, work.at<int32_t>(idx), work.at<float>(dist), pa, hs,
                                "fu_relocalise_keys")))
        return st;
    hipError_t e = hipMemcpyAsync(work.at<double>(fpos), frame_pos, sizeof(double) * 3 * nq, hipMemcpyHostToDevice, hs);
    int* dhead = work.at<int>(head);
    RatioPair* dpairs = work.at<RatioPair>(pairs);
    const RatioPoints points{dhead, dpairs, work.at<double>(fpos)};
    hipLaunchKernelGGL(k_ratio_pairs, dim3(1), dim3(1024), 0, hs, pa, dpairs, dhead);
    if (draws > 0)
        hipLaunchKernelGGL(k_hypotheses<RatioPoints>, dim3(draws), dim3(64), 0, hs, points, seed, 0ll, 0, dhead + 1);
    if (e == hipSuccess) e = hipGetLastError();
    // the pairs with the counts, as many as go with them
    std::vector<int> hhead(1 + draws);
    std::vector<RatioPair> hp(nq);
    const size_t hbytes = sizeof(int) * hhead.size();
    const int first = (int)std::min<size_t>(nq, (kMailBytes - hbytes) / sizeof(RatioPair));
    const int dev = keymap_device(km);
    // also after a failure: nothing queued may still read the caller's memory
    const hipError_t er = mail_read(dev, hhead.data(), dhead, hbytes, hp.data(), dpairs, sizeof(RatioPair) * first, hs);
    if (er == hipSuccess) scratch.done();
    if (e == hipSuccess) e = er;
    const int np = e == hipSuccess ? hhead[0] : 0;
    if (np > first) {
        e = hipMemcpyAsync(hp.data() + first, dpairs + first, sizeof(RatioPair) * (np - first), hipMemcpyDeviceToHost, hs);
        const hipError_t es = hipStreamSynchronize(hs);
        if (e == hipSuccess) e = es;
    }
    if (e != hipSuccess) return api_error(FU_ERR_HIP, "fu_relocalise_keys: %s", hipGetErrorString(e));
    if (n_pairs) *n_pairs = np;
    if (np < 3) return FU_OK;
    if (iterations < 0) return api_error(FU_ERR_ARG, "fu_pose_estimate: bad argument");
    std::vector<double> src(3 * (size_t)np), ref(3 * (size_t)np);
    for (int k = 0; k < np; ++k)
        for (int c = 0; c < 3; ++c) {
            src[3 * k + c] = frame_pos[3 * (size_t)hp[k].query + c];
            ref[3 * k + c] = (double)hp[k].pos[c];
        }
    Counts<RatioPoints> counts{points, seed, dev, hs, std::vector<int>(hhead.begin() + 1, hhead.end())};
    double T[16];
    int32_t good = 0;
    if ((st = pose_estimate(HostPoints{src.data(), ref.data()}, np, iterations, seed, counts, T, nullptr, &good))) return st;
    if (!good) return FU_OK;
    rigid_inverse(T, pose);
    *ok = 1;
    return FU_OK;
}

// GenerateGraph's selection on the device (Tracking.cc:515-596)
extern "C" fu_status fu_select_subgraphs(const float* matrix, int32_t n, int32_t n_lists, int32_t max_select,
                                         float min_score, float* rank_sum, int32_t* order, int32_t* n_selected,
                                         int32_t* n_refined, int32_t* refined, fu_stream s) {
    if (n < 0 || n > 46340 || n_lists < 1 || n_lists > 65535 || max_select < 1 || max_select > kMaxSelect)
        return api_error(FU_ERR_ARG, "fu_select_subgraphs: n %d (at most 46340), %d lists, %d per list (at most %d)", n,
                         n_lists, max_select, kMaxSelect);
    if (!n_selected || !n_refined || !refined || (n > 0 && (!matrix || !rank_sum || !order)))
        return api_error(FU_ERR_ARG, "fu_select_subgraphs: null argument");
    hipStream_t hs = (hipStream_t)s;
    if (n > 0) {
        hipLaunchKernelGGL(k_rank_sums, dim3((n + kSumCols - 1) / kSumCols), dim3(256), 0, hs, matrix, n, rank_sum);
        hipLaunchKernelGGL(k_rank_order, dim3((n + 63) / 64), dim3(1024), 0, hs, rank_sum, n, order);
    }
    const SelArgs a{matrix, order, n, max_select, min_score, n_selected, n_refined, refined};
    hipLaunchKernelGGL(k_select, dim3(n_lists), dim3(kSelLanes), 0, hs, a);
    const int longest = std::min(max_select, n);
    if (longest > 2) {  // no list of fewer is refined
        const int fours = (longest + 2) / 4;
        if ((long long)fours * n_lists <= kRefineGroups)
            hipLaunchKernelGGL(k_refine<false>, dim3(fours, n_lists), dim3(256), 0, hs, a);
        else
            hipLaunchKernelGGL(k_refine<true>, dim3(std::min(fours, std::max(4, kStagedGroups / n_lists)), n_lists), dim3(256), 0,
                               hs, a);
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return api_error(FU_ERR_HIP, "fu_select_subgraphs: %s", hipGetErrorString(e));
    return FU_OK;
}

// Tracker::Relocalise with useGraphMatching on (Tracking.cc:432-453) through GenerateGraph's
// PoseEstimate calls (:469-629): the match list keeps both nearest map keys of a query that
// fails the ratio test; pairs whose map key is not valid are dropped; their consistency
// matrix (BuildAdjacencyMatrix) and sub-graph selection run on the device; then PoseEstimate
// on the pairs of the first list of three or more selected pairs, once per kept list up to
// five (the reference's cv::sortIdx over its one-column list of counts leaves every index at
// 0, so each call takes that first list), when it holds four or more refined pairs.  Call c
// draws its samples from seed + c.  frame_pos (nq x 3) and frame_normal (nq x 4): host
// floats, the lifted keypoints.
extern "C" fu_status fu_relocalise_graph_candidates(fu_keymap* km, const float* frame_desc, const float* frame_pos,
                                                    const float* frame_normal, int32_t nq, int32_t iterations,
                                                    uint64_t seed, double poses[5 * 16], int32_t* n_poses,
                                                    int32_t* n_pairs, fu_stream s) {
    if (!km || !poses || !n_poses || nq < 0 || iterations < 0 ||
        (nq > 0 && (!frame_desc || !frame_pos || !frame_normal)))
        return api_error(FU_ERR_ARG, "fu_relocalise_graph_candidates: bad argument");
    constexpr int kLists = 10, kSelect = 400, kPoseLists = 5;  // Tracking.h:129-132
    constexpr float kMinScore = 0.1f;
    *n_poses = 0;
    if (n_pairs) *n_pairs = 0;
    const char* who = "fu_relocalise_graph_candidates";
    hipStream_t hs = (hipStream_t)s;
    uint32_t nk = 0;
    fu_status st = keymap_count(km, nk, hs);
    if (st) return st;
    if (nk == 0 || nq == 0) return FU_OK;  // no map keys (Tracking.cc:417-418)
    KeyScratch scratch(km, hs);
    const int dev = keymap_device(km);
    Block keys(hs), work(hs), graph(hs);
    const size_t nm = 2 * (size_t)nq;
    const size_t fpos = work.part(sizeof(float) * 3 * nq), fnrm = work.part(sizeof(float) * 4 * nq),
                 idx = work.part(sizeof(int32_t) * nm), dist = work.part(sizeof(float) * nm),
                 fk = work.part(sizeof(SurfHead) * nm), mk = work.part(sizeof(SurfHead) * nm),
                 dd = work.part(sizeof(float) * nm), cnt = work.part(sizeof(int) * 2);
    if (!work.allocate()) return api_error(FU_ERR_NOMEM, "%s: %d keypoints", who, nq);
    PairArgs pa{};
    if ((st = collect_and_match(km, scratch, frame_desc, nq, nk, keys, work.at<int32_t>(idx), work.at<float>(dist), pa, hs, who)))
        return st;
    hipError_t e = hipMemcpyAsync(work.at<float>(fpos), frame_pos, sizeof(float) * 3 * nq, hipMemcpyHostToDevice, hs);
    if (e == hipSuccess)
        e = hipMemcpyAsync(work.at<float>(fnrm), frame_normal, sizeof(float) * 4 * nq, hipMemcpyHostToDevice, hs);
    SurfHead *dfk = work.at<SurfHead>(fk), *dmk = work.at<SurfHead>(mk);
    hipLaunchKernelGGL(k_graph_pairs, dim3(1), dim3(1024), 0, hs, pa, work.at<float>(fpos), work.at<float>(fnrm), dfk, dmk,
                       work.at<float>(dd), work.at<int>(cnt));
    if (e == hipSuccess) e = hipGetLastError();
    int counted[2] = {0, 0};
    // also after a failure: nothing queued may still read the caller's memory
    const hipError_t er = mail_read(dev, counted, work.at<int>(cnt), sizeof(counted), hs);
    if (er == hipSuccess) scratch.done();
    if (e == hipSuccess) e = er;
    if (e != hipSuccess) return api_error(FU_ERR_HIP, "%s: %s", who, hipGetErrorString(e));
    if (n_pairs) *n_pairs = counted[0];
    const int n = counted[1];
    if (counted[0] < 3 || n == 0) return FU_OK;  // rank.cols == 0 (:523-524)
    if (n > 46340) return api_error(FU_ERR_ARG, "%s: %d pairs (at most 46340)", who, n);
    // counts of the lists, verdicts, points: read back together
    const int draws = std::min(iterations, kFirstDraws);
    constexpr size_t kCountInts = 2 * kLists;
    const size_t head_ints = kCountInts + (size_t)kPoseLists * draws;
    const size_t mat = graph.part(sizeof(float) * (size_t)n * n), rank = graph.part(sizeof(float) * n),
                 order = graph.part(sizeof(int32_t) * n),
                 sel = graph.part(sizeof(int32_t) * (kCountInts + (size_t)kLists * kSelect)),
                 head = graph.part(sizeof(int) * head_ints), pts = graph.part(sizeof(float) * 6 * kSelect);
    if (!graph.allocate()) return api_error(FU_ERR_NOMEM, "%s: %d pairs", who, n);
    int32_t* nsel = graph.at<int32_t>(sel);
    int* dhead = graph.at<int>(head);
    float* dpts = graph.at<float>(pts);
    if ((st = build_adjacency(dfk, dmk, 1, work.at<float>(dd), n, graph.at<float>(mat), hs))) return st;
    if ((st = fu_select_subgraphs(graph.at<float>(mat), n, kLists, kSelect, kMinScore, graph.at<float>(rank),
                                  graph.at<int32_t>(order), nsel, nsel + kLists, nsel + 2 * kLists, s)))
        return st;
    const ListPoints points{nsel, nsel + kLists, nsel + 2 * kLists, kLists, kSelect, dfk, dmk};
    hipLaunchKernelGGL(k_list_points, dim3(1), dim3(1024), 0, hs, points, dhead, dpts);
    if (draws > 0)
        hipLaunchKernelGGL(k_hypotheses<ListPoints>, dim3(draws, kPoseLists), dim3(64), 0, hs, points, seed, 0ll, draws,
                           dhead + kCountInts);
    e = hipGetLastError();
    std::vector<int> hhead(head_ints);
    std::vector<float> hpts(6 * kSelect);
    static_assert((kCountInts + kPoseLists * kFirstDraws + 6 * kSelect) * 4 <= kMailBytes, "one mail");
    const hipError_t er2 = mail_read(dev, hhead.data(), dhead, sizeof(int) * head_ints, hpts.data(), dpts,
                                     sizeof(float) * hpts.size(), hs);
    if (e == hipSuccess) e = er2;
    if (e != hipSuccess) return api_error(FU_ERR_HIP, "%s: %s", who, hipGetErrorString(e));
    const int* n_selected = hhead.data();
    const int* n_refined = hhead.data() + kLists;
    int kept = 0, first = -1;
    for (int i = 0; i < kLists; ++i)
        if (n_selected[i] >= 3) {
            if (first < 0) first = i;
            ++kept;
        }
    if (kept == 0) return FU_OK;  // "not enough points" (:591-594)
    const int M = std::min(kept, kPoseLists);
    const int R = n_refined[first];
    if (R <= 3) return FU_OK;  // every call skipped (:601-602)
    std::vector<double> src(3 * (size_t)R), ref(3 * (size_t)R);
    for (int k = 0; k < R; ++k)
        for (int c = 0; c < 3; ++c) {
            src[3 * k + c] = (double)hpts[6 * k + c];
            ref[3 * k + c] = (double)hpts[6 * k + 3 + c];
        }
    for (int c = 0; c < M; ++c) {
        const int* v = hhead.data() + kCountInts + (size_t)c * draws;
        Counts<ListPoints> counts{points, seed + (uint64_t)c, dev, hs, std::vector<int>(v, v + draws)};
        double T[16];
        int32_t good = 0;
        if ((st = pose_estimate(HostPoints{src.data(), ref.data()}, R, iterations, seed + (uint64_t)c, counts, T, nullptr,
                                &good)))
            return st;
        if (good) rigid_inverse(T, poses + 16 * (*n_poses)++);
    }
    return FU_OK;
}
