// Point-to-plane ICP: per-pixel association and Jacobian rows, compensated FP32
// reduction of the 29 sums, and (optionally) the FP64 solve and pose update on the device.
//
// Reference: Tracking/Reduction.cu ICPReduce::searchPoint (:227-257), getRow (:259-286),
// operator() (:288-312), Reduce<float,29> (:49-64), CreateMatrix<6,7> (:6-16), ICPStep
// (:319-375); Tracking/Tracking.cc Tracker::ComputeSE3 (:296-409).
//
// Each lane adds the products of its kIcpLanePixels pixels; a wave reduces its 29 sums with one
// reduce-scatter butterfly (wave_reduce_scatter32) and the waves are added through LDS into
// one partial row per work-group (frames with more pixel chunks than work-groups sum their
// chunks per lane with Neumaier-compensated FP32 adds first).
// The work-group whose row arrives last sums the rows with the same compensated tree and
// (mode 1) unpacks A (6x6) and b (6) in FP64, solves by Gauss-Jordan, takes the SE(3) exponential
// and composes the pose on its first wave: the only FP64 steps of the pipeline.
//
// With the photometric term (ComputeSE3 icpOnly = false) every iteration is two launches:
// the RGB residual pass (RGBReduction::ComputeResidual, Reduction.cu:469-483: one residual
// record per pixel and the integer sums of each work-group) and one pass that computes both
// the ICP rows of the pixels and the weighted RGB rows of the list in work-groups of their own (the
// latter first add the integer sums up to sigma themselves); the last to end blends
// A_rgb * 1e-4f + A_icp in FP64 before the solve.
#include "fu_device.h"
#include "fu_kernels.h"
#include "fu_track.h"
#include "fu_batch.h"

namespace fu {

struct Kahan {
    float s, c;
    __device__ void add(float v) {
        const float t = s + v;
        if (fabsf(s) >= fabsf(v))
            c += (s - t) + v;
        else
            c += (v - t) + s;
        s = t;
    }
    __device__ float val() const { return s + c; }
};

// ------------------------------------------------------------------ reduction kernel
// The poses of an iteration, read through the constant address space: the state changes only
// after every work-group has read them, so they are scalar loads even where the compiler sees
// later stores to the state (as vector loads they took up to 39 registers per lane).
#if defined(__HIP_DEVICE_COMPILE__)
#define FU_CPTR(T) const __attribute__((address_space(4))) T*
#else
#define FU_CPTR(T) const T*
#endif
__device__ __forceinline__ m3 load_m3(FU_CPTR(float) r) {
    return m3{mk3(r[0], r[1], r[2]), mk3(r[3], r[4], r[5]), mk3(r[6], r[7], r[8])};
}

// smallest float s with sqrtf(s) >= 0.6f, largest d with sqrtf(d) <= 0.1f, largest e with
// (double)sqrtf(e) < 0.1 (found by bisection over the floats with the host's IEEE sqrtf;
// tests/test_oracle.py checks all three)
constexpr float kSine2 = 0x1.70a3d8p-2f;
constexpr float kDist2 = 0x1.47ae16p-7f;
constexpr float kRgbDist2 = 0x1.47ae12p-7f;
constexpr bool angle_thresh_ok() { return kSine2 > 0.35f && kSine2 < 0.37f && kDist2 > 0.0099f && kDist2 < 0.0101f; }

struct IcpPose {
    m3 Rc, Rl, Rli;
    f3 tc, tl;
};
__device__ __forceinline__ IcpPose icp_pose(const TrackState* st_) {
    const auto st = (FU_CPTR(TrackState))st_;
    IcpPose P;
    P.Rc = load_m3(st->Rcurr);
    P.Rl = load_m3(st->Rlast);
    P.Rli = load_m3(st->RlastInv);
    P.tc = mk3(st->tcurr[0], st->tcurr[1], st->tcurr[2]);
    P.tl = mk3(st->tlast[0], st->tlast[1], st->tlast[2]);
    return P;
}

// ICPReduce::searchPoint + getRow (Reduction.cu:227-286) of a lane's pixel in three steps, so that
// the loads of a lane's pixels are in flight together: its own vertex and normal, which wait for
// nothing (not even the pose); the association's projection, which gives the last frame's pixel;
// that pixel's vertex and normal, and the row.  The reference's tests and arithmetic, as selects
// instead of early returns (lanes that fail a test read pixel 0 and contribute zeros), so a wave
// runs one path; a wave without any valid vertex skips the rest.
// Many sessions are bound by the maps' bytes (64 a pixel and iteration, from HBM: a session's maps do
// not stay in the caches), so a frame's own vertices are made from its depth, 12 bytes less
// (32 served sessions of 640x480, a frame each: 3,531 -> 3,420 us).
struct IcpPixel {
    bool in, ok;      // the lane has a pixel; it has passed the tests so far
    int i;            // the pixel
    f3 v, n;          // current vertex and normal (camera)
    f3 vg, vp;        // the vertex in the world and in the last camera frame
    f3 vl, nl;        // the associated vertex and normal (last camera)
};
__device__ __forceinline__ void icp_load(const IcpArgs& a, int i, bool in, IcpPixel& p) {
    const int ic = in ? i : 0;
    p.in = in;
    p.i = ic;
    if (a.zcurr)  // uniform
        p.v.z = FU_G(const float, a.zcurr)[ic];
    else
        p.v = xyz(FU_G(const f4, a.vcurr)[ic]);
    p.n = xyz(FU_G(const f4, a.ncurr)[ic]);
}
// the projection and the gathers; false (uniform) when no lane of the wave has a valid vertex
__device__ __forceinline__ bool icp_associate(const IcpArgs& a, const IcpPose& P, IcpPixel& p) {
    const int cols = a.cols, rows = a.rows;
    if (a.zcurr) {
        const int y = (int)__umulhi((unsigned)p.i, a.row_magic), x = p.i - y * cols;
        p.v = xyz(vertex_of(p.v.z, x, y, a.invfx, a.invfy, a.cx, a.cy, a.cutoff));
    }
    p.ok = p.in && !(isnanf_(p.v.x) || (double)p.v.z < 1e-3);
    if (ballot(p.ok) == 0ull) return false;
    p.vg = add(mv(P.Rc, p.v), P.tc);
    p.vp = mv(P.Rli, sub(p.vg, P.tl));
    // Reduction.cu:237-239: `float invz = 1.0 / z`, float products and sum, + 0.5 in double,
    // truncation.  The double quotient rounded to float is the float quotient 1.0f / z (double
    // rounding of a quotient of floats through a format of >= 2*24+2 bits is innocuous).  A lane
    // without a valid vertex divides by 1 (its result is discarded), so only a valid vertex
    // with |z| outside [2^-60, 2^30] takes the general division.
    const float zp = p.ok ? p.vp.z : 1.0f;
    const float azp = fabsf(zp);
    const float invz = (azp >= 0x1p-60f && azp <= 0x1p30f) ? fu_div_refined(1.0f, zp, fu_rcp_refined(zp)) : 1.0f / zp;
    const int u = d2i((double)(p.vp.x * invz * a.fx + a.cx) + 0.5);
    const int vv = d2i((double)(p.vp.y * invz * a.fy + a.cy) + 0.5);
    p.ok = p.ok && !(u < 0 || vv < 0 || u >= cols || vv >= rows);
    const int j = p.ok ? vv * cols + u : 0;
    p.vl = xyz(FU_G(const f4, a.vlast)[j]);
    p.nl = xyz(FU_G(const f4, a.nlast)[j]);
    return true;
}
// the row [-n, n x v_l, -n.(v_c - v_l)] (last camera frame) of a pixel with a correspondence, else
// zeros; returns whether there is one
__device__ __forceinline__ bool icp_row(const IcpPose& P, const IcpPixel& p, float (&row)[7]) {
    const f3 vlast_g = add(mv(P.Rl, p.vl), P.tl);
    const f3 ncurr_g = mv(P.Rc, p.n);
    const f3 nlast_g = mv(P.Rl, p.nl);
    const f3 dv = sub(vlast_g, p.vg);
    const f3 cr2 = cross(ncurr_g, nlast_g);
    const float dist2 = dot(dv, dv), sine2 = dot(cr2, cr2);
    const bool ok = p.ok && sine2 < kSine2 && dist2 <= kDist2 && !isnanf_(p.n.x) && !isnanf_(p.nl.x);
    const f3 nl = mv(P.Rli, nlast_g);
    const f3 vla = mv(P.Rli, sub(vlast_g, P.tl));
    const f3 mn = neg(nl);
    const f3 cr = cross(nl, vla);
    // a lane without a correspondence contributes +0 to every sum, as the products of a zero row
    row[0] = ok ? mn.x : 0.f;
    row[1] = ok ? mn.y : 0.f;
    row[2] = ok ? mn.z : 0.f;
    row[3] = ok ? cr.x : 0.f;
    row[4] = ok ? cr.y : 0.f;
    row[5] = ok ? cr.z : 0.f;
    row[6] = ok ? dot(mn, sub(p.vp, vla)) : 0.f;
    return ok;
}
// the 29 products of the row and the count 1 into v[0 .. 28] (kAdd: added to v instead)
template <bool kAdd>
__device__ __forceinline__ void icp_row_values(const IcpPose& P, const IcpPixel& p, bool any, float (&v)[32]) {
    if (!any) {
        if constexpr (!kAdd) {
#pragma unroll
            for (int k = 0; k < 29; ++k) v[k] = 0.f;
        }
        return;
    }
    float row[7];
    const bool ok = icp_row(P, p, row);
    int k = 0;
#pragma unroll
    for (int r = 0; r < 7; ++r)
#pragma unroll
        for (int c = r; c < 7; ++c) {
            if constexpr (kAdd)
                v[k] += row[r] * row[c];
            else
                v[k] = row[r] * row[c];
            ++k;
        }
    if constexpr (kAdd)
        v[28] += ok ? 1.0f : 0.f;
    else
        v[28] = ok ? 1.0f : 0.f;
}
// both pixels of a lane, loaded: their products added in pixel order
__device__ __forceinline__ void icp_pixels(const IcpArgs& a, const IcpPose& P, IcpPixel& p, IcpPixel& q, float (&v)[32]) {
    const bool any_p = icp_associate(a, P, p), any_q = icp_associate(a, P, q);
    icp_row_values<false>(P, p, any_p, v);
    icp_row_values<true>(P, q, any_q, v);
}

__device__ __forceinline__ void store_agent(float* p, float v);

// sums of a work-group of NW waves: each wave's totals into LDS, then one 29-float row
// (v[29..31] must be 0).  Value j of a wave's totals is held by lanes 2j and 2j+1 after the
// reduce-scatter; the waves are added as a pairwise tree.
template <int NW>
__device__ __forceinline__ void block_rows29(float (&v)[32], float (&wsum)[NW][32], float* out) {
    const float t = wave_reduce_scatter32(v);
    const int lane = lane_id();
    if (!(lane & 1)) wsum[threadIdx.x >> 6][lane >> 1] = t;
    __syncthreads();
    if (threadIdx.x < 29) {
        const int j = threadIdx.x;
        float w[NW];
#pragma unroll
        for (int k = 0; k < NW; ++k) w[k] = wsum[k][j];
#pragma unroll
        for (int h = NW / 2; h >= 1; h /= 2)
#pragma unroll
            for (int k = 0; k < h; ++k) w[k] = w[2 * k] + w[2 * k + 1];
        store_agent(out + j, w[0]);
    }
}

// ------------------------------------------------------------------ the last work-group's stage
// An iteration is one launch: the work-group whose partial row arrives last sums the rows and
// updates the pose.  Nobody waits: every work-group counts itself in st->arrived after its row
// is written, and the one that reads groups - 1 there goes on.  The rows travel as agent-scope
// relaxed atomic accesses, which are written through to and read from the memory that all XCDs
// share, so a work-group needs only its own stores complete (s_waitcnt) before it is counted,
// not a release, whose write-back of the XCD's whole L2 made such a ticket slower than a second
// launch.  As a second launch of one work-group this stage took 6.4 us an iteration (single
// 640x480 session) and 15 us (lanes of eleven sessions), most of it the launch, the rows' trip
// and one lane's serial FP64 chain.
__device__ __forceinline__ void store_agent(float* p, float v) {
    __hip_atomic_store(FU_G(float, p), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float load_agent(const float* p) {
    return __hip_atomic_load(FU_G(const float, p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// called by every lane once the first wave's lanes have stored the work-group's row: whether
// this is the last of `groups` work-groups (the same in every lane)
__device__ __forceinline__ bool last_to_arrive(TrackState* st, int groups) {
    __shared__ int last;
    if (threadIdx.x < 64) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the row is in place
        if (threadIdx.x == 0) {
            const unsigned before = __hip_atomic_fetch_add(FU_G(unsigned, &st->arrived), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            last = before == (unsigned)groups - 1u;
            if (last) __hip_atomic_store(FU_G(unsigned, &st->arrived), 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    __syncthreads();
    return last != 0;
}

// Sums of the partial rows of `chunks` pixel chunks into total[0..28] (LDS), by the NW waves of a
// work-group.  NW = 16: a row per chunk; NW = 4 (at most 128 chunks): four rows per chunk, one of
// each quarter.  The order is that of 256 lanes which each add the rows of chunks t, t + 256, ...
// (compensated), four waves reduced as wave_reduce_scatter32 does and added pairwise: lane (j, q)
// of a wave holds value j of chunks 64 w + q + 8 k, k = 0..7, so the loads of 64 rows are in
// flight together and a row is read in 32-byte pieces.
template <int NW>
__device__ __forceinline__ void sum_rows32(const float* parts, int chunks, float* total) {
    constexpr int kRows = NW == 16 ? 1 : 4;  // rows per chunk
    __shared__ float wsum[4][32];
    const int lane = lane_id(), wave = threadIdx.x >> 6;
    const int q = lane >> 3, j = ((wave & 3) << 3) | (lane & 7);
    // chunks past the end read chunk 0 and count as +0, which changes no sum (columns 29-31 of a
    // row are never written and never used)
    auto fetch = [&](int c0, float (&x)[8]) {
        float y[8][kRows];
#pragma unroll
        for (int u = 0; u < 8; ++u)
#pragma unroll
            for (int r = 0; r < kRows; ++r) {
                const int c = c0 + q + 8 * u;
                y[u][r] = load_agent(parts + ((c < chunks ? c : 0) * kRows + r) * 32 + j);
            }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            if constexpr (kRows == 1)
                x[u] = y[u][0];
            else
                x[u] = (y[u][0] + y[u][1]) + (y[u][2] + y[u][3]);
            x[u] = c0 + q + 8 * u < chunks ? x[u] : 0.f;
        }
    };
    // the tree of wave_reduce_scatter32 over 64 rows: partners 32, 16 and 8 apart, then row 7 - q
    // of each eight, then 2 and 1 apart
    auto tree = [&](const float (&x)[8]) {
        float t = ((x[0] + x[4]) + (x[2] + x[6])) + ((x[1] + x[5]) + (x[3] + x[7]));
        t += __shfl_xor(t, 56);
        t += __shfl_xor(t, 16);
        return t + __shfl_xor(t, 8);
    };
    if constexpr (NW == 16) {
        const int w = wave >> 2;
        float x[8] = {}, c[8] = {};
        if (w * 64 < chunks) fetch(w * 64, x);  // uniform
        for (int c0 = 256 + w * 64; c0 < chunks; c0 += 256) {
            float y[8];
            fetch(c0, y);
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                Kahan k{x[u], c[u]};
                k.add(y[u]);
                x[u] = k.s;
                c[u] = k.c;
            }
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) x[u] = x[u] + c[u];
        const float t = tree(x);
        if (q == 0) wsum[w][j] = t;
    } else {
#pragma unroll 1
        for (int w = 0; w < 4; ++w) {
            float t = 0.f;
            if (w * 64 < chunks) {
                float x[8];
                fetch(w * 64, x);
                t = tree(x);
            }
            if (q == 0) wsum[w][j] = t;
        }
    }
    __syncthreads();
    if (threadIdx.x < 29) {
        const int i = threadIdx.x;
        total[i] = (wsum[0][i] + wsum[1][i]) + (wsum[2][i] + wsum[3][i]);
    }
}

// LDS written by some lanes of a wave is read by others of the same wave: its LDS operations
// run in order, so only the compiler has to keep them so
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
__device__ __forceinline__ double readlane_f64(double v, int lane) {
    return __longlong_as_double((long long)readlane64((unsigned long long)__double_as_longlong(v), lane));
}
// 1 / s for normal s: v_rcp_f64 is good to about 2^-24, and one third-order step (the error
// cubed, 2^-72) leaves the rounding of the last sum, about one ulp
__device__ __forceinline__ double rcp_f64(double s) {
    const double y = __builtin_amdgcn_rcp(s);
    const double e = fma(-s, y, 1.0);
    return fma(y, fma(e, e, e), y);
}

// What the pose update of an iteration reads from the tracking state, one pose element per lane
// (element lane & 15), loaded ahead of the row sums so that its latency overlaps theirs.
struct UpdateIn {
    double last, delta, init;
    int iters;
};
__device__ __forceinline__ UpdateIn load_update(const TrackState* st_) {
    const auto st = FU_G(const TrackState, st_);
    const int e = threadIdx.x & 15;
    return UpdateIn{st->last_pose[e], st->delta[e], st->init_pose[e], st->iters_done};
}

// icp_update (fu_track.h) by the 64 lanes of one wave, from the totals in LDS: lane 8 i + m
// holds element (i, m) of the augmented matrix [A b], so an elimination step is one update for
// all its elements, and the poses are products of one element per lane.  The elimination runs
// over the rows above the pivot too, which leaves the solution in place of b (a back
// substitution's six dependent steps took 0.65 us); its pivots are the squares of Cholesky's
// diagonal, so the test for a positive definite matrix is the same.  The solution and the
// exponential's coefficients differ from icp_update's by a few ulp of FP64.  One lane's serial
// chain took 3.5 us and over 150 registers, which would have cost the reduction its occupancy.
template <bool kRgb>
__device__ __forceinline__ void icp_update_wave(const IcpArgs& a, const float* total, const UpdateIn& in, double* sm) {
    const auto st = FU_G(TrackState, a.st);
    const int lane = lane_id();
    const int e = lane & 15, i4 = e >> 2, j4 = e & 3;  // pose element of the lane
    // 4x4 matrices in LDS
    double* const X = sm;
    double* const Y = sm + 16;
    double* const last = sm + 32;
    double* const init = sm + 48;
    last[e] = in.last;
    init[e] = in.init;
    Y[e] = in.delta;
    const int i = lane >> 3, m = lane & 7;
    const bool el = i < 6 && m < 7;
    const int lo = min(i, m), hi = max(i, m);
    const int idx = el ? lo * 7 - lo * (lo - 1) / 2 + hi - lo : 0;  // element (lo, hi) of the 29 sums
    double v = (double)total[idx];
    bool good = true;
    if constexpr (kRgb) {
        const float rerr = sqrtf(total[32 + 27]) / total[32 + 28];
        const int rcnt = f2i(total[32 + 28]);
        good = !(isnanf_(rerr) || rcnt < a.min_count);
        v = (double)total[32 + idx] * (double)1e-4f + v;
        if (lane == 0) {
            st->rgb_error = rerr;
            st->rgb_count = rcnt;
        }
    }
    if (el) {
        if (m < 6)
            st->A[i * 6 + m] = v;
        else
            st->b[i] = v;
    }
    const float err = sqrtf(total[27]) / total[28];
    const int cnt = f2i(total[28]);
    good = good && !(isnanf_(err) || cnt < a.min_count);
    if (lane == 0) {
        st->residual[0] = total[27];
        st->residual[1] = total[28];
        st->icp_error = err;
        st->count = cnt;
        st->iters_done = in.iters + 1;
    }
#pragma unroll 1
    for (int j = 0; j < 6; ++j) {
        const double s = readlane_f64(v, j * 9);
        good = good && s > 0.0;
        const double c = v * rcp_f64(s > 0.0 ? s : 1.0);  // row j: the pivot row divided by the pivot
        const double l = __shfl(v, i * 8 + j), r = __shfl(c, j * 8 + m);
        v = i == j ? c : v - l * r;
    }
    double nx = in.last;
    int status = TS_FAILED;
    if (good) {  // uniform
        status = TS_RUNNING;
        if (i < 6 && m == 6) st->x[i] = v;
        // SE(3) exponential (se3_exp) of x / 2^n, squared n times: the coefficients sin(th)/th,
        // (1 - cos(th))/th^2 and (th - sin(th))/th^3 come from their series, whose six terms end
        // below 2^-60 for th up to an eighth of a radian, where an iteration's step lies (n = 0;
        // a squaring doubles the relative error, a few ulp at steps of a radian)
        double wx = readlane_f64(v, 3 * 8 + 6), wy = readlane_f64(v, 4 * 8 + 6), wz = readlane_f64(v, 5 * 8 + 6);
        double th2 = wx * wx + wy * wy + wz * wz;
        int n = 0;
        double scale = 1.0;
        while (th2 > 0x1p-6 && n < 60) {
            th2 *= 0.25;
            scale *= 0.5;
            ++n;
        }
        constexpr double f2 = 1.0 / 2, f3 = f2 / 3, f4 = f3 / 4, f5 = f4 / 5, f6 = f5 / 6, f7 = f6 / 7, f8 = f7 / 8,
                         f9 = f8 / 9, f10 = f9 / 10, f11 = f10 / 11, f12 = f11 / 12, f13 = f12 / 13;
        const double x2 = -th2;
        const double A = fma(fma(fma(fma(fma(f11, x2, f9), x2, f7), x2, f5), x2, f3), x2, 1.0);
        const double B = fma(fma(fma(fma(fma(f12, x2, f10), x2, f8), x2, f6), x2, f4), x2, f2);
        const double C = fma(fma(fma(fma(fma(f13, x2, f11), x2, f9), x2, f7), x2, f5), x2, f3);
        {
            // element (i4, j4) of R = I + A W + B W^2 and V = I + B W + C W^2, W^2 = w w^T - th^2 I
            const double wi = (i4 == 0 ? wx : i4 == 1 ? wy : wz) * scale, wj = (j4 == 0 ? wx : j4 == 1 ? wy : wz) * scale;
            const int k = 3 - i4 - j4;  // the third axis
            const double wk = (k == 0 ? wx : k == 1 ? wy : wz) * scale;
            const bool diag = i4 == j4;
            const double W = diag ? 0.0 : (j4 - i4 == 1 || j4 - i4 == -2) ? -wk : wk;
            const double W2 = diag ? wi * wj - th2 : wi * wj;
            const double I = diag ? 1.0 : 0.0;
            const double R = I + A * W + B * W2;
            const double u = __shfl(v, (j4 < 3 ? j4 : 0) * 8 + 6) * scale;
            const double vu = (I + B * W + C * W2) * u;  // lanes j4 < 3: a term of row i4 of V u
            const double t = __shfl(vu, e & 12) + __shfl(vu, (e & 12) | 1) + __shfl(vu, (e & 12) | 2);
            X[e] = i4 == 3 ? (j4 == 3 ? 1.0 : 0.0) : j4 < 3 ? R : t;
        }
        auto product = [&](const double* P, const double* Q) {
            wave_sync();
            double s = 0;
#pragma unroll
            for (int k = 0; k < 4; ++k) s += P[i4 * 4 + k] * Q[k * 4 + j4];
            wave_sync();
            return s;
        };
        // element of rigid_inv(M)
        auto inverse = [&](const double* M) {
            const double s = -(M[i4] * M[3] + M[4 + i4] * M[7] + M[8 + i4] * M[11]);
            return i4 == 3 ? (j4 == 3 ? 1.0 : 0.0) : j4 < 3 ? M[j4 * 4 + i4] : s;
        };
#pragma unroll 1
        for (; n > 0; --n) X[e] = product(X, X);
        const double d = product(X, Y);  // the accumulated step
        if (lane < 16) st->delta[e] = d;
        X[e] = d;
        wave_sync();
        Y[e] = inverse(X);
        nx = product(last, Y);
        if (a.final_iter) {
            Y[e] = nx;
            X[e] = inverse(init);
            const double q = product(X, Y);
            X[e] = q;
            wave_sync();
            const double tn = sqrt(X[3] * X[3] + X[7] * X[7] + X[11] * X[11]);
            const bool ok = err < a.thresh && sin_euler_norm(X) <= 0.1 && tn <= 0.1;
            status = ok ? TS_OK : TS_REJECTED;
            if (!ok) nx = in.last;
        }
    }
    if (lane < 16) {
        st->next_pose[e] = nx;
        if (i4 < 3) {
            if (j4 < 3) {
                st->Rcurr[i4 * 3 + j4] = (float)nx;
                st->RcurrInv[j4 * 3 + i4] = (float)nx;
            } else {
                st->tcurr[i4] = (float)nx;
            }
        }
    }
    if (lane == 0 && status != TS_RUNNING) st->status = status;
}

// the last stage of an ICP-only iteration, by a work-group of NW waves
template <int NW>
__device__ __forceinline__ void icp_last(const IcpArgs& a, int chunks, float* out = nullptr) {
    __shared__ float total[32];
    if (out) {
        sum_rows32<NW>(a.partials, chunks, total);
        if (threadIdx.x < 29) out[threadIdx.x] = total[threadIdx.x];  // the lane's own total
        return;
    }
    __shared__ double sm[64];
    const UpdateIn in = load_update(a.st);
    sum_rows32<NW>(a.partials, chunks, total);
    if (threadIdx.x >= 64) return;
    wave_sync();
    if (threadIdx.x < 29) a.st->sums[threadIdx.x] = total[threadIdx.x];
    if (a.mode == 1) icp_update_wave<false>(a, total, in, sm);
}

// How an ICP-only iteration is split over work-groups.  Every form computes the same sums in the
// same order, so a session's results do not depend on which one a launch takes.
//   kLoop     1024 lanes, chunks beyond the grid looped over with compensated per-lane sums
//             (frames of more than kIcpMaxBlocks chunks)
//   kChunk    1024 lanes a chunk of kIcpPixels pixels
//   kQuarter  256 lanes, a quarter of a chunk and a partial row each
// The last work-group of a session sums its rows and updates the pose, except in a launch of more
// than kLastGroups chunks, where a second launch does (kTicket).
enum IcpForm : int { kLoop, kChunk, kQuarter };

// `step`: a single reduction (ICPStep) at the pose given there, whose 29 sums go to step->out; the
// tracking state only counts the rows.
struct IcpStep {
    IcpPose pose;
    float* out;  // pinned host memory
};
template <int FORM, bool kTicket>
__device__ __forceinline__ void icp_body(WG g, const IcpArgs& a, const IcpStep* step = nullptr) {
    constexpr int NT = FORM == kQuarter ? 256 : kIcpThreads, NW = NT / 64;
    static_assert(kIcpLanePixels == 2, "a lane's pixels are loaded as a pair");
    const int N = a.cols * a.rows;
    // a chunk is kIcpPixels = kIcpLanePixels * kIcpThreads pixels: lane t of its kIcpThreads
    // adds the products of pixels t and t + kIcpThreads of the chunk, in that order, before the
    // wave reduction
    const int i0 = FORM == kQuarter ? (g.x >> 2) * kIcpPixels + (g.x & 3) * NT + threadIdx.x
                                    : g.x * kIcpPixels + threadIdx.x;
    IcpPixel p, q;
    icp_load(a, i0, i0 < N, p);
    icp_load(a, i0 + kIcpThreads, i0 + kIcpThreads < N, q);
    const auto st = FU_G(const TrackState, a.st);
    if (a.mode != 0 && st->status != TS_RUNNING) return;  // uniform: a failed frame skips
    const IcpPose P = step ? step->pose : icp_pose(a.st);
    __shared__ float wsum[NW][32];
    float v[32];
    v[29] = v[30] = v[31] = 0.f;
    icp_pixels(a, P, p, q, v);
    if constexpr (FORM == kLoop) {
        // more chunks than work-groups: compensated per-lane sums over the chunks, seeded
        // exactly by the first (so every form agrees when every group has one chunk)
        Kahan acc[29];
#pragma unroll
        for (int j = 0; j < 29; ++j) acc[j] = Kahan{v[j], 0.f};
        const int stride = g.nx * kIcpPixels;
        for (int c = g.x * kIcpPixels + stride; c < N; c += stride) {
            // the rows first, then each product pair into its sum: the sums leave no registers for
            // the products as well
            const int i = c + threadIdx.x;
            float rp[7] = {}, rq[7] = {};
            bool okp = false, okq = false;
            icp_load(a, i, i < N, p);
            if (icp_associate(a, P, p)) okp = icp_row(P, p, rp);
            icp_load(a, i + kIcpThreads, i + kIcpThreads < N, q);
            if (icp_associate(a, P, q)) okq = icp_row(P, q, rq);
            int k = 0;
#pragma unroll
            for (int r = 0; r < 7; ++r)
#pragma unroll
                for (int m = r; m < 7; ++m) {
                    acc[k].add(rp[r] * rp[m] + rq[r] * rq[m]);
                    ++k;
                }
            acc[28].add((okp ? 1.0f : 0.f) + (okq ? 1.0f : 0.f));
        }
#pragma unroll
        for (int j = 0; j < 29; ++j) v[j] = acc[j].val();
    }
    block_rows29(v, wsum, a.partials + g.x * 32);
    if constexpr (kTicket) {
        if (last_to_arrive(a.st, g.nx)) icp_last<NW>(a, FORM == kQuarter ? g.nx >> 2 : g.nx, step ? step->out : nullptr);
    }
}
template <int FORM>
__global__ __launch_bounds__(FORM == kQuarter ? 256 : kIcpThreads) void k_icp(IcpArgs a) {
    icp_body<FORM, true>(hw_wg(), a);
}
template <int FORM>
__global__ __launch_bounds__(FORM == kQuarter ? 256 : kIcpThreads) void k_icp_step(IcpArgs a, IcpStep step) {
    icp_body<FORM, true>(hw_wg(), a, &step);
}

// ------------------------------------------------------------------ photometric term
struct RgbPose {
    m3 Rc, Rci, Rl, Rli;
    f3 tc, tl;
};
__device__ __forceinline__ RgbPose rgb_pose(const TrackState* st_) {
    const auto st = (FU_CPTR(TrackState))st_;
    RgbPose P;
    P.Rc = load_m3(st->Rcurr);
    P.Rci = load_m3(st->RcurrInv);
    P.Rl = load_m3(st->Rlast);
    P.Rli = load_m3(st->RlastInv);
    P.tc = mk3(st->tcurr[0], st->tcurr[1], st->tcurr[2]);
    P.tl = mk3(st->tlast[0], st->tlast[1], st->tlast[2]);
    return P;
}

// The pose-independent part of RGBReduction::FindCorresp (Reduction.cu:420-433) for pixel
// (x, y): inside the 5-pixel margin, the 4x4 window [y-2, y+2) x [x-2, x+2) non-zero (the
// margin keeps it in the image, so the reference's clamps are inactive), a non-zero gradient
// (sqrtf(gx * gx + gy * gy) > 0: the integer sum is positive unless both are zero) and a valid
// vertex
__device__ __forceinline__ bool rgb_eligible(const IcpArgs& a, int x, int y) {
    const int cols = a.cols, rows = a.rows;
    if (!(x >= 5 && x < cols - 5 && y >= 5 && y < rows - 5)) return false;
    const auto inext = FU_G(const unsigned char, a.rgb.inext);
    bool valid = true;
#pragma unroll
    for (int u = -2; u < 2; ++u)
#pragma unroll
        for (int v = -2; v < 2; ++v) valid &= inext[(y + u) * cols + x + v] > 0;
    if (!valid) return false;
    const int i = y * cols + x;
    const int gx = FU_G(const short, a.rgb.dx)[i], gy = FU_G(const short, a.rgb.dy)[i];
    if (gx == 0 && gy == 0) return false;
    return !isnanf_(FU_G(const f4, a.vcurr)[i].x);
}

// the rest of FindCorresp (Reduction.cu:434-463) for an eligible pixel i: the last-frame
// pixel j and the intensity difference, or false
__device__ __forceinline__ bool rgb_corresp(const IcpArgs& a, const RgbPose& P, int i, int& j, int& diff) {
    const int cols = a.cols, rows = a.rows;
    const f4 vc = FU_G(const f4, a.vcurr)[i];
    const f3 vg = add(mv(P.Rc, xyz(vc)), P.tc);
    const f3 vl = mv(P.Rli, sub(vg, P.tl));
    // __float2int_rd(fx * x / z + cx + 0.5): float quotient and sum, 0.5 added in double,
    // the double rounded to float, then floor
    const int u = f2i(floorf((float)((double)(a.fx * vl.x / vl.z + a.cx) + 0.5)));
    const int v = f2i(floorf((float)((double)(a.fy * vl.y / vl.z + a.cy) + 0.5)));
    if (!(u >= 0 && v >= 0 && u < cols && v < rows)) return false;
    const int k = v * cols + u;
    const f4 la = FU_G(const f4, a.vlast)[k];
    const int lk = FU_G(const unsigned char, a.rgb.ilast)[k];
    // (double)norm4(...) < 0.1 on the squared norm: see kRgbDist2
    const f4 d4 = sub4(la, vc);
    if (!(!isnanf_(la.x) && dot4(d4, d4) <= kRgbDist2 && lk != 0)) return false;
    j = k;
    diff = (int)FU_G(const unsigned char, a.rgb.inext)[i] - lk;
    return true;
}

// RGBReduction::GetRow (Reduction.cu:485-520) of a valid residual: the last frame's vertex, the
// gradient and the intensity difference of its pixel
__device__ __forceinline__ void rgb_row(const IcpArgs& a, const RgbPose& P, const f4& la, int dx, int dy, int diff,
                                        float sigma, float (&row)[7]) {
    float w = sigma + (float)abs(diff);
    w = (double)w < 1e-3 ? 1.0f : 1.0f / w;
    if ((double)sigma < 1e-6) w = 1.0f;
    const f3 point = mv(P.Rci, sub(add(mv(P.Rl, xyz(la)), P.tl), P.tc));
    // (float)((double)s / 9.0) in the reference: for every short s this equals the correctly
    // rounded float quotient (s / 9 has a period-6 binary expansion, so rounding to double
    // first never lands on a float rounding boundary; checked for all 65536 values)
    const float gx = (float)dx / 9.0f;
    const float gy = (float)dy / 9.0f;
    const float invz = 1.0f / point.z;
    f3 left;
    left.x = gx * a.fx * invz;
    left.y = gy * a.fy * invz;
    left.z = -(left.x * point.x + left.y * point.y) * invz;
    const f3 c = cross(point, left);
    row[0] = w * left.x;
    row[1] = w * left.y;
    row[2] = w * left.z;
    row[3] = w * c.x;
    row[4] = w * c.y;
    row[5] = w * c.z;
    row[6] = -w * (float)diff;
}

// sum over the work-group of one int per lane (all lanes get it); `part` holds a slot per wave
__device__ __forceinline__ unsigned block_sum_u32(unsigned v, unsigned* part) {
    v = wave_sum_u32(v);
    if (lane_id() == 0) part[threadIdx.x >> 6] = v;
    __syncthreads();
    unsigned t = 0;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) t += part[w];
    return t;
}

// list building, pass 1: the eligibility of each pixel as one 64-bit word per wave (kept in
// the record buffer until pass 2) and the eligible pixels of each 1024-pixel work-group
__device__ __forceinline__ void rgb_count_body(WG g, const IcpArgs& a) {
    const int N = a.cols * a.rows;
    const int i = g.x * kIcpThreads + threadIdx.x;
    bool e = false;
    if (i < N) {
        const int y = i / a.cols;
        e = rgb_eligible(a, i - y * a.cols, y);
    }
    const unsigned long long m = ballot(e);
    __shared__ unsigned part[kIcpThreads / 64];
    if (lane_id() == 0) {
        part[threadIdx.x >> 6] = (unsigned)__popcll(m);
        FU_G(unsigned long long, a.rgb.rec)[g.x * (kIcpThreads / 64) + (threadIdx.x >> 6)] = m;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned t = 0;
        for (int w = 0; w < kIcpThreads / 64; ++w) t += part[w];
        FU_G(int, a.rgb.wgcnt)[g.x] = (int)t;
    }
}
// pass 2: each work-group writes its eligible pixels at the prefix of the counts before it
// (pixel order); the last work-group stores the total
__device__ __forceinline__ void rgb_scatter_body(WG g, const IcpArgs& a) {
    __shared__ unsigned part[kIcpThreads / 64];
    __shared__ unsigned wbase[kIcpThreads / 64];
    const auto wgcnt = FU_G(const int, a.rgb.wgcnt);
    unsigned before = 0;
    for (int t = threadIdx.x; t < g.x; t += blockDim.x) before += (unsigned)wgcnt[t];
    const unsigned base = block_sum_u32(before, part);
    const int wave = threadIdx.x >> 6;
    const unsigned long long m = FU_G(const unsigned long long, a.rgb.rec)[g.x * (kIcpThreads / 64) + wave];
    __syncthreads();  // part is reused
    if (lane_id() == 0) part[wave] = (unsigned)__popcll(m);
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned t = base;
        for (int w = 0; w < kIcpThreads / 64; ++w) {
            wbase[w] = t;
            t += part[w];
        }
        if (g.x == g.nx - 1) *FU_G(int, a.rgb.count) = (int)t;
    }
    __syncthreads();
    if ((m >> lane_id()) & 1ull) FU_G(int, a.rgb.list)[wbase[wave] + lane_rank(m)] = g.x * kIcpThreads + threadIdx.x;
}

// residual pass over the list: record (j << 9) | (diff + 256) or -1 per entry, and the
// work-group's {count, sum diff^2}; one entry per lane
__device__ __forceinline__ void rgb_resid_body(WG g, const IcpArgs& a) {
    const auto st = FU_G(const TrackState, a.st);
    if (a.mode != 0 && st->status != TS_RUNNING) return;  // uniform: a failed frame skips
    const int n = *FU_G(const int, a.rgb.count);
    const int k = g.x * kIcpThreads + threadIdx.x;
    int rec = -1, diff = 0;
    if (g.x * kIcpThreads < n) {  // uniform
        const RgbPose P = rgb_pose(a.st);
        if (k < n) {
            int j;
            if (rgb_corresp(a, P, FU_G(const int, a.rgb.list)[k], j, diff)) rec = (j << 9) | (diff + 256);
            FU_G(int, a.rgb.rec)[k] = rec;
        }
    }
    const bool ok = rec >= 0;
    const unsigned c = (unsigned)__popcll(ballot(ok));
    const unsigned q = wave_sum_u32(ok ? (unsigned)(diff * diff) : 0u);
    __shared__ unsigned part[kIcpThreads / 64][2];
    if (lane_id() == 0) {
        part[threadIdx.x >> 6][0] = c;
        part[threadIdx.x >> 6][1] = q;
    }
    __syncthreads();
    if (threadIdx.x < 2) {
        unsigned t = 0;
        for (int w = 0; w < kIcpThreads / 64; ++w) t += part[w][threadIdx.x];
        FU_G(int, a.rgb.corr)[g.x * 2 + threadIdx.x] = (int)t;
    }
}
__global__ __launch_bounds__(kIcpThreads) void k_rgb_resid(IcpArgs a) { rgb_resid_body(hw_wg(), a); }

// totals of the residual pass's {count, sum diff^2} over its `nparts` work-groups (32-bit,
// wrapping, as the reference's int sums), and sigma = sqrt(sum / count) (Reduction.cu:605)
__device__ __forceinline__ float rgb_sigma(const IcpArgs& a, int nparts, int& ci, int& qi) {
    __shared__ unsigned part[kIcpThreads / 64][2];
    const auto corr = FU_G(const int, a.rgb.corr);
    unsigned c = 0, q = 0;
    for (int t = threadIdx.x; t < nparts; t += blockDim.x) {
        c += (unsigned)corr[2 * t];
        q += (unsigned)corr[2 * t + 1];
    }
    c = wave_sum_u32(c);
    q = wave_sum_u32(q);
    if (lane_id() == 0) {
        part[threadIdx.x >> 6][0] = c;
        part[threadIdx.x >> 6][1] = q;
    }
    __syncthreads();
    unsigned tc = 0, tq = 0;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) {
        tc += part[w][0];
        tq += part[w][1];
    }
    ci = (int)tc;
    qi = (int)tq;
    return sqrtf((float)qi / (float)(ci == 0 ? 1 : ci));
}

// A lane's two list entries (n in the list) in two steps, so that their loads are in flight
// together: the residual record and pixel, then the associated vertex and the gradient.  The
// record of an entry outside the list is never read; lanes without a residual evaluate the row
// of pixel 0 and discard it.
struct RgbEntry {
    bool ok;
    int i, j, diff;
    f4 la;
    int gx, gy;
};
__device__ __forceinline__ void rgb_load(const IcpArgs& a, int k, int n, RgbEntry& e) {
    const int rec = k < n ? FU_G(const int, a.rgb.rec)[k] : -1;
    const int pix = k < n ? FU_G(const int, a.rgb.list)[k] : 0;
    e.ok = rec >= 0;
    e.i = e.ok ? pix : 0;
    e.j = e.ok ? rec >> 9 : 0;
    e.diff = e.ok ? (rec & 511) - 256 : 0;
}
__device__ __forceinline__ void rgb_gather(const IcpArgs& a, RgbEntry& e) {
    e.la = FU_G(const f4, a.vlast)[e.j];
    e.gx = FU_G(const short, a.rgb.dx)[e.i];
    e.gy = FU_G(const short, a.rgb.dy)[e.i];
}
// the 29 products of an entry's photometric row into v[0 .. 28] (kAdd: added), zeros for a lane
// without a residual
template <bool kAdd>
__device__ __forceinline__ void rgb_row_values(const IcpArgs& a, const RgbPose& Q, const RgbEntry& e, float sigma,
                                               float (&v)[32]) {
    if (ballot(e.ok) == 0ull) {
        if constexpr (!kAdd) {
#pragma unroll
            for (int k = 0; k < 29; ++k) v[k] = 0.f;
        }
        return;
    }
    float row[7];
    rgb_row(a, Q, e.la, e.gx, e.gy, e.diff, sigma, row);
#pragma unroll
    for (int k = 0; k < 7; ++k) row[k] = e.ok ? row[k] : 0.f;
    int k = 0;
#pragma unroll
    for (int r = 0; r < 7; ++r)
#pragma unroll
        for (int c = r; c < 7; ++c) {
            if constexpr (kAdd)
                v[k] += row[r] * row[c];
            else
                v[k] = row[r] * row[c];
            ++k;
        }
    if constexpr (kAdd)
        v[28] += e.ok ? 1.0f : 0.f;
    else
        v[28] = e.ok ? 1.0f : 0.f;
}

// Sums of the 64-float rows (columns 0-28 ICP, of nicp chunks; 32-60 photometric, of nrgb) into
// total[0..63] (LDS): four waves each add every fourth chunk in order (compensated, one value per
// lane) and are added pairwise.  NW = 16 waves (a row per chunk) bring the rows into LDS kSumTile
// at a time, eight loads of a lane in flight; NW = 4 (four rows per chunk, one of each quarter)
// add them as they come, eight chunks in flight.  Chunks past a column's end count as +0.
constexpr int kSumTile = 128;
template <int NW>
__device__ __forceinline__ void sum_rows64(const float* parts, int nicp, int nrgb, float* total) {
    __shared__ float wsum[4][64];
    const int lane = lane_id(), wave = threadIdx.x >> 6;
    const int mine = lane < 32 ? nicp : nrgb, most = max(nicp, nrgb);
    Kahan k{0.f, 0.f};
    if constexpr (NW == 16) {
        __shared__ float tile[kSumTile][64];
        for (int base = 0; base < most; base += kSumTile) {
            if (base) __syncthreads();  // the previous tile is added
            float x[kSumTile / 16];
#pragma unroll
            for (int u = 0; u < kSumTile / 16; ++u) {
                const int c = base + u * 16 + wave;
                x[u] = load_agent(parts + (c < mine ? c : 0) * 64 + lane);
            }
#pragma unroll
            for (int u = 0; u < kSumTile / 16; ++u) tile[u * 16 + wave][lane] = base + u * 16 + wave < mine ? x[u] : 0.f;
            __syncthreads();
            if (wave < 4)
                for (int c = wave; c < min(kSumTile, most - base); c += 4) k.add(tile[c][lane]);
        }
    } else {
        for (int base = wave; base < most; base += 32) {
            float x[8][4];
#pragma unroll
            for (int u = 0; u < 8; ++u)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int c = base + 4 * u;
                    x[u][r] = load_agent(parts + ((c < mine ? c : 0) * 4 + r) * 64 + lane);
                }
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const float t = (x[u][0] + x[u][1]) + (x[u][2] + x[u][3]);
                k.add(base + 4 * u < mine ? t : 0.f);
            }
        }
    }
    if (wave < 4) wsum[wave][lane] = k.val();
    __syncthreads();
    if (wave == 0) total[lane] = (wsum[0][lane] + wsum[1][lane]) + (wsum[2][lane] + wsum[3][lane]);
}

// ICP rows and photometric rows of the kRgbPixels chunks (two pixels or two list entries per lane,
// added before the wave reduction) by work-groups of their own: the first `nicp` take the pixels,
// the others the list, of which those past its end leave at once.  One work-group doing both kept
// the photometric rows to the few that hold list entries, which then took twice as long as the
// others, and 84 registers (one 1024-lane work-group per CU).  Row c: the ICP sums of chunk c in
// columns 0-28, its photometric sums in 32-60 (four rows per chunk in the kQuarter form).
// nresid: work-groups of the residual pass, whose integer sums give sigma.
__device__ __forceinline__ int rgb_icp_groups(const IcpArgs& a, int groups) {
    return a.ncurr ? groups >> 1 : 0;  // no normals: photometric rows only
}
// list chunks that hold entries; the first is always taken, so an iteration without any ends too
__device__ __forceinline__ int rgb_list_chunks(int n) { return max(1, (n + kRgbPixels - 1) / kRgbPixels); }

template <int FORM>
__device__ __forceinline__ void icp_rgb_last(const IcpArgs& a, int nicp, int nrgb) {
    __shared__ float total[64];
    __shared__ double sm[64];
    const UpdateIn in = load_update(a.st);
    sum_rows64<FORM == kQuarter ? 4 : 16>(a.partials, nicp, nrgb, total);
    if (threadIdx.x >= 64) return;
    wave_sync();
    const int lane = threadIdx.x;
    if (lane < 29) {
        a.st->sums[lane] = total[lane];
        a.st->rgb_sums[lane] = total[32 + lane];
    }
    if (a.mode == 1) icp_update_wave<true>(a, total, in, sm);
}

template <int FORM, bool kTicket>
__device__ __forceinline__ void icp_rgb_body(WG g, const IcpArgs& a, int nresid) {
    constexpr int NT = FORM == kQuarter ? 256 : kIcpThreads, NW = NT / 64, kParts = FORM == kQuarter ? 4 : 1;
    __shared__ float wsum[NW][32];
    const int nicp = rgb_icp_groups(a, g.nx);
    const bool list = g.x >= nicp;
    const int id = list ? g.x - nicp : g.x;
    const int i0 = id / kParts * kRgbPixels + id % kParts * NT + threadIdx.x, i1 = i0 + kIcpThreads;
    float v[32];
    int n;
    if (!list) {
        const int N = a.cols * a.rows;
        IcpPixel p, q;
        icp_load(a, i0, i0 < N, p);
        icp_load(a, i1, i1 < N, q);
        const auto st = FU_G(const TrackState, a.st);
        if (a.mode != 0 && st->status != TS_RUNNING) return;
        n = *FU_G(const int, a.rgb.count);
        icp_pixels(a, icp_pose(a.st), p, q, v);
        v[29] = v[30] = v[31] = 0.f;
        block_rows29(v, wsum, a.partials + id * 64);
    } else {
        const auto st = FU_G(const TrackState, a.st);
        if (a.mode != 0 && st->status != TS_RUNNING) return;
        n = *FU_G(const int, a.rgb.count);
        if (id / kParts >= rgb_list_chunks(n)) return;  // uniform
        RgbEntry e, f;
        rgb_load(a, i0, n, e);
        rgb_load(a, i1, n, f);
        rgb_gather(a, e);
        rgb_gather(a, f);
        int ci, qi;
        const float sigma = rgb_sigma(a, nresid, ci, qi);
        if (id == 0 && threadIdx.x == 0) {
            a.st->rgb_corresp[0] = ci;
            a.st->rgb_corresp[1] = qi;
            a.st->sigma = sigma;
        }
        const RgbPose Q = rgb_pose(a.st);
        rgb_row_values<false>(a, Q, e, sigma, v);
        rgb_row_values<true>(a, Q, f, sigma, v);
        v[29] = v[30] = v[31] = 0.f;
        block_rows29(v, wsum, a.partials + id * 64 + 32);
    }
    if constexpr (kTicket) {
        const int nrgb = rgb_list_chunks(n);
        if (last_to_arrive(a.st, nicp + nrgb * kParts)) icp_rgb_last<FORM>(a, nicp / kParts, nrgb);
    }
}
// eight waves per SIMD (64 registers), so that two 1024-lane work-groups share a CU
template <int FORM>
__global__ __launch_bounds__(FORM == kQuarter ? 256 : kIcpThreads) void k_icp_rgb(IcpArgs a, int nresid) {
    icp_rgb_body<FORM, true>(hw_wg(), a, nresid);
}

__global__ __launch_bounds__(kIcpThreads) void k_rgb_count(IcpArgs a) { rgb_count_body(hw_wg(), a); }
__global__ __launch_bounds__(kIcpThreads) void k_rgb_scatter(IcpArgs a) { rgb_scatter_body(hw_wg(), a); }
void launch_rgb_lists(const IcpArgs* a, const int* nblocks, int nlevels, hipStream_t s) {
    for (int l = 0; l < nlevels; ++l)
        if (a[l].use_rgb) {
            hipLaunchKernelGGL(k_rgb_count, dim3(nblocks[l]), dim3(kIcpThreads), 0, s, a[l]);
            hipLaunchKernelGGL(k_rgb_scatter, dim3(nblocks[l]), dim3(kIcpThreads), 0, s, a[l]);
        }
}

// A launch of up to kQuarterChunks chunks leaves most CUs idle with a chunk per work-group (a
// chunk's 2048 pixels are 3.5 us of VALU issue on one CU): its chunks are split in four.  More
// chunks would make the last work-group's rows (128 bytes each) cost what the split gains.
constexpr int kQuarterChunks = 128;
// Above kLastGroups chunks a launch is bound by issue, and a work-group that waits about a
// microsecond for its row and its count holds up the next: the rows are summed by a second launch.
constexpr int kLastGroups = 4096;

void launch_icp_step(const IcpArgs& a, int nblocks, const float Rcurr[9], const float tcurr[3], const float Rlast[9],
                     const float RlastInv[9], const float tlast[3], float* out, hipStream_t s) {
    auto m = [](const float* r) { return m3{mk3(r[0], r[1], r[2]), mk3(r[3], r[4], r[5]), mk3(r[6], r[7], r[8])}; };
    const IcpStep step{IcpPose{m(Rcurr), m(Rlast), m(RlastInv), mk3(tcurr[0], tcurr[1], tcurr[2]),
                               mk3(tlast[0], tlast[1], tlast[2])},
                       out};
    if ((long long)nblocks * kIcpPixels < (long long)a.cols * a.rows)
        hipLaunchKernelGGL(k_icp_step<kLoop>, dim3(nblocks), dim3(kIcpThreads), 0, s, a, step);
    else if (nblocks <= kQuarterChunks)
        hipLaunchKernelGGL(k_icp_step<kQuarter>, dim3(nblocks * 4), dim3(256), 0, s, a, step);
    else
        hipLaunchKernelGGL(k_icp_step<kChunk>, dim3(nblocks), dim3(kIcpThreads), 0, s, a, step);
}

void launch_icp(const IcpArgs& a, int nblocks, hipStream_t s) {
    if (a.use_rgb) {  // one pixel per lane (the caller sizes nblocks to cover the level)
        hipLaunchKernelGGL(k_rgb_resid, dim3(nblocks), dim3(kIcpThreads), 0, s, a);
        const int pairs = (nblocks + 1) / 2;  // kRgbPixels chunks of the combined pass
        const int kinds = a.ncurr ? 2 : 1;
        if (pairs <= kQuarterChunks)
            hipLaunchKernelGGL(k_icp_rgb<kQuarter>, dim3(pairs * kinds * 4), dim3(256), 0, s, a, nblocks);
        else
            hipLaunchKernelGGL(k_icp_rgb<kChunk>, dim3(pairs * kinds), dim3(kIcpThreads), 0, s, a, nblocks);
        return;
    }
    if ((long long)nblocks * kIcpPixels < (long long)a.cols * a.rows)
        hipLaunchKernelGGL(k_icp<kLoop>, dim3(nblocks), dim3(kIcpThreads), 0, s, a);
    else if (nblocks <= kQuarterChunks)
        hipLaunchKernelGGL(k_icp<kQuarter>, dim3(nblocks * 4), dim3(256), 0, s, a);
    else
        hipLaunchKernelGGL(k_icp<kChunk>, dim3(nblocks), dim3(kIcpThreads), 0, s, a);
}

// before tracking: a lost tracker does not track; otherwise the start of ComputeSE3
// (frame_begin)
__device__ __forceinline__ void track_begin_body(TrackState* st) {
    if (threadIdx.x != 0) return;
    frame_begin(st);
}
__global__ void k_track_begin(TrackState* st) { track_begin_body(st); }
// after tracking: the state machine decides what the frame does, and a swapped frame's pose
// becomes the last pose (frame_commit); the map's counters for the fusion that follows
__device__ __forceinline__ void track_commit_body(TrackState* st, unsigned* ctr) {
    if (threadIdx.x == 0) frame_commit(st);
    begin_pass(ctr, 3);
}
__global__ void k_track_commit(TrackState* st, unsigned* ctr) { track_commit_body(st, ctr); }
void launch_track_begin(TrackState* st, hipStream_t s) { hipLaunchKernelGGL(k_track_begin, dim3(1), dim3(64), 0, s, st); }
void launch_track_commit(TrackState* st, const MapView& m, hipStream_t s) {
    hipLaunchKernelGGL(k_track_commit, dim3(1), dim3(64), 0, s, st, m.ctr);
}

// ------------------------------------------------------------------ batched launches
// The iteration schedule is the union of the sessions' schedules: a session runs iteration
// `iter` of `level` only if it has that many, and its last iteration is final.
__device__ __forceinline__ bool icp_slot_args(const BatchLaunch& b, int s, IcpArgs& a, int& nblocks) {
    if (slot_first(b, s)) return false;
    const SessDesc& d = b.desc[b.sess[s]];
    const int l = b.level;
    if (b.iter >= d.iters[l]) return false;
    a = cload(d.icp[l]);
    a.final_iter = (l == d.last_level && b.iter == d.iters[l] - 1) ? 1 : 0;
    nblocks = d.icp_blocks[l];
    return true;
}

template <int FORM, bool kTicket>
__global__ __launch_bounds__(FORM == kQuarter ? 256 : kIcpThreads) void kb_icp(BatchLaunch b) {
    WG g;
    const int s = batch_slot(b, batch_wg(b), g);
    IcpArgs a;
    int nb;
    if (!icp_slot_args(b, s, a, nb)) return;
    icp_body<FORM, kTicket>(g, a);
}
// the rows of every session, where their work-groups do not sum them
__global__ __launch_bounds__(kIcpThreads) void kb_icp_last(BatchLaunch b) {
    IcpArgs a;
    int nb;
    if (!icp_slot_args(b, blockIdx.x, a, nb)) return;
    if (a.mode != 0 && FU_G(const TrackState, a.st)->status != TS_RUNNING) return;
    icp_last<kIcpThreads / 64>(a, nb);
}

__global__ __launch_bounds__(kIcpThreads) void kb_rgb_count(BatchLaunch b) {
    WG g;
    const int s = batch_slot(b, blockIdx.x, g);
    IcpArgs a;
    int nb;
    if (!icp_slot_args(b, s, a, nb)) return;
    rgb_count_body(g, a);
}
__global__ __launch_bounds__(kIcpThreads) void kb_rgb_scatter(BatchLaunch b) {
    WG g;
    const int s = batch_slot(b, blockIdx.x, g);
    IcpArgs a;
    int nb;
    if (!icp_slot_args(b, s, a, nb)) return;
    rgb_scatter_body(g, a);
}
__global__ __launch_bounds__(kIcpThreads) void kb_rgb_resid(BatchLaunch b) {
    WG g;
    const int s = batch_slot(b, batch_wg(b), g);
    IcpArgs a;
    int nb;
    if (!icp_slot_args(b, s, a, nb)) return;
    rgb_resid_body(g, a);
}
template <int FORM, bool kTicket>
__global__ __launch_bounds__(FORM == kQuarter ? 256 : kIcpThreads) void kb_icp_rgb(BatchLaunch b) {
    WG g;
    const int s = batch_slot(b, batch_wg(b), g);
    IcpArgs a;
    int nb;
    if (!icp_slot_args(b, s, a, nb)) return;
    icp_rgb_body<FORM, kTicket>(g, a, nb);
}
__global__ __launch_bounds__(kIcpThreads) void kb_icp_rgb_last(BatchLaunch b) {
    IcpArgs a;
    int nb;
    if (!icp_slot_args(b, blockIdx.x, a, nb)) return;
    if (a.mode != 0 && FU_G(const TrackState, a.st)->status != TS_RUNNING) return;
    icp_rgb_last<kChunk>(a, (nb + 1) / 2, rgb_list_chunks(*FU_G(const int, a.rgb.count)));
}

__global__ void kb_track_begin(BatchLaunch b) {
    const int s = blockIdx.x;
    if (slot_first(b, s)) return;
    track_begin_body(b.desc[b.sess[s]].st);
}
__global__ void kb_track_commit(BatchLaunch b) {
    const SessDesc& d = b.desc[b.sess[blockIdx.x]];
    track_commit_body(d.st, d.m.ctr);
}

// tracking result and map counters of every slot, into out[slot]
__global__ void kb_results(BatchLaunch b, FrameBrief* out) {
    const int s = blockIdx.x;
    const SessDesc& d = b.desc[b.sess[s]];
    const TrackState* st = d.st;
    FrameBrief* o = out + s;
    const int t = threadIdx.x;
    if (t < 16) o->pose[t] = st->next_pose[t];
    if (t == 16) o->status = st->status;
    if (t == 17) o->icp_error = st->icp_error;
    if (t == 18) o->icp_count = st->count;
    if (t == 19) o->n_visible = d.m.ctr[C_VISIBLE];
    if (t == 20) o->n_alloc = min(d.m.ctr[C_ALLOC], d.m.num_blocks);
    if (t == 21) o->flags = d.m.ctr[C_FLAGS];
    if (t == 22) o->rgb_count = d.use_rgb ? st->rgb_count : 0;
}
// the states of the first n sessions, one after the other
__global__ __launch_bounds__(256) void k_states(const SessDesc* desc, unsigned* out) {
    const auto src = FU_G(const unsigned, reinterpret_cast<const unsigned*>(desc[blockIdx.x].st));
    constexpr int n = (int)(sizeof(TrackState) / 4);
    for (int i = threadIdx.x; i < n; i += 256) out[blockIdx.x * n + i] = src[i];
}
void launch_states(const SessDesc* desc, int n, void* out, hipStream_t s) {
    hipLaunchKernelGGL(k_states, dim3(n), dim3(256), 0, s, desc, (unsigned*)out);
}
void launch_b_results(BatchLaunch& b, FrameBrief* out, hipStream_t s) {
    hipLaunchKernelGGL(kb_results, dim3(b.n), dim3(64), 0, s, b, out);
}

void launch_b_track_begin(BatchLaunch& b, const SessDesc* h, hipStream_t s) {
    (void)h;
    hipLaunchKernelGGL(kb_track_begin, dim3(b.n), dim3(64), 0, s, b);
}
void launch_b_icp(BatchLaunch& b, const SessDesc* h, int level, int iter, hipStream_t s) {
    b.level = level;
    b.iter = iter;
    b.xcd = xcd_order(FU_STAGE_ICP);
    if (h[b.sess[0]].use_rgb) {  // the sessions of a batch share the tracking mode
        const int grid = batch_layout(b, h, BT_ICP, level, 1);
        hipLaunchKernelGGL(kb_rgb_resid, dim3(grid), dim3(kIcpThreads), 0, s, b);
        // pixels and list entries in work-groups of their own
        const int pairs = batch_layout(b, h, BT_ICP_PAIRS, level, 2) / 2;
        if (pairs <= kQuarterChunks) {
            hipLaunchKernelGGL((kb_icp_rgb<kQuarter, true>), dim3(batch_layout(b, h, BT_ICP_PAIRS, level, 8)), dim3(256), 0,
                               s, b);
        } else if (pairs <= kLastGroups) {
            hipLaunchKernelGGL((kb_icp_rgb<kChunk, true>), dim3(pairs * 2), dim3(kIcpThreads), 0, s, b);
        } else {
            hipLaunchKernelGGL((kb_icp_rgb<kChunk, false>), dim3(pairs * 2), dim3(kIcpThreads), 0, s, b);
            hipLaunchKernelGGL(kb_icp_rgb_last, dim3(b.n), dim3(kIcpThreads), 0, s, b);
        }
        return;
    }
    bool one = true;
    for (int i = 0; i < b.n; ++i) {
        const SessDesc& d = h[b.sess[i]];
        one = one && (long long)d.icp_blocks[level] * kIcpPixels >= (long long)d.lc[level] * d.lr[level];
    }
    const int grid = batch_layout(b, h, BT_ICP, level, 1);
    if (grid > kLastGroups) {
        if (one)
            hipLaunchKernelGGL((kb_icp<kChunk, false>), dim3(grid), dim3(kIcpThreads), 0, s, b);
        else
            hipLaunchKernelGGL((kb_icp<kLoop, false>), dim3(grid), dim3(kIcpThreads), 0, s, b);
        hipLaunchKernelGGL(kb_icp_last, dim3(b.n), dim3(kIcpThreads), 0, s, b);
    } else if (!one) {
        hipLaunchKernelGGL((kb_icp<kLoop, true>), dim3(grid), dim3(kIcpThreads), 0, s, b);
    } else if (grid <= kQuarterChunks) {
        hipLaunchKernelGGL((kb_icp<kQuarter, true>), dim3(batch_layout(b, h, BT_ICP, level, 4)), dim3(256), 0, s, b);
    } else {
        hipLaunchKernelGGL((kb_icp<kChunk, true>), dim3(grid), dim3(kIcpThreads), 0, s, b);
    }
}
// the eligible-pixel lists of every level (iteration 0 of each level: a session without
// iterations at a level builds none)
void launch_b_rgb_lists(BatchLaunch& b, const SessDesc* h, hipStream_t s) {
    for (int l = 0; l < 3; ++l) {
        b.level = l;
        b.iter = 0;
        const int grid = batch_layout(b, h, BT_ICP, l, 1);
        hipLaunchKernelGGL(kb_rgb_count, dim3(grid), dim3(kIcpThreads), 0, s, b);
        hipLaunchKernelGGL(kb_rgb_scatter, dim3(grid), dim3(kIcpThreads), 0, s, b);
    }
}

void launch_b_track_commit(BatchLaunch& b, const SessDesc* h, hipStream_t s) {
    (void)h;
    hipLaunchKernelGGL(kb_track_commit, dim3(b.n), dim3(64), 0, s, b);
}

}  // namespace fu
