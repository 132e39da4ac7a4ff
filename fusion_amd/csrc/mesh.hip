// Two-pass marching cubes over all allocated blocks.
//
// Reference: Mapping/MeshScene.cu (checkBlocks :20-41, readNormal :43-103,
// readVertexAndColor :105-140, interp :142-150, buildVertexList :152-259,
// MarchingCube :261-295).  The reference runs one pass with a global atomic triangle
// counter and 32 hash lookups per voxel.  Here:
//   count  one work-group per block reads the block plus a one-voxel halo below and a
//          two-voxel halo above (11^3 sdf values, from the 27 neighbouring blocks looked up
//          once) as bit masks, a row of 11 voxels per mask: which are NaN, which are 1.0 and
//          which are negative.  A voxel's tests and its case are bits of 16 of those rows;
//   scan   exclusive scan of the per-block counts in chunks; the last chunk to be summed scans
//          the chunk sums;
//   emit   reads the blocks that have triangles again, now keeping values and colours in LDS,
//          lists their triangles in voxel-index order and makes one vertex per lane.
// Allocated blocks are read straight from the pool-ordered key array, so no compaction
// pass over the N_E hash entries is needed (checkBlocks).
//
// Measured on a room of 4,772 blocks and 427,000 triangles (10 mm): count 48 -> 21 us, scan
// (three launches before) 18 -> 5 us, emit 128 -> 37 us.  Before, every voxel tested 56
// values in LDS, and the few lanes with triangles made and wrote all of theirs one after the
// other, three floats or bytes at a time.
#include "fu_device.h"
#include "fu_kernels.h"
#include "mc_tables.h"

namespace fu {

__constant__ unsigned long long c_mc_tri[256];

void upload_mc_tables() {
    unsigned long long tri[256];
    for (int c = 0; c < 256; ++c) tri[c] = mc_packed(c);
    (void)hipMemcpyToSymbol(HIP_SYMBOL(c_mc_tri), tri, sizeof(tri));
}

// corners joined by edge e: edges 0-7 run around the bottom and top faces, 8-11 are the
// vertical edges (MeshScene.cu:185-256)
__device__ __forceinline__ int kMcEdgeCornerDev(int e, int k) {
    if (e < 8) return k == 0 ? e : ((e & 4) | ((e + 1) & 3));
    return k == 0 ? e - 8 : e - 4;
}

constexpr int kHalo = 11;  // voxels -1 .. 9 relative to the block origin
constexpr int kHalo3 = kHalo * kHalo * kHalo;
constexpr int kRows = kHalo * kHalo;  // rows of kHalo voxels along x

struct MeshMasks {
    int nb[27];
    // bit x + 1 of row (z + 1) * 11 + y + 1: the voxel is NaN (absent); NaN or exactly 1.0;
    // negative
    unsigned short nan[kRows], bad[kRows], neg[kRows];
    unsigned char ntri[256];  // triangles of each case
    int wsum[4];
};
struct MeshValues {
    float sdf[kHalo3];
    unsigned rgb[kHalo3];
};

__device__ __forceinline__ int hidx(int x, int y, int z) { return ((z + 1) * kHalo + (y + 1)) * kHalo + (x + 1); }

__device__ __forceinline__ void load_ntri(MeshMasks& s) {
    s.ntri[threadIdx.x] = (unsigned char)(c_mc_tri[threadIdx.x] >> 60);
}

// The halo of block bp into the masks (and, with val, the values): 16 lanes per row, so a load
// of a wave covers four rows and its ballots are their masks; a wave's eight loads go out together.
template <int F, bool kValues>
__device__ void stage_block(const MapView& m, i3 bp, MeshMasks& s, MeshValues* val) {
    using IO = VoxelIO<F>;
    const int t = threadIdx.x;
    if (t < 27) {
        const i3 nbp = mki3(bp.x + t % 3 - 1, bp.y + (t / 3) % 3 - 1, bp.z + t / 9 - 1);
        s.nb[t] = find_block(m, nbp);
    }
    __syncthreads();
    const int lane = lane_id(), wave = t >> 6, sub = lane >> 4, x = lane & 15;
    constexpr int kSteps = (kRows + 15) / 16;  // four waves, four rows each
    const int rx = x - 1, ox = rx < 0 ? 0 : (rx >= 8 ? 2 : 1);
    int heap[kSteps], li[kSteps];
    float sd[kSteps];
#pragma unroll
    for (int k = 0; k < kSteps; ++k) {
        const int row = (k * 4 + wave) * 4 + sub;
        const int rz = row / kHalo - 1, ry = row % kHalo - 1;
        const int oz = rz < 0 ? 0 : (rz >= 8 ? 2 : 1), oy = ry < 0 ? 0 : (ry >= 8 ? 2 : 1);
        const bool in = row < kRows && x < kHalo;
        heap[k] = in ? s.nb[oz * 9 + oy * 3 + ox] : -1;
        li[k] = ((rz & 7) * 8 + (ry & 7)) * 8 + (rx & 7);
        sd[k] = heap[k] >= 0 ? IO::sdf(IO::block(m, heap[k]), li[k]) : fnan();
    }
#pragma unroll
    for (int k = 0; k < kSteps; ++k) {
        const int row = (k * 4 + wave) * 4 + sub;
        const unsigned long long n = ballot(isnanf_(sd[k])), b = ballot(isnanf_(sd[k]) || sd[k] == 1.0f),
                                 g = ballot(sd[k] < 0);
        if (row < kRows) {
            if (x == 0) {  // bits past the row's 11 voxels are not looked at
                s.nan[row] = (unsigned short)(n >> (sub * 16));
                s.bad[row] = (unsigned short)(b >> (sub * 16));
                s.neg[row] = (unsigned short)(g >> (sub * 16));
            }
            if constexpr (kValues)
                if (x < kHalo) {
                    unsigned c = 0;
                    if (heap[k] >= 0) {
                        const VoxAux a = IO::aux(IO::block(m, heap[k]), li[k]);
                        c = (unsigned)a.r | ((unsigned)a.g << 8) | ((unsigned)a.b << 16);
                    }
                    val->sdf[row * kHalo + x] = sd[k];
                    val->rgb[row * kHalo + x] = c;
                }
        }
    }
    __syncthreads();
}

// corner c of the cell (MeshScene.cu:107-135 order)
__device__ __forceinline__ void corner_off(int c, int& dx, int& dy, int& dz) {
    dx = (c & 1) ^ ((c >> 1) & 1);
    dy = (c >> 1) & 1;
    dz = (c >> 2) & 1;
}

// The cube indices of the lane's voxels 2 t and 2 t + 1 (index z * 64 + y * 8 + x), 0 when a
// corner is NaN or exactly 1.0, a central-difference neighbour of a corner is NaN, or the case
// has no edges (buildVertexList, MeshScene.cu:152-183; case 0 has none)
__device__ __forceinline__ void classify2(const MeshMasks& s, int (&cube)[2]) {
    const int t = threadIdx.x, r = t >> 2, y = r & 7, z = r >> 3;
    const int r00 = (z + 1) * kHalo + y + 1;  // row (y, z); (y + 1, z) is the next, (y, z + 1) 11 on
    const unsigned corner = s.bad[r00] | s.bad[r00 + 1] | s.bad[r00 + kHalo] | s.bad[r00 + kHalo + 1];
    const unsigned along = s.nan[r00] | s.nan[r00 + 1] | s.nan[r00 + kHalo] | s.nan[r00 + kHalo + 1];
    const unsigned beside = s.nan[r00 - 1] | s.nan[r00 + 2] | s.nan[r00 + kHalo - 1] | s.nan[r00 + kHalo + 2] |
                            s.nan[r00 - kHalo] | s.nan[r00 - kHalo + 1] | s.nan[r00 + 2 * kHalo] |
                            s.nan[r00 + 2 * kHalo + 1];
    const unsigned n00 = s.neg[r00], n10 = s.neg[r00 + 1], n01 = s.neg[r00 + kHalo], n11 = s.neg[r00 + kHalo + 1];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int x = (t & 3) * 2 + h;
        // corners at x and x + 1 (bits x + 1, x + 2), their neighbours along x from x - 1 to x + 2
        const bool bad = ((((corner | beside) >> (x + 1)) & 3u) | ((along >> x) & 15u)) != 0;
        auto pair = [&](unsigned n) { return (n >> (x + 1)) & 3u; };
        auto back = [&](unsigned p) { return (p >> 1) | ((p & 1u) << 1); };  // corners 2, 3 run the other way
        const unsigned c = pair(n00) | back(pair(n10)) << 2 | pair(n01) << 4 | back(pair(n11)) << 6;
        cube[h] = bad ? 0 : (int)c;
    }
}

// wave-inclusive scan
__device__ __forceinline__ int wave_scan(int v) {
    const int lane = lane_id();
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int y = __shfl_up(v, d);
        if (lane >= d) v += y;
    }
    return v;
}

template <int F>
__global__ __launch_bounds__(256) void k_mesh_count(MapView m, unsigned* counts) {
    __shared__ MeshMasks s;
    load_ntri(s);
    if (blockIdx.x == 0 && threadIdx.x == 0) m.ctr[C_DONE] = 0;  // k_mesh_scan counts its chunks there
    const unsigned nalloc = min(m.ctr[C_ALLOC], m.num_blocks);
    for (unsigned b = blockIdx.x; b < nalloc; b += gridDim.x) {
        const unsigned long long key = m.block_key[b];
        if (key == kEmptyKey) {
            if (threadIdx.x == 0) counts[b] = 0;
            continue;
        }
        stage_block<F, false>(m, unpack_key(key), s, nullptr);
        int cube[2];
        classify2(s, cube);
        const int n = wave_scan((int)s.ntri[cube[0]] + (int)s.ntri[cube[1]]);
        if (lane_id() == 63) s.wsum[threadIdx.x >> 6] = n;
        __syncthreads();
        if (threadIdx.x == 0) counts[b] = (unsigned)(s.wsum[0] + s.wsum[1] + s.wsum[2] + s.wsum[3]);
    }
}

// ---- exclusive scan of counts[0..n) (n read from the allocation counter) ----------------
// Work-group c scans chunk c in place (offsets within the chunk) and hands on its sum and its
// number of blocks with triangles; the last of them to arrive scans those: base[c] is the first
// triangle of chunk c, base[chunks] their total.  The sums travel as agent-scope relaxed atomic
// accesses, counted once the storing wave's stores are complete (as the rows of an ICP iteration).
constexpr int kChunk = 2048;
constexpr int kScanLanes = 1024;  // two counts per lane

// exclusive scan over the work-group's lanes; `total` is uniform
__device__ __forceinline__ int scan_lanes(int v, int* wsum, int& total) {
    const int incl = wave_scan(v), w = threadIdx.x >> 6;
    __syncthreads();  // wsum may still be read from a previous scan
    if (lane_id() == 63) wsum[w] = incl;
    __syncthreads();
    int before = 0, all = 0;
#pragma unroll
    for (int k = 0; k < kScanLanes / 64; ++k) {
        before += k < w ? wsum[k] : 0;
        all += wsum[k];
    }
    total = all;
    return before + incl - v;
}
// `sums`: two words per chunk (triangles, blocks with triangles)
__global__ __launch_bounds__(kScanLanes) void k_mesh_scan(MapView m, unsigned* counts, unsigned* base, unsigned* sums) {
    __shared__ int wsum[kScanLanes / 64];
    __shared__ int last;
    const unsigned n = min(m.ctr[C_ALLOC], m.num_blocks);
    const int chunks = max(1, (int)((n + kChunk - 1) / kChunk));
    if ((int)blockIdx.x >= chunks) return;  // uniform
    const unsigned i = blockIdx.x * kChunk + 2 * threadIdx.x;
    const int v0 = i < n ? (int)counts[i] : 0, v1 = i + 1 < n ? (int)counts[i + 1] : 0;
    int total, occ;
    const int ex = scan_lanes(v0 + v1, wsum, total);
    if (i < n) counts[i] = (unsigned)ex;
    if (i + 1 < n) counts[i + 1] = (unsigned)(ex + v0);
    scan_lanes((v0 > 0) + (v1 > 0), wsum, occ);
    if (threadIdx.x < 64) {
        if (threadIdx.x == 0) {
            __hip_atomic_store(FU_G(unsigned, sums) + 2 * blockIdx.x, (unsigned)total, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(FU_G(unsigned, sums) + 2 * blockIdx.x + 1, (unsigned)occ, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the sums are in place
        if (threadIdx.x == 0) {
            const unsigned before = atomicAdd(&m.ctr[C_DONE], 1u);
            last = before == (unsigned)chunks - 1u;
        }
    }
    __syncthreads();
    if (!last) return;
    unsigned carry = 0, occupied = 0;
    for (int c0 = 0; c0 < chunks; c0 += kScanLanes) {
        const int c = c0 + (int)threadIdx.x;
        int t = 0, o = 0;
        if (c < chunks) {
            t = (int)__hip_atomic_load(FU_G(const unsigned, sums) + 2 * c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            o = (int)__hip_atomic_load(FU_G(const unsigned, sums) + 2 * c + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        const int e = scan_lanes(t, wsum, total);
        if (c < chunks) base[c] = carry + (unsigned)e;
        carry += (unsigned)total;
        scan_lanes(o, wsum, occ);
        occupied += (unsigned)occ;
    }
    if (threadIdx.x == 0) {
        base[chunks] = carry;
        m.ctr[C_TRI] = carry;
        m.ctr[C_OCC] = occupied;
    }
}

// ---- emit --------------------------------------------------------------------------------
__device__ __forceinline__ float mc_interp(float v1, float v2) {
    // MeshScene.cu:142-150 (fabs of a float compared against the double 1e-6)
    if ((double)fabsf(0.0f - v1) < 1e-6) return 0.0f;
    if ((double)fabsf(0.0f - v2) < 1e-6) return 1.0f;
    if ((double)fabsf(v1 - v2) < 1e-6) return 0.0f;
    return (0.0f - v1) / (v2 - v1);
}

// Lane v of a batch makes vertex v (three per triangle in list order), so the lanes share the work
// evenly however the triangles fall on the voxels, and a wave's vertices, normals and colours are
// contiguous in the output.
// Six waves per SIMD: a block is a chain of loads, so what counts is how many are under way (43 us
// with the 105 registers the compiler would take).
template <int F>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(6, 8))) void k_mesh_emit(MapView m, const unsigned* offsets, const unsigned* base, MeshOut o) {
    __shared__ MeshMasks s;
    __shared__ MeshValues val;
    __shared__ unsigned char cubes[512];
    __shared__ unsigned short list[512 * 5];  // voxel index << 3 | triangle of its case
    load_ntri(s);
    const unsigned nalloc = min(m.ctr[C_ALLOC], m.num_blocks);
    const int t = threadIdx.x;
    for (unsigned b = blockIdx.x; b < nalloc; b += gridDim.x) {
        const unsigned long long key = m.block_key[b];
        if (key == kEmptyKey) continue;
        const unsigned c = b / kChunk;
        const unsigned start = base[c] + offsets[b];
        const unsigned end = (b + 1 < nalloc && b + 1 < (c + 1) * kChunk) ? base[c] + offsets[b + 1] : base[c + 1];
        if (end == start || start >= o.max_tri) continue;
        const i3 bp = unpack_key(key);
        __syncthreads();  // the previous block's list is done
        stage_block<F, true>(m, bp, s, &val);
        int cube[2];
        classify2(s, cube);
        const int n0 = s.ntri[cube[0]], n1 = s.ntri[cube[1]];
        const int incl = wave_scan(n0 + n1);
        if (lane_id() == 63) s.wsum[t >> 6] = incl;
        cubes[2 * t] = (unsigned char)cube[0];
        cubes[2 * t + 1] = (unsigned char)cube[1];
        __syncthreads();
        int at = incl - n0 - n1;
        for (int k = 0; k < (t >> 6); ++k) at += s.wsum[k];
        for (int k = 0; k < n0; ++k) list[at + k] = (unsigned short)((2 * t) << 3 | k);
        for (int k = 0; k < n1; ++k) list[at + n0 + k] = (unsigned short)((2 * t + 1) << 3 | k);
        __syncthreads();
        const int nv = 3 * (int)(min(end, o.max_tri) - start);
        for (int v = t; v < nv; v += 256) {
            const int tri = v / 3, k = v - tri * 3;
            const int ent = list[tri], li = ent >> 3, q = ent & 7;
            const int lx = li & 7, ly = (li >> 3) & 7, lz = li >> 6;
            const int cb = cubes[li];
            const int e = (int)((c_mc_tri[cb] >> (4 * (3 * q + k))) & 0xF);
            const int ca = kMcEdgeCornerDev(e, 0), cc = kMcEdgeCornerDev(e, 1);
            int ax, ay, az, bx, by, bz;
            corner_off(ca, ax, ay, az);
            corner_off(cc, bx, by, bz);
            const int ha = hidx(lx + ax, ly + ay, lz + az), hb = hidx(lx + bx, ly + by, lz + bz);
            // corner normals: central differences (MeshScene.cu:43-103)
            auto grad = [&](int h) {
                return mk3(val.sdf[h + 1] - val.sdf[h - 1], val.sdf[h + kHalo] - val.sdf[h - kHalo],
                           val.sdf[h + kRows] - val.sdf[h - kRows]);
            };
            const float val1 = mc_interp(val.sdf[ha], val.sdf[hb]);
            const float ox = bx == ax ? (float)ax : (bx > ax ? (float)ax + val1 : (float)ax - val1);
            const float oy = by == ay ? (float)ay : (by > ay ? (float)ay + val1 : (float)ay - val1);
            const float oz = bz == az ? (float)az : (bz > az ? (float)az + val1 : (float)az - val1);
            const i3 vp = mki3(bp.x * 8 + lx, bp.y * 8 + ly, bp.z * 8 + lz);
            const f3 vtx = mul(mk3((float)vp.x + ox, (float)vp.y + oy, (float)vp.z + oz), m.voxel_size);
            const f3 na = grad(ha), nb = grad(hb);
            const f3 nv3 = normalised(add(na, mul(val1, sub(nb, na))));
            const int iv = f2i(val1);
            const unsigned cola = val.rgb[ha], colb = val.rgb[hb];
            unsigned char col[3];
#pragma unroll
            for (int ch = 0; ch < 3; ++ch) {
                const unsigned a8 = (cola >> (8 * ch)) & 0xFF, b8 = (colb >> (8 * ch)) & 0xFF;
                const unsigned char d = (unsigned char)(b8 - a8);
                const unsigned char prod = (unsigned char)(int)(d * iv);
                col[ch] = (unsigned char)(a8 + prod);
            }
            const size_t vi = (size_t)start * 3 + v;
            *(FU_GPTR(f3))(FU_G(float, o.vertex) + vi * 3) = vtx;
            *(FU_GPTR(f3))(FU_G(float, o.normal) + vi * 3) = nv3;
            FU_G(unsigned char, o.color)[vi * 3 + 0] = col[0];
            FU_G(unsigned char, o.color)[vi * 3 + 1] = col[1];
            FU_G(unsigned char, o.color)[vi * 3 + 2] = col[2];
            if (o.tri_meta && k == 0) {
                const auto meta = FU_G(int, o.tri_meta) + ((size_t)start + tri) * 4;
                meta[0] = vp.x;
                meta[1] = vp.y;
                meta[2] = vp.z;
                meta[3] = cb * 16 + q;
            }
        }
    }
}

// chunk: (num_blocks + 2047) / 2048 + 1 bases, then two words per chunk
template <int F>
static void mesh_f(const MapView& m, const MeshOut& o, unsigned* counts, unsigned* chunk, hipStream_t s) {
    const unsigned nchunks = (m.num_blocks + kChunk - 1) / kChunk;
    const unsigned groups = min(m.num_blocks, 4096u);
    hipLaunchKernelGGL(k_mesh_count<F>, dim3(groups), dim3(256), 0, s, m, counts);
    hipLaunchKernelGGL(k_mesh_scan, dim3(nchunks), dim3(kScanLanes), 0, s, m, counts, chunk, chunk + nchunks + 1);
    hipLaunchKernelGGL(k_mesh_emit<F>, dim3(groups), dim3(256), 0, s, m, counts, chunk, o);
}
void launch_mesh(const MapView& m, const MeshOut& o, unsigned* counts, unsigned* chunk, hipStream_t s) {
    switch (m.fmt) {
        case VF_F32_W8: mesh_f<VF_F32_W8>(m, o, counts, chunk, s); break;
        case VF_F32_W16: mesh_f<VF_F32_W16>(m, o, counts, chunk, s); break;
        default: mesh_f<VF_F16_W8>(m, o, counts, chunk, s); break;
    }
}

}  // namespace fu
