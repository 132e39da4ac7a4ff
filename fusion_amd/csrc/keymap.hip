// The keypoint map: a bucketed hash of SURF records keyed by 1 cm grid cells, and the
// adjacency (consistency) matrix of matched keypoint pairs.
//
// Reference: Mapping/DeviceMap.h KeyMap (:163-185), DeviceMap.cu KeyMap::Hash / FindKey /
// InsertKey / ResetKeys (:203-296), Mapping/FuseMap.cu ResetKeyPoints / CollectKeyPoints /
// InsertKeyPoints (:366-472), Tracking/KeyPoints.cu BuildAdjacencyMatrix (:12-77).
//
// Inserts are applied as if one key at a time in index order: each round, every key still
// waiting claims its bucket with an atomic minimum of its index, and the owner of each bucket
// inserts (buckets are independent); the others wait for the next round.  The reference's
// per-bucket try-lock drops a key that meets another in its bucket in the same launch.
#include <hip/hip_runtime.h>
#include <limits.h>
#include <stddef.h>
#include <string.h>

#include <atomic>
#include <mutex>
#include <vector>

#include "fu_api.h"
#include "fu_keys.h"
#include "fu_mail.h"

using namespace fu;

namespace {

struct alignas(16) Surf {  // fu_surf / SURF: valid, pos, normal, descriptor (288 bytes)
    unsigned char valid;
    unsigned char pad[3];
    float pos[3];
    float normal[4];
    float desc[64];
};
static_assert(sizeof(Surf) == sizeof(fu_surf) && sizeof(Surf) == 288, "SURF layout");
constexpr int kSurfHeads = kSlotHeads;
static_assert(sizeof(Surf) % sizeof(SurfHead) == 0, "records are whole heads apart");

// KeyMap::Hash (DeviceMap.cu:206-214): the signed remainder of the wrapped products' xor
__device__ __forceinline__ int key_hash(i3 p, int max_keys) {
    const int h = (int)(((uint32_t)p.x * 73856093u) ^ ((uint32_t)p.y * 19349669u) ^ ((uint32_t)p.z * 83492791u));
    int r = h % max_keys;
    return r < 0 ? r + max_keys : r;
}
// make_int3(pos / GridSize)
__device__ __forceinline__ i3 key_cell(const float* pos, float grid) {
    return i3{f2i(pos[0] / grid), f2i(pos[1] / grid), f2i(pos[2] / grid)};
}

struct KeyArgs {
    Surf* keys;        // the map: max_keys * nbuckets records
    int* mutex;        // KeyMap::Mutex (reset to -1; the inserts here do not lock)
    int* owner;        // per bucket: INT_MAX, or the lowest index of a waiting key this round
    unsigned* bits;    // a bit per slot: its key is valid
    unsigned* valid;   // their number
    int max_keys, nbuckets;
    float grid;
};

// ResetKeys (DeviceMap.cu:289-296)
__global__ void k_reset_keys(KeyArgs a, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    a.mutex[i] = -1;
    a.keys[i].valid = 0;
    if ((i & 31) == 0) a.bits[i >> 5] = 0u;
    if (i == 0) *a.valid = 0u;
    if (i < a.max_keys) a.owner[i] = INT_MAX;
}

// one round of inserts: the claim, then the owners' inserts
__global__ void k_insert_claim(KeyArgs a, const Surf* in, const unsigned char* done, int* bucket, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n || done[i]) return;
    const int b = key_hash(key_cell(in[i].pos, a.grid), a.max_keys);
    bucket[i] = b;
    atomicMin(&a.owner[b], i);
}
__global__ void k_insert_apply(KeyArgs a, Surf* in, int* index, unsigned char* done, const int* bucket, int n,
                               unsigned* left) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n || done[i]) return;
    const int b = bucket[i];
    if (a.owner[b] != i) {
        atomicAdd(left, 1u);
        return;
    }
    // KeyMap::FindKey(pos, first, buck, hashIndex) and InsertKey
    const i3 p = key_cell(in[i].pos, a.grid);
    int first = -1, found = -1;
    for (int j = 0; j < a.nbuckets; ++j) {
        const int s = b * a.nbuckets + j;
        const Surf& k = a.keys[s];
        if (!k.valid && first == -1) first = s;
        if (k.valid && eqi(key_cell(k.pos, a.grid), p)) {
            found = s;
            break;
        }
    }
    if (found >= 0) {
        index[i] = found;
        in[i].pos[0] = a.keys[found].pos[0];
        in[i].pos[1] = a.keys[found].pos[1];
        in[i].pos[2] = a.keys[found].pos[2];
    } else if (first != -1) {
        index[i] = first;
        const uint4* src = reinterpret_cast<const uint4*>(&in[i]);
        uint4* dst = reinterpret_cast<uint4*>(&a.keys[first]);
        for (int q = 0; q < (int)(sizeof(Surf) / 16); ++q) dst[q] = src[q];
        if (in[i].valid) {
            atomicOr(&a.bits[first >> 5], 1u << (first & 31));
            atomicAdd(a.valid, 1u);
        }
    }
    done[i] = 1;
    a.owner[b] = INT_MAX;
}

// CollectKeys (FuseMap.cu:384-406) in slot order: valid key j (0-based over the slots) goes to
// out[j] when 0 < j < cap (the reference copies only at offsets > 0).  k_collect_count counts the
// valid bits of each 1024-slot group, and its last work-group to end turns the counts into their
// exclusive prefix; the copies that follow read only the bits and the valid records (20,000 of
// 500,000 slots: a lane per record behind its slot's flag took 20 us, now 6).  Inserts keep the bits:
// reading a flag in every slot's record was 32 MB and 11 us, with the prefix 16, now 5.
constexpr int kCollect = 1024;              // slots per group
constexpr int kWords = kCollect / 64;       // 64-bit words per group
constexpr int kCountGroups = 256 / kWords;  // groups per work-group of k_collect_count, a word per lane
struct CollectArgs {
    const Surf* keys;
    int groups;
    unsigned* counts;                // per group
    unsigned* base;                  // their exclusive prefix
    unsigned* total;
    unsigned* arrived;               // work-groups that have counted; 0 between calls
    const unsigned long long* bits;  // kWords per group, zero past the slots
};
// between work-groups of a launch: through the memory that all XCDs share
__device__ __forceinline__ void store_shared(unsigned* p, unsigned v) {
    __hip_atomic_store(FU_G(unsigned, p), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned load_shared(const unsigned* p) {
    return __hip_atomic_load(FU_G(const unsigned, p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// slot (with kPack below, else null): the `cap` slots of the copy that follows, all -1 until it writes them
__global__ __launch_bounds__(256) void k_collect_count(CollectArgs a, int* slot, unsigned cap) {
    __shared__ unsigned wsum[4];
    __shared__ int last;
    if (slot)
        for (unsigned j = blockIdx.x * 256 + threadIdx.x; j < cap; j += gridDim.x * 256) slot[j] = -1;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int group = blockIdx.x * kCountGroups + threadIdx.x / kWords;
    unsigned c = group < a.groups ? (unsigned)__popcll(a.bits[blockIdx.x * 256 + threadIdx.x]) : 0u;
#pragma unroll
    for (int d = 1; d < kWords; d <<= 1) c += __shfl_xor(c, d);
    if (group < a.groups && threadIdx.x % kWords == 0) store_shared(&a.counts[group], c);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the wave's counts are in place
    __syncthreads();
    if (threadIdx.x == 0)
        last = atomicInc(a.arrived, gridDim.x - 1u) == gridDim.x - 1u;  // and back to 0
    __syncthreads();
    if (!last) return;  // uniform
    // lane t owns a run of consecutive counts; the runs' sums are scanned across the work-group
    // (integer sums: the same as one lane walking the counts in order)
    const int per = (a.groups + 255) / 256;
    const int b = min(a.groups, (int)threadIdx.x * per), e = min(a.groups, b + per);
    unsigned own = 0;
    for (int g = b; g < e; ++g) own += load_shared(&a.counts[g]);
    unsigned x = own;  // inclusive scan over the wave
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const unsigned y = __shfl_up(x, d);
        if (lane >= d) x += y;
    }
    if (lane == 63) wsum[w] = x;
    __syncthreads();
    unsigned before = 0, all = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        before += k < w ? wsum[k] : 0u;
        all += wsum[k];
    }
    unsigned run = before + x - own;
    for (int g = b; g < e; ++g) {
        const unsigned n = load_shared(&a.counts[g]);
        a.base[g] = run;
        run += n;
    }
    if (threadIdx.x == 0) *a.total = all;
}
// A wave per word of bits, 16 lanes per record, four records at a time.  kPack: the descriptors
// alone, packed for the matcher, and each one's slot (record 0 as the zeros that CollectKeys
// leaves there, slot -1), and such zeros up to `cap`; else whole records into `out`.  Nothing is
// written from `cap` on and every slot is one of the map's or -1, whatever the bits: an insert or a
// reset that runs beside the copy, which the caller has to rule out, may change what is found, but
// nothing is read or written outside the arrays.
template <bool kPack>
__global__ __launch_bounds__(256) void k_collect_copy(CollectArgs a, Surf* out, float* desc, int* slot, unsigned cap) {
    const int word = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if constexpr (kPack) {
        for (unsigned j = *a.total + blockIdx.x * 16 + threadIdx.x / 16; j < cap; j += gridDim.x * 16)
            reinterpret_cast<uint4*>(desc)[(size_t)j * 16 + threadIdx.x % 16] = make_uint4(0u, 0u, 0u, 0u);
    }
    if (word >= a.groups * kWords) return;  // uniform
    unsigned long long m = a.bits[word];
    if (!m) return;  // uniform
    const int w = word % kWords;
    // valid records of the group's words before this one
    unsigned before = 0;
    if (lane < w) before = (unsigned)__popcll(a.bits[word - w + lane]);
#pragma unroll
    for (int d = 1; d < kWords; d <<= 1) before += __shfl_xor(before, d);
    before = (unsigned)__builtin_amdgcn_readfirstlane((int)before);
    const unsigned j0 = a.base[word / kWords] + before;
    const int sub = lane >> 4, q = lane & 15, n = __popcll(m);
    for (int k = 0; k < sub; ++k) m &= m - 1;
    for (int r = sub; r < n; r += 4) {
        const int i = word * 64 + __builtin_ctzll(m);
        const unsigned j = j0 + r;
        const uint4* src = reinterpret_cast<const uint4*>(&a.keys[i]);
        if constexpr (kPack) {
            static_assert(offsetof(Surf, desc) == 32, "two 16-byte words ahead of the descriptor");
            if (j < cap) {
                uint4 v = src[2 + q];
                if (j == 0) v = make_uint4(0u, 0u, 0u, 0u);
                reinterpret_cast<uint4*>(desc)[(size_t)j * 16 + q] = v;
                if (q == 0) slot[j] = j == 0 ? -1 : i;
            }
        } else if (j > 0 && j < cap) {
            uint4* dst = reinterpret_cast<uint4*>(&out[j]);
            dst[q] = src[q];
            if (q < 2) dst[16 + q] = src[16 + q];
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) m &= m - 1;
    }
}

__device__ __forceinline__ float clamp1(float a) {  // KeyPoints.cu:6-10
    a = a > -1.f ? a : -1.f;
    a = a < 1.f ? a : 1.f;
    return a;
}
__device__ __forceinline__ f3 spos(const SurfHead& s) { return mk3(s.pos[0], s.pos[1], s.pos[2]); }
__device__ __forceinline__ f4 snrm(const SurfHead& s) { return mk4(s.normal[0], s.normal[1], s.normal[2], s.normal[3]); }
__device__ __forceinline__ float dot4f(f4 a, f4 b) { return a.x * b.x + a.y * b.y + a.z * b.z + a.w * b.w; }

// BuildAdjecencyMatrixKernel (KeyPoints.cu:12-57), one lane per entry of the n x n matrix; the
// records' heads, `stride` heads apart
__global__ void k_adjacency(const SurfHead* frame, const SurfHead* map, int stride, const float* dist, int n, float* out) {
    const int x = blockIdx.x * 16 + (threadIdx.x & 15);
    const int y = blockIdx.y * 16 + (threadIdx.x >> 4);
    if (x >= n || y >= n) return;
    float score = 0;
    if (x == y) {
        score = expf(-dist[x]);
    } else {
        const SurfHead &m0 = map[x * stride], &m1 = map[y * stride], &f0 = frame[x * stride], &f1 = frame[y * stride];
        const float d00 = norm(sub(spos(f0), spos(f1)));
        const float d01 = norm(sub(spos(m0), spos(m1)));
        const f3 e10 = normalised(sub(spos(f0), spos(f1)));
        const f3 e11 = normalised(sub(spos(m0), spos(m1)));
        const f4 d10 = mk4(e10.x, e10.y, e10.z, 1.0f), d11 = mk4(e11.x, e11.y, e11.z, 1.0f);
        if ((double)d00 <= 1e-2 || (double)d01 <= 1e-2) {
            score = 0;
        } else {
            const float alpha00 = acosf(clamp1(dot4f(snrm(f0), snrm(f1))));
            const float beta00 = acosf(clamp1(dot4f(d10, snrm(f0))));
            const float gamma00 = acosf(clamp1(dot4f(d10, snrm(f1))));
            const float alpha01 = acosf(clamp1(dot4f(snrm(m0), snrm(m1))));
            const float beta01 = acosf(clamp1(dot4f(d11, snrm(m0))));
            const float gamma01 = acosf(clamp1(dot4f(d11, snrm(m1))));
            score = expf(-(fabsf(d00 - d01) + fabsf(alpha00 - alpha01) + fabsf(beta00 - beta01) +
                           fabsf(gamma00 - gamma01)));
        }
    }
    if (isnanf_(score)) score = 0;
    out[(size_t)y * n + x] = score;
}

}  // namespace

struct fu_keymap {
    fu_keymap_params p;
    KeyArgs a;
    unsigned* aux = nullptr;    // [0] keys left in a round, [1] valid keys, from [4] the slots' valid bits
    // aux[1] as of the last insert or reset call, kUnknown while an insert runs and after one failed
    std::atomic<long long> n_valid{0};
    // scratch of the collections (KeyScratch): the sets that no call uses, and all there are
    std::mutex lock;
    std::vector<unsigned*> idle, sets;
    int dev = -1;               // the device the map was created on
    unsigned char* done = nullptr;  // per key of an insert call, grown on demand
    int* bucket = nullptr;
    int cap = 0;
};

#define KM_HIP(call)                                                                              \
    do {                                                                                          \
        hipError_t e_ = (call);                                                                   \
        if (e_ != hipSuccess) return api_error(FU_ERR_HIP, "%s: %s", #call, hipGetErrorString(e_)); \
    } while (0)

extern "C" void fu_keymap_params_default(fu_keymap_params* p) {
    // KeyMap's constants (DeviceMap.h:165-170)
    p->grid_size = 0.01f;
    p->max_keys = 100000;
    p->n_buckets = 5;
}

extern "C" fu_status fu_keymap_destroy(fu_keymap* k) {
    if (!k) return FU_OK;
    (void)hipFree(k->a.keys);
    (void)hipFree(k->a.mutex);
    (void)hipFree(k->a.owner);
    (void)hipFree(k->aux);
    (void)hipFree(k->done);
    (void)hipFree(k->bucket);
    for (unsigned* set : k->sets) (void)hipFree(set);
    delete k;
    return FU_OK;
}

static int n_slots(const fu_keymap* k) { return k->a.max_keys * k->a.nbuckets; }
static int n_groups(const fu_keymap* k) { return (n_slots(k) + kCollect - 1) / kCollect; }
static size_t aux_bytes(const fu_keymap* k) { return (4 + (size_t)n_groups(k) * (2 * kWords)) * 4; }
constexpr long long kUnknown = -1;

// A set: total, arrived, the groups' counts and their prefix.  One is made with the map, so that
// calls that follow one another never allocate; a further one for each call that runs beside others,
// on a stream or thread of its own (sharing one, the arrivals of two calls mixed, and a prefix was
// made of counts that were not all in place).
constexpr size_t kIdleSets = 16;
static unsigned* make_set(fu_keymap* k) {
    unsigned* set = nullptr;
    const size_t bytes = (2 + 2 * (size_t)n_groups(k)) * 4;
    // cleared before any stream may use it
    if (hipMalloc(&set, bytes) == hipSuccess && hipMemset(set, 0, bytes) == hipSuccess &&
        hipStreamSynchronize(nullptr) == hipSuccess) {
        std::lock_guard<std::mutex> g(k->lock);
        k->sets.push_back(set);
        return set;
    }
    (void)hipGetLastError();
    (void)hipFree(set);
    return nullptr;
}
fu::KeyScratch::KeyScratch(fu_keymap* km, hipStream_t s) : k(km), stream(s) {
    {
        std::lock_guard<std::mutex> g(k->lock);
        if (!k->idle.empty()) {
            set = k->idle.back();
            k->idle.pop_back();
            return;
        }
    }
    set = make_set(k);
}
fu::KeyScratch::~KeyScratch() {
    // a set that kernels may still write is not used again (it is freed with the map)
    if (!set || (!waited && hipStreamSynchronize(stream) != hipSuccess)) return;
    {
        std::lock_guard<std::mutex> g(k->lock);
        if (k->idle.size() < kIdleSets) {
            k->idle.push_back(set);
            return;
        }
        for (unsigned*& x : k->sets)
            if (x == set) {
                x = k->sets.back();
                k->sets.pop_back();
                break;
            }
    }
    (void)hipFree(set);
}
static CollectArgs collect_args(const fu_keymap* k, unsigned* set) {
    const int g = n_groups(k);
    return CollectArgs{k->a.keys, g, set + 2, set + 2 + g, set, set + 1, (const unsigned long long*)k->a.bits};
}

extern "C" fu_status fu_keymap_create(const fu_keymap_params* p, fu_keymap** out) {
    if (!p || !out) return api_error(FU_ERR_ARG, "fu_keymap_create: null argument");
    *out = nullptr;
    if (p->max_keys < 1 || p->n_buckets < 1 || (long long)p->max_keys * p->n_buckets > (1ll << 28) || !(p->grid_size > 0))
        return api_error(FU_ERR_ARG, "fu_keymap_create: %u keys x %u buckets, grid %g", p->max_keys, p->n_buckets,
                         (double)p->grid_size);
    fu_keymap* k = new fu_keymap();
    k->p = *p;
    k->a.max_keys = (int)p->max_keys;
    k->a.nbuckets = (int)p->n_buckets;
    k->a.grid = p->grid_size;
    const size_t n = (size_t)n_slots(k);
    if (hipMalloc(&k->a.keys, n * sizeof(Surf)) != hipSuccess || hipMalloc(&k->a.mutex, n * 4) != hipSuccess ||
        hipMalloc(&k->a.owner, (size_t)p->max_keys * 4) != hipSuccess ||
        hipMalloc(&k->aux, aux_bytes(k)) != hipSuccess || !make_set(k)) {
        (void)hipGetLastError();
        fu_keymap_destroy(k);
        return api_error(FU_ERR_NOMEM, "fu_keymap_create: allocation failed");
    }
    k->idle = k->sets;
    // records start zeroed (ResetKeys clears only the valid flags, so a record's other bytes
    // keep what the last key there left)
    k->dev = current_device();
    k->a.bits = k->aux + 4;
    k->a.valid = k->aux + 1;
    if (hipMemset(k->a.keys, 0, n * sizeof(Surf)) != hipSuccess || hipMemset(k->aux, 0, aux_bytes(k)) != hipSuccess) {
        (void)hipGetLastError();
        fu_keymap_destroy(k);
        return api_error(FU_ERR_HIP, "fu_keymap_create: clearing the records failed");
    }
    fu_status st = fu_reset_key_points(k, nullptr);
    if (st) {
        fu_keymap_destroy(k);
        return st;
    }
    if (hipStreamSynchronize(nullptr) != hipSuccess) {
        fu_keymap_destroy(k);
        return api_error(FU_ERR_HIP, "fu_keymap_create: reset failed");
    }
    *out = k;
    return FU_OK;
}

extern "C" fu_status fu_reset_key_points(fu_keymap* k, fu_stream s) {
    if (!k) return api_error(FU_ERR_ARG, "fu_reset_key_points: null key map");
    const int n = n_slots(k);
    k->n_valid = kUnknown;
    hipLaunchKernelGGL(k_reset_keys, dim3((n + 255) / 256), dim3(256), 0, (hipStream_t)s, k->a, n);
    KM_HIP(hipGetLastError());
    k->n_valid = 0;
    return FU_OK;
}

extern "C" fu_status fu_insert_key_points(fu_keymap* k, fu_surf* keys, int32_t* index, uint32_t n, fu_stream s) {
    if (!k || (n && (!keys || !index))) return api_error(FU_ERR_ARG, "fu_insert_key_points: null argument");
    if (n == 0) return FU_OK;  // InsertKeyPoints returns at once (FuseMap.cu:459-460)
    if (n > (1u << 24)) return api_error(FU_ERR_ARG, "fu_insert_key_points: %u keys (at most 2^24)", n);
    hipStream_t hs = (hipStream_t)s;
    if ((int)n > k->cap) {
        KM_HIP(hipStreamSynchronize(hs));
        (void)hipFree(k->done);
        (void)hipFree(k->bucket);
        k->done = nullptr;
        k->bucket = nullptr;
        k->cap = 0;
        if (hipMalloc(&k->done, n) != hipSuccess || hipMalloc(&k->bucket, (size_t)n * 4) != hipSuccess) {
            (void)hipGetLastError();
            return api_error(FU_ERR_NOMEM, "fu_insert_key_points: scratch allocation failed");
        }
        k->cap = (int)n;
    }
    k->n_valid = kUnknown;
    KM_HIP(hipMemsetAsync(k->done, 0, n, hs));
    const dim3 grid((n + 255) / 256);
    // rounds until every key is placed; each round places at least the lowest waiting index
    for (uint32_t round = 0; round <= n; ++round) {
        KM_HIP(hipMemsetAsync(k->aux, 0, 4, hs));
        hipLaunchKernelGGL(k_insert_claim, grid, dim3(256), 0, hs, k->a, (const Surf*)keys, k->done, k->bucket, (int)n);
        hipLaunchKernelGGL(k_insert_apply, grid, dim3(256), 0, hs, k->a, (Surf*)keys, index, k->done, k->bucket, (int)n,
                           k->aux);
        KM_HIP(hipGetLastError());
        unsigned aux[2] = {};
        KM_HIP(hipMemcpyAsync(aux, k->aux, sizeof(aux), hipMemcpyDeviceToHost, hs));
        KM_HIP(hipStreamSynchronize(hs));
        if (aux[0] == 0) {
            k->n_valid = aux[1];
            return FU_OK;
        }
    }
    return api_error(FU_ERR_STATE, "fu_insert_key_points: inserts did not finish");
}

static void launch_count(const CollectArgs& a, int* slot, unsigned cap, hipStream_t s) {
    hipLaunchKernelGGL(k_collect_count, dim3((a.groups + kCountGroups - 1) / kCountGroups), dim3(256), 0, s, a, slot, cap);
}

extern "C" fu_status fu_collect_key_points(fu_keymap* k, fu_surf* out, uint32_t cap, uint32_t* n_keys, fu_stream s) {
    if (!k || !n_keys || (cap && !out)) return api_error(FU_ERR_ARG, "fu_collect_key_points: null argument");
    hipStream_t hs = (hipStream_t)s;
    KeyScratch scratch(k, hs);
    if (!scratch.set) return api_error(FU_ERR_NOMEM, "fu_collect_key_points: scratch allocation failed");
    const CollectArgs a = collect_args(k, scratch.set);
    launch_count(a, nullptr, 0, hs);
    if (cap)
        hipLaunchKernelGGL(k_collect_copy<false>, dim3(a.groups * (kCollect / 256)), dim3(256), 0, hs, a, (Surf*)out,
                           nullptr, nullptr, cap);
    KM_HIP(hipGetLastError());
    KM_HIP(mail_read(k->dev, n_keys, a.total, 4, hs));
    scratch.done();
    return FU_OK;
}

namespace fu {
// the number of valid keys: as the host knows it (an insert returns when its keys are in place), else
// from the device
fu_status keymap_count(const fu_keymap* k, uint32_t& n, hipStream_t s) {
    const long long known = k->n_valid;
    n = (uint32_t)known;
    if (known == kUnknown) KM_HIP(mail_read(k->dev, &n, k->a.valid, 4, s));
    return FU_OK;
}
// for n of its keys: their descriptors (n x 64, 16-byte aligned) and slots, key 0 as zeros and slot -1
fu_status keymap_pack(fu_keymap* k, const KeyScratch& scratch, float* desc, int32_t* slot, uint32_t n, hipStream_t s) {
    if (!scratch.set) return api_error(FU_ERR_NOMEM, "key map: scratch allocation failed");
    const CollectArgs a = collect_args(k, scratch.set);
    launch_count(a, slot, n, s);
    hipLaunchKernelGGL(k_collect_copy<true>, dim3(a.groups * (kCollect / 256)), dim3(256), 0, s, a, nullptr, desc, slot, n);
    KM_HIP(hipGetLastError());
    return FU_OK;
}
const SurfHead* keymap_heads(const fu_keymap* k) { return (const SurfHead*)k->a.keys; }
int keymap_device(const fu_keymap* k) { return k->dev; }
// fu_build_adjacency_matrix on the records' heads alone
fu_status build_adjacency(const SurfHead* frame, const SurfHead* map, int stride, const float* dist, int n, float* matrix,
                          hipStream_t s) {
    const dim3 grid((n + 15) / 16, (n + 15) / 16);
    hipLaunchKernelGGL(k_adjacency, grid, dim3(256), 0, s, frame, map, stride, dist, n, matrix);
    KM_HIP(hipGetLastError());
    return FU_OK;
}
}  // namespace fu

extern "C" fu_status fu_keymap_read(fu_keymap* k, fu_surf* host, fu_stream s) {
    if (!k || !host) return api_error(FU_ERR_ARG, "fu_keymap_read: null argument");
    KM_HIP(hipMemcpyAsync(host, k->a.keys, (size_t)n_slots(k) * sizeof(Surf), hipMemcpyDeviceToHost, (hipStream_t)s));
    KM_HIP(hipStreamSynchronize((hipStream_t)s));
    return FU_OK;
}

extern "C" fu_status fu_build_adjacency_matrix(const fu_surf* frame_keys, const fu_surf* map_keys, const float* dist,
                                               int32_t n, float* matrix, fu_stream s) {
    if (n < 0 || (n && (!frame_keys || !map_keys || !dist || !matrix)))
        return api_error(FU_ERR_ARG, "fu_build_adjacency_matrix: null argument or negative size");
    if (n > 46340) return api_error(FU_ERR_ARG, "fu_build_adjacency_matrix: %d pairs (the matrix index is 32-bit)", n);
    if (n == 0) return FU_OK;
    return build_adjacency((const SurfHead*)frame_keys, (const SurfHead*)map_keys, kSurfHeads, dist, n, matrix,
                           (hipStream_t)s);
}
