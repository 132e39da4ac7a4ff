// What relocalisation (reloc.hip) uses of the keypoint map (keymap.hip) beside its C ABI.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/fusion_amd.h"

namespace fu {

// a fu_surf without its descriptor
struct alignas(16) SurfHead {
    unsigned char valid;
    unsigned char pad[3];
    float pos[3];
    float normal[4];
};

// The scratch of one call's collection, from its launch until the call has waited for its stream;
// `set` is null when there is no memory for it.
class KeyScratch {
public:
    KeyScratch(fu_keymap* k, hipStream_t s);
    ~KeyScratch();
    KeyScratch(const KeyScratch&) = delete;
    KeyScratch& operator=(const KeyScratch&) = delete;
    void done() { waited = true; }  // the stream has been waited for
    unsigned* set = nullptr;

private:
    fu_keymap* k;
    hipStream_t stream;
    bool waited = false;
};
fu_status keymap_count(const fu_keymap* k, uint32_t& n, hipStream_t s);
fu_status keymap_pack(fu_keymap* k, const KeyScratch& scratch, float* desc, int32_t* slot, uint32_t n, hipStream_t s);
const SurfHead* keymap_heads(const fu_keymap* k);  // of the map's slots, kSlotHeads apart
constexpr int kSlotHeads = sizeof(fu_surf) / sizeof(SurfHead);
int keymap_device(const fu_keymap* k);
fu_status build_adjacency(const SurfHead* frame, const SurfHead* map, int stride, const float* dist, int n, float* matrix,
                          hipStream_t s);

}  // namespace fu
